"""Layers and batches that the chain takes beside its own solved layers: objects
with the layer protocol, subclasses, hand-made S-matrices, empty batches."""
import numpy as np
import pytest
import torch


class Own:
    """The protocol of Crystal.add_layer: solve_batch(kp, wl, ws, rt_only)."""
    depth, fields, S = 0.3, False, None

    def solve_batch(self, kp, wl, ws=None, rt_only=False):
        self.S = (kp, wl, rt_only)


def test_layer_objects_with_the_plain_protocol():
    from khepri_amd.layer import Layer, plan_layers
    kp, wl = torch.zeros((2, 2), dtype=torch.complex128), torch.ones(2, dtype=torch.float64)
    ly = Own()
    assert plan_layers([ly], kp, wl) == {}
    Layer.solve_batch_many([ly], kp, wl, rt_only=True)
    assert ly.S[2] is True


def test_subclass_with_its_own_solve_batch():
    """Its solve decides what becomes of the S-matrix: nothing is planned for it."""
    from khepri_amd import Crystal
    from khepri_amd.layer import Layer, plan_layers

    class Sub(Layer):
        def solve_batch(self, kp, wl, ws=None, rt_only=False):
            self.S = kp
    kp, wl = torch.zeros((2, 2), dtype=torch.complex128), torch.ones(2, dtype=torch.float64)
    ly = Sub.pixmap(Crystal((1, 1)).expansion, np.eye(8) + 1.0, 0.3)
    assert plan_layers([ly], kp, wl) == {}
    Layer.solve_batch_many([ly], kp, wl)
    assert ly.S is kp


def test_extended_layer_over_such_a_base():
    from khepri_amd.extension import ExtendedLayer
    from khepri_amd.layer import Layer

    class Sub(Layer):
        def solve_batch(self, kp, wl, ws=None, rt_only=False):
            raise StopIteration                    # reached with the plain arguments
    base = Sub()
    base.formulation, base.expansion = 1, None
    ext = ExtendedLayer.__new__(ExtendedLayer)
    ext.__dict__.update(base=base, fields=False, mode=0, gs=np.zeros((2, 1)))
    kp, wl = torch.zeros((2, 2), dtype=torch.complex128), torch.ones(2, dtype=torch.float64)
    assert ext.plan(kp, wl) is None
    with pytest.raises(StopIteration):
        ext.solve_batch(kp, wl)


def _recorded(monkeypatch):
    """ops.redheffer replaced by a record of its operands."""
    from khepri_amd import ops
    seen = []

    def redheffer(SA, SB, ws=None, gj=False):
        seen.append((SA, SB))
        return SA, None
    monkeypatch.setattr(ops, "redheffer", redheffer)
    return seen


def test_stack_layers_reads_the_given_s(monkeypatch):
    """stack_layers multiplies the S-matrices that its layers hold, whatever their
    permittivity says and also where a layer has none."""
    from khepri_amd import Crystal
    from khepri_amd.layer import Layer, stack_layers
    e = Crystal((1, 1)).expansion
    seen = _recorded(monkeypatch)
    layers = [Layer(), Layer.half_infinite(e, "reflexion", 1), Layer.uniform(e, 1, 0.3), Layer.uniform(e, 2.0, 0.3)]
    for k, ly in enumerate(layers):
        ly.S = torch.full((1, 2, 2, 2, 2), k, dtype=torch.complex128)
    layers[2].X = torch.ones((1, 2), dtype=torch.complex128)   # of an earlier solve
    stack_layers(None, layers, [True, False, False, True], reverse=False)
    assert [id(b) for _, b in seen] == [id(ly.S) for ly in layers[1:]]
    assert seen[0][0] is layers[0].S


def test_fold_is_for_layers_as_solved_by_the_library(monkeypatch):
    """Where the stack was just solved, gap-medium layers fold; those of another solve_batch do not."""
    from khepri_amd import Crystal
    from khepri_amd.layer import Layer, stack_layers

    class Sub(Layer):
        def solve_batch(self, kp, wl, ws=None, rt_only=False):
            super().solve_batch(kp, wl, ws, rt_only)
    e = Crystal((1, 1)).expansion
    for kind, products in ((Layer, 0), (Sub, 1)):
        seen = _recorded(monkeypatch)
        layers = [kind.half_infinite(e, "reflexion", 1), Layer.uniform(e, 2.0, 0.3)]
        for ly in layers:
            ly.S = torch.zeros((1, 2, 2, 2, 2), dtype=torch.complex128)
        Stot = stack_layers(None, layers, [True, True], reverse=False, solved=True)[2]
        assert len(seen) == products
        assert Stot is (layers[1].S if products == 0 else layers[0].S)


def test_folded_stack_keeps_the_copies_the_mask_names(monkeypatch):
    """The mask of a stack without half spaces (void crystal) is two longer than the
    stack: its entry for the last layer decides, as it does without folding."""
    from khepri_amd import Crystal
    from khepri_amd.layer import Layer, stack_layers
    e = Crystal((1, 1)).expansion
    _recorded(monkeypatch)
    layers = [Layer.uniform(e, 2.0, 0.3), Layer.uniform(e, 3.0, 0.3)]
    for ly in layers:
        ly.S = torch.zeros((1, 2, 2, 2, 2), dtype=torch.complex128)
    for mask in ([True, False, False, True], [False, True], [True, True]):
        copies = [[S is not None for S in stack_layers(None, layers, mask, reverse=False, solved=solved)[0]]
                  for solved in (False, True)]
        assert copies[0] == copies[1] == mask[:2]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["pixmap", "uniform"])
def test_empty_batch(gpu, kind):
    """No sources: empty R and T of the streamed chain, an empty S of a layer; the
    resident chain, which multiplies S-matrices, refuses them."""
    from khepri_amd import Crystal, workloads as W
    cl = Crystal((3, 3))
    eps = W.disc_pixmap(64, 9.0, 0.3, 1.0) if kind == "pixmap" else 2.0
    (cl.add_layer_pixmap if kind == "pixmap" else cl.add_layer_uniform)("P", eps, 0.5)
    cl.set_device(["P"], False)
    cl.set_source(np.zeros(0), kp=np.zeros((0, 2)))
    cl.solve(rt_only=True)
    assert [len(x) for x in cl.poynting_flux_end()] == [0, 0]
    with pytest.raises(ValueError):
        cl.solve(rt_only=False)
    if kind == "pixmap":
        cl.layers["P"].solve(np.zeros((0, 2)), np.zeros(0))
        assert cl.layers["P"].S.shape == (0, 2, 2, 18, 18)
