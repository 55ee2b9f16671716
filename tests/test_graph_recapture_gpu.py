"""Captured graphs whose new sources want other doubling counts of the layer
S-matrices.  A replay is the eager call on the new sources, bit for bit: it runs
the same kernels on the same inputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIXELS = np.random.default_rng(5).uniform(2.0, 12.0, (32, 32))
WL = np.array([1.8, 1.9])
FAR = np.array([[0.3, 0.2], [90.0, 80.0]])   # far evanescent: more doublings


def crystal(pw=(7, 7), depth=0.3):
    from khepri_amd import Crystal
    cl = Crystal(pw)
    cl.add_layer_pixmap("P", PIXELS, depth)
    cl.set_device(["P"], False)
    return cl


def counts(cl, **source):
    """The doubling counts of a crystal's layer P at these sources."""
    import torch
    from khepri_amd.layer import plan_layers
    cl.set_source(WL, 1.0, 0.3, **source)
    kp, wl = (torch.as_tensor(x, device=cl._dev()) for x in (cl._kp, cl._wl))
    return list(plan_layers([cl.layers["P"]], kp, wl).values())[0].counts.tolist()


@pytest.mark.parametrize("source", [dict(theta=45.0), dict(kp=FAR)])
def test_gradient_graph_reads_the_new_sources(gpu, source):
    from khepri_amd.adjoint import flux_gradient
    from khepri_amd.graph import GradientGraph
    first = dict(theta=0.0)
    assert counts(crystal(), **first) != counts(crystal(), **source)
    cl = crystal()
    cl.set_source(WL, 1.0, 0.3, **first)
    g = GradientGraph(cl, wT=1.0)
    for src in (source, first, source):
        g.update_sources(WL, 1.0, 0.3, **src)
        R, T, grads = g.replay()
        ref = crystal()
        ref.set_source(WL, 1.0, 0.3, **src)
        Rr, Tr, gr = flux_gradient(ref, wT=1.0)
        np.testing.assert_array_equal(R, Rr)
        np.testing.assert_array_equal(T, Tr)
        np.testing.assert_array_equal(grads["P"].cpu().numpy(), gr["P"].cpu().numpy())


def test_solve_graph_after_an_eager_solve(gpu):
    """The eager solve in between leaves its own source tensors in the crystal."""
    from khepri_amd.graph import SolveGraph
    assert counts(crystal((3, 3)), theta=0.0) != counts(crystal((3, 3)), kp=FAR)
    cl = crystal((3, 3))
    cl.set_source(WL, 1.0, 0.3)
    g = SolveGraph(cl)
    cl.set_source(1.1 * WL, 0.2, 1.0, theta=12.0)
    cl.solve()
    g.update_sources(WL, 1.0, 0.3, kp=FAR)
    ref = crystal((3, 3))
    ref.set_source(WL, 1.0, 0.3, kp=FAR)
    ref.solve()
    for _ in range(2):
        for a, b in zip(g.replay(), ref.poynting_flux_end()):
            np.testing.assert_array_equal(a, b)


def test_gradient_graph_is_captured_once(gpu):
    """Its launches go through the modes: no new sources change them."""
    from khepri_amd.graph import GradientGraph
    cl = crystal((3, 3))
    cl.set_source(WL, 1.0, 0.3)
    g = GradientGraph(cl, wT=1.0)
    graph, buffers = g.graph, g.outputs[2]["P"].data_ptr()
    for src in (dict(kp=FAR), dict(kp=FAR), dict(theta=0.0)):
        g.update_sources(WL, 1.0, 0.3, **src)
        assert g.graph is graph and g.outputs[2]["P"].data_ptr() == buffers


def test_solve_graph_is_captured_once_per_plan(gpu):
    from khepri_amd.graph import SolveGraph
    cl = crystal((3, 3))
    cl.set_source(WL, 1.0, 0.3)
    g = SolveGraph(cl)
    graph = g.graph
    g.update_sources(1.01 * WL, 1.0, 0.3)
    assert g.graph is graph
    g.update_sources(WL, 1.0, 0.3, kp=FAR)
    graph2 = g.graph
    assert graph2 is not graph
    g.update_sources(1.01 * WL, 1.0, 0.3, kp=FAR)
    assert g.graph is graph2


@pytest.mark.parametrize("rt_only", [None, True])
def test_new_sources_leave_the_crystal_unsolved(gpu, rt_only):
    """update_sources ran nothing for the crystal itself, recaptured or not: its
    results, which a capture only records, cannot be read."""
    from khepri_amd.graph import SolveGraph
    cl = crystal((3, 3))
    cl.set_source(WL, 1.0, 0.3)
    g = SolveGraph(cl, rt_only=rt_only)
    for src in (dict(theta=1.0), dict(kp=FAR)):
        g.update_sources(WL, 1.0, 0.3, **src)
        assert not cl.solved
        with pytest.raises(AssertionError):
            cl.poynting_flux_end()
