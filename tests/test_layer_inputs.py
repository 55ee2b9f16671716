"""Layers and batches that the chain takes beside its own solved layers."""
import numpy as np
import pytest


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
