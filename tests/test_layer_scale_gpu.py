"""khx_layer_scale against the largest eigenvalue of P Q from numpy: ordinary,
lossy and metallic maps, one-dimensional bases, long waves, and maps whose
permittivity changes sign, whose largest eigenvalues come in pairs of opposite
sign so that one step of the power iteration grows and the next shrinks.

Bound: the approximant's error is one rounding (1e-16) up to |x| = 4.7 and grows
with the 35th power, so an estimate may be 0.85 of the true value (4 / 4.7)."""
import numpy as np
import pytest

from oracle import rcwa

pytestmark = pytest.mark.gpu


def draw(kind, seed):
    rng = np.random.default_rng(seed)
    x, y = np.meshgrid(np.linspace(-0.5, 0.5, 48), np.linspace(-0.5, 0.5, 48), indexing="ij")
    if kind == "sign":
        v = np.where(rng.random(3) < 0.5, rng.uniform(0.5, 6, 3), -rng.uniform(0.5, 6, 3)) - 1j * rng.uniform(0, 0.05, 3)
    elif kind == "metal":
        v = np.array([1.0, -12.0 - 1.0j, 2.25])
    else:
        v = rng.uniform(1.0, 12.0, 3) - 1j * (rng.uniform(0, 0.5, 3) if kind == "lossy" else 0)
    eps = np.full((48, 48), v[0])
    for k in (1, 2):
        cx, cy, r = rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3), rng.uniform(0.1, 0.4)
        eps[(x - cx) ** 2 + (y - cy) ** 2 < r * r] = v[k]
    pw = [(3, 3), (5, 5), (5, 3), (7, 1)][rng.integers(4)]
    return eps, pw, rng.uniform(0.6, 4), rng.uniform(-3, 3, 2)


@pytest.mark.parametrize("kind,seeds", [
    ("sign", [1490, 1592, 1366, 1543, 1421, 286, 547, 2570, 1978, 2112, 2036, 566]), ("real", range(12)),
    ("lossy", range(12)), ("metal", range(12))])
def test_estimate_is_not_far_below(gpu, kind, seeds):
    import torch
    from khepri_amd import Crystal, ops
    from khepri_amd.layer import Layer
    low = {}
    for seed in seeds:
        eps, pw, wl, kp = draw(kind, seed)
        e = Crystal(pw).expansion
        C, IC = Layer.pixmap(e, eps, 1.0).convolution_matrices(gpu)
        kx, ky = ops.kvectors(e.g_device(gpu), torch.as_tensor(kp[None] + 0j, device=gpu),
                              torch.as_tensor([wl], dtype=torch.float64, device=gpu))
        got = ops.layer_scale(C, IC, kx, ky, torch.ones(1, dtype=torch.float64, device=gpu)).item()
        ox, oy, _ = rcwa.k_vectors(rcwa.g_vectors(pw, rcwa.lattice_matrix("square")), kp, wl)
        _, _, lam = rcwa.structured_layer_modes(ox, oy, rcwa.convolution_matrix(eps, pw))
        low[seed] = got / (0.5 * np.abs(lam).max())
    assert min(low.values()) >= 0.85, low
