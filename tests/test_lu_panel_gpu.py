"""The LU's register panel against its LDS panel: pivot rows that tie (matrices of
small integers), one to three rows per thread, panels narrower than 16, few and
many right-hand sides.  The same pivots and the same sums: equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 100, 256, 257, 512, 513, 1025])
def test_ties_and_edges(gpu, monkeypatch, n):
    import torch
    from khepri_amd import ops
    rng = np.random.default_rng(n)
    A = np.stack([rng.integers(-2, 3, (n, n)) + 1j * rng.integers(-2, 3, (n, n)),
                  rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))])
    out = []
    for reg in ("0", "1"):
        monkeypatch.setenv("KHX_LU_PANEL_REG", reg)
        res = []
        for m in (3, 70):
            B = np.random.default_rng(m).normal(size=(2, n, m)) + 0j
            X, info = ops.solve(torch.as_tensor(A, device=gpu), torch.as_tensor(B, device=gpu))
            res += [X.cpu().numpy(), info.cpu().numpy()]
        res += [t.cpu().numpy() for t in ops.lu_factor(torch.as_tensor(A, device=gpu))]
        out.append(res)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
