"""Gauss-Jordan solve (khx_zgesv_ws, lu_gj.hip) against numpy, at the
orders where its tiling changes: one panel and less (1, 15, 16, 17), the edges of
the wavefront tilings (64/65, 128/129, 192/193, 256/257, 384/385, 512) and
beyond them (the LU path), right-hand sides around the 16- and 32-column strips,
batches below and above the strip rule.

Tolerance: forward error <= 1e-16 * n * cond(A) * 64 (growth of partial
pivoting on random matrices stays far below 64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(A, B, gpu):
    import torch
    from khepri_amd import ops
    X, info = ops.solve_conditioned(torch.as_tensor(A, device=gpu), torch.as_tensor(B, device=gpu))
    return X.cpu().numpy(), info.cpu().numpy()


@pytest.mark.parametrize("n,m,batch", [
    (1, 1, 3), (2, 5, 1), (15, 16, 2), (16, 17, 2), (17, 1, 2), (31, 33, 3), (50, 50, 70), (64, 31, 2), (65, 64, 2),
    (98, 97, 130), (128, 16, 2), (129, 40, 2), (162, 162, 3), (162, 162, 90), (192, 15, 2), (193, 33, 2),
    (256, 20, 2), (257, 50, 2), (338, 100, 2), (384, 32, 1), (385, 17, 1), (512, 48, 1), (513, 70, 1)])
def test_orders_and_strips(gpu, n, m, batch):
    rng = np.random.default_rng(n * 1000 + m)
    A = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    B = rng.normal(size=(batch, n, m)) + 1j * rng.normal(size=(batch, n, m))
    X, info = _solve(A, B, gpu)
    assert (info == 0).all()
    for b in {0, batch // 2, batch - 1}:
        ref = np.linalg.solve(A[b], B[b])
        err = np.linalg.norm(X[b] - ref) / np.linalg.norm(ref)
        assert err <= 64e-16 * n * np.linalg.cond(A[b]), (b, err)


@pytest.mark.parametrize("n", [18, 50, 130])
def test_pivots_far_from_the_diagonal(gpu, n):
    """A reversed diagonal with small noise: every pivot row lies in another
    wavefront's rows than its column; scales from 1e-200 to 1e200."""
    rng = np.random.default_rng(n)
    A = (rng.normal(size=(4, n, n)) + 1j * rng.normal(size=(4, n, n))) * 1e-3
    A[:, np.arange(n), n - 1 - np.arange(n)] += 2.0 + 1.0j
    scale = np.array([1.0, 1e-200, 1e200, 1e-30])[:, None, None]
    B = rng.normal(size=(4, n, 7)) + 1j * rng.normal(size=(4, n, 7))
    X, info = _solve(A * scale, B, gpu)
    assert (info == 0).all()
    for b in range(4):
        ref = np.linalg.solve(A[b], B[b])
        assert np.abs(X[b] * scale[b] - ref).max() <= 64e-16 * n * np.linalg.cond(A[b]) * np.abs(ref).max()


@pytest.mark.parametrize("n", [3, 50, 162])
def test_singular_and_nan_items(gpu, n):
    """An exactly singular item is reported with its first zero pivot and leaves
    the others alone; a NaN item gives NaN."""
    rng = np.random.default_rng(3)
    A = rng.normal(size=(4, n, n)) + 1j * rng.normal(size=(4, n, n))
    B = rng.normal(size=(4, n, 4)) + 0j
    A[1, :, n - 1] = 0.0
    A[2, n // 2, 0] = np.nan
    X, info = _solve(A, B, gpu)
    assert info[0] == 0 and info[3] == 0 and info[1] == n
    assert np.isnan(X[2]).all() and not np.isfinite(X[1]).any()
    for b in (0, 3):
        ref = np.linalg.solve(A[b], B[b])
        assert np.linalg.norm(X[b] - ref) <= 64e-16 * n * np.linalg.cond(A[b]) * np.linalg.norm(ref)


@pytest.mark.parametrize("n,m,batch", [
    (15, 3, 513), (64, 5, 513), (100, 4, 513), (129, 20, 33), (192, 9, 256), (193, 17, 255), (193, 17, 256),
    (256, 3, 256), (257, 40, 257)])
def test_columns_and_rows_by_batch(gpu, n, m, batch):
    """Around the batches and orders where the columns of a launch (32, 64, 128,
    all) and the rows of a wavefront change; a zero column, in a later launch
    where there are several, is reported."""
    rng = np.random.default_rng(n + batch)
    A = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    B = rng.normal(size=(batch, n, m)) + 1j * rng.normal(size=(batch, n, m))
    zero = 3 * n // 4
    A[1, :, zero] = 0.0
    X, info = _solve(A, B, gpu)
    assert info[1] == zero + 1 and (np.delete(info, 1) == 0).all()
    for b in (0, batch // 2, batch - 1):
        ref = np.linalg.solve(A[b], B[b])
        err = np.linalg.norm(X[b] - ref) / np.linalg.norm(ref)
        assert err <= 64e-16 * n * np.linalg.cond(A[b]), (b, err)


@pytest.mark.parametrize("n,batch,wide", [(2, 3, "neither"), (18, 40, "a"), (50, 2, "b"), (530, 2, "neither")])
def test_star_product_with_one_solve(gpu, n, batch, wide):
    """redheffer(gj=True) against the formula with two solves, per item and with
    either operand shared by the batch.  Blocks of norm ~1/2: cond(D) < 2, so the
    products' rounding is all there is (64 n eps)."""
    import torch
    from khepri_amd import ops
    rng = np.random.default_rng(n)

    def draw(count):
        S = rng.normal(size=(count, 2, 2, n, n)) + 1j * rng.normal(size=(count, 2, 2, n, n))
        return S / (4 * np.sqrt(2 * n))
    A, B = draw(1 if wide == "a" else batch), draw(1 if wide == "b" else batch)
    put = lambda S: torch.as_tensor(S[0] if wide != "neither" and len(S) == 1 else S, device=gpu)   # noqa: E731
    S, info = ops.redheffer(put(A), put(B), gj=True)
    assert (info.cpu().numpy() == 0).all()
    S = S.cpu().numpy()
    for b in (0, batch - 1):
        a, c = A[b % len(A)], B[b % len(B)]
        D, F = np.eye(n) - c[0, 0] @ a[1, 1], np.eye(n) - a[1, 1] @ c[0, 0]
        ref = np.array([[a[0, 0] + a[0, 1] @ np.linalg.solve(D, c[0, 0]) @ a[1, 0], a[0, 1] @ np.linalg.solve(D, c[0, 1])],
                        [c[1, 0] @ np.linalg.solve(F, a[1, 0]), c[1, 1] + c[1, 0] @ np.linalg.solve(F, a[1, 1]) @ c[0, 1]]])
        assert np.linalg.norm(S[b] - ref) <= 64e-16 * n * np.linalg.norm(ref)
