"""The GEMM tile the library takes without a tuning table, as the autotuner reports
it (no GPU)."""
import pytest


@pytest.mark.parametrize("M,N,batch,tile", [
    (162, 162, 1024, 5), (81, 162, 1, 5), (1, 1, 1, 5), (1250, 2500, 8, 4), (1250, 2500, 2, 5), (1024, 1024, 8, 4),
    (1024, 1024, 7, 5), (1023, 1024, 64, 5), (1024, 1023, 64, 5)])
def test_library_tile(M, N, batch, tile):
    from khepri_amd import autotune
    assert autotune.library_tile(M, N, batch) == tile


def test_bad_shapes_are_refused():
    from khepri_amd import autotune
    with pytest.raises(ValueError):
        autotune.library_tile(0, 4, 1)
