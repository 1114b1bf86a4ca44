"""The regression head at the edges of its kernel's sizes: the keys a lane holds (2, 4, 8, 16 for up to 128, 256, 512,
1,024 quantiles), row counts that leave a workgroup's last rows, wavefronts or lanes without work, and levels that
spread the reading over one to seven wavefronts. Against the host statement, as in test_gpu_quantiles: the moments and
inner quantiles bit for bit, the tails at its 5e-5."""
import numpy as np
import pytest

from conftest import pkg
from test_gpu_quantiles import host_stats, rows_of, say

dm, hip = pkg("devmem"), pkg("hip")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    g = hip.Gpu(0)
    yield g
    g.close()


@pytest.mark.parametrize("n,rows,levels", [(2, 5, 1), (3, 9, 0), (127, 513, 3), (128, 17, 64), (129, 1025, 8),
                                           (256, 40, 11), (257, 700, 2), (511, 33, 1), (512, 5, 6), (513, 4099, 6),
                                           (1000, 8209, 2), (1023, 31, 64), (1024, 520, 5)])
def test_quantile_sizes(gpu, n, rows, levels):
    say(f"quantile sizes n={n} rows={rows} levels={levels}")
    rng = np.random.default_rng(n + rows)
    q = rows_of(rng, rows, n) if n > 7 else rng.standard_normal((rows, n)).astype(np.float32)
    alphas = np.sort(rng.uniform(1e-4, 1 - 1e-4, levels)).astype(np.float32)
    got = gpu.quantile_stats(q, alphas)
    # every row's moments and order are the host's; a sample of the rows where there are many
    pick = np.unique(np.concatenate([np.arange(min(rows, 40)), np.arange(max(0, rows - 20), rows),
                                     rng.integers(0, rows, 40)]))
    want = host_stats(q[pick], alphas)
    got = got[pick]
    lo, hi = np.float32(1) / np.float32(n + 1), np.float32(n) / np.float32(n + 1)
    inner = np.concatenate([[True, True, True], (alphas >= lo) & (alphas <= hi)])
    assert np.array_equal(got[:, inner], want[:, inner], equal_nan=True)
    gt, wt = got[:, ~inner], want[:, ~inner]
    ok = np.isfinite(wt)
    assert np.array_equal(np.isfinite(gt), ok)
    if ok.any():
        assert (np.abs(gt[ok] - wt[ok]) / np.maximum(np.abs(wt[ok]), 1.0)).max() < 5e-5


def test_every_row_count(gpu):
    """The largest row count there is, two quantiles a row (43 GB of quantiles and statistics on the card): a million rows
    over and over, whose statistics come out alike everywhere, at the ends and wherever a launch could end."""
    rows, period = 2 ** 31 - 1, 1 << 20
    rng = np.random.default_rng(11)
    part = rng.standard_normal((period, 2)).astype(np.float32)
    want = gpu.quantile_stats(part, np.zeros(0, np.float32))
    try:
        q, out = dm.DeviceBuffer(rows * 8), dm.DeviceBuffer(rows * 12)
    except RuntimeError:
        pytest.skip("needs 43 GB of free memory on the card")
    say(f"quantile sizes n=2 rows={rows}")
    q.upload(part)
    at = period
    while at < rows:  # the rows so far once more behind themselves
        n = min(at, rows - at)
        assert dm.rt().hipMemcpy(q.ptr + 8 * at, q.ptr, 8 * n, 3) == 0
        at += n
    dm.synchronize()
    gpu.quantile_stats_dev(q.ptr, rows, 2, np.zeros(0, np.float32), out.ptr)
    got = np.empty((period, 3), np.float32)
    for k in sorted({0, 2047} | set(range(127, 2048, 128)) | set(range(128, 2048, 128))):
        n = min(period, rows - k * period)
        assert dm.rt().hipMemcpy(got.ctypes.data, out.ptr + 12 * k * period, 12 * n, dm.D2H) == 0
        assert np.array_equal(got[:n], want[:n]), k
    q.free()
    out.free()
