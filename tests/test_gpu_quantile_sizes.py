"""The regression head at the edges of its kernel's sizes: the keys a lane holds (2, 4, 8, 16 for up to 128, 256, 512,
1,024 quantiles), row counts that leave a workgroup's last rows, wavefronts or lanes without work, and levels that
spread the reading over one to seven wavefronts. Against the host statement, as in test_gpu_quantiles: the moments and
inner quantiles bit for bit, the tails at its 5e-5."""
import numpy as np
import pytest

from conftest import pkg
from test_gpu_quantiles import host_stats, rows_of, say

hip = pkg("hip")
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
