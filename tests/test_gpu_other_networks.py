"""Networks of other sizes than the published one on the kernels that take them too: the row stage over other embedding
widths, class-token counts and feed-forward widths (row blocks without the next block's keys and values or without the
feed-forward half, the per-head attention of 129 to 256 tokens), and a fit over other inducing-point counts, embedding
widths and feature groups. Against the oracle at the stages' raw-score tolerance, 5e-5."""
import numpy as np
import pytest

import oracle as orc
from conftest import pkg
from test_gpu_stages import TOL, say

fit, hip, M = pkg("fit"), pkg("hip"), pkg("model")
pytestmark = pytest.mark.gpu

ROWS = {"six class tokens": dict(row_num_cls=6, icl_nhead=12), "feed-forward 128": dict(ff_factor=1),
        "six class tokens, feed-forward 512": dict(row_num_cls=6, icl_nhead=12, ff_factor=4),
        "width 64": dict(embed_dim=64, row_nhead=4, col_nhead=4),
        "width 48": dict(embed_dim=48, row_nhead=3, col_nhead=3, icl_nhead=6)}
FITS = {"64 inducing points": dict(col_num_inds=64), "192 inducing points": dict(col_num_inds=192),
        "width 64": dict(embed_dim=64, row_nhead=4, col_nhead=4), "pairs of features": dict(col_feature_group_size=2),
        "five features": dict(col_feature_group_size=5),
        "width 48, regression": dict(embed_dim=48, row_nhead=3, col_nhead=3, icl_nhead=6, max_classes=0)}


@pytest.fixture(scope="module")
def gpu():
    g = hip.Gpu(0)
    yield g
    g.close()


def network(changes):
    return M.Model.random(dict(M.FULL_CLASSIFIER, icl_num_blocks=2, **changes), seed=4)


@pytest.mark.parametrize("name", ROWS)
def test_row_stage(gpu, name):
    m = network(ROWS[name])
    w = gpu.weights(m)
    for tokens, n in ((20, 130), (41, 131), (104, 128), (129, 9), (204, 130), (256, 129)):
        tok = np.random.default_rng(tokens).standard_normal((n, tokens, m.e)).astype(np.float32)
        err = np.abs(gpu.represent(w, tok) - orc.represent(m, tok)).max()
        say(f"{name}, {n} rows of {tokens} tokens: {err:.2e}")
        assert err < TOL
    w.free()


@pytest.mark.parametrize("name", FITS)
def test_fit(gpu, name):
    m = network(FITS[name])
    w = gpu.weights(m)
    # A row of missing values has cells of -100 plus an embedding of spread s: the layer norm's mean over them carries the
    # roundings of a sum of e terms of 100, at most about 100 2^-24 sqrt(e), and divides by s.
    spread = m.t["col_y"].reshape(-1, m.e).std(1).min()
    for rows, features, missing in ((1, 3, False), (130, 7, False), (600, 3, False), (1, 3, True), (130, 7, True)):
        rng = np.random.default_rng(rows)
        x = rng.standard_normal((rows, features)).astype(np.float32)
        if missing:
            x[rows // 2] = -100.0
        y = (rng.integers(0, 10, rows) if m.max_classes else rng.standard_normal(rows)).astype(np.float32)
        col, reps = gpu.fit_represent(w, x, y, [10], np.stack([fit.query_scale(b, rows) for b in m.col_a1]))
        want, emb = orc.fit_columns(m, x, y, [10], 256)
        err = max(np.abs(col - want).max(), np.abs(reps - orc.fit_rows(m, emb)).max())
        say(f"{name}, a fit of {rows} x {features}{' with a missing row' if missing else ''}: {err:.2e}")
        assert err < TOL + (100 * 2.0 ** -24 * np.sqrt(m.e) / spread if missing else 0.0)
    w.free()
