"""Heads of very different magnitude in the fused column and row blocks and the inducing points' attention: one head's numbers are 2^30 times the others' and
have no part in the result, so that the other heads must come out as if it were not there. Against the oracle at the
stages' raw-score tolerance, 5e-5; a scale shared with the large head would leave the others eight bits.

Queries: head 0's query bias is 2^30 and its keys are zero (its weights are equal). Values: head 7's are 2^30 and the
output projection's columns for it zero."""
import numpy as np
import pytest

import oracle as orc
from conftest import pkg
from test_gpu_stages import TOL, say

abi, fit, hip, M = pkg("abi"), pkg("fit"), pkg("hip"), pkg("model")
planmod = pkg("plan")
pytestmark = pytest.mark.gpu
BIG = np.float32(2.0 ** 30)


@pytest.fixture(scope="module")
def gpu():
    g = hip.Gpu(0)
    yield g
    g.close()


def large_queries():
    m = M.Model.random(M.FULL_CLASSIFIER, seed=2)
    for b in m.col_a1 + m.col_a2 + m.row[:-1]:
        e = b.d
        b.t["in_b"][:16] = BIG
        b.t["in_w"].reshape(3 * e, e)[e:e + 16] = 0.0
        b.t["in_b"][e:e + 16] = 0.0
    return m


def large_values():
    m = M.Model.random(M.FULL_CLASSIFIER, seed=2)
    for b in m.col_a1 + m.col_a2 + m.row[:-1]:
        e = b.d
        b.t["in_b"][2 * e + 112:] = BIG
        b.t["out_w"].reshape(e, e)[:, 112:] = 0.0
    return m


@pytest.fixture(scope="module", params=["queries", "values"])
def kind(request):
    return request.param


@pytest.fixture(scope="module")
def model(kind):
    return large_queries() if kind == "queries" else large_values()


@pytest.fixture(scope="module")
def weights(gpu, model):
    return gpu.weights(model)


@pytest.mark.parametrize("tokens,n", [(41, 131), (104, 130), (204, 129)])
def test_row_blocks(gpu, kind, model, weights, tokens, n):
    tok = np.random.default_rng(tokens).standard_normal((n, tokens, model.e)).astype(np.float32)
    err = np.abs(gpu.represent(weights, tok) - orc.represent(model, tok)).max()
    say(f"large {kind}, {n} rows of {tokens} tokens: {err:.2e}")
    assert err < TOL


def test_column_blocks(gpu, kind, model, weights):
    n, features, rows = 130, 9, 64
    rng = np.random.default_rng(5)
    col = (rng.standard_normal((features, 1, len(model.col_a2), 2, model.e, model.inds)) * 0.5).astype(np.float32)
    if kind == "queries":
        col[:, :, :, 0, :16] = 0.0
    else:
        col[:, :, :, 1, 112:] *= BIG
    layers = [orc.pack((rng.standard_normal(2 * model.d * rows) * 0.5).astype(np.float32), model.d, rows, abi.KV_F32)
              for _ in range(model.icl_layers)]
    scales = np.stack([orc.query_scale(b, rows) for b in model.icl])
    vm = gpu.load(weights, abi.KV_F32, rows, 64, layers, scales)
    vm.set_columns(col, features, 1)
    x = rng.standard_normal((n, features)).astype(np.float32)
    fitted = orc.Fitted(rows, features, 10, 64, abi.KV_F32,
                        planmod.Plan([10], [planmod.Node(None, [], 10, True, list(range(10)))]), col, [scales], [layers])
    err = np.abs(gpu.embed(weights, vm, x) - orc.embed(model, fitted, x)).max()
    say(f"large {kind}, embeddings: {err:.2e}")
    assert err < TOL


def test_fit_columns(gpu, kind, model, weights):
    rng = np.random.default_rng(7)
    x, y = rng.standard_normal((300, 5)).astype(np.float32), rng.integers(0, 10, 300).astype(np.float32)
    got, reps = gpu.fit_represent(weights, x, y, [10], np.stack([fit.query_scale(b, 300) for b in model.col_a1]))
    want, emb = orc.fit_columns(model, x, y, [10], 256)
    keep = np.abs(want) < 1e6  # all but the large head's values
    err = max(np.abs(got - want)[keep].max(), np.abs(reps - orc.fit_rows(model, emb)).max())
    say(f"large {kind}, a fit: {err:.2e}")
    assert err < TOL


@pytest.mark.parametrize("place", [0, 350, 699])
def test_outlying_cell(gpu, place):
    """A row a million times the others', first, within and last of the inducing points' ranges of cells: the scale that
    their keys and values take from it must not cost the others, nor depend on where it stands."""
    m = M.Model.random(M.FULL_CLASSIFIER, seed=2)
    w = gpu.weights(m)
    rng = np.random.default_rng(9)
    x, y = rng.standard_normal((700, 3)).astype(np.float32), rng.integers(0, 10, 700).astype(np.float32)
    x[place] *= 1e6
    got, reps = gpu.fit_represent(w, x, y, [10], np.stack([fit.query_scale(b, 700) for b in m.col_a1]))
    want, emb = orc.fit_columns(m, x, y, [10], 256)
    # head by head, each against its own size
    g, t = (a.reshape(3, 3, 2, 8, 16, m.inds) for a in (got, want))
    off = np.abs(g - t).max(axis=(0, 4, 5)) / np.abs(t).max(axis=(0, 4, 5))
    say(f"an outlying cell at {place}: {off.max():.2e} of a head, rows {np.abs(reps - orc.fit_rows(m, emb)).max():.2e}")
    assert off.max() < TOL and np.abs(reps - orc.fit_rows(m, emb)).max() < TOL
