"""Calls under a working-memory budget whose last batch is shorter than the others. From 128 rows (rows of more than 128
tokens; else 512) the row stage takes a compact layout, so that a shorter batch below that count needs more memory than a
full one above it: a budget between the two must give smaller batches, not an error on the last one, and a row batch
that a caller was told of must hold for every smaller call. Against the same calls without a budget."""
import numpy as np
import pytest

import oracle as orc
from conftest import pkg
from test_gpu_stages import TOL, say

abi, fit, hip, M = pkg("abi"), pkg("fit"), pkg("hip"), pkg("model")
pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def gpu():
    g = hip.Gpu(0)
    yield g
    g.close()


@pytest.fixture(scope="module")
def model():
    return M.Model.random(M.FULL_CLASSIFIER, seed=2)


@pytest.fixture(scope="module")
def weights(gpu, model):
    return gpu.weights(model)


def budgeted(gpu, megabytes, call):
    old = gpu.work_budget()
    gpu.release()
    try:
        gpu.set_work_budget(megabytes * MB)
        out = call()
        now, peak = gpu.working()
        assert peak <= megabytes * MB
        return out
    finally:
        gpu.set_work_budget(old)


@pytest.mark.parametrize("tokens,n,megabytes", [(204, 1033, 60), (204, 1033, 90), (257, 300, 90), (24, 1537, 30)])
def test_represent(gpu, model, weights, tokens, n, megabytes):
    say(f"{n} rows of {tokens} tokens in {megabytes} MB")
    tok = np.random.default_rng(tokens).standard_normal((n, tokens, model.e)).astype(np.float32)
    want = gpu.represent(weights, tok)
    got = budgeted(gpu, megabytes, lambda: gpu.represent(weights, tok))
    assert np.abs(got - want).max() < TOL


@pytest.mark.parametrize("n,features,megabytes", [(1033, 200, 64), (1033, 200, 96), (1537, 20, 40)])
def test_predict(gpu, model, weights, n, features, megabytes):
    say(f"{n} x {features} predicted in {megabytes} MB")
    rows = 64
    rng = np.random.default_rng(n + features)
    layers = [orc.pack((rng.standard_normal(2 * model.d * rows) * 0.5).astype(np.float32), model.d, rows, abi.KV_F32)
              for _ in range(model.icl_layers)]
    vm = gpu.load(weights, abi.KV_F32, rows, 64, layers, np.stack([orc.query_scale(b, rows) for b in model.icl]))
    vm.set_columns((rng.standard_normal((features, 1, len(model.col_a2), 2, model.e, model.inds)) * 0.5)
                   .astype(np.float32), features, 1)
    x = rng.standard_normal((n, features)).astype(np.float32)
    want = gpu.predict(weights, vm, x, 10)
    got = budgeted(gpu, megabytes, lambda: gpu.predict(weights, vm, x, 10))
    assert np.abs(got - want).max() < TOL


@pytest.mark.parametrize("features,megabytes", [(200, 100), (200, 160), (20, 60), (20, 200)])
def test_row_batch_holds_for_smaller_calls(gpu, model, weights, features, megabytes):
    rng = np.random.default_rng(features)

    def call():
        most = gpu.row_batch(weights, features)
        assert most > 0
        say(f"row batch of {features} features in {megabytes} MB: {most}")
        for n in sorted({k for k in (1, 127, 128, 511, 512, most // 2, most) if 0 < k <= most}):
            gpu.rows(weights, rng.standard_normal((n, features, model.e)).astype(np.float32))
        return most

    budgeted(gpu, megabytes, call)


def test_fit(gpu, model, weights):
    """A fit's row stage: 1,033 rows of 200 features, whose cells alone take 106 MB."""
    rng = np.random.default_rng(3)
    x, y = rng.standard_normal((1033, 200)).astype(np.float32), rng.integers(0, 10, 1033).astype(np.float32)
    scales = np.stack([fit.query_scale(b, 1033) for b in model.col_a1])
    want, reps = gpu.fit_represent(weights, x, y, [10], scales)
    for megabytes in (280, 320):
        got, r = budgeted(gpu, megabytes, lambda: gpu.fit_represent(weights, x, y, [10], scales))
        say(f"a fit in {megabytes} MB: {np.abs(r - reps).max():.2e}")
        assert max(np.abs(got - want).max(), np.abs(r - reps).max()) < TOL
