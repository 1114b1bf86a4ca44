"""The row stage at the edges of its kernels' token slots, 128 to 257 tokens a row: the four- and eight-wavefront row
block (129, 160 and 161, 192 and 193, 256 tokens: whole and partly idle wavefronts, 64-key steps past the row), the
class tokens' attention over up to 256 tokens, the per-head attention below 128 rows and the general path past 256.
Against the oracle at the stages' raw-score tolerance, 5e-5; a prediction too, whose column stage forms the first
block's keys and values."""
import numpy as np
import pytest

import oracle as orc
from conftest import pkg
from test_gpu_stages import TOL, say

abi, hip, M = pkg("abi"), pkg("hip"), pkg("model")
planmod = pkg("plan")
pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("tokens,n", [(128, 130), (129, 1), (129, 9), (129, 130), (160, 128), (161, 40), (192, 255),
                                      (193, 256), (204, 300), (256, 5), (256, 130), (256, 257), (257, 6), (257, 130)])
def test_wide_rows(gpu, model, weights, tokens, n):
    say(f"wide rows tokens={tokens} n={n}")
    m = model
    features = tokens - m.cls
    rng = np.random.default_rng(tokens * 1000 + n)
    tok = rng.standard_normal((n, tokens, m.e)).astype(np.float32)
    err = np.abs(gpu.represent(weights, tok) - orc.represent(m, tok)).max()
    say("  represent worst", err)
    assert err < TOL
    rows = chunk = 64
    layers = [orc.pack((rng.standard_normal(2 * m.d * rows) * 0.5).astype(np.float32), m.d, rows, abi.KV_F32)
              for _ in range(m.icl_layers)]
    scales = np.stack([orc.query_scale(b, rows) for b in m.icl])
    col_kv = (rng.standard_normal((features, 1, len(m.col_a2), 2, m.e, m.inds)) * 0.5).astype(np.float32)
    vm = gpu.load(weights, abi.KV_F32, rows, chunk, layers, scales)
    vm.set_columns(col_kv, features, 1)
    x = rng.standard_normal((n, features)).astype(np.float32)
    fitted = orc.Fitted(rows, features, 10, chunk, abi.KV_F32,
                        planmod.Plan([10], [planmod.Node(None, [], 10, True, list(range(10)))]), col_kv, [scales], [layers])
    err = np.abs(gpu.predict(weights, vm, x, 10) - orc.predict_raw(m, fitted, x)).max()
    say("  predict worst", err)
    assert err < TOL
