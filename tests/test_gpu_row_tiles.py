"""The fused row block by a row's tokens in tiles of 32: two rows a workgroup (up to 64 tokens; an odd count of rows leaves
its last one alone), one of three or four tiles, the edges of each. Against the oracle at the stages' raw-score
tolerance, 5e-5. Rows that share a workgroup do not see each other: one of infinities leaves its neighbours' bits."""
import numpy as np
import pytest

import oracle as orc
from conftest import pkg
from test_gpu_stages import TOL, say

hip, M = pkg("hip"), pkg("model")
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


@pytest.mark.parametrize("tokens,n", [(5, 129), (31, 512), (32, 129), (33, 130), (63, 513), (64, 131), (65, 128),
                                      (95, 130), (96, 513), (97, 129), (112, 128), (113, 130), (127, 515)])
def test_row_tiles(gpu, model, weights, tokens, n):
    say(f"row tiles tokens={tokens} n={n}")
    tok = np.random.default_rng(tokens * 1000 + n).standard_normal((n, tokens, model.e)).astype(np.float32)
    err = np.abs(gpu.represent(weights, tok) - orc.represent(model, tok)).max()
    say("  represent worst", err)
    assert err < TOL


@pytest.mark.parametrize("tokens,n", [(41, 513), (64, 512), (30, 515)])
def test_rows_of_a_workgroup_are_apart(gpu, model, weights, tokens, n):
    say(f"rows apart tokens={tokens} n={n}")
    tok = np.random.default_rng(tokens).standard_normal((n, tokens, model.e)).astype(np.float32)
    plain = gpu.represent(weights, tok)
    odd = [3, 200, n - 1]
    tok[odd[0], 2, 5], tok[odd[1], 7], tok[odd[2], tokens - 1, 0] = np.inf, np.nan, -np.inf
    got = gpu.represent(weights, tok)
    others = np.setdiff1d(np.arange(n), odd)
    assert np.array_equal(got[others], plain[others]) and np.isfinite(plain).all()
    assert np.isnan(got[odd]).any(axis=1).all()
