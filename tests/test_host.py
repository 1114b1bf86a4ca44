"""Host-side pieces of the drop-in surface that run without a GPU: the float32 restatement of the query scale and
its elementary functions (checked against the oracle, which is pinned to the reference), and the bundle format."""
import os

import numpy as np
import pytest

import oracle as orc
from conftest import GOLDEN, pkg

fit, B, M = pkg("fit"), pkg("bundle"), pkg("model")


def test_exp_erf_gelu_match_the_oracle_bit_for_bit():
    x = np.linspace(-30.0, 30.0, 20001, dtype=np.float32)
    l = orc.lib()
    assert np.array_equal(fit.exp1(x), np.array([l.orc_exp1(float(v)) for v in x], np.float32))
    assert np.array_equal(fit.erf1(x), np.array([l.orc_erf1(float(v)) for v in x], np.float32))
    g = x.copy()
    l.orc_gelu(orc.fp(g), g.size)
    assert np.array_equal(fit.gelu(x), g)


def test_query_scale_matches_the_oracle(tiny_model):
    full = M.Model.random(M.FULL_CLASSIFIER, seed=2)
    for m in (tiny_model, full):
        for b in list(m.icl) + list(m.col_a1) + list(m.col_a2):
            for n in (1, 120, 10000, 100000):
                want = orc.query_scale(b, n)
                got = fit.query_scale(b, n)
                # logf may differ by one unit in the last place between libraries
                assert np.abs(got - want).max() <= 2e-7 * max(1.0, np.abs(want).max()), (n,)


def test_query_scales_of_unlike_blocks():
    """Each block's own hidden units and head width, summed left to right, whatever the others' are."""
    rng = np.random.default_rng(3)
    F, d, blocks = np.float32, 48, []
    for heads, hid in ((4, 24), (3, 0), (6, 40), (4, 24), (2, 1)):
        t = {"l1b": np.zeros(1, F)}
        if hid:
            t.update(b0w=rng.standard_normal(hid), b0b=rng.standard_normal(hid), b2w=rng.standard_normal(d * hid),
                     b2b=rng.standard_normal(d))
        blocks.append(M.Block(d, heads, t))
    for n in (1, 777, 10000):
        got = fit.query_scales(blocks, n)
        for b, g in zip(blocks, got):
            inv = F(1.0) / np.sqrt(F(b.hd))
            want = np.full(d, inv, F)
            if b.ss_hidden:
                h = fit.gelu(b.t["b0w"] * np.log(F(n)) + b.t["b0b"])
                s = np.add.accumulate(b.t["b2w"].reshape(d, -1) * h[None, :], axis=1, dtype=F)[:, -1]
                want = (s + b.t["b2b"]) * inv
            assert np.array_equal(g, want) and np.array_equal(fit.query_scale(b, n), want)


def test_bundle_round_trip(tmp_path):
    t = {"a": np.arange(7, dtype=np.float32), "b": np.arange(6, dtype=np.int32).reshape(2, 3),
         "c": np.frombuffer(b"hello", dtype=np.uint8), "d": np.ones((2, 2), np.float16)}
    p = os.path.join(tmp_path, "x.tirs")
    raw = B.write(p, t)
    b = B.Bundle.open(p)
    assert b.bytes("c") == b"hello" and b.i32s("b").tolist() == list(range(6))
    assert b.f32s("d").tolist() == [1.0] * 4
    assert all(e.offset % 64 == 0 for e in b.entries)
    assert raw[:8] == b"TIRSBNDL"
    # the reference's own fixtures parse, and re-writing one reproduces its layout exactly
    g = B.Bundle.open(os.path.join(GOLDEN, "tiny-raw.tirs"))
    again = B.write(None, {e.name: g.array(e.name) for e in g.entries})
    assert again == bytes(g.data)


def test_copy_records_is_an_exact_copy():
    """The fit's record copy (sliced over threads from 4 MiB on) returns the same bytes, in a new array, at sizes
    below, at and above the threshold and not a multiple of the slice count."""
    rng = np.random.default_rng(5)
    for n in (0, 1, 4095, 1 << 22, (1 << 22) + 1, 41_156_608 + 7):
        src = rng.integers(0, 256, n, dtype=np.uint8)
        got = fit.copy_records(src)
        assert got.dtype == np.uint8 and got.shape == src.shape
        assert np.array_equal(got, src)
        if n:
            assert not np.shares_memory(got, src)


@pytest.mark.filterwarnings("ignore:Conversion of an array")
def test_plan_takes_any_sequence_of_numbers():
    """Targets as an array, a column, a list, texts, a generator, or values that only float() reads."""
    planmod = pkg("plan")

    class Number:
        def __init__(self, v):
            self.v = v

        def __float__(self):
            return float(self.v)

    values = [0, 3, 1, 12, 7, 5, 3, 11, 2, 4, 6, 8, 9, 10]
    want = planmod.Plan.new(10, values, 13)
    forms = [np.array(values, np.float32), np.array(values), np.array(values, object), np.array(values)[:, None],
             [str(v) for v in values], [Number(v) for v in values]]
    for y in forms:
        assert planmod.Plan.new(10, y, 13) == want
    assert planmod.Plan.new(10, (v for v in values), 13) == want
    assert planmod.Plan.new(0, np.array([0.5, -2.25], np.float32), 5).nodes[0].y == [0.5, -2.25]
