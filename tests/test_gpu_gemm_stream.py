"""Grouped GEMM of Q4_K banks on tiles of up to 8 rows: every row count around a tile's end, one super-block to a row up to sixteen (each number of
waves that a workgroup has its own share of columns for), in front of down banks of its own type, of Q6_K and of the int8 units' types; against
the f64 product of the dequantized weights."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 7, 8, 9, 0, 15, 16, 17, 2]


@pytest.mark.parametrize("H,I,down", [(256, 256, "Q4_K"), (512, 768, "Q4_K"), (768, 512, "Q4_K"), (1024, 1280, "Q4_K"), (1280, 2560, "Q4_K"),
                                      (1792, 2816, "Q4_K"), (2304, 256, "Q4_K"), (256, 256, "Q6_K"), (512, 768, "Q6_K"), (2048, 1024, "Q6_K"), (768, 2816, "Q6_K"), (2560, 640, "Q5_1"), (512, 384, "Q5_1"), (1024, 512, "Q8_0"), (2048, 768, "Q5_K"), (4096, 1536, "Q4_K"),
                                      (1536, 4096, "Q4_K")])
def test_tiles_of_8_rows(monkeypatch, H, I, down):
    monkeypatch.setenv("MUMMU_GEMM_TILE_ROWS", "8")
    monkeypatch.setenv("MUMMU_GEMM_MIN_TOKENS", "1")
    counts = COUNTS
    E, n = len(counts), sum(counts)
    rng = np.random.Generator(np.random.PCG64(H + I))
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (61, 62))
    downs = synth.random_bank_fast(getattr(M, down), [I, H, E], 63)
    ids = np.repeat(np.arange(E), counts)[rng.permutation(n)].astype(np.int32)[:, None]
    x = rng.standard_normal((n, H), dtype=np.float32) * np.exp2(rng.integers(-12, 1, (n, 1))).astype(np.float32)
    w = rng.random((n, 1), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, getattr(M, down))
        got, again = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids, w, x)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, orc.Q4_K, orc.Q4_K, getattr(orc, down)), ids, w, x)
    # (as the other forms on these units, 22 bits an element; in front of an int8 down product 16 bits and a scale per 64: each hidden element is off by
    # m / 65024, m the largest of its 64, at most and 9e-6 m in the mean square; m is up to eight times the mean size, which makes 7e-5 of the terms'
    # root sum of squares, and the worst of 10^5 outputs has five times that; 2.5e-4 to 3e-4 seen, two times allowed)
    assert orc.rel_err(got, want, mag).max() <= (6e-4 if down in ("Q5_1", "Q8_0", "Q5_K") else 1e-5)
    assert np.linalg.norm(got - want) <= (1e-4 if down in ("Q5_1", "Q8_0", "Q5_K") else 1e-6) * np.linalg.norm(want)


@pytest.mark.parametrize("H,I", [(1024, 1024), (2048, 512)])
@pytest.mark.parametrize("field,at", [("d", 0), ("dmin", 2)])
def test_an_infinite_scale_is_what_it_is_on_tiles_of_16_rows(monkeypatch, H, I, field, at):
    """A damaged block of the down bank: both halfs of a row's elements are summed before they meet it."""
    monkeypatch.setenv("MUMMU_GEMM_MIN_TOKENS", "1")
    E, n = 2, 13
    rng = np.random.Generator(np.random.PCG64(H))
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (64, 65))
    downs = synth.random_bank_fast(M.Q4_K, [I, H, E], 66)
    blocks = downs.reshape(E, H, I // 256, 144)
    blocks[:, ::3, I // 512, at:at + 2] = np.full(1, np.inf, np.float16).view(np.uint8)
    ids = (np.arange(n) % 5 == 0).astype(np.int32)[:, None]
    x = rng.standard_normal((n, H), dtype=np.float32)
    outs = []
    for rows in ("8", "16"):
        monkeypatch.setenv("MUMMU_GEMM_TILE_ROWS", rows)
        with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
            m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, M.Q4_K)
            outs.append(np.asarray(m.apply_routing(0, ids, np.ones((n, 1), np.float32), x)))
    assert np.isinf(outs[1][:, ::3]).any()
    assert np.array_equal(np.isnan(outs[0]), np.isnan(outs[1])) and np.array_equal(np.sign(outs[0][np.isinf(outs[1])]), np.sign(outs[1][np.isinf(outs[1])]))
    assert np.isfinite(outs[0][:, 1::3]).all()
