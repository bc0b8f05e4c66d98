"""The grouped GEMMs of Q4_K banks on tiles of up to 64 and of up to 16 rows: experts whose rows end just before, at and just after each half of a tile,
among experts without rows, against the f64 product of the dequantized weights.  One super-block to a row (the shortest loop over
K), an odd number of them, one to eight slabs of columns, which are whole (hidden and inter are multiples of 256 here).  The tolerance is
the 3e-5 of the other forms on these units; Q6_K downs likewise."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 0, 2]


@pytest.mark.parametrize("down,tile_rows", [(M.Q4_K, 64), (M.Q4_K, 16), (M.Q8_0, 64), (M.Q6_K, 16), (M.Q6_K, 32), (M.Q6_K, 64)])
@pytest.mark.parametrize("H,I", [(256, 256), (768, 512), (2048, 768)])
def test_every_tile_edge_matches_the_f64_reference(monkeypatch, H, I, down, tile_rows):
    monkeypatch.setenv("MUMMU_GEMM_TILE_ROWS", str(tile_rows))
    E, n = len(COUNTS), sum(COUNTS)
    rng = np.random.Generator(np.random.PCG64(H))
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (31, 32))
    downs = synth.random_bank_fast(down, [I, H, E], 33)
    ids = np.repeat(np.arange(E), COUNTS)[rng.permutation(n)].astype(np.int32)[:, None]
    x = rng.standard_normal((n, H), dtype=np.float32) * np.exp2(rng.integers(-12, 1, (n, 1))).astype(np.float32)
    w = rng.random((n, 1), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, down)
        got, again = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids, w, x)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    orc_down = {M.Q4_K: orc.Q4_K, M.Q6_K: orc.Q6_K, M.Q8_0: orc.Q8_0}[down]
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, orc.Q4_K, orc.Q4_K, orc_down), ids, w, x)
    # (activations in front of a Q8_0 bank: 16 bits and a scale per 64, the bar of experts.rs:1264-1271)
    assert orc.rel_err(got, want, mag).max() <= (2e-3 if down == M.Q8_0 else 3e-5)


# Lists of 16-row tiles in front of down banks of other types, which put together eight elements of an accumulator: every row count of a tile.
@pytest.mark.parametrize("name", ["Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("H,I", [(256, 256), (512, 640)])
def test_tiles_of_16_rows_in_front_of_other_down_banks(name, H, I):
    down = getattr(M, name)
    if down in (M.Q5_K, M.Q6_K) and I % 256:
        pytest.skip("rows of whole super-blocks")
    counts = list(range(17)) * 2
    E, n = len(counts), sum(counts)
    rng = np.random.Generator(np.random.PCG64(H + I))
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (51, 52))
    downs = synth.random_bank_fast(down, [I, H, E], 53)
    ids = np.repeat(np.arange(E), counts)[rng.permutation(n)].astype(np.int32)[:, None]
    x, w = rng.standard_normal((n, H), dtype=np.float32), rng.random((n, 1), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, down)
        got, again = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids, w, x)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, orc.Q4_K, orc.Q4_K, getattr(orc, name)), ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= (3e-5 if down == M.Q6_K else 2e-3)   # (experts.rs:1264-1271)


def test_gates_beyond_the_exponential():
    # gates from -2000 to 2000, e^-x past the largest f32 among them: the wide gates pass, the others leave nothing
    H, I, E, n = 256, 256, 2, 80
    row = np.zeros(144, np.uint8)
    row[:2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)   # d = 1, no offsets
    row[4:8], row[12:16] = 1, 1                                    # every sub-block's scale is 1
    gate = np.tile(row, (I, 1))
    gate[:, 16] = 8                                                # element 0: 8
    up = np.tile(row, (I, 1))
    up[:, 17] = 1                                                  # element 1: 1
    down = np.tile(row, (H, 1))
    down[:, 18] = 1                                                # hidden element 2
    x = np.zeros((n, H), np.float32)
    x[:, 0], x[:, 1] = np.linspace(-250.0, 250.0, n), 1.0
    ids = (np.arange(n, dtype=np.int32) % E)[:, None]
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, *sum(([np.tile(b, (E, 1)), M.Q4_K] for b in (gate, up, down)), []))
        got = m.apply_routing(0, ids, np.ones((n, 1), np.float32), x)
    g = 8.0 * x[:, :1].astype(np.float64)
    want = np.broadcast_to(g / (1.0 + np.exp(np.minimum(-g, 700.0))), (n, H))
    assert np.isfinite(got).all()
    # (a few roundings of f32; below -87 the product with 0 where the quotient is under 2e-36)
    assert (np.abs(got - want) <= 1e-6 * np.abs(want) + 2e-36).all()


@pytest.mark.parametrize("down", [M.Q4_K, M.Q8_0])
def test_last_tiles_of_every_number_of_sixteens(monkeypatch, down):
    """Tiles of up to 64 rows cost what they have in steps of 16: the steps that the counts above leave out, as only tile and behind a full one."""
    monkeypatch.setenv("MUMMU_GEMM_TILE_ROWS", "64")
    counts, H, I = [47, 48, 49, 46, 79, 80, 81, 111, 112, 113, 50, 3], 512, 768
    E, n = len(counts), sum(counts)
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (41, 42))
    downs = synth.random_bank_fast(down, [I, H, E], 43)
    rng = np.random.Generator(np.random.PCG64(3))
    ids = np.repeat(np.arange(E), counts)[rng.permutation(n)].astype(np.int32)[:, None]
    x, w = rng.standard_normal((n, H), dtype=np.float32), rng.random((n, 1), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, down)
        got = m.apply_routing(0, ids, w, x)
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, orc.Q4_K, orc.Q4_K, orc.Q4_K if down == M.Q4_K else orc.Q8_0), ids, w, x)
    # (the bars of the test above)
    assert orc.rel_err(got, want, mag).max() <= (2e-3 if down == M.Q8_0 else 3e-5)
