"""The 32-row grouped GEMM of Q8_0 banks on the f16 units: experts whose rows end just before, at and just after a tile, over
rows of one, two, three and five stages of K and down banks that are no multiple of its 256 columns, against the f64
reference; one expert alone likewise.  Rows carry 22 bits and sums 24: 3e-5, as for the Q4_K kernels of that form."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 15, 31, 32, 33, 63, 64, 65, 0, 97]


@pytest.mark.parametrize("H,I", [(128, 128), (256, 384), (640, 256)])
def test_tile_edges_match_the_f64_reference(H, I):
    E = 40
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (1, 2))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 3)
    ids = np.repeat(np.arange(E), EDGES + [1 + e % 3 for e in range(E - len(EDGES))])
    g = np.random.default_rng(H)
    ids = g.permutation(ids).astype(np.int32)[:, None]
    n = len(ids)
    x, w = g.standard_normal((n, H)).astype(np.float32), g.random((n, 1)).astype(np.float32)
    banks = orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got, again = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids, w, x)
        alone = {rows: m.expert_run(0, E - 1, x[:rows]) for rows in (64, 65, 96, 129)}
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(banks, ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 3e-5
    for rows, y in alone.items():
        want, mag = orc.moe_ref_f64(banks, np.full((rows, 1), E - 1, np.uint32), np.ones((rows, 1), np.float32), x[:rows])
        assert orc.rel_err(y, want, mag).max() <= 3e-5


def outlier_case(wide_block, n=130, factor=2.0 ** 20):
    # Rows with one element (or one block of 64) standing out by `factor`; the weights that meet it are 0, so that what comes out is
    # made of the small ones.
    H, I, E = 512, 256, 4
    banks = [np.frombuffer(synth.random_bank_fast(M.Q8_0, ne, s), np.uint8).copy() for s, ne in ((1, [H, I, E]), (2, [H, I, E]), (3, [I, H, E]))]
    x = np.random.default_rng(9).standard_normal((n, H)).astype(np.float32)
    blocks = [b.reshape(-1, H // 32, 34) for b in banks[:2]]
    if wide_block:
        x[:, :64] *= np.float32(factor)
        for b in blocks:
            b[:, :2, 2:] = 0
    else:
        x[:, 7] = np.float32(factor) * np.sign(x[:, 7])
        for b in blocks:
            b[:, 0, 2 + 7] = 0
    return H, I, E, n, banks, x


@pytest.mark.parametrize("factor", [1.0, 2000.0, 2.0 ** 20])
def test_rows_with_one_element_standing_out_keep_their_small_elements(factor):
    H, I, E, n = 512, 256, 4, 130
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (1, 2))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 3)
    x = np.random.default_rng(9).standard_normal((n, H)).astype(np.float32)
    x[:, 7] *= np.float32(factor)
    x[::3, 500] *= np.float32(-factor)
    ids, w = (np.arange(n, dtype=np.int32) % E)[:, None], np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got, alone = m.apply_routing(0, ids, w, x), m.expert_run(0, 1, x)
    banks = orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0)
    want, mag = orc.moe_ref_f64(banks, ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 3e-5
    want, mag = orc.moe_ref_f64(banks, np.ones((n, 1), np.uint32), w, x)
    assert orc.rel_err(alone, want, mag).max() <= 3e-5


@pytest.mark.parametrize("wide_block", [False, True])
def test_the_limit_of_one_scale_per_row(wide_block):
    # An element is off by at most 2^-34 of its row's largest (2^20 times up to 4.5 here), at random: at most 2^-11.8 of an element of
    # 1, by root mean square a quarter of that (rows' largest are half of it, errors are uniform), in gate and up alike, whose product
    # carries both: 2^-12 of the result in norm.  (That is with the row's largest below 2^10; it lies 2^5 higher, so 2^-17 comes out.)
    H, I, E, n, (gate, up, down), x = outlier_case(wide_block)
    ids, w = (np.arange(n, dtype=np.int32) % E)[:, None], np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got, alone = m.apply_routing(0, ids, w, x), m.expert_run(0, 1, x)
    banks = orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0)
    for y, e in ((got, ids), (alone, np.ones((n, 1)))):
        want, _ = orc.moe_ref_f64(banks, e.astype(np.uint32), w, x)
        assert np.linalg.norm(y - want) <= 2.0 ** -12 * np.linalg.norm(want)


# Blocks of 64 that stand out by up to 2^23 and meet no weight cost the rest of their row no more than 16 bits for each 64 elements do
# (4.6e-5): an element is off by at most 2^-39 of its row's largest (below 2^25.2 here), by root mean square 2^-15.8, at most 2^-14.8
# where the largest passes a power of two, in gate and up alike: 2^-14 of the result in norm.  Few rows per expert, and more than 190.
@pytest.mark.parametrize("rows", [32, 200])
@pytest.mark.parametrize("factor", [2.0 ** 16, 2.0 ** 23])
def test_blocks_standing_out_cost_no_more_than_a_scale_per_64(rows, factor):
    H, I, E, n, (gate, up, down), x = outlier_case(True, 4 * rows, factor)
    ids, w = (np.arange(n, dtype=np.int32) % E)[:, None], np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got = m.apply_routing(0, ids, w, x)
    want, _ = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0), ids, w, x)
    assert np.linalg.norm(got - want) <= 2.0 ** -14 * np.linalg.norm(want)


# Which form takes a batch shows in its error: 2.5e-7 for pairs of halfs, 4.5e-5 for 16 bits per 64 elements.
@pytest.mark.parametrize("E,I,rows,pairs", [(8, 128, 33, True), (8, 128, 34, False), (8, 128, 42, False), (8, 128, 45, True), (8, 128, 190, True),
                                            (8, 128, 191, False), (512, 384, 33, True), (512, 384, 47, False), (512, 384, 50, True)])
def test_the_form_by_rows_per_expert(E, I, rows, pairs):
    H, n = 128, rows * E
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (1, 2))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 3)
    x = np.random.default_rng(rows).standard_normal((n, H)).astype(np.float32)
    ids, w = (np.arange(n, dtype=np.int32) % E)[:, None], np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got = m.apply_routing(0, ids, w, x)[:E]
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0), ids[:E], w[:E], x[:E])
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2e-3 and (err <= 3e-6) == pairs, err


# More items (tiles by 128 rows of gate and up, or 256 of down) than workgroups, so that loads run on from one item into the next:
# rows of one, two, three, five and eight stages, a last slab that is half one; and more rows per expert than ragged shapes
# keep in this form.
@pytest.mark.parametrize("H,I,scale", [(128, 384, 1), (768, 128, 1), (640, 384, 1), (1024, 256, 1), (512, 768, 1), (256, 512, 8)])
def test_workgroups_of_several_items_match_the_f64_reference(H, I, scale):
    counts = np.array([0, 1, 16, 31, 32, 33, 64, 65, 0, 2] * (8 if scale == 1 else 2)) * scale
    E = len(counts)
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (11, 12))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 13)
    g = np.random.default_rng(H + I)
    ids = g.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    n = len(ids)
    x, w = g.standard_normal((n, H)).astype(np.float32) * np.exp2(g.integers(-12, 1, (n, 1))).astype(np.float32), g.random((n, 1)).astype(np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got, again = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids, w, x)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0), ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 3e-5


# Tiles of up to 16 rows (both halfs of a row in one product) beside fuller ones, a workgroup going from one kind to the other.
@pytest.mark.parametrize("H,I", [(128, 256), (640, 384), (1024, 256)])
def test_tiles_of_up_to_16_rows_match_the_f64_reference(H, I):
    counts = np.array([16, 17, 15, 32, 1, 24, 48, 49] * 32)
    E = len(counts)
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (21, 22))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 23)
    g = np.random.default_rng(H)
    ids = g.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    n = len(ids)
    x, w = g.standard_normal((n, H)).astype(np.float32), np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got = m.apply_routing(0, ids, w, x)
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0), ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 3e-5
    assert np.linalg.norm(got - want) <= 3e-6 * np.linalg.norm(want)


# The same for rows whose pieces begin at multiples of 16 bytes, which take pairs of halfs to 40 rows an expert, and from where a tile of 64 is too small.
@pytest.mark.parametrize("H,rows,pairs", [(256, 34, True), (256, 40, True), (256, 41, False), (256, 45, True), (2304, 33, True), (2304, 34, False)])
def test_the_form_by_rows_per_expert_and_their_length(H, rows, pairs):
    E, I, n = 8, 256, 8 * rows
    gate, up = (synth.random_bank_fast(M.Q8_0, [H, I, E], seed) for seed in (1, 2))
    down = synth.random_bank_fast(M.Q8_0, [I, H, E], 3)
    x = np.random.default_rng(rows).standard_normal((n, H)).astype(np.float32)
    ids, w = (np.arange(n, dtype=np.int32) % E)[:, None], np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q8_0, up, M.Q8_0, down, M.Q8_0)
        got = m.apply_routing(0, ids, w, x)[:E]
    want, _ = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q8_0), ids[:E], w[:E], x[:E])
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2e-3 and (err <= 3e-6) == pairs, err
