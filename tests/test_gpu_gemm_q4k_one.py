"""One Q4_K expert on its own on a few rows: row counts around the tiles of 16, one to ten super-blocks along K (with and without a wave
left over), rows of very different size, against the f64 reference.  The tolerance is the 3e-5 of the other Q4_K forms on these units."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


# (hidden, inter, the fewest rows that take this form)
@pytest.mark.parametrize("H,I,first", [(2048, 1024, 22), (4096, 1792, 7), (2560, 768, 23), (256, 4096, 43), (4608, 256, 39)])
def test_few_rows_of_one_expert_match_the_f64_reference(H, I, first):
    E, n = 2, 81
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (41, 42))
    down = synth.random_bank_fast(M.Q4_K, [I, H, E], 43)
    g = np.random.default_rng(H)
    x = g.standard_normal((n, H)).astype(np.float32) * np.exp2(g.integers(-12, 13, (n, 1))).astype(np.float32)
    x[3] = 0.0
    x[5, 256:] = 0.0
    counts = sorted({first, first + 1, 31, 32, 33, 47, 48, 49, 63, 64, 80, 81})
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, down, M.Q4_K)
        got = {rows: m.expert_run(0, 1, x[n - rows:]) for rows in counts if rows >= first}
        again = m.expert_run(0, 1, x[n - first:])
    assert np.array_equal(got[first].view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q4_K), np.ones((n, 1), np.uint32), np.ones((n, 1), np.float32), x)
    for rows, y in got.items():
        err = orc.rel_err(y, want[n - rows:], mag[n - rows:])
        assert np.isfinite(y).all() and err.max() <= 3e-5, (rows, err.max())


# Sub-blocks of 32 that stand out by up to 2^23 and meet no weight: an element is off by at most 2^-39 of its super-block's largest (below 2^25.2
# here), by root mean square at most 2^-14.8, the sums behind the offsets by 2^-25 of values of 2^-10.5 and more, in gate and up alike:
# 2^-14 of the result in norm.  (The per-row kernels with a scale per 16 elements: 1.8e-5 whatever stands out.)
@pytest.mark.parametrize("factor", [2.0 ** 16, 2.0 ** 23])
def test_sub_blocks_standing_out_leave_the_rest_of_their_super_block(factor):
    H, I, E, n = 2048, 1024, 2, 48
    gate, up, down = (np.frombuffer(synth.random_bank_fast(M.Q4_K, ne, s), np.uint8).copy() for s, ne in ((41, [H, I, E]), (42, [H, I, E]), (43, [I, H, E])))
    for bank in (gate, up):
        blocks = bank.reshape(-1, 144)
        blocks[:, 4] &= 0xC0   # scale and offset of sub-block 0 (the upper bits are sub-block 4's)
        blocks[:, 8] &= 0xC0
    x = np.random.default_rng(9).standard_normal((n, H)).astype(np.float32)
    x.reshape(n, H // 256, 8, 32)[:, :, 0] *= np.float32(factor)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, down, M.Q4_K)
        got = m.expert_run(0, 1, x)
    want, _ = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.Q4_K), np.ones((n, 1), np.uint32), np.ones((n, 1), np.float32), x)
    assert np.linalg.norm(got - want) <= 2.0 ** -14 * np.linalg.norm(want)
