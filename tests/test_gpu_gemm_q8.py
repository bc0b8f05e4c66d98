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
