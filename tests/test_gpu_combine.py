"""The weighted sum of a token's slots behind the grouped products: slot counts around eight (asked for at once) and around a wave's 64 lanes, where
the form with the slots in LDS takes over, hidden sizes that fill part of a workgroup, and a y large enough to be read past the caches' order of
use.  F32 banks against the f64 reference at their 1e-5: one slot left out, twice or with another's weight is off by a hundredth."""
import numpy as np
import pytest

from mummu_amd import moe as M, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,k,n", [(64, 1, 40), (64, 7, 40), (192, 8, 40), (1088, 9, 70), (64, 17, 33), (64, 63, 33), (128, 64, 33), (64, 65, 33),
                                   (2048, 8, 3051), (2048, 8, 3053)])
def test_sum_over_the_slots(H, k, n):
    I, E = 64, k + 3
    rng = synth.SplitMix64(H + 100 * k + n)
    gate, up, down = (synth.dense_bank(synth.F32, shape, rng) for shape in ([H, I, E], [H, I, E], [I, H, E]))
    router = rng.normal(E * H, 0.0, 0.05).astype(np.float16).reshape(E, H)
    x = rng.normal(n * H).astype(np.float32).reshape(n, H)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=n) as m:
        m.load_layer(0, router, M.F16, gate, M.F32, up, M.F32, down, M.F32)
        got = m.forward(x, k, True)
        r = m.route(x, k, True)
    some = np.unique(np.append(np.arange(0, n, 1 + n // 64), n - 1))
    ids, weights = (np.asarray(a).reshape(n, k)[some] for a in (r.ids, r.weights))
    banks = orc.LayerBanks(H, I, E, gate, up, down, synth.F32, synth.F32, synth.F32)
    want, mag = orc.moe_ref_f64(banks, ids.astype(np.int32), weights, x[some])
    assert orc.rel_err(got[some], want, mag).max() <= 1e-5
