"""The rows that the grouped products read are made by the dispatch launch, beside the sort: in each of their forms (halfs, scaled pairs of
halfs, two bytes and a scale per 64), by the one-launch sort and the two-launch one, with a last workgroup of one to three rows and rows
that are no multiple of what a workgroup takes at once.  Against the f64 reference, at the 2e-3 of experts.rs:1264-1271 in norm and twice that for an element (of halfs; the
other forms are nearer)."""
import numpy as np
import pytest

from mummu_amd import moe as M, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

FORMS = {"f16": synth.F16, "q4_k": synth.Q4_K, "q8_0": synth.Q8_0, "q5_0": synth.Q5_0}


@pytest.mark.parametrize("n", [33, 257, 258, 1537])   # (1 to 4 chunks of 1024 assignments)
@pytest.mark.parametrize("H", [256, 1280])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_batch_matches_the_f64_reference(form, H, n):
    t = FORMS[form]
    I, E, k = 256, 8, 2
    rng = synth.SplitMix64(H + n)
    bank = synth.dense_bank if form == "f16" else synth.synth_bank
    gate, up, down = bank(t, [H, I, E], rng), bank(t, [H, I, E], rng), bank(t, [I, H, E], rng)
    router = rng.normal(E * H, 0.0, 0.05).astype(np.float16).reshape(E, H)
    x = rng.normal(n * H).astype(np.float32).reshape(n, H)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=n) as m:
        m.load_layer(0, router, M.F16, gate, t, up, t, down, t)
        got = m.forward(x, k, False)
        r = m.route(x, k, False)
    banks = orc.LayerBanks(H, I, E, gate, up, down, t, t, t)
    want, mag = orc.moe_ref_f64(banks, r.ids.astype(np.int32), r.weights, x)
    assert orc.rel_err(got, want, mag).max() <= 4e-3
    assert (np.linalg.norm(got - want, axis=1) <= 2e-3 * np.linalg.norm(want, axis=1)).all()
