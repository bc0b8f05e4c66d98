"""The rows that the grouped products read are made by the dispatch launch, beside the sort: in each of their forms (halfs, scaled pairs of
halfs, two bytes and a scale per 64), by the one-launch sort (one to three chunks of 1024 assignments) and the two-launch one, with a last workgroup of one to
three rows, rows that are no multiple of what a workgroup takes at once, and more rows than a pass of the workgroups.  Against the f64 reference.  Halfs at the
2e-3 of experts.rs:1264-1271 in norm and twice that for an element.  Pairs of halfs at the 3e-5 for an element of the other tests of those forms, and 1e-5 in norm:
22 bits, where the upper halfs alone are 2^-12.  Two bytes at 3e-4 in norm: an element is off by up to 2^-16 of its 64's largest, some 2.5 times the others, 4e-5 over
both products; the upper byte alone is 256 times that."""
import numpy as np
import pytest

from mummu_amd import moe as M, synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu

FORMS = {"f16": synth.F16, "q4_k": synth.Q4_K, "q8_0": synth.Q8_0, "q5_0": synth.Q5_0}


BOUNDS = {"f16": (4e-3, 2e-3), "q4_k": (3e-5, 1e-5), "q8_0": (3e-5, 1e-5), "q5_0": (4e-3, 3e-4)}   # of an element, in norm


def check(form, H, n, every=1):
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
    some = np.unique(np.append(np.arange(0, n, every), np.arange(n - 8, n)))
    banks = orc.LayerBanks(H, I, E, gate, up, down, t, t, t)
    want, mag = orc.moe_ref_f64(banks, r.ids.astype(np.int32).reshape(n, k)[some], r.weights.reshape(n, k)[some], x[some])
    got = got[some]
    element, norm = BOUNDS[form]
    assert orc.rel_err(got, want, mag).max() <= element
    assert (np.linalg.norm(got - want, axis=1) <= norm * np.linalg.norm(want, axis=1)).all()


@pytest.mark.parametrize("n", [33, 257, 258, 515, 1027, 1537])   # (1 to 4 chunks of 1024 assignments; 1, 2 or 3 rows in the last workgroup)
@pytest.mark.parametrize("H", [256, 1280])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_batch_matches_the_f64_reference(form, H, n):
    check(form, H, n)


# (2048 workgroups make four rows of pairs or of two bytes each, or 4096 elements as halfs, at a time)
@pytest.mark.parametrize("form,H", [("f16", 1280), ("q4_k", 256), ("q8_0", 256), ("q5_0", 256)])
def test_more_rows_than_a_pass_of_the_workgroups(form, H):
    check(form, H, 8199, every=7)
