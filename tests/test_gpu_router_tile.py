"""Router logits of many tokens, four by four experts to a wave or sixteen by sixteen on the matrix units: bit for bit the oracle's fixed
summation order, at token and expert counts that end inside a tile, on one to four passes over the experts, for every router type."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,n", [(512, 3, 9), (512, 130, 12), (2560, 512, 67), (1024, 129, 33), (512, 512, 600), (512, 501, 1101), (8192, 17, 10), (4608, 512, 600),
                                   # (experts that leave most of a matrix tile's columns empty; the matrix units: more than 128 workgroups of 16 by 64;
                                   # one - 512, 600 and 1101 above - two, five and eight chunks of 512, the last workgroup one token)
                                   (4096, 65, 1041), (512, 16, 2100), (1024, 130, 689), (2560, 512, 257), (4096, 96, 1041)])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_logits_match_the_oracle_bit_for_bit(H, E, n, kind):
    rng = np.random.Generator(np.random.PCG64(H + E + n))
    w = rng.standard_normal((E, H), dtype=np.float32) * np.float32(0.05)
    w[0, :64] = 1e-6   # (subnormal halfs)
    if kind == "f16":
        w, t, ot = w.astype(np.float16), M.F16, orc.F16
    elif kind == "bf16":
        w, t, ot = (w.view(np.uint32) >> 16).astype(np.uint16), M.BF16, orc.BF16
    else:
        t, ot = M.F32, orc.F32
    x = rng.standard_normal((n, H), dtype=np.float32)
    x[1, ::3] *= 1e-30   # (subnormal products and sums)
    bank = synth.random_bank_fast(M.Q8_0, [H, 32, E], 1)
    with M.SparseMoe(M.SparseMoeConfig(H, 32, E, 2), max_tokens=n) as m:
        m.load_layer(0, w, t, bank, M.Q8_0, bank, M.Q8_0, synth.random_bank_fast(M.Q8_0, [32, H, E], 2), M.Q8_0)
        got = np.asarray(m.route(x, 2, True, return_logits=True)[-1]).reshape(n, E)
    want = orc.router_logits(x, w, ot, E).reshape(n, E)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


# Batches of up to 128 experts on either side of the line from which they take these tiles and a launch for the routing: the oracle's routing
# bit for bit, every row served counted once.
@pytest.mark.parametrize("E,n", [(128, 256), (128, 257), (65, 300), (64, 300), (128, 2100),
                                 # (57 to 64 experts from 1025 tokens, 33 to 56 from 2049: on the matrix units with the routing behind)
                                 (64, 2048), (64, 2049), (33, 2065), (32, 2100), (50, 4096)])
def test_routing_and_hits_of_a_batch(E, n):
    H, I, k = 512, 64, 2
    rng = np.random.Generator(np.random.PCG64(E + n))
    router = (rng.standard_normal((E, H), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    x = rng.standard_normal((n, H), dtype=np.float32)
    bank = synth.random_bank_fast(M.Q8_0, [H, I, E], 1)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=n) as m:
        m.load_layer(0, router, M.F16, bank, M.Q8_0, bank, M.Q8_0, synth.random_bank_fast(M.Q8_0, [I, H, E], 2), M.Q8_0)
        m.take_hits(0)
        m.forward(x, k, True)
        ids, w = m.last_routing(n, k)
        hits = np.asarray(m.take_hits(0))
    oids, ow = orc.route_olmoe(orc.router_logits(x, router, orc.F16, E), n, E, k, True)
    assert np.array_equal(ids, oids.astype(np.int32).reshape(n, k))
    assert np.array_equal(w.view(np.uint32), ow.reshape(n, k).view(np.uint32))
    assert np.array_equal(hits, np.bincount(ids.ravel(), minlength=E))


# The routing of 33 to 64 experts on either side of the line to the matrix units, and of few more tokens than a workgroup's: both forms sum a
# logit in the same order, so no bit of the routing may differ.
@pytest.mark.parametrize("E,n", [(64, 1024), (64, 1025), (33, 1030), (32, 1030), (50, 1537), (56, 1025), (57, 1025), (56, 2048), (56, 2049)])
def test_routing_at_the_line_to_the_matrix_units(E, n):
    test_routing_and_hits_of_a_batch(E, n)


# The matrix units with the routing behind, of two to eight chunks of 512 elements (a quarter of 16 rows in LDS at a time), every router type, few slots and
# more than the sixteen that the short ranking takes.
@pytest.mark.parametrize("H,E,n,k", [(1024, 64, 1030, 33), (1536, 57, 1025, 8), (1536, 33, 2049, 8), (2048, 64, 1041, 8), (2560, 50, 1039, 50), (4096, 64, 1040, 17)])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_routing_behind_several_chunks(H, E, n, k, kind):
    rng = np.random.Generator(np.random.PCG64(H + E + n))
    w32 = rng.standard_normal((E, H), dtype=np.float32) * np.float32(0.05)
    if kind == "f16":
        w, t, ot = w32.astype(np.float16), M.F16, orc.F16
    elif kind == "bf16":
        w = (w32.view(np.uint32) >> 16).astype(np.uint16)
        t, ot = M.BF16, orc.BF16
    else:
        w, t, ot = w32, M.F32, orc.F32
    x = rng.standard_normal((n, H), dtype=np.float32)
    bank = synth.random_bank_fast(M.Q8_0, [H, 64, E], 1)
    with M.SparseMoe(M.SparseMoeConfig(H, 64, E, k), max_tokens=n) as m:
        m.load_layer(0, w, t, bank, M.Q8_0, bank, M.Q8_0, synth.random_bank_fast(M.Q8_0, [64, H, E], 2), M.Q8_0)
        m.forward(x, k, True)
        ids, weights = m.last_routing(n, k)
    oids, ow = orc.route_olmoe(orc.router_logits(x, w, ot, E), n, E, k, True)
    assert np.array_equal(ids, oids.astype(np.int32).reshape(n, k))
    assert np.array_equal(weights.view(np.uint32), ow.reshape(n, k).view(np.uint32))


# A token whose row holds an infinity or a NaN is refused, on either side of the line to the matrix units.
@pytest.mark.parametrize("E,n", [(64, 40), (64, 2049), (130, 40), (130, 700)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_rows_that_are_not_finite_are_refused(E, n, value):
    H = 1024
    rng = np.random.Generator(np.random.PCG64(E + n))
    router = (rng.standard_normal((E, H), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    x = rng.standard_normal((n, H), dtype=np.float32)
    x[n - 1, H - 1] = value
    bank = synth.random_bank_fast(M.Q8_0, [H, 32, E], 1)
    with M.SparseMoe(M.SparseMoeConfig(H, 32, E, 2), max_tokens=n) as m:
        m.load_layer(0, router, M.F16, bank, M.Q8_0, bank, M.Q8_0, synth.random_bank_fast(M.Q8_0, [32, H, E], 2), M.Q8_0)
        for call in (m.route, m.forward):
            with pytest.raises(M.MoeError, match=f"token {n - 1} "):
                call(x, 2, True)
