"""Where a batch leaves the decode kernels: by what its slots' experts would read, from nine tokens on (banks on the f16 units).
On both sides of the line the block agrees with what the other form gives, the routing to the bit."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,E,k,bank,down,line", [(4096, 1792, 8, 4, "Q4_K", "Q4_K", 9), (2560, 640, 24, 10, "Q4_K", "Q5_1", 19), (2048, 1024, 16, 8, "Q8_0", "Q8_0", 13), (4096, 1792, 8, 4, "Q8_0", "Q8_0", 9),
                                                    (2048, 1024, 16, 8, "Q4_K", "Q4_K", 11), (2048, 1024, 16, 8, "Q4_K", "Q6_K", 12), (2048, 1024, 16, 8, "Q4_K", "Q5_1", 19), (1024, 512, 8, 4, "Q4_K", "Q4_K", 18)])
def test_both_sides_of_the_line(monkeypatch, H, I, E, k, bank, down, line):
    rng = np.random.Generator(np.random.PCG64(H + E))
    bt, dt = getattr(M, bank), getattr(M, down)
    gate, up = (synth.random_bank_fast(bt, [H, I, E], seed) for seed in (71, 72))
    downs = synth.random_bank_fast(dt, [I, H, E], 73)
    router = (rng.standard_normal((E, H)) * 0.02).astype(np.float16)
    x = rng.standard_normal((line, H), dtype=np.float32)

    def run(lines):
        if lines is not None:
            monkeypatch.setenv("MUMMU_GEMM_MIN_TOKENS", str(lines))
        with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=line) as m:
            m.load_layer(0, router, M.F16, gate, bt, up, bt, downs, dt)
            out = [(np.asarray(m.forward(x[:n], k, True)), m.last_routing(n, k)) for n in (line - 1, line)]
            return m.batched_from(0), out

    at, by_rule = run(None)
    assert at == line
    forced = {lines: run(lines)[1] for lines in (1, 1 << 20)}
    for i in range(2):
        same, other = forced[1 if i else 1 << 20][i], forced[1 << 20 if i else 1][i]
        assert np.array_equal(by_rule[i][0].view(np.uint32), same[0].view(np.uint32))
        assert all(np.array_equal(np.asarray(a), np.asarray(b)) for a, b in zip(by_rule[i][1][:2], other[1][:2]))
        # (16 bits and a scale per 16 elements in the decode kernels: 2^-17 of a block's largest element, twice and through three products)
        assert np.linalg.norm(by_rule[i][0] - other[0]) <= 2e-4 * np.linalg.norm(other[0])


@pytest.mark.parametrize("H,I,E,k", [(2048, 1024, 16, 8), (2560, 640, 16, 10)])
def test_few_rows_in_front_of_int8_downs_keep_a_scale_per_16(H, I, E, k):
    """Sixteen hidden rows in every 64 stand out by 2^8 and meet weights of 0: what the others lose to them is what a scale shared with
    them takes.  18 tokens: 2^-17 of a block's largest element, through three products."""
    gate, up = (synth.random_bank_fast(M.Q4_K, [H, I, E], seed) for seed in (77, 78))
    blocks = up.reshape(E, I, H // 256, 144)
    scales = blocks[..., :4].copy().view(np.float16)
    scales[:, np.arange(I) % 64 < 16] *= np.float16(256.0)
    blocks[..., :4] = scales.view(np.uint8)
    downs = synth.random_bank_fast(M.Q8_0, [I, H, E], 79)
    downs.reshape(E, H, I // 64, 2, 34)[..., 0, 2:18] = 0
    rng = np.random.Generator(np.random.PCG64(9))
    x = rng.standard_normal((18, H), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=18) as m:
        m.load_layer(0, (rng.standard_normal((E, H)) * 0.02).astype(np.float16), M.F16, gate, M.Q4_K, up, M.Q4_K, downs, M.Q8_0)
        got = np.asarray(m.forward(x, k, True))
        ids, w = m.last_routing(18, k)[:2]
    want, _ = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, orc.Q4_K, orc.Q4_K, orc.Q8_0), ids, w, x)
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"off by {off:.2e}")
    assert off <= 1e-4


def _top_k_handle(monkeypatch, k_handle, lines=None):
    if lines is None:
        monkeypatch.delenv("MUMMU_GEMM_MIN_TOKENS", raising=False)
    else:
        monkeypatch.setenv("MUMMU_GEMM_MIN_TOKENS", str(lines))
    H, I, E = 2048, 1024, 16
    m = M.SparseMoe(M.SparseMoeConfig(H, I, E, k_handle), max_tokens=18)
    rng = np.random.Generator(np.random.PCG64(5))
    banks = [synth.random_bank_fast(M.Q4_K, dims, seed) for dims, seed in (([H, I, E], 74), ([H, I, E], 75), ([I, H, E], 76))]
    m.load_layer(0, (rng.standard_normal((E, H)) * 0.02).astype(np.float16), M.F16, banks[0], M.Q4_K, banks[1], M.Q4_K, banks[2], M.Q4_K)
    return m, rng.standard_normal((18, H), dtype=np.float32)


@pytest.mark.parametrize("k_handle,k,line", [(8, 1, 18), (8, 2, 18), (8, 8, 11), (1, 8, 11)])
def test_the_line_is_that_of_the_calls_top_k(monkeypatch, k_handle, k, line):
    """What the slots of a call read goes by its own top_k; batched_from() answers for the configured one."""
    outs = {}
    for lines in (None, 1, 1 << 20):
        m, x = _top_k_handle(monkeypatch, k_handle, lines)
        with m:
            if lines is None:
                assert m.batched_from(0) == {8: 11, 1: 18}[k_handle]
            outs[lines] = {n: np.asarray(m.forward(x[:n], k, True)) for n in (10, 11, 17, 18)}
            ids, w = m.last_routing(18, k)[:2]
            outs[lines]["routed"] = {n: np.asarray(m.apply_routing(0, ids[:n], w[:n], x[:n])) for n in (10, 11, 17, 18)}
    for n in (10, 11, 17, 18):
        same = outs[1 if n >= line else 1 << 20]
        assert np.array_equal(outs[None][n].view(np.uint32), same[n].view(np.uint32)), n
        assert np.array_equal(outs[None]["routed"][n].view(np.uint32), same["routed"][n].view(np.uint32)), n
