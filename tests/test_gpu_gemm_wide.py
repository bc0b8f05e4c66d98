"""The wide grouped GEMM of F16 and BF16 banks: experts whose rows end just before, at and just after each step of 64 and
each tile of 320, over rows and banks that are no multiple of its slabs, against the f64 reference.  Every row is
held to the 2e-3 of experts.rs:1264-1271 in norm, every element to twice that (six million of them, one expert each)."""
import numpy as np
import pytest
import torch

from mummu_amd import moe as M
from oracle import binding as orc

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257, 319, 320, 321, 384, 385, 639, 640, 641, 0, 2]
H, I, E = 1088, 576, 64


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_every_tile_edge_matches_the_f64_reference(dtype):
    g = torch.Generator().manual_seed(7)
    torch_t, t, ot = (torch.float16, M.F16, orc.F16) if dtype == "f16" else (torch.bfloat16, M.BF16, orc.BF16)
    bank = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(torch_t).view(torch.int16).numpy().view(np.uint16)
    gate, up, down = bank(E, I, H), bank(E, I, H), bank(E, H, I)
    counts = EDGES + [1 + e % 3 for e in range(E - len(EDGES))]
    ids = np.repeat(np.arange(E), counts)
    ids = ids[np.random.default_rng(3).permutation(len(ids))].astype(np.int32)[:, None]
    n = len(ids)
    assert n >= 79 * E, "the batch is too small to be served by the wide kernel"
    x = torch.randn(n, H, generator=g).numpy()
    w = torch.rand(n, 1, generator=g).numpy()
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, bank(E, H), t, gate, t, up, t, down, t)
        got = m.apply_routing(0, ids, w, x)
        again = m.apply_routing(0, ids, w, x)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, ot), ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 4e-3
    assert (np.linalg.norm(got - want, axis=1) <= 2e-3 * np.linalg.norm(want, axis=1)).all()


def test_gates_far_beyond_the_exponential_keep_silu_finite():
    # Rows that are a power of two times one pattern: gates from -1000 to 1000, e^-x past the largest f32 among them.
    H, I, E, n = 256, 128, 224, 72 * 224
    row = lambda v: np.float16(v).view(np.uint16)
    gate = np.zeros((E, I, H), np.uint16)
    gate[:, :, 0] = row(np.linspace(-1000, 1000, I))
    up = np.full((E, I, H), row(0), np.uint16)
    up[:, :, 1] = row(1.0)
    down = np.zeros((E, H, I), np.uint16)
    down[:, np.arange(I), np.arange(I)] = row(1.0)
    x = np.zeros((n, H), np.float32)
    x[:, 0], x[:, 1] = np.where(np.arange(n) % 2, 1.0, 0.125), 1.0
    ids = (np.arange(n, dtype=np.int32) % E)[:, None]
    w = np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.uint16), M.F16, gate, M.F16, up, M.F16, down, M.F16)
        got = m.apply_routing(0, ids, w, x)[:, :I]
    g = x[:, :1].astype(np.float64) * gate[0, :, 0].view(np.float16).astype(np.float64)
    want = g / (1.0 + np.exp(np.minimum(-g, 700.0)))
    assert np.isfinite(got).all()
    # (silu carries an f32 rounding or three and is stored as a half: half an ulp, 2^-11; below 2^-14 half of its last bit)
    assert (np.abs(got - want) <= np.abs(want) * 2.0 ** -10.9 + 2.0 ** -24).all()


def test_infinite_gates_come_out_as_in_the_narrow_kernel():
    # x beyond the halfs is an infinity to both kernels: a gate of -inf is NaN (-inf * 0), one of +inf an infinity
    H, I, E, n = 256, 128, 224, 72 * 224
    one, minus = np.float16(1.0).view(np.uint16), np.float16(-1.0).view(np.uint16)
    gate, up, down = (np.full(s, one, np.uint16) for s in ((E, I, H), (E, I, H), (E, H, I)))
    gate[1::2] = minus   # every second expert
    x = np.full((n, H), 0.01, np.float32)
    x[5:7, 0] = 1e6
    ids = (np.arange(n, dtype=np.int32) % E)[:, None]   # rows 5 and 6: experts 5 and 6
    w = np.ones((n, 1), np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.uint16), M.F16, gate, M.F16, up, M.F16, down, M.F16)
        wide, narrow = m.apply_routing(0, ids, w, x), m.apply_routing(0, ids[:64], w[:64], x[:64])
    for got in (wide, narrow):
        assert np.isnan(got[5]).all()
        assert np.array_equal(got[6], np.full(H, np.inf, np.float32))
        assert np.isfinite(np.delete(got, (5, 6), 0)).all()


def few_steps(H, I, dtype, counts):
    """A batch of `counts` rows per expert on banks of a few steps of K, the same bits six times over; bounds as above."""
    E, n = len(counts), int(np.sum(counts))
    ids = np.random.default_rng(5).permutation(np.repeat(np.arange(E), counts)).astype(np.int32)[:, None]
    torch_t, t, ot = (torch.float16, M.F16, orc.F16) if dtype == "f16" else (torch.bfloat16, M.BF16, orc.BF16)
    g = torch.Generator().manual_seed(9)
    bank = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(torch_t).view(torch.int16).numpy().view(np.uint16)
    gate, up, down = bank(E, I, H), bank(E, I, H), bank(E, H, I)
    x, w = torch.randn(n, H, generator=g).numpy(), torch.rand(n, 1, generator=g).numpy()
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, bank(E, H), t, gate, t, up, t, down, t)
        got = m.apply_routing(0, ids, w, x)
        for _ in range(5):
            assert np.array_equal(got.view(np.uint32), m.apply_routing(0, ids, w, x).view(np.uint32))
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, ot), ids, w, x)
    assert orc.rel_err(got, want, mag).max() <= 4e-3
    assert (np.linalg.norm(got - want, axis=1) <= 2e-3 * np.linalg.norm(want, axis=1)).all()


FEW_STEPS = pytest.mark.parametrize("H, I", [(256, 128), (320, 192)], ids=["4 and 2 steps of K", "5 and 3"])


@FEW_STEPS
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_several_items_to_a_workgroup_of_few_steps(H, I, dtype):
    """More items than CUs, each height of a tile behind each other, with as few steps of K as the kernel takes and one more: what an
    item's first stages and the stores before them find in LDS and in the counters."""
    counts = np.random.default_rng(11).permutation(np.resize([1, 64, 65, 128, 130, 192, 200, 256, 257, 320, 321, 500, 640, 641, 900, 3, 0], 256))
    tiles = int(((counts + 319) // 320).sum())
    assert counts.sum() // 256 >= len(counts), "too few rows per expert for workgroups that take items in turn"
    assert tiles > 8 * 32 + 64, "too few items for every XCD's workgroups to take a second one"
    few_steps(H, I, dtype, counts)


@FEW_STEPS
def test_an_item_to_a_workgroup_of_few_steps(H, I):
    """The same heights and steps with fewer rows per expert, where every workgroup has one item."""
    counts = np.random.default_rng(11).permutation(np.resize([1, 64, 65, 128, 130, 192, 200, 256, 257, 320, 321, 0, 0, 0, 3, 2], 480))
    assert 72 * len(counts) <= counts.sum() < 256 * len(counts)
    few_steps(H, I, "f16", counts)


def test_either_side_of_the_line_from_the_narrow_tiles():
    """78 rows an expert and 79, of rows of 512 elements: the same rows off the f64 reference by no more than x and the activations as halfs make, on either kernel."""
    H = I = 512
    E = 112
    g = torch.Generator().manual_seed(4)
    bank = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(torch.float16).view(torch.int16).numpy().view(np.uint16)
    gate, up, down = bank(E, I, H), bank(E, I, H), bank(E, H, I)
    n = 79 * E
    x, ids = torch.randn(n, H, generator=g).numpy(), (np.arange(n, dtype=np.int32) % E)[:, None]
    w = np.ones((n, 1), np.float32)
    some = np.arange(0, 78 * E, 97)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, bank(E, H), M.F16, gate, M.F16, up, M.F16, down, M.F16)
        both = [m.apply_routing(0, ids[:k * E], w[:k * E], x[:k * E])[some] for k in (78, 79)]
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, down, orc.F16), ids[some], w[some], x[some])
    for got in both:
        assert orc.rel_err(got, want, mag).max() <= 4e-3
        assert (np.linalg.norm(got - want, axis=1) <= 2e-3 * np.linalg.norm(want, axis=1)).all()
