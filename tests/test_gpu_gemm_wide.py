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
    assert n >= 72 * E, "the batch is too small to be served by the wide kernel"
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
