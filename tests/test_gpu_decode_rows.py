"""Decode kernels: rows that end inside an iteration (64 short rows side by side, of which a matrix has 32 or 96), one to eight blocks to a row, and the
row iterations of one to eight tokens: each token as on its own, and against the f64 product of the dequantized weights."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["Q8_0", "Q5_1", "Q4_0"])
@pytest.mark.parametrize("H,I", [(32, 96), (96, 32), (64, 160), (160, 64)])
def test_short_rows(monkeypatch, name, H, I):
    _check(monkeypatch, name, name, H, I)


@pytest.mark.parametrize("bank,down", [("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("Q5_K", "Q5_K"), ("Q6_K", "Q6_K"), ("Q4_K", "Q5_1")])
@pytest.mark.parametrize("H,I", [(256, 256), (512, 768), (2304, 512)])
def test_super_blocks(monkeypatch, bank, down, H, I):
    _check(monkeypatch, bank, down, H, I)


def _check(monkeypatch, bank, down, H, I):
    monkeypatch.setenv("MUMMU_GEMM_MIN_TOKENS", "1000000")   # the decode kernels at every size
    E, k, most = 8, 4, 8
    bt, dt = getattr(M, bank), getattr(M, down)
    rng = np.random.Generator(np.random.PCG64(H * 31 + I))
    gate, up = (synth.random_bank_fast(bt, [H, I, E], seed) for seed in (81, 82))
    downs = synth.random_bank_fast(dt, [I, H, E], 83)
    router = (rng.standard_normal((E, H)) * 0.1).astype(np.float16)
    x = rng.standard_normal((most, H), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, k), max_tokens=most) as m:
        m.load_layer(0, router, M.F16, gate, bt, up, bt, downs, dt)
        alone = np.concatenate([np.asarray(m.forward(x[t:t + 1], k, True)) for t in range(most)])
        for n in (2, 3, 5, 8):
            assert np.array_equal(np.asarray(m.forward(x[:n], k, True)).view(np.uint32), alone[:n].view(np.uint32))
        m.forward(x, k, True)
        ids, w = m.last_routing(most, k)[:2]
    want, mag = orc.moe_ref_f64(orc.LayerBanks(H, I, E, gate, up, downs, getattr(orc, bank), getattr(orc, bank), getattr(orc, down)), ids, w, x)
    assert orc.rel_err(alone, want, mag).max() <= 2e-3   # (16-bit activations: experts.rs:1264-1271)
