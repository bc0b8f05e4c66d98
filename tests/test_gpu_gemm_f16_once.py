"""Grouped GEMM of 16-bit banks: experts whose rows fit one tile read their weights past the caches' order of use, those with several tiles do not.
Both kinds beside one another in a launch, in every place of the tile list."""
import numpy as np
import pytest

from mummu_amd import moe as M

pytestmark = pytest.mark.gpu


def _bf16(a):
    u = a.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("counts", [(40, 1, 0, 3), (1, 150, 31, 33), (5, 0, 90, 64), (140, 130, 1, 2)])
def test_one_tile_and_several(kind, counts):
    H, I, E = 192, 128, len(counts)
    rng = np.random.Generator(np.random.PCG64(sum(counts)))
    ids = np.repeat(np.arange(E, dtype=np.int32), counts)
    rng.shuffle(ids)
    n = ids.size
    x = rng.standard_normal((n, H), dtype=np.float32)
    w = [rng.standard_normal((E, o, i), dtype=np.float32) * np.float32(0.05) for o, i in ((I, H), (I, H), (H, I))]
    if kind == "f16":
        raw = [a.astype(np.float16) for a in w]
        w64 = [a.astype(np.float64) for a in raw]
        t = M.F16
    else:
        raw = [_bf16(a) for a in w]
        w64 = [(a.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for a in raw]
        t = M.BF16
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=n) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, *[v for a in raw for v in (a.reshape(-1).view(np.uint8), t)])
        got = np.asarray(m.apply_routing(0, ids[:, None], np.ones((n, 1), np.float32), x)).reshape(n, H)
    want = np.empty((n, H))
    for r in range(n):
        g, u = w64[0][ids[r]] @ x[r].astype(np.float64), w64[1][ids[r]] @ x[r].astype(np.float64)
        want[r] = w64[2][ids[r]] @ (g / (1.0 + np.exp(-g)) * u)
    # x and the activations between the products are halfs: 2^-12 of an element on average of each, twice
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 1e-3


# Tiles of 96 rows up to 84 rows an expert on average (504 of six; 505 are past the line), experts just below, at and above one and two of them; 128 from there.
@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("counts", [(67, 95, 96, 97, 0, 47), (83, 192, 193, 30, 0, 2), (84, 191, 96, 97, 0, 36), (84, 191, 96, 97, 0, 37), (84, 127, 128, 129, 0, 43)])
def test_tiles_of_96_rows(kind, counts):
    test_one_tile_and_several(kind, counts)
