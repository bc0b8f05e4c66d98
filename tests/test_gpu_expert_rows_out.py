"""One expert's rows from and to the host: up to 512 KB the down product leaves them in pinned memory itself, beyond they are copied.  The bits of the
device call on both sides of the line, whichever kernel the rows take, and with calls of either kind one after the other."""
import numpy as np
import pytest

from mummu_amd import moe as M
from mummu_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["Q4_K", "Q8_0", "Q5_1", "F16", "F32"])
def test_both_ways_out(name):
    H, I, E = 2048, 256, 2
    t = getattr(M, name)
    if name in ("F16", "F32"):
        rng = np.random.Generator(np.random.PCG64(7))
        banks = [(rng.standard_normal(E * I * H) * 0.05).astype(np.float16 if name == "F16" else np.float32).view(np.uint8) for _ in range(3)]
    else:
        banks = [synth.random_bank_fast(t, dims, seed) for dims, seed in (([H, I, E], 91), ([H, I, E], 92), ([I, H, E], 93))]
    counts = (65, 1, 64, 63, 130, 17, 64)   # 512 KB are 64 rows
    x = np.random.Generator(np.random.PCG64(8)).standard_normal((max(counts), H), dtype=np.float32)
    with M.SparseMoe(M.SparseMoeConfig(H, I, E, 1), max_tokens=max(counts)) as m:
        m.load_layer(0, np.zeros((E, H), np.float16), M.F16, banks[0], t, banks[1], t, banks[2], t)
        for n in counts:
            dx, dy = M.DeviceBuffer.from_array(x[:n]), M.DeviceBuffer(4 * n * H)
            m.expert_run_device(0, 1, dx, n, dy)
            m.check()
            want = dy.download(np.float32, (n, H))
            assert np.array_equal(np.asarray(m.expert_run(0, 1, x[:n])).view(np.uint32), want.view(np.uint32))
