"""The packed GEMV at the edges of its tiles: every count of rows where another form takes over, K around the 32 of a stage
and short of its slices, column counts that fill no group, and operands that are not 16-byte aligned - against the oracle,
and each row bit for bit as when it comes alone."""
import numpy as np
import pytest

from mummu_amd import moe as M
from oracle import binding as orc
from tests.packed_helpers import pack_words, quantize_block32

pytestmark = pytest.mark.gpu


class At:
    def __init__(self, buf, offset):
        self.buf, self.ptr = buf, buf.ptr + offset


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("k,n", [(31, 32), (32, 288), (33, 256), (444, 544), (1028, 1312), (2050, 96)])
def test_rows_and_edges(k, n, bits):
    g = np.random.default_rng(k + n + bits)
    codes, scales = quantize_block32(g.uniform(-1, 1, (k, n)).astype(np.float32), bits)
    words = pack_words(codes, bits)
    x = g.uniform(-1, 1, (64, k)).astype(np.float32)
    want = orc.q4s_gemv(words, scales, k, n, bits, x)
    peak = np.abs(want).max()
    # the words and x 4 bytes into their buffers
    wd = M.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.uint32), words.ravel()]))
    xd = M.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    sd, yd = M.DeviceBuffer.from_array(scales), M.DeviceBuffer(4 * 64 * n)
    with M.PackedWeight(words, scales, k, n, bits) as w, M.PackedWeight.wrap_device(At(wd, 4), sd, k, n, bits) as odd:
        alone = np.concatenate([w.gemv(x[i]).reshape(1, n) for i in range(64)])
        assert np.abs(alone - want).max() <= 1e-5 * peak
        for m in (2, 4, 5, 8, 9, 16, 17, 32, 33, 64):
            assert np.array_equal(w.gemv(x[:m]).view(np.uint32), alone[:m].view(np.uint32)), m
            odd.gemv_device(At(xd, 4), m, yd)
            assert np.array_equal(yd.download(np.float32, (64, n))[:m].view(np.uint32), alone[:m].view(np.uint32)), m


# Two or three workgroups along K, and from 17 rows on two row groups: whoever adds the partial sums may start when those of its
# rows are there and no earlier (up to 8 rows the last workgroup of a column group, one of all rows; then a launch of its own).
# Every call takes other rows, so that a sum read too early is the one of the call before.
@pytest.mark.parametrize("k,n", [(512, 4096), (640, 2048), (2048, 50304), (444, 544), (4096, 4096), (1024, 17408)])
def test_row_groups_add_their_own_partial_sums(k, n):
    g = np.random.default_rng(k + n)
    words = g.integers(0, 1 << 32, (k, n // 8), dtype=np.uint32)
    scales = g.uniform(0.001, 0.01, (k, n // 32)).astype(np.float32)
    x = g.standard_normal((96, k)).astype(np.float32)
    with M.PackedWeight(words, scales, k, n, 4) as w, M.PackedWeight(words, scales, k, n, 4) as one:
        for m, at in ((32, 0), (17, 32), (8, 60), (21, 64), (32, 64), (9, 11), (17, 0), (4, 90), (16, 40), (8, 33), (20, 32), (21, 0)):
            alone = np.concatenate([one.gemv(x[at + i]).reshape(1, n) for i in range(m)])
            assert np.array_equal(w.gemv(x[at:at + m]).view(np.uint32), alone.view(np.uint32)), (m, at)
        want = orc.q4s_gemv(words, scales, k, n, 4, x[:1])
        assert np.abs(one.gemv(x[0]) - want[0]).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("bits", [4, 8])
def test_infinite_rows_give_infinite_sums(bits):
    # an infinity times a code is an infinity of the code's sign, times 0 it is NaN; the rows beside it stay as they are
    k, n, m = 700, 288, 9
    g = np.random.default_rng(bits)
    codes, scales = quantize_block32(g.uniform(-1, 1, (k, n)).astype(np.float32), bits)
    words = pack_words(codes, bits)
    x = g.uniform(-1, 1, (m, k)).astype(np.float32)
    bad = x.copy()
    bad[1, 3], bad[4, 699], bad[6, 350], bad[8, 40], bad[8, 690] = np.inf, -np.inf, np.nan, 3.0e38, np.inf
    with M.PackedWeight(words, scales, k, n, bits) as w:
        got, plain = w.gemv(bad), w.gemv(x)
    want = orc.q4s_gemv(words, scales, k, n, bits, bad)
    for r in (1, 4, 6, 8):
        assert not np.isfinite(want[r]).any()
        assert np.array_equal(got[r], want[r], equal_nan=True), r
    ok = [r for r in range(m) if r not in (1, 4, 6, 8)]
    assert np.array_equal(got[ok].view(np.uint32), plain[ok].view(np.uint32))


@pytest.mark.parametrize("m", [1, 4, 8, 16, 32])
@pytest.mark.parametrize("bits", [4, 8])
def test_infinities_in_every_form_and_in_the_last_scale(bits, m):
    # (no code 0 beside an infinity: every sum is one; K ends inside a stage, so the infinite scale is that of its padding too)
    k, n = 1037, 288
    g = np.random.default_rng(bits + m)
    codes, scales = quantize_block32(g.uniform(-1, 1, (k, n)).astype(np.float32), bits)
    bad = m // 2
    x = g.uniform(0.5, 1, (m, k)).astype(np.float32)
    x[bad, 5] = np.inf
    codes[5][codes[5] == 0] = 1
    codes[k - 1] = np.where(codes[5] < 0, -1, 1)
    with M.PackedWeight(pack_words(codes, bits), scales, k, n, bits) as w:
        got = w.gemv(x)
    assert np.array_equal(got[bad], np.where(codes[5] < 0, -np.inf, np.inf).astype(np.float32))
    assert np.isfinite(np.delete(got, bad, 0)).all()
    scales[k - 1, 2] = np.inf
    with M.PackedWeight(pack_words(codes, bits), scales, k, n, bits) as w:
        got = w.gemv(x)
    want = np.where(codes[k - 1, 64:96] < 0, -np.inf, np.inf).astype(np.float32)
    assert np.array_equal(got[:, 64:96], np.broadcast_to(want, (m, 32)))
    assert np.isfinite(np.delete(np.delete(got, bad, 0), np.s_[64:96], 1)).all()


@pytest.mark.parametrize("bits", [4, 8])
def test_an_infinite_row_costs_a_second_pass_and_no_more(bits):
    # twice the loop, and the launch: under three times a call without one (a row and column redone term by term: over twenty)
    k, n, m = 5120, 4096, 4
    g = np.random.default_rng(bits)
    wd = M.DeviceBuffer.from_array(g.integers(0, 1 << 32, (k, n * bits // 32), dtype=np.uint32))
    sd = M.DeviceBuffer.from_array(g.uniform(0.001, 0.01, (k, n // 32)).astype(np.float32))
    x = g.standard_normal((m, k)).astype(np.float32)
    bad = x.copy()
    bad[1, 7] = np.inf
    yd = M.DeviceBuffer(4 * m * n)
    with M.SparseMoe(M.SparseMoeConfig(64, 64, 2, 1), max_tokens=1) as clock, M.PackedWeight.wrap_device(wd, sd, k, n, bits) as w:
        def best(rows):
            xd, times = M.DeviceBuffer.from_array(rows), []
            for _ in range(8):
                clock.timer_start()
                for _ in range(20):
                    w.gemv_device(xd, m, yd, clock.stream)
                times.append(clock.timer_stop())
            return min(times)
        plain, infinite = best(x), best(bad)
    assert infinite <= 3.0 * plain, (infinite, plain)
