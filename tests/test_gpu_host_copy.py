"""Large host arrays on their way to and from the device in pieces: sizes around pieces, slots and the sharing threshold, from
several threads on streams of their own, and where no thread helps."""
import threading
import time

import numpy as np
import pytest

import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L

pytestmark = pytest.mark.gpu
PIECE = L.STAGE


@pytest.mark.parametrize("nbytes", [L.SHARED // 2, L.SHARED + 8, 2 * PIECE, L.HOST_SLOTS * PIECE - 8, L.HOST_SLOTS * PIECE + 8, 3 * L.HOST_SLOTS * PIECE + 24])
def test_arrays_travel_whole(nbytes):
    tt = L.torch()
    rng = np.random.default_rng(nbytes)
    x = rng.standard_normal(nbytes // 8)
    for a in (x, x.astype(np.float32), x.astype(np.float16)):
        a.flags.writeable = False
        t = L.to_device(a)
        assert t.dtype == tt.from_numpy(a.copy()).dtype and np.array_equal(t.cpu().numpy(), a)
    i = rng.integers(0, 8, nbytes // 8)
    d, e = L.upload_indices(i, 8, x[:7].copy())
    assert d.dtype == tt.uint8 and np.array_equal(d.cpu().numpy(), i) and np.array_equal(e.cpu().numpy(), x[:7])
    for at in (0, i.size // 2, i.size - 1):
        for bad in (-1, 8, 1 << 40):
            j = i.copy()
            j[at] = bad
            with pytest.raises(ValueError, match="out of range"):
                L.upload_indices(j, 8)
    buf, (a, b) = L.device_block((i.shape, tt.uint8), (x.shape, tt.float64))
    a.copy_(d)
    b.copy_(L.to_device(x))
    wide, back = L.fetch(buf, (a, np.int64), (b, np.float64))
    assert wide.dtype == np.int64 and np.array_equal(wide, i) and np.array_equal(back, x)


def test_threads_with_streams_of_their_own(monkeypatch):
    """More jobs at a time than the copy threads can all help with; and none of them (the threads take no more work)."""
    tt = L.torch()
    kv = tqa.KVCacheCompressor(64, k_bits=3, v_bits=2, seed=3)
    x = [np.random.default_rng(s).standard_normal((1, 4, 20_000, 64)).astype(np.float32) for s in range(5)]
    want = [kv.decompress(kv.compress(a, -a)) for a in x]

    def run(s, bad):
        with tt.cuda.stream(tt.cuda.Stream()):
            for _ in range(3):
                k, v = kv.decompress(kv.compress(x[s], -x[s]))
                if not (np.array_equal(k, want[s][0]) and np.array_equal(v, want[s][1])):
                    bad.append(s)
    for helped in (True, False):
        if not helped:
            class Gone:
                def submit(self, *args):
                    raise RuntimeError("cannot schedule new futures after shutdown")
            monkeypatch.setattr(L, "_copy_pool", Gone)
        bad = []
        threads = [threading.Thread(target=run, args=(s, bad)) for s in range(len(x))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert bad == []


def test_a_result_behind_other_work_costs_one_processor():
    """While the stream works on something else nobody spins for a result but the thread that asked for it."""
    tt = L.torch()
    m = tt.randn((4096, 4096), device="cuda")
    buf, (t,) = L.device_block(((1 << 21,), tt.float64))
    t.fill_(1.5)
    L.fetch(buf, (t, np.float64))
    for _ in range(400):
        m @ m
    wall, cpu = time.perf_counter(), time.process_time()
    out, = L.fetch(buf, (t, np.float64))
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert (out == 1.5).all()
    assert cpu < 1.5 * wall + 0.05, (cpu, wall)
