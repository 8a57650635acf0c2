"""Device buffers that wait for their next owner (hm_buffer_take, hm_buffer_give):
reuse by size, refusal of foreign pointers, the device memory back once no block is
taken, and engine objects made, used and dropped in several threads at once, whose
results must equal those of one thread bit for bit."""
import ctypes
import subprocess
import sys
import threading

import numpy as np
import pytest

import henon_map_cpp_amd as hm
from henon_map_cpp_amd import _capi as C

pytestmark = pytest.mark.gpu


def take(nbytes):
    p = ctypes.c_void_p()
    C.check(C.lib().hm_buffer_take(ctypes.byref(p), nbytes))
    return p


def test_reuse_by_size():
    keep = take(8)  # the blocks below stay idle while one is taken
    sizes = [0, 1, 4096, 4097, (1 << 20) + 1, 37 << 20]
    blocks = [take(s) for s in sizes]
    assert len({b.value for b in blocks}) == len(sizes)
    for b in blocks:
        C.check(C.lib().hm_buffer_give(b))
    big = take(37 << 20)
    assert big.value == blocks[-1].value
    other = take(60 << 20)  # larger than any idle block of these
    assert other.value not in {b.value for b in blocks}
    for b in (big, other, keep):
        C.check(C.lib().hm_buffer_give(b))


def test_foreign_and_twice_given_pointers_are_refused():
    keep, b = take(8), take(100)
    C.check(C.lib().hm_buffer_give(b))
    for bad in (b, ctypes.c_void_p(b.value + 8)):
        assert C.lib().hm_buffer_give(bad) == C.HM_ERR_ARG
    C.check(C.lib().hm_buffer_give(None))
    C.check(C.lib().hm_buffer_give(keep))


def test_memory_goes_back_with_the_last_block():
    code = """
import ctypes
from henon_map_cpp_amd import _capi as C
L = C.lib()
def free():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    C.check(L.hm_mem_info(ctypes.byref(f), ctypes.byref(t)))
    return f.value
def take(n):
    p = ctypes.c_void_p()
    C.check(L.hm_buffer_take(ctypes.byref(p), n))
    return p
a = take(8)
before = free()
b = take(3 << 30)
C.check(L.hm_buffer_give(b))
assert before - free() > (3 << 30) - (64 << 20), "kept while a block is taken"
c = take(17 << 30)
C.check(L.hm_buffer_give(c))
assert before - free() < 4 << 30, "a block beyond the limit is not kept"
C.check(L.hm_buffer_give(a))
assert free() >= before - (64 << 20), "freed with the last block"
"""
    subprocess.run([sys.executable, "-c", code], check=True, timeout=100)


def test_threads_make_use_and_drop_engine_objects():
    def work(k):
        rng = np.random.default_rng(k)
        n, turns = 200 + 37 * k, 64
        t = hm.henon_tracker(turns + 1, 0.168, 0.201, "sps", epsilon=16.0)
        out = []
        for _ in range(3):
            p = hm.particles(*rng.uniform(-0.3, 0.3, (4, n)))
            birk, fft = t.tracker.all_tunes(p.particles, turns, 0.2, 10.0, float("nan"), False, [0], [31])
            out += [birk, fft, np.asarray(p.get_x())]
            q = hm.particles(*rng.uniform(-0.3, 0.3, (4, n)))
            out.append(t.tangent_indicators(q, turns, 0.2, 10.0, samples=[turns])["matrix"])
        return out

    want = [work(k) for k in range(4)]
    got = [None] * 4

    def run(k):
        got[k] = work(k)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(want, got):
        assert all(np.array_equal(u, v, equal_nan=True) for u, v in zip(a, b))
