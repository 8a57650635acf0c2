"""Idle blocks of hm_buffer_give stand in no other allocation's way: on a device with
little room left, hm_malloc and hm_buffer_take of more than is free succeed once the
idle blocks are gone (they are freed and the allocation tried again), and one that
does not fit even then is refused with its error code. The device is filled to about
9 GiB free, never beyond, and in a process of its own."""
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CODE = """
import ctypes
from henon_map_cpp_amd import _capi as C
L = C.lib()
G = 1 << 30
def free():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    C.check(L.hm_mem_info(ctypes.byref(f), ctypes.byref(t)))
    return f.value
def get(call, n):
    p = ctypes.c_void_p()
    return call(ctypes.byref(p), n), p
def have(call, n):
    rc, p = get(call, n)
    C.check(rc)
    return p
keep = have(L.hm_buffer_take, 8)          # blocks given below stay idle
filler = have(L.hm_malloc, free() - 21 * G)
for call, drop in ((L.hm_malloc, L.hm_free), (L.hm_buffer_take, L.hm_buffer_give)):
    for n in (7 * G, 5 * G):              # two idle blocks, 12 GiB
        idle = have(L.hm_buffer_take, n)
        print("idle", n, flush=True)
        if n == 7 * G:
            first = idle
        else:
            C.check(L.hm_buffer_give(idle))
    C.check(L.hm_buffer_give(first))
    room = free()
    assert 7 * G < room < 11 * G, room
    p = have(call, room + 4 * G)
    print("allocated", flush=True)
    C.check(drop(p))
    rc, p = get(call, 100 * G)
    assert rc == C.HM_ERR_ALLOC, rc
    print("refused", flush=True)
C.check(L.hm_free(filler))
C.check(L.hm_buffer_give(keep))
"""


def test_allocations_take_the_room_of_idle_blocks():
    subprocess.run([sys.executable, "-c", CODE], check=True, timeout=100)
