"""The binding's host-side short cuts: half scalars and the pending-error count."""
import ctypes as C
import random
import struct
import threading
import time

import numpy as np
import pytest

import cutorch_amd as thc


def test_half_scalars_round_as_numpy_rounds_them():
    rng = random.Random(3)
    values = [0.0, -0.0, 1, -3, 0.1, 65504, 65519.999, 65520.0, 1e30, -1e30, float("inf"), float("-inf"), float("nan"),
              2.0 ** -24, 2.0 ** -25, 3 * 2.0 ** -25, 10 ** 6, -(10 ** 6), True, np.float32(0.3), np.float64(-2.5)]
    values += [struct.unpack("<e", struct.pack("<H", rng.randrange(0x7c00)))[0] * (1 + rng.choice((0, 2.0 ** -11, -2.0 ** -12, 2.0 ** -40)))
               for _ in range(5000)]
    for v in values:
        assert thc._half_bits(v) == thc._half_bits_numpy(v), v


def test_errors_are_seen_by_the_thread_that_made_them():
    lib = thc.lib()
    lib.THCAmd_clearLastError()
    before = thc._pending.value

    def fail():
        st = C.c_void_p(lib.THCState_alloc())
        t = lib.THCudaTensor_new(st)                    # empty: asking for dim 3 is an argument error
        lib.THCudaTensor_size(st, t, 3)
        lib.THCudaTensor_size(st, t, 3)                 # counted once per thread, not per message
        lib.THCudaTensor_free(st, t)
        lib.THCState_free(st)

    failed, checked, raised = threading.Event(), threading.Event(), []

    def other():
        fail()
        failed.set()
        checked.wait()
        try:
            thc._check()
        except thc.THCError as e:
            raised.append(str(e))

    worker = threading.Thread(target=other)
    worker.start()
    failed.wait()
    assert thc._pending.value == before + 1
    thc._check()                                        # the other thread's message is not this one's
    checked.set()
    worker.join()
    assert raised and "out of range" in raised[0]
    assert thc._pending.value == before
    fail()
    with pytest.raises(thc.THCError):
        thc._check()
    thc._check()
    assert thc._pending.value == before


def test_a_thread_that_ends_without_reading_its_error_is_not_counted_on():
    lib = thc.lib()
    lib.THCAmd_clearLastError()
    before = thc._pending.value

    def fail():
        st = C.c_void_p(lib.THCState_alloc())
        t = lib.THCudaTensor_new(st)
        lib.THCudaTensor_size(st, t, 3)
        lib.THCudaTensor_free(st, t)
        lib.THCState_free(st)

    workers = [threading.Thread(target=fail) for _ in range(3)]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    deadline = time.time() + 20                         # (join returns a little before the thread's own end)
    while thc._pending.value != before and time.time() < deadline:
        time.sleep(0.01)
    assert thc._pending.value == before
