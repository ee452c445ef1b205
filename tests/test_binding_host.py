"""The binding's host-side short cuts: half scalars and the pending-error count."""
import ctypes as C
import os
import random
import struct
import subprocess
import sys
import sysconfig
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


def test_fast_calls_round_halves_as_numpy_does():
    """Scalars of half tensors: the nearest half of a double, ties to even, subnormals, overflow, signed zeros, NaN."""
    from cutorch_amd import _fastcall
    halves = np.arange(0x7c00, dtype=np.uint16).view(np.float16).astype(np.float64)
    mid = (halves[:-1] + halves[1:]) / 2
    rng = np.random.default_rng(3)
    values = np.concatenate([halves, mid, np.nextafter(mid, 1e9), np.nextafter(mid, -1e9), [65519.9, 65520.0, 65536.0, 1e300, np.inf, 0.0],
                             np.exp(rng.uniform(-25, 13, 20000))])
    with np.errstate(over="ignore"):
        for sign in (1, -1):
            want = (sign * values).astype(np.float16).view(np.uint16)
            got = np.array([_fastcall.half_bits(float(v)) for v in sign * values], dtype=np.uint16)
            assert np.array_equal(got, want)
        assert np.isnan(np.array(_fastcall.half_bits(float("nan")), dtype=np.uint16).view(np.float16))
    assert _fastcall.half_bits(3) == np.float16(3).view(np.uint16)
    with pytest.raises(TypeError):
        _fastcall.half_bits("3")


def test_every_method_has_a_fast_call():
    """The signatures of all entry points behind the Tensor methods are served, and what ctypes refuses is refused."""
    import ctypes
    from cutorch_amd import _fastcall
    lib = thc.lib()
    names = ("copy fill zero add sub mul div cadd csub cmul cdiv addcmul addcdiv exp abs clamp pow tpow cmaxValue fmod cpow cmax lerp "
             "copyCudaFloat copyCudaHalf ltValue ltValueT ltTensor ltTensorT equal sum prod mean norm cumsum cumprod renorm var std varall "
             "dist max min sumall prodall meanall normall maxall minall").split()
    served = 0
    for kind, (T, _, _, _) in thc._TYPES.items():
        for name in names:
            if not hasattr(lib, T + "_" + name):
                continue
            f = getattr(lib, T + "_" + name)
            if not f.argtypes:
                continue
            signature = "".join(thc._CODES.get(t, "?") for t in [f.restype] + list(f.argtypes[1:]))
            call = _fastcall.bind(ctypes.cast(f, ctypes.c_void_p).value, signature, 0)
            assert call is not None, (T, name, signature)
            served += 1
            with pytest.raises(TypeError):
                call(*[1] * len(f.argtypes))                  # one too many
            if "l" in signature[2:]:
                with pytest.raises(TypeError):
                    call(*[1.5] * (len(f.argtypes) - 1))      # a float for a whole number (the call itself is not reached)
    assert served > 200
    assert _fastcall.bind(0, "vzz", 0) is None


def test_the_binding_works_without_its_native_module():
    """An interpreter that csrc/fastcall.cpp was not built for calls the same entry points through ctypes."""
    code = """if True:
        import sys
        sys.modules["cutorch_amd._fastcall"] = None          # (an import of it raises ImportError)
        import cutorch_amd as thc
        thc._state = thc.lib().THCState_alloc()
        for kind in ("float", "half", "long"):
            t = thc.Tensor(kind)
            assert t.fill(3) is t and t.mul(t, 2) is t and t.cmul(t, t) is t and t.compare_value("lt", t, 1, True) is t
        f = thc.Tensor("float")
        for bad in (lambda: f.var(f, 2), lambda: f.max(thc.Tensor("long"), f, 3)):
            try:
                bad()
                raise SystemExit("no error")
            except thc.THCError as e:
                assert "out of range" in str(e), e
        print("ok", thc._fastcall)
    """
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                          cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert done.stdout.strip() == "ok None", done.stdout + done.stderr


def test_the_native_module_is_named_for_its_interpreter():
    """Its name holds the ABI that it was built for, so no other interpreter loads it."""
    from cutorch_amd import build
    assert build.BINDING.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and len(sysconfig.get_config_var("EXT_SUFFIX")) > len(".so")
    assert thc._fastcall is None or os.path.realpath(thc._fastcall.__file__) == os.path.realpath(build.BINDING)
