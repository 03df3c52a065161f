"""Plans with tall column passes (rocfft_amd/csrc/tall_kernels.hip) through the emulation, which runs
those passes when a test asks for them: what such a plan accepts is what the plan without them does."""
import ctypes

import numpy as np
import pytest

import rocfft_amd.binding as B


@pytest.fixture
def tall(emu):
    """the emulation with tall column passes; tall.tall(False) takes them out of the plans made next"""
    c = emu.c
    c.fftrt_emu_set_tall.argtypes = [ctypes.c_int]
    c.fftrt_emu_set_capturing.argtypes = [ctypes.c_int]
    c.fftrt_emu_tall_launches.restype = ctypes.c_long
    c.fftrt_emu_malloc_calls.restype = ctypes.c_long
    c.fftrt_emu_set_tall(1)
    yield emu
    c.fftrt_emu_set_tall(0)
    c.fftrt_emu_set_capturing(0)


def plans(lib, *args):
    """the same plan with and without tall column passes"""
    out = []
    for on in (1, 0):
        lib.c.fftrt_emu_set_tall(on)
        out.append(B.Plan(*args, lib=lib))
        assert ("tall" in lib.describe(*args)[1]) == bool(on)
    lib.c.fftrt_emu_set_tall(1)
    return out


def test_work_areas_accepted_do_not_depend_on_the_kernels(tall):
    """an area that is given has to hold what the plan without these kernels needs, and without one
    the stream must not be capturing, though the tall list itself needs none"""
    c = tall.c
    both = plans(tall, B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, [64, 960], 2)
    size = both[0].work_buffer_size
    assert size == both[1].work_buffer_size > 0
    x = np.random.default_rng(1).uniform(-1, 1, 64 * 960 * 2 * 2).astype(np.float32)
    y = np.empty_like(x)
    area = np.empty(size + 64, dtype=np.uint8)
    base = area.ctypes.data + -area.ctypes.data % 16
    result = []
    for plan in both:
        before = c.fftrt_emu_tall_launches()

        def status(given, capturing=0, static=False):
            info = B.ExecutionInfo(tall)
            if given is not None:
                info.set_work_buffer(base, given)
            c.fftrt_emu_set_capturing(capturing)
            run = plan.execute_static_status if static else plan.execute_status
            return run([x.ctypes.data], [y.ctypes.data], info)

        got = [status(size), status(size - 16), status(size, 1), status(None, 1), status(None, 1, True), status(None)]
        assert got == [0, B.STATUS_INVALID_WORK_BUFFER, 0, B.STATUS_INVALID_WORK_BUFFER, 0, 0], got
        result.append(c.fftrt_emu_tall_launches() - before)
    assert result == [4, 0]
    # nothing is allocated for a list that needs nothing
    calls = c.fftrt_emu_malloc_calls()
    both[0].execute([x.ctypes.data], [y.ctypes.data])
    assert c.fftrt_emu_malloc_calls() == calls
    both[1].execute([x.ctypes.data], [y.ctypes.data])
    assert c.fftrt_emu_malloc_calls() == calls + 1


def test_static_area_too_small_for_the_plan_without_tall_columns(tall):
    x = np.zeros(2 * 4096 * 2160, dtype=np.float32)
    y = np.full_like(x, 7)
    for plan in plans(tall, B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, [4096, 2160], 1):
        assert plan.work_buffer_size > B.STATIC_WORK_BYTES
        assert plan.execute_static_status([x.ctypes.data], [y.ctypes.data]) == B.STATUS_INVALID_WORK_BUFFER
        assert (y == 7).all()
