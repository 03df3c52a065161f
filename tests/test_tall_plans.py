"""Plans with tall column passes (rocfft_amd/csrc/tall_kernels.hip) through the emulation, which runs
those passes when a test asks for them: what such a plan accepts is what the plan without them does."""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

import helpers as H
import rocfft_amd.binding as B
from test_callbacks import ROOT, callback_library, check_case


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


# (precision, length): both tile widths, idle lanes, four passes, a prime factor of 17
TALL = [(B.SINGLE, 648), (B.SINGLE, 1020), (B.SINGLE, 1100), (B.SINGLE, 4096), (B.DOUBLE, 750), (B.DOUBLE, 1089),
        (B.DOUBLE, 2401), (B.DOUBLE, 3528)]


@pytest.mark.parametrize("prec,n", TALL, ids=lambda v: str(v))
def test_parameters_of_tall_columns(tall, prec, n):
    """The plan's strides, tiles and workgroups, run by a plain transform on exactly those: full tiles,
    remainders of 1 and W-1 columns, other row pitches, outer dimensions, in place, a scale factor."""
    before = tall.c.fftrt_emu_tall_launches()

    def columns(kind, cols, pitch=None, out_pitch=None, **kw):
        p = pitch or cols
        H.check(tall, H.HostBackend(), kind, [n], cols, prec, in_strides=[p], in_dist=1, out_strides=[out_pitch or p],
                out_dist=1, **kw)

    columns(B.COMPLEX_FORWARD, 16)
    columns(B.COMPLEX_INVERSE, 9, scale=0.25)
    columns(B.COMPLEX_INVERSE, 23, inplace=True)
    columns(B.COMPLEX_FORWARD, 8, pitch=21, out_pitch=32)
    columns(B.COMPLEX_FORWARD, 16, in_offsets=[3, 0], out_offsets=[1, 0])
    H.check(tall, H.HostBackend(), B.COMPLEX_INVERSE, [9, n, 2], 2, prec, inplace=True)
    H.check(tall, H.HostBackend(), B.REAL_FORWARD, [18, n], 2, prec)
    H.check(tall, H.HostBackend(), B.REAL_INVERSE, [18, 2, n], 1, prec)
    # rows as long as the permuted staging of a split wants them, another pitch on the input side
    H.check(tall, H.HostBackend(), B.COMPLEX_FORWARD, [72, n], 1, prec, in_strides=[1, 512], in_dist=512 * n,
            out_strides=[1, 80], out_dist=80 * n)
    assert tall.c.fftrt_emu_tall_launches() - before == 9


FORMS = [(B.COMPLEX_FORWARD, B.SINGLE, [24, 1080], 2), (B.COMPLEX_INVERSE, B.DOUBLE, [12, 960], 1),
         (B.REAL_FORWARD, B.SINGLE, [30, 648], 1), (B.REAL_INVERSE, B.SINGLE, [30, 648], 1),
         (B.COMPLEX_FORWARD, B.SINGLE, [10000, 648], 1)]


@pytest.mark.parametrize("which", ["load", "store", "load+store"])
def test_callbacks_take_a_list_without_tall_columns_where_they_have_to(tall, which):
    """A callback on the side of a tall pass sends the call to the other list (behind rows of 10000
    points to that list's own second list); on the other side the tall pass stays."""
    cblib = callback_library("libcb_host.so")
    for kind, prec, lengths, batch in FORMS:
        assert "tall" in tall.describe(B.NOTINPLACE, kind, prec, lengths, batch)[1], lengths
        before = tall.c.fftrt_emu_tall_launches()
        check_case(tall, H.HostBackend(), cblib, kind, lengths, batch, prec, {}, which)
        at_the_end = kind != B.REAL_INVERSE  # the pass over the columns is the last one, else the first
        stays = which == ("load" if at_the_end else "store") and lengths[0] < 10000
        assert tall.c.fftrt_emu_tall_launches() - before == int(stays), (lengths, which)


def test_buffers_aligned_to_a_scalar_take_a_list_without_tall_columns(tall):
    for kind, prec, lengths, batch in FORMS:
        if kind not in (B.COMPLEX_FORWARD, B.COMPLEX_INVERSE):
            continue
        rt = np.float32 if prec == B.SINGLE else np.float64
        total = 2 * batch * int(np.prod(lengths))
        x = np.random.default_rng(5).uniform(-1, 1, total).astype(rt)
        xs, ys = np.zeros(total + 4, dtype=rt), np.zeros(total + 4, dtype=rt)
        # (numpy's allocations are aligned to 16 bytes)
        shift = 1
        xs[shift:shift + total] = x
        want = np.empty_like(x)
        plan = B.Plan(B.NOTINPLACE, kind, prec, lengths, batch, lib=tall)
        before = tall.c.fftrt_emu_tall_launches()
        plan.execute([x.ctypes.data], [want.ctypes.data])
        assert tall.c.fftrt_emu_tall_launches() == before + 1
        plan.execute([xs.ctypes.data + xs.itemsize], [ys.ctypes.data + ys.itemsize])
        assert tall.c.fftrt_emu_tall_launches() == before + 1
        scale = np.abs(want).max()
        assert np.abs(ys[shift:shift + total] - want).max() <= 8 * np.finfo(rt).eps * scale * 4
        assert ys[0] == 0 and not ys[shift + total:].any()


def test_arrays_that_keep_the_passes_they_had(tall):
    """planar and half-precision arrays, and strides whose offsets inside a tile do not fit 32 bits"""
    for lengths in ([64, 960], [30, 1080], [128, 4096]):
        assert "tall" in tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, lengths, 2)[1]
        assert "tall" not in tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.HALF, lengths, 2)[1]
        for types in ((B.COMPLEX_PLANAR, B.COMPLEX_PLANAR), (B.COMPLEX_PLANAR, B.COMPLEX_INTERLEAVED),
                      (B.COMPLEX_INTERLEAVED, B.COMPLEX_PLANAR)):
            desc = B.PlanDescription(lib=tall).set_data_layout(*types)
            text = tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, lengths, 2, desc)[1]
            # (from planar to interleaved the rows write the interleaved array, which the columns then use)
            assert ("tall" in text) == (types[1] == B.COMPLEX_INTERLEAVED), (lengths, types)

    def columns(pitch):
        desc = B.PlanDescription(lib=tall)
        desc.set_data_layout(B.COMPLEX_INTERLEAVED, B.COMPLEX_INTERLEAVED, None, None, [pitch], 1, [pitch], 1)
        return tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, [960], 64, desc)[1]

    # (960 + 1) rows of the pitch and a tile of 8 columns stay below 2^32 bytes, or do not
    last = ((1 << 29) - 8 - 1) // 961
    assert "tall" in columns(last) and "tall" not in columns(last + 1)


def test_switch_without_tall_columns():
    """the product library's planner (no device needed) with and without ROCFFT_AMD_NO_TALL"""
    code = ("import rocfft_amd.binding as B; l = B.library();"
            "print('tall' in l.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, [4096, 960], 4)[1])")
    env = {k: v for k, v in os.environ.items() if not k.startswith("ROCFFT_AMD_")}
    for extra, want in (({}, "True"), ({"ROCFFT_AMD_NO_TALL": "1"}, "False")):
        out = subprocess.run([sys.executable, "-c", code], env=dict(env, **extra), cwd=ROOT, capture_output=True,
                             text=True, timeout=120)
        assert out.returncode == 0 and out.stdout.split()[-1] == want, (extra, out.stdout, out.stderr[-500:])


def is_tall(lib, prec, lengths, batch=1, pitch=None):
    desc = None
    if pitch:
        desc = B.PlanDescription(lib=lib)
        desc.set_data_layout(B.COMPLEX_INTERLEAVED, B.COMPLEX_INTERLEAVED, None, None, [pitch], 1, [pitch], 1)
    st, text, _ = lib.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, prec, lengths, batch, desc)
    assert st == 0
    return "tall" in text


# (precision, points, columns, taken): both sides of each line of tall_pays
RULE = [
    # in the place of one pass of the same width: always; four lengths from 112 workgroups on full lines
    (B.SINGLE, 704, 8, True), (B.DOUBLE, 1200, 5, True), (B.DOUBLE, 3000, 17, True),
    (B.SINGLE, 896, 880, False), (B.SINGLE, 896, 912, True), (B.SINGLE, 896, 913, False),
    # ... of half the width, rows that start on lines and rows that do not
    (B.SINGLE, 880, 496, False), (B.SINGLE, 880, 528, True), (B.SINGLE, 880, 1521, False), (B.SINGLE, 880, 1530, True),
    (B.SINGLE, 880, 2600, False), (B.SINGLE, 880, 3601, True),
    (B.DOUBLE, 1225, 376, False), (B.DOUBLE, 1225, 392, True), (B.DOUBLE, 1225, 570, False), (B.DOUBLE, 1225, 573, True),
    # in the place of two passes
    (B.SINGLE, 750, 8, True), (B.SINGLE, 960, 512, False), (B.SINGLE, 960, 576, True),
    (B.SINGLE, 2025, 1024, False), (B.SINGLE, 2025, 1088, True), (B.SINGLE, 2048, 512, False), (B.SINGLE, 2048, 576, True),
    (B.DOUBLE, 1080, 32, True), (B.DOUBLE, 1600, 128, False), (B.DOUBLE, 1600, 160, True),
    (B.DOUBLE, 2187, 256, False), (B.DOUBLE, 2187, 288, True),
    # ... with 32-byte runs, among them pitches that are multiples of 512 bytes
    (B.SINGLE, 3840, 640, False), (B.SINGLE, 3840, 704, True), (B.SINGLE, 3840, 315, False), (B.SINGLE, 3840, 321, True),
    (B.DOUBLE, 2816, 160, False), (B.DOUBLE, 2816, 192, True), (B.DOUBLE, 3840, 416, False), (B.DOUBLE, 3840, 448, True),
    (B.DOUBLE, 3168, 640, False), (B.DOUBLE, 3168, 864, True),
    (B.DOUBLE, 2401, 4096, False), (B.DOUBLE, 2430, 4096, True),
]


@pytest.mark.parametrize("prec,n,cols,taken", RULE, ids=lambda v: str(v))
def test_tall_rule(tall, prec, n, cols, taken):
    assert is_tall(tall, prec, [n], cols, cols) == taken


def test_tall_rule_counts_idle_columns(tall):
    """short rows that leave the last tile half empty keep the pass that folds the batch into its tiles"""
    assert is_tall(tall, B.SINGLE, [15, 1080], 240) and not is_tall(tall, B.SINGLE, [9, 1080], 240)
    assert is_tall(tall, B.SINGLE, [15, 880], 240) and not is_tall(tall, B.SINGLE, [13, 880], 240)
    # small problems as a whole: what the tile passes did faster
    for prec, lengths, batch in ((B.SINGLE, [70, 2048], 1), (B.SINGLE, [10, 1080], 3), (B.DOUBLE, [12, 2160], 1),
                                 (B.SINGLE, [64, 2187], 1), (B.DOUBLE, [16, 3993], 1)):
        assert not is_tall(tall, prec, lengths, batch), lengths


def test_tall_rule_where_the_pass_is_refused_later(tall):
    """The rows before a long strided dimension are written in permuted order exactly when that dimension
    is not one tall pass: here the offsets inside its tiles would not fit 32 bits."""
    for lengths, want in (([16384, 16, 2000], "tall"), ([16384, 16, 2048], "staged")):
        st, text, work = tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, lengths)
        assert st == 0 and want in text, text
        tall.c.fftrt_emu_set_tall(0)
        assert work == tall.describe(B.NOTINPLACE, B.COMPLEX_FORWARD, B.SINGLE, lengths)[2]
        tall.c.fftrt_emu_set_tall(1)


def tall_schedules():
    """(double precision?, length, radices, threads per transform, columns, padding shift)"""
    text = open(os.path.join(ROOT, "rocfft_amd", "csrc", "tall_schedules.h")).read()
    for m in re.finditer(r"^TALL_SCHED\(\d+, (float|double), ([\d, ]+)\)", text, re.M):
        v = [int(x) for x in m.group(2).split(",")]
        yield m.group(1) == "double", v[0], [r for r in v[1:5] if r > 1], v[5], v[6], v[7]


def test_schedules_fit_registers_and_lds():
    """At most 12 values of a thread in double precision, one radix-12 pass (two of them took up to 76 bytes
    of scratch a lane); a padding of the LDS tile never costs the second workgroup of a compute unit."""
    gen = subprocess.run([sys.executable, os.path.join(ROOT, "rocfft_amd", "csrc", "gen_tall_schedules.py")],
                         capture_output=True, text=True, check=True).stdout
    assert gen == open(os.path.join(ROOT, "rocfft_amd", "csrc", "tall_schedules.h")).read()
    rows = list(tall_schedules())
    assert len(rows) > 300
    for double, n, radix, tpt, width, shift in rows:
        assert int(np.prod(radix)) == n
        held = max(-(-(n // r) // tpt) * r for r in radix)
        assert held <= (12 if double else 20) and not (double and radix.count(12) > 1), (n, radix)
        size = width * (16 if double else 8)
        lds = (n + ((n - 1) >> shift)) * size
        assert lds <= 160 * 1024
        if n <= 1200 and 2 * n * size <= 160 * 1024:
            assert 2 * lds <= 160 * 1024, (double, n)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["load", "store", "load+store"])
def test_callbacks_beside_tall_columns_on_the_gpu(gpu_lib, which):
    cblib = callback_library("libcb_device.so")
    for kind, prec, lengths, batch in FORMS:
        print("tall callback case", kind, prec, lengths, which, flush=True)
        assert "tall" in gpu_lib.describe(B.NOTINPLACE, kind, prec, lengths, batch)[1], lengths
        check_case(gpu_lib, H.TorchBackend(), cblib, kind, lengths, batch, prec, {}, which)
