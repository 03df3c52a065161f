#!/usr/bin/env python3
"""Writes tall_schedules.h: the lengths and radix schedules of the column kernels in
tall_kernels.hip.

Run by hand when the list changes:  python3 gen_tall_schedules.py > tall_schedules.h

Every length with a compile-time-schedule tile kernel (fast_schedules.h) from 641 points to the
last whose tile fits 160 KB of LDS.  Columns per workgroup: 64-byte runs (8 single, 4 double) up to
2400 points, 32-byte runs beyond.  Measured in single precision from 2400 to 3500 points against the
two passes of a split, 32-byte runs are faster with three radix passes (2560 x 50000 851 -> 837 us,
2744 x 3000 53 -> 43 us, 3072 x 8001 189 -> 176 us, 3120 x 800 25 -> 16 us) and mostly slower with four
(3200 x 40000 817 -> 887 us, 3456 x 20000 455 -> 476 us), which are left out.
"""
import os
import re

RADICES = [17, 16, 15, 14, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2]
# additions and multiplications of a butterfly relative to radix 2, per butterfly
COST = {2: 2, 3: 4, 4: 4, 5: 9, 6: 8, 7: 16, 8: 9, 9: 17, 10: 16, 11: 40, 12: 17, 13: 52, 14: 28, 15: 30, 16: 22,
        17: 90}
LDS_BYTES = 160 * 1024
SLICES = 4
NO_PAD = 31
# Lengths left out because the passes they would replace are faster: in single precision 714 and 784 points, whose
# tile pass has 8 columns too (x 4096 columns 18.1 against 20.5 and 20.0 against 23.8 us), 1300 (x 16384 146 against
# 161 us), 2448 (x 3001 53 against 61 us) and 2601 (x 1500 33 against 38 us); in double 2420 and 2500 with rows of
# 32 KB and more (1.04x to 1.3x) and 2904 (x 2000 70 against 79 us)
LEFT_OUT = {False: (714, 784, 1300, 2448, 2601), True: (2420, 2500, 2904)}


def pitch(n, shift):
    """LDS positions of a column: one position of padding every 2**shift elements"""
    return n + ((n - 1) >> shift)


def exchange_cycles(n, sch, t, width, double, shift):
    """LDS cycles of the exchanges between the passes, relative to accesses without bank conflicts:
    64 banks of 4 bytes, 256 bytes a cycle"""
    group, cycles, ideal, cum = (16 if double else 32), 0, 0, 1
    lanes = [(i // width, i % width) for i in range(t * width)]
    for p, r in enumerate(sch):
        m = n // r
        for s in range(-(-m // t)):
            for k in range(r):
                for read in (True, False):
                    if p == (0 if read else len(sch) - 1):
                        continue
                    for g in range(0, len(lanes), group):
                        banks = {}
                        for tt, w in lanes[g:g + group]:
                            b = tt + s * t
                            if b < m:
                                j = b + k * m if read else b // cum * r * cum + b % cum + k * cum
                                bank = ((j + (j >> shift)) * width + w) % group
                                banks[bank] = banks.get(bank, 0) + 1
                        if banks:
                            cycles += max(banks.values())
                            ideal += 1
        cum *= r
    return cycles / ideal


def padding(n, sch, t, width, double):
    """the padding with the fewest LDS cycles among those whose tiles leave room for as many workgroups"""
    size = width * (16 if double else 8)
    room = LDS_BYTES // (2 if 2 * pitch(n, NO_PAD) * size <= LDS_BYTES and n <= 1200 else 1)
    fit = [s for s in (NO_PAD, 5, 4, 3) if pitch(n, s) * size <= room]
    return min(fit, key=lambda s: (round(exchange_cycles(n, sch, t, width, double, s), 2), -s))


def schedules(n, acc=()):
    if n == 1:
        if len(acc) >= 2:
            yield acc
        return
    if len(acc) == 4:
        return
    for r in RADICES:
        if n % r == 0:
            yield from schedules(n // r, acc + (r,))


def best(n, lo, hi, values):
    """fewest passes, then least work of all lanes (idle ones count), then fewest values a thread"""
    res = None
    for sch in schedules(n):
        for t in range(max(lo, 1), hi + 1):
            slots = [-(-(n // r) // t) for r in sch]
            held = max(s * r for s, r in zip(slots, sch))
            if held > values:
                continue
            work = t * sum(s * (COST[r] + 3 * r) for s, r in zip(slots, sch)) / n
            key = (len(sch), round(work, 1), held, sch[0], t, sch)
            if res is None or key < res[0]:
                res = (key, sch, t)
    return res


def pick(n, double):
    """schedule, threads per transform and columns per workgroup, or None"""
    if double:
        width = 4 if n <= 2400 else 2
        tries = [(n // 11, 1024 // width, 11), (n // 12, 1024 // width, 12)]
    else:
        width = 8 if n <= 2400 else 4
        # up to 1200 points two workgroups of 512 threads share a compute unit; beyond, one: as many threads as
        # it can have
        tries = [(64, 128, 18)] if n <= 1200 else [(96, 128, 20)] if n <= 2400 else [(144, 256, 18)] if n <= 3500 else [(200, 256, 17)]
    if pitch(n, 4) * width * (16 if double else 8) > LDS_BYTES:
        return None
    found = None
    for lo, hi, values in tries:
        b = best(n, lo, hi, values)
        if not b or (not double and 2400 < n <= 3500 and len(b[1]) > 3):
            continue
        # Double precision: 11 values of a thread and their twiddles fit 128 registers; 12 take up to 44 bytes
        # of scratch a lane (76 with two passes of radix 12), which pays where it saves an exchange through LDS
        # (1200 points x 2048 columns 28.2 against 26.8 us) and not otherwise (750 x 8000 61.9 against 54.2 us).
        if found and (len(b[1]) >= len(found[1]) or b[1].count(12) > 1):
            continue
        if not found and values == 12 and b[1].count(12) > 1:
            continue
        found = b
    return (found[1], found[2], width) if found else None


def main():
    here = os.path.dirname(os.path.abspath(__file__))
    lengths = set()
    with open(os.path.join(here, "fast_schedules.h")) as f:
        for line in f:
            m = re.match(r"FAST_SCHED\((\d+), (\d+), (\d+)", line)
            if m:
                lengths.add(int(m.group(3)))
    print("// written by gen_tall_schedules.py: slice, type, length, radices, threads per transform, columns, LDS padding")
    i = 0
    for n in sorted(x for x in lengths if 640 < x <= 4096):
        for double in (False, True):
            p = n not in LEFT_OUT[double] and pick(n, double)
            if p:
                sch = list(p[0]) + [1] * (4 - len(p[0]))
                print("TALL_SCHED(%d, %s, %d, %d, %d, %d, %d, %d, %d, %d)"
                      % (i % SLICES, "double" if double else "float", n, *sch, p[1], p[2], padding(n, p[0], p[1], p[2], double)))
                i += 1


if __name__ == "__main__":
    main()
