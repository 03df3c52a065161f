"""What making a plan costs on the host."""
import time

import numpy as np

import rocfft_amd.binding as B


def fastest(fn, runs=30):
    best = 1e9
    for _ in range(runs):
        t = time.perf_counter()
        fn()
        best = min(best, time.perf_counter() - t)
    return best


def test_tables_take_few_cosines(emu):
    """Making a plan computes its tables (no other plan holds them here): far less time than a cosine
    and a sine in long double for every value of the table would take by themselves."""
    for prec in (B.SINGLE, B.DOUBLE):
        for n in (4096, 3993):
            angles = np.arange(n, dtype=np.longdouble) * (2 * np.pi / n)
            every_value = fastest(lambda: (np.cos(angles), np.sin(angles)))
            made = fastest(lambda: B.Plan(B.NOTINPLACE, B.COMPLEX_FORWARD, prec, [n], 4, lib=emu).destroy())
            assert made < 0.5 * every_value, (prec, n, made, every_value)
