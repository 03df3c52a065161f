"""The library's build as a list of compiler runs: none of them long, each of them reported when it ends."""
import os
import re
import subprocess
from collections import Counter

import __graft_entry__ as entry

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rocfft_amd", "csrc")


def test_translation_units_are_small_and_all_built():
    """A length costs 2 to 15 s of compiler time (two or three kernels, twelve for powers of two); a unit
    stays below about a minute, and the makefile builds every unit that the list names."""
    text = open(os.path.join(CSRC, "fast_schedules.h")).read()
    units = int(re.search(r"#define FAST_SLICES (\d+)", text).group(1))
    rows = [tuple(map(int, m.group(1).split(",")[:2])) for m in re.finditer(r"^FAST_SCHED\(([\d, ]+)\)", text, re.M)]
    lengths = Counter(unit for unit, _ in rows)
    assert sorted(lengths) == list(range(units))
    assert max(lengths.values()) <= 16, lengths.most_common(3)
    plan = subprocess.run(["make", "-n", "-B", "-C", CSRC, "all"], capture_output=True, text=True, check=True).stdout
    built = [int(u) for u in re.findall(r"-DFAST_SLICE=(\d+)", plan)]
    assert sorted(built) == list(range(units))
    # make -s prints the echo of every finished unit and nothing else
    compiled = re.findall(r" -c \S+ -o \S*/(\S+\.o)$", plan, re.M)
    assert len(compiled) > units and sorted(compiled) == sorted(re.findall(r'echo "built (\S+)"', plan))


def test_number_of_compiler_runs_follows_the_machine(monkeypatch):
    monkeypatch.delenv("MAX_JOBS", raising=False)
    assert 1 <= entry._jobs() <= 16 and entry._jobs() <= len(os.sched_getaffinity(0))
    for value, want in (("3", 3), ("400", 16), ("0", 1)):
        monkeypatch.setenv("MAX_JOBS", value)
        assert entry._jobs() == want
