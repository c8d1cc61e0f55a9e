"""The launch choices by list sizes (apbf_amd/csrc/launch_rules.h), compiled for
the CPU: the lines lie where their measurements put them."""
import os
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(__file__), "cpp", "launch_rules_check.cpp")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path_factory.mktemp("rules") / "launch_rules_check")
    subprocess.run([gxx, "-std=c++17", "-O1", "-o", exe, SRC], check=True, timeout=120)

    def ask(*requests):
        text = "".join(" ".join(str(int(w) if isinstance(w, bool) else w) for w in r) + "\n" for r in requests)
        r = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True)
        return [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
    return ask


def test_walk_lanes(rules):
    known = [(1, 64), (8191, 64), (8192, 16), (40959, 16), (40960, 8), (131071, 8), (131072, 4), (8000000, 4)]
    assert rules(*[("walk", n, False) for n, _ in known]) == [(lanes,) for _, lanes in known]
    # long rows: never 4 lanes; below 128 K particles the row length changes nothing
    assert rules(*[("walk", n, True) for n, _ in known]) == [(max(lanes, 8),) for _, lanes in known]


def test_the_autotuner_tries_what_the_rule_takes(rules):
    sizes = [1, 8192, 40960, 131072]
    taken = {lanes for (lanes,) in rules(*[("walk", n, long_rows) for n in sizes for long_rows in (False, True)])}
    assert taken <= set(rules(("walks",))[0])


def test_solver_rows_per_flush(rules):
    assert rules(("few", 1), ("few", 131071), ("few", 131072)) == [(1,), (1,), (0,)]


def test_sort_plans(rules):
    """(digit bits, passes, one block) of a sort: short lists in one launch
    whatever their keys (but a single 9-bit pass beyond 1 024 values), 9-bit digits only where they save a pass of a longer
    list with bounded keys, and the passes cover every key."""
    def plan(cap, upper, bits=8, below=True):
        return rules(("sort", cap, upper, bits, below))[0]
    for key_bits in range(1, 32):
        assert plan(1024, 1 << key_bits) == (8, (key_bits + 7) // 8, 1), key_bits
        for cap in (1025, 4096):
            assert plan(cap, 1 << key_bits) == ((8, (key_bits + 7) // 8, 1) if key_bits != 9 else (9, 1, 0)), key_bits
        nine = (key_bits + 8) // 9 < (key_bits + 7) // 8
        want = (9, (key_bits + 8) // 9, 0) if nine else (8, (key_bits + 7) // 8, 0)
        assert plan(4097, 1 << key_bits) == want, key_bits
        # keys of any size are sorted by the 8-bit digits that cover the bound
        assert plan(4097, 1 << key_bits, below=False) == (8, key_bits // 8 + 1, 0)
        for shape in (4, 11):  # other shapes keep their digits and launches
            assert plan(100, 1 << key_bits, shape) == (shape, (key_bits + shape - 1) // shape, 0)
    assert plan(4097, 0xFFFFFFFF, below=False) == (8, 4, 0)
    assert plan(4097, 1) == (8, 0, 0) and plan(4097, 0, below=False) == (8, 0, 0)
