"""The page table a prefill workgroup stages (csrc/prefill_span.h) holds every
page its keys touch, for all windows the entry point accepts: the header is
compiled alone on the host and compared with the pages counted key by key."""
import os
import random
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INT64_MAX = 2 ** 63 - 1


@pytest.fixture(scope="module")
def span(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("span") / "driver")
    subprocess.run([cxx, "-std=c++20", "-O2", "-I" + os.path.join(ROOT, "sandyrt_amd", "csrc"),
                    os.path.join(ROOT, "tests", "binding", "prefill_span_driver.cpp"), "-o", exe], check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=60).stdout
        return [int(x) for x in out.split()]
    return run


def pages_touched(tk, window, rw, group, lp, base, tq):
    """Most pages a workgroup touches when the first query sits at `base`."""
    most, rows = 0, group * tq
    for r0 in range(0, rows, 32 * rw):
        first = base + r0 // group + 1 - window if window > 0 else 0
        last = min(base + min(rows - 1, r0 + 32 * rw - 1) // group, tk - 1)
        first = max(0, first)
        if first <= last:
            most = max(most, (last >> lp) - (first >> lp) + 1)
    return most


def test_span_covers_every_workgroup(span):
    r = random.Random(7)
    cases = []
    for _ in range(3000):
        tk, lp = r.randrange(1, 3000), r.choice([0, 1, 4, 6, 8])
        window = r.choice([0, 1, 2, r.randrange(1, 300), r.randrange(1, 4000), INT64_MAX - r.randrange(100), INT64_MAX])
        cases.append((tk, window, r.choice([1, 2]), r.choice([1, 2, 3, 6, 8, 40]), lp))
    for c, got in zip(cases, span(cases)):
        tk, window, rw, group, lp = c
        base, tq = r.randrange(0, tk + 40), r.randrange(2, 80)
        assert pages_touched(*c, base, tq) <= got <= (tk >> lp) + 1, (c, base, tq, got)


@pytest.mark.parametrize("window", [INT64_MAX - d for d in (0, 1, 5, 9, 33, 64, 65, 66)])
def test_unbounded_windows_span_the_whole_list(span, window):
    cases = [(tk, window, rw, g, lp) for tk in (40, 600, 9000) for rw in (1, 2) for g in (1, 8) for lp in (4, 6, 8)]
    assert span(cases) == [(c[0] >> c[4]) + 1 for c in cases]
