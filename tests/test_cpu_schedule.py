"""The partial rows of hub tasks at precisions above 10: their bytes stay within the two
register buffers (or 1 GiB) whatever the degrees, lists are cut at 256 arcs where that fits,
and every cut list is covered.  Host code only, compiled from the engine's header."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    src, lib = str(d / "rule.cpp"), str(d / "rule.so")
    with open(src, "w") as fh:
        fh.write('#include "%s"\n' % os.path.join(ROOT, "sparkx_amd", "csrc", "hb_schedule.h") +
                 'extern "C" uint64_t tasks(const uint32_t *o, uint32_t n, uint64_t l) { return hb::wide_tasks(o, n, l); }\n'
                 'extern "C" uint64_t task_len(const uint32_t *o, uint32_t n, int p) { return hb::wide_task_len(o, n, p); }\n')
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", src, "-o", lib],
                   check=True)
    so = C.CDLL(lib)
    u32p = np.ctypeslib.ndpointer(np.uint32, flags="C")
    so.tasks.argtypes, so.tasks.restype = [u32p, C.c_uint32, C.c_uint64], C.c_uint64
    so.task_len.argtypes, so.task_len.restype = [u32p, C.c_uint32, C.c_int], C.c_uint64
    return so


def _offsets(degrees):
    off = np.zeros(len(degrees) + 1, np.uint64)
    np.cumsum(degrees, out=off[1:])
    assert off[-1] < 2**32
    return off.astype(np.uint32)


@pytest.mark.parametrize("p", [11, 12, 14, 16])
@pytest.mark.parametrize("kind", ["dense", "denser", "power", "star", "small", "sparse", "empty"])
def test_partial_rows_are_bounded(rule, p, kind):
    deg = {"dense": np.full(65536, 10_000), "denser": np.full(65536, 65_535),  # 0.66 and 4.29 G arcs
           "power": np.maximum(1, 2_000_000 // np.arange(1, 1_000_001)), "star": np.r_[4_000_000, np.ones(4_000_000)],
           "small": np.r_[np.full(100, 900), np.full(5000, 3)], "sparse": np.full(100_000, 256),
           "empty": np.zeros(3)}[kind].astype(np.int64)
    off, n = _offsets(deg), len(deg)
    ln = rule.task_len(off, n, p)
    tasks = rule.tasks(off, n, ln)
    assert tasks == sum(-(-d // ln) for d in deg[deg > ln].tolist())
    room = max(n << (p + 1), 1 << 30)
    assert tasks << p <= room
    # the shortest of 256, 512, ... that fits
    assert ln == 256 or (ln % 512 == 0 and rule.tasks(off, n, ln // 2) << p > room)
    if kind in ("small", "sparse", "empty", "star"):
        assert ln == 256
