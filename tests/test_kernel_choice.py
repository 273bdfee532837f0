"""The rules that send batches to the split and panel kernels (overfit_amd/csrc/mid_rule.h), compiled for the host.

Their choice cannot be seen in the outputs, which are the same bits from every kernel. Checked here: the shapes by which
test_gpu_split.py and test_gpu_q8_mid.py mean to run a kernel do run it; batches that measured faster on the kernels used otherwise stay there; the
bounds on which the kernels' addressing rests.
"""
import ctypes
import os
import shutil
import subprocess

import pytest

import test_gpu_q8_mid as q8_mid
import test_gpu_split as split

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "overfit_amd", "csrc")
FORMATS = {"q4k": 12, "q6k": 14}
SOURCE = """
#include "mid_rule.h"
extern "C" int choice(int type, int in, int rows, long tiles, int count) {
    return (int)ovfq::mid_choice(type, in, rows, tiles, count);
}
extern "C" int choice_prepared(int type, int in, int rows, long tiles, int count) {
    return (int)ovfq::mid_choice(type, in, rows, tiles, count, true);
}
extern "C" int over_decode(int type, int in, int rows, long tiles, int count) {
    return ovfq::mid_over_decode(type, in, rows, tiles, count);
}
extern "C" int q8_mid(int in, long out, int rows) { return ovfq::q8_mid_choice(in, out, rows); }
extern "C" int panel_tiles(int type, long o_tiles, long subs) {
    int T;
    ovfq::panel_cost(type, o_tiles, subs, &T);
    return T;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "rule.so"), str(d / "rule.cpp")],
                   check=True)
    lib = ctypes.CDLL(str(d / "rule.so"))
    args = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_int]
    lib.choice.argtypes = lib.choice_prepared.argtypes = lib.over_decode.argtypes = args
    lib.q8_mid.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_int]
    lib.panel_tiles.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long]
    return lib


def choose(rule, fmt, k, rows, ns):
    """The kernel of an automatic call, as use_mid and use_gemv_rows of api.cpp combine the rule with the multi-row decode
    kernel's range (2 .. 8 rows, rows x inputs up to 32768, up to 4 rows or three weights)."""
    tiles = sum((n + 15) // 16 for n in ns)
    decode = rows <= 8 and rows * k <= 32768 and (rows <= 4 or len(ns) >= 3)
    if decode and not rule.over_decode(FORMATS[fmt], k, rows, tiles, len(ns)):
        return "none"
    return ("none", "split", "panel")[rule.choice(FORMATS[fmt], k, rows, tiles, len(ns))]


@pytest.mark.parametrize("fmt", list(FORMATS))
def test_split_and_panel_tests_run_what_they_name(rule, fmt):
    for rows, k, n in split.SPLIT:
        assert choose(rule, fmt, k, rows, [n]) == "split", (fmt, rows, k, n)
    for rows, k, ns in split.PANEL:
        assert choose(rule, fmt, k, rows, ns) == "panel", (fmt, rows, k, ns)
    for rows, k, ns in split.SPLIT_FUSED:
        assert choose(rule, "q4k", k, rows, ns) == "split", (rows, k, ns)
    for rows, k, n in split.PANEL_OF_FIVE:
        assert choose(rule, "q4k", k, rows, [n]) == "panel"
        assert rule.panel_tiles(12, (n + 63) // 64, (rows + 15) // 16) == 5


# (format, inputs, rows, outputs, the kernel that measured faster), by MI355X times of every kernel on the shape: a split
# kernel 10 to 60 % slower than what the shape had before, or a panel kernel 5 to 15 %.
FASTER = [
    ("q4k", 256, 8, [5120], "none"), ("q4k", 1536, 16, [4368], "none"), ("q4k", 2560, 10, [4336], "none"),
    ("q4k", 4352, 3, [912], "none"), ("q4k", 5120, 3, [440], "none"), ("q4k", 5376, 2, [5376, 672, 672], "none"),
    ("q4k", 5376, 6, [5872, 5872], "none"), ("q4k", 256, 39, [16848, 16848], "none"),
    ("q4k", 1280, 59, [9136], "panel"), ("q4k", 256, 61, [11168], "panel"),
    ("q6k", 256, 16, [6000], "none"), ("q6k", 1536, 11, [4448], "none"), ("q6k", 4352, 4, [1584], "none"),
    ("q6k", 256, 143, [5408], "panel"), ("q6k", 256, 506, [1744], "panel"), ("q6k", 1536, 206, [3376], "panel"),
    ("q6k", 1280, 455, [1280, 160, 160], "panel"), ("q6k", 256, 459, [13392], "none"), ("q6k", 512, 506, [22064], "none"),
    ("q6k", 1024, 387, [32752, 32752], "none"),
    # and where the split kernel is the faster one
    ("q4k", 4096, 64, [4096], "split"), ("q4k", 1024, 529, [720], "split"), ("q4k", 2560, 15, [400, 232, 232], "split"),
    ("q6k", 14336, 24, [4096], "split"), ("q6k", 3584, 481, [912], "split"), ("q6k", 1024, 10, [4256], "split"),
]


@pytest.mark.parametrize("fmt,k,rows,ns,kernel", FASTER)
def test_short_and_small_batches_take_the_faster_kernel(rule, fmt, k, rows, ns, kernel):
    assert choose(rule, fmt, k, rows, ns) == kernel


@pytest.mark.parametrize("k,n,rows,kernel", [
    (4096, 14336, 64, "panel"), (4096, 14336, 160, "none"), (4096, 14336, 512, "none"), (8192, 28672, 128, "panel"),
    (8192, 28672, 160, "none"), (8192, 8192, 320, "none"), (2048, 2048, 400, "none"), (2048, 2048, 256, "split"),
    (14336, 4096, 64, "split"), (14336, 4096, 160, "split"), (14336, 4096, 256, "none"), (14336, 1024, 512, "split"),
    (4096, 4096, 160, "split"), (4096, 4096, 200, "none"),
])
def test_prepared_weights_use_their_copy(rule, k, n, rows, kernel):
    """Q6_K weights with the MFMA-ready copy: past 128 rows never the panel kernel, which builds the operands again."""
    assert ("none", "split", "panel")[rule.choice_prepared(14, k, rows, (n + 15) // 16, 1)] == kernel
    for r in range(129, 1100, 37):
        assert rule.choice_prepared(14, k, r, (n + 15) // 16, 1) != 2


@pytest.mark.parametrize("n,rows,height", [(2304, 512, 3), (2304, 464, 3), (3456, 512, 4), (1024, 512, 2), (3072, 416, 3),
                                           (6144, 331, 5), (6144, 512, 4)])
def test_panel_height_is_the_fastest(rule, n, rows, height):
    """Q4_K tile heights that measured fastest, by more than 2 %."""
    assert rule.panel_tiles(12, (n + 63) // 64, (rows + 15) // 16) == height


def test_q8_0(rule):
    for rows, k, n in q8_mid.PROJECT + [(512, 32, 2040)]:
        assert not (rows <= 8 and rows * k <= 32768)  # the decode kernel
        assert rule.q8_mid(k, n, rows), (rows, k, n)
    # measured faster on the 64 x 64 tile kernel by 5 to 20 %, or on these by 4 to 30 %
    for k, n, rows in [(32, 14146, 146), (64, 4736, 473), (96, 21403, 499), (320, 32729, 214), (672, 24718, 179), (1216, 18313, 375)]:
        assert not rule.q8_mid(k, n, rows), (k, n, rows)
    for k, n, rows in [(128, 4096, 256), (320, 2000, 300), (1024, 4096, 512), (4096, 14336, 512), (14336, 4096, 300), (4096, 4096, 12)]:
        assert rule.q8_mid(k, n, rows), (k, n, rows)


@pytest.mark.parametrize("fmt", list(FORMATS))
def test_bounds(rule, fmt):
    """Never for one row, or where a workgroup's rows pass 32-bit offsets (64 rows of 2^26 inputs)."""
    for tiles in (1, 100, 800, 5000):
        assert rule.choice(FORMATS[fmt], 4096, 1, tiles, 1) == 0
        for rows in (2, 5, 17, 64, 65, 513):
            assert rule.choice(FORMATS[fmt], 1 << 26, rows, tiles, 1) == 0
        for subs in range(1, 40):
            t = rule.panel_tiles(FORMATS[fmt], tiles, subs)
            assert 1 <= t <= (5 if fmt == "q4k" else 4) and t <= subs
