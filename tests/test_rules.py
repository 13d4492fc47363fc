"""CPU: the rules that choose between two routes to the same result (ptha_amd/csrc/swh_rules.h),
built for the host, against kernel times measured on an MI355X for both routes: the chosen one
is nowhere more than a quarter slower than the other.

Tables are of measured times; both routes' results are compared in the GPU tests."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = r"""
#include "swh_rules.h"
extern "C" int lists_fit(int nsrc, int ng, long long samples, long long events, long long entries, int w, int maxima)
{
    return swh::superpose_lists_fit(nsrc, ng, samples, events, entries, w != 0, maxima != 0);
}
extern "C" int least_run(long long cells, int simple, int fp64, int due, int odd)
{
    return swh::fused_least_run(cells, simple != 0, fp64 != 0, due != 0, odd != 0);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("rules")
    src, so = str(d / "rules.cpp"), str(d / "librules.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    inc = os.path.join(os.path.dirname(HERE), "ptha_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", inc, src, "-o", so],
                   check=True)
    lib = ctypes.CDLL(so)
    q = ctypes.c_longlong
    lib.lists_fit.argtypes = [ctypes.c_int, ctypes.c_int, q, q, q, ctypes.c_int, ctypes.c_int]
    lib.least_run.argtypes = [q] + 4 * [ctypes.c_int]
    return lib


# sources, gauges, samples, events, sources named in all, weights, maxima; ms of the dense
# product, of the lists
EVENTS = [
    (10, 200, 20, 4096, 12288, 0, 1, 0.0606, 0.1082),
    (20, 64, 100, 1000, 6000, 1, 1, 0.0692, 0.1109),
    (10, 5, 100, 4096, 4096, 1, 1, 0.0475, 0.0746),
    (30, 64, 300, 2048, 22528, 0, 1, 0.1652, 0.5140),
    (50, 64, 100, 4096, 61440, 0, 1, 0.2047, 0.2979),
    (30, 64, 100, 4096, 4096, 1, 1, 0.1390, 0.2635),
    (50, 64, 100, 4096, 8192, 0, 1, 0.2011, 0.2651),
    (10, 64, 100, 16, 48, 1, 1, 0.0453, 0.0160),
    (20, 200, 20, 128, 128, 0, 1, 0.0676, 0.0163),
    (30, 16, 20, 128, 128, 0, 1, 0.0698, 0.0114),
    (200, 64, 100, 128, 7680, 1, 1, 0.7289, 0.0332),
    (512, 64, 100, 16, 5312, 0, 1, 1.8681, 0.0326),
    (639, 64, 100, 16, 496, 0, 1, 2.3374, 0.0242),
    (100, 64, 100, 1000, 30000, 0, 1, 0.3767, 0.0989),
    (1000, 200, 20, 128, 38400, 1, 1, 3.5998, 0.0594),
    (640, 5, 100, 128, 4096, 1, 1, 1.2828, 0.0214),
    (1000, 64, 100, 128, 38400, 1, 1, 3.6637, 0.0996),
    (30, 64, 300, 300, 2700, 1, 0, 0.0701, 0.0823),
    (10, 64, 100, 128, 768, 0, 0, 0.0108, 0.0138),
    (30, 64, 100, 128, 1152, 1, 0, 0.0170, 0.0196),
    (50, 16, 20, 16, 32, 1, 0, 0.0146, 0.0062),
    (30, 16, 20, 16, 144, 1, 0, 0.0095, 0.0061),
    (75, 64, 100, 16, 352, 1, 0, 0.0210, 0.0095),
    (640, 64, 100, 300, 57600, 0, 0, 0.4047, 0.1733),
    (512, 16, 20, 128, 19584, 1, 0, 0.0906, 0.0255),
    (512, 200, 20, 128, 3200, 0, 0, 0.1377, 0.0335),
    (1279, 200, 20, 128, 49024, 1, 0, 0.3326, 0.1525),
]


@pytest.mark.parametrize("row", EVENTS)
def test_events_take_the_faster_route(rules, row):
    *args, dense, lists = row
    chosen = lists if rules.lists_fit(*args) else dense
    assert chosen <= 1.25 * min(dense, lists)


def test_lists_only_where_they_fit(rules):
    assert rules.lists_fit(1279, 64, 100, 100, 1000, 0, 1)
    assert not rules.lists_fit(1280, 64, 100, 100, 1000, 0, 1)


# cells, truely linear without friction, FP64, max_stage after every step; us of a fused launch of
# three steps, of what it replaces (three single steps, or one and a half pairs), and of the
# extra launch that ends a run
RUNS = [
    (48, 1, 1, 0, 9.9, 11.5, 7.2), (48, 1, 1, 1, 10.5, 14.2, 7.4), (48, 0, 0, 1, 12.9, 14.2, 7.1),
    (2000, 1, 1, 0, 10.5, 13.0, 7.6), (2000, 0, 1, 0, 14.4, 16.9, 7.7), (2000, 0, 0, 1, 12.9, 14.5, 8.3),
    (22500, 1, 1, 0, 10.5, 14.2, 8.2), (22500, 1, 1, 1, 11.4, 15.4, 8.3), (22500, 0, 1, 0, 12.3, 14.2, 7.8),
    (22500, 0, 0, 0, 12.3, 18.4, 7.8), (22500, 0, 1, 1, 15.6, 16.9, 8.0), (160000, 1, 1, 0, 12.6, 17.8, 7.8),
    (160000, 1, 0, 0, 10.2, 17.2, 7.8), (160000, 1, 1, 1, 13.5, 25.9, 7.8), (160000, 0, 1, 0, 15.0, 17.5, 7.9),
    (160000, 0, 0, 0, 15.3, 22.0, 7.4), (160000, 0, 1, 1, 21.3, 26.5, 8.2), (350000, 1, 1, 0, 13.8, 22.6, 7.4),
    (350000, 0, 1, 1, 23.4, 36.1, 7.6), (1048576, 1, 1, 0, 24.8, 31.3, 8.5), (1048576, 1, 0, 0, 19.1, 24.4, 8.5),
    (1048576, 0, 1, 0, 40.1, 43.9, 9.2), (1048576, 0, 0, 1, 36.2, 58.3, 8.6), (1650000, 0, 0, 0, 25.8, 30.1, 8.6),
    (4194304, 1, 0, 0, 39.0, 54.1, 8.6), (4194304, 0, 1, 0, 106.8, 137.5, 8.2), (4194304, 0, 0, 1, 76.4, 167.7, 8.1),
]


@pytest.mark.parametrize("row", RUNS)
def test_runs_of_fused_launches_pay(rules, row):
    cells, simple, fp64, due, fused, replaced, flush = row
    least = rules.least_run(cells, simple, fp64, due, 0)
    assert 1 <= least <= 5
    assert least * fused + flush <= 1.08 * least * replaced
    # and those that pay clearly are taken
    assert 5 * fused + flush > 0.75 * 5 * replaced or least < 5
    assert due or least > 1      # (a lone launch in an even stretch leaves a single step)
    assert rules.least_run(cells, simple, fp64, due, 1) <= least
