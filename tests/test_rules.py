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
