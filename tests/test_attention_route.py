"""Which path an int8 attention call takes (attention_route.h): for calls whose two paths were
measured more than a tenth apart, the rule takes the faster one."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fusor-ai_amd", "csrc")

# head_dim, images, heads, queries, keys, fast exponentials, microseconds in one launch and unit by unit
MEASURED = [
    (128, 1, 3, 1024, 512, True, 86.0, 72.0), (128, 1, 6, 1024, 1024, True, 145.0, 123.0),
    (116, 1, 3, 426, 533, True, 98.0, 64.5), (120, 1, 3, 92, 424, False, 90.9, 66.0),
    (120, 2, 1, 2309, 395, False, 90.7, 66.6), (120, 1, 15, 80, 1738, True, 254.2, 191.1),
    (120, 1, 11, 134, 1095, False, 201.9, 149.4), (116, 1, 14, 95, 1378, False, 232.5, 182.3),
    (120, 1, 1, 274, 274, False, 70.9, 56.5), (112, 2, 3, 3866, 3866, False, 507.7, 425.3),
    (108, 1, 1, 19, 369, True, 60.5, 47.2), (100, 2, 2, 728, 728, True, 98.4, 82.6),
    (88, 1, 3, 483, 483, False, 84.9, 67.6), (84, 2, 6, 1338, 6407, False, 805.6, 657.1),
    (88, 1, 5, 1415, 1415, True, 174.9, 145.4), (4, 2, 3, 97, 3684, True, 164.2, 139.2),
    (20, 1, 7, 1, 1814, False, 117.7, 103.1), (64, 1, 1, 1024, 1024, True, 75.0, 56.0),
    (64, 1, 12, 1, 4096, True, 249.0, 210.0), (64, 1, 6, 1024, 1024, True, 76.0, 109.0),
    (64, 1, 12, 1024, 4096, True, 256.0, 371.0), (28, 1, 43, 88, 91, False, 25.9, 347.5),
    (92, 2, 10, 1, 2270, False, 218.5, 283.5), (72, 1, 16, 4096, 4096, True, 369.0, 941.0),
    (64, 4, 12, 729, 729, False, 97.0, 506.0),
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    where = tmp_path_factory.mktemp("route")
    source, lib = where / "route.cpp", where / "route.so"
    source.write_text('#include "attention_route.h"\n'
                      'extern "C" int one_launch(size_t i, size_t h, size_t d, size_t q, size_t k, int fast)\n'
                      '{ return fg::attend_in_one_launch(i, h, d, q, k, fast != 0); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).one_launch
    fn.argtypes = [ctypes.c_size_t] * 5 + [ctypes.c_int]
    return fn


@pytest.mark.parametrize("call", MEASURED)
def test_the_faster_path(rule, call):
    head_dim, images, heads, queries, keys, fast, launch, steps = call
    assert rule(images, heads, head_dim, queries, keys, fast) == (launch < steps)


def test_the_one_launch_tests_take_the_one_launch(rule):
    from test_gpu_attention_fused import LONG, RECORDS, SHAPES
    for H, _, D, I, Q, K, fast in SHAPES + RECORDS + LONG:
        assert rule(I, H, D, Q, K, fast), (H, D, I, Q, K, fast)
