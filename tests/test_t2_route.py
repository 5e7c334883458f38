"""Which kernel a T2b128 product takes (t2_route.h): for products whose two kernels were measured more
than 4 % apart, the rule takes the faster one."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fusor-ai_amd", "csrc")

# rows, outputs, groups of 128 inputs, microseconds on the staged tiles and on the waves' own
MEASURED = [
    (65, 12800, 64, 78.1, 59.7), (80, 12800, 64, 76.9, 62.3), (96, 12800, 64, 76.8, 65.9), (65, 13568, 112, 132.9, 103.5),
    (96, 13568, 112, 132.0, 113.0), (72, 14336, 64, 77.1, 67.0), (80, 16384, 64, 77.1, 69.0), (65, 18944, 48, 64.2, 57.6),
    (72, 16384, 48, 58.8, 53.1), (65, 12800, 32, 36.5, 32.9), (72, 13568, 32, 35.8, 34.2), (65, 13000, 32, 35.9, 32.9),
    (65, 12800, 16, 21.0, 18.9), (72, 13568, 16, 20.6, 19.2), (65, 12800, 12, 16.8, 14.8),
    (96, 14336, 32, 35.0, 39.4), (80, 14336, 24, 28.0, 30.8), (96, 12800, 24, 27.3, 29.1), (96, 16384, 16, 20.5, 23.2),
    (80, 18944, 16, 22.5, 24.3), (96, 14336, 112, 132.2, 145.5), (72, 16384, 112, 133.0, 158.6),
    (65, 22016, 64, 84.4, 93.4), (65, 25600, 32, 43.5, 54.5), (65, 14336, 4, 8.3, 9.6), (65, 12800, 2, 7.5, 9.7),
    (64, 25600, 64, 78.0, 82.5), (33, 25600, 16, 20.3, 25.8), (129, 12800, 48, 62.0, 66.6), (129, 8600, 32, 36.1, 38.5),
    (512, 14336, 32, 63.0, 116.2), (257, 5120, 32, 36.4, 41.6), (256, 1024, 32, 12.5, 10.8),
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    where = tmp_path_factory.mktemp("route")
    source, lib = where / "route.cpp", where / "route.so"
    source.write_text('#include "t2_route.h"\n'
                      'extern "C" int staged(long rows, long outputs, long groups)\n'
                      '{ return fg::t2_takes_staged(rows, outputs, groups); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).staged
    fn.argtypes = [ctypes.c_long] * 3
    return fn


@pytest.mark.parametrize("product", MEASURED)
def test_the_faster_kernel(rule, product):
    *sizes, staged, waves = product
    assert rule(*sizes) == (staged < waves)


def test_the_staged_tests_take_the_staged_tiles(rule):
    from test_gpu_t2_staged import STAGED, WAVES
    for rows, outputs, groups in STAGED:  # whole, and the range of four columns less at both ends
        assert rule(rows, outputs, groups) and rule(rows, (outputs + 3) // 4 * 4 - 8, groups), (rows, outputs, groups)
    for sizes in WAVES:
        assert not rule(*sizes), sizes
