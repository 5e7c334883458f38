"""Which kernels a prefill chunk's attention takes (prefill_route.h): for chunks measured more than a
tenth apart over caches past attn_rows_kernel's LDS, and a twentieth over short ones, the rule takes
the faster."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fusor-ai_amd", "csrc")

# head_dim, heads, kv_heads, rows, keys, rows fit, microseconds of the flash kernel and of the others
MEASURED = [
    (128, 7, 1, 32, 6532, False, 1447, 847), (128, 4, 1, 32, 6032, False, 1354, 510),
    (128, 8, 2, 48, 6048, False, 1347, 1141), (128, 4, 4, 48, 6048, False, 1363, 937),
    (64, 4, 4, 32, 7232, False, 868, 620), (64, 4, 4, 48, 5048, False, 675, 564),
    (64, 8, 2, 32, 5032, False, 673, 462), (64, 2, 2, 48, 7048, False, 858, 576),
    (32, 4, 1, 32, 7032, False, 587, 495), (32, 2, 1, 40, 7040, False, 607, 521),
    (128, 7, 1, 96, 6596, False, 1452, 2071), (128, 8, 2, 96, 6096, False, 1353, 2074),
    (128, 14, 2, 48, 6048, False, 1369, 1927), (64, 4, 4, 96, 5096, False, 689, 922),
    (64, 14, 2, 48, 3548, False, 543, 730), (64, 12, 12, 48, 3148, False, 501, 876),
    (32, 8, 8, 48, 3048, False, 384, 510), (32, 12, 2, 48, 7048, False, 605, 857),
    (32, 28, 4, 48, 2048, False, 327, 544), (32, 28, 4, 1, 65, True, 189, 179),
    (32, 8, 2, 2, 66, True, 206, 189), (64, 14, 2, 2, 66, True, 204, 190), (64, 14, 2, 4, 68, True, 213, 201),
    (64, 14, 2, 8, 208, True, 222, 243), (32, 28, 4, 4, 204, True, 196, 216), (128, 7, 1, 8, 208, True, 255, 277),
    (64, 14, 2, 1, 901, True, 252, 352), (64, 14, 2, 64, 264, True, 252, 268),
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    where = tmp_path_factory.mktemp("route")
    source, lib = where / "route.cpp", where / "route.so"
    source.write_text('#include "prefill_route.h"\n'
                      'extern "C" int flash(int d, int heads, int kv, int n, int keys, int fit)\n'
                      '{ return fg::prefill_takes_flash(d, heads, kv, n, keys, fit != 0); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib)).flash


@pytest.mark.parametrize("chunk", MEASURED)
def test_the_faster_kernels(rule, chunk):
    *sizes, flash, others = chunk
    assert rule(*sizes) == (flash < others)


def test_the_flash_tests_take_the_flash_kernel(rule):
    from test_gpu_prefill_flash import CASES, HEADS, LONG
    for case in CASES:
        d, rows, first = case
        assert rule(d, *HEADS[d], rows, rows + first, case not in LONG), case
