"""T2b128 products on the staged tiles (t2_lds_kernel: more than 32 rows, 200 or more workgroups of
64 x 128), where their tiles, quads and three stage buffers end: 1 to 5 groups, row and column
remainders, column ranges, bias, adding to the output, the fused scaling; and the wave tiles that
large tables of few rows, or of few past 64 and many groups, keep. Every output is the oracle's bits."""
import numpy as np
import pytest

from gpu_data import activations, synthetic_table
from oracle import oracle as O
from test_gpu_product import first_mismatch, gpu_product, oracle_product, same_bits, table

pytestmark = pytest.mark.gpu


# outputs are drawn so that ceil(rows / 64) * ceil(outputs / 128) >= 200 for the column range too
STAGED = [(33, 25732, 1), (64, 25600, 2), (65, 12932, 3), (127, 12801, 4), (449, 3458, 5), (200, 6500, 3)]
WAVES = [(20, 131076, 1), (65, 12932, 9)]


@pytest.mark.parametrize("rows,outputs,groups", STAGED + WAVES)
def test_staged_t2_tiles(gpu, rows, outputs, groups):
    import fusor_kernels as fk
    import torch
    print("t2 staged", rows, outputs, groups, flush=True)
    cols = 128 * groups
    data = synthetic_table(O.T2B128, outputs, cols, seed=rows + groups)
    t = table(fk, O.T2B128, outputs, cols, data)
    x = activations(rows, cols, seed=rows, outliers=0.02)
    bias = np.random.default_rng(rows).standard_normal(outputs).astype(np.float32)
    want = oracle_product(O.T2B128, outputs, cols, data, x, rows, bias=bias)
    got = gpu_product(fk, t, x, rows, bias=bias)
    assert same_bits(got, want), first_mismatch(got, want)
    lo, hi = 4, (outputs + 3) // 4 * 4 - 4
    want_r = oracle_product(O.T2B128, outputs, cols, data, x, rows, lo, hi)
    assert same_bits(gpu_product(fk, t, x, rows, cols=range(lo, hi)), want_r)
    out = torch.ones((rows, hi - lo + 3), device="cuda")  # a stride wider than the range
    fk.matmul(t.matrix(), fk.Input(f32=torch.from_numpy(x).cuda()), range(lo, hi), out=out, accumulate=True)
    added = out.cpu().numpy()
    assert same_bits(np.ascontiguousarray(added[:, :hi - lo]), np.float32(1) + want_r) and (added[:, hi - lo:] == 1).all()
    want_f = oracle_product(O.T2B128, outputs, cols, data, x, rows, fused=True)
    assert same_bits(gpu_product(fk, t, x, rows, fused_scale=True), want_f)
