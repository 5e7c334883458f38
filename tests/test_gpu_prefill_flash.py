"""The prefill's parallel-order attention (attn_flash_kernel) where its blocks of 32 rows and 32 keys
end: every head size, rows and positions around 32 and around the eight waves' turn of 256 keys.
The rows of a two-layer read leave their second layer's keys and values in the caches, so the
caches hold every row's attention output as the next layer sees it; they are compared with the
exact-order read of the same rows."""
import numpy as np
import pytest

from gpu_data import qwen2_model
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# A row that differs by an f32 rounding may quantize to a neighbouring level, a step of 1/127 of a
# group's largest value (about 3 standard deviations of its values): 2.4e-2 of a value at most,
# spread over the 32 products and more that a key or value sums.
LEVEL_STEP = 2.4e-2


def read_caches(fk, params, embeddings, first, chunk, exact):
    import torch
    from test_gpu_prefill import gpu_model
    model, kd, vd = gpu_model(fk, O.Q7B32, params, exact=exact)
    model.read(torch.from_numpy(embeddings).cuda(), first, chunk)
    torch.cuda.synchronize()
    n = len(embeddings)
    return [t.cpu().numpy()[1, :, first:first + n] for t in (kd, vd)]


def model_of(head_dim, capacity, seed):
    heads, kv_heads = {32: (6, 3), 64: (4, 1), 128: (2, 2)}[head_dim]
    return qwen2_model(O.Q7B32, hidden=128, layers=2, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ffn=256, vocab=64,
                       capacity=capacity, seed=seed, synthetic=False)


@pytest.mark.parametrize("head_dim", [32, 64, 128])
# more than 64 keys (112 for heads of 128), or the kernel for few keys takes the chunk
@pytest.mark.parametrize("rows,first", [(1, 112), (31, 82), (32, 96), (33, 95), (65, 63), (129, 0), (40, 255), (33, 700)])
def test_rows_equal_the_exact_order_reads(gpu, head_dim, rows, first):
    import fusor_kernels as fk
    print("flash prefill", head_dim, rows, first, flush=True)
    params = model_of(head_dim, 768, head_dim + rows + first)
    embeddings = np.random.default_rng(rows).standard_normal((rows, 128)).astype(np.float32)
    want = read_caches(fk, params, embeddings, first, rows, exact=True)
    got = read_caches(fk, params, embeddings, first, rows, exact=False)
    for g, w in zip(got, want):
        rel = np.linalg.norm(g - w, axis=(0, 2)) / np.linalg.norm(w, axis=(0, 2))  # a row's error
        assert rel.max() < LEVEL_STEP, rel


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_row_that_is_not_finite_reaches_no_earlier_row(gpu, bad):
    """Row 20 holds a value that is not finite: the rows before it, in its own block of keys among
    them, are what they are without it."""
    import fusor_kernels as fk
    params = model_of(64, 128, 9)
    embeddings = np.random.default_rng(2).standard_normal((48, 128)).astype(np.float32)
    clean = read_caches(fk, params, embeddings, 70, 48, exact=False)
    embeddings[20, 3] = bad
    for exact in (True, False):
        got = read_caches(fk, params, embeddings, 70, 48, exact=exact)
        for g, c in zip(got, clean):
            assert np.isfinite(g[:, :20]).all()
            rel = np.linalg.norm(g[:, :20] - c[:, :20], axis=(0, 2)) / np.linalg.norm(c[:, :20], axis=(0, 2))
            assert rel.max() < LEVEL_STEP
