"""The prefill's parallel-order attention (attn_flash_kernel) where its blocks of 32 rows and 32 keys
end: every head size, rows and positions around 32 and around the eight waves' turn of 256 keys, and
caches past what attn_rows_kernel's LDS holds.
The rows of a two-layer read leave their second layer's keys and values in the caches, so the
caches hold every row's attention output as the next layer sees it; they are compared with the
exact-order read of the same rows. The first layer's attention is nearly all that reaches them: its
residual rows are small and its feed-forward adds nothing, so one key wrongly seen or missed moves a
row well past the limit (test_prefill_flash_limit.py plants such mistakes)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# The two orders' attention rows differ by f32 roundings, so a row's levels differ in a value or two that
# lie at a tie: a step of 1/127 of its group's largest value (about 3 standard deviations), 2.4e-2 of
# one value, 0.2e-2 of a row of 128. Each such step moves the next layer's inputs by 0.2e-2, a twelfth
# of their own levels' steps, so a twelfth of those step too: 2.4e-2 * sqrt(1/12) = 0.7e-2 of a row. Two of them
# at once: 1e-2, and 0.3e-2 of their own.
LIMIT = 1.3e-2

HIDDEN, FFN = 128, 32
SEED = 112  # inputs in which every planted mistake moves some row by 3.7e-2 or more
HEADS = {32: (6, 3), 64: (4, 1), 128: (2, 2)}


def weights_of(head_dim, seed):
    """Two layers' f32 weights, their feed-forward adding nothing."""
    heads, kv_heads = HEADS[head_dim]
    rng = np.random.default_rng(seed)
    width, qkv_w = heads * head_dim, (heads + 2 * kv_heads) * head_dim
    layers = []
    for _ in range(2):
        w = {name: (rng.standard_normal(size) / math.sqrt(size[1])).astype(np.float32) for name, size in
             {"qkv": (qkv_w, HIDDEN), "o": (HIDDEN, width), "gate": (FFN, HIDDEN), "up": (FFN, HIDDEN)}.items()}
        w["down"] = np.zeros((HIDDEN, FFN), np.float32)
        layers.append(w)
    return layers


def caches_of(head_dim, capacity, seed):
    rng = np.random.default_rng(seed + 1)
    return [rng.standard_normal((2, HEADS[head_dim][1], capacity, head_dim)).astype(np.float32) for _ in range(2)]


def embeddings_of(rows):
    return 0.01 * np.random.default_rng(rows).standard_normal((rows, HIDDEN)).astype(np.float32)


def model_of(head_dim, capacity, seed):
    heads, kv_heads = HEADS[head_dim]
    layers = []
    for w in weights_of(head_dim, seed):
        layer = {name: O.encode(O.Q7B32, *v.shape, v) for name, v in w.items()}
        layer["norm1"] = layer["norm2"] = np.ones(HIDDEN, np.float32)
        layer["qkv_bias"] = np.zeros(len(w["qkv"]), np.float32)
        layers.append(layer)
    table = O.encode(O.Q7B32, 64, HIDDEN, np.random.default_rng(seed).standard_normal((64, HIDDEN)).astype(np.float32))
    sh = O.Qwen2Shape(hidden=HIDDEN, layers=2, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ffn=FFN, vocab=64,
                      capacity=capacity, rope_base=1e6, eps=1e-6, dtype=O.Q7B32)
    return (sh, layers, np.ones(HIDDEN, np.float32), table, *caches_of(head_dim, capacity, seed))


def row_errors(got, want):
    return np.linalg.norm(got - want, axis=(0, 2)) / np.linalg.norm(want, axis=(0, 2))


def read_caches(fk, params, embeddings, first, chunk, exact):
    import torch
    from test_gpu_prefill import gpu_model
    model, kd, vd = gpu_model(fk, O.Q7B32, params, exact=exact)
    model.read(torch.from_numpy(embeddings).cuda(), first, chunk)
    torch.cuda.synchronize()
    n = len(embeddings)
    return [t.cpu().numpy()[1, :, first:first + n] for t in (kd, vd)]


# few keys stay with attn_rows_kernel: up to 64 (heads of 128: 112), of fewer than 32 rows up to
# 144 (160)
SHAPES = [(1, 160), (7, 158), (31, 130), (32, 96), (33, 95), (65, 63), (129, 0), (40, 255), (33, 700)]
# past 1484, 2988 and 5996 keys (heads of 32, 64, 128) attn_rows_kernel does not hold a block's scores
LONG = [(32, 48, 1480), (64, 110, 2900), (128, 180, 5850)]
CASES = [(d, *s) for d in (32, 64, 128) for s in SHAPES] + LONG


def seed_of(head_dim, rows, first):
    return SEED + head_dim + rows + first


def capacity_of(rows, first):
    return (rows + first + 63) // 32 * 32


@pytest.mark.parametrize("head_dim,rows,first", CASES)
def test_rows_equal_the_exact_order_reads(gpu, head_dim, rows, first):
    import fusor_kernels as fk
    print("flash prefill", head_dim, rows, first, flush=True)
    params = model_of(head_dim, capacity_of(rows, first), seed_of(head_dim, rows, first))
    want = read_caches(fk, params, embeddings_of(rows), first, rows, exact=True)
    got = read_caches(fk, params, embeddings_of(rows), first, rows, exact=False)
    for g, w in zip(got, want):
        assert row_errors(g, w).max() < LIMIT, row_errors(g, w)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_row_that_is_not_finite_reaches_no_earlier_row(gpu, bad):
    """Row 20 holds a value that is not finite: the rows before it, in its own block of keys among
    them, are what they are without it."""
    import fusor_kernels as fk
    params = model_of(64, 128, 9)
    embeddings = embeddings_of(48)
    clean = read_caches(fk, params, embeddings, 70, 48, exact=False)
    embeddings[20, 3] = bad
    for exact in (True, False):
        got = read_caches(fk, params, embeddings, 70, 48, exact=exact)
        for g, c in zip(got, clean):
            assert np.isfinite(g[:, :20]).all()
            assert row_errors(g[:, :20], c[:, :20]).max() < LIMIT
