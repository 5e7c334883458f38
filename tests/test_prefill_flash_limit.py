"""The limit of test_gpu_prefill_flash.py is one that mistakes in the attention exceed: that test's
model in 64-bit numpy, with a key missed or wrongly seen by every row, or a block of keys lost."""
import math

import numpy as np
import pytest

from test_gpu_prefill_flash import CASES, HEADS, HIDDEN, LIMIT, caches_of, capacity_of, embeddings_of, row_errors, seed_of, weights_of


def rotated(x, positions):
    half = x.shape[-1] // 2
    angle = positions[:, None] * (1.0 / 1e6 ** (np.arange(half) * 2 / x.shape[-1]))
    c, s = np.cos(angle)[:, None], np.sin(angle)[:, None]
    a, b = x[..., :half], x[..., half:]
    return np.concatenate([a * c - b * s, b * c + a * s], -1)


def normed(x):
    return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-6)


def next_rows(head_dim, rows, first, mistake):
    """The second layer's keys and values of the read, with `mistake` (from the rows' masks) in the first's."""
    seed, capacity = seed_of(head_dim, rows, first), capacity_of(rows, first)
    heads, kv_heads = HEADS[head_dim]
    w0, w1 = weights_of(head_dim, seed)
    kc, vc = (c[0].astype(np.float64) for c in caches_of(head_dim, capacity, seed))
    positions = np.arange(first, first + rows)
    x = embeddings_of(rows).astype(np.float64)

    def projected(w, x):
        qkv = (normed(x) @ w["qkv"].T.astype(np.float64)).reshape(rows, heads + 2 * kv_heads, head_dim)
        q, k, v = np.split(qkv, [heads, heads + kv_heads], 1)
        return rotated(q, positions), rotated(k, positions), v

    q, k, v = projected(w0, x)
    kc[:, first:first + rows], vc[:, first:first + rows] = k.transpose(1, 0, 2), v.transpose(1, 0, 2)
    mask = mistake(np.arange(capacity)[None] <= positions[:, None], positions)
    out = np.empty((rows, heads, head_dim))
    for h in range(heads):
        kv = h // (heads // kv_heads)
        s = np.where(mask, q[:, h] @ kc[kv].T / math.sqrt(head_dim), -np.inf)
        e = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = e / e.sum(1, keepdims=True) @ vc[kv]
    _, k, v = projected(w1, x + out.reshape(rows, -1) @ w0["o"].T.astype(np.float64))
    return k.transpose(1, 0, 2), v.transpose(1, 0, 2)


def without(keys):
    """Every row misses the keys that `keys(positions)` gives it."""
    def mistake(mask, positions):
        mask = mask.copy()
        lost = keys(positions)
        for r, row in enumerate(mask):
            row[lost[r]] = False
        return mask
    return mistake


def one_later(mask, positions):
    mask = mask.copy()
    mask[np.arange(len(mask)), positions + 1] = True
    return mask


MISTAKES = {
    "own key missed": without(lambda p: [[i] for i in p]),
    "key before missed": without(lambda p: [[i - 1] for i in p]),
    "first key missed": without(lambda p: [[0] for _ in p]),
    "one later key seen": one_later,
    "last whole block of keys missed": without(lambda p: [slice((i + 1) // 32 * 32 - 32, (i + 1) // 32 * 32) for i in p]),
    "second block of keys missed": without(lambda p: [slice(32, 64) for _ in p]),
}


@pytest.mark.parametrize("head_dim,rows,first", CASES)
def test_mistakes_exceed_the_limit(head_dim, rows, first):
    right = next_rows(head_dim, rows, first, lambda mask, positions: mask)
    for name, mistake in MISTAKES.items():
        if first == 0 and "missed" in name:  # rows of few keys would have none left
            continue
        wrong = next_rows(head_dim, rows, first, mistake)
        worst = max(row_errors(g, w).max() for g, w in zip(wrong, right))
        assert worst > 2.5 * LIMIT, (name, worst)
