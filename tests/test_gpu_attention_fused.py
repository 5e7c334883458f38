"""The int8 attention in one launch (attention_fused.hip) at the sizes where its tiles end: head
sizes around 8 and 32 channels, keys around a run of 8, a block of 32, a stage of 64 and the keys'
mean's 512 and 1024, queries around a wave's 32 and a workgroup's 128. Every call's outputs are the oracle's bits, and those of
the step-by-step kernels (FG_ATTEND_UNITS selects them) on the same inputs."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [  # heads, kv_heads, head_dim, images, queries, keys, fast
    (12, 12, 4, 1, 1, 1, True), (12, 12, 8, 1, 33, 7, False), (12, 4, 12, 1, 31, 8, True), (12, 12, 32, 1, 32, 31, True),
    (12, 12, 36, 1, 33, 32, False), (16, 4, 40, 2, 127, 33, True), (12, 12, 64, 1, 128, 63, False),
    (12, 12, 64, 1, 129, 64, True), (12, 12, 72, 2, 65, 65, True), (12, 12, 80, 1, 20, 96, False),
    (12, 12, 88, 1, 40, 97, True), (12, 12, 96, 1, 40, 127, True), (12, 6, 100, 1, 70, 129, False),
    (12, 12, 112, 1, 33, 160, True), (12, 12, 120, 1, 5, 200, True), (12, 2, 128, 1, 130, 513, False),
]

# every record (blocks of 32 channels, eights of channels in the last) over two whole stages of 64 keys and
# a remainder, with both exponentials
RECORDS = [(12, 12 if d % 16 else 3, d, 1, 35, 128 + r, fast) for d, r in
           [(4, 1), (8, 33), (12, 8), (16, 31), (24, 32), (32, 63), (36, 7), (40, 40), (48, 1), (56, 33), (64, 9), (72, 31),
            (80, 32), (88, 63), (96, 5), (104, 40), (112, 1), (120, 33), (128, 17)] for fast in (True, False)]

# the keys' mean goes through two buffers of 512 keys: one and two turns of both, with remainders,
# and the longest a model asks for
LONG = [(24, 6, 64, 1, 33, 1023, True), (24, 24, 8, 1, 20, 1024, False), (24, 6, 64, 1, 33, 1025, False),
        (24, 3, 40, 2, 17, 1536, True), (24, 24, 72, 1, 20, 1537, False), (24, 8, 32, 1, 33, 2048, True),
        (48, 8, 128, 1, 16, 2049, False), (24, 24, 72, 1, 20, 4096, True), (24, 6, 64, 1, 33, 4095, False)]


def call_with(H, KV, D, I, Q, K, q, k, v, fast, pad=0):
    import torch

    import fusor_kernels as fk
    q, k, v = (torch.from_numpy(np.pad(a, ((0, 0), (pad, 0)))).cuda() for a in (q, k, v))
    base = torch.full((I * Q * H * D + pad,), float("nan"), device="cuda")
    out = base[pad:].view(I * Q, H * D)  # a pad of 1: rows that allow no 16-byte access
    fk.attend(fk.Call(H, KV, D, I, Q, K, fk.Operand(q, H * D + pad, pad), fk.Operand(k, KV * D + pad, pad),
                      fk.Operand(v, KV * D + pad, pad), fk.Exponentials.FAST if fast else fk.Exponentials.EXACT), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def inputs(H, KV, D, I, Q, K, spread, seed):
    rng = np.random.default_rng(seed)
    q = (spread * rng.standard_normal((I * Q, H * D))).astype(np.float32)
    return q, *(rng.standard_normal((I * K, KV * D)).astype(np.float32) for _ in range(2))


# spread 1: every weight near the row's largest; 40: most of them below 2^-52 (groups outside the
# shared reciprocal's range) and many at the exponentials' clamp
@pytest.mark.parametrize("spread", [1.0, 40.0])
@pytest.mark.parametrize("shape", SHAPES + RECORDS + LONG)
def test_one_launch_is_the_oracles_bits(gpu, monkeypatch, shape, spread):
    H, KV, D, I, Q, K, fast = shape
    print("attend", shape, spread, flush=True)
    q, k, v = inputs(H, KV, D, I, Q, K, spread, seed=D * 1000 + K)
    want = O.attend(H, KV, D, I, Q, K, q, k, v, fast=fast)
    monkeypatch.delenv("FG_ATTEND_UNITS", raising=False)
    for pad in (0, 1):
        got = call_with(H, KV, D, I, Q, K, q, k, v, fast, pad)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (pad, np.max(np.abs(got - want)))
    monkeypatch.setenv("FG_ATTEND_UNITS", "64")
    steps = call_with(H, KV, D, I, Q, K, q, k, v, fast)
    assert np.array_equal(steps.view(np.uint32), want.view(np.uint32))


def test_one_launch_with_infinities_and_nan(gpu, monkeypatch):
    """Infinite and NaN queries, keys and values: the same values as the step-by-step kernels (NaN
    where they are NaN, equal elsewhere)."""
    H, KV, D, I, Q, K = 12, 12, 64, 1, 40, 70
    q, k, v = inputs(H, KV, D, I, Q, K, 1.0, seed=4)
    q[3, 5], q[4, 70], k[9, 130], v[11, 200], v[12, 300] = np.inf, np.nan, np.nan, np.inf, np.nan
    k[20, 400] = -np.inf
    monkeypatch.delenv("FG_ATTEND_UNITS", raising=False)
    for fast in (True, False):
        got = call_with(H, KV, D, I, Q, K, q, k, v, fast)
        monkeypatch.setenv("FG_ATTEND_UNITS", "64")
        want = call_with(H, KV, D, I, Q, K, q, k, v, fast)
        monkeypatch.delenv("FG_ATTEND_UNITS")
        assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("fast", [True, False])
def test_one_launch_with_subnormal_scales(gpu, monkeypatch, fast):
    """The first stage's keys take all of the weight, but its values are 0, so the outputs are sums of
    weights at the exponentials' clamp (e^-87): their groups' scales, and the products of those
    scales with the values' scales, are subnormal."""
    H, KV, D, I, Q, K = 12, 12, 96, 1, 40, 150
    q, k, v = inputs(H, KV, D, I, Q, K, 1.0, seed=6)
    q, k = np.abs(q) + 1, 0.1 * k
    k[:64] += 30
    v[:64] = 0
    v[100:] *= 1e3
    want = O.attend(H, KV, D, I, Q, K, q, k, v, fast=fast)
    assert 0 < np.abs(want).max() < 1e-33 and (np.abs(want[want != 0]) < 2.0 ** -126).any()
    monkeypatch.delenv("FG_ATTEND_UNITS", raising=False)
    got = call_with(H, KV, D, I, Q, K, q, k, v, fast)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.max(np.abs(got - want))
