"""GPU parity of decode calls by the count of their partitions, which mi355_attn_decode_plan_probe confirms: every edge of the
merges (rows of 16 a wave, two rows of 16 at a time in the launch, one to four waves and up to four trips in the merge launch),
by explicit counts and by the rule, up to the most (256); the same partitions merged in the launch and by the merge launch;
the fused step; and lengths read from tables. Against the float64 oracle.

Bounds, of the largest value: 1e-5 for a float32 cache, 2e-3 otherwise (half operands; bfloat16 outputs are compared after
discounting the half ulp of the format).
"""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from __graft_entry__ import load_package  # noqa: E402
from oracle import attn_oracle as orc  # noqa: E402
from oracle import c_oracle  # noqa: E402

A = load_package().attn
DEV = "cuda:0"
TDT = {A.F32: torch.float32, A.F16: torch.float16, A.BF16: torch.bfloat16, A.I8: torch.int8}
D = 256
PAIRS = [(A.F32, A.F32), (A.F16, A.F16), (A.BF16, A.BF16), (A.I8, A.F16)]


def rnd(seed, shape, dtype):
    x = torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)
    return (x * 40).round().clamp(-127, 127).to(torch.int8) if dtype == torch.int8 else x.to(dtype)


def host(x):
    return x.float().cpu().numpy()


def handle(kv, io, hq, hkv, ctx, batch=1):
    return A.Attn(1, hq, hkv, D, ctx, batch, kv, io, scale=0.07, stream=torch.cuda.current_stream().cuda_stream)


def fill(at, kv, seq, n, hkv, seed):
    k, v = (rnd(seed + i, (n, hkv, D), TDT[kv]) for i in range(2))
    at.kv_append(0, seq, 0, k, v)
    if kv == A.I8:
        s = torch.rand((2, hkv, D), generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV) * 0.01 + 0.02
        at.kv_set_scales(0, seq, s[0].contiguous(), s[1].contiguous())
        return host(k) * host(s[0]), host(v) * host(s[1])
    return host(k), host(v)


def check(got, q, k, v, n, kv, io, what):
    ref = c_oracle.sdpa_f64(host(q), k, v, 0.07, q_pos0=n - 1, kv_len=n)
    got = host(got)
    err = orc.rel_err_beyond_bf16_rounding(got, ref) if io == A.BF16 else float(np.abs(got - ref).max() / np.abs(ref).max())
    assert err < (1e-5 if kv == A.F32 else 2e-3), (what, err)


def call(at, lens, q, splits=0, seq_ids=None):
    out = torch.full_like(q, float("nan"))
    for _ in range(2):  # (the second call finds the tickets as the first has left them)
        at.decode(0, lens, q, out, num_splits=splits, seq_ids=seq_ids)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("hq,hkv", [(4, 1), (16, 1), (16, 8)])
def test_exact_counts(kv, io, hq, hkv):
    ctx = 64 * 256
    with handle(kv, io, hq, hkv, ctx) as at:
        k, v = fill(at, kv, 0, ctx, hkv, 1)
        q = rnd(7, (1, hq, D), TDT[io])
        for count in (2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256):
            n = 64 * count - (count * 7) % 64  # whole 64 tokens a partition, the last one short
            plan = A.decode_plan(kv, hq, hkv, [0], [n], count)
            assert plan[0] == count and plan[1] == (count <= 64 and count * hkv <= 256)
            check(call(at, [n], q, count), q, k, v, n, kv, io, count)


@pytest.mark.parametrize("kv,io", PAIRS)
def test_counts_by_the_rule(kv, io):
    hq, hkv, ctx = 4, 1, 33000
    lens = [(n + 1) // 2 if kv == A.F32 else n for n in (4300, 8000, 8193, 12400, 16385, 24700, 32768, 32769)]
    counts = [A.decode_plan(kv, hq, hkv, [0], [n])[0] for n in lens]
    if kv != A.I8:
        assert max(counts) == 256
    assert sum(n > 64 for n in counts) >= 4 and sum(n > 128 for n in counts) >= 2
    with handle(kv, io, hq, hkv, ctx) as at:
        k, v = fill(at, kv, 0, ctx, hkv, 3)
        q, nk, nv = (rnd(9 + i, (1, h, D), TDT[io]) for i, h in enumerate((hq, hkv, hkv)))
        at.set_layer_transform(0, norm_q=True, norm_k=True, eps=1e-6, rope_inv_freq=(10000.0 ** -(np.arange(0, D, 2) / D)).astype(np.float32))
        for n, count in reversed(list(zip(lens, counts))):  # (the step writes row n - 1: longest first)
            check(call(at, [n], q), q, k, v, n, kv, io, (n, count))
            step, two, turned = (torch.full_like(q, float("nan")) for _ in range(3))
            at.decode_step(0, [n], q, nk, nv, step)
            at.pre_attention(0, 0, n - 1, q, nk, nv, turned)
            at.decode(0, [n], turned, two)
            torch.cuda.synchronize()
            assert torch.isfinite(step.float()).all() and torch.equal(step, two), (n, count)


@pytest.mark.parametrize("kv,io", PAIRS)
def test_merged_in_the_launch_or_by_the_merge_launch(kv, io):
    """A sequence alone and among others, in the same partitions by the same waves: the same bits from either merge."""
    hq, hkv, batch = 8, 2, 65
    with handle(kv, io, hq, hkv, 64 * 64, batch) as at:
        for b in range(batch):
            fill(at, kv, b, 64 * 64 if b == 0 else 64, hkv, 2 * b)
        at.set_option("decode_waves", 1)
        q = rnd(5, (batch, hq, D), TDT[io])
        for count in (2, 16, 17, 33, 48, 49, 64):
            n = 64 * count - 5
            lens = [n] + [64] * (batch - 1)
            assert A.decode_plan(kv, hq, hkv, [0], [n], count)[:2] == (count, True)
            assert A.decode_plan(kv, hq, hkv, [0], lens, count)[:2] == (count, False)
            assert torch.equal(call(at, [n], q[:1].contiguous(), count)[0], call(at, lens, q, count)[0]), count


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("batch,n,splits", [(65, 500, 2), (100, 700, 2), (128, 1000, 2), (85, 700, 3), (100, 700, 0)])
def test_lengths_in_tables(kv, io, batch, n, splits):
    """More sequences than a launch carries, in partitions that the launch merges itself."""
    hq, hkv = 4, 1
    lens = [max(1, n - (37 * b) % n) for b in range(batch)]
    plan = A.decode_plan(kv, hq, hkv, [0], lens, splits)
    assert splits == 0 or plan[:2] == (splits, True)
    with handle(kv, io, hq, hkv, n, batch) as at:
        rows = [fill(at, kv, b, lens[b], hkv, 2 * b) for b in range(batch)]
        order = [(b * 7 + 3) % batch if batch % 7 else b for b in range(batch)]
        q = rnd(11, (batch, hq, D), TDT[io])
        out = call(at, [lens[b] for b in order], q, splits, seq_ids=order)
        for j, b in enumerate(order):
            check(out[j:j + 1], q[j:j + 1], *rows[b], lens[b], kv, io, (j, b))
