"""GPU parity of decode launches of up to one workgroup a compute unit, whose partials are merged by the workgroup that
writes the last of them, and of the launches next to them, against the float64 oracle: partitions of one key block up to
more than the merge has in one trip, contexts that end inside, at and behind a block (exact counts of partitions, up to the
most, are in test_gpu_decode_partitions.py), sequences of unequal lengths (some with a single partition), windows, more different windows than a
launch carries, 16 query heads on a KV head, repeated calls (the tickets are zero again), replays of a graph; and the fused
step against its two calls on both sides of the line between row waves of their own and shared ones.

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
TDT = {A.F32: torch.float32, A.F16: torch.float16, A.BF16: torch.bfloat16}
D = 256


def gen(seed, *shape):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def rounded(x, dt):
    t = torch.from_numpy(np.ascontiguousarray(x)).to(DEV).to(TDT[dt]).contiguous()
    return t, t.float().cpu().numpy()


def fill(at, kv, layer, seq, n, hkv, seed):
    k, v = gen(seed, n, hkv, D), gen(seed + 1, n, hkv, D)
    if kv == A.I8:
        kq, ks = orc.quantize_kv_int8(k)
        vq, vs = orc.quantize_kv_int8(v)
        at.kv_append(layer, seq, 0, torch.from_numpy(kq).to(DEV), torch.from_numpy(vq).to(DEV))
        at.kv_set_scales(layer, seq, torch.from_numpy(ks).to(DEV), torch.from_numpy(vs).to(DEV))
        return orc.dequantize_kv_int8(kq, ks), orc.dequantize_kv_int8(vq, vs)
    kd, kr = rounded(k, kv)
    vd, vr = rounded(v, kv)
    at.kv_append(layer, seq, 0, kd, vd)
    return kr, vr


def check(got, ref, kv, io, what):
    err = orc.rel_err_beyond_bf16_rounding(got, ref) if io == A.BF16 else float(np.abs(got - ref).max() / np.abs(ref).max())
    assert err < (1e-5 if kv == A.F32 else 2e-3), (what, err)


def stream():
    return torch.cuda.current_stream().cuda_stream


PAIRS = [(A.F32, A.F32), (A.F16, A.F16), (A.BF16, A.BF16), (A.F16, A.F32), (A.I8, A.F16), (A.I8, A.BF16)]


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2), (16, 1), (3, 1)])
def test_partitions_on_both_sides_of_every_line(kv, io, hq, hkv):
    L = 2200
    windows = [0, 100, 1000]
    lens = [L, 1, 15, 64, 1057, 2049]
    with A.Attn(len(windows), hq, hkv, D, L, len(lens), kv, io, layer_window=windows, scale=0.07, stream=stream()) as at:
        rows = [[fill(at, kv, layer, b, L, hkv, 100 * layer + 7 * b + 1) for b in range(len(lens))] for layer in range(len(windows))]
        for layers in ((0, 1), (1, 1), (2, 1), (0, 3)):
            qd, qr = rounded(gen(5 + layers[0], layers[1], len(lens), hq, D), io)
            if io == A.F32 and kv in (A.F16, A.BF16):  # (what the matrix cores take, by definition)
                qd, qr = rounded(rounded(qr, kv)[1], A.F32)
            ref = [[c_oracle.sdpa_f64(qr[i, b:b + 1], *rows[layers[0] + i][b], 0.07, q_pos0=n - 1, window=windows[layers[0] + i], kv_len=n)
                    for b, n in enumerate(lens)] for i in range(layers[1])]
            for batch in ([0], [4], [0, 1, 2, 3, 4, 5]):
                q = qd[:, batch].contiguous()
                for splits in (0, 2, 5, 16, 17, 33, 40, 64, 65):
                    out = torch.full_like(q, float("nan"))
                    for _ in range(2):  # (the second call finds the tickets as the first has left them)
                        at.decode(layers[0], [lens[b] for b in batch], q, out, seq_ids=batch, num_splits=splits, n_layers=layers[1])
                    torch.cuda.synchronize()
                    got = out.float().cpu().numpy()
                    for i in range(layers[1]):
                        for j, b in enumerate(batch):
                            check(got[i, j], ref[i][b][0], kv, io, (layers, batch, splits, i, b))


def test_more_windows_than_a_launch_carries():
    hq, hkv, n = 4, 1, 300
    windows = [0, 10, 40, 130, 200, 1]
    with A.Attn(len(windows), hq, hkv, D, n, 1, A.F16, A.F16, layer_window=windows, stream=stream()) as at:
        rows = [fill(at, A.F16, layer, 0, n, hkv, 3 * layer) for layer in range(len(windows))]
        qd, qr = rounded(gen(8, len(windows), 1, hq, D), A.F16)
        out = torch.empty_like(qd)
        at.decode(0, [n], qd, out, n_layers=len(windows))
        torch.cuda.synchronize()
        for i, w in enumerate(windows):
            ref = c_oracle.sdpa_f64(qr[i], *rows[i], D ** -0.5, q_pos0=n - 1, window=w, kv_len=n)
            check(out[i].float().cpu().numpy(), ref, A.F16, A.F16, w)


@pytest.mark.parametrize("kv", [A.F16, A.BF16, A.F32, A.I8])
@pytest.mark.parametrize("batch,hkv,ctx", [(1, 1, 260), (1, 4, 2000), (8, 1, 700), (64, 4, 60), (64, 4, 700), (33, 2, 1100)])
def test_fused_step_equals_its_two_calls(kv, batch, hkv, ctx):
    hq, io = 2 * hkv, A.F16 if kv == A.I8 else kv
    with A.Attn(1, hq, hkv, D, ctx, batch, kv, io, layer_window=[600], stream=stream()) as at:
        at.set_layer_transform(0, norm_q=True, norm_k=True, q_weight=0.1 * gen(1, D), k_weight=0.1 * gen(2, D), eps=1e-6,
                               weight_offset=1.0, rope_inv_freq=(10000.0 ** -(np.arange(0, D, 2) / D)).astype(np.float32))
        lens = [ctx - (7 * b) % (ctx // 2) for b in range(batch)]
        for b in range(batch):
            fill(at, kv, 0, b, lens[b] - 1, hkv, b)
        q, k, v = (rounded(gen(60 + i, batch, h, D), io)[0] for i, h in enumerate((hq, hkv, hkv)))
        step, two = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
        for _ in range(2):
            at.decode_step(0, lens, q, k, v, step)
        turned = torch.empty_like(q)
        for b in range(batch):
            at.pre_attention(0, b, lens[b] - 1, q[b:b + 1], k[b:b + 1], v[b:b + 1], turned[b:b + 1])
        at.decode(0, lens, turned, two)
        torch.cuda.synchronize()
        assert torch.isfinite(step.float()).all()
        assert torch.equal(step, two)


def test_replays_of_a_launch_that_merges_itself():
    hq, hkv, n = 4, 1, 1152
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        with A.Attn(1, hq, hkv, D, n, 1, A.F16, A.F16, stream=side.cuda_stream) as at:
            fill(at, A.F16, 0, 0, n, hkv, 1)
            q = rounded(gen(2, 1, hq, D), A.F16)[0]
            eager, out = torch.empty_like(q), torch.empty_like(q)
            at.decode(0, [n], q, eager)
            side.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side):
                at.decode(0, [n], q, out)
            for _ in range(4):
                out.fill_(float("nan"))
                g.replay()
                at.decode(0, [n], q, eager)
                side.synchronize()
                assert torch.equal(out, eager)
            del g
