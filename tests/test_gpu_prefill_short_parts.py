"""GPU parity of short prefill calls whose tiles are cut over the keys into parts that the launch merges itself, against the
float64 oracle: from one tile (eight parts) to 128 (two, which fill the workspace and the tickets to their end) and one more
(none), contexts that leave the last part short or missing, windows that cut the tiles unequally, several layers and KV heads,
one to 16 query heads a KV head, soft-capped scores, every pair of types, repeated calls (the tickets are zero again) and
replays of a graph recorded before any eager call.

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


def fill(at, kv, layer, n, hkv, seed):
    k, v = gen(seed, n, hkv, D), gen(seed + 1, n, hkv, D)
    if kv == A.I8:
        kq, ks = orc.quantize_kv_int8(k)
        vq, vs = orc.quantize_kv_int8(v)
        at.kv_append(layer, 0, 0, torch.from_numpy(kq).to(DEV), torch.from_numpy(vq).to(DEV))
        at.kv_set_scales(layer, 0, torch.from_numpy(ks).to(DEV), torch.from_numpy(vs).to(DEV))
        return orc.dequantize_kv_int8(kq, ks), orc.dequantize_kv_int8(vq, vs)
    kd, kr = rounded(k, kv)
    vd, vr = rounded(v, kv)
    at.kv_append(layer, 0, 0, kd, vd)
    return kr, vr


PAIRS = [(A.F32, A.F32), (A.F16, A.F16), (A.BF16, A.BF16), (A.BF16, A.F32), (A.I8, A.F16), (A.I8, A.BF16)]


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2), (3, 1)])
def test_parts_of_tiles(kv, io, hq, hkv):
    L = 2300
    windows = [0, 1500]
    with A.Attn(len(windows), hq, hkv, D, L, 1, kv, io, layer_window=windows, scale=0.07,
                stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_option("prefill_short", 1)
        rows = [fill(at, kv, layer, L, hkv, 10 * layer + 1) for layer in range(len(windows))]
        # (tiles of 4 positions: from one of them to more than 128)
        for q_pos0, n in ((2299, 1), (2049, 3), (1000, 63), (1, 300), (1780, 513)):
            for layers in ((0, 1), (0, 2)):
                qd, qr = rounded(gen(900 + n, layers[1], n, hq, D), io)
                if io == A.F32 and kv in (A.F16, A.BF16):  # (what the matrix cores take, by definition)
                    qd, qr = rounded(rounded(qr, kv)[1], A.F32)
                out = torch.full_like(qd, float("nan"))
                for _ in range(2):  # (the second call finds the tickets as the first has left them)
                    at.prefill(layers[0], 0, q_pos0, n, qd, out, n_layers=layers[1])
                torch.cuda.synchronize()
                got = out.float().cpu().numpy()
                for i in range(layers[1]):
                    k, v = rows[layers[0] + i]
                    ref = c_oracle.sdpa_f64(qr[i], k, v, 0.07, q_pos0=q_pos0, window=windows[layers[0] + i], kv_len=q_pos0 + n)
                    err = orc.rel_err_beyond_bf16_rounding(got[i], ref) if io == A.BF16 else float(np.abs(got[i] - ref).max() / np.abs(ref).max())
                    assert err < (1e-5 if kv == A.F32 else 2e-3), (q_pos0, n, layers, i, err)


# query heads, KV heads, start, rows, parts of a tile, soft cap
SHAPES = [(4, 1, 1500, 512, 2, 0.0), (4, 1, 1500, 512, 2, 30.0), (4, 1, 1500, 513, 1, 0.0), (16, 1, 3000, 20, 8, 0.0), (16, 1, 3000, 100, 2, 30.0),
          (1, 1, 3000, 300, 8, 0.0), (1, 1, 3001, 64, 8, 30.0), (8, 2, 3000, 64, 8, 0.0)]


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("hq,hkv,start,n,parts,softcap", SHAPES)
def test_counts_of_parts(kv, io, hq, hkv, start, n, parts, softcap):
    if parts > 1:
        assert A.prefill_route(kv, hq, hkv, [0], start, n) == (A.ROUTE_SHORT, parts)
    with A.Attn(1, hq, hkv, D, start + n, 1, kv, io, scale=0.07, softcap=softcap, stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_option("prefill_short", 1)
        k, v = fill(at, kv, 0, start + n, hkv, 3)
        qd, qr = rounded(gen(n, n, hq, D), io)
        if io == A.F32 and kv in (A.F16, A.BF16):  # (what the matrix cores take, by definition)
            qd, qr = rounded(rounded(qr, kv)[1], A.F32)
        out = torch.full_like(qd, float("nan"))
        for _ in range(2):  # (the second call finds the tickets as the first has left them)
            at.prefill(0, 0, start, n, qd, out)
        torch.cuda.synchronize()
        got = out.float().cpu().numpy()
        ref = c_oracle.sdpa_f64(qr, k, v, 0.07, q_pos0=start, softcap=softcap, kv_len=start + n)
        err = orc.rel_err_beyond_bf16_rounding(got, ref) if io == A.BF16 else float(np.abs(got - ref).max() / np.abs(ref).max())
        assert err < (1e-5 if kv == A.F32 else 2e-3), err


@pytest.mark.parametrize("kv", [A.F16, A.F32, A.I8])
def test_recorded_first_and_replayed(kv):
    io = A.F16 if kv == A.I8 else kv
    hq, hkv, start, n = 4, 1, 1500, 40
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        with A.Attn(1, hq, hkv, D, start + n, 1, kv, io, stream=side.cuda_stream) as at:
            at.set_option("prefill_short", 1)
            fill(at, kv, 0, start + n, hkv, 1)
            q = rounded(gen(2, n, hq, D), io)[0]
            eager, out = torch.empty_like(q), torch.empty_like(q)
            side.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side):
                at.prefill(0, 0, start, n, q, out)
            for _ in range(4):
                out.fill_(float("nan"))
                g.replay()
                at.prefill(0, 0, start, n, q, eager)
                side.synchronize()
                assert torch.equal(out, eager)
            del g
