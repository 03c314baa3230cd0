"""Prefill launches of few, long tiles: the keys of a tile are cut into as few parts as do, of the same length but for
the last, and, where the measured times say so, run as a direct launch (a workgroup per item on 16x16x32 MFMAs, no work
plan). Checked against the float64 oracle where it can go wrong: tiles whose block counts leave parts empty or a block shorter than the others, ragged
ends, windows on some layers only (their tiles have fewer parts than the launch has room for), more parts than the
merge asks for at once, float32 output, and an int8 cache through its staged planes.

Bound: 2e-3 of the largest value (half operands; the queries enter the oracle as the matrix cores take them).
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
D = 256


def gen(seed, *shape):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def half(x):
    t = torch.from_numpy(np.ascontiguousarray(x)).to(DEV).half().contiguous()
    return t, t.float().cpu().numpy()


@pytest.mark.parametrize("kv", [A.F16, A.I8])
@pytest.mark.parametrize("io", [A.F16, A.F32])
@pytest.mark.parametrize("hq,hkv,start,n,windows,key_split", [
    (8, 2, 4000, 2047, [0], -1),          # 128 items, four parts each: the direct launch, by rule
    (8, 2, 3990, 1400, [0, 900], -1),     # two layers, two parts; the windowed tiles are whole, their second part is empty
    (8, 2, 6000, 1000, [0, 2500], -1),    # four parts; the windowed tiles have two of them
    (6, 2, 5001, 1500, [0], -1),          # three heads a KV head: 128 positions a tile
    (4, 1, 1000, 333, [0, 200], 3),    # up to 14 parts: more than the merge asks for at once
])
def test_split_tiles_against_the_oracle(kv, io, hq, hkv, start, n, windows, key_split):
    L, nl = start + n, len(windows)
    if key_split < 0:
        route, parts = A.prefill_route(kv, hq, hkv, windows, start, n)
        assert route == A.ROUTE_DIRECT16 and parts > 1
    with A.Attn(nl, hq, hkv, D, L, 1, kv, io, layer_window=windows, stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_option("prefill_short", 0)
        at.set_option("prefill_key_split", key_split)
        k, v = gen(1, L, hkv, D), gen(2, L, hkv, D)
        if kv == A.I8:
            kq, ks = orc.quantize_kv_int8(k)
            vq, vs = orc.quantize_kv_int8(v)
            kd, vd = torch.from_numpy(kq).to(DEV), torch.from_numpy(vq).to(DEV)
            k, v = orc.dequantize_kv_int8(kq, ks), orc.dequantize_kv_int8(vq, vs)
        else:
            (kd, k), (vd, v) = half(k), half(v)
        for layer in range(nl):
            at.kv_append(layer, 0, 0, kd, vd)
            if kv == A.I8:
                at.kv_set_scales(layer, 0, torch.from_numpy(ks).to(DEV), torch.from_numpy(vs).to(DEV))
        qd, qr = half(gen(3, nl, n, hq, D))
        if io == A.F32:
            qd = qd.float()
        out = torch.full_like(qd, float("nan"))
        for _ in range(2):
            at.prefill(0, 0, start, n, qd, out, n_layers=nl)
        torch.cuda.synchronize()
        got = out.float().cpu().numpy()
        assert np.isfinite(got).all()
        # (every 7th row and the ends of the call: the oracle is float64 on the CPU)
        rows = sorted(set(range(0, n, 7)) | set(range(n - 40, n)) | set(range(40)))
        for layer, w in enumerate(windows):
            worst = 0.0
            for r in rows[::4]:
                ref = c_oracle.sdpa_f64(qr[layer, r:r + 1], k, v, D ** -0.5, q_pos0=start + r, window=w, kv_len=start + r + 1)
                worst = max(worst, float(np.abs(got[layer, r] - ref[0]).max() / np.abs(ref).max()))
            assert worst < 2e-3, (layer, worst)
