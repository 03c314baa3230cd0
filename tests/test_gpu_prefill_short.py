"""GPU parity of the prefill kernel for short calls (16 columns of positions x query heads per workgroup, the keys dealt
out over its waves) against the float64 oracle, at the sizes where it can go wrong: one row, tiles that start in front
of the call's first row or end behind its last, group sizes that leave columns empty, windows of one key up to wider
than the context, one key block per tile and more blocks than waves, both wave counts (launches of up to 256 workgroups
run eight waves each, larger ones four), every pair of cache and activation type, soft cap.

Bounds: 1e-5 for a float32 cache; 2e-3 of the largest value otherwise (half operands), where bfloat16 outputs are
compared after discounting the half ulp of the output format, and bfloat16 keys and queries enter the oracle rounded.
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


def queries(x, kv, io):
    """In the activation type, with values that the matrix cores take as they are: float32 queries over a 16-bit cache are
    rounded to the cache's type by definition, so the oracle gets the rounded values too."""
    if io == A.F32 and kv in (A.F16, A.BF16):
        return rounded(rounded(x, kv)[1], A.F32)
    return rounded(x, io)


def fill(at, kv, layer, seq, L, hkv, seed):
    k, v = gen(seed, L, hkv, D), gen(seed + 1, L, hkv, D)
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
    if io == A.BF16:
        err = orc.rel_err_beyond_bf16_rounding(got, ref)
    else:
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
    assert err < (1e-5 if kv == A.F32 else 2e-3), (what, err)


PAIRS = [(A.F32, A.F32), (A.F16, A.F16), (A.F16, A.F32), (A.BF16, A.BF16), (A.BF16, A.F32), (A.I8, A.F16), (A.I8, A.BF16),
         (A.I8, A.F32)]


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2), (3, 1), (16, 1), (2, 2), (9, 1)])
def test_edges_of_tiles_windows_and_groups(kv, io, hq, hkv):
    L = 400
    windows = [0, 1, 17, 70, 1000]
    # (rows, windows and lengths on both sides of the 16- and 64-token blocks; the context goes on behind the call)
    with A.Attn(len(windows), hq, hkv, D, L, 2, kv, io, layer_window=windows, scale=0.07,
                stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_option("prefill_short", 1)
        rows = [fill(at, kv, layer, 1, L, hkv, 10 * layer + 1) for layer in range(len(windows))]
        for q_pos0, n in ((0, 1), (0, 15), (0, 64), (3, 30), (63, 2), (70, 129), (399, 1), (50, 350)):
            for layers in ((0, 5), (3, 1)):  # all layers in one call; one layer
                qd, qr = queries(gen(900 + n, layers[1], n, hq, D), kv, io)
                out = torch.full_like(qd, float("nan"))
                at.prefill(layers[0], 1, q_pos0, n, qd, out, n_layers=layers[1])
                torch.cuda.synchronize()
                got = out.float().cpu().numpy()
                for i in range(layers[1]):
                    k, v = rows[layers[0] + i]
                    ref = c_oracle.sdpa_f64(qr[i], k, v, 0.07, q_pos0=q_pos0, window=windows[layers[0] + i], kv_len=q_pos0 + n)
                    check(got[i], ref, kv, io, (q_pos0, n, layers, i))


@pytest.mark.parametrize("kv,io", PAIRS)
@pytest.mark.parametrize("n", [1021, 1025])
def test_both_wave_counts(kv, io, n):
    # 4 heads on 1 KV head behind 2 rows: 256 tiles of four positions (eight waves) and 257 (four waves)
    hq, hkv, q_pos0 = 4, 1, 2
    L = q_pos0 + n
    with A.Attn(1, hq, hkv, D, L, 1, kv, io, layer_window=[600], softcap=20.0, stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_option("prefill_short", 1)
        k, v = fill(at, kv, 0, 0, L, hkv, 71)
        qd, qr = queries(2.0 * gen(72, n, hq, D), kv, io)
        out = torch.full_like(qd, float("nan"))
        at.prefill(0, 0, q_pos0, n, qd, out)
        torch.cuda.synchronize()
        ref = c_oracle.sdpa_f64(qr, k, v, D ** -0.5, q_pos0=q_pos0, window=600, softcap=20.0, kv_len=L)
        check(out.float().cpu().numpy(), ref, kv, io, n)


def test_rule_and_switch():
    # a short call takes the kernel by rule (same bits as the switch), a call over many layers does not, and an option
    # that asks for one of the other kernels is followed
    hq, hkv, n, nl = 4, 1, 512, 26
    with A.Attn(nl, hq, hkv, D, n, 1, A.F16, A.F16, stream=torch.cuda.current_stream().cuda_stream) as at:
        for layer in range(nl):
            fill(at, A.F16, layer, 0, n, hkv, 5)
        qd, _ = rounded(gen(7, nl, n, hq, D), A.F16)

        def run(layers, **options):
            for name, value in options.items():
                at.set_option(name, value)
            q = qd[:layers].contiguous()
            out = torch.empty_like(q)
            at.prefill(0, 0, 0, n, q, out, n_layers=layers)
            torch.cuda.synchronize()
            return out

        short = run(1, prefill_short=1)
        assert torch.equal(run(1, prefill_short=-1), short)
        assert not torch.equal(run(1, prefill_rows16=0), short)
        at.set_option("prefill_rows16", -1)
        whole = run(nl, prefill_short=0)
        assert torch.equal(run(nl, prefill_short=-1), whole)
        assert not torch.equal(run(nl, prefill_short=1), whole)
        with pytest.raises(A.AttnError):
            at.set_option("prefill_short", 2)


@pytest.mark.parametrize("option,value", [("prefill_rows16", 1), ("prefill_key_split", 0), ("prefill_workgroups", 7)])
def test_float32_cache_under_options_of_the_tiled_kernels(option, value):
    # no tiled kernel takes a float32 cache, so options that choose among them leave its calls where they are (they used
    # to send them to the row-wise path, at two to four times the time)
    hq, hkv, n = 4, 1, 200
    with A.Attn(1, hq, hkv, D, n, 1, A.F32, A.F32, stream=torch.cuda.current_stream().cuda_stream) as at:
        fill(at, A.F32, 0, 0, n, hkv, 5)
        qd, _ = rounded(gen(7, n, hq, D), A.F32)

        def run():
            out = torch.empty_like(qd)
            at.prefill(0, 0, 0, n, qd, out)
            torch.cuda.synchronize()
            return out

        want = run()
        at.set_option(option, value)
        assert torch.equal(run(), want)
        at.set_option("rowwise_prefill", 1)
        assert not torch.equal(run(), want)  # (that path sums in another order)
