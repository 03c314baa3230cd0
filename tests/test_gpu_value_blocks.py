"""The value rows of the step before attention: blocks of the V plane that a call covers as a whole are assembled in LDS
and written as 16-byte chunks, the ends row by row (over an int8 cache short calls go row by row altogether). Both ways
must leave the same bytes: a call over n rows against n calls of one row each (which never cover a block), for every
cache and activation type, with and without the norm of the values, at starts and lengths on both sides of the blocks (16,
32 or 64 rows), and without touching the rows around it."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from __graft_entry__ import load_package  # noqa: E402

A = load_package().attn
DEV = "cuda:0"
TDT = {A.F32: torch.float32, A.F16: torch.float16, A.BF16: torch.bfloat16, A.I8: torch.int8}
D = 256


@pytest.mark.parametrize("kv,io", [(A.F32, A.F32), (A.F16, A.F16), (A.F16, A.F32), (A.BF16, A.BF16), (A.BF16, A.F32),
                                   (A.I8, A.F16), (A.I8, A.BF16), (A.I8, A.F32)])
@pytest.mark.parametrize("norm_v", [False, True])
def test_whole_blocks_equal_single_rows(kv, io, norm_v):
    hq, hkv, L = 4, 2, 260
    gen = torch.Generator(device=DEV).manual_seed(7)
    stream = torch.cuda.current_stream().cuda_stream
    with A.Attn(1, hq, hkv, D, L, 2, kv, io, stream=stream) as at:
        at.set_layer_transform(0, norm_q=True, norm_k=True, norm_v=norm_v, rope_inv_freq=np.linspace(1.0, 1e-3, D // 2))
        before = torch.randint(-100, 100, (L, hkv, D), generator=gen, device=DEV).to(TDT[kv])
        if kv == A.I8:
            s = torch.rand((2, hkv, D), generator=gen, device=DEV) * 0.01 + 0.02
            for seq in (0, 1):
                at.kv_set_scales(0, seq, s[0].contiguous(), s[1].contiguous())
        for pos, n in ((0, 1), (0, 16), (0, 64), (0, 63), (1, 64), (31, 33), (15, 17), (64, 65), (60, 200), (5, 250), (191, 69)):
            q, k, v = (torch.randn((n, h, D), generator=gen, device=DEV).to(TDT[io]) for h in (hq, hkv, hkv))
            read = []
            for seq, step in ((0, n), (1, 1)):
                at.kv_append(0, seq, 0, before, before)
                out = torch.empty_like(q)
                for i in range(0, n, step):
                    part = out[i:i + step]
                    at.pre_attention(0, seq, pos + i, q[i:i + step], k[i:i + step], v[i:i + step], part)
                ko, vo = torch.empty_like(before), torch.empty_like(before)
                at.kv_read(0, seq, 0, L, ko, vo)
                torch.cuda.synchronize()
                read.append((out, ko, vo))
            for got, want in zip(*read):
                assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), (kv, io, pos, n)
            rest = torch.ones(L, dtype=torch.bool, device=DEV)
            rest[pos:pos + n] = False
            if kv != A.BF16:  # (whole numbers up to 100 are exact in every type)
                assert torch.equal(read[0][2][rest], before[rest])
            if not norm_v and kv == io and kv != A.BF16:
                assert torch.equal(read[0][2][pos:pos + n], v)


@pytest.mark.parametrize("io", [A.F16, A.BF16, A.F32])
@pytest.mark.parametrize("pos,n", [(0, 512), (0, 640), (1, 575), (63, 577), (64, 511), (40, 700)])
def test_long_int8_calls_equal_short_ones(io, pos, n):
    # 16 rows a token: from 512 tokens on the whole blocks of an int8 call go through LDS; parts of 50 tokens never do
    hq, hkv, L = 8, 4, 760
    gen = torch.Generator(device=DEV).manual_seed(9)
    with A.Attn(1, hq, hkv, D, L, 2, A.I8, io, stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_layer_transform(0, norm_q=True, norm_k=True, norm_v=True, rope_inv_freq=np.linspace(1.0, 1e-3, D // 2))
        before = torch.randint(-100, 100, (L, hkv, D), generator=gen, device=DEV).to(torch.int8)
        q, k, v = (torch.randn((n, h, D), generator=gen, device=DEV).to(TDT[io]) for h in (hq, hkv, hkv))
        read = []
        for seq, step in ((0, n), (1, 50)):
            s = torch.linspace(0.01, 0.04, hkv * D, device=DEV).reshape(hkv, D)
            at.kv_set_scales(0, seq, s, s)
            at.kv_append(0, seq, 0, before, before)
            out = torch.empty_like(q)
            for i in range(0, n, step):
                e = min(n, i + step)
                at.pre_attention(0, seq, pos + i, q[i:e], k[i:e], v[i:e], out[i:e])
            ko, vo = torch.empty_like(before), torch.empty_like(before)
            at.kv_read(0, seq, 0, L, ko, vo)
            torch.cuda.synchronize()
            read.append((out, ko, vo))
        for got, want in zip(*read):
            assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        assert torch.equal(read[0][2][:pos], before[:pos]) and torch.equal(read[0][2][pos + n:], before[pos + n:])


@pytest.mark.parametrize("kv,io", [(A.I8, A.BF16), (A.I8, A.F32), (A.BF16, A.BF16)])
def test_ends_of_a_call_take_no_longer_than_its_rows(kv, io):
    # rows that fill no block have a wave each, so 63 rows take what 16 take (a launch of that size is latency); walked
    # by one workgroup a block they took 1.3 (bfloat16) to 3.3 (int8) times as long
    with A.Attn(1, 4, 1, D, 128, 1, kv, io, stream=torch.cuda.current_stream().cuda_stream) as at:
        at.set_layer_transform(0, norm_q=True, norm_k=True, rope_inv_freq=np.linspace(1.0, 1e-3, D // 2))
        at.set_timing(True)
        times = {}
        for n in (16, 63):
            q, k, v = (torch.randn((n, h, D), device=DEV).to(TDT[io]) for h in (4, 1, 1))
            out, ms = torch.empty_like(q), []
            for _ in range(40):
                for _ in range(3):
                    at.pre_attention(0, 0, 0, q, k, v, out)
                torch.cuda.synchronize()
                ms.append(at.last_kernel_ms())
            times[n] = sorted(ms)[20]
        assert times[63] < 1.25 * times[16], times
