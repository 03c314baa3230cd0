"""The value rows of the step before attention: blocks of the V plane that a call covers as a whole are assembled in LDS
and written as 16-byte chunks, the ends row by row. Both ways must leave the same bytes: a call over n rows against n
calls of one row each (which never cover a block), for every cache and activation type, with and without the norm of the
values, at starts and lengths on both sides of the blocks (16, 32 or 64 rows), and without touching the rows around it."""
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
