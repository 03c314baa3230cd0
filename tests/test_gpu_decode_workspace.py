"""Decode calls that are recorded into HIP graphs beside other calls of the same handle: as the first call of the handle, and
with later calls of other lengths, batches and partition counts between the replays. A replay gives the bits of the same call
on a handle of its own, and a call that the handle has no room for is refused with a message that leaves the capture alive.
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

A = load_package().attn
DEV = "cuda:0"
TDT = {A.F32: torch.float32, A.F16: torch.float16, A.BF16: torch.bfloat16, A.I8: torch.int8}
D = 256


def rnd(seed, shape, dtype):
    x = torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)
    return (x * 40).round().clamp(-127, 127).to(torch.int8) if dtype == torch.int8 else x.to(dtype)


def handle(kv, io, hq, hkv, ctx, batch, stream):
    at = A.Attn(1, hq, hkv, D, ctx, batch, kv, io, stream=stream.cuda_stream)
    at.set_layer_transform(0, norm_q=True, norm_k=True, eps=1e-6,
                           rope_inv_freq=(10000.0 ** -(np.arange(0, D, 2) / D)).astype(np.float32))
    for b in range(batch):
        if kv == A.I8:
            s = torch.full((2, hkv, D), 0.025, device=DEV)
            at.kv_set_scales(0, b, s[0].contiguous(), s[1].contiguous())
        at.kv_append(0, b, 0, rnd(2 * b, (ctx, hkv, D), TDT[kv]), rnd(2 * b + 1, (ctx, hkv, D), TDT[kv]))
    return at


@pytest.mark.parametrize("step", [False, True])
@pytest.mark.parametrize("kv,io,recorded", [(A.F16, A.F16, 300), (A.BF16, A.F32, 512), (A.F32, A.F32, 200), (A.I8, A.BF16, 1100)])
def test_first_call_recorded_and_longer_calls_between_its_replays(kv, io, recorded, step):
    hq, hkv, ctx = 4, 1, 2200
    assert A.decode_plan(kv, hq, hkv, [0], [recorded])[0] > 1  # (there are partials to keep)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side), handle(kv, io, hq, hkv, ctx, 2, side) as own, handle(kv, io, hq, hkv, ctx, 2, side) as at:
        q, k, v = (rnd(90 + i, (2, h, D), TDT[io]) for i, h in enumerate((hq, hkv, hkv)))

        def call(h, n, out, batch=1):
            qs, ks, vs = q[:batch].contiguous(), k[:batch].contiguous(), v[:batch].contiguous()
            h.decode_step(0, [n] * batch, qs, ks, vs, out) if step else h.decode(0, [n] * batch, qs, out)

        want, out, other = torch.empty_like(q[:1]), torch.empty_like(q[:1]), torch.empty_like(q)
        call(own, recorded, want)
        side.synchronize()
        args = tuple(x[:1].contiguous() for x in (q, k, v))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            at.decode_step(0, [recorded], *args, out) if step else at.decode(0, [recorded], args[0], out)
        for n, batch in ((recorded + 1, 1), (recorded + 200, 1), (recorded + 600, 2), (2200, 1), (2200, 2), (64, 1)):
            if step and n < recorded:
                continue  # (would write a row that the recorded call sees)
            call(at, n, other[:batch], batch)
            held = torch.full((64 << 20,), 7, dtype=torch.uint8, device=DEV)  # (what is freed now is written over)
            out.fill_(float("nan"))
            g.replay()
            side.synchronize()
            assert torch.equal(out, want), (n, batch)
            assert bool((held == 7).all()), (n, batch)
            del held
        del g


def test_recorded_call_keeps_its_workspace_when_a_later_one_outgrows_it():
    hq, hkv, ctx, B = 8, 2, 2200, 64
    plan = [A.decode_plan(A.F16, hq, hkv, [0], [ctx] * B, s) for s in (16, 35)]
    assert plan[0][3] < plan[0][2] <= 2048 * (hq // hkv) < plan[1][2]  # behind the fixed room, in the reserve, beyond it
    side = torch.cuda.Stream()
    with torch.cuda.stream(side), handle(A.F16, A.F16, hq, hkv, ctx, B, side) as at:
        q = rnd(5, (B, hq, D), torch.float16)
        out, want, other = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
        g = torch.cuda.CUDAGraph()
        codes = []
        with torch.cuda.graph(g, stream=side):
            try:
                at.decode(0, [ctx] * B, q, out, num_splits=16)
            except A.AttnError as e:
                codes.append((e.code, "capture" in e.message))
            at.decode(0, [300] * 4, q[:4], out[:4])
        assert codes == [(A.FAILED_PRECONDITION, True)]
        at.decode(0, [300] * 4, q[:4], want[:4])
        out.fill_(float("nan"))
        g.replay()
        side.synchronize()
        assert torch.equal(out[:4], want[:4])
        del g
        at.decode(0, [ctx] * B, q, want, num_splits=16)
        side.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            at.decode(0, [ctx] * B, q, out, num_splits=16)
        for splits in (0, 35, 16):
            at.decode(0, [ctx] * B, q, other, num_splits=splits)
            held = torch.full((64 << 20,), 7, dtype=torch.uint8, device=DEV)
            out.fill_(float("nan"))
            g.replay()
            side.synchronize()
            assert torch.equal(out, want), splits
            assert bool((held == 7).all()), splits
            del held
        assert torch.equal(other, want)
        del g


def test_large_call_on_the_default_stream_while_another_stream_is_captured():
    hq, hkv, ctx, B = 8, 2, 1024, 40
    side = torch.cuda.Stream()
    with A.Attn(1, hq, hkv, D, ctx, B, A.F16, A.F16, stream=0) as at:
        for b in range(B):
            at.kv_append(0, b, 0, rnd(2 * b, (ctx, hkv, D), torch.float16), rnd(2 * b + 1, (ctx, hkv, D), torch.float16))
        q = rnd(5, (B, hq, D), torch.float16)
        want, out, x = torch.empty_like(q), torch.empty_like(q), torch.zeros(4, device=DEV)
        at.decode(0, [ctx] * B, q, want, num_splits=16)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side, capture_error_mode="thread_local"):
            x += 1
            at.decode(0, [ctx] * B, q, out, num_splits=16)  # (runs: the handle's stream is not the one captured)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        del g


def test_noalloc_calls_of_more_results_than_a_handle_has_room_for_are_ordered_across_streams():
    hq, hkv, ctx, B = 8, 2, 1024, 40
    assert A.decode_plan(A.F16, hq, hkv, [0], [ctx] * B, 16)[2] > A.decode_plan(A.F16, hq, hkv, [0], [ctx] * B, 16)[3]
    streams = [torch.cuda.Stream() for _ in range(2)]
    with handle(A.F16, A.F16, hq, hkv, ctx, B, streams[0]) as at0, handle(A.F16, A.F16, hq, hkv, ctx, B, streams[1]) as at1:
        torch.cuda.synchronize()
        qs = [rnd(7 + i, (B, hq, D), torch.float16) for i in range(2)]
        want = [torch.empty_like(q) for q in qs]
        got = [[torch.empty_like(q) for _ in range(10)] for q in qs]
        torch.cuda.synchronize()
        for at, q, o in zip((at0, at1), qs, want):
            at.decode(0, [ctx] * B, q, o, num_splits=16)
        torch.cuda.synchronize()
        for rep in range(10):
            for i, at in enumerate((at0, at1)):
                at.decode_noalloc(0, [ctx] * B, qs[i], got[i][rep], num_splits=16)
        torch.cuda.synchronize()
        for i in range(2):
            assert all(torch.equal(x, want[i]) for x in got[i])


def test_overlapping_replays_leave_later_calls_alone():
    """Replays of one handle that run at the same time spoil each other's results at most: what follows is right again."""
    hq, hkv, ctx = 4, 1, 1152
    side, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(side), handle(A.F32, A.F32, hq, hkv, ctx, 1, side) as at:
        qd, qp = rnd(1, (1, hq, D), torch.float32), rnd(2, (100, hq, D), torch.float32)
        assert A.decode_plan(A.F32, hq, hkv, [0], [ctx])[1] and A.decode_plan(A.F32, hq, hkv, [0], [700])[1]
        calls = [lambda o: at.decode(0, [ctx], qd, o), lambda o: at.decode(0, [700], qd, o), lambda o: at.prefill(0, 0, 1000, 100, qp, o)]
        want = [torch.empty_like(q) for q in (qd, qd, qp)]
        for call, o in zip(calls, want):
            call(o)
        graphs = []
        for call, q in zip(calls, (qd, qd, qp)):
            out = torch.empty_like(q)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side):
                call(out)
            graphs.append((g, out))
        side.synchronize()
        for rep in range(20):
            for i in range(30):
                with torch.cuda.stream(side if i % 2 else second):
                    graphs[(i + rep) % 3][0].replay()
            torch.cuda.synchronize()
            for (g, out), call, w in zip(graphs, calls, want):
                out.fill_(float("nan"))
                g.replay()
                side.synchronize()
                assert torch.equal(out, w), rep
                out.fill_(float("nan"))
                call(out)
                side.synchronize()
                assert torch.equal(out, w), rep
        del g, graphs
