"""Which kernel a prefill call takes by rule, through mi355_attn_prefill_route_probe (host only): calls whose times on the
short kernel and on the tiled kernels were measured (MI355X, us) and lie clearly apart go to the faster one, calls the
short kernel cannot take go elsewhere, and the split of long tiles is what its launches are tested with."""
import ctypes
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from __graft_entry__ import load_package  # noqa: E402

A = load_package().attn


def windows(layers, local):
    return [local if (l + 1) % 6 else 0 for l in range(layers)] if layers > 1 else [local]


# cache, query heads, KV heads, layers, window of the local layers, start, rows, tiled us, short us
MEASURED = [
    # one XCD has the global layer's tiles to itself (a number of units that shares a factor with eight)
    (A.BF16, 4, 1, 8, 512, 1059, 1686, 92.0, 203.6),
    (A.F16, 16, 2, 8, 512, 4227, 265, 172.0, 298.6),
    (A.F16, 4, 1, 8, 512, 1556, 639, 61.4, 79.4),
    # ... or one engine of an XCD (a factor of 32)
    (A.BF16, 8, 2, 16, 1024, 3058, 108, 62.8, 102.6),
    (A.F16, 8, 4, 12, 512, 4822, 107, 67.8, 100.3),
    # more planes than an L2 holds, walked by few tiles each
    (A.F16, 2, 2, 26, 512, 79, 589, 33.6, 49.8),
    (A.BF16, 16, 2, 26, 0, 2068, 16, 51.1, 70.3),
    (A.F16, 2, 2, 26, 0, 3559, 57, 46.0, 56.6),
    # a few workgroups more than compute units, and more than two rounds of them
    (A.F16, 16, 2, 2, 0, 4139, 150, 46.8, 65.7),
    (A.I8, 8, 2, 1, 0, 3072, 1100, 65.9, 81.1),
    (A.I8, 8, 2, 1, 0, 3072, 600, 47.4, 56.1),
    # the tiled kernels' own ground
    (A.BF16, 8, 2, 26, 0, 1686, 78, 67.9, 144.3),
    (A.F16, 8, 4, 26, 512, 718, 196, 59.2, 140.4),
    (A.F16, 4, 1, 1, 0, 3000, 2048, 58.5, 76.6),
    (A.F16, 8, 2, 1, 0, 6157, 2047, 146.4, 239.0),
    # short calls, whole prompts of one layer, a chat's next turn
    (A.BF16, 4, 1, 1, 0, 0, 64, 9.9, 5.1),
    (A.BF16, 4, 1, 1, 0, 0, 1024, 25.7, 13.6),
    (A.BF16, 4, 1, 1, 512, 0, 1024, 24.9, 10.0),
    (A.F16, 4, 1, 1, 0, 1207, 17, 19.4, 14.4),
    (A.BF16, 4, 1, 1, 0, 1943, 281, 27.6, 20.9),
    (A.BF16, 3, 1, 1, 0, 1492, 203, 24.2, 17.4),
    (A.BF16, 4, 1, 1, 0, 0, 2048, 35.2, 28.6),
    (A.F16, 16, 2, 1, 0, 0, 1321, 57.4, 43.2),
    (A.F16, 8, 2, 2, 0, 167, 1247, 61.2, 45.7),
    (A.I8, 8, 2, 1, 0, 0, 300, 24.0, 10.0),
    (A.I8, 8, 2, 1, 0, 3072, 256, 47.0, 31.0),
    (A.I8, 4, 1, 1, 0, 3072, 1024, 42.7, 37.0),
    (A.I8, 8, 4, 2, 512, 31, 762, 37.3, 24.1),
    # few tiles behind a long context, in parts
    (A.F16, 8, 1, 1, 0, 6843, 26, 38.4, 17.2),
]


@pytest.mark.parametrize("kv,hq,hkv,layers,local,start,n,tiled,short", MEASURED)
def test_measured_calls_take_the_faster_kernel(kv, hq, hkv, layers, local, start, n, tiled, short):
    route, _ = A.prefill_route(kv, hq, hkv, windows(layers, local), start, n)
    assert (route == A.ROUTE_SHORT) == (short < tiled), (route, tiled, short)


def test_routes_at_their_limits():
    assert A.prefill_route(A.F32, 4, 1, [0], 0, 300)[0] == A.ROUTE_SHORT  # a float32 cache has no tiled kernel
    assert A.prefill_route(A.F32, 4, 1, [0] * 65, 0, 300)[0] == A.ROUTE_ROWWISE  # more layers than the argument block holds
    assert A.prefill_route(A.F32, 4, 1, [0], 0, 65536)[0] == A.ROUTE_ROWWISE
    assert A.prefill_route(A.F16, 4, 1, [0] * 65, 0, 16)[0] in (A.ROUTE_TILED32, A.ROUTE_PLANNED16)
    assert A.prefill_route(A.I8, 8, 2, [0], 100, 15)[0] == A.ROUTE_ROWWISE  # under prefill_i8_min_rows
    assert A.prefill_route(A.I8, 8, 2, [0], 100, 16)[0] == A.ROUTE_SHORT
    # 26 layers of a 1,024-token prompt in one call: the planned kernel; the late chunk of a long document: parts, no plan
    assert A.prefill_route(A.BF16, 4, 1, windows(26, 512), 0, 1024) == (A.ROUTE_PLANNED16, 1)
    assert A.prefill_route(A.F16, 8, 2, [0], 6157, 2047) == (A.ROUTE_DIRECT16, 4)
    assert A.prefill_route(A.I8, 8, 2, [0], 3072, 1024) == (A.ROUTE_TILED32, 4)


def test_parts_of_short_calls():
    """Few tiles of many key blocks are cut over the keys, into at most eight parts and 256 workgroups."""
    for kv, hq, hkv, start, n, parts in ((A.F16, 8, 1, 6843, 26, 8), (A.F32, 4, 1, 0, 300, 3), (A.F32, 4, 1, 1000, 100, 8), (A.I8, 8, 2, 3000, 64, 8),
                                         (A.F32, 4, 1, 1500, 512, 2), (A.F32, 4, 1, 1500, 513, 1), (A.F32, 4, 1, 0, 64, 1)):
        assert A.prefill_route(kv, hq, hkv, [0], start, n) == (A.ROUTE_SHORT, parts), (kv, start, n)


def test_arguments_are_checked():
    w = (ctypes.c_int32 * 1)(0)
    probe = A.lib().mi355_attn_prefill_route_probe
    assert probe(A.F16, 1, 64, 0, 4, 1, w, 256, None) == A.ROUTE_SHORT
    for bad in ((-1, 1, 64, 0, 4, 1, w, 256), (4, 1, 64, 0, 4, 1, w, 256), (A.F16, 0, 64, 0, 4, 1, w, 256), (A.F16, 1, 0, 0, 4, 1, w, 256),
                (A.F16, 1, 64, -1, 4, 1, w, 256), (A.F16, 1, 64, 0, 5, 2, w, 256), (A.F16, 1, 64, 0, 4, 0, w, 256),
                (A.F16, 1, 64, 0, 17, 1, w, 256), (A.F16, 1, 64, 0, 4, 1, None, 256), (A.F16, 1, 64, 0, 4, 1, w, 0)):
        assert probe(*bad, None) < 0, bad
