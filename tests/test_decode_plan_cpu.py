"""Partitions of decode calls and the room for their partial results, through mi355_attn_decode_plan_probe (host only): what
fits the room that a handle holds from its creation on needs no allocation, so a call can be recorded first thing and no
later call moves what a recorded one writes to."""
import ctypes
import os
import random
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from __graft_entry__ import load_package  # noqa: E402

A = load_package().attn
DTYPES = [A.F32, A.F16, A.BF16, A.I8]
HEADS = [(1, 1), (3, 1), (4, 1), (8, 1), (16, 1), (8, 2), (8, 4), (32, 2), (64, 4), (8, 8), (128, 8)]


@pytest.mark.parametrize("kv", DTYPES)
@pytest.mark.parametrize("hq,hkv", HEADS)
def test_contexts_of_up_to_512_tokens_need_no_workspace(kv, hq, hkv):
    for layers in (1, 2, 26, 64):
        for windows in ([0] * layers, [100] * layers, [0 if (l + 1) % 6 == 0 else 300 for l in range(layers)]):
            for batch in (1, 2, 3, 7, 16, 63, 64, 65, 128, 200, 300):
                for n in (1, 128, 129, 200, 256, 257, 300, 384, 500, 512):
                    splits, _, rows, fixed = A.decode_plan(kv, hq, hkv, windows, [n] * (batch - 1) + [max(1, n // 9)])
                    assert splits >= 1 and rows <= fixed, (layers, batch, n)


def test_launches_that_merge_themselves_need_no_workspace_and_no_rule_asks_for_more_than_the_reserve():
    rng = random.Random(5)
    merged = many = 0
    for _ in range(20000):
        kv, (hq, hkv) = rng.choice(DTYPES), rng.choice(HEADS)
        layers, batch = rng.choice((1, 1, 2, 6, 26, 65)), max(1, round(2 ** rng.uniform(0, 8)))
        n = max(1, round(2 ** rng.uniform(0, 17)))
        windows = [rng.choice((0, 512, n, 1)) for _ in range(layers)]
        lens = [n] * (batch - 1) + [max(1, round(n * rng.random()))]
        asked = rng.choice((0, 0, 0, 2, 16, 64, 256))
        splits, in_launch, rows, fixed = A.decode_plan(kv, hq, hkv, windows, lens, asked)
        assert rows == (layers * batch * hq * splits if splits > 1 else 0)
        assert splits <= (asked or 256)
        if in_launch:
            assert layers * batch * hkv * splits <= 256 and 1 < splits <= 64 and rows <= fixed
        if not asked:
            assert rows <= 2048 * (hq // hkv)
        merged += in_launch
        many += splits > 64
    assert merged > 1000 and many > 100


def test_partitions_that_hold_nothing_are_not_counted():
    assert A.decode_plan(A.F16, 8, 2, [0], [4096], 18)[0] == 16  # 18 of 228 tokens each: 16 of 256
    assert A.decode_plan(A.F16, 8, 2, [512], [4096], 18)[0] == 9  # 575 tokens from an aligned row on
    assert A.decode_plan(A.F16, 8, 2, [0], [1], 64)[0] == 1


@pytest.mark.parametrize("kv,hq,hkv,layers,batch,n,splits", [
    (A.F16, 8, 2, 30, 1, 4096, 16), (A.I8, 8, 2, 1, 32, 4096, 16), (A.F16, 8, 2, 1, 64, 2000, 8), (A.BF16, 4, 1, 1, 40, 3000, 24),
    (A.I8, 8, 2, 1, 32, 2490, 13), (A.BF16, 4, 1, 26, 1, 6000, 32), (A.I8, 4, 1, 1, 64, 6000, 16), (A.F16, 8, 2, 6, 8, 2000, 11)])
def test_large_launches_run_in_about_1024_workgroups(kv, hq, hkv, layers, batch, n, splits):
    """Half as many lose precision: the heaviest key of a wave is the one whose probability is exact in half."""
    assert A.decode_plan(kv, hq, hkv, [0] * layers, [n] * batch)[0] == splits


def test_arguments_are_checked():
    w = (ctypes.c_int32 * 1)(0)
    probe = A.lib().mi355_attn_decode_plan_probe
    assert probe(A.F16, 1, 1, 4, 1, w, 64, 64, 0, None, None, None) == 1
    for bad in ((-1, 1, 1, 4, 1, w, 64, 64, 0), (4, 1, 1, 4, 1, w, 64, 64, 0), (A.F16, 0, 1, 4, 1, w, 64, 64, 0),
                (A.F16, 1, 0, 4, 1, w, 64, 64, 0), (A.F16, 1, 1, 5, 2, w, 64, 64, 0), (A.F16, 1, 1, 17, 1, w, 64, 64, 0),
                (A.F16, 1, 1, 4, 0, w, 64, 64, 0), (A.F16, 1, 1, 4, 1, None, 64, 64, 0), (A.F16, 1, 1, 4, 1, w, 64, 65, 0),
                (A.F16, 1, 1, 4, 1, w, 64, 0, 0), (A.F16, 1, 1, 4, 1, w, 64, 64, -1), (A.F16, 1, 1, 4, 1, w, 64, 64, 257)):
        assert probe(*bad, None, None, None) < 0, bad
