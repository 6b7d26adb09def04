"""The choice of attention launches (attention_plan), without a device: block
tables over random window layouts, and what a launch capture may take."""

import random

import pytest

from kernrt_amd import AttnSpec, Window
from kernrt_amd.backends import attention_plan

SEQ = 16384
GEOMETRIES = [(15, 5, 64), (4, 4, 64), (16, 2, 64), (16, 8, 128), (12, 2, 128), (16, 1, 128), (16, 2, 32), (8, 2, 96)]


def spec(n_heads, n_kv, hs, seq=SEQ):
    return AttnSpec(n_heads, n_heads // n_kv, hs, n_kv * hs, seq)


def layout(w):
    return w.att_start, w.shared


def sequences(rng, total, longest):
    """Rows of ragged sequences, some with a shared prefix, packed one after another."""
    out, base = [], 0
    prefix = rng.choice((0, 0, rng.randint(1, 200)))
    base = prefix
    while len(out) < total:
        n = rng.randint(1, longest)
        start = rng.choice((0, rng.randint(0, 900)))
        out += [Window(base, base + start + i, (0, prefix)) for i in range(min(n, total - len(out)))]
        base += start + n
    return out if base < SEQ else out[:1]


@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_block_tables_keep_layouts_apart(geometry):
    rng, seen = random.Random(sum(geometry)), set()
    for _ in range(400):
        ws = sequences(rng, rng.choice((1, 2, 5, 30, 100, 400)), rng.choice((1, 3, 20, 90, 400)))
        kind, blocks = attention_plan(ws, spec(*geometry))
        seen.add((kind, bool(blocks)))
        if not blocks:
            continue
        assert kind in ("rows", "mx")
        assert blocks[0] == 0 and blocks[-1] == len(ws) and all(a < b for a, b in zip(blocks, blocks[1:]))
        longest = max(b - a for a, b in zip(blocks, blocks[1:]))
        for a, b in zip(blocks, blocks[1:]):
            assert len({layout(w) for w in ws[a:b]}) == 1
            # a block ends at its layout's end, or full
            assert b == len(ws) or layout(ws[b]) != layout(ws[a]) or b - a == longest
    assert geometry[2] == 96 or len(seen) > 1


@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_a_capture_takes_no_table_and_no_new_scratch_for_regular_rows(geometry):
    rng, sp = random.Random(sum(geometry)), spec(*geometry)
    for _ in range(200):
        ws = sequences(rng, rng.choice((1, 2, 30, 400)), rng.choice((1, 20, 400)))
        assert attention_plan(ws, sp, capturing=True)[1] == []
    for n, start in ((1, 0), (1, 3000), (2, 40), (9, 500), (30, 150), (200, 100), (500, 20), (40, 900)):
        kind, blocks = attention_plan([Window(0, start + i) for i in range(n)], sp, capturing=True)
        # heads of 32 have no blocks for windows past what the LDS holds
        assert kind != "split" or (n > 1 and start + n > 700 and geometry[2] == 32), (n, start, kind)
        assert n > 1 or kind == "general"


def test_large_scratch_is_not_taken_by_choice():
    # 200 rows of 16 heads: 12.8 MB of scores at 1024 slots, 1.6 GB at 131072
    ws = [Window(0, 100 + i) for i in range(200)]
    assert attention_plan(ws, spec(16, 8, 128, 1024))[0] == "split"
    assert attention_plan(ws, spec(16, 8, 128, 131072))[0] != "split"


def test_short_windows_of_128_wide_heads():
    def equal(n, length):  # sequences of one length: regular blocks
        return [Window(i // length * length, i) for i in range(n)]

    # one query head per KV head: blocks from 2048 (row, KV head) pairs on
    assert attention_plan(equal(256, 128), spec(8, 8, 128, 2048))[0] == "split"
    assert attention_plan(equal(264, 8), spec(8, 8, 128, 2048)) == ("rows", [])
    assert attention_plan(equal(2000, 40), spec(16, 8, 128, 2048))[0] == "split"
    # more rows than a grid dimension has workgroups
    assert attention_plan([Window(0, 0)] * 65536, spec(2, 1, 128, 8))[0] == "rows"


def test_refused_windows():
    for w in (Window(5, 4), Window(0, SEQ), Window(0, 1, (3, 2)), Window(0, 1, (0, SEQ + 1)), Window(0, SEQ - 1, (0, 1))):
        with pytest.raises(ValueError):
            attention_plan([w], spec(4, 4, 64))
