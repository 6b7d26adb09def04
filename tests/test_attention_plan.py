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
    # 100 rows of 16 heads: 6.6 MB of scores at 1024 slots, 0.84 GB at 131072
    ws = [Window(0, 100 + i) for i in range(100)]
    assert attention_plan(ws, spec(16, 8, 128, 1024))[0] == "split"
    assert attention_plan(ws, spec(16, 8, 128, 131072))[0] == "mx"
    # rows without blocks have nothing else
    ws = [Window(50 * i, 50 * i + 20) for i in range(100)]
    assert attention_plan(ws, spec(16, 8, 128, 131072))[0] == "split"


def test_short_windows_of_128_wide_heads():
    def equal(n, length):  # sequences of one length: regular blocks
        return [Window(i // length * length, i) for i in range(n)]

    # one query head per KV head: blocks from 2048 (row, KV head) pairs on
    assert attention_plan(equal(256, 128), spec(8, 8, 128, 2048))[0] == "split"
    assert attention_plan(equal(264, 8), spec(8, 8, 128, 2048)) == ("rows", [])
    assert attention_plan(equal(2000, 40), spec(16, 8, 128, 2048))[0] == "split"
    # more rows than a grid dimension has workgroups
    assert attention_plan([Window(0, 0)] * 65536, spec(2, 1, 128, 8))[0] == "rows"


# both sides of the lines at which blocks overtake the per-row launches: rows of
# one sequence ending at `end`
@pytest.mark.parametrize("geometry,n,end,kind", [
    ((16, 8, 128), 128, 1536, "split"), ((16, 8, 128), 129, 1536, "mx"), ((16, 8, 128), 96, 1537, "split"),
    ((16, 8, 128), 97, 1537, "mx"), ((12, 4, 128), 160, 500, "split"), ((12, 4, 128), 161, 500, "mx"),
    ((16, 2, 128), 256, 900, "split"), ((16, 2, 128), 257, 900, "mx"), ((16, 4, 64), 320, 1000, "split"),
    ((16, 4, 64), 321, 1000, "mx"), ((15, 5, 64), 192, 3000, "split"), ((15, 5, 64), 193, 3000, "mx"),
    ((15, 5, 64), 100, 193, "split"), ((15, 5, 64), 100, 192, "rows"), ((15, 5, 64), 103, 400, "rows"),
    ((16, 16, 64), 20, 199, "split"), ((16, 16, 64), 21, 199, "rows"), ((16, 16, 64), 32, 200, "split"),
    ((16, 2, 64), 100, 513, "split"), ((16, 2, 64), 100, 512, "rows"), ((16, 2, 64), 129, 600, "rows"),
    ((8, 1, 128), 20, 100, "rows"), ((32, 8, 128), 140, 150, "split"), ((16, 2, 32), 64, 100, "rows"),
    ((15, 5, 64), 1, 255, "general"), ((15, 5, 64), 1, 256, "split"), ((16, 8, 128), 1, 255, "general"),
    ((16, 2, 32), 1, 511, "general"), ((16, 2, 32), 1, 3072, "split"), ((16, 2, 32), 1, 3073, "general"),
    ((16, 2, 64), 1, 3073, "general"), ((16, 2, 128), 1, 3073, "split"),
])
def test_lines_between_rows_and_blocks(geometry, n, end, kind):
    ws = [Window(0, end - n + i) for i in range(n)]
    assert attention_plan(ws, spec(*geometry, 4096)) == (kind, [])


# sequences of their own lengths: tables where they are shorter than the per-row launches
@pytest.mark.parametrize("geometry,lens,shared,kind", [
    ((15, 5, 64), [10, 11, 9, 13, 7], 0, "split"), ((15, 5, 64), [50, 51, 52, 53, 7], 0, "rows"),
    ((16, 8, 32), [50, 51, 52, 53, 57] * 3, 0, "split"), ((16, 8, 128), [50, 51, 52, 53, 7], 0, "split"),
    ((15, 5, 64), [3, 4, 5, 2] * 50, 1200, "split"), ((15, 5, 64), [103, 104, 105, 201], 1200, "mx"),
    ((16, 8, 128), [103, 104, 105], 200, "mx"), ((16, 8, 128), [83, 84, 85], 200, "split"),
    ((12, 2, 128), [101, 102, 103, 50], 150, "mx"), ((12, 2, 128), [101, 102, 103], 150, "general"),
    ((12, 2, 64), [101, 102, 103] * 3, 0, "rows"), ((12, 2, 64), [101, 102, 103] * 2, 0, "general"),
    ((12, 1, 32), [101, 102, 103] * 9, 0, "general"),
])
def test_lines_for_ragged_sequences(geometry, lens, shared, kind):
    ws, base = [], shared
    for n in lens:
        ws += [Window(base, base + i, (0, shared)) for i in range(n)]
        base += n
    got, blocks = attention_plan(ws, spec(*geometry, 4096))
    assert got == kind and bool(blocks) == (kind in ("rows", "mx"))


def test_refused_windows():
    for w in (Window(5, 4), Window(0, SEQ), Window(0, 1, (3, 2)), Window(0, 1, (0, SEQ + 1)), Window(0, SEQ - 1, (0, 1))):
        with pytest.raises(ValueError):
            attention_plan([w], spec(4, 4, 64))
