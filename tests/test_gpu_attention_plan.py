"""The choice of attention launches (attention_plan) on both sides of its lines:
every window layout gives the oracle's outputs and probabilities bit for bit,
whichever launches take it."""

import numpy as np
import pytest

import kernrt_amd as K
import oracle as O
from helpers import product_matrix
from test_gpu_ops import _attention_case

pytestmark = pytest.mark.gpu


def causal(n, start=0, base=0, shared=0):
    return [(base, base + start + i, 0, shared) for i in range(n)]


def ragged(lens, shared=0):
    out, base = [], shared
    for n in lens:
        out += causal(n, 0, base, shared)
        base += n
    return out


# one row: below and at the split's first window, 4- and 16-dim slices (n_kv hs
# / 4 workgroups up to and past 256), passes of the V slice
@pytest.mark.parametrize("n_heads,n_kv,hs,count", [
    (15, 5, 64, 255), (15, 5, 64, 256), (32, 32, 64, 700), (16, 8, 128, 3), (16, 8, 128, 300), (32, 16, 128, 2900),
    (4, 2, 32, 300), (4, 2, 32, 512), (16, 2, 64, 3072), (16, 2, 64, 3073),
])
def test_one_row(n_heads, n_kv, hs, count):
    kinds = _attention_case(count + 5, n_heads, n_kv, hs, [(2, count + 1, 0, 0)], count)
    general = count < (512 if hs == 32 else 256) or count == 3073
    assert kinds == (["general"] if general else ["split", "general"])


# few rows at long windows: slices of 4 and 16 dims, a workgroup per (row, KV
# head), and blocks beyond the number of pairs that the per-row launches take
@pytest.mark.parametrize("n_heads,n_kv,hs,n,start", [
    (15, 5, 64, 3, 300), (15, 5, 64, 12, 290), (15, 5, 64, 13, 290), (6, 2, 64, 256, 70), (6, 2, 64, 257, 70),
    (4, 4, 64, 30, 800), (16, 8, 128, 2, 150), (16, 8, 128, 30, 150), (16, 8, 128, 225, 3), (8, 8, 32, 65, 60),
    (16, 1, 128, 9, 130), (12, 2, 128, 9, 130),
])
def test_rows_of_one_sequence(n_heads, n_kv, hs, n, start):
    kinds = _attention_case(start + n + 3, n_heads, n_kv, hs, causal(n, start), n + start)
    by_blocks = (n, start) in ((257, 70), (225, 3), (65, 60)) or n_heads // n_kv in (6, 16)
    assert kinds[0] in (("rows", "mx") if by_blocks else ("split",)) and kinds[-1] in ("rows", "mx")


# sequences whose lengths leave blocks of every size: block tables for
# k_attn_rows and for the matrix core (1, 2, 4 and 8 query heads per workgroup),
# with and without a shared prefix; too ragged for blocks; a row alone at the end
@pytest.mark.parametrize("n_heads,n_kv,hs,lens,shared,kind", [
    (15, 5, 64, [1, 5, 6, 37, 64, 3, 2, 1], 0, "rows"), (15, 5, 64, [70, 33, 48], 9, "rows"),
    (4, 4, 64, [7, 50, 1, 9], 20, "split"), (6, 2, 64, [1, 1, 2, 1, 1], 0, "split"),
    (16, 8, 128, [100, 30, 66, 1], 0, "split"), (16, 8, 128, [180, 17, 1, 15], 12, "split"),
    (16, 8, 128, [180, 17, 1, 70], 12, "mx"), (4, 2, 64, [790, 495, 1], 0, "mx"), (8, 4, 32, [40, 3, 25], 7, "split"),
    (12, 1, 32, [40, 3, 25], 7, "general"), (8, 8, 128, [90, 60, 40, 30, 44], 0, "split"),
    (12, 2, 64, [99, 101, 98, 97, 103, 102, 95], 3, "rows"), (12, 2, 128, [190, 150, 3], 5, "mx"), (4, 4, 64, [790, 30, 1], 9, "mx"), (16, 4, 128, [300, 120, 100], 4, "mx"),
    (16, 2, 64, [790, 30, 1], 0, "mx"),
])
def test_rows_of_ragged_sequences(n_heads, n_kv, hs, lens, shared, kind):
    wins = ragged(lens, shared)
    kinds = _attention_case(shared + sum(lens) + 2, n_heads, n_kv, hs, wins, sum(lens) + shared)
    spec = K.AttnSpec(n_heads, n_heads // n_kv, hs, n_kv * hs, shared + sum(lens) + 2)
    _, blocks = K.backends.attention_plan([K.Window(a, s, (x, y)) for a, s, x, y in wins], spec)
    assert kinds[0] == kind and bool(blocks) == (kind in ("rows", "mx"))


# a batch of sequences: a workgroup per (row, KV head), slices of 4 and of 16 dims,
# on both sides of their shortest window; eight query heads without slices of 16
@pytest.mark.parametrize("n_heads,n_kv,hs,n,count", [
    (15, 5, 64, 2, 255), (15, 5, 64, 2, 256), (15, 5, 64, 6, 256), (15, 5, 64, 13, 256), (8, 8, 128, 2, 127),
    (8, 8, 128, 2, 128), (16, 2, 64, 8, 576), (16, 2, 64, 9, 576), (16, 8, 32, 3, 200), (8, 4, 32, 32, 200),
])
def test_independent_rows(n_heads, n_kv, hs, n, count):
    windows = [(count * i, count * i + count - 1 - 3 * (i % 4), 0, 0) for i in range(n)]
    assert "split" in _attention_case(count * n + 1, n_heads, n_kv, hs, windows, n + count)


@pytest.mark.parametrize("n,hs", [(1, 64), (1, 128), (6, 64)])
def test_growing_windows_leave_the_scratch_in_place(n, hs):
    # a conversation's window grows past 512, 1024, 1536 positions: what the
    # first call laid out (and a recorded decode step holds) stays
    hip, seq = K.open("hip"), 2048
    emb = hip.upload_matrix(product_matrix(O.Matrix(np.ones((8, 32), np.float32), "q8_0")))
    hip.bind_handles(emb, 0xFFFFFFFF, [{}])
    hip.prepare(None, K.KvSpec(1, 2 * hs, seq))
    q, out, att = hip.alloc(n * 4 * hs), hip.alloc(n * 4 * hs), hip.alloc(n * 4 * seq)
    spec = K.AttnSpec(4, 2, hs, 2 * hs, seq)
    epochs = []
    for end in (20, 100, 300, 512, 513, 900, 1025, 1600, 2040):
        hip.attention(q, out, att, 0, [K.Window(0, end + r, (0, 0)) for r in range(n)], spec)
        epochs.append(hip.dbg_epoch())
    assert epochs == epochs[:1] * len(epochs)
    hip.close()
