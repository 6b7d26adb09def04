"""A recorded launch sequence keeps the memory and the row lists it was recorded
with: eager calls between its replays grow every workspace, rotation table and
list of the context, and each replay still gives the eager result."""

import numpy as np
import pytest

import kernrt_amd as K
import oracle as O
from helpers import assert_bits_equal, product_matrix

pytestmark = pytest.mark.gpu

DIM, HEADS, KV_HEADS, HS, SEQ = 128, 6, 2, 64, 3100


def rows_of(lens, start=0):
    out, base = [], 0
    for n in lens:
        out += [(base, base + start + i, 0, 0) for i in range(n)]
        base += start + n
    return out


# one row and a few at long windows (per-row launches), one sequence's rows and
# ragged sequences (row blocks), many rows at long windows (matrix core)
@pytest.mark.parametrize("windows", [rows_of([1], 300), rows_of([5], 290), rows_of([70]), rows_of([70, 33, 48, 1]),
                                     rows_of([300, 200, 160], 780)[300:]])
def test_replays_between_eager_calls(windows):
    rng = np.random.default_rng(len(windows))
    n, q_dim, kv_dim = len(windows), HEADS * HS, KV_HEADS * HS
    hip = K.open("hip")
    mats = {name: hip.upload_matrix(product_matrix(O.Matrix(rng.normal(0, 0.02, size=(w, DIM)).astype(np.float32), "q8_0")))
            for name, w in (("q", q_dim), ("k", kv_dim), ("v", kv_dim))}
    emb = hip.upload_matrix(product_matrix(O.Matrix(rng.normal(size=(8, DIM)).astype(np.float32), "q8_0")))
    hip.bind_handles(emb, 0xFFFFFFFF, [mats])
    hip.prepare(None, K.KvSpec(1, kv_dim, SEQ))
    fill = rng.normal(size=SEQ * kv_dim).astype(np.float32)
    hip.kv_upload(0, 0, fill)
    hip.kv_upload(1, 0, fill)
    x = hip.upload(rng.normal(size=n * DIM).astype(np.float32))
    q, k, v, out = (hip.alloc(n * w) for w in (q_dim, kv_dim, kv_dim, q_dim))
    att = hip.alloc(n * HEADS * SEQ)
    spec, rope = K.AttnSpec(HEADS, HEADS // KV_HEADS, HS, kv_dim, SEQ), K.RopeSpec(HS, 10_000.0, False)
    slots = [s for _, s, _, _ in windows]
    wins = [K.Window(a, s, (c, d)) for a, s, c, d in windows]

    def sequence():
        hip.project_qkv(0, x, q, k, v, n)
        hip.rope(q, k, q_dim, kv_dim, n, slots, rope)
        hip.kv_write(0, np.array(slots, np.uint64), k, v, n)
        hip.attention(q, out, att, 0, wins, spec)

    sequence()
    want = hip.read(out, n * q_dim)
    hip.capture_begin()
    sequence()
    hip.capture_end()
    zeros = np.zeros(n * q_dim, np.float32)
    for i in range(4):
        # more rows than before, at longer windows and positions
        m = n + 30 * (i + 1)
        bx, bq = (hip.upload(rng.normal(size=m * w).astype(np.float32)) for w in (DIM, q_dim))
        bk, bo, ba = hip.alloc(m * kv_dim), hip.alloc(m * q_dim), hip.alloc(m * HEADS * SEQ)
        hip.project_qkv(0, bx, bq, bk, bk, m)
        hip.rope(bq, bk, q_dim, kv_dim, m, [SEQ + 4000 * i + r for r in range(m)], rope)
        hip.attention(bq, bo, ba, 0, [K.Window(r // 50, 900 + 300 * i + r, (0, 0)) for r in range(m)], spec)
        noise = hip.upload(np.full(1 << 20, -1e30, np.float32))  # into what may have been freed
        hip.copy(hip.upload(zeros), 0, out, 0, n * q_dim)
        hip.replay(2)
        assert_bits_equal(hip.read(out, n * q_dim), want, f"replay {i}")
        hip.read(noise, 1 << 20)
    # the next capture starts anew, after one eager pass
    sequence()
    hip.capture_begin()
    sequence()
    hip.capture_end()
    hip.replay(1)
    assert_bits_equal(hip.read(out, n * q_dim), want, "a second capture")
    hip.close()


@pytest.mark.parametrize("warm,wins", [
    ([(0, 100 + i, 0, 0) for i in range(600)], rows_of([9], 400)),      # one sequence's rows: blocks
    ([(0, 100 + i, 0, 0) for i in range(600)], rows_of([1], 400)),
    ([(0, 20 + i, 0, 0) for i in range(40)], rows_of([20, 11, 9], 60)),  # per-row launches without their scratch
])
def test_capture_of_windows_that_no_call_had_before(warm, wins):
    # a capture cannot allocate: it takes the launches that the memory of the
    # eager calls before it serves
    rng = np.random.default_rng(len(wins))
    hip, kv_dim, q_dim, seq = K.open("hip"), KV_HEADS * HS, HEADS * HS, 16384
    emb = hip.upload_matrix(product_matrix(O.Matrix(np.ones((8, 32), np.float32), "q8_0")))
    hip.bind_handles(emb, 0xFFFFFFFF, [{}])
    hip.prepare(None, K.KvSpec(1, kv_dim, seq))
    for which in (0, 1):
        hip.kv_upload(which, 0, rng.normal(size=1200 * kv_dim).astype(np.float32))
    n = max(len(warm), len(wins))
    q = hip.upload(rng.normal(size=n * q_dim).astype(np.float32))
    out, att = hip.alloc(n * q_dim), hip.alloc(n * HEADS * seq)
    spec = K.AttnSpec(HEADS, HEADS // KV_HEADS, HS, kv_dim, seq)
    wins, warm = ([K.Window(a, s, (c, d)) for a, s, c, d in w] for w in (wins, warm))
    hip.attention(q, out, att, 0, warm, spec)
    epoch = hip.dbg_epoch()
    hip.capture_begin()
    hip.attention(q, out, att, 0, wins, spec)
    assert hip.dbg_epoch() == epoch
    hip.capture_end()
    hip.replay(1)
    got = hip.read(out, len(wins) * q_dim)
    hip.attention(q, out, att, 0, wins, spec)
    assert_bits_equal(got, hip.read(out, len(wins) * q_dim), "eager")
    hip.replay(2)
    assert_bits_equal(got, hip.read(out, len(wins) * q_dim), "again")
    hip.close()
