"""The backend's projections as one launch: the workspace they leave behind,
outputs that repeat or are the input, and rows whose quantization runs inside
the launch; the final norm over picked rows. Bit for bit against the oracle."""

import numpy as np
import pytest

import kernrt_amd as K
import oracle as O
from helpers import assert_bits_equal, gaussian_weights, gpu_model, product_matrix

pytestmark = pytest.mark.gpu


# 2048 is the widest row that one launch quantizes, 2080 the first that takes two
@pytest.mark.parametrize("storage", ["q8_0", "q8_0x4"])
@pytest.mark.parametrize("dim,rows", [(64, 1), (96, 1), (2048, 1), (2080, 1), (96, 3), (96, 9)])
def test_projections_and_their_workspace(storage, dim, rows):
    rng = np.random.default_rng(dim + rows)
    shapes = {"q": 128, "k": 64, "v": 64, "gate": 96, "up": 96}
    ms = {n: O.Matrix(rng.normal(0, 0.02, size=(w, dim)).astype(np.float32), storage) for n, w in shapes.items()}
    hip = K.open("hip")
    h = {n: hip.upload_matrix(product_matrix(m)) for n, m in ms.items()}
    emb = hip.upload_matrix(product_matrix(O.Matrix(rng.normal(size=(8, dim)).astype(np.float32), storage)))
    hip.bind_handles(emb, 0xFFFFFFFF, [h])
    hip.prepare(None, K.KvSpec(1, 64, 16))
    x = rng.normal(size=(rows, dim)).astype(np.float32)
    want = {n: m.project_cpu(x).ravel() for n, m in ms.items()}
    xb = hip.upload(x)
    y = {n: hip.alloc(rows * w) for n, w in shapes.items()}
    hip.project_qkv(0, xb, y["q"], y["k"], y["v"], rows)
    hip.project_gate_up(0, xb, y["gate"], y["up"], rows)
    for n, w in shapes.items():
        assert_bits_equal(hip.read(y[n], rows * w), want[n], n)
    # the quantized rows stay in the workspace
    other = hip.upload(rng.normal(size=(rows, dim)).astype(np.float32))
    hip.quantize_rows(other, rows, dim)
    hip.project(0, "v", xb, y["v"], rows)
    hip.matmul_quantized(h["q"], y["q"], rows)
    assert_bits_equal(hip.read(y["q"], rows * 128), want["q"], "from the workspace")
    # one buffer for two outputs: the later one stays
    hip.project_gate_up(0, xb, y["gate"], y["gate"], rows)
    assert_bits_equal(hip.read(y["gate"], rows * 96), want["up"], "repeated output")
    # an output over the input
    big = hip.alloc(rows * max(dim, 128))
    hip.copy(xb, 0, big, 0, rows * dim)
    hip.project(0, "q", big, big, rows)
    assert_bits_equal(hip.read(big, rows * 128), want["q"], "over the input")
    hip.close()


# a single row over many outputs: 2048 x 12288 in all is the first that is
# quantized before the launch (as gate and up of 6144), 12256 the last inside it
@pytest.mark.parametrize("storage", ["q8_0", "q8_0x4"])
@pytest.mark.parametrize("gate,up", [(6144, 6112), (6144, 6144)])
def test_one_row_over_many_outputs(storage, gate, up):
    dim = 2048
    rng = np.random.default_rng(gate + up)
    small = rng.normal(0, 0.02, size=(64, dim)).astype(np.float32)
    # every 64 rows of the oracle's matrix again: its projection repeats too
    ms = O.Matrix(small, storage)
    big = {n: O.Matrix(np.resize(small, (w, dim)), storage) for n, w in (("gate", gate), ("up", up))}
    hip = K.open("hip")
    h = {n: hip.upload_matrix(product_matrix(m)) for n, m in big.items()}
    emb = hip.upload_matrix(product_matrix(ms))
    hip.bind_handles(emb, 0xFFFFFFFF, [h])
    hip.prepare(None, K.KvSpec(1, 64, 16))
    x = rng.normal(size=(1, dim)).astype(np.float32)
    want = ms.project_cpu(x).ravel()
    y = {"gate": hip.alloc(gate), "up": hip.alloc(up)}
    hip.project_gate_up(0, hip.upload(x), y["gate"], y["up"], 1)
    for n, w in (("gate", gate), ("up", up)):
        assert_bits_equal(hip.read(y[n], w), np.resize(want, w), n)
    z = hip.alloc(gate)
    hip.matmul_quantized(h["gate"], z, 1)
    assert_bits_equal(hip.read(z, gate), np.resize(want, gate), "from the workspace")
    hip.close()


@pytest.mark.parametrize("storage,lens", [("q8_0", [3, 0, 9, 1, 0]), ("q8_0x4", [1, 0, 40]), ("q8_0", [0, 0]),
                                          ("q8_0", [70, 60])])
def test_hidden_rows_with_empty_sequences(storage, lens):
    # [70, 60]: dim 1024 leaves the last down projection as four planes
    dim = 1024 if lens == [70, 60] else 128
    c = O.Config(dim=dim, hidden_dim=256, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=64, seq_len=160,
                 rms_eps=1e-5, rope_theta=10_000.0, rope_interleaved=False, head_dim=32)
    ow = gaussian_weights(c, storage, seed=sum(lens) + dim)
    gpu, cpu = gpu_model(c, ow), O.Model(c, ow, "cpu")
    seqs = [[(7 * i + 3 * s) % 64 for i in range(n)] for s, n in enumerate(lens)]
    got, want = gpu.prefill_multi(seqs), cpu.prefill_multi(seqs)
    assert_bits_equal(got, want, "multi")
    assert_bits_equal(gpu.prefill_shared([5, 6, 7], seqs), cpu.prefill_shared([5, 6, 7], seqs), "shared")
