"""The per-wave GEMM (gemm_direct.hip) and the Q8_0x4 tile forms (gemm.hip) at
the edges of their tiles and of the dispatch, bit for bit against the oracle's
cpu backend."""

import numpy as np
import pytest

import kernrt_amd as K
import oracle as O
from helpers import assert_bits_equal, gaussian_weights, gpu_model, product_matrix

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    h = K.open("hip")
    yield h
    h.close()


def check_matmul(hip, storage, n, k, rows, scale=1.0):
    rng = np.random.default_rng(n + 3 * k + rows)
    m = O.Matrix(rng.normal(0, 0.02 * scale, size=(n, k)).astype(np.float32), storage)
    x = (rng.normal(size=(rows, k)) * scale).astype(np.float32)
    mat = hip.upload_matrix(product_matrix(m))
    y = hip.alloc(rows * n)
    hip.matmul(mat, hip.upload(x), y, rows)
    assert_bits_equal(hip.read(y, rows * n), m.project_cpu(x).ravel(), f"{storage} {n}x{k} rows={rows}")
    hip.free_matrix(mat)


# 1 to 4 blocks short of a group of four, fewer groups than the loads kept
# ahead, one, two and many rounds of them; 16-row and 16-column remainders
@pytest.mark.parametrize("storage", ["q8_0", "q8_0x4"])
@pytest.mark.parametrize("k", [32, 96, 128, 416, 544, 576, 2048])
@pytest.mark.parametrize("rows,n", [(5, 3204), (8, 4), (15, 20), (16, 16), (17, 36), (33, 132)])
def test_direct_gemm_edges(hip, storage, k, rows, n):
    check_matmul(hip, storage, n, k, rows)


# both sides of the dispatch: 1408 units of 16x16 (64x64 tiles above), 512 tiles
# of 64x64 (128x128 above, 64x64 again where those take a second round) for
# Q8_0x4; 512 units for Q8_0; five to seven rows of a narrow output (GEMV below
# an eighth of the inner dimension)
@pytest.mark.parametrize("storage,n,k,rows", [
    ("q8_0x4", 4096, 160, 80), ("q8_0x4", 4096, 160, 96), ("q8_0x4", 4100, 96, 130),
    ("q8_0x4", 4096, 96, 512), ("q8_0x4", 4096, 96, 513), ("q8_0x4", 4096, 96, 640), ("q8_0x4", 4164, 160, 700),
    ("q8_0x4", 9216, 96, 385), ("q8_0x4", 64, 544, 5), ("q8_0x4", 68, 544, 7), ("q8_0", 2048, 96, 64), ("q8_0", 2048, 96, 80),
])
def test_gemm_dispatch_edges(hip, storage, n, k, rows):
    check_matmul(hip, storage, n, k, rows)


def test_subnormal_scale_products(hip):
    # the scale products of blocks of about 1e-21 fall below the normal range
    for rows in (8, 40):
        check_matmul(hip, "q8_0", 64, 256, rows, scale=1e-20)


# hidden blocks, heads and rows that leave the last tile of each form partly
# empty: direct (2, 7, 40 rows), 64x64 tiles (100 rows of 33 blocks and of 38
# heads), 128x128 tiles (1300 rows of 33 blocks: 693 tiles of 64x64)
@pytest.mark.parametrize("storage,hidden,n_heads,rows", [
    ("q8_0x4", 96, 6, 2), ("q8_0x4", 96, 6, 7), ("q8_0", 160, 6, 7), ("q8_0x4", 1056, 30, 40),
    ("q8_0x4", 1056, 30, 100), ("q8_0x4", 1056, 30, 700), ("q8_0x4", 1056, 30, 1300), ("q8_0", 96, 6, 40),
])
def test_prefill_epilogues(storage, hidden, n_heads, rows):
    c = O.Config(dim=160, hidden_dim=hidden, n_layers=1, n_heads=n_heads, n_kv_heads=n_heads // 6 if n_heads == 6 else 5,
                 vocab_size=64, seq_len=rows + 8, rms_eps=1e-5, rope_theta=10_000.0, rope_interleaved=False,
                 head_dim=64)
    ow = gaussian_weights(c, storage, seed=hidden + rows)
    gpu, cpu = gpu_model(c, ow), O.Model(c, ow, "cpu")
    prompt = [(i * 11 + 5) % c.vocab_size for i in range(rows)]
    assert_bits_equal(gpu.prefill(prompt, 0), cpu.prefill(prompt, 0), "prefill")
    assert_bits_equal(gpu.prefill([3, 9], rows), cpu.prefill([3, 9], rows), "two rows more")
