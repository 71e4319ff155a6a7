"""Tiled GEMM of K-quant weights and Q8_K activations with integer fp16 operands (mh_gemm_int16.hip) against the CPU oracle,
at the edges of its two tile forms and of the rule that chooses one (x16_form, 256 compute units)."""
import numpy as np
import pytest

from marmot_amd.capi import DT_F32
from oracle.pyoracle import KIND_Q4_K, KIND_Q5_K, KIND_Q6_K
from tests.test_gpu_moe import check_moe_stages
from tests.util import assert_matmul_parity, gaussian

pytestmark = pytest.mark.gpu

KINDS = {"q4_k": KIND_Q4_K, "q5_k": KIND_Q5_K, "q6_k": KIND_Q6_K}


@pytest.fixture(scope="module")
def hip():
    from marmot_amd import HipBackend

    b = HipBackend(0)
    yield b
    b.close()


@pytest.mark.parametrize("name,N,M,K", [
    ("q4_k", 500, 14335, 512),    # 256 x 128 tiles, the last ones ragged in both directions
    ("q4_k", 449, 14081, 256),    # one block per row, one weight row in the last tile
    ("q5_k", 512, 14336, 768),    # whole tiles, three blocks
    ("q5_k", 129, 16641, 256),    # 128 x 64 tiles, one token and one weight row in the last ones
    ("q6_k", 193, 4229, 1280),    # rows of 5 blocks: every row starts at another offset in its 16-byte piece
    ("q6_k", 64, 16513, 256),     # one token tile, one block
])
def test_integer_operand_gemm_matches_oracle(hip, oracle, name, N, M, K):
    """The bound is the suite's for matmul outputs (1e-3, floored): exact integer block sums on both sides, so only the
    fp32 sum over at most five blocks is ordered differently."""
    kind = KINDS[name]
    blocks = hip.quantize_weights(kind, gaussian(700 + N, (M, K), 0.02))
    x = gaussian(701 + N, (N, K))
    bias = gaussian(702, (M,))
    got = hip.linear(x, blocks, kind, M, bias=bias)
    assert hip.last_route() == f"mmq_{name}_q8_k_mfma_tile"
    assert_matmul_parity(got, oracle.matmul(kind, blocks, x, M, bias=bias, threads=16), what=f"{name} {N} x {K} x {M}")


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
def test_moe_experts_on_the_tiled_gemm(hip, oracle, name):
    """Experts that see 333 routes each, in items of 64 with a ragged last one, through the grouped form: two tiles per
    compute unit in both projections and 32 routes per expert are the line from which the expert layer takes it. Stage by
    stage with the bounds of the expert tests (the product of gate and up is quantized again in between)."""
    E, F, H, k, T = 3, 2048, 4096, 2, 500
    kind = KINDS[name]
    gate, up = (hip.quantize_weights(kind, gaussian(710 + i, (E * F, H), 0.02)) for i in range(2))
    down = hip.quantize_weights(kind, gaussian(712, (E * H, F), 0.02))
    hidden = gaussian(713, (T, H))
    vals, ids = oracle.topk(gaussian(714, (T, E)), k)
    w = oracle.softmax_rows(vals)
    ref = oracle.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind, threads=16)
    check_moe_stages(hip, oracle, hidden, gate, up, down, ids, w, F, E, kind, ref, f"tiled experts {name}")


@pytest.mark.parametrize("N,M,K", [
    (130, 8225, 256),   # 2 bytes; one block per row: the end arrives with the first block; one row in the last wavefront
    (130, 8229, 768),   # the matrix ends 14 bytes into a 16-byte piece
    (193, 6333, 1536),  # 12 bytes; 29 rows in the last wavefront
    (130, 8232, 256),   # whole 16-byte pieces
])
def test_end_of_a_q6_k_matrix(hip, oracle, N, M, K):
    """210-byte blocks: the last 16-byte piece may hold bytes that are not the matrix's. They are left alone (here NaN scales
    follow at once), and the bytes in front of them arrive."""
    blocks = hip.quantize_weights(KIND_Q6_K, gaussian(720 + M, (M, K), 0.02))
    x = gaussian(721 + M, (N, K))
    size = blocks.nbytes
    d_w, d_x, d_out = hip.alloc(size + 64), hip.to_device(x), hip.alloc(4 * N * M)
    try:
        d_w.upload(np.concatenate([blocks.reshape(-1), np.full(64, 0xFF, np.uint8)]))
        hip.linear_d(KIND_Q6_K, d_w, d_x, DT_F32, N, K, M, d_out, DT_F32)
        assert hip.last_route() == "mmq_q6_k_q8_k_mfma_tile"
        got = d_out.download(np.float32, (N, M))
    finally:
        for b in (d_w, d_x, d_out):
            b.free()
    assert_matmul_parity(got, oracle.matmul(KIND_Q6_K, blocks, x, M, threads=16), what=f"q6_k end {N} x {K} x {M}")
