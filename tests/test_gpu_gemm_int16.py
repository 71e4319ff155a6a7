"""Tiled GEMM of K-quant weights and Q8_K activations with integer fp16 operands (mh_gemm_int16.hip) against the CPU oracle,
at the edges of its two tile forms and of the rule that chooses one (x16_form, 256 compute units)."""
import pytest

from oracle.pyoracle import KIND_Q4_K, KIND_Q5_K, KIND_Q6_K
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
