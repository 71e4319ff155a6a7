"""Tiled GEMM of Q4_K / Q5_K weights and Q8_K activations with integer fp16 operands (mh_gemm_int16.hip) against the CPU oracle,
at the edges of its 256 x 128 tile and of the rule that takes it (x16_form, 256 compute units), and the int8 planes beside it
(mh_gemm_planes.hip) where a Q6_K matrix ends, with several weights in a launch and with FLOAT16 outputs."""
import numpy as np
import pytest

from marmot_amd.capi import DT_F32
from oracle.pyoracle import KIND_Q4_K, KIND_Q5_K, KIND_Q6_K
from tests.test_gpu_moe import check_moe_stages
from tests.util import assert_matmul_parity, gaussian, random_valid_blocks

pytestmark = pytest.mark.gpu

KINDS = {"q4_k": KIND_Q4_K, "q5_k": KIND_Q5_K, "q6_k": KIND_Q6_K}


@pytest.fixture(scope="module")
def hip():
    from marmot_amd import HipBackend

    b = HipBackend(0)
    yield b
    b.close()


@pytest.mark.parametrize("name,form,N,M,K", [
    ("q4_k", "fp16_tile_256x128", 500, 14335, 512),    # 256 x 128 tiles, the last ones ragged in both directions
    ("q4_k", "fp16_tile_256x128", 449, 14081, 256),    # one block per row, one weight row in the last tile
    ("q5_k", "fp16_tile_256x128", 512, 14336, 768),    # whole tiles, three blocks
    ("q5_k", "int8_planes_128x64", 129, 16641, 256),    # 128 x 64 tiles, one token and one weight row in the last ones
    ("q6_k", "int8_planes_128x64_k2", 193, 4229, 1280),    # rows of 5 blocks: every row starts at another offset in its 16-byte piece
    ("q6_k", "int8_planes_128x64_k2", 64, 16513, 256),     # one token tile, one block
])
def test_integer_operand_gemm_matches_oracle(hip, oracle, name, form, N, M, K):
    """The bound is the suite's for matmul outputs (1e-3, floored): exact integer block sums on both sides, so only the
    fp32 sum over at most five blocks is ordered differently."""
    kind = KINDS[name]
    blocks = hip.quantize_weights(kind, gaussian(700 + N, (M, K), 0.02))
    x = gaussian(701 + N, (N, K))
    bias = gaussian(702, (M,))
    got = hip.linear(x, blocks, kind, M, bias=bias)
    assert hip.last_route() == f"mmq_{name}_q8_k_{form}"
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
    hip.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind)
    assert hip.last_route() == "moe_experts_tiled"


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
        assert hip.last_route() == "mmq_q6_k_q8_k_int8_planes_128x64_k2"
        got = d_out.download(np.float32, (N, M))
    finally:
        for b in (d_w, d_x, d_out):
            b.free()
    assert_matmul_parity(got, oracle.matmul(KIND_Q6_K, blocks, x, M, threads=16), what=f"q6_k end {N} x {K} x {M}")


@pytest.mark.parametrize("name,form,N,M", [("q4_k", "fp16_tile_256x128", 290, 21500), ("q5_k", "fp16_tile_256x128", 290, 21500),
                                           ("q5_k", "int8_planes_128x64", 130, 16600),
                                           ("q6_k", "int8_planes_128x64_k2", 130, 6000)])
def test_random_blocks(hip, oracle, name, form, N, M):
    """Arbitrary block bytes: every nibble, scale (Q6_K: -128 among them) and minimum."""
    kind, K = KINDS[name], 512
    blocks = random_valid_blocks(np.random.default_rng(730), kind, M, K)
    x = gaussian(731, (N, K))
    got = hip.linear(x, blocks, kind, M)
    assert hip.last_route() == f"mmq_{name}_q8_k_{form}"
    assert_matmul_parity(got, oracle.matmul(kind, blocks, x, M, threads=16), what=f"random blocks {name} {form}")


@pytest.mark.parametrize("name,form,N,M", [("q4_k", "fp16_tile_256x128", 290, 21500), ("q5_k", "fp16_tile_256x128", 290, 21500),
                                           ("q5_k", "int8_planes_128x64", 130, 16600),
                                           ("q6_k", "int8_planes_128x64_k2", 130, 6000)])
@pytest.mark.parametrize("large", [False, True])
def test_block_sums(hip, name, form, N, M, large):
    """One block per row, activation and block scales of 1, minimum scale 0: the output is the integer block sum. Below
    2^24 it must be exact. Sums of one sign at the largest values go to 2^24.9 (Q5_K 2^25.9, Q6_K 2^26.9). On int8 planes they are
    rounded once; on fp16 operands 16 instructions round by at most one unit in the last place each, and a factor of two for
    the smaller partial sums of a chain whose parts differ in sign."""
    kind, K, rng = KINDS[name], 256, np.random.default_rng(740)
    rows = rng.integers(0, 256, (4, 4096), dtype=np.uint8)  # a few distinct blocks, repeated
    bb = {"q4_k": 144, "q5_k": 176, "q6_k": 210}[name]
    few = rows[:, :bb].copy()
    one, zero = np.float16(1.0).tobytes(), np.float16(0.0).tobytes()
    if name == "q6_k":
        few[:, 192:208] = 127 if large else rng.integers(-31, 32, (4, 16)).astype(np.int8).view(np.uint8)
        few[:, 208:210] = np.frombuffer(one, np.uint8)
        if large:
            few[:, :192] = rng.choice(np.array([0xFF, 0xFE, 0xEF], np.uint8), (4, 192))
        ql, qh = few[:, :128].astype(np.int64).reshape(4, 2, 2, 32), few[:, 128:192].astype(np.int64).reshape(4, 2, 32)
        u = np.stack([((ql[:, :, g & 1] >> (4 * (g >> 1))) & 15) | (((qh >> (2 * g)) & 3) << 4) for g in range(4)], axis=2)
        w = (u - 32).reshape(4, 16, 16) * few[:, 192:208].view(np.int8).astype(np.int64)[:, :, None]
    else:
        qs = 16 if name == "q4_k" else 48
        few[:, 0:2], few[:, 2:4] = np.frombuffer(one, np.uint8), np.frombuffer(zero, np.uint8)
        if large:
            few[:, 4:16] = 0xFF
            few[:, 16:] = rng.choice(np.array([0xFF, 0xEF, 0xFE], np.uint8), (4, bb - 16))
        s = few[:, 4:16].astype(np.int64)
        sc = np.concatenate([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], axis=1)
        q = few[:, qs:qs + 128].astype(np.int64).reshape(4, 4, 1, 32)
        q = np.concatenate([q & 15, q >> 4], axis=2).reshape(4, 8, 32)
        if name == "q5_k":
            h = few[:, 16:48].astype(np.int64)
            q = q + np.stack([((h >> b) & 1) << 4 for b in range(8)], axis=1)
        w = q * sc[:, :, None]
    codes = (rng.integers(120, 128, (N, K)) if large else rng.integers(-127, 128, (N, K))).astype(np.int8)
    want = codes.astype(np.int64) @ w.reshape(4, K).T
    assert (np.abs(want).max() > 2 ** 24) == large
    lay = hip.packed_activation_layout(kind, N, K)
    image = np.zeros(lay.total_bytes, np.uint8)
    vals = np.zeros((N, lay.values_per_row), np.int8)
    vals[:, :K] = codes
    image[lay.values_offset:lay.values_offset + vals.size] = vals.view(np.uint8).reshape(-1)
    image[lay.scales_offset:lay.scales_offset + 4 * N] = np.ones(N, np.float32).view(np.uint8)
    sums = codes.reshape(N, 16, 16).sum(axis=2, dtype=np.int16)
    image[lay.sums_offset:lay.sums_offset + sums.nbytes] = sums.view(np.uint8).reshape(-1)
    d_w, d_p, d_out = hip.to_device(few[np.arange(M) % 4]), hip.to_device(image), hip.alloc(4 * N * M)
    try:
        hip.linear_prepacked_d(kind, d_w, d_p, N, K, M, d_out)
        assert hip.last_route() == f"mmq_{name}_q8_k_{form}"
        got = d_out.download(np.float32, (N, M))
    finally:
        for b in (d_w, d_p, d_out):
            b.free()
    want = want[:, np.arange(M) % 4]
    if large and form.startswith("fp16"):
        # (a unit in the last place is at most 2^-23 of the value)
        assert np.max(np.abs(got - want) / np.abs(want)) <= 2 * 16 * 2.0 ** -23
    else:
        assert np.array_equal(got, want.astype(np.float32))


@pytest.mark.parametrize("name,form,N,M,K", [("q4_k", "fp16_tile_256x128", 300, 10752, 256), ("q6_k", "int8_planes_128x64_k2", 130, 3000, 512)])
def test_two_weights_in_one_launch(hip, oracle, name, form, N, M, K):
    kind = KINDS[name]
    a, b = (hip.quantize_weights(kind, gaussian(750 + i, (M, K), 0.02)) for i in range(2))
    x = gaussian(752, (N, K))
    got = hip.linear_dual(x, a, b, kind, M)
    assert hip.last_route() == f"mmq_{name}_q8_k_{form}"
    for g, w in zip(got, (a, b)):
        assert_matmul_parity(g, oracle.matmul(kind, w, x, M, threads=16), what=f"two weights {name}")


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_three_weights_and_float16_outputs(hip, oracle, dtype):
    """Query, key and value projection: the bias joins before the one rounding to FLOAT16; a single linear rounds first and
    adds the bias in FLOAT16. The suite's bound, with two roundings to FLOAT16 (2^-10) on top."""
    kind, N, M, K = KIND_Q6_K, 130, 2000, 512
    ws = [hip.quantize_weights(kind, gaussian(760 + i, (M, K), 0.02)) for i in range(3)]
    x = gaussian(763, (N, K)).astype(dtype)
    biases = [gaussian(764, (M,)).astype(dtype), None, gaussian(765, (M,)).astype(dtype)]
    tol = 1e-3 if dtype == np.float32 else 2e-3
    got = hip.linear_qkv(x, *ws, kind, M, bq=biases[0], bv=biases[2])
    assert hip.last_route() == "mmq_q6_k_q8_k_int8_planes_128x64_k2"
    for g, r in zip(got, oracle.matmul_qkv(kind, *ws, x, M, bq=biases[0], bv=biases[2])):
        assert g.dtype == dtype
        assert_matmul_parity(g, r, tol=tol, what="three weights")
    if dtype == np.float16:
        w = hip.quantize_weights(kind, gaussian(766, (6000, K), 0.02))
        bias = gaussian(767, (6000,)).astype(np.float16)
        dot = None
        for b in (None, bias):
            one = hip.linear(x, w, kind, 6000, bias=b, out_dtype=np.float16, force_pack=True)
            assert hip.last_route() == "mmq_q6_k_q8_k_int8_planes_128x64_k2"
            ref = oracle.matmul(kind, w, x, 6000, bias=b, out_dtype=np.float16, force_pack=True, threads=16)
            # a product on a tie rounds the other way, and so may the sum with the bias: one unit (2^-10) of each
            dot = one.astype(np.float64) if b is None else dot
            bound = 2.0 ** -10 * (np.abs(dot) + np.abs(ref.astype(np.float64))) + 2.0 ** -24
            assert np.all(np.abs(one.astype(np.float64) - ref) <= bound), "FLOAT16 output"


def test_q6_k_experts_at_two_byte_alignment(hip, oracle):
    """Expert stacks that do not start on a 16-byte boundary keep the kernel in passes."""
    E, F, H, k, T = 3, 2048, 4096, 2, 500
    stacks = [hip.quantize_weights(KIND_Q6_K, gaussian(770 + i, s, 0.02)) for i, s in enumerate(((E * F, H), (E * F, H), (E * H, F)))]
    hidden = gaussian(773, (T, H))
    vals, ids = oracle.topk(gaussian(774, (T, E)), k)
    w = oracle.softmax_rows(vals)
    out = []
    for pad in (0, 2):
        d = [hip.to_device(np.concatenate([np.zeros(pad, np.uint8), s.reshape(-1)])) for s in stacks]
        rest = [hip.to_device(hidden), hip.to_device(ids.astype(np.int32)), hip.to_device(w), hip.alloc(4 * T * H)]
        try:
            hip.moe_experts_d(rest[0], T, H, F, E, k, KIND_Q6_K, KIND_Q6_K, *d, *rest[1:], gate_offset=pad, up_offset=pad,
                              down_offset=pad)
            assert hip.last_route() == ("moe_experts_tiled" if pad == 0 else "moe_experts_grouped")
            out.append(rest[3].download(np.float32, (T, H)))
        finally:
            for b in d + rest:
                b.free()
    # the product of gate and up is quantized again: a difference in the last place moves single codes by a step, 1 / 127 of
    # their block's largest value, in one of the 2048 terms of an output
    diff, rms = np.abs(out[1].astype(np.float64) - out[0]), np.sqrt(np.mean(out[0].astype(np.float64) ** 2))
    assert diff.sum() <= 4e-4 * np.abs(out[0]).sum() and diff.max() <= rms / 50
