"""Tiled GEMM of K-quant weights and Q8_K activations on int8 planes (mh_gemm_planes.hip) against the CPU oracle, at the edges
of its forms and of the rule that chooses one (planes_form, 256 compute units): 64 x 64 tiles with four K groups per workgroup, 128
rows with two or one, 64 or 128 tokens per tile, last tiles with one to four token tiles, one block per row (the second K group has none) and odd counts."""
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


CASES = [
    # (kinds, form, tokens, rows, K); mfma_tile: the kernels of mh_gemm_i8.hip
    ("q4_k q5_k", "mfma_tile", 128, 10400, 256),               # few blocks
    ("q4_k q5_k", "mfma_tile", 97, 12801, 768),
    ("q6_k", "128x64_k2", 128, 10400, 256),                    # two K groups, 64 tokens, the second group without a block
    ("q6_k", "128x64_k2", 97, 12801, 768),                     # odd block counts, one row and 33 tokens in the last tiles
    ("q4_k", "128x64_k2", 128, 9900, 3584),
    ("q4_k", "128x64_k2", 97, 9985, 3840),
    ("q4_k", "mfma_tile", 128, 9900, 3328),                    # (13 blocks)
    ("q5_k", "128x64_k2", 128, 10400, 1536),
    ("q5_k", "128x64_k2", 97, 12801, 1792),
    ("q5_k", "mfma_tile", 97, 12801, 1280),                    # (5 blocks)
    ("q6_k", "64x64_k4", 33, 11000, 1280),
    ("q4_k q5_k q6_k", "64x64_k4", 65, 2085, 256),             # four K groups, 64 rows: three without a block, one token and 37 rows in the last tiles
    ("q4_k q5_k q6_k", "64x64_k4", 130, 1401, 1280),           # (five blocks, one row in the last tile)
    ("q4_k q5_k q6_k", "64x64_k4", 257, 3232, 768),            # (255 tiles of 256)
    ("q4_k q5_k q6_k", "64x64_k4", 129, 3700, 4352),           # (more than 16 blocks)
    ("q6_k", "64x64_k4", 17, 8200, 512),                       # (17 tokens of two token tiles)
    ("q6_k", "mfma_tile", 64, 5440, 6144),                     # 85 tiles of 24 blocks
    ("q6_k", "64x64_k4", 64, 5441, 6144),                      # 86 of them
    ("q6_k", "mfma_tile", 17, 4224, 4352),                     # 66 tiles of 17 blocks, 17 tokens in each
    ("q6_k", "64x64_k4", 32, 4224, 4352),                      # 32 tokens
    ("q4_k", "mfma_tile", 33, 6144, 4096),                     # 16 blocks: 96 tiles of 33 tokens
    ("q4_k", "64x64_k4", 33, 8192, 4096),                      # 128 of them
    ("q5_k", "mfma_tile", 64, 4800, 4096),                     # 75 tiles of 64 tokens
    ("q5_k", "64x64_k4", 64, 4864, 4096),                      # 76 of them
    ("q4_k q5_k q6_k", "128x128_k2", 257, 6785, 768),          # two K groups, 128 tokens, one token in the last tile
    ("q4_k q5_k q6_k", "128x128_k2", 380, 8200, 256),
    ("q4_k q5_k", "128x64", 130, 16600, 512),                  # one K group, 64 tokens
    ("q4_k q5_k", "128x64", 161, 18500, 256),                  # (two token tiles in the last one)
    ("q6_k", "128x128", 257, 11000, 512),                      # one K group, 128 tokens: one, two, three and four token tiles in the last one
    ("q6_k", "128x128", 300, 11000, 256),
    ("q6_k", "128x128", 340, 11000, 768),
    ("q6_k", "128x128", 384, 11001, 512),
]


@pytest.mark.parametrize("name,form,N,M,K", [(n, t, *rest) for names, t, *rest in CASES for n in names.split()])
def test_forms_match_oracle(hip, oracle, name, form, N, M, K):
    """The bound is the suite's for matmul outputs (1e-3, floored): exact integer block sums on both sides, so only the fp32
    sum over at most 24 blocks is ordered differently. Arbitrary block bytes: every nibble, scale (Q6_K: -128 among them,
    products -4064 .. 4096 in two bytes) and minimum."""
    kind = KINDS[name]
    blocks = random_valid_blocks(np.random.default_rng(800 + N), kind, M, K)
    x, bias = gaussian(801 + N, (N, K)), gaussian(802, (M,))
    got = hip.linear(x, blocks, kind, M, bias=bias)
    assert hip.last_route() == f"mmq_{name}_q8_k_{'' if form == 'mfma_tile' else 'int8_planes_'}{form}"
    assert_matmul_parity(got, oracle.matmul(kind, blocks, x, M, bias=bias, threads=16), what=f"{name} {N} x {K} x {M}")


@pytest.mark.parametrize("name,form,N,M,K", [
    ("q4_k", "128x64_k2", 100, 3700, 1024),
    ("q4_k", "128x64_k2", 200, 2050, 2048),
    ("q5_k", "128x64_k2", 130, 3300, 256),
    ("q4_k", "64x64_k4", 33, 2050, 4096),    # 99 tiles of 33 tokens
    ("q5_k", "64x64_k4", 200, 500, 4096),
    ("q6_k", "64x64_k4", 64, 1500, 6144),    # 72 tiles of 24 blocks
])
def test_sets_of_weights_have_lines_of_their_own(hip, oracle, name, form, N, M, K):
    """Three weights in one launch, on forms that one weight with as many tiles leaves to the kernels of mh_gemm_i8.hip."""
    kind = KINDS[name]
    ws = [random_valid_blocks(np.random.default_rng(860 + i), kind, M, K) for i in range(3)]
    x = gaussian(863, (N, K))
    got = hip.linear_qkv(x, *ws, kind, M)
    assert hip.last_route() == f"mmq_{name}_q8_k_int8_planes_{form}"
    for g, r in zip(got, oracle.matmul_qkv(kind, *ws, x, M)):
        assert_matmul_parity(g, r, what=f"three weights {name} {N} x {K} x {M}")


@pytest.mark.parametrize("name,N,M", [("q4_k", 130, 16600), ("q5_k", 130, 16600), ("q6_k", 300, 11000),  # one K group
                                      ("q4_k", 257, 6800), ("q5_k", 257, 6800), ("q6_k", 257, 6800),  # two
                                      ("q4_k", 70, 2100), ("q5_k", 70, 2100), ("q6_k", 70, 2100)])  # four
@pytest.mark.parametrize("scale", ["largest", "mixed"])
def test_block_sums_are_exact(hip, name, N, M, scale):
    """One block per row, activation and block scales of 1, minimum scale 0: the output is the integer block sum rounded
    once, also where it does not fit 24 bits (sums of one sign at the largest values reach 2^24.9, Q5_K 2^25.9, Q6_K 2^26.9)."""
    kind, K, rng = KINDS[name], 256, np.random.default_rng(810)
    bb = {"q4_k": 144, "q5_k": 176, "q6_k": 210}[name]
    few = rng.integers(0, 256, (4, bb), dtype=np.uint8)  # a few distinct blocks, repeated
    one, zero = np.float16(1.0).tobytes(), np.float16(0.0).tobytes()
    if name == "q6_k":
        few[:, 208:210] = np.frombuffer(one, np.uint8)
        if scale == "largest":
            few[:, 192:208] = np.array([127, 128, 127, 128], np.uint8)[:, None]
            few[:, :192] = np.array([0, 0, 255, 255], np.uint8)[:, None]
        ql, qh = few[:, :128].astype(np.int64).reshape(4, 2, 2, 32), few[:, 128:192].astype(np.int64).reshape(4, 2, 32)
        u = np.stack([((ql[:, :, g & 1] >> (4 * (g >> 1))) & 15) | (((qh >> (2 * g)) & 3) << 4) for g in range(4)], axis=2)
        w = (u - 32).reshape(4, 16, 16) * few[:, 192:208].view(np.int8).astype(np.int64)[:, :, None]
    else:
        qs = 16 if name == "q4_k" else 48
        few[:, 0:2], few[:, 2:4] = np.frombuffer(one, np.uint8), np.frombuffer(zero, np.uint8)
        if scale == "largest":
            few[:, 4:] = 0xFF
        s = few[:, 4:16].astype(np.int64)
        sc = np.concatenate([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], axis=1)
        q = few[:, qs:qs + 128].astype(np.int64).reshape(4, 4, 1, 32)
        q = np.concatenate([q & 15, q >> 4], axis=2).reshape(4, 8, 32)
        if name == "q5_k":
            h = few[:, 16:48].astype(np.int64)
            q = q + np.stack([((h >> b) & 1) << 4 for b in range(8)], axis=1)
        w = q * sc[:, :, None]
    codes = (rng.integers(120, 128, (N, K)) if scale == "largest" else rng.integers(-127, 128, (N, K))).astype(np.int8)
    want = codes.astype(np.int64) @ w.reshape(4, K).T
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
        got = d_out.download(np.float32, (N, M))
    finally:
        for b in (d_w, d_p, d_out):
            b.free()
    assert np.array_equal(got, want[:, np.arange(M) % 4].astype(np.float32))


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
def test_experts_in_more_tiles_than_the_chip_holds(hip, oracle, name):
    """About 30 items of 32 tiles in both projections: workgroups go on to a second tile, of the other weight or another expert,
    ragged last items among them. Stage by stage with the bounds of the expert tests."""
    E, F, H, k, T = 3, 2048, 4096, 2, 900
    kind = KINDS[name]
    gate, up = (hip.quantize_weights(kind, gaussian(820 + i, (E * F, H), 0.02)) for i in range(2))
    down = hip.quantize_weights(kind, gaussian(822, (E * H, F), 0.02))
    hidden = gaussian(823, (T, H))
    vals, ids = oracle.topk(gaussian(824, (T, E)), k)
    w = oracle.softmax_rows(vals)
    ref = oracle.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind, threads=16)
    check_moe_stages(hip, oracle, hidden, gate, up, down, ids, w, F, E, kind, ref, f"experts from tile to tile {name}")
    hip.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind)
    assert hip.last_route() == "moe_experts_tiled"


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("H,F,T", [(2048, 256, 8200), (256, 2304, 16500)])  # one block per row: down, gate and up
def test_experts_of_a_call_and_of_its_halves(hip, name, H, F, T):
    """A token's result does not depend on the others, bit for bit: the halves of a call fit the chip in one of the two
    projections, the whole call does not."""
    E, k, kind = 4, 2, KINDS[name]
    gate, up = (random_valid_blocks(np.random.default_rng(830 + i), kind, E * F, H) for i in range(2))
    down = random_valid_blocks(np.random.default_rng(832), kind, E * H, F)
    hidden, rng = gaussian(833, (T, H)), np.random.default_rng(834)
    ids = np.argsort(rng.random((T, E)), axis=1)[:, :k].astype(np.int32)
    w = np.full((T, k), 0.5, np.float32)
    whole = hip.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind)
    assert hip.last_route() == "moe_experts_tiled"
    for part in (slice(0, T // 2), slice(T // 2, T)):
        got = hip.moe_experts(hidden[part], gate, up, down, ids[part], w[part], F, E, kind, kind)
        assert hip.last_route() == "moe_experts_tiled"
        assert np.array_equal(got.view(np.uint32), whole[part].view(np.uint32))


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("H,F,T", [(1024, 768, 2100), (2048, 512, 2077)])
def test_gated_product_in_the_gemm(hip, name, H, F, T):
    """The call whose GEMM forms the gated product against the one that stores gate and up outputs and forms it when they are
    packed (a call that looks at the stages): the same sums through the same function, bit for bit. Items of one to 64 routes."""
    E, k, kind = 6, 2, KINDS[name]
    gate, up = (hip.quantize_weights(kind, gaussian(840 + i, (E * F, H), 0.02)) for i in range(2))
    down = hip.quantize_weights(kind, gaussian(842, (E * H, F), 0.02))
    hidden, rng = gaussian(843, (T, H)), np.random.default_rng(844)
    ids = np.argsort(rng.random((T, E)) * np.array([1, 1, 1, 2, 3, 6]), axis=1)[:, :k].astype(np.int32)
    w = np.abs(gaussian(845, (T, k)))
    got = hip.moe_experts(hidden, gate, up, down, ids, w, F, E, kind, kind)
    assert hip.last_route() == "moe_experts_tiled"
    stages = hip.moe_experts_probe(hidden, gate, up, down, ids, w, F, E, kind, kind)
    assert np.array_equal(got.view(np.uint32), stages["out"].view(np.uint32))


def test_experts_in_more_items_than_a_grid_dimension_holds(hip):
    """66048 work items (tiles are counted in one dimension): 4096 tokens 129 times over, each with the bits of the call of 4096."""
    E, F, H, k, T, times = 8, 256, 256, 8, 4096, 129
    gate, up = (random_valid_blocks(np.random.default_rng(850 + i), KIND_Q4_K, E * F, H) for i in range(2))
    down = random_valid_blocks(np.random.default_rng(852), KIND_Q4_K, E * H, F)
    hidden = gaussian(853, (T, H))
    ids, w = np.tile(np.arange(E, dtype=np.int32), (T, 1)), np.abs(gaussian(854, (T, k)))
    want = hip.moe_experts(hidden, gate, up, down, ids, w, F, E, KIND_Q4_K, KIND_Q4_K)
    assert hip.last_route() == "moe_experts_tiled"
    got = hip.moe_experts(*(np.tile(a, (times, 1)) if a is hidden else a for a in (hidden, gate, up, down)),
                          np.tile(ids, (times, 1)), np.tile(w, (times, 1)), F, E, KIND_Q4_K, KIND_Q4_K)
    assert hip.last_route() == "moe_experts_tiled"
    for part in got.reshape(times, T, H):
        assert np.array_equal(part.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("name,N,M,K", [("q4_k", 33, 4224, 4096), ("q5_k", 80, 2560, 4096), ("q6_k", 64, 4224, 8192)])
def test_captured_without_an_eager_run(oracle, name, N, M, K):
    """Packed activations, on sizes whose K is split over workgroups with partial sums in the workspace: a fresh device object
    captures the call all the same, on tiles that need none, and splits once it may allocate."""
    from marmot_amd import HipBackend

    kind, hip = KINDS[name], HipBackend(0)
    blocks, x = random_valid_blocks(np.random.default_rng(870), kind, M, K), gaussian(871, (N, K))
    want = oracle.matmul(kind, blocks, x, M, threads=16)
    bufs = [hip.to_device(blocks), hip.to_device(x), hip.alloc(hip.packed_activation_bytes(kind, N, K)), hip.alloc(4 * N * M)]
    d_w, d_x, d_p, d_out = bufs
    try:
        hip.pack_activations_d(kind, d_x, DT_F32, N, K, d_p)
        graph = hip.graph_capture(lambda: hip.linear_prepacked_d(kind, d_w, d_p, N, K, M, d_out))
        assert hip.last_route() == f"mmq_{name}_q8_k_int8_planes_64x64_k4"
        for _ in range(3):
            d_out.upload(np.full((N, M), np.nan, np.float32))
            hip.graph_launch(graph)
            hip.synchronize()
            assert_matmul_parity(d_out.download(np.float32, (N, M)), want, what=f"captured {name}")
            hip.linear_prepacked_d(kind, d_w, d_p, N, K, M, d_out)
            assert hip.last_route() == f"mmq_{name}_q8_k_mfma_tile"
            assert_matmul_parity(d_out.download(np.float32, (N, M)), want, what=f"eager {name}")
        hip.graph_destroy(graph)
    finally:
        for b in bufs:
            b.free()
        hip.close()
