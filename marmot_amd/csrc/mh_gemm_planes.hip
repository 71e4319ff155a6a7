// Prompts with packed (Q8_K) activations: K-quant weights x activation codes as a tiled GEMM on the int8 matrix cores, the
// product of a weight and its sub-block scale cut into two int8 planes.
//
// Per 256-value block the reference forms (cpu_vec_dot_q{4,5,6}_k_q8_k, src/backends/cpu/ops/matmul/quantized/
// vec_dot_impl.h:689-860) y += a.d * (w.d * isum - w.dmin * msum) with isum = sum_j sc_j * (q_j . a_j) and msum = sum_j mn_j *
// (sum of a over sub-block j). sc * q does not fit int8, but two numbers that do make it up: Q4_K q * (sc & 7) and q * (sc >> 3)
// (at most 105); Q5_K (0 .. 1953) and Q6_K (-4064 .. 4096) the product itself as 256 * h + l, its high byte and its low byte
// as signed numbers. One chain of v_mfma_i32_32x32x32_i8 per plane over the whole block gives isum = X + 2^SHIFT * Y exactly
// (below 2^27), in the matrix time of one fp16 operand, since the int8 instructions run at twice the rate. Beside fp16
// operands (mh_gemm_int16.hip, which need two for Q6_K) the activations stay the bytes they are packed as: half the reads
// from LDS, no conversion, direct-to-LDS loads; the price is a shift-add and a conversion per output and block. The sums of
// 16 codes (at most 2032) and the mins are exact in fp16: one fp16 instruction per block and tile gives msum.
//
// What bounds it: the issue port, most of all vector instructions. Per wavefront and block, 32 rows x 128 tokens, a kernel issues
// 64 (68) matrix instructions beside 700 (Q6_K), 736 (Q5_K) or 534 (Q4_K) vector ones: 256 or 320 of the fp32 step (one output:
// shift-add, conversion, two or three multiply-adds), 50 / 16 per 32 values of unpacking (Q6_K, Q5_K / Q4_K), the rest addresses.
// Counted for 1024 x 14336 x 4096 (two K groups): 720, 755 and 553 vector instructions with the start and the end shared out; all
// instructions hold the port for 74, 86 and 78 % of a SIMD's clocks, vector ones for 60, 69 and 61, while the matrix cores are busy
// for 39, 46 and 53 %. Q6_K waits more: its raw blocks are read from LDS at two-byte offsets (LDS busy for 51 %, Q5_K 26).
// Hence the tile: what a lane unpacks meets up to four token tiles, and everything else waits in LDS so that two wavefronts
// fit a SIMD.
//
// A wavefront owns 32 weight rows x 32 CT tokens: lane (row j, half kh) unpacks the bytes only it reads, a run of 32 values
// (a step: 2 CT matrix instructions) ahead of its use, a quarter between every two matrix instructions. A stage is half a block
// of activation codes (two buffers, one barrier per stage); raw weight blocks go through a private LDS area of the wavefront,
// whose next block is requested as soon as the last bytes of this one are in registers. The fp32 step of a block is done
// half at the end of its second stage and half at the beginning of the next block's first, which makes stages equally long.
// KG = 2: eight wavefronts, two K groups with buffers of their own that take every second block, one stage apart (one does its
// fp32 step while the other multiplies), sums joined in LDS at the end: for calls that have one tile per compute unit, which
// would leave a SIMD one wavefront. KG = 4 halves the tile's rows besides (RG = 2 wavefronts of them, four K groups): a call of
// half a chip of 128 x 64 tiles, the k and v projections of a prompt, takes a whole chip of these. KG = 1: four wavefronts, two
// or three workgroups per compute unit; the last tiles of a ragged token count run on as many of the C token tiles as hold a
// token.
// Measured (us of whole calls in a row, the quantization of 6 - 17 included; before: the best of the kernels of
// mh_gemm_int16.hip and mh_gemm_i8.hip; tokens x K x M):
//          1024 x 14336 x 4096   1000 x 4096 x 14336   1024 x 4096 x 4096   300 x 4096 x 4096
//   Q6_K   308 / 162             302 / 185             99 / 59              61 / 39
//   Q5_K   203 / 154             -                     67 / 55              38 / 35
//   Q4_K   189 / 143             -                     62 / 52              31 / 30
// and routed experts (E = 128, top 8, H = 2048, F = 768, 2048 tokens) Q6_K 650 / 455, Q4_K 395 / 373.
// Experts have few blocks per row (3 and 8 there), so a tile is over soon after its first operands have arrived. Their form
// (LOOP) keeps as many workgroups as the chip holds and has each request the first codes and weights of its next tile during
// the last block of this one: the calls above 384 -> 373 and 464 -> 455, 1500 tokens of 64 Q5_K experts of 512 228 -> 212. The
// gate and up projections share a tile (GLU: 64 rows of each), so that their gated product is formed from sums that are still in
// registers: 50 MB written and read in the place of 100, 376 -> 350 us for the Q4_K call, its packing 28 -> 19 us. (Linears
// of 16 blocks and more would lose up to 4 % to the registers that LOOP takes.)
#include "mh_rows.h"

#include <type_traits>

namespace mh {

typedef int pl_i32x4 __attribute__((ext_vector_type(4)));
typedef int pl_i32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 pl_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 pl_half8 __attribute__((ext_vector_type(8)));
typedef float pl_float16 __attribute__((ext_vector_type(16)));
typedef unsigned short pl_u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t pl_u32x4 __attribute__((ext_vector_type(4)));

struct GemmPlanesParams {
    const uint8_t *w[3];   // weights: M rows of nb blocks each
    const int8_t *qs;      // activation codes, rows of kp bytes
    const float *ad;       // activation block scales [rows][nb]
    const int16_t *sums;   // sums of 16 codes [rows][16 nb]
    size_t kp, N, M, nb;
    void *out[3];
    const void *bias[3];
    int bias_is_f16, bias_first, out_is_f16;
    uint32_t row_tiles, col_tiles, weights;
    // grouped (MoE): work items (expert, first route, routes) in the place of col_tiles; activation row of a route through
    // act_index (null: the route itself), output row = route
    const int4 *items;
    const int *n_items;
    const uint32_t *act_index;
    size_t expert_stride;
};

// Per format: 16-byte pieces that cover a row's block from the boundary below its start, whether a minimum exists, and the
// weight of the second plane
template <int KIND>
struct PlanesFormat;
template <>
struct PlanesFormat<MARMOT_HIP_KIND_Q4_K> {
    static constexpr int BYTES = Q4_K_BYTES, PIECES = 9, SHIFT = 3;
    static constexpr bool MIN = true;
};
template <>
struct PlanesFormat<MARMOT_HIP_KIND_Q5_K> {
    static constexpr int BYTES = Q5_K_BYTES, PIECES = 11, SHIFT = 8;
    static constexpr bool MIN = true;
};
template <>
struct PlanesFormat<MARMOT_HIP_KIND_Q6_K> {
    static constexpr int BYTES = Q6_K_BYTES, PIECES = 14, SHIFT = 8;  // 14 + 210 bytes at most
    static constexpr bool MIN = false;
};

// RG: wavefronts along the rows of a workgroup's tile
template <int KIND, int C, int KG, bool LOOP, int RG>
struct PlanesLds {
    static constexpr int ROWS = 64 / PlanesFormat<KIND>::PIECES;  // whole rows per direct-to-LDS load
    static constexpr int DMA = (32 + ROWS - 1) / ROWS;            // such loads of a wavefront per block
    static constexpr int ACT = 32 * C * 128;                      // one stage: 32 C tokens x 128 codes
    static constexpr int W0 = KG * 2 * ACT;
    static constexpr int WAVE_W = 32 * 16 * PlanesFormat<KIND>::PIECES;
    static constexpr int S0 = W0 + RG * KG * WAVE_W;
    static constexpr int SUMS = PlanesFormat<KIND>::MIN ? 32 * C * 32 : 0;  // sums of a block as fp16: [token][16]
    static constexpr int SD = SUMS + 32 * C * 4;                            // then the activation scales [token]
    static constexpr int OFFS = S0 + 2 * KG * SD;  // lane offsets of the activation loads: [this tile, next][wavefront][load][lane]
    static constexpr int OFF_N = 4 * C / RG + 1 + (PlanesFormat<KIND>::MIN ? 1 : 0);
    static constexpr int TABLE = RG * KG * OFF_N * 256;
    static constexpr int NEXT = OFFS + (LOOP ? 2 : 1) * TABLE;  // activation rows of the next tile's tokens, per wavefront
    static constexpr int BYTES = NEXT + (LOOP ? RG * 128 * C : 0);
};

__device__ __forceinline__ pl_u16x2 pl_v(uint32_t v) {
    return __builtin_bit_cast(pl_u16x2, v);
}
__device__ __forceinline__ uint32_t pl_u(pl_u16x2 v) {
    return __builtin_bit_cast(uint32_t, v);
}

// (a & 0x0f0f0f0f) | (b & 0xf0f0f0f0) in one instruction, whatever is done with the result
__device__ __forceinline__ uint32_t pl_nibbles(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(0x0f0f0f0fu), "v"(a), "v"(b));
    return r;
}
// e: products of bytes 0 and 2, o: of bytes 1 and 3, each + 128, as 16-bit numbers: their high bytes and their low bytes - 128
__device__ __forceinline__ void pl_split(uint32_t e, uint32_t o, int &lo, int &hi) {
    lo = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
    hi = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
}

// The lane's part of a block: row j, values 16 kh .. 16 kh + 15 of each of the eight runs of 32 values. A half block is four
// steps; step i unpacks run sub(i) of it, both nibbles of the same 16 bytes one after the other.
template <int KIND>
struct PlanesRaw;

template <>
struct PlanesRaw<MARMOT_HIP_KIND_Q6_K> {
    uint4 ql, qh;
    uint32_t scw[2];
    float d, ndmin;
    static constexpr int sub(int i) {
        return (i & 1) * 2 + (i >> 1);
    }
    __device__ __forceinline__ void load_low(const uint8_t *at, int hb, int pair, int kh) {
        __builtin_memcpy(&ql, at + 64 * hb + 32 * pair + 16 * kh, 16);
    }
    __device__ __forceinline__ void load_half(const uint8_t *at, int hb, int kh) {
        __builtin_memcpy(&qh, at + 128 + 32 * hb + 16 * kh, 16);
        __builtin_memcpy(scw, at + 192 + 8 * hb, 8);
        scw[0] <<= 8 * (1 - kh);  // bytes 1 and 3: this lane's groups
        scw[1] <<= 8 * (1 - kh);
    }
    __device__ __forceinline__ void load_header(const uint8_t *at, int) {
        uint16_t v;
        __builtin_memcpy(&v, at + 208, 2);
        d = h2f(v);
        asm volatile("" : "+v"(d));
        ndmin = 0.0f;
    }
    __device__ __forceinline__ pl_half8 mins() const {
        return pl_half8{};
    }
    struct Scale {
        pl_u16x2 m, c;
    };
    __device__ __forceinline__ Scale scale(int, int i) const {
        const uint32_t word = scw[sub(i) >> 1];
        const uint32_t m = __builtin_amdgcn_perm(0u, word, (sub(i) & 1) ? 0x09030903u : 0x08010801u);
        return {pl_v(m), pl_v(m) * pl_u16x2{(unsigned short)-32, (unsigned short)-32} + pl_u16x2{128, 128}};
    }
    __device__ __forceinline__ void planes(const Scale &sc, int, int i, int piece, int &lo, int &hi) const {
        const uint32_t lw[4] = {ql.x, ql.y, ql.z, ql.w};
        const uint32_t hw[4] = {qh.x, qh.y, qh.z, qh.w};
        const int s = sub(i);
        const uint32_t l = (i & 1) ? lw[piece] >> 4 : lw[piece];
        const uint32_t h = s == 0 ? hw[piece] << 4 : s == 1 ? hw[piece] << 2 : s == 2 ? hw[piece] : hw[piece] >> 2;
        const uint32_t x = pl_nibbles(l, h);
        const pl_u16x2 e = pl_v(x & 0x003f003fu), o = pl_v((x >> 8) & 0x003f003fu);
        pl_split(pl_u(e * sc.m + sc.c), pl_u(o * sc.m + sc.c), lo, hi);
    }
};

template <>
struct PlanesRaw<MARMOT_HIP_KIND_Q4_K> {
    uint4 q;
    uint32_t sc, mn;
    float d, ndmin;
    static constexpr int sub(int i) {
        return i;
    }
    __device__ __forceinline__ void load_low(const uint8_t *at, int hb, int pair, int kh) {
        q = *(const uint4 *)(at + 16 + 64 * hb + 32 * pair + 16 * kh);
    }
    // 6-bit scales and mins as bytes (get_scale_min_k4, kquant_common.h:29-37)
    __device__ __forceinline__ void load_half(const uint8_t *at, int hb, int) {
        const uint4 hdr = *(const uint4 *)at;
        sc = hb == 0 ? hdr.y & 0x3f3f3f3fu : (hdr.w & 0x0f0f0f0fu) | (((hdr.y >> 6) & 0x03030303u) << 4);
    }
    __device__ __forceinline__ void load_header(const uint8_t *at, int kh) {
        const uint4 hdr = *(const uint4 *)at;
        d = h2f((uint16_t)(hdr.x & 0xffffu));
        ndmin = -h2f((uint16_t)(hdr.x >> 16));
        asm volatile("" : "+v"(d), "+v"(ndmin));  // plain fp32 values: no mixed-precision multiply-adds later
        mn = kh == 0 ? hdr.z & 0x3f3f3f3fu : ((hdr.w >> 4) & 0x0f0f0f0fu) | (((hdr.z >> 6) & 0x03030303u) << 4);
        asm volatile("" : "+v"(mn));
    }
    // mins as the fp16 operand of the sums: sum 8 kh + e belongs to sub-block 4 kh + e / 2
    __device__ __forceinline__ pl_half8 mins() const {
        pl_half8 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            r[2 * i] = r[2 * i + 1] = (_Float16)(unsigned short)((mn >> (8 * i)) & 0xffu);
        }
        return r;
    }
    struct Scale {
        pl_u16x2 lo, hi;
    };
    __device__ __forceinline__ uint32_t splat(int i) const {
        return __builtin_amdgcn_perm(0u, sc, i == 0 ? 0x0c000c00u : i == 1 ? 0x0c010c01u : i == 2 ? 0x0c020c02u : 0x0c030c03u);
    }
    __device__ __forceinline__ Scale scale(int, int i) const {
        const uint32_t v = splat(i);
        return {pl_v(v & 0x00070007u), pl_v(v >> 3 & 0x00070007u)};
    }
    __device__ __forceinline__ void planes(const Scale &s, int, int i, int piece, int &lo, int &hi) const {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        const pl_u16x2 x = pl_v((i & 1) ? (w[piece] >> 4) & 0x0f0f0f0fu : w[piece] & 0x0f0f0f0fu);
        lo = (int)pl_u(x * s.lo);
        hi = (int)pl_u(x * s.hi);
    }
};

template <>
struct PlanesRaw<MARMOT_HIP_KIND_Q5_K> {
    PlanesRaw<MARMOT_HIP_KIND_Q4_K> k4;
    uint4 h;  // fifth bits of this lane's 16 positions of every run: bit 4 hb + i
    float d, ndmin;
    static constexpr int sub(int i) {
        return i;
    }
    __device__ __forceinline__ void load_low(const uint8_t *at, int hb, int pair, int kh) {
        k4.load_low(at + 32, hb, pair, kh);
    }
    __device__ __forceinline__ void load_half(const uint8_t *at, int hb, int kh) {
        k4.load_half(at, hb, kh);
        if (hb == 0) {
            h = *(const uint4 *)(at + 16 + 16 * kh);
        }
    }
    __device__ __forceinline__ void load_header(const uint8_t *at, int kh) {
        k4.load_header(at, kh);
        d = k4.d;
        ndmin = k4.ndmin;
    }
    __device__ __forceinline__ pl_half8 mins() const {
        return k4.mins();
    }
    struct Scale {
        pl_u16x2 m;
    };
    __device__ __forceinline__ Scale scale(int, int i) const {
        return {pl_v(k4.splat(i))};
    }
    __device__ __forceinline__ void planes(const Scale &s, int hb, int i, int piece, int &lo, int &hi) const {
        const uint32_t w[4] = {k4.q.x, k4.q.y, k4.q.z, k4.q.w};
        const uint32_t hw[4] = {h.x, h.y, h.z, h.w};
        const int bit = 4 * hb + i;
        const uint32_t l = (i & 1) ? w[piece] >> 4 : w[piece];
        const uint32_t f = bit < 4 ? hw[piece] << (4 - bit) : hw[piece] >> (bit - 4);
        const uint32_t x = pl_nibbles(l, f);
        const pl_u16x2 e = pl_v(x & 0x001f001fu), o = pl_v((x >> 8) & 0x001f001fu);
        const pl_u16x2 c = {128, 128};
        pl_split(pl_u(e * s.m + c), pl_u(o * s.m + c), lo, hi);
    }
};

// 64 x 16 bytes from base + voff (per lane) to LDS address lds_addr + 16 * lane (see dma16_to_lds). The s_nop separates the
// load from a vector instruction that may have written the scalar base right before it (v_readlane of a spilled scalar
// register): a memory instruction must not read such a register within five wait states, and the compiler does not look
// into the assembly to keep them apart.
__device__ __forceinline__ void planes_dma16(uint32_t lds_addr, const uint8_t *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base)
                 : "memory");
}
// The same for the lanes of `mask` only (every lane is active around it): a branch here would be a block of its own, and the
// compiler moves the arithmetic that belongs before it behind it.
__device__ __forceinline__ void planes_dma16_of(uint64_t mask, uint32_t lds_addr, const uint8_t *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base), "s"(mask)
                 : "memory");
}
// 64 x 4 bytes, to lds_addr + 4 * lane
__device__ __forceinline__ void planes_dma4(uint32_t lds_addr, const uint8_t *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void planes_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// LOOP: a workgroup goes from tile to tile. GLU: its first two wavefronts hold rows of weight 0, the others the same rows of weight 1,
// and the output is silu(first) * second.
template <int KIND, int C, int KG, bool LOOP = false, int RG = 4, bool GLU = false>
__global__ __launch_bounds__(64 * RG * KG, C == 2 && KG == 1 ? 3 : 2) void k_gemm_planes(const GemmPlanesParams p) {
    using F = PlanesFormat<KIND>;
    using L = PlanesLds<KIND, C, KG, LOOP, RG>;
    static_assert(!LOOP || KG == 1, "one K group");
    static_assert(!GLU || LOOP, "the join of the two weights' sums borrows the place of the codes between two tiles");
    constexpr int TOK = 32 * C;
    // direct-to-LDS loads of codes per wavefront and stage, 8 tokens each: the i-th of all wavefronts is tile i (RG == 4)
    constexpr int APW = 4 * C / RG;
    static_assert(RG == 4 || (RG == 2 && C == 2 && KG == 4), "a token tile is four loads; two wavefronts load the sums of 64 tokens");
    warm_kernel_arguments<sizeof(GemmPlanesParams)>();
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gw = wave % RG, kg = wave / RG;  // row group, K group
    const uint32_t nb = (uint32_t)p.nb;
    // Tile t of the call: rows fastest, then weights, then tokens (or work items). KG == 1: a workgroup takes every gridDim.x-th.
    struct Tile {
        const uint8_t *w;
        uint32_t which, row0, tok0, toks;  // row0: this wavefront's first weight row; tok0: first output row
    };
    typedef const __attribute__((address_space(4))) int uniform_int;
    uint32_t cols = p.col_tiles;
    if (p.items != nullptr) {
        cols = (uint32_t)*(uniform_int *)(uintptr_t)p.n_items;
    }
    const uint32_t tiles_all = p.row_tiles * p.weights * cols;
    auto tile_at = [&](uint32_t t) {
        Tile r;
        const uint32_t rest = t / p.row_tiles, y = rest / p.weights;
        r.which = rest - y * p.weights;
        r.row0 = (t - rest * p.row_tiles) * (GLU ? 64u : 32u * RG) + 32u * (uint32_t)(GLU ? gw & 1 : gw);
        r.w = p.w[GLU ? (uint32_t)gw >> 1 : r.which];
        if (p.items != nullptr) {
            uniform_int *it = (uniform_int *)(uintptr_t)(p.items + y);
            r.w += (size_t)it[0] * p.expert_stride;
            r.tok0 = (uint32_t)it[1];
            r.toks = (uint32_t)it[2];
        } else {
            r.tok0 = y * TOK;
            r.toks = (uint32_t)p.N - r.tok0 < (uint32_t)TOK ? (uint32_t)p.N - r.tok0 : (uint32_t)TOK;
        }
        return r;
    };
    if (blockIdx.x >= tiles_all) {
        return;
    }
    uint32_t tile = blockIdx.x;
    const Tile first = tile_at(tile);
    uint32_t toks = first.toks;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_u8_t *)lds;

    // ---- activation codes: load q of a stage brings tokens 8 q .. 8 q + 7, 128 bytes each. Lane l's 16 bytes land in slot l % 8 of
    // token 8 q + l / 8, which holds chunk (slot ^ swizzle(token)), swizzle(t) = t % 8 ^ (t / 8) % 2: eight, and sixteen, lanes with
    // consecutive tokens that read one chunk touch different banks.
    const uint32_t a_group = lds_base + (uint32_t)(kg * 2 * L::ACT);
    uint32_t table = 0;  // this tile's
    auto offs = [&](uint32_t table, int i) -> uint32_t & {
        return ((uint32_t *)(lds + L::OFFS + table * (uint32_t)L::TABLE))[wave * (L::OFF_N * 64) + 64 * i + lane];
    };
    const uint32_t s_tok = (uint32_t)((gw * 64 + lane) >> 1) % TOK;
    auto fill_offs = [&](uint32_t table, auto act_row) {  // act_row: the activation row of a tile's token
#pragma unroll
        for (int i = 0; i < APW; ++i) {
            const uint32_t q = (uint32_t)(RG * i + gw);
            const uint32_t chunk = ((uint32_t)lane & 7u) ^ ((uint32_t)lane >> 3) ^ (q & 1u);
            offs(table, i) = act_row(8u * q + ((uint32_t)lane >> 3)) * (uint32_t)p.kp + 16u * chunk;
        }
        // scales, sums (tokens wrap around: several lanes then bring the same bytes)
        offs(table, APW) = act_row(((uint32_t)gw * 64u + (uint32_t)lane) % TOK) * nb * 4u;
        if constexpr (F::MIN) {
            offs(table, APW + 1) = act_row(s_tok) * nb * 32u + 16u * (lane & 1);
        }
    };
    fill_offs(0u, [&](uint32_t t) {  // tokens beyond the last one re-read it and are never stored
        const uint32_t row = first.tok0 + (t < toks ? t : toks - 1u);
        return p.act_index != nullptr ? p.act_index[row] : row;
    });
    auto request_acts = [&](uint32_t half, int buffer, int i, uint32_t off) {
        planes_dma16(a_group + (uint32_t)(buffer * L::ACT + 1024 * (RG * i + gw)), (const uint8_t *)p.qs + (size_t)half * 128u, off);
    };
    // ---- scales and sums of a block, in places that alternate with its number since the workgroup began
    const uint32_t sd_at = lds_base + (uint32_t)(L::S0 + 2 * kg * L::SD);
    pl_u32x4 s_next = {};
    auto request_scales = [&](uint32_t b, uint32_t number, uint32_t off) {
        if (64u * (uint32_t)gw < toks) {
            planes_dma4(sd_at + (uint32_t)((number & 1u) * L::SD + L::SUMS + 256 * gw), (const uint8_t *)p.ad + (size_t)b * 4u, off);
        }
    };
    auto request_sums = [&](uint32_t b, uint32_t off) {
        if constexpr (F::MIN) {
            glb_u8_t *sums = (glb_u8_t *)p.sums + (size_t)b * 32u;
            asm("" : "+s"(sums));
            s_next = *(const __attribute__((address_space(1))) pl_u32x4 *)(sums + (size_t)off);
        }
    };
    auto store_block = [&](uint32_t number) {
        if constexpr (F::MIN) {
            const uint32_t v[4] = {s_next.x, s_next.y, s_next.z, s_next.w};
            uint32_t e[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                e[c] = __builtin_bit_cast(uint32_t, pl_half2{(_Float16)(int16_t)(v[c] & 0xffffu), (_Float16)(int16_t)(v[c] >> 16)});
            }
            uint8_t *sums = lds + L::S0 + (2 * kg + (number & 1u)) * L::SD;
            *(uint4 *)(sums + s_tok * 32u + 16u * (lane & 1)) = make_uint4(e[0], e[1], e[2], e[3]);
        }
    };

    // ---- weights: load i of a block brings rows ROWS i .. + ROWS - 1 of the wavefront: lane l the 16-byte piece l % PIECES
    // of row l / PIECES, counted from the 16-byte boundary at or below the row's block; a piece that holds no byte of the
    // block re-reads the last one that does, lanes behind the last row and rows behind the matrix re-read a row before.
    const uint32_t row_bytes = (uint32_t)p.nb * F::BYTES;
    const uint32_t w_r = (uint32_t)lane / F::PIECES < L::ROWS ? (uint32_t)lane / F::PIECES : L::ROWS - 1u;
    const uint32_t w_piece = 16u * ((uint32_t)lane - F::PIECES * w_r < F::PIECES ? (uint32_t)lane - F::PIECES * w_r : F::PIECES - 1u);
    const uint32_t w_lds = lds_base + (uint32_t)(L::W0 + wave * L::WAVE_W);
    // Q6_K: the piece that holds the end of the matrix may reach up to 14 bytes behind it (its size need not be a multiple
    // of 16), and those bytes need not exist. The wavefront of the last row brings the piece before in its place (one
    // operand more of a minimum that is there anyway) and copies the bytes that exist when the block is read (bring_end).
    const uint8_t *wbase;
    uint32_t low4, last_row, w_first, w_last, w_end, w_most, end_block, my_row;
    auto aim = [&](const Tile &t) {  // where the weights of tile t are
        const uint32_t M = (uint32_t)p.M;
        const uint8_t *at = t.w + (size_t)(t.row0 < M ? t.row0 : M - 1u) * row_bytes;
        low4 = (uint32_t)((uintptr_t)at & 15u);
        wbase = uniform_pointer(at - low4);
        last_row = t.row0 >= M ? 0u : M - t.row0 < 32u ? M - t.row0 - 1u : 31u;
        w_first = low4 + w_r * row_bytes + (F::BYTES % 16 != 0 ? 0u : w_piece);
        w_last = low4 + last_row * row_bytes + (F::BYTES % 16 != 0 ? 0u : w_piece);
        w_end = low4 + (last_row + 1u) * row_bytes;
        const bool ragged = F::BYTES % 16 != 0 && t.row0 + 32u >= M && (w_end & 15u) != 0;
        w_most = ragged ? (w_end & ~15u) - 16u : ~0u;
        end_block = ragged ? nb - 1u : ~0u;
        my_row = low4 + ((uint32_t)j < last_row ? (uint32_t)j : last_row) * row_bytes;
    };
    aim(first);
    auto request_weights = [&](uint32_t b, int i) {
        uint32_t at = w_first;
        asm volatile("" : "+v"(at));  // formed at each load: kept in registers, the L::DMA offsets would be spilled
        at += (uint32_t)i * (L::ROWS * row_bytes);
        at = at < w_last ? at : w_last;
        const uint32_t to = w_lds + (uint32_t)(i * L::ROWS * 16 * F::PIECES);
        if constexpr (F::BYTES % 16 != 0) {
            at += b * (uint32_t)F::BYTES;
            const uint32_t last = (at + (uint32_t)F::BYTES - 1u) & ~15u;
            at = (at & ~15u) + w_piece;
            at = at < last ? at : last;
            at = at < w_most ? at : w_most;
        }
        const uint8_t *base = F::BYTES % 16 != 0 ? wbase : wbase + (size_t)b * F::BYTES;
        // (the launcher checks that rows of whole 16-byte pieces start on 16-byte boundaries)
        // lanes without a row write nothing: the place behind the rows of this load belongs to the next one
        constexpr int ALL = L::ROWS * F::PIECES, LAST = (32 - L::ROWS * (L::DMA - 1)) * F::PIECES;
        planes_dma16_of(~0ull >> (64 - (i + 1 < L::DMA ? ALL : LAST)), to, base, at);
    };
    // After the loads of block b have arrived: the end of the matrix, two bytes per lane
    auto bring_end = [&](uint32_t b) {
        if constexpr (F::BYTES % 16 != 0) {
            if (b == end_block) {
                const uint32_t block = low4 + last_row * row_bytes + b * (uint32_t)F::BYTES;
                const uint32_t from = (w_end & ~15u) + 2u * (uint32_t)lane;
                if (from < w_end) {
                    uint8_t *to = lds + L::W0 + wave * L::WAVE_W + last_row * (16 * F::PIECES) + (from - (block & ~15u));
                    *(uint16_t *)to = *(const __attribute__((address_space(1))) uint16_t *)(wbase + from);
                }
            }
        }
    };
    const uint8_t *my_w = lds + L::W0 + wave * L::WAVE_W + j * (16 * F::PIECES);
    auto my_block = [&](uint32_t b) {  // (blocks of whole pieces start at the beginning of their place)
        return F::BYTES % 16 != 0 ? my_w + ((my_row + b * (uint32_t)F::BYTES) & 15u) : my_w;
    };

    uint32_t number = 0;  // blocks of this K group so far
    // (looked up where it is needed: two of them in registers throughout would be spilled)
    auto look_up = [&](uint32_t t) {
        asm volatile("" : "+s"(t));
        return tile_at(t);
    };
    // CT: the token tiles that hold a token
    auto walk = [&](auto tiles_c, bool first_tile) {
    constexpr int CT = decltype(tiles_c)::value;
    const bool more = LOOP && tile + gridDim.x < tiles_all;  // another tile of this workgroup
    pl_float16 total[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            total[t][r] = 0.0f;
        }
    }
    pl_i32x16 X[CT], Y[CT];
    PlanesRaw<KIND> raw;
    const uint32_t a_at = a_group + (uint32_t)(j * 128 + 16 * (kh ^ (j & 7) ^ ((j >> 3) & 1)));

    // fp32 step of a block: y += a.d * (w.d * isum - w.dmin * msum)
    auto finish = [&](uint32_t number, int first, int last) {
        const uint8_t *sd = lds + L::S0 + (2 * kg + (number & 1u)) * L::SD;
        pl_half8 sums = {}, mins = {};
        if constexpr (F::MIN) {
            sums = *(const pl_half8 *)(sd + (32 * first + j) * 32 + 16 * kh);
            mins = raw.mins();
        }
#pragma unroll
        for (int t = first; t < last; ++t) {
            pl_float16 T = {};
            if constexpr (F::MIN) {
                T = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, mins, T, 0, 0, 0);
                if (t + 1 < last) {
                    sums = *(const pl_half8 *)(sd + (32 * (t + 1) + j) * 32 + 16 * kh);
                }
            }
            float4 da4 = *(const float4 *)(sd + L::SUMS + 4 * (32 * t + 4 * kh));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float da[4] = {da4.x, da4.y, da4.z, da4.w};
                if (q < 3) {
                    da4 = *(const float4 *)(sd + L::SUMS + 4 * (32 * t + 8 * (q + 1) + 4 * kh));
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * q + e;
                    float v = raw.d * (float)((Y[t][r] << F::SHIFT) + X[t][r]);
                    if constexpr (F::MIN) {
                        v = __builtin_fmaf(raw.ndmin, T[r], v);
                    }
                    total[t][r] = __builtin_fmaf(da[e], v, total[t][r]);
                }
            }
            asm volatile("" : "+v"(total[t]));  // done here: the sums of a block's products are not carried further
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Blocks kg, kg + KG, ... are this K group's.
    const uint32_t mine = nb > (uint32_t)kg ? (nb - (uint32_t)kg + KG - 1u) / KG : 0u;
    const uint32_t stages = 2u * ((nb + KG - 1u) / KG) + (KG > 1 ? 1u : 0u);  // barriers of every wavefront
    uint32_t passed = 0;
    pl_i32x4 lo[2], hi[2];
    // The weights of block b have been requested: unpacks its first step
    auto first_load = [&](uint32_t b) {
        bring_end(b);
        raw.load_half(my_block(b), 0, kh);
        raw.load_low(my_block(b), 0, 0, kh);
    };
    auto first_step = [&](uint32_t b) {
        const auto sc = raw.scale(0, 0);
#pragma unroll
        for (int piece = 0; piece < 4; ++piece) {
            int l, h;
            raw.planes(sc, 0, 0, piece, l, h);
            lo[0][piece] = l;
            hi[0][piece] = h;
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (first_tile && mine != 0) {
#pragma unroll
        for (int i = 0; i < L::DMA; ++i) {
            request_weights((uint32_t)kg, i);
        }
#pragma unroll
        for (int i = 0; i < CT * 4 / RG; ++i) {
            request_acts(2u * (uint32_t)kg, 0, i, offs(table, i));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (first_tile) {
        planes_barrier();
    }
    if (KG > 1 && kg >= KG / 2) {  // (wavefronts w and w + 4 share a SIMD)
        planes_barrier();
        ++passed;
    }
    for (uint32_t ib = 0; ib < mine; ++ib, ++number) {
        const uint32_t b = (uint32_t)kg + KG * ib;
        const bool last = ib + 1 == mine;
        // (behind the workgroup's last block some block is requested again rather than branched around)
        const uint32_t bn = !last ? b + KG : LOOP ? 0u : b;
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            constexpr int STEPS = 4 * CT, AHEAD = 2, LOADS = CT * 4 / RG;
            pl_i32x4 ring[AHEAD];
            uint32_t a_addr = 0;
            auto read_a = [&](int st) {
                const int s = st / CT, t = st % CT;
                if (t == 0) {
                    asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a_addr) : "s"(32 * PlanesRaw<KIND>::sub(s)), "v"(a_at));
                }
                ring[st % AHEAD] = *(const __attribute__((address_space(3))) pl_i32x4 *)(
                    (const lds_u8_t *)(uintptr_t)a_addr + hb * L::ACT + t * 4096);
            };
            if (hb == 0) {
                // (Q6_K's blocks are the largest and arrive last: read behind the fp32 step, 3 % of 1024 x 14336 x 4096)
                if (ib != 0 && F::BYTES % 16 == 0) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                if (F::BYTES % 16 == 0) {
                    first_load(b);
                }
                if (ib != 0) {
                    finish(number - 1u, CT / 2, CT);
                    if (F::BYTES % 16 != 0) {
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                }
                if (F::BYTES % 16 != 0) {
                    first_load(b);
                }
                first_step(b);
                raw.load_header(my_block(b), kh);
                if (LOOP && ib == 0 && more) {
                    if (p.act_index != nullptr) {  // read behind the end of this stage
                        const Tile next = look_up(tile + gridDim.x);
#pragma unroll
                        for (int i = 0; i < C / 2; ++i) {
                            const uint32_t t = 64u * i + (uint32_t)lane;
                            planes_dma4(lds_base + (uint32_t)(L::NEXT + wave * 128 * C + 256 * i),
                                        (const uint8_t *)(p.act_index + next.tok0), 4u * (t < next.toks ? t : next.toks - 1u));
                        }
                    }
                }
            }
            const uint8_t *block = my_block(b);
            if (LOOP && hb == 1 && last && more) {
                // from here on the requests are the next tile's
                const Tile next = look_up(tile + gridDim.x);
                fill_offs(table ^ 1u, [&](uint32_t t) {
                    const uint32_t in = t < next.toks ? t : next.toks - 1u;
                    return p.act_index != nullptr ? ((const uint32_t *)(lds + L::NEXT))[wave * (32 * C) + in] : next.tok0 + in;
                });
                table ^= 1u;
                aim(next);
            }
#pragma unroll
            for (int st = 0; st < AHEAD; ++st) {
                read_a(st);
            }
            uint32_t off = offs(table, 0);  // of the next load of the activations
            // Steps before fp32 steps of the other K group's wavefront on this SIMD, which fill what matrix instructions leave (2 - 3 %;
            // independent workgroups are 4 % slower with it)
            if (KG > 1) {
                __builtin_amdgcn_s_setprio(1);
            }
            __builtin_amdgcn_sched_barrier(0);
            typename PlanesRaw<KIND>::Scale sc = {};
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                const int s = st / CT, t = st % CT;
                const pl_i32x4 a = ring[st % AHEAD];
                const pl_i32x16 zero = {};
                X[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, lo[s & 1], hb == 0 && s == 0 ? zero : X[t], 0, 0, 0);
                Y[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, hi[s & 1], hb == 0 && s == 0 ? zero : Y[t], 0, 0, 0);
                if (st + AHEAD < STEPS) {
                    read_a(st + AHEAD);
                }
                // the next stage's codes, then scales and sums of this block: one load per place
                if (st < LOADS) {
                    request_acts(hb == 0 ? 2u * b + 1u : 2u * bn, hb ^ 1, st, off);
                    if (st + 1 < LOADS) {
                        off = offs(table, st + 1);
                    } else if (hb == 0) {
                        off = offs(table, APW);
                    } else if (LOOP && CT < C && last) {  // the next tile may have more of them
#pragma unroll
                        for (int i = CT; i < C; ++i) {
                            request_acts(2u * bn, hb ^ 1, i, offs(table, i));
                        }
                    }
                } else if (st == LOADS && hb == 0) {
                    request_scales(b, number, off);
                    if (F::MIN) {
                        off = offs(table, APW + 1);
                    }
                } else if (st == LOADS + 1 && hb == 0) {
                    request_sums(b, off);
                }
                // the operands of the next step, a quarter at a time
                const int hn = s < 3 ? hb : 1, sn = (s + 1) & 3;
                if (t == 0) {
                    if (s == 3 && hb == 0) {
                        if (RG == 4) {
                            store_block(number);
                        }
                        raw.load_half(block, hn, kh);
                    }
                    if (s == 1 || (s == 3 && hb == 0)) {
                        raw.load_low(block, hn, sn / 2, kh);
                    }
                }
                // The last bytes of this block have been read: its place is the next one's. (Waited for: the request alone does
                // not keep the new bytes behind a read that still queues for LDS.)
                constexpr int FREE = CT == 1 ? 2 : 3 * CT / 2;
                if (hb == 1 && st == FREE) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                if (hb == 1) {
#pragma unroll
                    for (int i = 0; i < L::DMA; ++i) {
                        if (st == FREE + i * CT / L::DMA) {
                            request_weights(bn, i);
                        }
                    }
                }
#pragma unroll
                for (int piece = 0; piece < 4; ++piece) {
                    // (not at once: the bytes are on their way from LDS)
                    if ((s < 3 || hb == 0) && (piece + 1 < 4 ? piece + 1 : 3) * CT / 4 == t) {
                        if (piece == 0) {
                            sc = raw.scale(hn, sn);
                        }
                        int l, h;
                        raw.planes(sc, hn, sn, piece, l, h);
                        lo[sn & 1][piece] = l;
                        hi[sn & 1][piece] = h;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (KG > 1) {
                __builtin_amdgcn_s_setprio(0);
            }
            if (hb == 0) {
                if (RG != 4) {  // (requested later than with four)
                    store_block(number);
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else {
                finish(number, 0, CT / 2);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L::DMA) : "memory");  // all but the weights, the last requests
            }
            planes_barrier();
            ++passed;
        }
    }
    // The first weights of the next tile (in front of the stores, which would be waited for too). Behind the last tile some were
    // requested all the same, and must not land in the LDS of the workgroup that comes after.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (mine != 0) {
        finish(number - 1u, CT / 2, CT);
    }
    if constexpr (KG > 1) {
        for (; passed < stages; ++passed) {
            planes_barrier();
        }
        static_assert(CT == C, "whole tiles");
    }
    if constexpr (KG == 4) {
        // the K groups' sums meet in LDS: each keeps a quarter of the outputs, half a token tile, and gives away the others
        static_assert(C == 2 && RG * 4 * 4 * 2048 <= L::W0, "the mail fits the codes' place");
        float4 *mail = (float4 *)lds + gw * 2048 + lane;  // [to][from][two][lane]
#pragma unroll
        for (int to = 0; to < 4; ++to) {
            if (to != kg) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const pl_float16 &v = total[to >> 1];
                    const int r = 8 * (to & 1) + 4 * q;
                    mail[512 * to + 128 * kg + 64 * q] = make_float4(v[r], v[r + 1], v[r + 2], v[r + 3]);
                }
            }
        }
        planes_barrier();
        float own[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float low = kg == 0 ? total[0][i] : total[0][8 + i], high = kg == 2 ? total[1][i] : total[1][8 + i];
            own[i] = kg < 2 ? low : high;
        }
#pragma unroll
        for (int from = 0; from < 4; ++from) {  // in the order of K
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float4 v = make_float4(own[4 * q], own[4 * q + 1], own[4 * q + 2], own[4 * q + 3]);
                if (from != kg) {
                    v = mail[512 * kg + 128 * from + 64 * q];
                }
                const float add[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    total[0][4 * q + e] = from == 0 ? add[e] : total[0][4 * q + e] + add[e];
                }
            }
        }
    }
    if constexpr (KG == 2) {
        // the K groups' sums meet in LDS: each gives the other half of its token tiles and keeps the other half
        static_assert(C % 2 == 0, "halves of whole token tiles");
        float *mail = (float *)lds + (size_t)wave * (C / 2) * 1024 + lane * 4;
        const float *from = (const float *)lds + (size_t)(wave ^ RG) * (C / 2) * 1024 + lane * 4;
#pragma unroll
        for (int t = 0; t < C / 2; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4 v;
                v.x = kg == 0 ? total[C / 2 + t][4 * q] : total[t][4 * q];
                v.y = kg == 0 ? total[C / 2 + t][4 * q + 1] : total[t][4 * q + 1];
                v.z = kg == 0 ? total[C / 2 + t][4 * q + 2] : total[t][4 * q + 2];
                v.w = kg == 0 ? total[C / 2 + t][4 * q + 3] : total[t][4 * q + 3];
                *(float4 *)(mail + (4 * t + q) * 256) = v;
            }
        }
        planes_barrier();
#pragma unroll
        for (int t = 0; t < C / 2; ++t) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = *(const float4 *)(from + (4 * t + q) * 256);
                const float add[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * q + e;
                    // (in the order of K: group 0's sum first)
                    total[t][r] = kg == 0 ? total[t][r] + add[e] : add[e] + total[C / 2 + t][r];
                }
            }
        }
    }

    if constexpr (GLU) {
        // Wavefronts gw and gw ^ 2 exchange halves of a token tile's sums and form the products of one half each. The second buffer of
        // the codes was read before the last barrier, and the next tile's codes come into it behind the next one.
        float4 *mail = (float4 *)(lds + L::ACT) + lane;  // [wavefront][two][lane]
        static_assert(RG * 2 * 1024 <= L::ACT, "half a token tile per wavefront");
        const bool second = gw >= 2;
#pragma unroll
        for (int t = 0; t < CT; ++t) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = second ? total[t][4 * q + e] : total[t][8 + 4 * q + e];
                }
                mail[128 * gw + 64 * q] = make_float4(v[0], v[1], v[2], v[3]);
            }
            planes_barrier();
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float4 v = mail[128 * (gw ^ 2) + 64 * q];
                const float other[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float mine = second ? total[t][8 + 4 * q + e] : total[t][4 * q + e];
                    const float gate = second ? other[e] : mine, up = second ? mine : other[e];
                    total[t][4 * q + e] = gate / (1.0f + expf(-gate)) * up;  // cpu_silu_f32 (elementwise_f32_scalar.c:11-13)
                }
            }
            planes_barrier();
        }
    }

    // lane (j, kh) holds weight row row0 + j for tokens 32 t + 8 (r / 4) + 4 kh + r % 4: 32 rows of a token per store
    const Tile cur = LOOP ? look_up(tile) : first;
    if (cur.row0 + (uint32_t)j >= p.M) {
        return;
    }
    const size_t m = cur.row0 + j, tok0 = cur.tok0;
    const uint32_t which = cur.which;
    uint32_t kh4 = 4u * (uint32_t)kh;
    asm volatile("" : "+v"(kh4));  // (the places of the outputs are not kept from tile to tile)
    // token tiles this wavefront stores, outputs of one
    constexpr int OUT = KG == 4 ? 1 : KG == 2 ? C / 2 : CT, REGS = KG == 4 || GLU ? 8 : 16;
    const uint32_t n0 = (uint32_t)(KG == 4 ? 16 * kg : KG == 2 ? 32 * kg * OUT : GLU ? 16 * (gw >> 1) : 0);
    const void *bias_p = p.bias[which];
    const bool has_bias = bias_p != nullptr;
    const float bias = !has_bias ? 0.0f : p.bias_is_f16 ? h2f(((const uint16_t *)bias_p)[m]) : ((const float *)bias_p)[m];
    if (!p.out_is_f16) {
        float *out = (float *)p.out[which] + tok0 * p.M + m;
#pragma unroll
        for (int t = 0; t < OUT; ++t) {
#pragma unroll
            for (int r = 0; r < REGS; ++r) {
                const uint32_t n = n0 + 32u * t + 8u * (r >> 2) + kh4 + (r & 3u);
                if (n < toks) {
                    out[(size_t)n * p.M] = has_bias ? total[t][r] + bias : total[t][r];
                }
            }
        }
    } else {
        uint16_t *out = (uint16_t *)p.out[which] + tok0 * p.M + m;
        const bool bias_first = p.bias_first != 0;
#pragma unroll
        for (int t = 0; t < OUT; ++t) {
#pragma unroll
            for (int r = 0; r < REGS; ++r) {
                const uint32_t n = n0 + 32u * t + 8u * (r >> 2) + kh4 + (r & 3u);
                if (n < toks) {
                    // without bias_first: round to the output type, then add the bias in it
                    const uint16_t first = f2h(has_bias && bias_first ? total[t][r] + bias : total[t][r]);
                    out[(size_t)n * p.M] = has_bias && !bias_first ? f2h(h2f(first) + bias) : first;
                }
            }
        }
    }
    };
    if constexpr (KG == 1) {
        for (bool first_tile = true;; first_tile = false) {
            const uint32_t tiles = (toks + 31u) / 32u;
            if (C >= 4 && tiles == 4) {
                walk(std::integral_constant<int, C < 4 ? 1 : 4>{}, first_tile);
            } else if (C >= 3 && tiles == 3) {
                walk(std::integral_constant<int, C < 3 ? 1 : 3>{}, first_tile);
            } else if (tiles == 2) {
                walk(std::integral_constant<int, 2>{}, first_tile);
            } else {
                walk(std::integral_constant<int, 1>{}, first_tile);
            }
            tile += gridDim.x;
            if (!LOOP || tile >= tiles_all) {
                return;
            }
            toks = look_up(tile).toks;
        }
    } else {
        walk(std::integral_constant<int, C>{}, true);
    }
}

// cols: tiles along the tokens, or work items at most. LOOP: as many workgroups as the chip holds at once (three per compute unit).
template <int KIND, int C, int KG, bool LOOP = false, int RG = 4, bool GLU = false>
static int planes_launch(marmot_hip_device *dev, GemmPlanesParams &p, size_t cols, unsigned weights) {
    MH_TRY(allow_large_lds(dev, (const void *)k_gemm_planes<KIND, C, KG, LOOP, RG, GLU>));
    constexpr size_t ROWS = GLU ? 64 : 32 * RG;
    p.row_tiles = (uint32_t)((p.M + ROWS - 1) / ROWS);
    p.col_tiles = (uint32_t)cols;
    p.weights = weights;
    const size_t tiles = (size_t)p.row_tiles * cols * weights;
    const size_t places = (size_t)dev->props.multiProcessorCount * 3;
    const dim3 grid((unsigned)(LOOP && tiles > places ? places : tiles));
    hipLaunchKernelGGL((k_gemm_planes<KIND, C, KG, LOOP, RG, GLU>), grid, dim3(64 * RG * KG),
                       (PlanesLds<KIND, C, KG, LOOP, RG>::BYTES), dev->stream, p);
    MH_HIP(hipGetLastError());
    return MARMOT_HIP_SUCCESS;
}

static bool planes_kind(int kind) {
    return kind == MARMOT_HIP_KIND_Q4_K || kind == MARMOT_HIP_KIND_Q5_K || kind == MARMOT_HIP_KIND_Q6_K;
}

// Which form (10 C + KG), or none (0), by the tiles a call has. The kernels of mh_gemm_i8.hip split K over workgroups where
// tiles are few, which pays the partial sums and wins while the chip is mostly empty; K groups in one workgroup want one
// tile per compute unit, and beyond that workgroups share one. Measured as time of the form over time of those kernels (Q6_K from
// form 42 on: of the fp16 tile that was there), whole calls in a row, about 400 sizes per format; tiles on 256 compute units:
//   24, 64 x 64, four K groups, up to a tile per compute unit. It takes a whole tile's time for any number of tokens in it.
//     Q6_K   up to 16 blocks from 65 tiles on 0.95 - 0.55, also at 17 tokens (66 tiles of 4 / 8 / 16 blocks 0.70, 0.83, 0.95)
//            17 - 23 blocks at 66 tiles 0.94 at 64 tokens, 1.03 at 17; 24 and more 1.03 - 1.31 (80 tiles 1.00 - 1.10), 88 tiles 0.88 - 0.98
//     Q4_K   up to 8 blocks 0.95 - 0.66. 16 blocks, 66 tiles with 33 / 64 tokens 1.08 / 0.99, 96 with 33 / 48 / 80 1.02, 1.00, 1.02,
//            128 with 33 / 80 0.98, 0.98; 12 blocks 1.01 / 0.92 and 0.93; beyond 16 blocks 160 tiles 1.03 - 1.09, 172 0.90
//     Q5_K   up to 8 blocks 0.98 - 0.65. 16 blocks, 66 tiles 1.12 / 1.03, 96 1.04, 1.01, 1.04, 128 1.01, 0.99; 12 blocks
//            1.09 / 0.98 and 0.98; beyond 16 blocks 160 tiles 1.00 - 1.04, 172 0.84
//            (One size goes the other way: 1024 x 4096 x 512, 128 tiles, 1.02 for both)
//   22, 128 x 64, two K groups, up to a tile per compute unit
//     Q6_K   0.77 (4 blocks) - 0.50
//     Q4_K   144 - 256 tiles of 4 / 8 / 10 / 12 / 14 / 16 blocks 1.14 - 1.06, 1.06 - 1.02, 1.04 - 1.01, 1.03 - 1.00, 1.02 - 0.99,
//            1.01 - 0.98, 32 and more 0.98 - 0.91
//     Q5_K   4 / 5 / 6 / 8 blocks 1.07 - 1.02, 1.04 - 1.00, 1.01 - 0.98, 0.99 - 0.96, 16 and more 0.93 - 0.85
//            (Both: up to three fifths of the compute units the split of more than 8 blocks fills the chip better)
//   42, 128 x 128, two K groups, up to a tile per compute unit (130 - 256 of them, 260 - 512 of 128 x 64)
//     Q6_K   0.76 - 0.46; the forms with one K group over it: 41 1.19 - 1.42, 21 1.01 - 1.54
//     Q4_K   0.96 - 0.67; 41 1.18 - 1.39, 21 1.00 - 1.26 but for 4 blocks (0.96 - 1.04) and 140 tokens (two tiles for little more
//            than one: 0.88 of 4 blocks, 0.91 of 16)
//     Q5_K   0.93 - 0.59; 41 1.17 - 1.37, 21 1.03 - 1.41 but for 140 and 200 tokens of 4 blocks (0.91, 0.95)
//   more tiles: Q6_K 41, 0.91 - 0.52 (21 against it 0.86 at 258 - 344 tiles of 128 x 128 and few blocks, 0.95 - 1.25 else); Q4_K, Q5_K 21,
//            0.99 - 0.68 (41 against it 0.97 - 1.21 and, Q5_K, 0.87 - 1.16)
// Several weights in one call: the other kernels take them one after the other, each split by itself, so the lines above that
// keep few blocks and badly filled tiles away are not theirs (three weights, other kernels / here: Q4_K 128 x 1024 x 4096 37.9 / 13.8
// us, 33 x 4096 x 2048 36.5 / 17.3, Q5_K 200 x 4096 x 512 40.9 / 21.3). Nor are they a call's that has no room for the partial sums of
// a split (a capture without an eager run before): no_split.
// Q4_K and Q5_K: where mh_gemm_int16.hip has a form of 256 x 128 for the call, that one is as fast or faster (1024 x 4096 x 14336
// Q4_K 156 us against 155, Q5_K 162 against 169; 1024 x 1024 x 8192 31 against 35).
static int planes_form(const marmot_hip_device *dev, int kind, size_t N, size_t M, size_t nb, size_t weights, bool no_split) {
    const size_t cus = (size_t)dev->props.multiProcessorCount;
    const size_t rows = (M + 127) / 128 * weights, rows64 = (M + 63) / 64 * weights;
    const size_t small = (N + 63) / 64 * rows, large = (N + 127) / 128 * rows, least = (N + 63) / 64 * rows64;
    const bool q6 = kind == MARMOT_HIP_KIND_Q6_K, q5 = kind == MARMOT_HIP_KIND_Q5_K;
    no_split = no_split || weights > 1;
    if (least <= cus) {
        const size_t used = N * rows64;  // 64 per tile if tokens fill them
        bool takes;
        if (no_split) {
            takes = q6 || nb <= 16 || 3 * least > 2 * cus;
        } else if (q6) {
            takes = nb <= 16 || 3 * least > cus || (nb < 24 && used >= 8 * cus);
        } else if (nb > 16) {
            takes = 3 * least > 2 * cus;
        } else {  // (16 blocks: from 16 and 19 tokens of a row tile per compute unit on)
            takes = nb <= 8 || 2 * used >= cus * (3 * nb - (q5 ? 10 : 16));
        }
        return 4 * least > cus && takes ? 24 : 0;
    }
    if (small <= cus) {
        return q6 || ((no_split || nb >= (q5 ? 6u : 14u)) && (nb <= 8 || 5 * small > 3 * cus)) ? 22 : 0;
    }
    return large <= cus ? 42 : q6 ? 41 : 21;
}

bool gemm_planes_applies(const marmot_hip_device *dev, int kind, size_t N, size_t K, size_t M, int weights,
                         const ActScratch &act, bool no_split) {
    if (dev->knobs.no_gemm_i8 || !planes_kind(kind) || K % QK_K != 0) {
        return false;
    }
    if ((((uintptr_t)act.qs) & 15) != 0 || act.kp % 16 != 0 || N * act.kp >= ((size_t)1 << 32) ||
        32 * (K / QK_K) * block_bytes(kind) >= ((size_t)1 << 31) || N > (size_t)65535 * 64) {
        return false;  // 32-bit lane offsets
    }
    return planes_form(dev, kind, N, M, K / QK_K, (size_t)weights, no_split) != 0;
}

// Rows x tokens of a tile, and the K groups of a workgroup (_k2, _k4)
#define PLANES_ROUTE(form)                                                                    \
    (KIND == MARMOT_HIP_KIND_Q4_K ? "mmq_q4_k_q8_k_int8_planes_" form                         \
     : KIND == MARMOT_HIP_KIND_Q5_K ? "mmq_q5_k_q8_k_int8_planes_" form : "mmq_q6_k_q8_k_int8_planes_" form)

template <int KIND>
static int planes_launch_kind(marmot_hip_device *dev, GemmPlanesParams &p, unsigned weights, bool no_split) {
    const int form = planes_form(dev, KIND, p.N, p.M, p.nb, weights, no_split);
    const unsigned t64 = (unsigned)((p.N + 63) / 64), t128 = (unsigned)((p.N + 127) / 128);
    if (form == 22) {
        set_route(PLANES_ROUTE("128x64_k2"));
        return planes_launch<KIND, 2, 2>(dev, p, t64, weights);
    }
    if (form == 24) {
        set_route(PLANES_ROUTE("64x64_k4"));
        return planes_launch<KIND, 2, 4, false, 2>(dev, p, t64, weights);
    }
    if (form == 42) {
        set_route(PLANES_ROUTE("128x128_k2"));
        return planes_launch<KIND, 4, 2>(dev, p, t128, weights);
    }
    if constexpr (KIND == MARMOT_HIP_KIND_Q6_K) {
        set_route(PLANES_ROUTE("128x128"));
        return planes_launch<KIND, 4, 1>(dev, p, t128, weights);
    } else {
        set_route(PLANES_ROUTE("128x64"));
        return planes_launch<KIND, 2, 1>(dev, p, t64, weights);
    }
}
#undef PLANES_ROUTE

int launch_gemm_planes(marmot_hip_device *dev, int kind, const WeightSet &ws, const ActScratch &act, size_t N, size_t K,
                       size_t M, int out_dtype, bool no_split) {
    GemmPlanesParams p = {};
    for (int i = 0; i < ws.count; ++i) {
        p.w[i] = (const uint8_t *)ws.w[i];
        p.out[i] = ws.out[i];
        p.bias[i] = ws.bias[i];
    }
    p.qs = act.qs;
    p.ad = act.d;
    p.sums = act.sums;
    p.kp = act.kp;
    p.N = N;
    p.M = M;
    p.nb = K / QK_K;
    p.bias_is_f16 = ws.bias_dtype == MARMOT_HIP_DTYPE_F16;
    p.bias_first = ws.bias_first ? 1 : 0;
    p.out_is_f16 = out_dtype == MARMOT_HIP_DTYPE_F16;
    const unsigned weights = (unsigned)ws.count;
    switch (kind) {
    case MARMOT_HIP_KIND_Q4_K:
        return planes_launch_kind<MARMOT_HIP_KIND_Q4_K>(dev, p, weights, no_split);
    case MARMOT_HIP_KIND_Q5_K:
        return planes_launch_kind<MARMOT_HIP_KIND_Q5_K>(dev, p, weights, no_split);
    default:
        return planes_launch_kind<MARMOT_HIP_KIND_Q6_K>(dev, p, weights, no_split);
    }
}

// ------------------------------------------------------------------ grouped (MoE)
bool gemm_planes_grouped_supported(const marmot_hip_device *dev, int kind, size_t rows, size_t K, size_t M, size_t max_items,
                                   const void *w0, const void *w1) {
    // (Q6_K rows are loaded from the 16-byte boundary below: the first one must not begin behind it. Tiles are counted in 32 bits.)
    return !dev->knobs.no_gemm_i8 && planes_kind(kind) && K % QK_K == 0 && rows * K < ((size_t)1 << 32) &&
           32 * (K / QK_K) * block_bytes(kind) < ((size_t)1 << 31) && M < ((size_t)1 << 31) &&
           2 * ((M + 63) / 64) * max_items < ((size_t)1 << 31) && ((((uintptr_t)w0) | ((uintptr_t)w1)) & 15) == 0;
}

int launch_gemm_planes_grouped(marmot_hip_device *dev, int kind, const void *d_w0, const void *d_w1, size_t expert_stride,
                               const ActScratch &act, const uint32_t *d_act_index, const int4 *d_items, const int *d_n_items,
                               size_t max_items, size_t K, size_t M, void *d_out0, void *d_out1, bool swiglu) {
    GemmPlanesParams p = {};
    p.w[0] = (const uint8_t *)d_w0;
    p.w[1] = (const uint8_t *)d_w1;
    p.out[0] = d_out0;
    p.out[1] = d_out1;
    p.qs = act.qs;
    p.ad = act.d;
    p.sums = act.sums;
    p.kp = act.kp;
    p.M = M;
    p.nb = K / QK_K;
    p.items = d_items;
    p.n_items = d_n_items;
    p.act_index = d_act_index;
    p.expert_stride = expert_stride;
    const unsigned weights = d_w1 != nullptr && !swiglu ? 2 : 1;
    if (swiglu) {  // silu(d_w0's outputs) * d_w1's, into d_out0
        switch (kind) {
        case MARMOT_HIP_KIND_Q4_K:
            return planes_launch<MARMOT_HIP_KIND_Q4_K, 2, 1, true, 4, true>(dev, p, max_items, 1);
        case MARMOT_HIP_KIND_Q5_K:
            return planes_launch<MARMOT_HIP_KIND_Q5_K, 2, 1, true, 4, true>(dev, p, max_items, 1);
        default:
            return planes_launch<MARMOT_HIP_KIND_Q6_K, 2, 1, true, 4, true>(dev, p, max_items, 1);
        }
    }
    // Items of 64 routes and three workgroups per compute unit: with items of 128 and two of them, 2048 tokens of 128 experts
    // take 401 us for 393 (Q4_K), 452 for 460 (Q6_K).
    switch (kind) {
    case MARMOT_HIP_KIND_Q4_K:
        return planes_launch<MARMOT_HIP_KIND_Q4_K, 2, 1, true>(dev, p, max_items, weights);
    case MARMOT_HIP_KIND_Q5_K:
        return planes_launch<MARMOT_HIP_KIND_Q5_K, 2, 1, true>(dev, p, max_items, weights);
    default:
        return planes_launch<MARMOT_HIP_KIND_Q6_K, 2, 1, true>(dev, p, max_items, weights);
    }
}

} // namespace mh
