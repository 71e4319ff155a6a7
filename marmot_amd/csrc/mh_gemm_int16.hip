// Long prompts with packed (Q8_K) activations: Q4_K / Q5_K weights x activation codes as a tiled GEMM on the fp16 matrix cores,
// both operands integers that fp16 holds exactly.
//
// Per 256-value block the reference forms (cpu_vec_dot_q{4,5}_k_q8_k, src/backends/cpu/ops/matmul/quantized/
// vec_dot_impl.h:689-787) y += a.d * (w.d * isum - w.dmin * msum) with isum = sum_j sc_j * (q_j . a_j) and msum = sum_j mn_j *
// (sum of a over sub-block j). Here the sub-block scale goes into the weight operand: sc * q is at most 63 * 15 = 945 (Q4_K)
// or 63 * 31 = 1953 (Q5_K), below 2048, so it is exact in fp16, and the activation codes (-127 .. 127) are too: ONE chain of
// v_mfma_f32_32x32x16_f16 per block gives isum in fp32 (exact below 2^24; from there on, up to 2^24.9 for Q4_K and 2^25.9 for
// Q5_K, where the reference rounds isum once, every instruction of the chain may round: at most 16 units in the last place),
// and one more instruction on the stored sums of 16 codes (at most 2032, exact) and the mins gives msum. fp32 work per output
// and block: three multiply(-add)s.
//
// What bounds it: vector instructions. A SIMD issues one per 4.2 clocks, a matrix instruction holds the issue port for 8 of
// its 32 clocks (measured with two wavefronts per SIMD), and per 32 x 32 outputs and block this kernel issues 17 matrix
// instructions beside 48 vector instructions of the fp32 step and its share of the unpacking (190 / 250 per 32 rows and block)
// and of the conversion of the activations. The int8 planes of mh_gemm_planes.hip take the same matrix time and as many
// vector instructions; what this kernel has is one workgroup of 256 x 128 outputs per compute unit, so it is taken where
// such tiles fill the chip well (x16_form).
//
// A wavefront owns 32 weight rows x 128 tokens: its lane (row j, half kh) unpacks, in registers, the bytes only it reads.
// Activations pass through LDS as fp16 (converted once per workgroup on the way from memory: code -> byte under the
// exponent of 1024 -> minus 1152), half a block (128 values) per stage, two stages, one barrier per stage; raw weight
// blocks go through a private LDS area of the wavefront (direct-to-LDS loads in whole 16-byte pieces, a block ahead).
// Everything that is not a matrix instruction is spread between them, a few instructions per step. The eight wavefronts of
// the workgroup meet at the same barriers, so the second wavefront of a SIMD does its fp32 step one stage late: without that
// both do it at once and the matrix core idles meanwhile.
// Measured (us of whole calls in a row, the quantization of 6 - 17 included; tile = k_gemm_q{4,5}k_q8k_tile of
// mh_gemm_i8.hip, flat = this kernel with flat loads of the activations, which count as LDS accesses too: an operand read then
// waited for memory; tokens x K x M):
//                          1000 x 4096 x 14336   2048 x 4096 x 4096
//   Q4_K tile / flat / now   193 / 163 / 155       118 / 94 / 88
//   Q5_K tile / flat / now   247 / 178 / 162       146 / 101 / 92
// 155 us with 7 of quantization are 790 TOP/s. The matrix instructions alone are about half of it at the clock the chip holds
// under them (1.7 - 1.9 GHz), the stores of the 57 MB of output 12, waits for the weights 12; what is left is unpacking and the
// conversion of the activations, which every row tile repeats.
#include "mh_rows.h"

#include <type_traits>

namespace mh {

typedef _Float16 x_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 x_half8 __attribute__((ext_vector_type(8)));
typedef float x_float16 __attribute__((ext_vector_type(16)));
typedef uint32_t x_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) x_u32x4 glb_u32x4_t;

struct GemmX16Params {
    const uint8_t *w[3];   // weights: M rows of nb blocks each
    const int8_t *qs;      // activation codes, rows of kp bytes
    const float *ad;       // activation block scales [rows][nb]
    const int16_t *sums;   // sums of 16 codes [rows][16 nb]
    size_t kp, N, M, nb;
    void *out[3];
    const void *bias[3];
    int bias_is_f16, bias_first, out_is_f16;
};

// Per format: bytes of a block, in whole 16-byte pieces
template <int KIND>
struct X16Format;
template <>
struct X16Format<MARMOT_HIP_KIND_Q4_K> {
    static constexpr int BYTES = Q4_K_BYTES, PIECES = 9;
};
template <>
struct X16Format<MARMOT_HIP_KIND_Q5_K> {
    static constexpr int BYTES = Q5_K_BYTES, PIECES = 11;
};

constexpr int X16_TILES = 4, X16_ROWS = 8;  // token tiles of a wavefront, wavefronts along the rows

template <int KIND>
struct X16Lds {
    static constexpr int C = X16_TILES, RG = X16_ROWS;
    static constexpr int ROWS = 64 / X16Format<KIND>::PIECES;             // whole rows per direct-to-LDS load
    static constexpr int DMA = (32 + ROWS - 1) / ROWS;                    // such loads of a wavefront per block
    static constexpr int ACT = 32 * C * 256;                              // one stage: 32 C tokens x 128 fp16
    static constexpr int W0 = 2 * ACT;
    static constexpr int WAVE_W = 32 * 16 * X16Format<KIND>::PIECES;
    static constexpr int S0 = W0 + RG * WAVE_W;                           // sums of the block as fp16: [token][16]
    static constexpr int SUMS = 32 * C * 32;
    static constexpr int SD = SUMS + 32 * C * 4;                          // then the activation scales [token]; two blocks
    static constexpr int BYTES = S0 + 2 * SD;
};

__device__ __forceinline__ x_half2 x_h2(uint32_t v) {
    return __builtin_bit_cast(x_half2, v);
}
__device__ __forceinline__ uint32_t x_u(x_half2 v) {
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ x_half2 x_splat(_Float16 v) {
    return x_half2{v, v};
}
// (v & mask) | magic in one instruction: two 32-bit literals do not fit one, so both sit in registers
struct X16Masks {
    uint32_t magic, low, high;
    __device__ __forceinline__ X16Masks() : magic(0x64006400u), low(0x000f000fu), high(0x00f000f0u) {
        asm volatile("" : "+v"(magic), "+v"(low), "+v"(high));
    }
};
__device__ __forceinline__ x_half2 x_and_or(uint32_t v, uint32_t mask, uint32_t magic) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(mask), "v"(magic));
    return x_h2(r);
}
// bytes 0, 2 (odd = 0) or 1, 3 (odd = 1) of v as fp16 1024 + byte
template <int ODD>
__device__ __forceinline__ x_half2 x_bytes(uint32_t v) {
    return x_h2(__builtin_amdgcn_perm(0x64646464u, v, ODD ? 0x04030401u : 0x04020400u));
}

__device__ __forceinline__ void x_put(x_half8 &op, int half, x_half2 e0, x_half2 e1) {
    op[4 * half] = e0[0];
    op[4 * half + 1] = e0[1];
    op[4 * half + 2] = e1[0];
    op[4 * half + 3] = e1[1];
}

// Weight operands of the 32 values (group g, lane half kh: values 32 g + 16 kh .. + 15 of half block hb), two
// instructions of 8 values; inside every four values the order is 0, 2, 1, 3 in both operands of the product. `raw`
// holds the lane's bytes of the block.
template <int KIND>
struct X16Raw;

template <>
struct X16Raw<MARMOT_HIP_KIND_Q4_K> {
    uint32_t sc_lo, sc_hi, mn_lo, mn_hi;
    float d, ndmin;
    uint4 q[4];
    x_half2 sc[4];
    __device__ __forceinline__ void header(const uint4 &hdr) {
        d = h2f((uint16_t)(hdr.x & 0xffffu));
        ndmin = -h2f((uint16_t)(hdr.x >> 16));
        asm volatile("" : "+v"(d), "+v"(ndmin));  // plain fp32 values: no mixed-precision multiply-adds later
        // 6-bit scales and mins as bytes (get_scale_min_k4, kquant_common.h:29-37)
        const uint32_t s_lo = hdr.y & 0x3f3f3f3fu;
        const uint32_t s_hi = (hdr.w & 0x0f0f0f0fu) | (((hdr.y >> 6) & 0x03030303u) << 4);
        mn_lo = hdr.z & 0x3f3f3f3fu;
        mn_hi = ((hdr.w >> 4) & 0x0f0f0f0fu) | (((hdr.z >> 6) & 0x03030303u) << 4);
        const x_half2 k = x_splat((_Float16)1024.0f);
        sc[0] = x_bytes<0>(s_lo) - k;  // scales 0, 2
        sc[1] = x_bytes<1>(s_lo) - k;  // scales 1, 3
        sc[2] = x_bytes<0>(s_hi) - k;
        sc[3] = x_bytes<1>(s_hi) - k;
    }
    uint4 hdr;
    __device__ __forceinline__ void load_head(const uint8_t *at, int kh) {
        hdr = *(const uint4 *)at;
        q[0] = *(const uint4 *)(at + 16 + 16 * kh);
        q[1] = *(const uint4 *)(at + 48 + 16 * kh);
    }
    __device__ __forceinline__ void load_tail(const uint8_t *at, int kh) {
        q[2] = *(const uint4 *)(at + 80 + 16 * kh);
        q[3] = *(const uint4 *)(at + 112 + 16 * kh);
    }
    __device__ __forceinline__ void decode_head(int) {
        header(hdr);
    }
    // mins as the fp16 operand of the sums: sum 8 kh + e belongs to sub-block 4 kh + e / 2
    __device__ __forceinline__ x_half8 mins(int kh) const {
        const uint32_t m = kh ? mn_hi : mn_lo;
        const x_half2 k = x_splat((_Float16)1024.0f);
        x_half8 r;
        const x_half2 m02 = x_bytes<0>(m) - k, m13 = x_bytes<1>(m) - k;
        r[0] = r[1] = m02[0];
        r[2] = r[3] = m13[0];
        r[4] = r[5] = m02[1];
        r[6] = r[7] = m13[1];
        return r;
    }
    __device__ __forceinline__ x_half2 scale(int sub) const {  // sub-block 0 .. 7 (compile time)
        const x_half2 pair = sc[(sub >> 2) * 2 + (sub & 1)];
        return x_splat((sub & 2) ? pair[1] : pair[0]);
    }
    __device__ __forceinline__ void operands(int hb, int g, int, int piece, const X16Masks &mk,
                                             x_half8 (&op)[2]) const {
        const int sub = 4 * hb + g;
        const uint4 &v = q[2 * hb + (g >> 1)];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        const x_half2 s = scale(sub);
        // the high nibbles stay where they are (16 q): their multiplier is sc / 16
        const x_half2 m = (g & 1) ? s * x_splat((_Float16)0.0625f) : s;
        const x_half2 c = m * x_splat((_Float16)-1024.0f);
        const uint32_t mask = (g & 1) ? mk.high : mk.low;
        const uint32_t x = w[piece];
        x_put(op[piece >> 1], piece & 1, __builtin_elementwise_fma(x_and_or(x, mask, mk.magic), m, c),
              __builtin_elementwise_fma(x_and_or(x >> 8, mask, mk.magic), m, c));
    }
};

template <>
struct X16Raw<MARMOT_HIP_KIND_Q5_K> {
    X16Raw<MARMOT_HIP_KIND_Q4_K> k4;
    float d, ndmin;
    uint4 h;  // fifth bits of this lane's 16 positions of every group: bit 4 hb + g
    uint4 h_next;
    __device__ __forceinline__ void load_head(const uint8_t *at, int kh) {
        k4.hdr = *(const uint4 *)at;
        h_next = *(const uint4 *)(at + 16 + 16 * kh);
        k4.q[0] = *(const uint4 *)(at + 48 + 16 * kh);
        k4.q[1] = *(const uint4 *)(at + 80 + 16 * kh);
    }
    __device__ __forceinline__ void load_tail(const uint8_t *at, int kh) {
        k4.q[2] = *(const uint4 *)(at + 112 + 16 * kh);
        k4.q[3] = *(const uint4 *)(at + 144 + 16 * kh);
    }
    __device__ __forceinline__ void decode_head(int kh) {
        k4.decode_head(kh);
        h = h_next;
        d = k4.d;
        ndmin = k4.ndmin;
    }
    __device__ __forceinline__ x_half8 mins(int kh) const {
        return k4.mins(kh);
    }
    __device__ __forceinline__ void operands(int hb, int g, int, int piece, const X16Masks &mk,
                                             x_half8 (&op)[2]) const {
        const int sub = 4 * hb + g;
        const uint4 &v = k4.q[2 * hb + (g >> 1)];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        const uint32_t hw[4] = {h.x, h.y, h.z, h.w};
        const x_half2 m = k4.scale(sub);
        const x_half2 c = m * x_splat((_Float16)-1024.0f);
        // four 5-bit values as bytes
        const uint32_t nib = (g & 1) ? (w[piece] >> 4) & 0x0f0f0f0fu : w[piece] & 0x0f0f0f0fu;
        const uint32_t b = nib | (((hw[piece] >> sub) & 0x01010101u) << 4);
        x_put(op[piece >> 1], piece & 1, __builtin_elementwise_fma(x_bytes<0>(b), m, c),
              __builtin_elementwise_fma(x_bytes<1>(b), m, c));
    }
};

// 64 x 16 bytes from base + voff (per lane) to LDS address lds_addr + 16 * lane (see dma16_to_lds). The s_nop separates the
// load from a vector instruction that may have written the scalar base right before it (v_readlane of a spilled scalar
// register): a memory instruction must not read such a register within five wait states, and the compiler does not look
// into the assembly to keep them apart.
__device__ __forceinline__ void x16_dma(uint32_t lds_addr, const uint8_t *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void x16_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int KIND>
__global__ __launch_bounds__(64 * X16_ROWS, 2) void k_gemm_x16(const GemmX16Params p) {
    using F = X16Format<KIND>;
    using L = X16Lds<KIND>;
    constexpr int C = X16_TILES, RG = X16_ROWS;
    constexpr int THREADS = 64 * RG, TOK = 32 * C;
    constexpr int APT = 8 * TOK / THREADS;  // 16-byte pieces of codes per thread and stage
    static_assert(8 * TOK % THREADS == 0, "whole pieces per thread");
    warm_kernel_arguments<sizeof(GemmX16Params)>();
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int which = blockIdx.z;
    const size_t row0 = (size_t)blockIdx.x * (32 * RG) + 32 * wave;  // this wavefront's first weight row
    const uint8_t *w = p.w[which];
    const size_t tok0 = (size_t)blockIdx.y * TOK;  // first output row
    const uint32_t toks = (uint32_t)(p.N - tok0 < (size_t)TOK ? p.N - tok0 : (size_t)TOK);
    // ---- activations: piece `tid + THREADS i` of a stage is 16 codes (part q % 8) of token q / 8; rows beyond the last
    // token re-read it and are never stored
    uint32_t a_row[APT];
    uint32_t a_lds[APT];  // where its 2 x 8 fp16 values go: chunk c of a token sits in slot c ^ (token % 16)
#pragma unroll
    for (int i = 0; i < APT; ++i) {
        const uint32_t q = (uint32_t)(tid + THREADS * i), t = q >> 3, part = q & 7u;
        const uint32_t row = (uint32_t)tok0 + (t < toks ? t : toks - 1u);
        a_row[i] = row * (uint32_t)p.kp + 16u * part;
        a_lds[i] = t * 256u + 16u * ((2u * part) ^ (t & 15u));
    }
    // sums and scales of a block: thread's piece (tokens wrap around: several threads then write the same bytes)
    const uint32_t s_tok = (uint32_t)(tid >> 1) % TOK, d_tok = (uint32_t)tid % TOK;
    const uint32_t s_row = (uint32_t)tok0 + (s_tok < toks ? s_tok : toks - 1u);
    const uint32_t d_row = (uint32_t)tok0 + (d_tok < toks ? d_tok : toks - 1u);
    const uint32_t s_off = s_row * (uint32_t)p.nb * 32u + 16u * (tid & 1);
    const uint32_t d_off = d_row * (uint32_t)p.nb * 4u;

    // ---- weights: load i of a block brings rows ROWS i .. + ROWS - 1 of the wavefront: lane l the 16-byte piece l % PIECES
    // of row l / PIECES; lanes behind the last row and rows behind the matrix re-read a row before.
    const uint32_t row_bytes = (uint32_t)p.nb * F::BYTES;
    const uint32_t rows = (uint32_t)(row0 < p.M ? (p.M - row0 < 32 ? p.M - row0 : 32) : 0);
    const uint8_t *wbase = w + (row0 < p.M ? row0 : p.M - 1) * row_bytes;
    wbase = uniform_pointer(wbase);
    const uint32_t last_row = rows == 0 ? 0 : rows - 1u;
    const uint32_t w_r = (uint32_t)lane / F::PIECES < L::ROWS ? (uint32_t)lane / F::PIECES : L::ROWS - 1u;
    const uint32_t w_piece = 16u * ((uint32_t)lane - F::PIECES * w_r < F::PIECES ? (uint32_t)lane - F::PIECES * w_r : F::PIECES - 1u);
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_u8_t *)lds;
    const uint32_t w_lds = lds_base + (uint32_t)(L::W0 + wave * L::WAVE_W);
    const uint32_t w_first = w_r * row_bytes + w_piece;
    const uint32_t w_last = last_row * row_bytes + w_piece;
    auto request_weights = [&](uint32_t b, int i) {
        uint32_t at = w_first;
        asm volatile("" : "+v"(at));  // formed at each load: kept in registers, the L::DMA offsets would be spilled
        at += (uint32_t)i * (L::ROWS * row_bytes);
        at = at < w_last ? at : w_last;
        const uint32_t to = w_lds + (uint32_t)(i * L::ROWS * 16 * F::PIECES);
        const uint8_t *base = wbase + (size_t)b * F::BYTES;
        // (the launcher checks that rows of whole 16-byte pieces start on 16-byte boundaries)
        // lanes without a row write nothing: the place behind the rows of this load belongs to the next one
        if ((uint32_t)lane < (i + 1 < L::DMA ? L::ROWS : 32 - L::ROWS * (L::DMA - 1)) * F::PIECES) {
            x16_dma(to, base, at);
        }
    };
    const uint8_t *my_w = lds + L::W0 + wave * L::WAVE_W + j * (16 * F::PIECES);

    x_u32x4 a_next[APT];
    x_u32x4 s_next;
    float d_next = 0.0f;
    auto request_acts = [&](uint32_t stage) {
        // The asm keeps a scalar base + 32-bit lane offsets, not a 64-bit address per lane and load; the pointer says that
        // it is global memory, since a flat load also counts as an LDS access and every operand read then waits for it.
        glb_u8_t *base = (glb_u8_t *)p.qs + (size_t)stage * 128u;
        asm("" : "+s"(base));
#pragma unroll
        for (int i = 0; i < APT; ++i) {
            a_next[i] = *(const glb_u32x4_t *)(base + (size_t)a_row[i]);
        }
    };
    auto request_block = [&](uint32_t b) {
        {
            glb_u8_t *sums = (glb_u8_t *)p.sums + (size_t)b * 32u;
            asm("" : "+s"(sums));
            s_next = *(const glb_u32x4_t *)(sums + (size_t)s_off);
        }
        glb_u8_t *ad = (glb_u8_t *)p.ad + (size_t)b * 4u;
        asm("" : "+s"(ad));
        d_next = *(const __attribute__((address_space(1))) float *)(ad + (size_t)d_off);
    };
    auto store_acts = [&](int buffer, int i) {
        uint8_t *stage = lds + buffer * L::ACT;
        const x_half2 k = x_splat((_Float16)1152.0f);
        const uint32_t v[4] = {a_next[i].x ^ 0x80808080u, a_next[i].y ^ 0x80808080u, a_next[i].z ^ 0x80808080u,
                               a_next[i].w ^ 0x80808080u};
        uint32_t e[8];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            e[2 * c] = x_u(x_bytes<0>(v[c]) - k);
            e[2 * c + 1] = x_u(x_bytes<1>(v[c]) - k);
        }
        *(uint4 *)(stage + a_lds[i]) = make_uint4(e[0], e[1], e[2], e[3]);
        *(uint4 *)(stage + (a_lds[i] ^ 16u)) = make_uint4(e[4], e[5], e[6], e[7]);
    };
    auto store_block = [&](uint32_t b) {
        uint8_t *sd = lds + L::S0 + (b & 1u) * L::SD;
        {
            const uint32_t v[4] = {s_next.x, s_next.y, s_next.z, s_next.w};
            uint32_t e[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                e[c] = x_u(x_half2{(_Float16)(int16_t)(v[c] & 0xffffu), (_Float16)(int16_t)(v[c] >> 16)});
            }
            *(uint4 *)(sd + s_tok * 32u + 16u * (tid & 1)) = make_uint4(e[0], e[1], e[2], e[3]);
        }
        *(float *)(sd + L::SUMS + d_tok * 4u) = d_next;
    };

    float total[C][16];
#pragma unroll
    for (int t = 0; t < C; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            total[t][r] = 0.0f;
        }
    }
    const uint32_t nb = (uint32_t)p.nb;
    const X16Masks mk;
    // A operand of (g, kh, i): chunk 4 g + 2 kh + i of token 32 t + j. One address register: the others differ from it in
    // bits 4 .. 7 and are formed where they are used (kept out of registers by the volatile asm).
    const uint32_t a_at = lds_base + (uint32_t)(j * 256 + 16 * ((2 * kh) ^ (j & 15)));
    // fp32 step of a block, token tile t: y += a.d * (w.d * isum - w.dmin * msum)
    x_float16 P[C];
    float d = 0.0f, ndmin = 0.0f;
    x_half8 mins = {};
    auto finish = [&](uint32_t b) {
        const uint8_t *sd = lds + L::S0 + (b & 1u) * L::SD;
        x_half8 sums = *(const x_half8 *)(sd + j * 32 + 16 * kh);
#pragma unroll
        for (int t = 0; t < C; ++t) {
            x_float16 T = {};
            T = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, mins, T, 0, 0, 0);
            if (t + 1 < C) {
                sums = *(const x_half8 *)(sd + (32 * (t + 1) + j) * 32 + 16 * kh);
            }
            float4 da4[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                da4[q] = *(const float4 *)(sd + L::SUMS + 4 * (32 * t + 8 * q + 4 * kh));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float da[4] = {da4[q].x, da4[q].y, da4[q].z, da4[q].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * q + e;
                    const float v = __builtin_fmaf(ndmin, T[r], d * P[t][r]);
                    total[t][r] = __builtin_fmaf(da[e], v, total[t][r]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Two wavefronts share a SIMD and its matrix core. With the fp32 step at the same place in both, the matrix core
    // would idle during it; so the second half of the workgroup's wavefronts does it one stage later, while the first
    // half's matrix instructions run.
    X16Raw<KIND> raw;
#pragma unroll
    for (int i = 0; i < L::DMA; ++i) {
        request_weights(0, i);
    }
    request_acts(0);
    request_block(0);
#pragma unroll
    for (int i = 0; i < APT; ++i) {
        store_acts(0, i);
    }
    store_block(0);
    request_acts(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    raw.load_head(my_w, kh);
    x16_barrier();
    auto walk = [&](auto late_c) {
    constexpr bool LATE = decltype(late_c)::value;
    for (uint32_t b = 0; b < nb; ++b) {
        const uint32_t bn = b + 1 < nb ? b + 1 : b;  // (the last block is requested again rather than branched around)
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            // Steps (g, i, t): one matrix instruction each, consecutive ones on different accumulators. The A operand
            // of a step is read AHEAD steps before it, the weight operands of group g + 1 are unpacked, a quarter at a time,
            // between the steps of group g. AHEAD is what the register budget carries without spills.
            constexpr int STEPS = 8 * C, AHEAD = 3;
            x_half8 ring[AHEAD];
            uint32_t a_addr[2];
            auto read_a = [&](int s) {
                const int g = s / (2 * C), t = s % C, i = (s / C) & 1;
                if (t == 0) {
                    asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a_addr[i]) : "s"(16 * (4 * g + i)), "v"(a_at));
                }
                ring[s % AHEAD] = *(const __attribute__((address_space(3))) x_half8 *)(
                    (const lds_u8_t *)(uintptr_t)a_addr[i] + hb * L::ACT + t * 8192);
            };
            x_half8 op[2][2];
            if (hb == 0 && LATE && b != 0) {
                finish(b - 1);
            }
            if (hb == 0) {
                raw.load_tail(my_w, kh);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) {
                read_a(s);
            }
            if (hb == 0) {
                raw.decode_head(kh);
                d = raw.d;
                ndmin = raw.ndmin;
                mins = raw.mins(kh);
            }
#pragma unroll
            for (int piece = 0; piece < 4; ++piece) {
                raw.operands(hb, 0, kh, piece, mk, op[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int g = s / (2 * C), t = s % C, i = (s / C) & 1;
                const x_half8 a = ring[s % AHEAD];
                const x_float16 zero = {};
                P[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, op[g & 1][i], hb == 0 && g == 0 && i == 0 ? zero : P[t], 0, 0, 0);
                if (s + AHEAD < STEPS) {
                    read_a(s + AHEAD);
                }
                if (g < 3) {
#pragma unroll
                    for (int piece = 0; piece < 4; ++piece) {
                        if (piece * 2 * C / 4 == s % (2 * C)) {
                            raw.operands(hb, g + 1, kh, piece, mk, op[(g + 1) & 1]);
                        }
                    }
                }
                // Between the steps: the wavefront's next weight block (its area is free once the block is in registers: the
                // reads were issued before the operands of step 0), the codes of the next stage into the other buffer (free
                // since the barrier that ended the previous stage), then the requests for the stage after it.
                const auto at = [&](int x) { return s == x * C / 4; };
                if (hb == 0) {
#pragma unroll
                    for (int i = 0; i < L::DMA; ++i) {
                        if (at(2 + i * 10 / L::DMA)) {
                            request_weights(bn, i);
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < APT; ++i) {
                    if (at(13 + 2 * i)) {
                        store_acts(hb ^ 1, i);
                    }
                }
                if (hb == 0 && at(17)) {
                    store_block(b);
                }
                if (at(19)) {
                    if (hb == 1) {
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the weight block, requested before the codes
                    }
                    request_acts(2 * bn + hb);
                    if (hb == 0) {
                        request_block(bn);
                    }
                }
                if (hb == 1 && at(24)) {
                    raw.load_head(my_w, kh);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (hb == 1 && !LATE) {
                finish(b);
            }
            x16_barrier();
        }
    }
    if (LATE) {
        finish(nb - 1);
    }
    };
    if (wave >= 4) {
        walk(std::true_type{});
    } else {
        walk(std::false_type{});
    }

    // lane (j, kh) holds weight row row0 + j for tokens 32 t + 8 (r / 4) + 4 kh + r % 4: 32 rows of a token per store
    if ((uint32_t)j >= rows) {
        return;
    }
    const size_t m = row0 + j;
    const void *bias_p = p.bias[which];
    const bool has_bias = bias_p != nullptr;
    const float bias = !has_bias ? 0.0f : p.bias_is_f16 ? h2f(((const uint16_t *)bias_p)[m]) : ((const float *)bias_p)[m];
    if (!p.out_is_f16) {
        float *out = (float *)p.out[which] + tok0 * p.M + m;
#pragma unroll
        for (int t = 0; t < C; ++t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t n = (uint32_t)(32 * t + 8 * (r >> 2) + 4 * kh + (r & 3));
                if (n < toks) {
                    out[(size_t)n * p.M] = has_bias ? total[t][r] + bias : total[t][r];
                }
            }
        }
    } else {
        uint16_t *out = (uint16_t *)p.out[which] + tok0 * p.M + m;
        const bool bias_first = p.bias_first != 0;
#pragma unroll
        for (int t = 0; t < C; ++t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t n = (uint32_t)(32 * t + 8 * (r >> 2) + 4 * kh + (r & 3));
                if (n < toks) {
                    // without bias_first: round to the output type, then add the bias in it
                    const uint16_t first = f2h(has_bias && bias_first ? total[t][r] + bias : total[t][r]);
                    out[(size_t)n * p.M] = has_bias && !bias_first ? f2h(h2f(first) + bias) : first;
                }
            }
        }
    }
}

// Whether a call takes this kernel. A compute unit takes as long for one 256 x 128 tile as for three rounds of 128 x 64 tiles
// (2048 x 4096 x 4096, one large tile per compute unit: 85 us; four rounds of small ones: 107 us in mh_gemm_i8.hip, 101 us in
// mh_gemm_planes.hip), so the large tile has to save a round.
static bool x16_form(const marmot_hip_device *dev, size_t N, size_t M, size_t weights) {
    const size_t cus = (size_t)dev->props.multiProcessorCount;
    const size_t small = ((N + 63) / 64) * ((M + 127) / 128) * weights;
    const size_t large = ((N + 127) / 128) * ((M + 255) / 256) * weights;
    return 3 * ((large + cus - 1) / cus) < (small + cus - 1) / cus;
}

bool gemm_x16_applies(const marmot_hip_device *dev, int kind, size_t N, size_t K, size_t M, int weights,
                      const ActScratch &act) {
    if (dev->knobs.no_gemm_i8 || (kind != MARMOT_HIP_KIND_Q4_K && kind != MARMOT_HIP_KIND_Q5_K) || K % QK_K != 0) {
        return false;
    }
    if ((((uintptr_t)act.qs) & 15) != 0 || act.kp % 16 != 0 || N * act.kp >= ((size_t)1 << 32) ||
        32 * (K / QK_K) * block_bytes(kind) >= ((size_t)1 << 31) || N > (size_t)65535 * 64) {
        return false;  // 32-bit lane offsets
    }
    return x16_form(dev, N, M, (size_t)weights);
}

template <int KIND>
static int x16_launch(marmot_hip_device *dev, const GemmX16Params &p, unsigned weights) {
    MH_TRY(allow_large_lds(dev, (const void *)k_gemm_x16<KIND>));
    const dim3 grid((unsigned)((p.M + 32 * X16_ROWS - 1) / (32 * X16_ROWS)), (unsigned)((p.N + 127) / 128), weights);
    hipLaunchKernelGGL((k_gemm_x16<KIND>), grid, dim3(64 * X16_ROWS), X16Lds<KIND>::BYTES, dev->stream, p);
    MH_HIP(hipGetLastError());
    set_route(KIND == MARMOT_HIP_KIND_Q4_K ? "mmq_q4_k_q8_k_fp16_tile_256x128" : "mmq_q5_k_q8_k_fp16_tile_256x128");
    return MARMOT_HIP_SUCCESS;
}

int launch_gemm_x16(marmot_hip_device *dev, int kind, const WeightSet &ws, const ActScratch &act, size_t N, size_t K,
                    size_t M, int out_dtype) {
    GemmX16Params p = {};
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
    return kind == MARMOT_HIP_KIND_Q4_K ? x16_launch<MARMOT_HIP_KIND_Q4_K>(dev, p, weights)
                                        : x16_launch<MARMOT_HIP_KIND_Q5_K>(dev, p, weights);
}

} // namespace mh
