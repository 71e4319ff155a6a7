// Paged attention (marmot_paged_attention; CPU counterpart cpu_paged_attention_impl,
// src/backends/cpu/ops/paged_attention/paged_attention_ref.c:573-1082): every token's new key / value rows are written
// into the paged cache at the token's kv_slot, then every (token, query head) attends over positions 0 .. pos of its
// sequence through the block table.
//
// Attention kernel: one workgroup of 16 groups of 16 lanes per (token, up to four query heads of one key / value
// head). A group walks the positions g, g + 16, g + 32, ...: its 16 lanes split the head dimension (a lane holds EPL consecutive values of the
// query, of the running output and of each key / value row, so a row is read as one contiguous run by the group), the
// dot product is reduced inside the group with data-parallel-primitive moves, and the group keeps its own running
// maximum, sum and output (online softmax). The groups meet in LDS at the end. All arithmetic is fp32 like the
// reference's; only the order of the sums differs (per group instead of per block of positions). Rows are read with
// 16-byte loads when the head dimension is exactly 16 x EPL values with unit stride, element by element otherwise.
// A token whose sequence slot or cache block is out of range is skipped (the host rejects such calls when it may read
// the metadata, like the reference).
#include "mh_common.h"

#include <math.h>

namespace mh {

constexpr uint32_t PA_NO_BLOCK = 0xFFFFFFFFu;

struct PaParams {
    uint32_t token_count, layer_idx, num_q_heads, num_kv_heads, head_dim, block_size;
    float scale;
    int act_dtype, kv_dtype;
    const uint32_t *meta;
    size_t meta_stride[2];
    const void *q, *k_new, *v_new;
    size_t q_stride[3], k_stride[3], v_stride[3];
    void *kv_k, *kv_v;
    size_t kv_stride[5];
    size_t kv_blocks, kv_layers;
    const uint32_t *table;
    size_t table_stride[2];
    size_t max_seqs, max_blocks;
    void *out;
    size_t out_stride[3];
    uint32_t shift, mask, group;
    int q_vec, kv_vec;  // 16-byte loads of the query / of the cache rows
    int *flag;          // metadata check: 1 + index of an offending token (maximum)
    float *k_scale, *v_scale;  // FLOAT8_E4M3 cache: scales [blocks][layers][kv heads] at scale_stride
    size_t scale_stride[3];
    uint32_t *new_kmax, *new_vmax;  // scratch [blocks][kv heads]: largest new magnitudes as float bits
    uint32_t *min_off;              // scratch [blocks]: first offset this call writes (block_size = untouched)
    uint32_t *claim;                // scratch [blocks][kv heads]: the token whose workgroup rescales the block (~0 = none yet)
    uint32_t splits;    // workgroups along the history of one (token, heads) pair
    float *partial;     // splits > 1: [token][query head][partial_splits][2 + head_dim]: maximum, sum, unnormalized output
    uint32_t partial_splits;  // the largest split count of the call: every (token, head) pair has room for any kernel
    uint32_t tile_tokens;  // tokens per tile of the prompt kernel (k_pa_prompt), 0 = not launched
    uint32_t tile_splits;  // prompt kernel: workgroups along a history
    uint32_t long_from;    // prompt kernel: positions the longest history of the call has at least
    uint32_t *tiled;       // scratch [token_count]: 1 = the prompt kernel takes the token, 2 = a token in share_splits shares
    uint32_t share_splits; // workgroups along the history of a token by itself in a call whose runs are in tiles
    int out_vec;           // prompt kernel: FLOAT32 output rows at 16-byte boundaries
};

// The prompt kernel takes a token when its tile (tile_tokens consecutive tokens of the call) holds at least PA_RUN_MIN
// tokens of the token's sequence, that sequence has long_from / 2 positions or more and some sequence of the call has
// long_from; the other kernels of the call take the rest. A pass over a history costs the prompt kernel the same for one
// token as for the whole tile, so the decode tokens of a mixed call stay where every token has workgroups of its own.
// The lengths are those of the tile's tokens and of 64 probes, tokens spread evenly over the call (its last one among
// them): what the block table has room for says nothing about a call. The launch that writes the cache finds the answer
// and leaves it in p.tiled (in the workgroups of the other kernels it cost 12 - 20 us of 256-token calls).
constexpr uint32_t PA_RUN_MIN = 4;

// positions that token t sees, none behind the table's last block
__device__ __forceinline__ uint32_t pa_visible(const PaParams &p, uint32_t position) {
    const uint64_t limit = (uint64_t)p.max_blocks << p.shift;
    const uint32_t len = position + 1u;
    return len < limit ? len : (uint32_t)limit;
}
__device__ __forceinline__ uint32_t pa_probe(const PaParams &p, uint32_t i) {
    const uint32_t step = (p.token_count + 63u) / 64u, t = (i + 1u) * step - 1u;
    return t < p.token_count ? t : p.token_count - 1u;
}

// Whole wavefront: 1 = the prompt kernel takes token t. 2 = not a run, beside one that it takes, and a long history: the
// few tokens that are left do not fill the chip, so their histories are split (100 tokens over 4000 positions and 16 decode
// tokens over 2000: 110 us unsplit). Else 0.
__device__ __forceinline__ uint32_t pa_in_run(const PaParams &p, uint32_t t, uint32_t seq) {
    const uint32_t first = t / p.tile_tokens * p.tile_tokens, lane = threadIdx.x & 63u;
    const size_t probe = (size_t)pa_probe(p, lane) * p.meta_stride[0];
    const uint32_t probe_seq = p.meta[probe], probe_len = pa_visible(p, p.meta[probe + p.meta_stride[1]]);
    bool far = probe_seq < p.max_seqs && probe_len >= p.long_from;
    bool own = probe_seq == seq && probe_len >= p.long_from / 2u;
    uint32_t same = 0;
    for (uint32_t i = 0; i < p.tile_tokens; i += 64u) {
        const uint32_t other = first + i + lane;
        const bool inside = i + lane < p.tile_tokens && other < p.token_count;
        const size_t at = (size_t)(inside ? other : t) * p.meta_stride[0];
        const uint32_t s = p.meta[at], len = pa_visible(p, p.meta[at + p.meta_stride[1]]);
        same += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(inside && s == seq));
        far = far || (s < p.max_seqs && len >= p.long_from);
        own = own || (s == seq && len >= p.long_from / 2u);
    }
    if (seq >= p.max_seqs || __builtin_amdgcn_ballot_w64(far) == 0 || __builtin_amdgcn_ballot_w64(own) == 0) {
        return 0u;
    }
    return same >= PA_RUN_MIN ? 1u : 2u;
}

// marmot_f32_to_bf16_ref / marmot_bf16_to_f32_ref (src/utils/dtype_ref.c:86-104): round to nearest even on the bits
__device__ __forceinline__ uint16_t pa_f2bf(float v) {
    const uint32_t bits = __float_as_uint(v);
    return (uint16_t)((bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float pa_bf2f(uint16_t h) {
    return __uint_as_float((uint32_t)h << 16);
}

// The reference's e4m3 (marmot_fp8_dequantize / marmot_fp8_quantize with 4 exponent bits, 3 mantissa bits, bias 7,
// no infinity, largest finite value 240: src/utils/dtype_ref.c:118-212).
__device__ __forceinline__ float pa_fp8_to_f32(uint32_t c) {
    const uint32_t field = (c >> 3) & 15u, mant = c & 7u, sign = (c & 0x80u) << 24;
    if (field == 15u) {
        return __uint_as_float(0x7fc00000u);
    }
    if (field == 0u) {
        return __uint_as_float(__float_as_uint((float)mant * 0.001953125f) | sign);  // mant / 8 * 2^-6
    }
    return __uint_as_float(sign | ((field + 120u) << 23) | (mant << 20));  // (1 + mant / 8) * 2^(field - 7)
}

__device__ __forceinline__ uint32_t pa_f32_to_fp8(float value) {
    if (value != value) {
        return 0x79u;
    }
    const uint32_t sign = value < 0.0f ? 0x80u : 0u;
    const float mag = fabsf(value);
    if (mag > 240.0f) {  // infinity included
        return sign | 0x77u;
    }
    if (mag == 0.0f) {
        return sign;
    }
    int e;
    float m = frexpf(mag, &e);  // mag = m * 2^e, m in [0.5, 1)
    m *= 2.0f;
    e -= 1;
    int field = e + 7;
    if (field > 0 && field < 15) {
        int r = (int)rintf((m - 1.0f) * 8.0f);  // nearest, ties to even
        if (r == 8) {
            r = 0;
            field += 1;
            if (field >= 15) {
                return sign | 0x77u;
            }
        }
        return sign | ((uint32_t)field << 3) | (uint32_t)(r & 7);
    }
    int r = (int)rintf(ldexpf(mag, 9));  // below the smallest normal 2^-6: multiples of 2^-9, never rounded up into
    if (r == 0) {                        // the normal range
        return sign;
    }
    return sign | (uint32_t)(r > 7 ? 7 : r);
}

// cpu_paged_attention_fp8_quant / _dequant / _scale_from_max (paged_attention_ref.c:142-163)
__device__ __forceinline__ uint32_t pa_fp8_quant(float value, float scale) {
    return scale > 0.0f ? pa_f32_to_fp8(value / scale) : 0u;
}
__device__ __forceinline__ float pa_fp8_dequant(uint32_t c, float scale) {
    return scale > 0.0f ? pa_fp8_to_f32(c) * scale : 0.0f;
}

__device__ __forceinline__ float pa_load(const void *data, int dtype, size_t i) {
    if (dtype == MARMOT_HIP_DTYPE_F8_E4M3) {  // the code's value; the caller applies the block's scale
        return pa_fp8_to_f32(((const uint8_t *)data)[i]);
    }
    if (dtype == MARMOT_HIP_DTYPE_F16) {
        return h2f(((const uint16_t *)data)[i]);
    }
    if (dtype == MARMOT_HIP_DTYPE_BF16) {
        return pa_bf2f(((const uint16_t *)data)[i]);
    }
    return ((const float *)data)[i];
}

__device__ __forceinline__ void pa_store(void *data, int dtype, size_t i, float v) {
    if (dtype == MARMOT_HIP_DTYPE_F16) {
        ((uint16_t *)data)[i] = f2h(v);
    } else if (dtype == MARMOT_HIP_DTYPE_BF16) {
        ((uint16_t *)data)[i] = pa_f2bf(v);
    } else {
        ((float *)data)[i] = v;
    }
}

// exp(x) for x <= 0 (softmax weights and rescaling factors): the hardware's base-2 exponential, about 2 units in the
// last place -- far inside the tolerance of the output, and a fraction of the library routine's instructions
__device__ __forceinline__ float pa_exp(float x) {
    return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f);
}

// A query row is split into FLOAT16 parts after an exact scaling: by the power of two that brings its largest magnitude
// `most` to 2^14 .. 2^15. Unscaled, values from 65520 on are infinite as FLOAT16, and the second part of a value below
// 1/8 is subnormal (rms relative error of the split, queries of size 0.09 / 0.01 / 0.001: 2e-7 / 2e-6 / 2e-5). Scaled, the
// parts leave at most 2^-23 of a value and 2^-40 of the row's largest. (Bounded so that both powers are normal numbers.)
__device__ __forceinline__ int pa_split_exponent(float most) {
    int e;
    (void)frexpf(most, &e);
    e = 15 - e;
    return e < -113 ? -113 : (e > 100 ? 100 : e);
}

// EPL consecutive values starting at element `first` (unit stride, 16-byte aligned start for the storage type)
template <int EPL>
__device__ __forceinline__ void pa_load_run(const void *data, int dtype, size_t first, float (&v)[EPL]) {
    if (dtype == MARMOT_HIP_DTYPE_F8_E4M3) {
        uint32_t w[EPL / 4];
        if constexpr (EPL == 4) {
            w[0] = *(const uint32_t *)((const uint8_t *)data + first);
        } else if constexpr (EPL == 8) {
            const uint2 u = *(const uint2 *)((const uint8_t *)data + first);
            w[0] = u.x, w[1] = u.y;
        } else {
            const uint4 u = *(const uint4 *)((const uint8_t *)data + first);
            w[0] = u.x, w[1] = u.y, w[2] = u.z, w[3] = u.w;
        }
        // Codes whose exponent field is below 15 mean the same in this format and in the hardware's e4m3 (bias 7,
        // same subnormals), which converts two bytes per instruction; a word that holds a field of 15 (this format's
        // NaN) takes the bit-level decoder.
        typedef float pa_f2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int i = 0; i < EPL / 4; ++i) {
            if (((((w[i] & 0x78787878u) + 0x08080808u) & 0x80808080u)) == 0u) {
                const pa_f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], false);
                const pa_f2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], true);
                v[4 * i] = lo.x, v[4 * i + 1] = lo.y, v[4 * i + 2] = hi.x, v[4 * i + 3] = hi.y;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[4 * i + e] = pa_fp8_to_f32((w[i] >> (8 * e)) & 0xffu);
                }
            }
        }
    } else if (dtype == MARMOT_HIP_DTYPE_F32) {
#pragma unroll
        for (int e = 0; e < EPL; e += 4) {
            const float4 f = *(const float4 *)((const float *)data + first + e);
            v[e] = f.x, v[e + 1] = f.y, v[e + 2] = f.z, v[e + 3] = f.w;
        }
    } else {
        uint32_t w[EPL / 2];
        if constexpr (EPL == 4) {
            const uint2 u = *(const uint2 *)((const uint16_t *)data + first);
            w[0] = u.x, w[1] = u.y;
        } else {
#pragma unroll
            for (int e = 0; e < EPL / 2; e += 4) {
                const uint4 u = *(const uint4 *)((const uint16_t *)data + first + 2 * e);
                w[e] = u.x, w[e + 1] = u.y, w[e + 2] = u.z, w[e + 3] = u.w;
            }
        }
#pragma unroll
        for (int e = 0; e < EPL / 2; ++e) {
            if (dtype == MARMOT_HIP_DTYPE_F16) {
                v[2 * e] = h2f((uint16_t)(w[e] & 0xffffu));
                v[2 * e + 1] = h2f((uint16_t)(w[e] >> 16));
            } else {
                v[2 * e] = __uint_as_float(w[e] << 16);
                v[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
            }
        }
    }
}

// ---- metadata check (paged_attention_ref.c:809-823): sequence slots inside the block table, kv slots inside the cache
__global__ __launch_bounds__(256) void k_pa_check(const PaParams p) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= p.token_count) {
        return;
    }
    const uint32_t seq = p.meta[t * p.meta_stride[0]];
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    if (seq >= p.max_seqs || (slot >> p.shift) >= p.kv_blocks) {
        atomicMax(p.flag, (int)(p.token_count - t));  // the maximum names the first offender
    }
}

// ---- cache write (cpu_paged_attention_kv_write_range, :346-373): one workgroup per (token, kv head)
__global__ __launch_bounds__(128) void k_pa_write(const PaParams p) {
    const uint32_t t = blockIdx.x, h = blockIdx.y;
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    const uint32_t block = slot >> p.shift;
    if (p.tile_tokens != 0u && h == 0 && threadIdx.x < 64u) {
        const uint32_t tiled = pa_in_run(p, t, p.meta[t * p.meta_stride[0]]);
        if (threadIdx.x == 0) {
            p.tiled[t] = tiled;
        }
    }
    if (block >= p.kv_blocks) {
        return;
    }
    const size_t dst0 = (size_t)block * p.kv_stride[0] + (size_t)p.layer_idx * p.kv_stride[1] + (size_t)h * p.kv_stride[2] +
                        (size_t)(slot & p.mask) * p.kv_stride[3];
    const size_t k0 = (size_t)t * p.k_stride[0] + (size_t)h * p.k_stride[1];
    const size_t v0 = (size_t)t * p.v_stride[0] + (size_t)h * p.v_stride[1];
    const bool bits16 = p.act_dtype == p.kv_dtype && p.act_dtype != MARMOT_HIP_DTYPE_F32;
    for (uint32_t d = threadIdx.x; d < p.head_dim; d += blockDim.x) {
        const size_t dst = dst0 + d * p.kv_stride[4];
        if (bits16) {  // same 16-bit storage type: the bits travel unchanged
            ((uint16_t *)p.kv_k)[dst] = ((const uint16_t *)p.k_new)[k0 + d * p.k_stride[2]];
            ((uint16_t *)p.kv_v)[dst] = ((const uint16_t *)p.v_new)[v0 + d * p.v_stride[2]];
        } else {
            pa_store(p.kv_k, p.kv_dtype, dst, pa_load(p.k_new, p.act_dtype, k0 + d * p.k_stride[2]));
            pa_store(p.kv_v, p.kv_dtype, dst, pa_load(p.v_new, p.act_dtype, v0 + d * p.v_stride[2]));
        }
    }
}

// The same for 16-bit caches where eight values are 16 aligned bytes (pa_write_rows): one workgroup per token, eight values of a
// row per thread and step, and a wavefront of its own for the look at the call's lengths, which is a chain of loads as long
// as the copy's. 1024 tokens of 8 heads of 128 beside a prompt: 9.7 -> 7.2 us (a workgroup per row is 8192 small ones).
constexpr uint32_t PA_WRITE_THREADS = 256;
__global__ __launch_bounds__(PA_WRITE_THREADS + 64) void k_pa_write_rows(const PaParams p) {
    const uint32_t t = blockIdx.x;
    if (threadIdx.x >= PA_WRITE_THREADS) {  // (launched beside k_pa_prompt only)
        const uint32_t tiled = pa_in_run(p, t, p.meta[t * p.meta_stride[0]]);
        if (threadIdx.x == PA_WRITE_THREADS) {
            p.tiled[t] = tiled;
        }
        return;
    }
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    const uint32_t block = slot >> p.shift;
    if (block >= p.kv_blocks) {
        return;
    }
    const size_t dst0 = (size_t)block * p.kv_stride[0] + (size_t)p.layer_idx * p.kv_stride[1] + (size_t)(slot & p.mask) * p.kv_stride[3];
    const bool bits16 = p.act_dtype == p.kv_dtype;
    const uint32_t per_head = p.head_dim / 8u, pieces = p.num_kv_heads * per_head;
    for (uint32_t i = threadIdx.x; i < 2u * pieces; i += PA_WRITE_THREADS) {
        const bool is_value = i >= pieces;
        const uint32_t u = is_value ? i - pieces : i, h = u / per_head, d = 8u * (u - h * per_head);
        const void *src = is_value ? p.v_new : p.k_new;
        const size_t token_stride = is_value ? p.v_stride[0] : p.k_stride[0], head_stride = is_value ? p.v_stride[1] : p.k_stride[1];
        const size_t from = (size_t)t * token_stride + (size_t)h * head_stride + d;
        uint16_t *dst = (uint16_t *)(is_value ? p.kv_v : p.kv_k) + dst0 + (size_t)h * p.kv_stride[2] + d;
        if (bits16) {
            *(uint4 *)dst = *(const uint4 *)((const uint16_t *)src + from);
        } else {
            float v[8];
            pa_load_run<8>(src, p.act_dtype, from, v);
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = v[2 * e], b = v[2 * e + 1];
                w[e] = p.kv_dtype == MARMOT_HIP_DTYPE_F16 ? (uint32_t)f2h(a) | (uint32_t)f2h(b) << 16
                                                          : (uint32_t)pa_f2bf(a) | (uint32_t)pa_f2bf(b) << 16;
            }
            *(uint4 *)dst = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// ---- the FLOAT8_E4M3 cache write (paged_attention_ref.c:825-989) in four launches
// 1. scratch: no new magnitudes, no block touched
__global__ __launch_bounds__(256) void k_pa_fp8_init(const PaParams p) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < p.kv_blocks * p.num_kv_heads) {
        p.new_kmax[i] = 0u;
        p.new_vmax[i] = 0u;
        p.claim[i] = 0xffffffffu;
    }
    if (i < p.kv_blocks) {
        p.min_off[i] = p.block_size;
    }
}

__device__ __forceinline__ float pa_block_max(float v, float *red) {  // maximum over a workgroup of 128 threads
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = 64; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        }
        __syncthreads();
    }
    const float r = red[0];
    __syncthreads();
    return r;
}

// 2. per (token, kv head): the largest magnitudes of the new key and value rows into their block's entry (non-negative
//    floats order like their bits), and the first offset written in the block
__global__ __launch_bounds__(128) void k_pa_fp8_scan_new(const PaParams p) {
    __shared__ float red[128];
    const uint32_t t = blockIdx.x, h = blockIdx.y;
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    const uint32_t block = slot >> p.shift;
    if (block >= p.kv_blocks) {
        return;
    }
    float km = 0.0f, vm = 0.0f;
    for (uint32_t d = threadIdx.x; d < p.head_dim; d += 128u) {
        km = fmaxf(km, fabsf(pa_load(p.k_new, p.act_dtype, (size_t)t * p.k_stride[0] + (size_t)h * p.k_stride[1] + d * p.k_stride[2])));
        vm = fmaxf(vm, fabsf(pa_load(p.v_new, p.act_dtype, (size_t)t * p.v_stride[0] + (size_t)h * p.v_stride[1] + d * p.v_stride[2])));
    }
    km = pa_block_max(km, red);
    vm = pa_block_max(vm, red);
    if (threadIdx.x == 0) {
        atomicMax(p.new_kmax + (size_t)block * p.num_kv_heads + h, __float_as_uint(km));
        atomicMax(p.new_vmax + (size_t)block * p.num_kv_heads + h, __float_as_uint(vm));
        if (h == 0) {
            atomicMin(p.min_off + block, slot & p.mask);
        }
    }
}

// Maxima of four values over a workgroup of 128 threads (two wavefronts): lanes first, then the two wavefronts
// through LDS. `red` holds 8 floats and is free again on return.
__device__ __forceinline__ void pa_block_max4(float (&v)[4], float *red) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = fmaxf(v[i], __shfl_xor(v[i], s));
        }
    }
    if ((threadIdx.x & 63u) == 0u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            red[(threadIdx.x >> 6) * 4 + i] = v[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = fmaxf(red[i], red[4 + i]);
    }
    __syncthreads();
}

// The rows already in one (block, kv head): the first `existing` positions. `vec`: rows of a multiple of 16 codes at
// 16-byte aligned addresses, taken 16 codes at a time.
struct PaFp8Rows {
    uint8_t *kc, *vc;
    size_t si;
    uint32_t existing;
    bool vec;
};

__device__ __forceinline__ PaFp8Rows pa_fp8_rows(const PaParams &p, uint32_t b, uint32_t h, uint32_t existing) {
    PaFp8Rows r;
    const size_t base = (size_t)b * p.kv_stride[0] + (size_t)p.layer_idx * p.kv_stride[1] + (size_t)h * p.kv_stride[2];
    r.kc = (uint8_t *)p.kv_k + base, r.vc = (uint8_t *)p.kv_v + base;
    r.si = (size_t)b * p.scale_stride[0] + (size_t)p.layer_idx * p.scale_stride[1] + (size_t)h * p.scale_stride[2];
    r.existing = existing;
    r.vec = p.kv_stride[4] == 1 && (p.head_dim & 15u) == 0u && (p.kv_stride[3] & 15u) == 0u &&
            (((uintptr_t)r.kc | (uintptr_t)r.vc) & 15u) == 0u;
    return r;
}

__device__ __forceinline__ uint32_t pa_fp8_big_field(uint32_t big, uint32_t word) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t c = (word >> (8 * e)) & 0x7fu;
        big = c < 0x78u && c > big ? c : big;
    }
    return big;
}

// This thread's share of the largest finite magnitude fields (low seven bits) among the rows already there: a finite
// code's magnitude grows with that field, so the largest one is found first and decoded once (NaN codes, field 15
// of the exponent, never win a maximum).
__device__ __forceinline__ void pa_fp8_scan_rows(const PaParams &p, const PaFp8Rows &r, uint32_t &kbig, uint32_t &vbig) {
    kbig = vbig = 0u;
    if (r.vec) {
        const uint32_t per_row = p.head_dim >> 4, chunks = r.existing * per_row;
        for (uint32_t c = threadIdx.x; c < chunks; c += 128u) {
            const uint32_t pos = c / per_row;
            const size_t at = (size_t)pos * p.kv_stride[3] + (size_t)(c - pos * per_row) * 16u;
            const uint4 k = *(const uint4 *)(r.kc + at), v = *(const uint4 *)(r.vc + at);
            kbig = pa_fp8_big_field(pa_fp8_big_field(pa_fp8_big_field(pa_fp8_big_field(kbig, k.x), k.y), k.z), k.w);
            vbig = pa_fp8_big_field(pa_fp8_big_field(pa_fp8_big_field(pa_fp8_big_field(vbig, v.x), v.y), v.z), v.w);
        }
        return;
    }
    const uint32_t cells = r.existing * p.head_dim;
    for (uint32_t c = threadIdx.x; c < cells; c += 128u) {
        const uint32_t pos = c / p.head_dim, d = c - pos * p.head_dim;
        const size_t at = (size_t)pos * p.kv_stride[3] + (size_t)d * p.kv_stride[4];
        const uint32_t kb = r.kc[at] & 0x7fu, vb = r.vc[at] & 0x7fu;
        kbig = kb < 0x78u && kb > kbig ? kb : kbig;
        vbig = vb < 0x78u && vb > vbig ? vb : vbig;
    }
}

__device__ __forceinline__ uint32_t pa_fp8_recode4(uint32_t word, float old_scale, float new_scale) {
    uint32_t out = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        out |= pa_fp8_quant(pa_fp8_dequant((word >> (8 * e)) & 0xffu, old_scale), new_scale) << (8 * e);
    }
    return out;
}

// The new scale of one cache tensor of the block from the largest magnitude field found in it and the largest new
// magnitude; the rows already there are re-encoded when the scale changes. `old_scale` was read before any thread
// could have written the new one (a barrier lies between).
__device__ __forceinline__ float pa_fp8_rescale_rows(const PaParams &p, const PaFp8Rows &r, int which, uint32_t big_field,
                                                     float new_max, float old_scale) {
    uint8_t *cache = which ? r.vc : r.kc;
    const float big = fmaxf(pa_fp8_dequant(big_field, old_scale), new_max);
    const float new_scale = big > 0.0f ? big / 240.0f : 1.0f;
    if (r.existing > 0 && new_scale != old_scale) {
        if (r.vec) {
            const uint32_t per_row = p.head_dim >> 4, chunks = r.existing * per_row;
            for (uint32_t c = threadIdx.x; c < chunks; c += 128u) {
                const uint32_t pos = c / per_row;
                uint4 *cell = (uint4 *)(cache + (size_t)pos * p.kv_stride[3] + (size_t)(c - pos * per_row) * 16u);
                uint4 w = *cell;
                w.x = pa_fp8_recode4(w.x, old_scale, new_scale), w.y = pa_fp8_recode4(w.y, old_scale, new_scale);
                w.z = pa_fp8_recode4(w.z, old_scale, new_scale), w.w = pa_fp8_recode4(w.w, old_scale, new_scale);
                *cell = w;
            }
        } else {
            const uint32_t cells = r.existing * p.head_dim;
            for (uint32_t c = threadIdx.x; c < cells; c += 128u) {
                const uint32_t pos = c / p.head_dim, d = c - pos * p.head_dim;
                uint8_t *cell = cache + (size_t)pos * p.kv_stride[3] + (size_t)d * p.kv_stride[4];
                *cell = (uint8_t)pa_fp8_quant(pa_fp8_dequant(*cell, old_scale), new_scale);
            }
        }
    }
    if (threadIdx.x == 0) {
        (which ? p.v_scale : p.k_scale)[r.si] = new_scale;
    }
    return new_scale;
}

// The work on one (block, kv head): the new scales from the rows already there (the first `existing` positions) and
// this thread's share of the largest new magnitudes; the rows already there are re-encoded where a scale changes.
// Whole workgroup of 128.
__device__ __forceinline__ void pa_fp8_rescale_block(const PaParams &p, uint32_t b, uint32_t h, uint32_t existing,
                                                     float new_km, float new_vm, float *red, float *new_scales) {
    const PaFp8Rows r = pa_fp8_rows(p, b, h, existing);
    const float old_k = p.k_scale[r.si], old_v = p.v_scale[r.si];
    uint32_t kbig, vbig;
    pa_fp8_scan_rows(p, r, kbig, vbig);
    float m[4] = {new_km, new_vm, (float)kbig, (float)vbig};
    pa_block_max4(m, red);
    new_scales[0] = pa_fp8_rescale_rows(p, r, 0, (uint32_t)m[2], m[0], old_k);
    new_scales[1] = pa_fp8_rescale_rows(p, r, 1, (uint32_t)m[3], m[1], old_v);
}

// 3. per (touched block, kv head): the new scale; rows already in the block are re-encoded when it changes. A token
//    that writes the block's first new row does the block's work, so the launch grows with the call, not the cache;
//    when several tokens of a call carry that offset (the same kv_slot twice), the first workgroup to claim the block
//    does it alone: two of them would read each other's new scale as the old one and encode the rows twice. The
//    reference touches each block once, whatever duplicates a call holds (paged_attention_ref.c:866-946).
__global__ __launch_bounds__(128) void k_pa_fp8_rescale(const PaParams p) {
    __shared__ float red[128];
    const uint32_t t = blockIdx.x, h = blockIdx.y;
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    const uint32_t b = slot >> p.shift;
    if (b >= p.kv_blocks) {
        return;
    }
    const uint32_t existing = p.min_off[b];
    if ((slot & p.mask) != existing) {
        return;
    }
    if (threadIdx.x == 0) {
        red[0] = __uint_as_float(atomicCAS(p.claim + (size_t)b * p.num_kv_heads + h, 0xffffffffu, t));
    }
    __syncthreads();
    const bool mine = __float_as_uint(red[0]) == 0xffffffffu;
    __syncthreads();
    if (!mine) {
        return;
    }
    float scales[2];
    pa_fp8_rescale_block(p, b, h, existing, __uint_as_float(p.new_kmax[(size_t)b * p.num_kv_heads + h]),
                         __uint_as_float(p.new_vmax[(size_t)b * p.num_kv_heads + h]), red, scales);
}

// 4. per (token, kv head): the new rows, encoded with their block's scale
__global__ __launch_bounds__(128) void k_pa_fp8_store(const PaParams p) {
    const uint32_t t = blockIdx.x, h = blockIdx.y;
    const uint32_t slot = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]];
    const uint32_t block = slot >> p.shift;
    if (block >= p.kv_blocks) {
        return;
    }
    const size_t si = (size_t)block * p.scale_stride[0] + (size_t)p.layer_idx * p.scale_stride[1] + (size_t)h * p.scale_stride[2];
    const float ks = p.k_scale[si], vs = p.v_scale[si];
    const size_t dst0 = (size_t)block * p.kv_stride[0] + (size_t)p.layer_idx * p.kv_stride[1] + (size_t)h * p.kv_stride[2] +
                        (size_t)(slot & p.mask) * p.kv_stride[3];
    for (uint32_t d = threadIdx.x; d < p.head_dim; d += 128u) {
        const float kx = pa_load(p.k_new, p.act_dtype, (size_t)t * p.k_stride[0] + (size_t)h * p.k_stride[1] + d * p.k_stride[2]);
        const float vx = pa_load(p.v_new, p.act_dtype, (size_t)t * p.v_stride[0] + (size_t)h * p.v_stride[1] + d * p.v_stride[2]);
        ((uint8_t *)p.kv_k)[dst0 + d * p.kv_stride[4]] = (uint8_t)pa_fp8_quant(kx, ks);
        ((uint8_t *)p.kv_v)[dst0 + d * p.kv_stride[4]] = (uint8_t)pa_fp8_quant(vx, vs);
    }
}

// The same update in one launch, for calls of at most PA_FP8_ONE_TOKENS tokens. Every (token, kv head) workgroup finds
// the tokens of the call that write its block; the workgroup of the first of them does the block's work alone (largest
// new magnitudes, new scales, re-encoding, then the new rows in token order, so of two tokens with one kv_slot the
// later one stays, as in the reference's token loop) and the others leave. No scratch memory, no order between
// workgroups: each (block, kv head) is touched by exactly one.
constexpr uint32_t PA_FP8_ONE_TOKENS = 1024;
__global__ __launch_bounds__(128) void k_pa_fp8_update(const PaParams p) {
    __shared__ float red[128];
    __shared__ uint32_t members[PA_FP8_ONE_TOKENS / 32];
    __shared__ uint32_t first_off;
    const uint32_t t = blockIdx.x, h = blockIdx.y;
    const uint32_t b = p.meta[t * p.meta_stride[0] + 2 * p.meta_stride[1]] >> p.shift;
    if (b >= p.kv_blocks) {
        return;
    }
    if (threadIdx.x < PA_FP8_ONE_TOKENS / 32) {
        members[threadIdx.x] = 0u;
    }
    if (threadIdx.x == 0) {
        first_off = p.block_size;
    }
    __syncthreads();
    for (uint32_t u = threadIdx.x; u < p.token_count; u += 128u) {
        const uint32_t slot = p.meta[u * p.meta_stride[0] + 2 * p.meta_stride[1]];
        if ((slot >> p.shift) == b) {
            atomicOr(members + (u >> 5), 1u << (u & 31u));
            atomicMin(&first_off, slot & p.mask);
        }
    }
    __syncthreads();
    bool first = (members[t >> 5] & ((1u << (t & 31u)) - 1u)) == 0u;
    for (uint32_t w = 0; w < (t >> 5); ++w) {
        first = first && members[w] == 0u;
    }
    if (!first) {
        return;
    }
    const uint32_t words = (p.token_count + 31u) >> 5;
    float km = 0.0f, vm = 0.0f;
    for (uint32_t w = t >> 5; w < words; ++w) {
        for (uint32_t bits = members[w]; bits != 0u; bits &= bits - 1u) {
            const uint32_t u = w * 32u + (uint32_t)__ffs(bits) - 1u;
            for (uint32_t d = threadIdx.x; d < p.head_dim; d += 128u) {
                km = fmaxf(km, fabsf(pa_load(p.k_new, p.act_dtype, (size_t)u * p.k_stride[0] + (size_t)h * p.k_stride[1] + d * p.k_stride[2])));
                vm = fmaxf(vm, fabsf(pa_load(p.v_new, p.act_dtype, (size_t)u * p.v_stride[0] + (size_t)h * p.v_stride[1] + d * p.v_stride[2])));
            }
        }
    }
    float scales[2];
    pa_fp8_rescale_block(p, b, h, first_off, km, vm, red, scales);
    const size_t dst0 = (size_t)b * p.kv_stride[0] + (size_t)p.layer_idx * p.kv_stride[1] + (size_t)h * p.kv_stride[2];
    for (uint32_t w = t >> 5; w < words; ++w) {
        for (uint32_t bits = members[w]; bits != 0u; bits &= bits - 1u) {
            const uint32_t u = w * 32u + (uint32_t)__ffs(bits) - 1u;
            const uint32_t slot = p.meta[u * p.meta_stride[0] + 2 * p.meta_stride[1]];
            const size_t dst = dst0 + (size_t)(slot & p.mask) * p.kv_stride[3];
            for (uint32_t d = threadIdx.x; d < p.head_dim; d += 128u) {
                const float kx = pa_load(p.k_new, p.act_dtype, (size_t)u * p.k_stride[0] + (size_t)h * p.k_stride[1] + d * p.k_stride[2]);
                const float vx = pa_load(p.v_new, p.act_dtype, (size_t)u * p.v_stride[0] + (size_t)h * p.v_stride[1] + d * p.v_stride[2]);
                ((uint8_t *)p.kv_k)[dst + d * p.kv_stride[4]] = (uint8_t)pa_fp8_quant(kx, scales[0]);
                ((uint8_t *)p.kv_v)[dst + d * p.kv_stride[4]] = (uint8_t)pa_fp8_quant(vx, scales[1]);
            }
        }
    }
}

// ---- attention (cpu_paged_attention_attention_range, :398-569)
// One workgroup of 16 groups of 16 lanes per (token, QH query heads that share a key / value head): every key and
// value row is fetched, converted and located once for the QH heads. A group takes two positions per step and
// requests both before it works on either.
constexpr int PA_GROUPS = 16;

template <int EPL, int QH>
__global__ __launch_bounds__(16 * PA_GROUPS) void k_pa_attend(const PaParams p) {
    warm_kernel_arguments<sizeof(PaParams), sizeof(PaParams)>();
    __shared__ float s_acc[PA_GROUPS][QH][16 * EPL];
    __shared__ float s_m[PA_GROUPS][QH], s_l[PA_GROUPS][QH];
    const uint32_t t = blockIdx.x;
    const uint32_t qh0 = blockIdx.y * QH;  // first query head of this workgroup; QH divides the heads per kv head
    const int tid = threadIdx.x, g = tid >> 4, l = tid & 15;
    const uint32_t seq = p.meta[t * p.meta_stride[0]];
    const uint32_t pos = p.meta[t * p.meta_stride[0] + p.meta_stride[1]];
    uint32_t splits = p.splits;
    if (p.tile_tokens != 0u) {
        const uint32_t tiled = __builtin_amdgcn_readfirstlane(p.tiled[t]);  // (the loop over the shares stays scalar)
        splits = tiled == 2u ? p.share_splits : splits;
        if (tiled == 1u || blockIdx.z >= splits) {
            return;
        }
    }
    const uint32_t kv_len = seq < p.max_seqs ? pos + 1u : 0u;
    const uint32_t kvh = qh0 / p.group;
    const uint32_t d0 = (uint32_t)l * EPL;  // this lane's first value of the head dimension

    float qv[QH][EPL];
#pragma unroll
    for (int h = 0; h < QH; ++h) {
        const size_t q_base = (size_t)t * p.q_stride[0] + (size_t)(qh0 + h) * p.q_stride[1];
        if (p.q_vec) {
            pa_load_run<EPL>(p.q, p.act_dtype, q_base + d0, qv[h]);
        } else {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                qv[h][e] = d0 + e < p.head_dim ? pa_load(p.q, p.act_dtype, q_base + (size_t)(d0 + e) * p.q_stride[2]) : 0.0f;
            }
        }
        if (p.scale != 1.0f) {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                qv[h][e] *= p.scale;
            }
        }
    }

    float m[QH], lsum[QH], acc[QH][EPL];
#pragma unroll
    for (int h = 0; h < QH; ++h) {
        m[h] = -INFINITY;
        lsum[h] = 0.0f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            acc[h][e] = 0.0f;
        }
    }
    const size_t head_base = (size_t)p.layer_idx * p.kv_stride[1] + (size_t)kvh * p.kv_stride[2];
    const uint32_t *table_row = p.table + (size_t)seq * p.table_stride[0];
    // the cache row of position pp, or false when the position has no block (beyond the table, or a hole)
    const bool fp8 = p.kv_dtype == MARMOT_HIP_DTYPE_F8_E4M3;
    auto locate = [&](uint32_t pp, size_t &base, uint32_t &tb_out) -> bool {
        if (pp >= kv_len) {
            return false;
        }
        const uint32_t logical = pp >> p.shift;
        if (logical >= p.max_blocks) {
            return false;
        }
        const uint32_t tb = table_row[(size_t)logical * p.table_stride[1]];
        if (tb == PA_NO_BLOCK || tb >= p.kv_blocks) {
            return false;
        }
        base = (size_t)tb * p.kv_stride[0] + head_base + (size_t)(pp & p.mask) * p.kv_stride[3];
        tb_out = tb;
        return true;
    };
    auto fetch = [&](size_t base, uint32_t tb, float (&kr)[EPL], float (&vr)[EPL]) {
        if (p.kv_vec) {
            pa_load_run<EPL>(p.kv_k, p.kv_dtype, base + d0, kr);
            pa_load_run<EPL>(p.kv_v, p.kv_dtype, base + d0, vr);
        } else {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const bool in = d0 + e < p.head_dim;
                const size_t i = base + (size_t)(d0 + e) * p.kv_stride[4];
                kr[e] = in ? pa_load(p.kv_k, p.kv_dtype, i) : 0.0f;
                vr[e] = in ? pa_load(p.kv_v, p.kv_dtype, i) : 0.0f;
            }
        }
        if (fp8) {  // code value times the block's scale: the reference's decoded element (:474-498)
            const size_t si = (size_t)tb * p.scale_stride[0] + (size_t)p.layer_idx * p.scale_stride[1] +
                              (size_t)kvh * p.scale_stride[2];
            const float ks = p.k_scale[si], vs = p.v_scale[si];
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                kr[e] = ks > 0.0f ? kr[e] * ks : 0.0f;
                vr[e] = vs > 0.0f ? vr[e] * vs : 0.0f;
            }
        }
    };
    auto absorb = [&](const float (&kr)[EPL], const float (&vr)[EPL]) {
#pragma unroll
        for (int h = 0; h < QH; ++h) {
            float dot = 0.0f;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                dot = __builtin_fmaf(qv[h][e], kr[e], dot);
            }
            dot = row16_sum(dot);
            if (dot > m[h]) {  // the same decision in all 16 lanes of the group
                const float corr = m[h] == -INFINITY ? 0.0f : pa_exp(m[h] - dot);
                lsum[h] *= corr;
#pragma unroll
                for (int e = 0; e < EPL; ++e) {
                    acc[h][e] *= corr;
                }
                m[h] = dot;
            }
            const float w = pa_exp(dot - m[h]);
            lsum[h] += w;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                acc[h][e] = __builtin_fmaf(w, vr[e], acc[h][e]);
            }
        }
    };
    // this workgroup's share of the history (the whole of it without a split)
    const uint32_t chunk = (kv_len + splits - 1u) / splits;
    const uint32_t first = blockIdx.z * chunk;
    const uint32_t stop = first + chunk < kv_len ? first + chunk : kv_len;
    for (uint32_t pp = first + (uint32_t)g; pp < stop; pp += 2u * PA_GROUPS) {
        size_t base0 = 0, base1 = 0;
        uint32_t tb0 = 0, tb1 = 0;
        const bool have0 = locate(pp, base0, tb0), have1 = pp + PA_GROUPS < stop && locate(pp + PA_GROUPS, base1, tb1);
        float k0[EPL], v0[EPL], k1[EPL], v1[EPL];
        if (have0) {
            fetch(base0, tb0, k0, v0);
        }
        if (have1) {
            fetch(base1, tb1, k1, v1);
        }
        if (have0) {
            absorb(k0, v0);
        }
        if (have1) {
            absorb(k1, v1);
        }
    }

    // the groups meet: out = sum_g acc_g * exp(m_g - M) / sum_g l_g * exp(m_g - M)
#pragma unroll
    for (int h = 0; h < QH; ++h) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            s_acc[g][h][d0 + e] = acc[h][e];
        }
        if (l == 0) {
            s_m[g][h] = m[h];
            s_l[g][h] = lsum[h];
        }
    }
    __syncthreads();
    for (uint32_t idx = (uint32_t)tid; idx < (uint32_t)QH * p.head_dim; idx += 16u * PA_GROUPS) {
        uint32_t h = 0, d = idx;  // idx = h * head_dim + d
        while (d >= p.head_dim) {
            d -= p.head_dim;
            ++h;
        }
        float big = -INFINITY;
#pragma unroll
        for (int gg = 0; gg < PA_GROUPS; ++gg) {
            big = fmaxf(big, s_m[gg][h]);
        }
        float o = 0.0f, total = 0.0f;
        // a NaN score (NaN in the query or in a row of the history) leaves a NaN sum of weights in its group: the head's
        // output is NaN then, as in the reference, whatever the maxima say (they skip NaN)
        bool bad = false;
#pragma unroll
        for (int gg = 0; gg < PA_GROUPS; ++gg) {
            bad = bad || s_l[gg][h] != s_l[gg][h];
        }
        if (big != -INFINITY) {  // has_any (:552-557)
#pragma unroll
            for (int gg = 0; gg < PA_GROUPS; ++gg) {
                const float f = s_m[gg][h] == -INFINITY ? 0.0f : pa_exp(s_m[gg][h] - big);
                total = __builtin_fmaf(s_l[gg][h], f, total);
                o = __builtin_fmaf(s_acc[gg][h][d], f, o);
            }
        }
        if (splits > 1u) {  // the shares of the history meet in k_pa_merge
            float *part = p.partial + (((size_t)t * p.num_q_heads + qh0 + h) * p.partial_splits + blockIdx.z) * (p.head_dim + 2u);
            if (d == 0) {
                part[0] = big;
                part[1] = bad ? __uint_as_float(0x7fc00000u) : total;
            }
            part[2 + d] = o;
            continue;
        }
        o = bad ? __uint_as_float(0x7fc00000u) : (total > 0.0f ? o * (1.0f / total) : 0.0f);
        const size_t out_base = (size_t)t * p.out_stride[0] + (size_t)(qh0 + h) * p.out_stride[1];
        pa_store(p.out, p.act_dtype, out_base + (size_t)d * p.out_stride[2], o);
    }
}

// ---- attention with the scores on the matrix cores (FLOAT16 or BFLOAT16 cache rows of 128 values, blocks of 16
// positions or more)
// One workgroup of four wavefronts per (token, QH query heads of one key / value head, share of the history); a
// wavefront takes tiles of 16 consecutive positions (one cache block, or a 16-aligned part of one).
//   * Scores: S[position][head] = K[position][:] . q[head][:] as v_mfma_f32_16x16x16_f16 with the KEY ROWS as the row
//     operand, read from the cache straight into operand registers (lane (r, j) = (lane % 16, lane / 16) reads the 64
//     contiguous bytes of dimensions 32 j .. 32 j + 31 of position r: the k index of the c-th instruction stands for
//     dimensions 32 j + 4 c .. + 3, the same in both operands, so no value moves between lanes and none is converted).
//     The query is the column operand, scaled (see pa_split_exponent) and split once into a FLOAT16 high part and a
//     FLOAT16 remainder (two instructions per step: products of FLOAT16 values are exact in fp32); for
//     a BFLOAT16 cache (v_mfma_f32_16x16x16_bf16) into three BFLOAT16 parts of 8 bits each. Columns beyond QH are zero.
//   * The result layout puts positions 4 j + i (i = 0..3) of head n in lane (n, j): the online softmax of a head runs in
//     the four lanes n, n + 16, n + 32, n + 48 (two cross-lane exchanges per maximum and per sum).
//   * Output: the 16 lanes of group j hold dimensions 8 n .. 8 n + 7 of the value rows of THEIR four positions; the
//     weights of head h for these positions are fetched from lane (h, j) with ds_swizzle broadcasts; fp32
//     multiply-adds as before. The running output is rescaled only when a maximum moved (wavefront-wide test).
// The 16 partial outputs (4 wavefronts x 4 groups) meet in LDS like the 16 groups of k_pa_attend. fp32 accumulation
// everywhere; only the order of the sums differs from the reference.
typedef _Float16 pa_half4 __attribute__((ext_vector_type(4)));
typedef short pa_short4 __attribute__((ext_vector_type(4)));
typedef float pa_float4 __attribute__((ext_vector_type(4)));

template <int PATTERN>
__device__ __forceinline__ float pa_swizzle(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), PATTERN));
}
// value of lane (h, j) in every lane of the 16-lane group j (bit-mask mode: lane' = (lane & 0x10) | h inside each half)
template <int H>
__device__ __forceinline__ float pa_group_bcast(float v) {
    return pa_swizzle<0x10 | (H << 5)>(v);
}
// exchange with the lane 16 / 32 lanes away
__device__ __forceinline__ float pa_xor16(float v) {
    return pa_swizzle<0x1f | (0x10 << 10)>(v);
}
__device__ __forceinline__ float pa_xor32(float v) {
    return __shfl_xor(v, 32);
}

// Two e4m3 codes of a word (bytes 0, 1 or 2, 3) as a pair of FLOAT16 values in one instruction (gfx950's conversion
// with a power-of-two scale, here 1): exact, denormal codes included (both formats are linear there). Codes with all
// exponent bits set (NaN in the reference's e4m3, finite or NaN in the hardware's) are found by pa_fp8_nan_bits and
// take the reference's decoder.
typedef _Float16 pa_half2 __attribute__((ext_vector_type(2)));
template <int HI>
__device__ __forceinline__ uint32_t pa_fp8x2_to_f16(uint32_t w) {
    const pa_half2 v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, HI != 0);
    return __builtin_bit_cast(uint32_t, v);
}
// bit 7 of a byte is set iff that byte of w is a NaN code (exponent field 15)
__device__ __forceinline__ uint32_t pa_fp8_nan_bits(uint32_t w) {
    return (w & 0x78787878u) + 0x08080808u;
}
// the same two words through the reference's decoder (NaN codes become NaN)
template <int HI>
__device__ __forceinline__ uint32_t pa_fp8x2_to_f16_slow(uint32_t w) {
    const uint32_t c0 = (w >> (HI ? 16 : 0)) & 0xffu, c1 = (w >> (HI ? 24 : 8)) & 0xffu;
    return (uint32_t)f2h(pa_fp8_to_f32(c0)) | ((uint32_t)f2h(pa_fp8_to_f32(c1)) << 16);
}

constexpr int PA_KV_F16 = 0, PA_KV_BF16 = 1, PA_KV_FP8 = 2;
constexpr uint32_t PA_PIPELINE_TILES = 24;  // tiles per workgroup (six per wavefront) from which the tile loop is pipelined

template <int QH, int KVT, bool PIPE>
__global__ __launch_bounds__(256) void k_pa_attend_mfma(const PaParams p) {
    constexpr bool BF16 = KVT == PA_KV_BF16, FP8 = KVT == PA_KV_FP8;
    constexpr int EPL = 8;  // head_dim == 128
    __shared__ float s_acc[PA_GROUPS][QH][16 * EPL];
    __shared__ float s_m[PA_GROUPS][QH], s_l[PA_GROUPS][QH];
    const uint32_t t = blockIdx.x;
    const uint32_t qh0 = blockIdx.y * QH;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, j = lane >> 4;
    const uint32_t seq = p.meta[t * p.meta_stride[0]];
    const uint32_t pos = p.meta[t * p.meta_stride[0] + p.meta_stride[1]];
    uint32_t splits = p.splits;
    if (p.tile_tokens != 0u) {
        const uint32_t tiled = __builtin_amdgcn_readfirstlane(p.tiled[t]);  // (the loop over the shares stays scalar)
        splits = tiled == 2u ? p.share_splits : splits;
        if (tiled == 1u || blockIdx.z >= splits) {
            return;
        }
    }
    const uint32_t kv_len = seq < p.max_seqs ? pos + 1u : 0u;
    const uint32_t kvh = qh0 / p.group;

    // the query: head n (zero beyond QH), dimensions 32 j .. 32 j + 31, scaled, as high part + remainder(s); FLOAT16 parts
    // are those of the row in units of `unit` (see pa_split_exponent)
    constexpr int PARTS = BF16 ? 3 : 2;
    float unit = 1.0f;
    uint2 qpart[PARTS][8];  // four 16-bit values of the storage type each
    {
        float qv[32];
#pragma unroll
        for (int e = 0; e < 32; ++e) {
            qv[e] = 0.0f;
        }
        if (n < QH) {
            const size_t q_base = (size_t)t * p.q_stride[0] + (size_t)(qh0 + n) * p.q_stride[1];
            if (p.q_vec) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float part[8];
                    pa_load_run<8>(p.q, p.act_dtype, q_base + 32u * j + 8u * c, part);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        qv[8 * c + e] = part[e];
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 32; ++e) {
                    qv[e] = pa_load(p.q, p.act_dtype, q_base + (size_t)(32 * j + e) * p.q_stride[2]);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 32; ++e) {
            qv[e] = p.scale != 1.0f ? qv[e] * p.scale : qv[e];
        }
        int up = 0;
        if constexpr (!BF16) {
            float most = 0.0f;
#pragma unroll
            for (int e = 0; e < 32; ++e) {
                most = fmaxf(most, fabsf(qv[e]));
            }
            most = fmaxf(most, pa_xor16(most));
            up = pa_split_exponent(fmaxf(most, pa_xor32(most)));
            unit = ldexpf(1.0f, -up);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            uint16_t bits[PARTS][4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = BF16 ? qv[4 * c + e] : ldexpf(qv[4 * c + e], up);
#pragma unroll
                for (int part = 0; part < PARTS; ++part) {  // each remainder is exact in fp32
                    if constexpr (BF16) {
                        bits[part][e] = pa_f2bf(v);
                        v -= pa_bf2f(bits[part][e]);
                    } else {
                        bits[part][e] = f2h(v);
                        v -= h2f(bits[part][e]);
                    }
                }
            }
#pragma unroll
            for (int part = 0; part < PARTS; ++part) {
                qpart[part][c] = make_uint2((uint32_t)bits[part][0] | ((uint32_t)bits[part][1] << 16),
                                            (uint32_t)bits[part][2] | ((uint32_t)bits[part][3] << 16));
            }
        }
    }
    auto mma = [&](const uint2 kbits, const uint2 qbits, const pa_float4 c_in) -> pa_float4 {
        if constexpr (BF16) {
            return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(pa_short4, kbits),
                                                             __builtin_bit_cast(pa_short4, qbits), c_in, 0, 0, 0);
        } else {
            return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(pa_half4, kbits),
                                                         __builtin_bit_cast(pa_half4, qbits), c_in, 0, 0, 0);
        }
    };

    float m = -INFINITY, lsum = 0.0f;  // of head n (replicated in the four lanes n + 16 j)
    float acc[QH][EPL];
#pragma unroll
    for (int h = 0; h < QH; ++h) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            acc[h][e] = 0.0f;
        }
    }
    const size_t head_base = (size_t)p.layer_idx * p.kv_stride[1] + (size_t)kvh * p.kv_stride[2];
    const uint32_t *table_row = p.table + (size_t)seq * p.table_stride[0];
    // this workgroup's share of the history, in whole tiles of 16 positions
    const uint32_t tiles = (kv_len + 15u) >> 4;
    const uint32_t tiles_per_split = (tiles + splits - 1u) / splits;
    const uint32_t tile_first = blockIdx.z * tiles_per_split;
    const uint32_t tile_stop = tile_first + tiles_per_split < tiles ? tile_first + tiles_per_split : tiles;
    // Tiles of this wavefront: tile_first + wave, + 4, ... Two memory latencies lie in front of a tile's arithmetic, the
    // block table entry and then the rows it points to; with a handful of tiles per wavefront they were most of the
    // kernel's time. So the loop of the PIPE form runs a pipeline: while tile k is worked on, the rows of tile k + 1 and the table entry
    // of tile k + 2 are in flight. All of these loads are unconditional (a tile that does not exist or has no block
    // reads block 0 and is marked): a load behind a branch would make the compiler wait for everything in flight.
    struct TileRaw {
        uint4 k[4], v[4];  // FLOAT8_E4M3: k[0..1] = the 32 key codes, v[0..1] = 4 x 8 value codes
        float ks, vs;
        uint32_t p0;
        bool ok;
    };
    const uint32_t table_last = p.max_blocks > 0u ? p.max_blocks - 1u : 0u;
    auto table_entry = [&](uint32_t tile) -> uint32_t {
        const uint32_t logical = (tile << 4) >> p.shift;
        return table_row[(size_t)(logical < table_last ? logical : table_last) * p.table_stride[1]];
    };
    auto request = [&](TileRaw &r, uint32_t tile, uint32_t tb) {
        const uint32_t logical = (tile << 4) >> p.shift;
        r.ok = tile < tile_stop && logical < p.max_blocks && tb != PA_NO_BLOCK && tb < p.kv_blocks;  // else: a hole
        r.p0 = r.ok ? tile << 4 : 0u;
        const uint32_t tbs = r.ok ? tb : 0u;
        const size_t tile_base = (size_t)tbs * p.kv_stride[0] + head_base + (size_t)(r.p0 & p.mask) * p.kv_stride[3];
        // key rows: position n of the tile, dimensions 32 j .. + 31; value rows: positions 4 j + i, dimensions 8 n .. + 7
        if constexpr (FP8) {
            const size_t si = (size_t)tbs * p.scale_stride[0] + (size_t)p.layer_idx * p.scale_stride[1] +
                              (size_t)kvh * p.scale_stride[2];
            r.ks = p.k_scale[si];
            r.vs = p.v_scale[si];
            const uint8_t *krow = (const uint8_t *)p.kv_k + tile_base + (size_t)n * p.kv_stride[3] + 32u * j;
            r.k[0] = *(const uint4 *)krow;
            r.k[1] = *(const uint4 *)(krow + 16);
            uint2 vr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vr[i] = *(const uint2 *)((const uint8_t *)p.kv_v + tile_base + (size_t)(4 * j + i) * p.kv_stride[3] + 8u * n);
            }
            r.v[0] = make_uint4(vr[0].x, vr[0].y, vr[1].x, vr[1].y);
            r.v[1] = make_uint4(vr[2].x, vr[2].y, vr[3].x, vr[3].y);
        } else {
            const uint16_t *krow = (const uint16_t *)p.kv_k + tile_base + (size_t)n * p.kv_stride[3] + 32u * j;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                r.k[c] = *(const uint4 *)(krow + 8 * c);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                r.v[i] = *(const uint4 *)((const uint16_t *)p.kv_v + tile_base + (size_t)(4 * j + i) * p.kv_stride[3] + 8u * n);
            }
        }
    };
    auto consume = [&](const TileRaw &r) {
        if (!r.ok) {
            return;
        }
        const uint32_t p0 = r.p0;  // first position of the tile
        uint4 kq[4], vq[4];
        float k_unit = 1.0f, v_unit = 1.0f;  // FLOAT8_E4M3: what one unit of the FLOAT16 operands stands for
        if constexpr (FP8) {
            // codes -> FLOAT16 operands in registers (exact); the block's scale is applied to the scores and to the
            // softmax weights. A scale that is not positive decodes to zeros (the reference's
            // cpu_paged_attention_fp8_dequant); a tile that holds a NaN code takes the reference's decoder.
            const float ks = r.ks, vs = r.vs;
            const uint32_t kw[8] = {r.k[0].x, r.k[0].y, r.k[0].z, r.k[0].w, r.k[1].x, r.k[1].y, r.k[1].z, r.k[1].w};
            const uint2 vr[4] = {make_uint2(r.v[0].x, r.v[0].y), make_uint2(r.v[0].z, r.v[0].w),
                                 make_uint2(r.v[1].x, r.v[1].y), make_uint2(r.v[1].z, r.v[1].w)};
                uint32_t nan_k = 0, nan_v = 0;
    #pragma unroll
                for (int c = 0; c < 8; ++c) {
                    nan_k |= pa_fp8_nan_bits(kw[c]);
                }
    #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    nan_v |= pa_fp8_nan_bits(vr[i].x) | pa_fp8_nan_bits(vr[i].y);
                }
                const bool k_live = ks > 0.0f, v_live = vs > 0.0f;
                const bool slow = ((nan_k & 0x80808080u) != 0 && k_live) || ((nan_v & 0x80808080u) != 0 && v_live);
                if (__builtin_amdgcn_ballot_w64(slow) == 0) {
    #pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        kq[c] = make_uint4(pa_fp8x2_to_f16<0>(kw[2 * c]), pa_fp8x2_to_f16<1>(kw[2 * c]),
                                           pa_fp8x2_to_f16<0>(kw[2 * c + 1]), pa_fp8x2_to_f16<1>(kw[2 * c + 1]));
                    }
    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        vq[i] = make_uint4(pa_fp8x2_to_f16<0>(vr[i].x), pa_fp8x2_to_f16<1>(vr[i].x),
                                           pa_fp8x2_to_f16<0>(vr[i].y), pa_fp8x2_to_f16<1>(vr[i].y));
                    }
                } else {
    #pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        kq[c] = make_uint4(pa_fp8x2_to_f16_slow<0>(kw[2 * c]), pa_fp8x2_to_f16_slow<1>(kw[2 * c]),
                                           pa_fp8x2_to_f16_slow<0>(kw[2 * c + 1]), pa_fp8x2_to_f16_slow<1>(kw[2 * c + 1]));
                    }
    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        vq[i] = make_uint4(pa_fp8x2_to_f16_slow<0>(vr[i].x), pa_fp8x2_to_f16_slow<1>(vr[i].x),
                                           pa_fp8x2_to_f16_slow<0>(vr[i].y), pa_fp8x2_to_f16_slow<1>(vr[i].y));
                    }
                }
                if (!k_live) {
    #pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        kq[c] = make_uint4(0, 0, 0, 0);
                    }
                }
                if (!v_live) {
    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        vq[i] = make_uint4(0, 0, 0, 0);
                    }
                }
                k_unit = k_live ? ks : 0.0f;
                v_unit = v_live ? vs : 0.0f;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                kq[c] = r.k[c];
                vq[c] = r.v[c];
            }
        }
            pa_float4 sc = {0.0f, 0.0f, 0.0f, 0.0f};
    #pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint2 k0 = make_uint2(kq[c].x, kq[c].y), k1 = make_uint2(kq[c].z, kq[c].w);
    #pragma unroll
                for (int part = 0; part < PARTS; ++part) {
                    sc = mma(k0, qpart[part][2 * c], sc);
                }
    #pragma unroll
                for (int part = 0; part < PARTS; ++part) {
                    sc = mma(k1, qpart[part][2 * c + 1], sc);
                }
            }
            // positions beyond the sequence (the last tile): no score, no value
            const bool whole = p0 + 16u <= kv_len;
            float s4[4] = {sc[0], sc[1], sc[2], sc[3]};
            if constexpr (FP8) {
    #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s4[i] *= k_unit;
                }
            }
            if (!whole) {
    #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (p0 + 4u * j + (uint32_t)i >= kv_len) {
                        s4[i] = -INFINITY;
                        vq[i] = make_uint4(0, 0, 0, 0);
                    }
                }
            }
            // online softmax of head n over the tile's 16 positions (lanes n, n + 16, n + 32, n + 48)
            float big = fmaxf(fmaxf(s4[0], s4[1]), fmaxf(s4[2], s4[3]));
            big = fmaxf(big, pa_xor16(big));
            big = fmaxf(big, pa_xor32(big)) * unit;
            const float m_new = fmaxf(m, big);
            const float corr = m == -INFINITY ? 0.0f : pa_exp(m - m_new);
            float w4[4];
    #pragma unroll
            for (int i = 0; i < 4; ++i) {
                w4[i] = pa_exp(__builtin_fmaf(s4[i], unit, -m_new));
            }
            float tsum = (w4[0] + w4[1]) + (w4[2] + w4[3]);
            tsum += pa_xor16(tsum);
            tsum += pa_xor32(tsum);
            lsum = lsum * corr + tsum;
            const bool moved = m_new != m;
            m = m_new;
            // rescale the running output of the heads whose maximum moved
            if (__builtin_amdgcn_ballot_w64(moved && n < QH) != 0) {
                float f[QH];
                f[0] = pa_group_bcast<0>(corr);
                if constexpr (QH > 1) {
                    f[1] = pa_group_bcast<1>(corr);
                }
                if constexpr (QH > 2) {
                    f[2] = pa_group_bcast<2>(corr);
                    f[3] = pa_group_bcast<3>(corr);
                }
    #pragma unroll
                for (int h = 0; h < QH; ++h) {
    #pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        acc[h][e] *= f[h];
                    }
                }
            }
            // values: this group's four positions, dimensions 8 n .. 8 n + 7
    #pragma unroll
            for (int i = 0; i < 4; ++i) {
                float vr[EPL];
                const uint32_t vw[4] = {vq[i].x, vq[i].y, vq[i].z, vq[i].w};
    #pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (BF16) {
                        vr[2 * e] = __uint_as_float(vw[e] << 16);
                        vr[2 * e + 1] = __uint_as_float(vw[e] & 0xffff0000u);
                    } else {
                        vr[2 * e] = h2f((uint16_t)(vw[e] & 0xffffu));
                        vr[2 * e + 1] = h2f((uint16_t)(vw[e] >> 16));
                    }
                }
                float wh[QH];
                const float wi = FP8 ? w4[i] * v_unit : w4[i];  // the value rows' unit goes with the weight
                wh[0] = pa_group_bcast<0>(wi);
                if constexpr (QH > 1) {
                    wh[1] = pa_group_bcast<1>(wi);
                }
                if constexpr (QH > 2) {
                    wh[2] = pa_group_bcast<2>(wi);
                    wh[3] = pa_group_bcast<3>(wi);
                }
    #pragma unroll
                for (int h = 0; h < QH; ++h) {
    #pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        acc[h][e] = __builtin_fmaf(wh[h], vr[e], acc[h][e]);
                    }
                }
            }
    };
    const bool any_tile = p.kv_blocks > 0u && p.max_blocks > 0u && tile_first + (uint32_t)wave < tile_stop;
    // Few tiles per wavefront (short histories, the tokens of a prompt): one after the other; the pipeline's extra
    // requests (a tile and two table entries beyond the end) cost more than they hide there (16 x 512 positions
    // 18.7 -> 22.9 us, a prompt of 512 tokens 76 -> 101 us with the pipeline everywhere).
    if (any_tile && (!PIPE || tile_stop - tile_first < PA_PIPELINE_TILES)) {
        TileRaw r;
        for (uint32_t tile = tile_first + (uint32_t)wave; tile < tile_stop; tile += 4u) {
            request(r, tile, table_entry(tile));
            consume(r);
        }
    } else if (any_tile) {
        if constexpr (PIPE) {
            uint32_t tile = tile_first + (uint32_t)wave;
            TileRaw ra, rb;
            uint32_t e1 = table_entry(tile + 4u), e2 = table_entry(tile + 8u);
            request(ra, tile, table_entry(tile));
            for (; tile < tile_stop; tile += 8u) {
                request(rb, tile + 4u, e1);
                const uint32_t e3 = table_entry(tile + 12u);
                consume(ra);
                request(ra, tile + 8u, e2);
                const uint32_t e4 = table_entry(tile + 16u);
                consume(rb);
                e1 = e3;
                e2 = e4;
            }
        }
    }

    // the 16 partial outputs meet: group g = 4 wave + j; a wavefront's sum of weights is counted once (its group 0)
    const int g = 4 * wave + j;
    const uint32_t d0 = (uint32_t)n * EPL;
#pragma unroll
    for (int h = 0; h < QH; ++h) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            s_acc[g][h][d0 + e] = acc[h][e];
        }
    }
    if (n < QH) {
        s_m[g][n] = m;
        s_l[g][n] = j == 0 ? lsum : 0.0f;
    }
    __syncthreads();
    for (uint32_t idx = (uint32_t)tid; idx < (uint32_t)QH * 128u; idx += 256u) {
        const uint32_t h = idx >> 7, d = idx & 127u;
        float top = -INFINITY;
#pragma unroll
        for (int gg = 0; gg < PA_GROUPS; ++gg) {
            top = fmaxf(top, s_m[gg][h]);
        }
        float o = 0.0f, total = 0.0f;
        // a NaN score (NaN in the query or in a row of the history) leaves a NaN sum of weights in its group: the head's
        // output is NaN then, as in the reference, whatever the maxima say (they skip NaN)
        bool bad = false;
#pragma unroll
        for (int gg = 0; gg < PA_GROUPS; ++gg) {
            bad = bad || s_l[gg][h] != s_l[gg][h];
        }
        if (top != -INFINITY) {
#pragma unroll
            for (int gg = 0; gg < PA_GROUPS; ++gg) {
                const float f = s_m[gg][h] == -INFINITY ? 0.0f : pa_exp(s_m[gg][h] - top);
                total = __builtin_fmaf(s_l[gg][h], f, total);
                o = __builtin_fmaf(s_acc[gg][h][d], f, o);
            }
        }
        if (splits > 1u) {
            float *part = p.partial + (((size_t)t * p.num_q_heads + qh0 + h) * p.partial_splits + blockIdx.z) * (p.head_dim + 2u);
            if (d == 0) {
                part[0] = top;
                part[1] = bad ? __uint_as_float(0x7fc00000u) : total;
            }
            part[2 + d] = o;
            continue;
        }
        o = bad ? __uint_as_float(0x7fc00000u) : (total > 0.0f ? o * (1.0f / total) : 0.0f);
        const size_t out_base = (size_t)t * p.out_stride[0] + (size_t)(qh0 + h) * p.out_stride[1];
        pa_store(p.out, p.act_dtype, out_base + (size_t)d * p.out_stride[2], o);
    }
}

// ---- prompts: tiles of tokens that share the key / value rows (FLOAT16 or BFLOAT16 cache, rows of 64 or 128 values)
// One workgroup of eight wavefronts per (tile of tokens, key / value head, share of the history). Its 128 rows are the
// (token, query head) pairs of 128 / group consecutive tokens; wavefronts w and w + 4 own rows 32 w .. + 31, lane l row l % 32,
// each for one half (32 positions) of every tile of the history, with a maximum, a sum and outputs of its own; the halves
// meet in LDS at the end. Two wavefronts per SIMD: one multiplies while the other is at its softmax. The workgroup walks the
// histories of the sequences in its tile (one, mostly) in tiles of 64 positions: keys as rows in two buffers, values
// transposed in three, both requested one tile ahead through registers.
//   * Scores: S[position][row] = K . q as v_mfma_f32_32x32x16 with the key rows as row operand; lane (row, h = l / 32)
//     receives positions 8 q + 4 h + e in register 4 q + e, so a row's softmax is 16 registers and one exchange. Most of the
//     query's parts wait in LDS (rows of 128): 256 registers hold neither them nor a copy of the outputs beside the rest.
//   * Output: O[dimension][row] += V^T . P with the weights as column operand: registers 8 i .. 8 i + 7 ARE the operand of
//     instruction i (the k index of lane half h stands for positions 16 i + 4 h + 0..3 and 16 i + 8 + 4 h + 0..3), and the
//     transposed values are stored in that order, so no weight moves between lanes.
//   * Precision: query and weights stay fp32 quantities, split into two FLOAT16 parts (rounded to nearest: 2^-23; query rows
//     are scaled first, see pa_split_exponent, weights by 2^14, so that the parts of small ones are normal numbers) or three
//     BFLOAT16 parts (24 bits, exact), one instruction per part, fp32 accumulation.
//   * A value that is not finite would reach rows that may not see it (0 x infinity): a tile that holds one takes the
//     products of its visible positions one by one, with the weights in fp32.
//   * Scores of -inf weigh nothing as long as the row has others, in whichever half, tile or share of its history; a row that
//     has no others is NaN. (The reference looks for the maximum a block of 64 - 256 positions at a time and gives NaN for a row whose
//     first block holds nothing else.)
// The kernel per token reads a history once per token and head group and uses a quarter of its matrix instructions; this
// one reads it once per 128 / group tokens. Two sequences x 512 tokens over 2048 cached ones, 32 / 8 heads of 128, BFLOAT16 cache,
// whole call: 756 us per token; 249 with four wavefronts that own 32 positions at a time and the table entry read in front of
// each tile; 166 with 64 at a time (one wavefront per SIMD: scores, softmax and output one after the other); 148 with
// eight wavefronts; 136 - 145 (by card) now that one wavefront locates a tile's rows for all and the values' infinities are
// looked for by two maxima per word. Bound by the issue port: per SIMD and tile of 6700 clocks 1330 instructions take it for
// 5300 (counted: 790 vector, 96 matrix, 190 scalar, 90 LDS), the matrix cores are busy for 3070; 20 us are the start and the
// end (the query's parts 6, the join of the halves 4, the first tile 8).
// Error against 64 bits there: 3.6e-7 per token, 2.2e-7 here.
typedef float pa_float16v __attribute__((ext_vector_type(16)));
typedef _Float16 pa_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 pa_bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t pa_uint4 __attribute__((ext_vector_type(4)));

constexpr uint32_t PA_PROMPT_ROWS = 128;
constexpr uint32_t PA_PROMPT_SHARE = 256;  // positions a share of a history has at least
constexpr uint32_t PA_LONG = 512, PA_MANY = 256, PA_ANY_TABLE = 512;
constexpr size_t PA_PROMPT_WORK = (size_t)3 << 19;
constexpr uint32_t PA_SHARES = 4;  // of the history of a token that is left over

constexpr uint32_t PA_PROMPT_WAVES = 8;

template <int HD, bool BF16>
struct PaPromptLds {
    static constexpr uint32_t KROW = 2 * HD + 16;   // bytes; 16 of padding: rows 4 banks apart
    static constexpr uint32_t K = 64 * KROW, V = HD * 128;
    static constexpr uint32_t V0 = 2 * K;          // two buffers of keys, three of values
    static constexpr uint32_t Q = V0 + 3 * V;      // small parts of the query: [part][16 dimensions][wavefront][lane] x 16 bytes
    static constexpr uint32_t QPARTS = HD == 128 ? (BF16 ? 2 : 1) : 0;
    // sequence, length, longest history: 128 words each; nine words
    static constexpr uint32_t TOKENS = Q + QPARTS * PA_PROMPT_ROWS * HD * 2;
    // two tiles: places of 64 rows; then which of them exist
    static constexpr uint32_t ROWS = TOKENS + (3 * PA_PROMPT_ROWS + 12) * 4;
    static constexpr uint32_t BYTES = ROWS + (2 * 64 + 2) * 8;
    static constexpr uint32_t MAIL = PA_PROMPT_WAVES * HD / 64 * 4096;  // at the end: outputs, then maximum and sum of every lane
    static_assert(MAIL + PA_PROMPT_WAVES * 512 <= Q, "the mail fits the stages");
};

// byte offset of chunk c (16 bytes: eight positions) of dimension d in the transposed values; the exclusive or spreads
// eight consecutive dimensions (reads) and dimensions four apart (writes) over the banks
__device__ __forceinline__ uint32_t pa_vt_chunk(uint32_t d, uint32_t c) {
    return d * 128u + 16u * (c ^ ((d >> 2) & 7u) ^ ((d & 3u) << 1));
}

template <bool BF16>
__device__ __forceinline__ pa_float16v pa_mma32(const uint4 a, const uint4 b, const pa_float16v c) {
    if constexpr (BF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(pa_bf8, a), __builtin_bit_cast(pa_bf8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pa_half8, a), __builtin_bit_cast(pa_half8, b), c, 0, 0,
                                                      0);
    }
}

template <int HD, bool BF16>
__global__ __launch_bounds__(64 * PA_PROMPT_WAVES, 2) void k_pa_prompt(const PaParams p) {
    using L = PaPromptLds<HD, BF16>;
    constexpr int PARTS = BF16 ? 3 : 2, QC = HD / 16, DB = HD / 32, QREGS = PARTS - L::QPARTS;
    constexpr uint32_t THREADS = 64 * PA_PROMPT_WAVES;
    constexpr int KN = 64 * HD / 8 / THREADS;   // per thread and tile: 16-byte key chunks
    constexpr uint32_t VUNITS = 16 * HD / 4;    // of a tile: 4 x 4 blocks of values, one per thread at most
    static_assert(KN >= 1 && VUNITS <= THREADS && VUNITS % 64 == 0, "a tile's rows over the threads");
    constexpr float UNIT = BF16 ? 1.0f : 16384.0f;
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint32_t *s_seq = (uint32_t *)(lds + L::TOKENS), *s_len = s_seq + PA_PROMPT_ROWS, *s_longest = s_len + PA_PROMPT_ROWS;
    uint64_t *s_firsts = (uint64_t *)(s_longest + PA_PROMPT_ROWS);  // which tokens are the first of their sequence
    uint32_t *s_odd = (uint32_t *)(s_firsts + 2);  // per buffer: 1 + number of its tile if that holds a value that is not finite
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 31u, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), rows = wave & 3u, half = wave >> 2;
    const uint32_t tt = p.tile_tokens, t0 = (gridDim.x - 1u - blockIdx.x) * tt, kvh = blockIdx.y;  // long histories first

    // the tile's tokens: sequence (NONE: not this kernel's), visible positions, and at the first token of a sequence the
    // largest number of them
    const bool mine = tid < tt && t0 + tid < p.token_count && p.tiled[t0 + tid] == 1u;
    static_assert(PA_PROMPT_ROWS == 2 * 64, "tokens of a tile: in the first two wavefronts");
    const unsigned long long any_mine = __builtin_amdgcn_ballot_w64(mine);
    if (lane == 0 && wave < 2u) {
        s_odd[3 + wave] = any_mine != 0 ? 1u : 0u;
    }
    __syncthreads();
    if ((s_odd[3] | s_odd[4]) == 0u) {
        return;
    }
    if (tid < PA_PROMPT_ROWS) {
        const size_t at = (size_t)(t0 + tid) * p.meta_stride[0];
        s_seq[tid] = mine ? p.meta[at] : NONE;
        s_len[tid] = mine ? pa_visible(p, p.meta[at + p.meta_stride[1]]) : 0u;
    }
    if (tid < 3) {
        s_odd[tid] = 0;
    }
    __syncthreads();
    if (tid < PA_PROMPT_ROWS) {
        const uint32_t seq = s_seq[tid];
        uint32_t longest = 0;
        bool first = true;
        for (uint32_t i = 0; i < tt; i += 4u) {  // (behind the tile's tokens: nobody's)
            const uint4 lens = *(const uint4 *)(s_len + i), seqs = *(const uint4 *)(s_seq + i);
            const uint32_t len[4] = {lens.x, lens.y, lens.z, lens.w}, other[4] = {seqs.x, seqs.y, seqs.z, seqs.w};
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) {
                const bool eq = other[e] == seq;
                first = first && !(eq && i + e < tid);
                longest = eq && len[e] > longest ? len[e] : longest;
            }
        }
        s_longest[tid] = longest;
        const uint64_t firsts = __builtin_amdgcn_ballot_w64(mine && first);
        if (lane == 0) {
            s_firsts[wave] = firsts;
        }
    }
    __syncthreads();

    const uint32_t row = 32u * rows + n, tl = row / p.group, g = row - tl * p.group;
    const bool have = tl < tt;
    const uint32_t row_seq = have ? s_seq[tl] : NONE;
    const uint32_t full_len = row_seq != NONE ? s_len[tl] : 0u;
    const uint32_t t = t0 + tl, qh = kvh * p.group + g;

    // the query of this lane's row: dimensions 16 c + 8 h .. + 7, scaled and split. Rows that are not contiguous pass
    // through LDS (element loads in a loop of their own instead of 64 copies of them here).
    float *staged = (float *)lds;  // [128][HD]
    static_assert(L::TOKENS >= PA_PROMPT_ROWS * HD * 4, "the query rows fit the stages");
    if (!p.q_vec) {
        for (uint32_t i = tid; i < PA_PROMPT_ROWS * HD; i += THREADS) {
            const uint32_t r = i / HD, token = r / p.group;
            if (token < tt && s_seq[token] != NONE) {
                staged[i] = pa_load(p.q, p.act_dtype, (size_t)(t0 + token) * p.q_stride[0] +
                                    (size_t)(kvh * p.group + (r - token * p.group)) * p.q_stride[1] + (i % HD) * p.q_stride[2]);
            }
        }
        __syncthreads();
    }
    float qv[QC][8];
    const size_t q_base = (size_t)t * p.q_stride[0] + (size_t)qh * p.q_stride[1];
#pragma unroll
    for (int c = 0; c < QC; ++c) {
        const uint32_t d = 16u * c + 8u * h;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            qv[c][e] = 0.0f;
        }
        if (row_seq != NONE) {
            if (!p.q_vec) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    qv[c][e] = staged[row * HD + d + e];
                }
            } else if (p.act_dtype == MARMOT_HIP_DTYPE_F32) {
                const float4 a = *(const float4 *)((const float *)p.q + q_base + d);
                const float4 b = *(const float4 *)((const float *)p.q + q_base + d + 4u);
                const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    qv[c][e] = v[e];
                }
            } else {
                const uint2 a = *(const uint2 *)((const uint16_t *)p.q + q_base + d);
                const uint2 b = *(const uint2 *)((const uint16_t *)p.q + q_base + d + 4u);
                const uint32_t words[4] = {a.x, a.y, b.x, b.y};
                const bool f16 = p.act_dtype == MARMOT_HIP_DTYPE_F16;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint16_t bits = (uint16_t)(words[e >> 1] >> (16 * (e & 1)));
                    qv[c][e] = f16 ? h2f(bits) : pa_bf2f(bits);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            qv[c][e] = p.scale != 1.0f ? qv[c][e] * p.scale : qv[c][e];
        }
    }
    // FLOAT16 parts: the row times the power of two that brings its largest value to 2^14 .. 2^15; `unit` undoes it on
    // the scores
    int up = 0;
    float unit = 1.0f;
    if constexpr (!BF16) {
        float most = 0.0f;
#pragma unroll
        for (int c = 0; c < QC; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                most = fmaxf(most, fabsf(qv[c][e]));
            }
        }
        up = pa_split_exponent(fmaxf(most, pa_xor32(most)));
        unit = ldexpf(1.0f, -up);
    }
    uint4 qpart[QREGS][QC];
    uint8_t *q_small = lds + L::Q + rows * 1024u + 16u * lane;
#pragma unroll
    for (int c = 0; c < QC; ++c) {
        uint32_t w[PARTS][4];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = BF16 ? qv[c][e] : ldexpf(qv[c][e], up);
#pragma unroll
            for (int part = 0; part < PARTS; ++part) {  // each remainder is exact in fp32
                uint32_t bits;
                if constexpr (BF16) {  // cut off: rounding up would make infinity of the largest values
                    bits = __float_as_uint(v) >> 16;
                    v -= pa_bf2f((uint16_t)bits);
                } else {
                    bits = f2h(v);
                    v -= h2f((uint16_t)bits);
                }
                w[part][e >> 1] = (e & 1) == 0 ? bits : (w[part][e >> 1] | (bits << 16));
            }
        }
#pragma unroll
        for (int part = 0; part < PARTS; ++part) {
            const uint4 v = make_uint4(w[part][0], w[part][1], w[part][2], w[part][3]);
            if (part < QREGS) {
                qpart[part][c] = v;
            } else {  // (both halves' wavefronts hold the same rows)
                *(uint4 *)(q_small + 4096 * (QC * (part - QREGS) + c)) = v;
            }
        }
    }

    if (!p.q_vec) {
        __syncthreads();
    }

    const pa_float16v zero = {};
    pa_float16v out[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d) {
        out[d] = zero;
    }
    float m = -INFINITY, lsum = 0.0f;  // of this wavefront's positions; lsum: of this lane's part of them
    const size_t head_base = (size_t)p.layer_idx * p.kv_stride[1] + (size_t)kvh * p.kv_stride[2];
    const uint8_t *keys = (const uint8_t *)((const uint16_t *)p.kv_k + head_base);
    const uint8_t *values = (const uint8_t *)((const uint16_t *)p.kv_v + head_base);
    // a thread's part of a tile: 16 bytes of every THREADS / (HD / 8)-th key row, four dimensions of four consecutive value rows.
    // (The chunk of dimension 4 i + e: that of dimension 4 i with 2 e in an exclusive or, 128 e bytes on.)
    const uint32_t v_at = pa_vt_chunk(4u * (tid % (HD / 4)), 2u * (tid / HD) + (tid / (HD / 4) & 1u)) + 8u * (tid / (HD / 2) & 1u);
    const uint32_t v_from = pa_vt_chunk(n, 4u * half + h);
    uint64_t *s_rows = (uint64_t *)(lds + L::ROWS);
    // tiles staged so far, over all sequences: keys in buffer count & 1, values at `now`, the ones before at `before`
    uint32_t count = 0, now = L::V0, before = L::V0 + 2u * L::V;
    pa_uint4 kreg[KN];
    uint2 vreg[4];
    uint64_t mask_next = 0;  // positions of the requested tile that exist

    auto uniform64 = [](uint64_t v) {
        return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
               (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32;
    };
    // (a look at every token instead is a chain of as many reads from LDS: 3 of the 30 us of 512 fresh tokens, 128 of them in a tile)
    uint64_t firsts = uniform64(s_firsts[0]), firsts_high = uniform64(s_firsts[1]);
    while ((firsts | firsts_high) != 0u) {
        uint32_t first;
        if (firsts != 0u) {
            first = (uint32_t)__builtin_ctzll(firsts);
            firsts &= firsts - 1u;
        } else {
            first = 64u + (uint32_t)__builtin_ctzll(firsts_high);
            firsts_high &= firsts_high - 1u;
        }
        const uint32_t longest = __builtin_amdgcn_readfirstlane(s_longest[first]);
        if (longest == 0u) {
            continue;
        }
        const uint32_t seq = __builtin_amdgcn_readfirstlane(s_seq[first]);
        const uint32_t row_len = row_seq == seq ? full_len : 0u;
        const uint32_t *table_row = p.table + (size_t)seq * p.table_stride[0];
        const uint32_t tiles = (longest + 63u) / 64u;
        // shares of PA_PROMPT_SHARE positions at least; the others hold nothing
        const uint32_t most = (longest + PA_PROMPT_SHARE - 1u) / PA_PROMPT_SHARE, shares = p.tile_splits < most ? p.tile_splits : most;
        const uint32_t per_share = (tiles + shares - 1u) / shares;
        const uint32_t begin = blockIdx.z * per_share;
        const uint32_t end = begin + per_share < tiles ? begin + per_share : tiles;
        if (begin >= end) {
            continue;
        }
        // The first wavefront locates the rows two tiles ahead, lane i position i; rows without a block read block 0.
        auto table_entry = [&](uint32_t tile) -> uint32_t {
            const uint32_t logical = (64u * tile + lane) >> p.shift;
            return table_row[(size_t)(logical < p.max_blocks ? logical : p.max_blocks - 1u) * p.table_stride[1]];
        };
        auto locate = [&](uint32_t tile, uint32_t tb) {
            const uint32_t pos = 64u * tile + lane, logical = pos >> p.shift, buffer = (tile - begin) & 1u;
            const bool ok = pos < longest && logical < p.max_blocks && tb != PA_NO_BLOCK && tb < p.kv_blocks;
            const uint64_t exist = __builtin_amdgcn_ballot_w64(ok);
            s_rows[64u * buffer + lane] = ok ? 2u * ((uint64_t)tb * p.kv_stride[0] + (uint64_t)(pos & p.mask) * p.kv_stride[3]) : 0u;
            if (lane == 0) {
                s_rows[128u + buffer] = exist;
            }
        };
        auto request = [&](uint32_t tile) {
            const uint32_t buffer = (tile - begin) & 1u;
            mask_next = uniform64(s_rows[128u + buffer]);
            uint32_t tid = threadIdx.x;
            asm volatile("" : "+v"(tid));  // (places formed from it here, not kept throughout: there are no registers for them)
            const uint64_t *k_rows = s_rows + 64u * buffer + tid / (HD / 8);
            const uint8_t *k_base = keys + 16u * (tid % (HD / 8));
#pragma unroll
            for (int i = 0; i < KN; ++i) {
                kreg[i] = *(const pa_uint4 *)(k_base + k_rows[THREADS / (HD / 8) * i]);
            }
            if (VUNITS == THREADS || tid < VUNITS) {
                const uint64_t *v_rows = s_rows + 64u * buffer + 4u * (tid / (HD / 4));
                const uint8_t *v_base = values + 8u * (tid % (HD / 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    vreg[e] = *(const uint2 *)(v_base + v_rows[e]);
                }
            }
        };
        auto store = [&](uint32_t number, uint32_t values_at) {
            uint32_t tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            uint8_t *stage = lds + (number & 1u) * L::K + tid / (HD / 8) * L::KROW + 16u * (tid % (HD / 8));
#pragma unroll
            for (int i = 0; i < KN; ++i) {
                *(pa_uint4 *)(stage + THREADS / (HD / 8) * i * L::KROW) = kreg[i];
            }
            if (VUNITS == THREADS || tid < VUNITS) {
                if (mask_next != ~0ull) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        vreg[e] = (mask_next >> (4u * (tid / (HD / 4)) + e)) & 1u ? vreg[e] : make_uint2(0, 0);
                    }
                }
                // largest halves as unsigned numbers (negative values) and as signed ones (positive values): has one of them all
                // bits of its exponent set?
                typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
                typedef short i16x2 __attribute__((ext_vector_type(2)));
                u16x2 below = {0, 0};
                i16x2 above = {0, 0};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const u16x2 ux = __builtin_bit_cast(u16x2, vreg[e].x), uy = __builtin_bit_cast(u16x2, vreg[e].y);
                    const i16x2 ix = __builtin_bit_cast(i16x2, vreg[e].x), iy = __builtin_bit_cast(i16x2, vreg[e].y);
                    below = __builtin_elementwise_max(below, __builtin_elementwise_max(ux, uy));
                    above = __builtin_elementwise_max(above, __builtin_elementwise_max(ix, iy));
                }
                constexpr uint32_t ONE = BF16 ? 0x00800080u : 0x04000400u;
                const uint32_t low = __builtin_bit_cast(uint32_t, below) & 0x7fff7fffu;
                const uint32_t high = __builtin_bit_cast(uint32_t, above) & 0x7fff7fffu;
                const uint32_t odd = (low + ONE) | (high + ONE);
                uint8_t *vt = lds + values_at;
                constexpr uint32_t LOW = 0x05040100u, HIGH = 0x07060302u;
                auto pair = [](uint32_t b, uint32_t a, uint32_t sel) { return __builtin_amdgcn_perm(b, a, sel); };
                *(uint2 *)(vt + v_at) = make_uint2(pair(vreg[1].x, vreg[0].x, LOW), pair(vreg[3].x, vreg[2].x, LOW));
                *(uint2 *)(vt + (v_at ^ 32u) + 128) = make_uint2(pair(vreg[1].x, vreg[0].x, HIGH), pair(vreg[3].x, vreg[2].x, HIGH));
                *(uint2 *)(vt + (v_at ^ 64u) + 256) = make_uint2(pair(vreg[1].y, vreg[0].y, LOW), pair(vreg[3].y, vreg[2].y, LOW));
                *(uint2 *)(vt + (v_at ^ 96u) + 384) = make_uint2(pair(vreg[1].y, vreg[0].y, HIGH), pair(vreg[3].y, vreg[2].y, HIGH));
                if ((odd & 0x80008000u) != 0u) {
                    s_odd[number % 3u] = number + 1u;
                }
            }
        };
        pa_float16v s = zero;
        uint32_t see = 0;   // the positions of this wavefront's half of a tile that the lane's row sees
        bool some = false;  // some row sees one of them
        auto scores = [&](uint32_t tile, uint32_t number, uint64_t mask) {
            const uint32_t p0 = 64u * tile + 32u * half;
            some = __builtin_amdgcn_ballot_w64(row_len > p0) != 0;
            if (!some) {
                return;
            }
            const uint8_t *stage = lds + (number & 1u) * L::K + (32u * half + n) * L::KROW + 16u * h;
            uint4 k[QC];
#pragma unroll
            for (int c = 0; c < QC; ++c) {
                k[c] = *(const uint4 *)(stage + 32u * c);
            }
            s = zero;
#pragma unroll
            for (int part = PARTS - 1; part >= 0; --part) {  // small parts first
#pragma unroll
                for (int c = 0; c < QC; ++c) {
                    const uint4 q = part < QREGS ? qpart[part < QREGS ? part : 0][c]
                                                 : *(const uint4 *)(q_small + 4096 * (QC * (part - QREGS) + c));
                    s = pa_mma32<BF16>(k[c], q, s);
                }
            }
            const uint32_t left = row_len > p0 ? row_len - p0 : 0u;
            see = (uint32_t)(mask >> (32u * half)) & (left >= 32u ? ~0u : (1u << left) - 1u);
            if (__builtin_amdgcn_ballot_w64(see != ~0u) != 0) {
                const uint32_t bits = see >> (4u * h);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[r] = (bits >> (8 * (r >> 2) + (r & 3))) & 1u ? s[r] : -INFINITY;
                }
            }
        };
        auto output = [&](uint32_t number, uint32_t values_at) {
            if (!some) {
                return;
            }
            const bool odd = __builtin_amdgcn_readfirstlane(s_odd[number % 3u]) == number + 1u;
            float big = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) {
                big = fmaxf(big, s[r]);
            }
            big = fmaxf(big, pa_xor32(big)) * unit;
            const float m_new = fmaxf(m, big);
            // While every score so far is -inf, weights are 0, and a sum above 0 says that there were scores at all (then the output is
            // NaN if it stays so over the whole row: exp(-inf + inf)); the first larger score drops it.
            const float corr = m == m_new ? 1.0f : pa_exp(m - m_new);
            const bool lost = m_new == -INFINITY;
            const float m_use = lost ? 0.0f : m_new;
            m = m_new;
            float w[16], sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                w[r] = pa_exp(__builtin_fmaf(s[r], unit, -m_use)) * UNIT;
                sum[r & 3] += w[r];
            }
            lsum = lsum * corr + ((sum[0] + sum[1]) + (sum[2] + sum[3])) + (lost && see != 0u ? 1.0f : 0.0f);
            const uint8_t *vt = lds + values_at;
            // The weights as operands, in parts; or as they are, weight r in word 8 (r / 8) + r % 8 of the first two parts, for a tile with
            // a value that is not finite: two FLOAT16 parts hold nothing below 2^-39, and 0 x infinity is not what a small weight gives
            uint32_t wp[2][PARTS][4] = {};
            if (odd) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    wp[r >> 3][(r >> 2) & 1][r & 3] = __float_as_uint(w[r]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float a = w[8 * i + 2 * e], b = w[8 * i + 2 * e + 1];
#pragma unroll
                        for (int part = 0; part < PARTS; ++part) {
                            if constexpr (BF16) {  // eight bits at a time, cut off: the third part is exact
                                const uint32_t ab = __float_as_uint(a), bb = __float_as_uint(b);
                                wp[i][part][e] = __builtin_amdgcn_perm(bb, ab, 0x07060302u);
                                a -= __uint_as_float(ab & 0xFFFF0000u);
                                b -= __uint_as_float(bb & 0xFFFF0000u);
                            } else {
                                const uint16_t ah = f2h(a), bh = f2h(b);
                                wp[i][part][e] = (uint32_t)ah | ((uint32_t)bh << 16);
                                a -= h2f(ah);
                                b -= h2f(bh);
                            }
                        }
                    }
                }
            }
            // The tile's products are summed by themselves, small parts first, and join the running output in one rounding
            // (a third of the error of a chain through the running output, and the rescaling costs nothing)
            uint4 v[2][2];
            auto read_v = [&](int d) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    v[d & 1][i] = *(const uint4 *)(vt + (v_from ^ (32u * i)) + 4096 * d);
                }
            };
            read_v(0);
            __builtin_amdgcn_s_setprio(1);  // in front of the other half's softmax (0.6 us of 147)
#pragma unroll
            for (int d = 0; d < DB; ++d) {
                pa_float16v tile_out = zero;
                if (d + 1 < DB) {
                    read_v(d + 1);
                }
                if (!odd) {
#pragma unroll
                    for (int part = PARTS - 1; part >= 0; --part) {
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            tile_out = pa_mma32<BF16>(
                                v[d & 1][i], make_uint4(wp[i][part][0], wp[i][part][1], wp[i][part][2], wp[i][part][3]), tile_out);
                        }
                    }
                } else {
                    uint32_t h = lane >> 5;
                    asm volatile("" : "+v"(h));
                    for (uint32_t i = 0; i < 32u; ++i) {
                        // position i: weight 4 (i / 8) + i % 4 of lane half (i / 4) % 2
                        const uint32_t at = 4u * (i >> 3) + (i & 3u);
                        uint32_t mine_w = 0;
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            mine_w = (uint32_t)r == at ? wp[r >> 3][(r >> 2) & 1][r & 3] : mine_w;
                        }
                        const float wi = __uint_as_float(__shfl(mine_w, (int)(n + 32u * ((i >> 2) & 1u))));
                        if ((see >> i) & 1u) {
                            const uint32_t chunk = 4u * half + 2u * (i >> 4) + ((i >> 2) & 1u), in = 8u * ((i >> 3) & 1u) + 2u * (i & 3u);
#pragma unroll
                            for (int r = 0; r < 16; ++r) {
                                const uint32_t dim = 32u * d + 8u * (r >> 2) + 4u * h + (r & 3);
                                const uint16_t one = *(const uint16_t *)(vt + pa_vt_chunk(dim, chunk) + in);
                                tile_out[r] = __builtin_fmaf(wi, BF16 ? pa_bf2f(one) : h2f(one), tile_out[r]);
                                __builtin_amdgcn_sched_barrier(0);  // (rare, and short of registers otherwise)
                            }
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    out[d][r] = __builtin_fmaf(out[d][r], corr, tile_out[r]);
                }
                asm volatile("" : "+v"(out[d]));  // in place, one after the other
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        };
        // Between two barriers tile k + 1 is stored, half 0 takes tile k whole, half 1 the output of tile k - 1 and then
        // the scores of tile k: one uses the matrix cores while the other is at its softmax. Tile k + 1 goes to buffers
        // last read before the barrier: the keys of tile k - 1, the values of tile k - 2.
        auto after = [&](uint32_t at) { return at == L::V0 + 2u * L::V ? L::V0 : at + L::V; };
        uint32_t entry = 0;
        if (wave == 0u) {
            const uint32_t entry0 = table_entry(begin), entry1 = table_entry(begin + 1u);
            entry = table_entry(begin + 2u);
            locate(begin, entry0);
            locate(begin + 1u, entry1);
        }
        __syncthreads();
        request(begin);
        store(count, now);
        uint64_t mask = mask_next;
        __syncthreads();
        for (uint32_t tile = begin; tile <= end; ++tile) {
            const bool more = tile + 1u < end;
            if (half == 0u && tile < end) {
                scores(tile, count, mask);
            }
            if (more) {
                request(tile + 1u);
                if (wave == 0u) {
                    locate(tile + 2u, entry);
                    entry = table_entry(tile + 3u);
                }
            }
            if (half == 0u ? tile < end : tile != begin) {
                output(count - half, half == 0u ? now : before);
            }
            // (the requests behind half 0's scores and the stores in front of half 1's: 1 - 2.5 % of long histories)
            const uint64_t mask_now = mask;
            if (more) {
                store(count + 1u, after(now));
                mask = mask_next;
            }
            if (half != 0u && tile < end) {
                scores(tile, count, mask_now);
            }
            if (tile == end) {
                break;  // (the stores of the next sequence's first tile go to other buffers than the last output's)
            }
            ++count;
            before = now;
            now = after(now);
            __syncthreads();
        }
    }

    // The halves' sums meet in LDS: each gives half of its dimensions to the other and keeps the other half
    lsum += pa_xor32(lsum);
    __syncthreads();
    {
        float2 *ml = (float2 *)(lds + L::MAIL);
        ml[tid] = make_float2(m, lsum);
        float4 *mail = (float4 *)lds + wave * (HD / 64 * 256u) + lane;
#pragma unroll
        for (int d = 0; d < DB / 2; ++d) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = half == 0u ? out[DB / 2 + d][4 * q + e] : out[d][4 * q + e];
                    out[d][4 * q + e] = half == 0u ? out[d][4 * q + e] : out[DB / 2 + d][4 * q + e];
                }
                mail[64 * (4 * d + q)] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        __syncthreads();
        const float2 other = ml[tid ^ 256u];
        const float m_all = fmaxf(m, other.x);
        const float f_own = m == m_all ? 1.0f : pa_exp(m - m_all), f_other = other.x == m_all ? 1.0f : pa_exp(other.x - m_all);
        lsum = __builtin_fmaf(other.y, f_other, lsum * f_own);
        m = m_all;
        const float4 *from = (const float4 *)lds + (wave ^ 4u) * (HD / 64 * 256u) + lane;
#pragma unroll
        for (int d = 0; d < DB / 2; ++d) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = from[64 * (4 * d + q)];
                const float add[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    out[d][4 * q + e] = __builtin_fmaf(add[e], f_other, out[d][4 * q + e] * f_own);
                }
            }
        }
    }
    const uint32_t dim0 = half * (HD / 2);
    if (row_seq == NONE) {
        return;
    }
    const bool bad = lsum != lsum;
    if (p.tile_splits > 1u) {
        float *part = p.partial + (((size_t)t * p.num_q_heads + qh) * p.partial_splits + blockIdx.z) * (HD + 2u);
        if (h == 0 && half == 0u) {
            part[0] = m;
            part[1] = lsum;
        }
        if (m == -INFINITY && !bad) {  // a share that holds nothing but scores of -inf, if any: k_pa_merge leaves its outputs alone
            return;
        }
#pragma unroll
        for (int d = 0; d < DB / 2; ++d) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float2 *dst = (float2 *)(part + 2 + dim0 + 32 * d + 8 * q + 4 * h);
                dst[0] = make_float2(out[d][4 * q], out[d][4 * q + 1]);
                dst[1] = make_float2(out[d][4 * q + 2], out[d][4 * q + 3]);
            }
        }
        return;
    }
    const float inv = bad || (m == -INFINITY && lsum > 0.0f) ? __uint_as_float(0x7fc00000u) : (lsum > 0.0f ? 1.0f / lsum : 0.0f);
    const size_t base = (size_t)t * p.out_stride[0] + (size_t)qh * p.out_stride[1];
#pragma unroll
    for (int d = 0; d < DB / 2; ++d) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t dim = dim0 + 32u * d + 8u * q + 4u * h;
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[e] = bad || lsum > 0.0f ? out[d][4 * q + e] * inv : 0.0f;
            }
            if (p.out_vec) {
                *(float4 *)((float *)p.out + base + dim) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pa_store(p.out, p.act_dtype, base + (size_t)(dim + e) * p.out_stride[2], o[e]);
                }
            }
        }
    }
}

// the shares of a (token, head) pair's history: out = sum_s o_s * exp(M_s - M) / sum_s l_s * exp(M_s - M)
// (TILES: beside the prompt kernel, whose tokens have a split count of their own; without it the look at p.tiled costs a
// decode step 0.9 us)
template <bool TILES>
__global__ __launch_bounds__(256) void k_pa_merge(const PaParams p) {
    __shared__ float s_big[64], s_tot[64];  // splits <= 64
    const uint32_t t = blockIdx.x, qh = blockIdx.y;
    uint32_t splits = p.splits;
    if constexpr (TILES) {
        const uint32_t tiled = __builtin_amdgcn_readfirstlane(p.tiled[t]);
        splits = tiled == 1u ? p.tile_splits : (tiled == 2u ? p.share_splits : splits);
        if (splits <= 1u) {
            return;  // the token's own kernel has written its output
        }
    }
    const float *part = p.partial + ((size_t)t * p.num_q_heads + qh) * (TILES ? p.partial_splits : splits) * (p.head_dim + 2u);
    if (threadIdx.x < splits) {
        s_big[threadIdx.x] = part[(size_t)threadIdx.x * (p.head_dim + 2u)];
        s_tot[threadIdx.x] = part[(size_t)threadIdx.x * (p.head_dim + 2u) + 1];
    }
    __syncthreads();
    float big = -INFINITY;
    for (uint32_t z = 0; z < splits; ++z) {
        big = fmaxf(big, s_big[z]);
    }
    const size_t out_base = (size_t)t * p.out_stride[0] + (size_t)qh * p.out_stride[1];
    for (uint32_t d = threadIdx.x; d < p.head_dim; d += blockDim.x) {
        float o = 0.0f, total = 0.0f;
        bool bad = false;  // a share saw a NaN score, or all of them none but -inf (k_pa_prompt: a sum beside that maximum)
        for (uint32_t z = 0; z < splits; ++z) {
            bad = bad || s_tot[z] != s_tot[z] || (TILES && big == -INFINITY && s_tot[z] > 0.0f);
        }
        if (big != -INFINITY) {
            for (uint32_t z = 0; z < splits; ++z) {
                const bool empty = TILES && s_big[z] == -INFINITY;  // (k_pa_prompt leaves the outputs of such a share unwritten)
                const float f = s_big[z] == -INFINITY ? 0.0f : pa_exp(s_big[z] - big);
                total = __builtin_fmaf(s_tot[z], f, total);
                const float v = part[(size_t)z * (p.head_dim + 2u) + 2 + d];
                o = empty ? o : __builtin_fmaf(v, f, o);
            }
        }
        o = bad ? __uint_as_float(0x7fc00000u) : (total > 0.0f ? o * (1.0f / total) : 0.0f);
        pa_store(p.out, p.act_dtype, out_base + (size_t)d * p.out_stride[2], o);
    }
}

template <int EPL, int QH>
static void pa_launch(marmot_hip_device *dev, const PaParams &p) {
    hipLaunchKernelGGL((k_pa_attend<EPL, QH>), dim3(p.token_count, p.num_q_heads / QH, p.share_splits),
                       dim3(16 * PA_GROUPS), 0, dev->stream, p);
}

template <int HD, bool BF16>
static int pa_launch_prompt(marmot_hip_device *dev, const PaParams &p) {
    MH_TRY(allow_large_lds(dev, (const void *)k_pa_prompt<HD, BF16>));
    const unsigned tiles = (p.token_count + p.tile_tokens - 1) / p.tile_tokens;
    hipLaunchKernelGGL((k_pa_prompt<HD, BF16>), dim3(tiles, p.num_kv_heads, p.tile_splits), dim3(64 * PA_PROMPT_WAVES),
                       (PaPromptLds<HD, BF16>::BYTES), dev->stream, p);
    MH_HIP(hipGetLastError());
    return MARMOT_HIP_SUCCESS;
}

// k_pa_write_rows takes the call: rows of whole 16-byte pieces, in the cache and in the new rows, and more of them than run at once
// as workgroups of their own (a decode step of 16 tokens of 8 heads is 0.7 % of a layer faster with those: all start together)
static bool pa_write_rows(const marmot_hip_device *dev, const marmot_hip_paged_attention_t *a, size_t act_size) {
    if ((size_t)a->token_count * a->num_kv_heads < 4 * (size_t)dev->props.multiProcessorCount) {
        return false;
    }
    bool ok = (a->kv_dtype == MARMOT_HIP_DTYPE_F16 || a->kv_dtype == MARMOT_HIP_DTYPE_BF16) && a->head_dim % 8 == 0 &&
              a->kv_stride[4] == 1 && a->k_stride[2] == 1 && a->v_stride[2] == 1;
    ok = ok && (((uintptr_t)a->d_kv_k | (uintptr_t)a->d_kv_v | (uintptr_t)a->d_k_new | (uintptr_t)a->d_v_new) & 15) == 0;
    for (int i = 0; i < 4; ++i) {
        ok = ok && (a->kv_stride[i] * 2) % 16 == 0;
    }
    for (int i = 0; i < 2; ++i) {
        ok = ok && (a->k_stride[i] * act_size) % 16 == 0 && (a->v_stride[i] * act_size) % 16 == 0;
    }
    return ok;
}

static bool pa_float_dtype(int d) {
    return d == MARMOT_HIP_DTYPE_F32 || d == MARMOT_HIP_DTYPE_F16 || d == MARMOT_HIP_DTYPE_BF16;
}

static size_t pa_elem_size(int d) {
    return d == MARMOT_HIP_DTYPE_F32 ? 4 : (d == MARMOT_HIP_DTYPE_F8_E4M3 ? 1 : 2);
}

} // namespace mh

using namespace mh;

extern "C" int marmot_hip_fill_bytes_internal(marmot_hip_device_t *dev, void *d_dst, int value, size_t size);

extern "C" int marmot_hip_paged_attention(marmot_hip_device_t *dev, const marmot_hip_paged_attention_t *a,
                                          int validate_meta) {
    if (dev == nullptr) {
        return set_error(MARMOT_HIP_ERROR_DEVICE_NOT_AVAILABLE, "HIP device is not initialised");
    }
    if (a == nullptr || a->d_token_meta == nullptr || a->d_q == nullptr || a->d_k_new == nullptr ||
        a->d_v_new == nullptr || a->d_kv_k == nullptr || a->d_kv_v == nullptr || a->d_block_table == nullptr ||
        a->d_out == nullptr) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention descriptor invalid");
    }
    if (a->token_count == 0) {
        return MARMOT_HIP_SUCCESS;
    }
    if (a->num_q_heads == 0 || a->num_kv_heads == 0 || a->head_dim == 0 || a->block_size == 0) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention requires non-zero dimensions");
    }
    if ((a->block_size & (a->block_size - 1u)) != 0) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention block_size must be power of two");
    }
    if (a->num_q_heads % a->num_kv_heads != 0) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention requires num_q_heads divisible by num_kv_heads");
    }
    const bool fp8 = a->kv_dtype == MARMOT_HIP_DTYPE_F8_E4M3;
    if (!pa_float_dtype(a->act_dtype) || (!fp8 && !pa_float_dtype(a->kv_dtype))) {
        return set_error(MARMOT_HIP_ERROR_UNSUPPORTED_DTYPE, "paged_attention dtype not supported");
    }
    if (fp8 && (a->d_kv_k_scale == nullptr || a->d_kv_v_scale == nullptr)) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention FP8 KV requires scale tensors");
    }
    if (!fp8 && (a->d_kv_k_scale != nullptr || a->d_kv_v_scale != nullptr)) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "paged_attention scale tensors require FP8 KV");
    }
    if (a->kv_layers <= a->layer_idx) {
        return set_error(MARMOT_HIP_ERROR_DIMENSION_MISMATCH, "paged_attention layer_idx out of range");
    }
    if (a->head_dim > 256) {
        return set_error(MARMOT_HIP_ERROR_NOT_IMPLEMENTED, "paged_attention: head_dim %u is more than 256", a->head_dim);
    }
    if (a->num_q_heads > 65535u || a->num_kv_heads > 65535u) {
        return set_error(MARMOT_HIP_ERROR_NOT_IMPLEMENTED, "paged_attention: more than 65535 heads");
    }
    MH_HIP(hipSetDevice(dev->device_index));
    PaParams p;
    p.token_count = a->token_count, p.layer_idx = a->layer_idx, p.num_q_heads = a->num_q_heads;
    p.num_kv_heads = a->num_kv_heads, p.head_dim = a->head_dim, p.block_size = a->block_size;
    p.scale = a->scale, p.act_dtype = a->act_dtype, p.kv_dtype = a->kv_dtype;
    p.meta = a->d_token_meta, p.q = a->d_q, p.k_new = a->d_k_new, p.v_new = a->d_v_new;
    p.kv_k = a->d_kv_k, p.kv_v = a->d_kv_v, p.table = a->d_block_table, p.out = a->d_out;
    for (int i = 0; i < 2; ++i) {
        p.meta_stride[i] = a->meta_stride[i];
        p.table_stride[i] = a->table_stride[i];
    }
    for (int i = 0; i < 3; ++i) {
        p.q_stride[i] = a->q_stride[i], p.k_stride[i] = a->k_stride[i], p.v_stride[i] = a->v_stride[i];
        p.out_stride[i] = a->out_stride[i];
    }
    for (int i = 0; i < 5; ++i) {
        p.kv_stride[i] = a->kv_stride[i];
    }
    p.kv_blocks = a->kv_blocks, p.kv_layers = a->kv_layers, p.max_seqs = a->max_seqs, p.max_blocks = a->max_blocks_per_seq;
    p.shift = 0;
    while ((1u << p.shift) < a->block_size) {
        ++p.shift;
    }
    p.mask = a->block_size - 1u;
    p.group = a->num_q_heads / a->num_kv_heads;
    const int epl = a->head_dim <= 64 ? 4 : (a->head_dim <= 128 ? 8 : 16);
    // 16-byte runs: the head dimension is exactly 16 lanes x EPL values, unit stride, every row start 16-byte aligned
    const size_t asz = pa_elem_size(a->act_dtype), ksz = pa_elem_size(a->kv_dtype);
    const size_t run_a = (size_t)epl * asz < 16 ? (size_t)epl * asz : 16, run_k = (size_t)epl * ksz < 16 ? (size_t)epl * ksz : 16;
    const bool exact = a->head_dim == (uint32_t)(16 * epl);
    p.q_vec = exact && a->q_stride[2] == 1 && (((uintptr_t)a->d_q) % run_a) == 0 && (a->q_stride[0] * asz) % run_a == 0 &&
              (a->q_stride[1] * asz) % run_a == 0;
    p.kv_vec = exact && a->kv_stride[4] == 1 && (((uintptr_t)a->d_kv_k) % run_k) == 0 &&
               (((uintptr_t)a->d_kv_v) % run_k) == 0;
    for (int i = 0; i < 4 && p.kv_vec; ++i) {
        p.kv_vec = (a->kv_stride[i] * ksz) % run_k == 0;
    }
    p.k_scale = a->d_kv_k_scale, p.v_scale = a->d_kv_v_scale;
    for (int i = 0; i < 3; ++i) {
        p.scale_stride[i] = a->scale_stride[i];
    }
    p.new_kmax = p.new_vmax = p.min_off = p.claim = nullptr;
    p.flag = nullptr;
    if (validate_meta != 0 && !dev->capturing) {
        void *ws = nullptr;
        MH_TRY(workspace_reserve(dev, 256, &ws));
        p.flag = (int *)ws;
        MH_TRY(marmot_hip_fill_bytes_internal(dev, ws, 0, sizeof(int)));
        hipLaunchKernelGGL(k_pa_check, dim3((a->token_count + 255) / 256), dim3(256), 0, dev->stream, p);
        MH_HIP(hipGetLastError());
        int host_flag = 0;
        MH_HIP(hipMemcpyAsync(&host_flag, p.flag, sizeof(int), hipMemcpyDeviceToHost, dev->stream));
        MH_HIP(hipStreamSynchronize(dev->stream));
        if (host_flag != 0) {
            return set_error(MARMOT_HIP_ERROR_DIMENSION_MISMATCH,
                             "paged_attention seq_slot or kv_slot block out of range at token %u",
                             a->token_count - (uint32_t)host_flag);
        }
    }
    // workspace: [fp8 scratch][the tokens in tiles][partial results of split histories]
    const size_t fp8_words = fp8 ? 3 * a->kv_blocks * a->num_kv_heads + a->kv_blocks : 0;
    const size_t fp8_bytes = (fp8_words * sizeof(uint32_t) + 255) & ~(size_t)255;
    // query heads per workgroup: as many heads of one key / value head as the LDS tile of the final merge allows
    const int qh_max = epl == 16 ? 2 : 4;
    const int qh = (p.group % 4 == 0 && qh_max >= 4) ? 4 : (p.group % 2 == 0 ? 2 : 1);
    // few (token, heads) pairs (a decode step): the history is split over workgroups until the chip is about eight
    // (three for the matrix-core kernel) workgroups per compute unit deep, and a second kernel joins the shares
    const size_t pairs = (size_t)a->token_count * (a->num_q_heads / (uint32_t)qh);
    // FLOAT16 cache rows of 128 contiguous values in blocks of 16 positions or more: the scores on the matrix cores
    const bool kv_bf16 = a->kv_dtype == MARMOT_HIP_DTYPE_BF16;
    bool rows16 = (((uintptr_t)a->d_kv_k) & 15) == 0;  // FLOAT8_E4M3: 16 codes per load of a key row
    for (int i = 0; i < 4; ++i) {
        rows16 = rows16 && (a->kv_stride[i] * ksz) % 16 == 0;
    }
    const bool mfma_scores = (a->kv_dtype == MARMOT_HIP_DTYPE_F16 || kv_bf16 || (fp8 && rows16)) && p.kv_vec &&
                             a->head_dim == 128 && a->block_size >= 16 && !dev->knobs.no_attention_mfma;
    // (measured, 16 sequences x 4096 / x 512 positions, 32 / 8 heads: the matrix-core kernel 57.6 / 22.1 us at eight
    // workgroups per compute unit, 56.2 / 16.2 at four, 50.5 / 17.0 at three, 52.1 / 15.5 at two, 76.1 / 17.0 at one)
    const size_t want = (mfma_scores ? 3u : 8u) * (size_t)dev->props.multiProcessorCount;
    p.splits = 1;
    p.partial = nullptr;
    if (pairs * 2 <= want) {
        size_t sp = (want + pairs - 1) / pairs;
        p.splits = (uint32_t)(sp > 64 ? 64 : sp);
    }
    // Prompts: k_pa_prompt beside the kernel per token. Which tokens it takes is found on the device (pa_in_run): those of
    // calls with PA_PROMPT_WORK (token, head group, position) triples and more, counted with the longest history; a call of
    // fewer than PA_MANY tokens needs 2 PA_LONG positions too. Whole call, us per token / tiles, 32 / 8 heads of 128, FLOAT16:
    // fresh prompts of 100 tokens 15.5 / 29, 300 41.5 / 41.5, 400 56 / 45, 440 65 / 47, 512 78 / 49, 1024 210 / 65; 16 tokens
    // of four sequences over 1000 42 / 48, of BFLOAT16 64 tokens over 4000 115 / 45, 4 x 8 over 100 18 / 47; 32 / 8 heads of 64,
    // 100 tokens 23 / 24, 200 31 / 28, 300 50 / 31, 4 x 100 over 500 138 / 45. (The line, 430 fresh tokens here, is that of slower
    // tiles: from 300 tokens on, 200 with rows of 64, these would not lose.) It is launched where that can be: two tokens and
    // more per row of the block table, or PA_ANY_TABLE tokens (a decode step has one token per row at most and would pay for
    // an empty launch), and room for such a history in the table. A table with more room than the call needs costs the
    // empty launch: 100 fresh tokens 16.2 / 21.3, 256 in 32 short runs 22.0 / 28.5, 512 decode tokens over 100 54.2 / 56.7.
    // 16-byte key rows, 8-byte value rows.
    const bool any = dev->knobs.attention_prompt_any, many = a->token_count >= PA_MANY;
    const size_t enough = (PA_PROMPT_WORK + pairs - 1) / pairs, least = many || enough > 2 * PA_LONG ? enough : 2 * PA_LONG;
    const bool runs = a->token_count / 2 >= a->max_seqs;
    const bool prompt_size = (runs || a->token_count >= PA_ANY_TABLE) && (size_t)p.max_blocks * a->block_size >= least;
    bool prompt = (a->kv_dtype == MARMOT_HIP_DTYPE_F16 || kv_bf16) && rows16 && p.kv_vec &&
                        (a->head_dim == 64 || a->head_dim == 128) && p.group <= 32 && !dev->knobs.no_attention_mfma &&
                        (prompt_size || any);
    // (a history counts in whole blocks, like the room for it)
    p.long_from = any ? 0u : (uint32_t)(least > p.mask ? least - p.mask : 1u);
    p.tile_tokens = 0;
    p.tile_splits = 1, p.share_splits = p.splits;
    p.out_vec = 0;
    if (prompt) {
        p.tile_tokens = PA_PROMPT_ROWS / p.group;
        p.out_vec = a->act_dtype == MARMOT_HIP_DTYPE_F32 && a->out_stride[2] == 1 && (((uintptr_t)a->d_out) & 15) == 0 &&
                    a->out_stride[0] % 4 == 0 && a->out_stride[1] % 4 == 0;
        const size_t tiles = (a->token_count + p.tile_tokens - 1) / p.tile_tokens * a->num_kv_heads;
        // (what may be a decode step of many sequences is spared the launch that joins two shares: 512 x 100 positions
        // 57.9 us without tiles, 65.3 with both launches)
        const size_t cus = (size_t)dev->props.multiProcessorCount, sp = !runs && 2 * tiles >= cus ? 1 : cus / tiles;
        p.tile_splits = (uint32_t)(sp < 1 ? 1 : (sp > 16 ? 16 : sp));
        const uint32_t shares = p.tile_splits < PA_SHARES ? p.tile_splits : PA_SHARES;
        p.share_splits = runs && shares > p.splits ? shares : p.splits;
    }
    size_t tiled_bytes = 0, partial_bytes = 0;
    auto scratch = [&]() {
        p.partial_splits = p.share_splits > p.tile_splits ? p.share_splits : p.tile_splits;
        tiled_bytes = prompt ? ((size_t)a->token_count * sizeof(uint32_t) + 255) & ~(size_t)255 : 0;
        partial_bytes = p.partial_splits > 1u ? (size_t)a->token_count * a->num_q_heads * p.partial_splits *
                                                    (a->head_dim + 2u) * sizeof(float)
                                              : 0;
        return fp8_bytes + tiled_bytes + partial_bytes;
    };
    if (scratch() > workspace_room(dev) && prompt) {  // captured without an eager run before: the kernel per token needs less
        prompt = false;
        p.tile_tokens = 0, p.tile_splits = 1, p.share_splits = p.splits;
        (void)scratch();
    }
    p.tiled = nullptr;
    if (fp8_bytes + tiled_bytes + partial_bytes != 0) {
        void *ws = nullptr;
        MH_TRY(workspace_reserve(dev, fp8_bytes + tiled_bytes + partial_bytes, &ws));
        if (fp8) {
            p.new_kmax = (uint32_t *)ws;
            p.new_vmax = p.new_kmax + a->kv_blocks * a->num_kv_heads;
            p.min_off = p.new_vmax + a->kv_blocks * a->num_kv_heads;
            p.claim = p.min_off + a->kv_blocks;
        }
        p.tiled = prompt ? (uint32_t *)((uint8_t *)ws + fp8_bytes) : nullptr;
        p.partial = p.partial_splits > 1u ? (float *)((uint8_t *)ws + fp8_bytes + tiled_bytes) : nullptr;
    }
    const dim3 per_token(a->token_count, a->num_kv_heads);
    if (fp8) {
        const size_t cells = a->kv_blocks * a->num_kv_heads;
        if (cells > ((size_t)1 << 32)) {
            return set_error(MARMOT_HIP_ERROR_NOT_IMPLEMENTED, "paged_attention: FP8 cache of %zu blocks", a->kv_blocks);
        }
        if (a->token_count <= PA_FP8_ONE_TOKENS && !dev->knobs.no_fp8_update_fused) {
            hipLaunchKernelGGL(k_pa_fp8_update, per_token, dim3(128), 0, dev->stream, p);
        } else {
            hipLaunchKernelGGL(k_pa_fp8_init, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, dev->stream, p);
            hipLaunchKernelGGL(k_pa_fp8_scan_new, per_token, dim3(128), 0, dev->stream, p);
            hipLaunchKernelGGL(k_pa_fp8_rescale, per_token, dim3(128), 0, dev->stream, p);
            hipLaunchKernelGGL(k_pa_fp8_store, per_token, dim3(128), 0, dev->stream, p);
        }
    } else if (pa_write_rows(dev, a, asz)) {
        hipLaunchKernelGGL(k_pa_write_rows, dim3(a->token_count), dim3(PA_WRITE_THREADS + (prompt ? 64 : 0)), 0, dev->stream, p);
    } else {
        hipLaunchKernelGGL(k_pa_write, per_token, dim3(a->head_dim <= 64 ? 64 : 128), 0, dev->stream, p);
    }
    MH_HIP(hipGetLastError());
    if (prompt) {
        if (kv_bf16) {
            MH_TRY((a->head_dim == 64 ? pa_launch_prompt<64, true>(dev, p) : pa_launch_prompt<128, true>(dev, p)));
        } else {
            MH_TRY((a->head_dim == 64 ? pa_launch_prompt<64, false>(dev, p) : pa_launch_prompt<128, false>(dev, p)));
        }
    }
    if (mfma_scores) {
        const dim3 grid(p.token_count, p.num_q_heads / (uint32_t)qh, p.share_splits), block(256);
        // FLOAT8_E4M3 decode steps over long contexts (few tokens, a block table of 2048 positions or more): the form
        // whose tile loop is pipelined (16 x 4096 positions 60.7 -> 48.7 us). It needs the registers of a third
        // resident wavefront per SIMD, which short histories and prompts miss more than they gain (FLOAT16, pipeline
        // compiled in: 16 x 512 positions 18.7 -> 23.9 us, a prompt of 512 tokens 76 -> 105 us), and a FLOAT16 cache at
        // 4096 positions runs at the memory's rate either way (53.0 / 53.0 us).
        const bool pipe = fp8 && p.splits > 1u && (size_t)p.max_blocks * a->block_size >= 2048u;
        if (fp8 && pipe) {
            if (qh == 4) {
                hipLaunchKernelGGL((k_pa_attend_mfma<4, PA_KV_FP8, true>), grid, block, 0, dev->stream, p);
            } else if (qh == 2) {
                hipLaunchKernelGGL((k_pa_attend_mfma<2, PA_KV_FP8, true>), grid, block, 0, dev->stream, p);
            } else {
                hipLaunchKernelGGL((k_pa_attend_mfma<1, PA_KV_FP8, true>), grid, block, 0, dev->stream, p);
            }
        } else if (fp8) {
            if (qh == 4) {
                hipLaunchKernelGGL((k_pa_attend_mfma<4, PA_KV_FP8, false>), grid, block, 0, dev->stream, p);
            } else if (qh == 2) {
                hipLaunchKernelGGL((k_pa_attend_mfma<2, PA_KV_FP8, false>), grid, block, 0, dev->stream, p);
            } else {
                hipLaunchKernelGGL((k_pa_attend_mfma<1, PA_KV_FP8, false>), grid, block, 0, dev->stream, p);
            }
        } else if (kv_bf16) {
            if (qh == 4) {
                hipLaunchKernelGGL((k_pa_attend_mfma<4, PA_KV_BF16, false>), grid, block, 0, dev->stream, p);
            } else if (qh == 2) {
                hipLaunchKernelGGL((k_pa_attend_mfma<2, PA_KV_BF16, false>), grid, block, 0, dev->stream, p);
            } else {
                hipLaunchKernelGGL((k_pa_attend_mfma<1, PA_KV_BF16, false>), grid, block, 0, dev->stream, p);
            }
        } else if (qh == 4) {
            hipLaunchKernelGGL((k_pa_attend_mfma<4, PA_KV_F16, false>), grid, block, 0, dev->stream, p);
        } else if (qh == 2) {
            hipLaunchKernelGGL((k_pa_attend_mfma<2, PA_KV_F16, false>), grid, block, 0, dev->stream, p);
        } else {
            hipLaunchKernelGGL((k_pa_attend_mfma<1, PA_KV_F16, false>), grid, block, 0, dev->stream, p);
        }
    } else if (epl == 4) {
        qh == 4 ? pa_launch<4, 4>(dev, p) : qh == 2 ? pa_launch<4, 2>(dev, p) : pa_launch<4, 1>(dev, p);
    } else if (epl == 8) {
        qh == 4 ? pa_launch<8, 4>(dev, p) : qh == 2 ? pa_launch<8, 2>(dev, p) : pa_launch<8, 1>(dev, p);
    } else {
        qh == 2 ? pa_launch<16, 2>(dev, p) : pa_launch<16, 1>(dev, p);
    }
    MH_HIP(hipGetLastError());
    if (p.partial_splits > 1u) {
        const dim3 grid(a->token_count, a->num_q_heads), block(a->head_dim <= 64 ? 64 : 128);
        if (prompt) {
            hipLaunchKernelGGL(k_pa_merge<true>, grid, block, 0, dev->stream, p);
        } else {
            hipLaunchKernelGGL(k_pa_merge<false>, grid, block, 0, dev->stream, p);
        }
        MH_HIP(hipGetLastError());
    }
    set_route(prompt        ? "paged_attention_tiles"
              : mfma_scores ? "paged_attention_mfma_scores"
                            : "paged_attention");
    return MARMOT_HIP_SUCCESS;
}
