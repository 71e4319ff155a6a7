// MoE on the HIP backend: router helpers (top-k, softmax over the selected logits) and the grouped
// expert FFN: route sort -> shared activation quantization -> grouped gate/up matvec -> SwiGLU + requantize ->
// grouped down matvec -> weighted combine in the reference's accumulation order.
// Compile with -ffp-contract=off.
#include "mh_common.h"

#include <float.h>
#include <stdlib.h>

namespace mh {

constexpr int MOE_ITEM_COLS = 8;   // routes per grouped work item (16 or 32 when experts see many routes, see moe_item_cols)
// Routes per expert from which prompts take the tiled GEMM (mh_gemm_planes.hip, 64 routes per item) instead of passes of
// 16 or 32 routes, given two of its tiles per compute unit in both projections. us of whole calls, passes / tiled, E = 128, top 8,
// H = 2048, F = 768, at 12, 16, 24, 32, 56 and 128 routes per expert:
//   Q4_K 137 / 131, 161 / 133, 171 / 143, 210 / 155, 303 / 196, 600 / 361
//   Q5_K 149 / 152, 174 / 155, 204 / 165, 262 / 174, 364 / 212, 730 / 403
//   Q6_K 225 / 170, 276 / 173, 376 / 183, 439 / 194, 718 / 240, 1417 / 447
// (64 experts, top 4, F = 1024: Q4_K 88 / 92, 100 / 89, 107 / 95; Q5_K 99 / 106, 117 / 108, 137 / 114.) The line is that of the kernel
// this one replaced (248 / 182 at 32 routes); with this one passes lose from 16 routes on, and from 12 on for Q6_K.
constexpr size_t MOE_TILED_ROUTES = 32;
constexpr int MOE_MAX_EXPERTS = 1024;
constexpr int MOE_MAX_TOPK = 64;

// ------------------------------------------------------------------ top-k (cpu_topk_impl, moe_ops.c:789-889)
// The reference inserts the columns in ascending order into a k-long list sorted by value, a new value going in
// front of the first strictly smaller one: the result is the first k columns under the total order (value
// descending, column ascending) among the values greater than -FLT_MAX; NaNs never compare true and are skipped;
// unfilled slots keep (-FLT_MAX, -1). One wavefront per row selects that sequence directly: round r finds the
// largest element that comes strictly after the previous pick in the same order.
__global__ __launch_bounds__(256) void k_topk(const float *__restrict__ x, size_t rows, size_t cols, size_t k,
                                              float *__restrict__ values, int32_t *__restrict__ indices) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= rows) {
        return;  // uniform per wavefront
    }
    const float *in = x + row * cols;
    float last_v = INFINITY;
    int last_i = -1;
    bool done = false;
    for (size_t r = 0; r < k; ++r) {
        float bv = -FLT_MAX;
        int bi = -1;
        if (!done) {
            for (size_t col = lane; col < cols; col += 64) {
                const float v = in[col];
                const bool after_last = v < last_v || (v == last_v && (int)col > last_i);
                if (after_last && v > bv) {  // ascending columns: an equal later value never replaces
                    bv = v;
                    bi = (int)col;
                }
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const float ov = __shfl_xor(bv, d, 64);
                const int oi = __shfl_xor(bi, d, 64);
                if (ov > bv || (ov == bv && oi >= 0 && oi < bi)) {
                    bv = ov;
                    bi = oi;
                }
            }
            if (bi < 0) {
                done = true;
            } else {
                last_v = bv;
                last_i = bi;
            }
        }
        if (lane == 0) {
            values[row * k + r] = bv;
            indices[row * k + r] = bi;
        }
    }
}

// softmax over each row of k selected logits: max-subtract, expf, in-order sum, divide
__global__ __launch_bounds__(64) void k_softmax_rows(const float *__restrict__ x, size_t rows, size_t k,
                                                     float *__restrict__ out) {
    const size_t row = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows) {
        return;
    }
    const float *in = x + row * k;
    float *o = out + row * k;
    float mx = in[0];
    for (size_t i = 1; i < k; ++i) {
        mx = in[i] > mx ? in[i] : mx;
    }
    float sum = 0.0f;
    for (size_t i = 0; i < k; ++i) {
        const float e = expf(in[i] - mx);
        o[i] = e;
        sum += e;
    }
    for (size_t i = 0; i < k; ++i) {
        o[i] = o[i] / sum;
    }
}

// ------------------------------------------------------------------ route sort
// cpu_moe_execute_grouped (moe_ops.c:905-974): count routes per expert, exclusive prefix over experts, then a
// stable fill in token-then-slot order. `decode_order` reproduces cpu_moe_execute_decode (moe_ops.c:643-717), where
// experts are laid out in order of first appearance instead of ascending id. Also cuts every expert's segment into
// work items of up to MOE_ITEM_COLS routes for the grouped matvec.
struct RouteArgs {
    const int32_t *topk_ids;      // [T, k]
    const float *topk_weights;    // [T, k]
    float *weights;               // [T, k] a copy: the combine runs when the caller's may already be overwritten (by d_out)
    uint32_t *sorted_tokens;      // [routes]
    int *route_pos;               // [T, k] position of each (token, slot) in the sorted order
    int4 *items;                  // work items
    int *n_items;
    int *error_flag;              // 1 when an expert id is out of range, else 0: device memory, or pinned host memory
    int T, k, E;
    int decode_order;
    int item_cols;                // routes per work item: 8, 16, 32 or 64
    int id_bits;                  // bits of an expert id
    int span;                     // routes per workgroup
    int *table;                   // [workgroups, E + 1] routes per expert, and whether an id is bad; null for one workgroup
};

constexpr int MOE_ROUTE_LDS = 4096;    // routes of a workgroup whose expert ids are kept in LDS
constexpr int MOE_ROUTE_WAVES = 16;    // wavefronts of the route kernel; each fills one contiguous chunk of routes
// From more routes than this on the sort is spread over workgroups: one launch counts every workgroup's routes, in the next
// each places its own. One compute unit alone is bound by its atomics in LDS and by stores to scattered addresses
// (128 experts, us of one workgroup and the launch that wrote its records / of these two: 2240 routes 10.1 / 9.7, 4096
// 11.6 / 9.8, 8192 15.7 / 9.8, 16384 24.4 / 11.4; the ids of 16384 routes kept in LDS left the one workgroup at 23).
constexpr int MOE_SPLIT_ROUTES = 2048;
constexpr int MOE_SPLIT_SPAN = 1024;   // routes per workgroup: one round of every wavefront
constexpr int MOE_SPLIT_GROUPS = 64;   // at most, as each reads every one's counts; with more routes the spans grow

// exclusive prefix sum over the 64 lanes of a wavefront; *total receives the sum over all lanes
__device__ __forceinline__ int wave_excl_scan(int v, int lane, int *total) {
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d, 64);
        if (lane >= d) {
            incl += up;
        }
    }
    *total = __shfl(incl, 63, 64);
    return incl - v;
}

// rank = number of lower lanes holding the same id, cnt = number of lanes holding it. One ballot per bit of the ids (`bits`
// of them; id -1 counts as an id of its own through its sign bit).
__device__ __forceinline__ void wave_rank(int id, int lane, int bits, int *rank, int *cnt) {
    unsigned long long same = __ballot(id < 0);
    same = id < 0 ? same : ~same;
    for (int i = 0; i < bits; ++i) {
        const bool set = (id >> i) & 1;
        const unsigned long long with = __ballot(set);
        same &= set ? with : ~with;
    }
    *rank = __builtin_popcountll(same & ((1ull << lane) - 1ull));
    *cnt = __builtin_popcountll(same);
}

__device__ __forceinline__ void route_emit(const RouteArgs &a, int r, int pos, float weight) {
    a.route_pos[r] = pos;
    a.weights[r] = weight;
    if (pos >= 0) {
        a.sorted_tokens[pos] = (uint32_t)r / (uint32_t)a.k;
    }
}

// Routes per expert of every workgroup's span, for k_moe_route
__global__ __launch_bounds__(256) void k_moe_count(const RouteArgs a) {
    __shared__ int counts[MOE_MAX_EXPERTS + 1];
    for (int e = threadIdx.x; e <= a.E; e += blockDim.x) {
        counts[e] = 0;
    }
    __syncthreads();
    const int routes = a.T * a.k;
    const int first = (int)blockIdx.x * a.span;
    const int last = routes - first < a.span ? routes : first + a.span;
    for (int base = first; base < last; base += 1024) {
        int id[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = base + 256 * i + (int)threadIdx.x;
            id[i] = a.topk_ids[r < last ? r : last - 1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (base + 256 * i + (int)threadIdx.x < last) {
                if (id[i] < 0 || id[i] >= a.E) {
                    counts[a.E] = 1;
                } else {
                    atomicAdd(&counts[id[i]], 1);
                }
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e <= a.E; e += blockDim.x) {
        a.table[(size_t)blockIdx.x * (a.E + 1) + e] = counts[e];
    }
}

// Bound by latencies: loads of the ids are batched and ranks come from ballots. The weights of the routes are copied as they
// are; the combine scales them, by token.
__global__ __launch_bounds__(MOE_ROUTE_WAVES * 64) void k_moe_route(const RouteArgs a) {
    warm_kernel_arguments<sizeof(RouteArgs), sizeof(RouteArgs)>();
    __shared__ int counts[MOE_MAX_EXPERTS];
    __shared__ int wcount[MOE_ROUTE_WAVES][MOE_MAX_EXPERTS];  // per chunk: routes of each expert, then its cursor
    __shared__ int before[MOE_MAX_EXPERTS];  // routes of each expert in the spans of earlier workgroups
    __shared__ int bad_id;
    __shared__ int ids_l[MOE_ROUTE_LDS];  // expert id of each route of this workgroup (-1 = invalid)
    const int routes = a.T * a.k;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    if (a.decode_order) {
        // At most 64 routes: one wavefront, one round. Experts are laid out in order of first appearance, so the
        // segment of an expert starts at the number of routes whose expert appeared earlier: an exclusive scan of
        // the expert's route count over the lanes that hold a first appearance.
        if (wave != 0) {
            return;
        }
        int id = -1;
        float weight = 0.0f;
        if (lane < routes) {
            id = a.topk_ids[lane];
            weight = a.topk_weights[lane];
            if (id < 0 || id >= a.E) {
                id = -1;
            }
        }
        const unsigned long long bad = __ballot(lane < routes && id < 0);
        int rank, cnt;
        wave_rank(id, lane, a.id_bits, &rank, &cnt);
        const bool first = id >= 0 && rank == 0;
        int total, n_items;
        const int seg = wave_excl_scan(first ? cnt : 0, lane, &total);
        const int item0 = wave_excl_scan(first ? (cnt + a.item_cols - 1) / a.item_cols : 0, lane, &n_items);
        if (first) {
            counts[id] = seg;
            int n = item0;
            for (int j = 0; j < cnt; j += a.item_cols) {
                a.items[n++] = make_int4(id, seg + j, (cnt - j) < a.item_cols ? (cnt - j) : a.item_cols, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the segment starts are in LDS (same wavefront)
        if (lane < routes) {
            route_emit(a, lane, id >= 0 ? counts[id] + rank : -1, weight);
        }
        if (lane == 0) {
            *a.n_items = n_items;
            *a.error_flag = bad != 0 ? 1 : 0;
        }
        return;
    }

    const int first = (int)blockIdx.x * a.span;
    const int last = routes - first < a.span ? routes : first + a.span;
    const bool in_lds = last - first <= MOE_ROUTE_LDS;
    for (int e = tid; e < a.E; e += blockDim.x) {
#pragma unroll
        for (int w = 0; w < MOE_ROUTE_WAVES; ++w) {
            wcount[w][e] = 0;
        }
    }
    if (tid == 0) {
        bad_id = 0;
    }
    __syncthreads();
    // chunk of wavefront w: routes [first + w * chunk, first + (w + 1) * chunk), a multiple of 64
    const int chunk = ((last - first + MOE_ROUTE_WAVES * 64 - 1) / (MOE_ROUTE_WAVES * 64)) * 64;
    const int r_begin = first + wave * chunk;
    const int r_end = r_begin + chunk < last ? r_begin + chunk : last;
    float next_weight = r_begin + lane < r_end ? a.topk_weights[r_begin + lane] : 0.0f;  // requested before the ids are waited for
    constexpr int BATCH = 8;  // loads in flight per lane: with one, a prompt's counting loop is a chain of memory latencies
    for (int base = r_begin; base < r_end; base += 64 * BATCH) {
        int id[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int r = base + 64 * i + lane;
            id[i] = a.topk_ids[r < r_end ? r : r_end - 1];
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int r = base + 64 * i + lane;
            if (r < r_end) {
                if (id[i] < 0 || id[i] >= a.E) {
                    bad_id = 1;
                    id[i] = -1;
                } else {
                    atomicAdd(&wcount[wave][id[i]], 1);
                }
                if (in_lds) {
                    ids_l[r - first] = id[i];
                }
            }
        }
    }
    __syncthreads();
    for (int e = tid; e < a.E; e += blockDim.x) {
        int c = 0, b = 0;
        if (a.table != nullptr) {
            const int groups = (int)gridDim.x;
            for (int g0 = 0; g0 < groups; g0 += 16) {
                int n[16];
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    n[g] = a.table[(size_t)(g0 + g < groups ? g0 + g : groups - 1) * (a.E + 1) + e];
                }
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    c += g0 + g < groups ? n[g] : 0;
                    b += g0 + g < (int)blockIdx.x ? n[g] : 0;
                }
            }
        } else {
#pragma unroll
            for (int w = 0; w < MOE_ROUTE_WAVES; ++w) {
                c += wcount[w][e];
            }
        }
        counts[e] = c;
        before[e] = b;
    }
    __syncthreads();
    // exclusive prefix over experts in ascending id and the work items of every expert: lane l of the first
    // wavefront owns the experts [l * per, (l + 1) * per)
    if (wave == 0) {
        const int per = (a.E + 63) / 64;
        const int e0 = lane * per;
        const int e1 = e0 + per < a.E ? e0 + per : a.E;
        int c_sum = 0, i_sum = 0;
        for (int e = e0; e < e1; ++e) {
            const int c = counts[e];
            c_sum += c;
            i_sum += (c + a.item_cols - 1) / a.item_cols;
        }
        int total, n_items;
        int prefix = wave_excl_scan(c_sum, lane, &total);
        int n = wave_excl_scan(i_sum, lane, &n_items);
        for (int e = e0; e < e1; ++e) {
            const int c = counts[e];
            counts[e] = prefix;  // from here on: start of the expert's segment
            for (int j = 0; blockIdx.x == 0 && j < c; j += a.item_cols) {
                a.items[n++] = make_int4(e, prefix + j, (c - j) < a.item_cols ? (c - j) : a.item_cols, 0);
            }
            prefix += c;
        }
        if (blockIdx.x == 0) {
            int bad = bad_id;
            if (a.table != nullptr) {  // (at most one workgroup per lane)
                bad = __ballot(lane < (int)gridDim.x && a.table[(size_t)lane * (a.E + 1) + a.E] != 0) != 0 ? 1 : 0;
            }
            if (lane == 0) {
                *a.n_items = n_items;
                *a.error_flag = bad;
            }
        }
    }
    __syncthreads();
    // cursor of chunk w for expert e: segment start + routes of e in earlier chunks
    for (int e = tid; e < a.E; e += blockDim.x) {
        int run = counts[e] + before[e];
#pragma unroll
        for (int w = 0; w < MOE_ROUTE_WAVES; ++w) {
            const int c = wcount[w][e];
            wcount[w][e] = run;
            run += c;
        }
    }
    __syncthreads();
    // Stable fill, every wavefront over its own chunk, 64 routes per round in route order: a route's position is its
    // expert's cursor plus the number of earlier lanes of the round with the same expert.
    int *cursor = wcount[wave];
    auto id_of = [&](int r) {
        if (in_lds) {
            return ids_l[r - first];
        }
        const int id = a.topk_ids[r];
        return id < 0 || id >= a.E ? -1 : id;
    };
    int next = r_begin + lane < r_end ? id_of(r_begin + lane) : -1;
    for (int base = r_begin; base < r_end; base += 64) {
        const int r = base + lane;
        const int id = next;
        const float weight = next_weight;
        next = r + 64 < r_end ? id_of(r + 64) : -1;
        next_weight = r + 64 < r_end ? a.topk_weights[r + 64] : 0.0f;
        int rank, cnt;
        wave_rank(id, lane, a.id_bits, &rank, &cnt);
        int pos = -1;
        if (id >= 0) {
            pos = cursor[id] + rank;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // this round's cursor reads are complete before the update below
        if (id >= 0 && rank == cnt - 1) {
            cursor[id] += cnt;
        }
        if (r < r_end) {
            route_emit(a, r, pos, weight);
        }
    }
}

// ------------------------------------------------------------------ weighted combine
// out[t, :] = sum over the token's routes, in ascending sorted position (moe_ops.c:1034-1042), of
// weight * down_row; tokens without a valid route get zeros (moe_ops.c:944-947, 984-986).
// One workgroup per token and 1024 columns (4 per thread, VEC: as one 16-byte access); the rows of COMBINE_BATCH routes are
// requested before the first is added (2048 tokens, top 8, 2048 columns: 45 -> 24 us, one column per
// thread and one row at a time before; reading the 134 MB of route rows takes 22).
constexpr int COMBINE_BATCH = 8;
template <bool VEC>
__global__ __launch_bounds__(256) void k_moe_combine(const float *__restrict__ route_down,
                                                     const float *__restrict__ weights, float weights_scale,
                                                     int renormalize, const int *__restrict__ route_pos, int k, size_t H,
                                                     float *__restrict__ out) {
    __shared__ int raw[MOE_MAX_TOPK], pos[MOE_MAX_TOPK];
    __shared__ float raw_w[MOE_MAX_TOPK], wts[MOE_MAX_TOPK];
    const size_t t = blockIdx.x;
    const int s = threadIdx.x;
    const int p = s < k ? route_pos[t * k + s] : -1;
    const float w = s < k ? weights[t * k + s] : 0.0f;
    if (s < k) {
        raw[s] = p;
        raw_w[s] = w;
    }
    __syncthreads();
    int n = 0, rank = 0;
    float wsum = 0.0f;  // of every slot, in slot order, those of an invalid id too
    for (int i = 0; i < k; ++i) {
        wsum += raw_w[i];
        n += raw[i] >= 0 ? 1 : 0;
        rank += raw[i] >= 0 && raw[i] < p ? 1 : 0;  // (the positions of a token's routes are distinct)
    }
    if (p >= 0) {
        pos[rank] = p;
        const float norm = !renormalize ? weights_scale : wsum > FLT_MIN ? weights_scale / wsum : 0.0f;
        wts[rank] = w * norm;
    }
    __syncthreads();
    const size_t h = (size_t)blockIdx.y * 1024 + 4 * (size_t)threadIdx.x;
    if (h >= H) {
        return;
    }
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int cols = H - h < 4 ? (int)(H - h) : 4;
    for (int j0 = 0; j0 < n; j0 += COMBINE_BATCH) {
        float row[COMBINE_BATCH][4];
#pragma unroll
        for (int j = 0; j < COMBINE_BATCH; ++j) {
            const float *src = route_down + (size_t)pos[j0 + j < n ? j0 + j : n - 1] * H + h;
            if constexpr (VEC) {
                const float4 v = *(const float4 *)src;
                row[j][0] = v.x, row[j][1] = v.y, row[j][2] = v.z, row[j][3] = v.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    row[j][e] = src[e < cols ? e : 0];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < COMBINE_BATCH; ++j) {
            if (j0 + j < n) {
                const float wj = wts[j0 + j];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[e] += wj * row[j][e];
                }
            }
        }
    }
    float *dst = out + t * H + h;
    if constexpr (VEC) {
        *(float4 *)dst = make_float4(acc[0], acc[1], acc[2], acc[3]);
    } else {
        for (int e = 0; e < cols; ++e) {
            dst[e] = acc[e];
        }
    }
}

static inline size_t round256(size_t v) {
    return (v + 255) & ~(size_t)255;
}

} // namespace mh

using namespace mh;

extern "C" {

int marmot_hip_topk(marmot_hip_device_t *dev, const float *d_x, size_t rows, size_t cols, size_t k, float *d_values,
                    int32_t *d_indices) {
    if (dev == nullptr) {
        return set_error(MARMOT_HIP_ERROR_DEVICE_NOT_AVAILABLE, "HIP device is not initialised");
    }
    if (d_x == nullptr || d_values == nullptr || d_indices == nullptr) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "TopK descriptor is incomplete");
    }
    if (k == 0 || k > cols) {
        return set_error(MARMOT_HIP_ERROR_DIMENSION_MISMATCH, "TopK shapes do not match");
    }
    if (rows == 0) {
        return MARMOT_HIP_SUCCESS;
    }
    hipLaunchKernelGGL(k_topk, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, dev->stream, d_x, rows, cols, k,
                       d_values, d_indices);
    MH_HIP(hipGetLastError());
    return MARMOT_HIP_SUCCESS;
}

int marmot_hip_softmax_rows(marmot_hip_device_t *dev, const float *d_x, size_t rows, size_t k, float *d_out) {
    if (dev == nullptr) {
        return set_error(MARMOT_HIP_ERROR_DEVICE_NOT_AVAILABLE, "HIP device is not initialised");
    }
    if (d_x == nullptr || d_out == nullptr || k == 0) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "softmax_rows: bad argument");
    }
    if (rows == 0) {
        return MARMOT_HIP_SUCCESS;
    }
    hipLaunchKernelGGL(k_softmax_rows, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, dev->stream, d_x, rows, k,
                       d_out);
    MH_HIP(hipGetLastError());
    return MARMOT_HIP_SUCCESS;
}

} // extern "C"

// The pinned word and the event of the expert-id check, made by the device object's first checked call
static int host_word_init(marmot_hip_device *dev) {
    if (dev->host_word_event != nullptr) {
        return MARMOT_HIP_SUCCESS;
    }
    if (dev->host_word == nullptr) {
        MH_HIP(hipHostMalloc((void **)&dev->host_word, 64, hipHostMallocDefault));
    }
    MH_HIP(hipEventCreateWithFlags(&dev->host_word_event, hipEventDisableTiming));
    return MARMOT_HIP_SUCCESS;
}

// One body for marmot_hip_moe_experts and its stage-probing variant. `probe` (may be null) names device buffers that
// receive the intermediate arrays, and optionally the packed activations the down projection reads instead of the
// ones this call quantized.
static int moe_experts_impl(marmot_hip_device_t *dev, const float *d_hidden, size_t T, size_t H, size_t F, size_t E,
                            size_t k_per_token, int kind_gate_up, int kind_down, const void *d_gate, const void *d_up,
                            const void *d_down, const int32_t *d_topk_ids, const float *d_topk_weights,
                            float weights_scale, int router_weight_policy, int ffn_type, float *d_out,
                            const marmot_hip_moe_probe_t *probe) {
    if (dev == nullptr) {
        return set_error(MARMOT_HIP_ERROR_DEVICE_NOT_AVAILABLE, "HIP device is not initialised");
    }
    if (d_hidden == nullptr || d_gate == nullptr || d_up == nullptr || d_down == nullptr || d_topk_ids == nullptr ||
        d_topk_weights == nullptr || d_out == nullptr) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "MoE experts requires non-null context and tensors");
    }
    if (router_weight_policy < 0 || router_weight_policy > MARMOT_HIP_ROUTER_RENORMALIZE_SELECTED) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "MoE experts requires a valid router weight policy");
    }
    if (ffn_type != MARMOT_HIP_FFN_SWIGLU && ffn_type != MARMOT_HIP_FFN_GEGLU) {
        return set_error(MARMOT_HIP_ERROR_NOT_IMPLEMENTED, "MoE experts currently supports SwiGLU and GeGLU only");
    }
    const size_t bv_gu = block_values(kind_gate_up), bv_dn = block_values(kind_down);
    if (bv_gu == 0 || bv_dn == 0 || kind_gate_up == MARMOT_HIP_KIND_Q8_K || kind_down == MARMOT_HIP_KIND_Q8_K) {
        return set_error(MARMOT_HIP_ERROR_NOT_IMPLEMENTED, "MoE experts: unsupported expert quant kinds %d / %d",
                         kind_gate_up, kind_down);
    }
    if (E == 0 || E > (size_t)MOE_MAX_EXPERTS || k_per_token == 0 || k_per_token > (size_t)MOE_MAX_TOPK || H == 0 ||
        F == 0) {
        return set_error(MARMOT_HIP_ERROR_DIMENSION_MISMATCH, "MoE expert tensor shapes do not match");
    }
    if (T == 0) {
        return MARMOT_HIP_SUCCESS;
    }
    MH_HIP(hipSetDevice(dev->device_index));

    const size_t routes = T * k_per_token;
    // Routes per work item. A work item streams its expert's rows once for its routes, so prompts, where an expert
    // sees dozens of routes, take wider items (the small-batch kernels on the int8 matrix cores hold 16 or 32 activation
    // rows per pass; the dot-product kernel of the 32-value formats holds 8): E = 128, top 8, 512 tokens: 325 us with 8.
    const bool mmq_gu = mmq_grouped_supported(dev, kind_gate_up, H), mmq_dn = mmq_grouped_supported(dev, kind_down, F);
    const auto q45 = [](int kind) { return kind == MARMOT_HIP_KIND_Q4_K || kind == MARMOT_HIP_KIND_Q5_K; };
    size_t item_cols = MOE_ITEM_COLS;
    if (mmq_gu && mmq_dn && routes >= 12 * E) {
        item_cols = (routes >= 24 * E && q45(kind_gate_up) && q45(kind_down)) ? 32 : 16;
    }
    // Prompts with many routes per expert: the tiled GEMM on int8 planes, 64 routes per item
    const size_t tiled_items = routes / 64 + E / 2, two_per_cu = 2 * (size_t)dev->props.multiProcessorCount;
    const bool tiled = routes >= MOE_TILED_ROUTES * E && tiled_items * 2 * ((F + 127) / 128) >= two_per_cu &&
                       tiled_items * ((H + 127) / 128) >= two_per_cu &&
                       gemm_planes_grouped_supported(dev, kind_gate_up, T, H, F, E + routes / 64, d_gate, d_up) &&
                       gemm_planes_grouped_supported(dev, kind_down, routes, F, H, E + routes / 64, d_down, d_down);
    if (tiled) {
        item_cols = 64;
    }
    const size_t max_items = routes < E + routes / item_cols ? routes : E + routes / item_cols;
    const int act_gu = is_k_quant(kind_gate_up) ? MARMOT_HIP_KIND_Q8_K : MARMOT_HIP_KIND_Q8_0;
    const int act_dn = is_k_quant(kind_down) ? MARMOT_HIP_KIND_Q8_K : MARMOT_HIP_KIND_Q8_0;

    // workspace carve-up
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off += round256(bytes);
        return o;
    };
    const size_t o_hidden_q = take(act_scratch_layout(act_gu, T, H, nullptr, nullptr));
    const size_t o_fused_q = take(act_scratch_layout(act_dn, routes, F, nullptr, nullptr));
    const size_t o_tokens = take(routes * sizeof(uint32_t));
    const size_t o_weights = take(routes * sizeof(float));
    const size_t o_pos = take(routes * sizeof(int));
    const size_t o_items = take((max_items + 1) * sizeof(int4));
    const size_t o_flags = take(2 * sizeof(int));
    const size_t split_span = (routes + (size_t)MOE_SPLIT_GROUPS * MOE_SPLIT_SPAN - 1) /
                              ((size_t)MOE_SPLIT_GROUPS * MOE_SPLIT_SPAN) * MOE_SPLIT_SPAN;
    const size_t route_groups = routes > (size_t)MOE_SPLIT_ROUTES ? (routes + split_span - 1) / split_span : 1;
    const size_t table_bytes = route_groups > 1 ? route_groups * (E + 1) * sizeof(int) : 0;
    const size_t gate_bytes = routes * F * sizeof(float);
    const size_t o_gate = take(gate_bytes > table_bytes ? gate_bytes : table_bytes);  // the counts lie where gate comes later
    // (laid out also where the GEMM forms the gated product and leaves it alone: a workspace that held a prompt holds every shorter one,
    // also in a capture, which may not let it grow)
    const size_t o_up = take(routes * F * sizeof(float));
    const size_t o_down = take(routes * H * sizeof(float));
    void *ws = nullptr;
    int st = workspace_reserve(dev, off, &ws);
    if (st != MARMOT_HIP_SUCCESS) {
        return st;
    }
    uint8_t *base = (uint8_t *)ws;
    ActScratch hidden_q, fused_q;
    act_scratch_layout(act_gu, T, H, base + o_hidden_q, &hidden_q);
    act_scratch_layout(act_dn, routes, F, base + o_fused_q, &fused_q);
    uint32_t *sorted_tokens = (uint32_t *)(base + o_tokens);
    float *weights = (float *)(base + o_weights);
    int *route_pos = (int *)(base + o_pos);
    int4 *items = (int4 *)(base + o_items);
    int *flags = (int *)(base + o_flags);  // [0] = number of items, [1] = error flag; both set by the route kernel
    float *gate_out = (float *)(base + o_gate);
    float *up_out = (float *)(base + o_up);
    float *route_down = (float *)(base + o_down);

    RouteArgs ra;
    ra.topk_ids = d_topk_ids;
    ra.topk_weights = d_topk_weights;
    ra.weights = weights;
    ra.sorted_tokens = sorted_tokens;
    ra.route_pos = route_pos;
    ra.items = items;
    ra.n_items = flags;
    // Expert ids are validated on the device. The route kernel leaves the answer in pinned host memory and the call waits
    // for that kernel only, not for the experts; skipped while the stream is being captured into a graph or when the
    // device object was created with MARMOT_HIP_MOE_NO_VALIDATE set.
    const bool validate = !dev->capturing && !dev->knobs.moe_no_validate;
    if (validate) {
        MH_TRY(host_word_init(dev));
    }
    ra.error_flag = validate ? dev->host_word : flags + 1;
    ra.T = (int)T;
    ra.k = (int)k_per_token;
    ra.E = (int)E;
    // cpu_moe_should_use_decode_path (moe_ops.c:417-424)
    ra.decode_order = (T <= 4 && routes <= 64) ? 1 : 0;
    ra.item_cols = (int)item_cols;
    ra.id_bits = 1;
    while (((size_t)1 << ra.id_bits) < E) {
        ++ra.id_bits;
    }
    ra.span = (int)(route_groups > 1 ? split_span : routes);
    ra.table = route_groups > 1 ? (int *)(base + o_gate) : nullptr;
    if (route_groups > 1) {
        hipLaunchKernelGGL(k_moe_count, dim3((unsigned)route_groups), dim3(256), 0, dev->stream, ra);
        MH_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_moe_route, dim3((unsigned)route_groups), dim3(MOE_ROUTE_WAVES * 64), 0, dev->stream, ra);
    MH_HIP(hipGetLastError());
    if (validate) {
        MH_HIP(hipEventRecord(dev->host_word_event, dev->stream));
    }

    // hidden states are quantized once per token; routes refer to them through sorted_tokens
    st = launch_quantize_act_soa(dev, act_gu, d_hidden, MARMOT_HIP_DTYPE_F32, T, H, hidden_q);
    if (st != MARMOT_HIP_SUCCESS) {
        return st;
    }
    const size_t gu_stride = F * ((H + bv_gu - 1) / bv_gu) * block_bytes(kind_gate_up);
    const size_t dn_stride = H * ((F + bv_dn - 1) / bv_dn) * block_bytes(kind_down);
    // K-quant experts run on the matrix cores (long prompts on the tiled GEMM on int8 planes, else passes), the 32-value formats on
    // the dot-product matvec
    // Tiled, SwiGLU: the GEMM forms the gated product itself, which is written and read once in the place of two arrays (a call
    // that looks at the stages gets both)
    const bool gated = tiled && ffn_type != MARMOT_HIP_FFN_GEGLU && probe == nullptr;
    st = tiled  ? launch_gemm_planes_grouped(dev, kind_gate_up, d_gate, d_up, gu_stride, hidden_q, sorted_tokens, items, flags,
                                          max_items, H, F, gate_out, up_out, gated)
        : mmq_gu ? launch_mmq_grouped(dev, kind_gate_up, d_gate, d_up, gu_stride, hidden_q, sorted_tokens, items, flags,
                                     max_items, H, F, gate_out, up_out, (int)item_cols)
                : launch_matvec_grouped(dev, kind_gate_up, d_gate, d_up, gu_stride, hidden_q, sorted_tokens, items, flags,
                                        max_items, H, F, gate_out, up_out);
    if (st != MARMOT_HIP_SUCCESS) {
        return st;
    }
    st = gated ? launch_quantize_act_soa(dev, act_dn, gate_out, MARMOT_HIP_DTYPE_F32, routes, F, fused_q)
               : launch_quantize_glu_soa(dev, act_dn, gate_out, up_out, ffn_type == MARMOT_HIP_FFN_GEGLU, routes, F, fused_q);
    if (st != MARMOT_HIP_SUCCESS) {
        return st;
    }
    if (probe != nullptr) {
        const size_t fused_bytes = act_scratch_layout(act_dn, routes, F, nullptr, nullptr);
        const struct {
            void *dst;
            const void *src;
            size_t bytes;
        } copies[] = {
            {probe->d_sorted_tokens, sorted_tokens, routes * sizeof(uint32_t)},
            {probe->d_route_pos, route_pos, routes * sizeof(int)},
            {probe->d_gate_out, gate_out, routes * F * sizeof(float)},
            {probe->d_up_out, up_out, routes * F * sizeof(float)},
            {probe->d_fused_packed, base + o_fused_q, fused_bytes},
        };
        for (const auto &c : copies) {
            if (c.dst != nullptr) {
                MH_HIP(hipMemcpyAsync(c.dst, c.src, c.bytes, hipMemcpyDeviceToDevice, dev->stream));
            }
        }
        if (probe->d_fused_override != nullptr) {
            MH_HIP(hipMemcpyAsync(base + o_fused_q, probe->d_fused_override, fused_bytes, hipMemcpyDeviceToDevice,
                                  dev->stream));
        }
    }
    st = tiled  ? launch_gemm_planes_grouped(dev, kind_down, d_down, nullptr, dn_stride, fused_q, nullptr, items, flags,
                                          max_items, F, H, route_down, nullptr, false)
        : mmq_dn ? launch_mmq_grouped(dev, kind_down, d_down, nullptr, dn_stride, fused_q, nullptr, items, flags, max_items,
                                     F, H, route_down, nullptr, (int)item_cols)
                : launch_matvec_grouped(dev, kind_down, d_down, nullptr, dn_stride, fused_q, nullptr, items, flags,
                                        max_items, F, H, route_down, nullptr);
    if (st != MARMOT_HIP_SUCCESS) {
        return st;
    }
    const int renormalize = router_weight_policy == MARMOT_HIP_ROUTER_RENORMALIZE_SELECTED;
    const dim3 combine_grid((unsigned)T, (unsigned)((H + 1023) / 1024));
    if (H % 4 == 0 && (((uintptr_t)d_out) & 15) == 0) {
        hipLaunchKernelGGL(k_moe_combine<true>, combine_grid, dim3(256), 0, dev->stream, route_down, weights, weights_scale,
                           renormalize, route_pos, (int)k_per_token, H, d_out);
    } else {
        hipLaunchKernelGGL(k_moe_combine<false>, combine_grid, dim3(256), 0, dev->stream, route_down, weights, weights_scale,
                           renormalize, route_pos, (int)k_per_token, H, d_out);
    }
    MH_HIP(hipGetLastError());
    set_route(tiled ? "moe_experts_tiled" : "moe_experts_grouped");

    if (validate) {
        MH_HIP(hipEventSynchronize(dev->host_word_event));
        if (*(volatile int *)dev->host_word != 0) {
            // the caller takes the call for refused: its buffers are its own again
            MH_HIP(hipStreamSynchronize(dev->stream));
            return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "MoE expert id is out of range");
        }
    }
    return MARMOT_HIP_SUCCESS;
}

extern "C" {

int marmot_hip_moe_experts(marmot_hip_device_t *dev, const float *d_hidden, size_t T, size_t H, size_t F, size_t E,
                           size_t k_per_token, int kind_gate_up, int kind_down, const void *d_gate, const void *d_up,
                           const void *d_down, const int32_t *d_topk_ids, const float *d_topk_weights,
                           float weights_scale, int router_weight_policy, int ffn_type, float *d_out) {
    return moe_experts_impl(dev, d_hidden, T, H, F, E, k_per_token, kind_gate_up, kind_down, d_gate, d_up, d_down,
                            d_topk_ids, d_topk_weights, weights_scale, router_weight_policy, ffn_type, d_out, nullptr);
}

int marmot_hip_moe_experts_probe(marmot_hip_device_t *dev, const float *d_hidden, size_t T, size_t H, size_t F,
                                 size_t E, size_t k_per_token, int kind_gate_up, int kind_down, const void *d_gate,
                                 const void *d_up, const void *d_down, const int32_t *d_topk_ids,
                                 const float *d_topk_weights, float weights_scale, int router_weight_policy,
                                 int ffn_type, float *d_out, const marmot_hip_moe_probe_t *probe) {
    if (probe == nullptr) {
        return set_error(MARMOT_HIP_ERROR_INVALID_ARGUMENT, "MoE experts probe requires a probe description");
    }
    if (dev != nullptr && dev->capturing) {
        return set_error(MARMOT_HIP_ERROR_INVALID_OPERATION, "MoE experts probe cannot be captured into a graph");
    }
    return moe_experts_impl(dev, d_hidden, T, H, F, E, k_per_token, kind_gate_up, kind_down, d_gate, d_up, d_down,
                            d_topk_ids, d_topk_weights, weights_scale, router_weight_policy, ffn_type, d_out, probe);
}

} // extern "C"
