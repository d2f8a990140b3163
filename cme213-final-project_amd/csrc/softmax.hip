// Row softmax and softmax cross-entropy for gfx950.
//
// Reference behaviour: FINAL_CLEAN_CODE/src/kernels/activations.cu:394-532.
//  * softmax_forward (:394-435): out = e / sum with e = expf(x - max), one
//    block per row walking the row three times in global memory.
//  * cross_entropy_kernel (:438-477): p = e * (1 / (sum + 1e-9)),
//    loss = -logf(p[t] + 1e-9), grad = (p - onehot(t)) * scale; one 32-lane
//    warp per row.
//  * cross_entropy_forward (:479-499): scale 1; the per-row losses are
//    copied to the host and summed there in order; returns the mean.
//  * cross_entropy_forward_v2 (:517-532): scale 1 / batch; the mean loss
//    stays on the device (memset + atomicAdd tree + a divide kernel).
//
// Here a "row group" of G waves holds a row in registers (K accesses of
// 4 or 16 bytes per lane), so the row is read from HBM once and the output written once.  The
// row maximum and sum are wave reductions (DPP) combined across the G waves
// in a fixed order through LDS.  Rows longer than 65536 use a block-per-row
// kernel that streams the row three times, as the reference does.  The
// device mean loss is one single-workgroup reduction in a fixed order: no
// memset (graph-capture safe) and bitwise reproducible.
#include <cfloat>
#include <vector>

#include "mi_common.hpp"

namespace mi {

namespace {

constexpr float kCeEps = 1e-9f;  // activations.cu:461,470
constexpr float kLog2e = 1.4426950408889634f;

// Raw buffer resource over one row of `cols` floats (word 3 as for every
// gfx9 raw buffer: 32-bit data, no swizzle).  Loads past the end return 0 and
// stores past the end are dropped, which bounds the row in hardware.
constexpr int kBufWord3 = 0x00020000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const float* p, int cols) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, cols * 4, kBufWord3);
}

// G waves per row, K elements per lane.  Workgroups hold 4 waves (4 / G
// rows) for G < 4, otherwise one row of G waves.
template <int G>
constexpr int sm_threads() {
    return (G < 4 ? 4 : G) * kWave;
}

// V = 4 takes 16-byte accesses, V = 1 4-byte ones; K accesses per lane.
//
// Memory-bound.  16-byte stores carry the non-temporal hint: [16384, 1024]
// softmax 34.7 -> 26.3 us, [16384, 1100] 51.7 -> 27.1, [4096, 32000] 194 -> 180,
// cross-entropy [8192, 32000] 373 -> 360 (180 -> 173 and 360 -> 344 with it on
// the loads too, see stream_rows).  4-byte accesses do better without: their
// rows start anywhere, and lines shared by two waves are then written twice.
// Sharing one long row between workgroups that each read all of it and store a
// part was slower ([64, 32000] 7.1 -> 8.8 us, 16 rows of 50257 9.4 -> 21).
constexpr int kNontemporal = 2;  // cache-policy bit of the buffer accesses

template <int G, int K, bool CE, int V, bool NT>
__global__ __launch_bounds__(sm_threads<G>()) void row_softmax_kernel(
    const float* __restrict__ x, float* __restrict__ out, int rows, int cols,
    const int* __restrict__ targets, float* __restrict__ losses, float scale) {
    constexpr int GPB = G < 4 ? 4 / G : 1;  // row groups per workgroup
    constexpr int GT = G * kWave;            // lanes per row
    __shared__ float red_max[GPB][G];
    __shared__ float red_sum[GPB][G];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int grp = wave / G;
    const int wig = wave % G;
    const int t = wig * kWave + lane;
    const int row = blockIdx.x * GPB + grp;
    // Groups past the last row process a copy of the last row and store
    // nothing, so every wave reaches the barriers.
    const bool valid = row < rows;
    const int rr = valid ? row : rows - 1;
    const float* xr = x + static_cast<size_t>(rr) * cols;

    // Raw buffer loads bounded by the row length: slots past the end read 0
    // in hardware, so no index is clamped and every load shares one lane
    // offset plus a per-slot scalar offset.  Masked slots then take
    // -FLT_MAX, the reference's initial maximum, and give exp(.) = 0 below.
    const __amdgpu_buffer_rsrc_t rin = row_rsrc(xr, cols);
    float v[K][V];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if constexpr (V == 4) {
            const auto a = __builtin_amdgcn_raw_buffer_load_b128(rin, t * 16, k * GT * 16,
                                                                 NT ? kNontemporal : 0);
            const bool ok = 4 * (t + k * GT) < cols;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[k][e] = ok ? __int_as_float(a[e]) : -FLT_MAX;
        } else {
            const float a =
                __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rin, t * 4, k * GT * 4, 0));
            v[k][0] = (t + k * GT) < cols ? a : -FLT_MAX;
        }
    }
    float m = -FLT_MAX;
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int e = 0; e < V; ++e) m = fmaxf(m, v[k][e]);
    m = wave_max(m);
    if constexpr (G > 1) {
        if (lane == 0) red_max[grp][wig] = m;
        __syncthreads();
        m = red_max[grp][0];
#pragma unroll
        for (int w = 1; w < G; ++w) m = fmaxf(m, red_max[grp][w]);
    }

    // e = exp(x - m) as 2^(x log2 e - m log2 e) on v_exp_f32, the exponent
    // formed by one FMA.  The rounding of m log2 e scales every e of the row
    // by the same factor, which cancels in the normalisation; masked slots
    // (-FLT_MAX) give 2^-inf = 0.
    const float mL = m * kLog2e;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const float ex = __builtin_amdgcn_exp2f(fmaf(v[k][e], kLog2e, -mL));
            v[k][e] = ex;
            s += ex;
        }
    s = wave_sum(s);
    if constexpr (G > 1) {
        if (lane == 0) red_sum[grp][wig] = s;
        __syncthreads();
        s = red_sum[grp][0];
#pragma unroll
        for (int w = 1; w < G; ++w) s += red_sum[grp][w];
    }
    if (!valid) return;  // after the last barrier

    // Buffer stores past the row end are dropped in hardware.
    const __amdgpu_buffer_rsrc_t rout = row_rsrc(out + static_cast<size_t>(row) * cols, cols);
    auto store = [&](int k, const float (&y)[V]) __attribute__((always_inline)) {
        if constexpr (V == 4) {
            typedef int i32x4 __attribute__((ext_vector_type(4)));
            const i32x4 q = {__float_as_int(y[0]), __float_as_int(y[1]), __float_as_int(y[2]),
                             __float_as_int(y[3])};
            // The slot's offset is in the lane offset, not a scalar one: a
            // 16-byte buffer store must not be followed at once by a write of
            // its data registers, and the compiler leaves that wait out for
            // stores with a scalar offset register, which gave wrong first
            // elements here.
            __builtin_amdgcn_raw_buffer_store_b128(q, rout, (t + k * GT) * 16, 0, kNontemporal);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(y[0]), rout, t * 4, k * GT * 4, 0);
        }
    };
    if constexpr (!CE) {
        const float inv = 1.0f / s;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            float y[V];
#pragma unroll
            for (int e = 0; e < V; ++e) y[e] = v[k][e] * inv;
            store(k, y);
        }
    } else {
        const float inv = 1.0f / (s + kCeEps);
        const int tgt = targets[row];
        float pt = 0.0f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            float y[V];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float p = v[k][e] * inv;
                const bool hit = V * (t + k * GT) + e == tgt;
                pt = hit ? p : pt;
                y[e] = (hit ? p - 1.0f : p) * scale;
            }
            store(k, y);
        }
        // One lane owns the target and writes the loss; an invalid target
        // gives NaN (written by lane 0 of the group).
        if (tgt >= 0 && tgt < cols) {
            if (tgt / V % GT == t) losses[row] = -logf(pt + kCeEps);
        } else if (t == 0) {
            losses[row] = __int_as_float(0x7fc00000);
        }
    }
}

// Block-per-row fallback for rows longer than the register-resident shapes:
// max, sum of exponentials and the output are three passes over the row.
constexpr int kLongThreads = 1024;

template <int NW>
__device__ __forceinline__ float block_reduce(float v, float* red, bool is_max) {
    v = is_max ? wave_max(v) : wave_sum(v);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) r = is_max ? fmaxf(r, red[i]) : r + red[i];
    __syncthreads();
    return r;
}

template <bool CE>
__global__ __launch_bounds__(kLongThreads) void long_row_softmax_kernel(
    const float* __restrict__ x, float* __restrict__ out, int cols,
    const int* __restrict__ targets, float* __restrict__ losses, float scale) {
    constexpr int NW = kLongThreads / kWave;
    __shared__ float red[NW];
    const int row = blockIdx.x;
    const float* xr = x + static_cast<size_t>(row) * cols;
    float* orow = out + static_cast<size_t>(row) * cols;
    float m = -FLT_MAX;
    for (int j = threadIdx.x; j < cols; j += kLongThreads) m = fmaxf(m, xr[j]);
    m = block_reduce<NW>(m, red, true);
    float s = 0.0f;
    for (int j = threadIdx.x; j < cols; j += kLongThreads) s += expf(xr[j] - m);
    s = block_reduce<NW>(s, red, false);
    if constexpr (!CE) {
        for (int j = threadIdx.x; j < cols; j += kLongThreads) orow[j] = expf(xr[j] - m) / s;
    } else {
        const float inv = 1.0f / (s + kCeEps);
        const int tgt = targets[row];
        if ((tgt < 0 || tgt >= cols) && threadIdx.x == 0) losses[row] = __int_as_float(0x7fc00000);
        for (int j = threadIdx.x; j < cols; j += kLongThreads) {
            float p = expf(xr[j] - m) * inv;
            if (j == tgt) {
                losses[row] = -logf(p + kCeEps);
                p -= 1.0f;
            }
            orow[j] = p * scale;
        }
    }
}

// Mean of n per-row losses into *out, in a fixed order: thread i sums
// elements i, i + 1024, ... sequentially, the waves reduce with DPP and the
// 16 wave totals are added in wave order.
__global__ __launch_bounds__(kLongThreads) void loss_mean_kernel(const float* __restrict__ losses,
                                                                 int n, float* __restrict__ out) {
    constexpr int NW = kLongThreads / kWave;
    __shared__ float red[NW];
    float s = 0.0f;
    for (int i = threadIdx.x; i < n; i += kLongThreads) s += losses[i];
    s = wave_sum(s);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = red[0];
#pragma unroll
        for (int i = 1; i < NW; ++i) total += red[i];
        *out = total / static_cast<float>(n);
    }
}

struct SmPlan {
    int G = 0, K = 0;  // G == 0: long-row kernel
};

// The fewest waves, then the fewest accesses per lane that hold the row.  An
// access is 16 bytes (vec4) or 4.
SmPlan plan_softmax(int cols, bool vec4) {
    static const int kK1[] = {1, 2, 3, 4, 6, 8, 10, 12, 14, 16};
    static const int kK16[] = {10, 12, 14, 16, 24, 32, 40, 48, 56, 64};
    static const int kV1[] = {1, 2, 3, 4};
    static const int kV16[] = {3, 4, 5, 6, 7, 8, 10, 12, 14, 16};
    const int n = vec4 ? cols / 4 : cols;  // accesses
    for (int g = 1; g <= 16; g *= 2) {
        if (vec4 && g < 16) {
            for (int k : kV1)
                if (n <= g * kWave * k) return {g, k};
        } else {
            for (int k : (g < 16 ? kK1 : vec4 ? kV16 : kK16))
                if (n <= g * kWave * k) return {g, k};
        }
    }
    return {};
}

// Whether the loads of rows over 8 waves or more (past 4096 columns) carry the
// hint too: where the logits are half as large again as the 256 MB last-level
// cache, so that they come from memory, and rows past 49152 columns.  Time of
// the hinted form over the plain one's, logits from memory / in the cache: [4096,
// 8192] 0.94 / 1.09, [4096, 16384] 0.96 / 1.15, [2048, 32000] 0.97 / 1.14, [1000, 32000]
// 0.95 / 1.11, but [4096, 32000] 0.96 and [8192, 32000] 0.95 always, [256, 50304]
// 0.95 / 0.91, [300, 64000] 0.97 / 1.00, [512, 65536] 0.92 / 1.04.  The longest rows
// gain over 4-byte accesses except where one or two fall to each CU and the
// logits are in the cache (65536 columns: 64 rows 0.72 / 0.63, 256 rows 0.98 / 1.14,
// 512 rows 0.94 / 1.20, 768 rows 0.91 / 0.89).
bool stream_rows(int rows, int cols) {
    return cols > 49152 || static_cast<long long>(rows) * cols > (3ll << 25);
}

template <int G, int K, bool CE, int V>
void launch_rows(int rows, int cols, hipStream_t st, const float* x, float* out, const int* tg,
                 float* losses, float scale) {
    constexpr int GPB = G < 4 ? 4 / G : 1;
    const dim3 grid(static_cast<unsigned>((static_cast<long long>(rows) + GPB - 1) / GPB));
    if constexpr (V == 4 && G >= 8) {
        if (stream_rows(rows, cols)) {
            hipLaunchKernelGGL((row_softmax_kernel<G, K, CE, V, true>), grid,
                               dim3(sm_threads<G>()), 0, st, x, out, rows, cols, tg, losses, scale);
            return;
        }
    }
    hipLaunchKernelGGL((row_softmax_kernel<G, K, CE, V, false>), grid, dim3(sm_threads<G>()), 0,
                       st, x, out, rows, cols, tg, losses, scale);
}

template <bool CE>
void launch_softmax(int rows, int cols, hipStream_t st, const float* x, float* out, const int* tg,
                    float* losses, float scale) {
    // Up to 64 columns a 4-byte access already holds the row, and a 16-byte one
    // leaves most lanes idle: its time over the other's, 65536 rows of 16, 32, 64,
    // 68, 96 columns, 1.16, 1.11, 1.05, 0.85, 0.80.
    const bool vec4 = cols > 64 && cols % 4 == 0 && aligned16(x) && aligned16(out);
    const SmPlan p = plan_softmax(cols, vec4);
#define MI_SM_CASE(GG, KK, VV)                                                  \
    if (p.G == GG && p.K == KK && vec4 == (VV == 4)) {                           \
        launch_rows<GG, KK, CE, VV>(rows, cols, st, x, out, tg, losses, scale);  \
        return;                                                                  \
    }
    MI_SM_CASE(1, 1, 4)
    MI_SM_CASE(1, 2, 4)
    MI_SM_CASE(1, 3, 4)
    MI_SM_CASE(1, 4, 4)
    MI_SM_CASE(2, 3, 4)
    MI_SM_CASE(2, 4, 4)
    MI_SM_CASE(4, 3, 4)
    MI_SM_CASE(4, 4, 4)
    MI_SM_CASE(8, 3, 4)
    MI_SM_CASE(8, 4, 4)
    MI_SM_CASE(16, 3, 4)
    MI_SM_CASE(16, 4, 4)
    MI_SM_CASE(16, 5, 4)
    MI_SM_CASE(16, 6, 4)
    MI_SM_CASE(16, 7, 4)
    MI_SM_CASE(16, 8, 4)
    MI_SM_CASE(16, 10, 4)
    MI_SM_CASE(16, 12, 4)
    MI_SM_CASE(16, 14, 4)
    MI_SM_CASE(16, 16, 4)
    MI_SM_CASE(1, 1, 1)
    MI_SM_CASE(1, 2, 1)
    MI_SM_CASE(1, 3, 1)
    MI_SM_CASE(1, 4, 1)
    MI_SM_CASE(1, 6, 1)
    MI_SM_CASE(1, 8, 1)
    MI_SM_CASE(1, 10, 1)
    MI_SM_CASE(1, 12, 1)
    MI_SM_CASE(1, 14, 1)
    MI_SM_CASE(1, 16, 1)
    MI_SM_CASE(2, 10, 1)
    MI_SM_CASE(2, 12, 1)
    MI_SM_CASE(2, 14, 1)
    MI_SM_CASE(2, 16, 1)
    MI_SM_CASE(4, 10, 1)
    MI_SM_CASE(4, 12, 1)
    MI_SM_CASE(4, 14, 1)
    MI_SM_CASE(4, 16, 1)
    MI_SM_CASE(8, 10, 1)
    MI_SM_CASE(8, 12, 1)
    MI_SM_CASE(8, 14, 1)
    MI_SM_CASE(8, 16, 1)
    MI_SM_CASE(16, 10, 1)
    MI_SM_CASE(16, 12, 1)
    MI_SM_CASE(16, 14, 1)
    MI_SM_CASE(16, 16, 1)
    MI_SM_CASE(16, 24, 1)
    MI_SM_CASE(16, 32, 1)
    MI_SM_CASE(16, 40, 1)
    MI_SM_CASE(16, 48, 1)
    MI_SM_CASE(16, 56, 1)
    MI_SM_CASE(16, 64, 1)
#undef MI_SM_CASE
    hipLaunchKernelGGL((long_row_softmax_kernel<CE>), dim3(rows), dim3(kLongThreads), 0, st, x,
                       out, cols, tg, losses, scale);
}

int check_ce_args(const char* name, const float* logits, const int* targets, const float* grad,
                  int batch, int vocab) {
    if (batch < 0 || vocab <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: invalid shape batch=%d vocab=%d", name, batch,
                         vocab);
    if (batch > 0 && (!logits || !targets || !grad))
        return set_error(MI_ERR_INVALID_ARG, "%s: NULL pointer", name);
    return MI_OK;
}

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" {

int mi_softmax_forward(const float* x, float* out, int rows, int cols, void* stream) {
    const char* name = "mi_softmax_forward";
    if (rows < 0 || cols <= 0)
        return set_error(MI_ERR_INVALID_ARG, "%s: invalid shape rows=%d cols=%d", name, rows,
                         cols);
    if (rows == 0) return MI_OK;
    if (!x || !out) return set_error(MI_ERR_INVALID_ARG, "%s: NULL pointer", name);
    launch_softmax<false>(rows, cols, to_stream(stream), x, out, nullptr, nullptr, 1.0f);
    return check_launch(name);
}

int mi_cross_entropy_forward(const float* logits, const int* targets, float* grad, int batch,
                             int vocab, float* loss, void* stream) {
    const char* name = "mi_cross_entropy_forward";
    int rc = check_ce_args(name, logits, targets, grad, batch, vocab);
    if (rc != MI_OK) return rc;
    if (!loss) return set_error(MI_ERR_INVALID_ARG, "%s: NULL loss pointer", name);
    if (batch == 0) {
        *loss = 0.0f / static_cast<float>(batch);  // the reference's total / batch
        return MI_OK;
    }
    hipStream_t st = to_stream(stream);
    int err = MI_OK;
    char* ws = static_cast<char*>(
        workspace_get(colsum_part_offset() + static_cast<size_t>(batch) * sizeof(float), st, &err));
    if (!ws) return err;
    float* losses = reinterpret_cast<float*>(ws + colsum_part_offset());
    launch_softmax<true>(batch, vocab, st, logits, grad, targets, losses, 1.0f);
    rc = check_launch(name);
    if (rc != MI_OK) return rc;
    // As the reference: the per-row losses come back to the host and are
    // summed there in row order.
    std::vector<float> h(static_cast<size_t>(batch));
    hipError_t e = hipMemcpyAsync(h.data(), losses, h.size() * sizeof(float),
                                  hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return set_error(static_cast<int>(e), "%s: copying the losses failed: %s", name,
                         hipGetErrorString(e));
    float total = 0.0f;
    for (float l : h) total += l;
    *loss = total / static_cast<float>(batch);
    return MI_OK;
}

int mi_cross_entropy_forward_v2(const float* logits, const int* targets, float* grad,
                                float* losses, float* loss_out, int batch, int vocab,
                                void* stream) {
    const char* name = "mi_cross_entropy_forward_v2";
    int rc = check_ce_args(name, logits, targets, grad, batch, vocab);
    if (rc != MI_OK) return rc;
    if (!loss_out || (batch > 0 && !losses))
        return set_error(MI_ERR_INVALID_ARG, "%s: NULL pointer", name);
    hipStream_t st = to_stream(stream);
    if (batch > 0) {
        launch_softmax<true>(batch, vocab, st, logits, grad, targets, losses,
                             1.0f / static_cast<float>(batch));
        rc = check_launch(name);
        if (rc != MI_OK) return rc;
    }
    hipLaunchKernelGGL(loss_mean_kernel, dim3(1), dim3(kLongThreads), 0, st, losses, batch,
                       loss_out);
    return check_launch(name);
}

size_t mi_cross_entropy_workspace(int batch) {
    return batch > 0 ? colsum_part_offset() + static_cast<size_t>(batch) * sizeof(float) : 0;
}

}  // extern "C"
