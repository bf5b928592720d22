// Plain FP32 form of the fully fused MLP (tiny-cuda-nn src/fully_fused_mlp.cu,
// no biases): forward, backward through the layers, and weight gradients.
//
// A workgroup of 256 lanes owns a tile of T queries and keeps the tile's
// activations in LDS ([unit][query], FP32).  Each layer is an LDS-resident
// GEMM out[W][T] = A[W][K] . in[K][T]: the current weight matrix is staged
// k-major in LDS, and every lane accumulates a (W/16 units x T/16 queries)
// register block with FP32 FMAs (one float4 of weights and T/64 float4s of
// activations per 4*(T/16)... FMAs).  Weight gradients are batch reductions
// dW = delta . act^T on FP32 MFMAs, split over query chunks, with a
// deterministic second-pass reduction.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "model.h"
#include "nlod_common.h"
#include "wgrad.h"

namespace nlod {
namespace {

constexpr int kThreads = 256;
constexpr uint32_t kChunkK = 64;  // layer-0 / d_enc rows handled per pass

struct MlpArgs {
    uint32_t n_input, n_hidden_layers, n_output, n_output_padded;
    int32_t act, out_act;
};

// Q: queries per lane.  8 (4 at width 128) reuse a staged weight more; batches
// that give fewer such tiles than there are CUs take 4 (module forward and backward
// of 20011 queries, 64 x 5: 0.55 -> 0.48 ms; inference of 1000 queries 56 -> 39 us,
// but of 50000, two small tiles a CU, 98 -> 112 us).
template <int W, int Q>
struct Tiling {
    static constexpr int UB = W / 16;  // units per lane
    static constexpr int QB = Q;       // queries per lane
    static constexpr int T = 16 * QB;  // queries per tile
};
template <int W>
constexpr int kLargeQ = W >= 128 ? 4 : 8;

// acc[UB][QB] += sum_k AT[k][u0 + i] * X[k][q0 + j]; AT is [kk][W] (k-major), X is [kk][T]
template <int W, int Q>
__device__ __forceinline__ void lds_gemm(const float* __restrict__ AT, const float* __restrict__ X, uint32_t kk,
                                         int u0, int q0, float (&acc)[Tiling<W, Q>::UB][Tiling<W, Q>::QB]) {
    constexpr int UB = Tiling<W, Q>::UB, QB = Tiling<W, Q>::QB, T = Tiling<W, Q>::T;
#pragma unroll 2
    for (uint32_t k = 0; k < kk; ++k) {
        float a[UB], x[QB];
#pragma unroll
        for (int i = 0; i < UB; i += (UB >= 4 ? 4 : UB)) {
            if constexpr (UB >= 4) {
                const float4 v = *reinterpret_cast<const float4*>(AT + k * W + u0 + i);
                a[i] = v.x; a[i + 1] = v.y; a[i + 2] = v.z; a[i + 3] = v.w;
            } else {
#pragma unroll
                for (int t = 0; t < UB; ++t) a[t] = AT[k * W + u0 + t];
            }
        }
#pragma unroll
        for (int j = 0; j < QB; j += 4) {
            const float4 v = *reinterpret_cast<const float4*>(X + k * T + q0 + j);
            x[j] = v.x; x[j + 1] = v.y; x[j + 2] = v.z; x[j + 3] = v.w;
        }
#pragma unroll
        for (int i = 0; i < UB; ++i)
#pragma unroll
            for (int j = 0; j < QB; ++j) acc[i][j] += a[i] * x[j];
    }
}

// Stage rows [r0, r0+rows) x cols of a row-major matrix (stride ld) into LDS,
// transposed to [col][W-strided row]: dst[c * W + (r - r0)].
__device__ __forceinline__ void stage_transposed(float* dst, const float* __restrict__ src, uint32_t rows,
                                                 uint32_t cols, uint32_t ld, uint32_t col0, uint32_t Wd) {
    for (uint32_t idx = threadIdx.x; idx < rows * cols; idx += kThreads) {
        const uint32_t r = idx / cols, c = idx - r * cols;
        dst[c * Wd + r] = src[(size_t)r * ld + col0 + c];
    }
}

// Stage rows [k0, k0+kk) of a row-major [*, ld] matrix as-is: dst[k * ld + m].
__device__ __forceinline__ void stage_rows(float* dst, const float* __restrict__ src, uint32_t kk, uint32_t ld,
                                           uint32_t m0, uint32_t mm, uint32_t Wd) {
    for (uint32_t idx = threadIdx.x; idx < kk * mm; idx += kThreads) {
        const uint32_t k = idx / mm, m = idx - k * mm;
        dst[k * Wd + m] = src[(size_t)k * ld + m0 + m];
    }
}

// Load rows [k0, k0+kk) of a SoA [*][N] global matrix for the tile into X[kk][T] (0 beyond N).
template <int T>
__device__ __forceinline__ void load_tile_rows(float* X, const float* __restrict__ src, uint32_t k0, uint32_t kk,
                                               uint32_t N, uint32_t tq0) {
    for (uint32_t idx = threadIdx.x; idx < kk * T; idx += kThreads) {
        const uint32_t k = idx / T, q = idx - k * T;
        X[idx] = (tq0 + q < N) ? src[(size_t)(k0 + k) * N + tq0 + q] : 0.0f;
    }
}

template <int W, int Q>
__global__ __launch_bounds__(kThreads) void mlp_fwd_kernel(uint32_t N, MlpArgs a, const float* __restrict__ w,
                                                           const float* __restrict__ enc, float* __restrict__ out,
                                                           float* __restrict__ hidden) {
    using Tl = Tiling<W, Q>;
    constexpr int UB = Tl::UB, QB = Tl::QB, T = Tl::T;
    constexpr int R = W > (int)kChunkK ? W : (int)kChunkK;  // rows of the staging buffers
    extern __shared__ float4 smem4[];
    float* bufA = reinterpret_cast<float*>(smem4);  // [R][T]
    float* bufB = bufA + R * T;                      // [W][T]
    float* wt = bufB + W * T;                        // [R][W]
    const int tu = threadIdx.x >> 4, tq = threadIdx.x & 15;
    const int u0 = tu * UB, q0 = tq * QB;
    const uint32_t K = a.n_input;
    const uint32_t n_tiles = (N + T - 1) / T;
    for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const uint32_t tq0 = tile * T;
        float acc[UB][QB];
#pragma unroll
        for (int i = 0; i < UB; ++i)
#pragma unroll
            for (int j = 0; j < QB; ++j) acc[i][j] = 0.0f;
        for (uint32_t k0 = 0; k0 < K; k0 += kChunkK) {
            const uint32_t kc = min(kChunkK, K - k0);
            __syncthreads();
            load_tile_rows<T>(bufA, enc, k0, kc, N, tq0);
            stage_transposed(wt, w, W, kc, K, k0, W);
            __syncthreads();
            lds_gemm<W, Q>(wt, bufA, kc, u0, q0, acc);
        }
        float* cur = bufB;
        float* nxt = bufA;
        for (uint32_t layer = 0;; ++layer) {
            // activation -> LDS tile (and the saved activations for backward)
#pragma unroll
            for (int i = 0; i < UB; ++i) act_fwd_n<QB>(a.act, acc[i]);
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) {
                    const float h = acc[i][j];
                    cur[(u0 + i) * T + q0 + j] = h;
                    if (hidden && tq0 + q0 + j < N) hidden[((size_t)layer * W + u0 + i) * N + tq0 + q0 + j] = h;
                }
            if (layer + 1 >= a.n_hidden_layers) break;
            __syncthreads();
            stage_transposed(wt, w + (size_t)W * K + (size_t)layer * W * W, W, W, W, 0, W);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) acc[i][j] = 0.0f;
            lds_gemm<W, Q>(wt, cur, W, u0, q0, acc);
            float* t = cur;
            cur = nxt;
            nxt = t;
        }
        __syncthreads();
        // output layer: lane t < T computes query t's outputs (weights broadcast from global/L1)
        const float* w_out = w + (size_t)W * K + (size_t)(a.n_hidden_layers - 1) * W * W;
        for (uint32_t t = threadIdx.x; t < (uint32_t)T; t += kThreads) {
            if (tq0 + t >= N) continue;
            for (uint32_t r = 0; r < a.n_output; ++r) {
                float s = 0.0f;
#pragma unroll 8
                for (int k = 0; k < W; ++k) s += w_out[r * W + k] * cur[k * T + t];
                out[(size_t)(tq0 + t) * a.n_output + r] = act_fwd(a.out_act, s);
            }
        }
    }
}

// Backward through the layers for a tile: delta_l (SoA [L][W][N], dL/d pre-activation),
// delta_out (SoA [n_out_padded][N]) and dL/d(enc) (SoA [K][N], optional).
template <int W, int Q>
__global__ __launch_bounds__(kThreads) void mlp_bwd_delta_kernel(uint32_t N, MlpArgs a, const float* __restrict__ w,
                                                                 const float* __restrict__ hidden,
                                                                 const float* __restrict__ out,
                                                                 const float* __restrict__ d_out,
                                                                 float* __restrict__ delta,
                                                                 float* __restrict__ delta_out,
                                                                 float* __restrict__ d_enc) {
    using Tl = Tiling<W, Q>;
    constexpr int UB = Tl::UB, QB = Tl::QB, T = Tl::T;
    constexpr int R = W > (int)kChunkK ? W : (int)kChunkK;
    extern __shared__ float4 smem4[];
    float* bufA = reinterpret_cast<float*>(smem4);  // [R][T]
    float* bufB = bufA + R * T;                      // [W][T]
    float* wt = bufB + W * T;                        // [R][W]
    const int tu = threadIdx.x >> 4, tq = threadIdx.x & 15;
    const int u0 = tu * UB, q0 = tq * QB;
    const uint32_t K = a.n_input, L = a.n_hidden_layers;
    const uint32_t n_tiles = (N + T - 1) / T;
    for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const uint32_t tq0 = tile * T;
        __syncthreads();
        // output activation transfer (fully_fused_mlp.cu:757-760): dz[r][t] in bufA rows 0..15
        for (uint32_t idx = threadIdx.x; idx < 16u * T; idx += kThreads) {
            const uint32_t r = idx / T, t = idx - r * T, q = tq0 + t;
            float v = 0.0f;
            if (q < N && r < a.n_output)
                v = d_out[(size_t)q * a.n_output + r] * act_bwd(a.out_act, out[(size_t)q * a.n_output + r]);
            bufA[idx] = v;
            if (q < N && r < a.n_output_padded) delta_out[(size_t)r * N + q] = v;
        }
        // W_out [16][W] row-major is already k-major for the transposed product
        stage_rows(wt, w + (size_t)W * K + (size_t)(L - 1) * W * W, a.n_output, W, 0, W, W);
        __syncthreads();
        float acc[UB][QB];
#pragma unroll
        for (int i = 0; i < UB; ++i)
#pragma unroll
            for (int j = 0; j < QB; ++j) acc[i][j] = 0.0f;
        lds_gemm<W, Q>(wt, bufA, a.n_output, u0, q0, acc);
        for (int layer = (int)L - 1; layer >= 0; --layer) {
            // through the hidden activation: delta = acc * act'(h_layer)
#pragma unroll
            for (int i = 0; i < UB; ++i) {
                float hv[QB], dv[QB];
#pragma unroll
                for (int j = 0; j < QB; ++j) {
                    const uint32_t q = tq0 + q0 + j;
                    hv[j] = q < N ? hidden[((size_t)layer * W + u0 + i) * N + q] : 0.0f;
                }
                act_bwd_n<QB>(a.act, hv, dv);
#pragma unroll
                for (int j = 0; j < QB; ++j) {
                    const uint32_t q = tq0 + q0 + j;
                    acc[i][j] *= dv[j];
                    if (q < N) delta[((size_t)layer * W + u0 + i) * N + q] = acc[i][j];
                }
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) bufB[(u0 + i) * T + q0 + j] = acc[i][j];
            if (layer == 0) break;
            stage_rows(wt, w + (size_t)W * K + (size_t)(layer - 1) * W * W, W, W, 0, W, W);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) acc[i][j] = 0.0f;
            lds_gemm<W, Q>(wt, bufB, W, u0, q0, acc);
        }
        if (!d_enc) continue;
        // dL/d(enc)[m][t] = sum_u W0[u][m] delta_0[u][t], in chunks of W rows of m
        for (uint32_t m0 = 0; m0 < K; m0 += W) {
            const uint32_t mm = min((uint32_t)W, K - m0);
            __syncthreads();
            stage_rows(wt, w, W, K, m0, mm, W);
            for (uint32_t idx = threadIdx.x; idx < (uint32_t)W * (W - mm); idx += kThreads) {
                const uint32_t k = idx / (W - mm), m = mm + idx % (W - mm);
                wt[k * W + m] = 0.0f;
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) acc[i][j] = 0.0f;
            lds_gemm<W, Q>(wt, bufB, W, u0, q0, acc);
#pragma unroll
            for (int i = 0; i < UB; ++i)
#pragma unroll
                for (int j = 0; j < QB; ++j) {
                    const uint32_t m = m0 + u0 + i, q = tq0 + q0 + j;
                    if (m < K && q < N) d_enc[(size_t)m * N + q] = acc[i][j];
                }
        }
    }
}

// ---- weight gradients: C[m][k] = sum_q A[m][q] * B[k][q], grid (chunks of
// queries, 64 x 64 tiles of all matrices), see wgrad.h.  On
// v_mfma_f32_16x16x4_f32 (FP32 products and sums) with the queries as the
// reduction dimension: lane group g holds 4 consecutive queries of a 16-query
// step in one 16-byte load, and the step's four MFMAs take one of them each.
// One launch for all matrices: at 20011 queries the 20 blocks of 1024 queries
// per matrix left most of the chip idle (236 us for each 64 x 64 matrix of the
// 5-layer throughput network; its forward and backward 1.97 -> 0.59 ms).
constexpr uint32_t kWgradQueries = 16;  // queries per step

template <int RT, int CT>
__device__ __forceinline__ void wgrad_tile(uint32_t N, const WgradItem& it, uint32_t step0, uint32_t step1,
                                           const float* __restrict__ A, const float* __restrict__ B,
                                           float* __restrict__ p, uint32_t ld, float4* lds) {
    const int lane = threadIdx.x & 63, g = lane >> 4, m16 = lane & 15, wave = threadIdx.x >> 6;
    typedef float floatx4 __attribute__((ext_vector_type(4)));
    floatx4 acc[RT * CT];
#pragma unroll
    for (int t = 0; t < RT * CT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    const float* ap = A + (size_t)(it.row0 + m16) * N + 4 * g;
    const float* bp = B + (size_t)(it.col0 + m16) * N + 4 * g;
    auto load = [&](uint32_t step, floatx4 (&x)[RT], floatx4 (&y)[CT]) {
        const uint32_t q0 = step * kWgradQueries;
        if (q0 + kWgradQueries <= N) {
            // rows start at any multiple of 4 bytes
#pragma unroll
            for (int r = 0; r < RT; ++r) __builtin_memcpy(&x[r], ap + (size_t)(16 * r) * N + q0, 16);
#pragma unroll
            for (int c = 0; c < CT; ++c) __builtin_memcpy(&y[c], bp + (size_t)(16 * c) * N + q0, 16);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = q0 + 4 * g + j < N;
#pragma unroll
                for (int r = 0; r < RT; ++r) x[r][j] = in ? ap[(size_t)(16 * r) * N + q0 + j] : 0.0f;
#pragma unroll
                for (int c = 0; c < CT; ++c) y[c][j] = in ? bp[(size_t)(16 * c) * N + q0 + j] : 0.0f;
            }
        }
    };
    floatx4 nx[RT], ny[CT];
    uint32_t step = step0 + (uint32_t)wave;
    if (step < step1) load(step, nx, ny);
    for (; step < step1; step += 4) {
        floatx4 x[RT], y[CT];
#pragma unroll
        for (int r = 0; r < RT; ++r) x[r] = nx[r];
#pragma unroll
        for (int c = 0; c < CT; ++c) y[c] = ny[c];
        if (step + 4 < step1) load(step + 4, nx, ny);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    acc[r * CT + c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r][j], y[c][j], acc[r * CT + c], 0, 0, 0);
    }
    wgrad_add_waves<RT * CT>(acc, lds);
    if (wave != 0) return;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                p[(size_t)(it.row0 + 16 * r + 4 * g + i) * ld + it.col0 + 16 * c + m16] = acc[r * CT + c][i];
}

__global__ __launch_bounds__(256, 3) void wgrad_partial_kernel(uint32_t N, WgradShape a,
                                                               const float* __restrict__ enc,
                                                               const float* __restrict__ hidden,
                                                               const float* __restrict__ delta,
                                                               const float* __restrict__ delta_out,
                                                               float* __restrict__ partial, uint32_t n_params,
                                                               uint32_t chunk_steps) {
    __shared__ float4 lds[2 * 16 * 64];
    const WgradItem it = wgrad_item(blockIdx.y, a);
    const uint32_t n_steps = (N + kWgradQueries - 1) / kWgradQueries;
    const uint32_t step0 = min(n_steps, blockIdx.x * chunk_steps), step1 = min(n_steps, step0 + chunk_steps);
    const size_t layer = (size_t)a.W * N;
    const float* A = it.layer == a.L ? delta_out : delta + it.layer * layer;
    const float* B = it.layer == 0 ? enc : hidden + (it.layer - 1) * layer;
    const uint32_t rows = it.layer == a.L ? a.out_rows : a.W, cols = it.layer == 0 ? a.cols0 : a.W;
    float* p = partial + (size_t)blockIdx.x * n_params +
               (it.layer == 0 ? 0 : (size_t)a.W * a.cols0 + (size_t)(it.layer - 1) * a.W * a.W);
    auto run = [&](auto RTc, auto CTc) {
        wgrad_tile<decltype(RTc)::value, decltype(CTc)::value>(N, it, step0, step1, A, B, p, cols, lds);
    };
    auto run_rows = [&](auto RTc) {  // every dimension is a multiple of 16
        const uint32_t ct = (cols - it.col0) / 16;
        if (ct >= 4) run(RTc, std::integral_constant<int, 4>{});
        else if (ct == 3) run(RTc, std::integral_constant<int, 3>{});
        else if (ct == 2) run(RTc, std::integral_constant<int, 2>{});
        else run(RTc, std::integral_constant<int, 1>{});
    };
    const uint32_t rt = (rows - it.row0) / 16;
    if (rt >= 4) run_rows(std::integral_constant<int, 4>{});
    else if (rt >= 2) run_rows(std::integral_constant<int, 2>{});
    else run_rows(std::integral_constant<int, 1>{});
}

template <typename K>
void by_width(uint32_t W, K&& k) {
    switch (W) {
        case 16: k(std::integral_constant<int, 16>{}); break;
        case 32: k(std::integral_constant<int, 32>{}); break;
        case 64: k(std::integral_constant<int, 64>{}); break;
        case 128: k(std::integral_constant<int, 128>{}); break;
        default: fail(NLOD_ERR_CONFIG, "unsupported network width");
    }
}

MlpArgs make_args(const NetShape& n) {
    return MlpArgs{n.n_input, n.n_hidden_layers, n.n_output, n.n_output_padded, n.activation, n.output_activation};
}

template <int W, int Q>
size_t smem_bytes() {
    constexpr int T = Tiling<W, Q>::T;
    constexpr int R = W > (int)kChunkK ? W : (int)kChunkK;
    return sizeof(float) * ((size_t)R * T + (size_t)W * T + (size_t)R * W);
}

template <int W, int Q, typename Kern>
uint32_t grid_for(Kern kern, uint32_t N) {
    const int occ = occupancy_blocks((const void*)kern, kThreads, smem_bytes<W, Q>());
    const uint32_t tiles = div_round_up(N, Tiling<W, Q>::T);
    return std::min<uint32_t>(tiles, (uint32_t)(cu_count() * occ));
}

// Calls k with the width and the queries per lane that suit N.
template <typename K>
void by_tiling(uint32_t W, uint32_t N, K&& k) {
    by_width(W, [&](auto Wc) {
        constexpr int Q = kLargeQ<decltype(Wc)::value>;
        if (Q > 4 && div_round_up(N, 16 * Q) < (uint32_t)cu_count()) k(Wc, std::integral_constant<int, 4>{});
        else k(Wc, std::integral_constant<int, Q>{});
    });
}

uint32_t wgrad_steps(uint32_t N) { return div_round_up(std::max<uint32_t>(N, 1), kWgradQueries); }
WgradShape wgrad_shape(const NetShape& n) { return {n.width, n.n_input, n.n_hidden_layers, n.n_output_padded}; }
uint32_t wgrad_chunks_of(const NetShape& net, uint32_t N) {
    return wgrad_chunks(wgrad_items(wgrad_shape(net)), wgrad_steps(N));
}

}  // namespace

void mlp_forward_f32(hipStream_t stream, const NetShape& net, const float* weights, const float* enc, uint32_t N,
                     float* out, float* hidden) {
    if (N == 0) return;
    const MlpArgs a = make_args(net);
    by_tiling(net.width, N, [&](auto Wc, auto Qc) {
        constexpr int W = decltype(Wc)::value, Q = decltype(Qc)::value;
        auto kern = mlp_fwd_kernel<W, Q>;
        const uint32_t blocks = grid_for<W, Q>(kern, N);
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), (smem_bytes<W, Q>()), stream, N, a, weights, enc, out,
                           hidden);
    });
    NLOD_LAUNCH_CHECK();
}

void mlp_backward_delta_f32(hipStream_t stream, const NetShape& net, const float* weights, const float* hidden,
                            const float* out, const float* d_out, uint32_t N, float* delta, float* delta_out,
                            float* d_enc) {
    if (N == 0) return;
    const MlpArgs a = make_args(net);
    by_tiling(net.width, N, [&](auto Wc, auto Qc) {
        constexpr int W = decltype(Wc)::value, Q = decltype(Qc)::value;
        auto kern = mlp_bwd_delta_kernel<W, Q>;
        const uint32_t blocks = grid_for<W, Q>(kern, N);
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), (smem_bytes<W, Q>()), stream, N, a, weights, hidden, out,
                           d_out, delta, delta_out, d_enc);
    });
    NLOD_LAUNCH_CHECK();
}

size_t mlp_weight_grad_workspace_floats(const NetShape& net, uint32_t N) {
    return (size_t)wgrad_chunks_of(net, N) * net.n_params();
}

void mlp_weight_grad_f32(hipStream_t stream, const NetShape& net, const float* enc, const float* hidden,
                         const float* delta, const float* delta_out, uint32_t N, float* grads, float* workspace,
                         size_t workspace_floats, bool accumulate) {
    if (workspace_floats < mlp_weight_grad_workspace_floats(net, N)) fail(NLOD_ERR_STATE, "weight-gradient workspace too small");
    if (N == 0) {
        if (!accumulate) fill_f32(stream, grads, net.n_params(), 0.0f);
        return;
    }
    const uint32_t n_params = (uint32_t)net.n_params();
    const uint32_t chunks = wgrad_chunks_of(net, N);
    const WgradShape a = wgrad_shape(net);
    hipLaunchKernelGGL(wgrad_partial_kernel, dim3(chunks, wgrad_items(a)), dim3(256), 0, stream, N, a, enc, hidden,
                       delta, delta_out, workspace, n_params, div_round_up(wgrad_steps(N), chunks));
    NLOD_LAUNCH_CHECK();
    partial_reduce(stream, n_params, chunks, workspace, grads, accumulate);
}

}  // namespace nlod
