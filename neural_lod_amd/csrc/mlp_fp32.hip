// Plain FP32 form of the fully fused MLP (tiny-cuda-nn src/fully_fused_mlp.cu,
// no biases): forward, backward through the layers, and weight gradients.
//
// Every product runs on v_mfma_f32_16x16x4_f32 (FP32 operands, products and
// sums).  A wave owns 16 queries and keeps their activations in registers
// from the first layer to the last: the accumulator layout (lane group
// g = lane / 16 holds units 16t + 4g .. 16t + 4g + 3 of query lane % 16) is, one
// register at a time, the B operand of four products over the units
// {16t + 4g' + r, g' = 0..3}.  The matching A operands are four consecutive
// floats of a weight row, one 16-byte LDS read in the forward pass; the backward
// pass reads the same staged rows transposed, a dword at a time.  Only the
// current weight matrix is in LDS, staged by the block as it lies in memory; the
// next one is loaded into registers while the current one is used.  Weight
// gradients are batch reductions dW = delta . act^T, split over query chunks,
// with a deterministic second-pass reduction.
//
// Bound: the FP32 matrix rate for large batches; below two tiles a CU the serial
// chain of one wave (layers x products of 32 cycles, the weight loads between
// them).  Blocks of FP32 FMAs per lane, with the weights transposed on their way
// into LDS (all 64 lanes of a store on one bank), took, encoding included: 64 x 4
// network, 1000 queries 49 us, now 15; 20011, 76 and 38; 2^20, 1382 and 931;
// 128 x 4 network 89 and 33, 206 and 65, 5252 and 1727.  Two query tiles per wave
// (each weight staged for twice the queries) gave 899 us for the 931, three waves
// per SIMD by spilling 968.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "model.h"
#include "nlod_common.h"
#include "wgrad.h"

namespace nlod {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kChunkK = 64;  // columns of the first matrix staged at a time
constexpr uint32_t kTile = 16 * (kThreads / 64);  // queries per block: 16 per wave

struct MlpArgs {
    uint32_t n_input, n_hidden_layers, n_output, n_output_padded;
    int32_t act, out_act;
};

// Floats between the staged rows: 4 mod 16, so that neither the 16-byte reads of
// 16 rows nor the dword reads of 4 x 16 (rows 4 apart, columns consecutive) meet
// in an LDS bank.
template <int W>
constexpr int kLd = (W > kChunkK ? W : kChunkK) + 4;

// R rows x up to C columns (multiples of 4) of a row-major matrix, on their way
// into LDS: load() into registers, store() behind the barrier that frees the
// buffer.  Rows start at any multiple of 4 bytes.
template <int R, int C>
struct Staged {
    static constexpr int kLanes = C / 4, kRows = kThreads / kLanes, kSteps = (R + kRows - 1) / kRows;
    floatx4 v[kSteps];
    __device__ __forceinline__ void load(const float* __restrict__ src, uint32_t rows, uint32_t cols, uint32_t ld) {
        const uint32_t c = threadIdx.x % kLanes * 4;
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const uint32_t r = threadIdx.x / kLanes + i * kRows;
            v[i] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (r < rows && c < cols) __builtin_memcpy(&v[i], src + (size_t)r * ld + c, 16);
        }
    }
    __device__ __forceinline__ void store(float* dst, uint32_t ld) const {
        const uint32_t c = threadIdx.x % kLanes * 4;
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const uint32_t r = threadIdx.x / kLanes + i * kRows;
            if (R % kRows == 0 || r < (uint32_t)R) *reinterpret_cast<floatx4*>(dst + r * ld + c) = v[i];
        }
    }
};

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The W = 16 MT sums of a layer for 16 queries.  Input tiles alternate between two
// accumulators: half the chain of dependent products, and half the rounding
// errors in a row (against 64 bits, 64 x 5 and 128 x 4 networks: the outputs' relative
// error 2.0e-7 and 2.8e-7, 2.8e-7 and 3.8e-7 with one accumulator).
template <int MT>
struct Sums {
    floatx4 v[2][MT];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int m = 0; m < MT; ++m) v[0][m] = v[1][m] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ floatx4 sum(int m) const { return v[0][m] + v[1][m]; }

    // sums[m] += A[16m + .][16k .. 16k + 15] . x: 16 input units, held as an accumulator tile
    __device__ __forceinline__ void add_rows(const float* __restrict__ A, uint32_t ld, int k, floatx4 x) {
        const uint32_t lane = threadIdx.x & 63, g = lane >> 4, m16 = lane & 15;
        floatx4 a[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
            a[m] = *reinterpret_cast<const floatx4*>(A + (16 * m + m16) * ld + 16 * k + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int m = 0; m < MT; ++m) v[k & 1][m] = mfma4(a[m][r], x[r], v[k & 1][m]);
    }
    // sums[m] += A[16k .. 16k + 15][16m + .]^T . x
    __device__ __forceinline__ void add_cols(const float* __restrict__ A, uint32_t ld, int k, floatx4 x) {
        const uint32_t lane = threadIdx.x & 63, g = lane >> 4, m16 = lane & 15;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float a[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) a[m] = A[(16 * k + 4 * g + r) * ld + 16 * m + m16];
#pragma unroll
            for (int m = 0; m < MT; ++m) v[k & 1][m] = mfma4(a[m], x[r], v[k & 1][m]);
        }
    }
};

template <int W>
__global__ __launch_bounds__(kThreads, W >= 128 ? 1 : 2) void mlp_fwd_kernel(uint32_t N, MlpArgs a, const float* __restrict__ w,
                                               const float* __restrict__ enc, float* __restrict__ out,
                                               float* __restrict__ hidden) {
    constexpr int MT = W / 16, LD = kLd<W>;
    extern __shared__ float4 smem4[];
    float* w_lds = reinterpret_cast<float*>(smem4);  // [W][LD]: the current matrix
    float* out_lds = w_lds + W * LD;                 // [16][LD]: the output matrix
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, n16 = lane & 15;
    const uint32_t K = a.n_input, L = a.n_hidden_layers;
    const float* w_hidden = w + (size_t)W * K;  // L - 1 matrices [W][W]
    {
        Staged<16, W> so;
        so.load(w_hidden + (size_t)(L - 1) * W * W, a.n_output, W, W);
        so.store(out_lds, LD);
    }
    const uint32_t n_tiles = (N + kTile - 1) / kTile;
    for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const uint32_t q = tile * kTile + wave * 16 + n16;
        const bool valid = q < N;
        Sums<MT> acc;
        acc.clear();
        Staged<W, kChunkK> s0;
        s0.load(w, W, min((uint32_t)kChunkK, K), K);
        for (uint32_t k0 = 0; k0 < K; k0 += kChunkK) {
            const uint32_t kc = min((uint32_t)kChunkK, K - k0);  // a multiple of 16
            floatx4 x[kChunkK / 16];
#pragma unroll
            for (int c = 0; c < kChunkK / 16; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t k = 16 * c + 4 * g + r;
                    x[c][r] = k < kc && valid ? enc[(size_t)(k0 + k) * N + q] : 0.0f;
                }
            __syncthreads();
            s0.store(w_lds, LD);
            __syncthreads();
            if (k0 + kChunkK < K) s0.load(w + k0 + kChunkK, W, min((uint32_t)kChunkK, K - k0 - kChunkK), K);
#pragma unroll
            for (int c = 0; c < kChunkK / 16; ++c)
                if (16u * c < kc) acc.add_rows(w_lds, LD, c, x[c]);
        }
        Staged<W, W> s;
        if (L > 1) s.load(w_hidden, W, W, W);
        floatx4 h[MT];
        for (uint32_t layer = 0;; ++layer) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const floatx4 z = acc.sum(m);
                float y[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = z[r];
                act_fwd_n<4>(a.act, y);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h[m][r] = y[r];
                    if (hidden && valid) hidden[((size_t)layer * W + 16 * m + 4 * g + r) * N + q] = y[r];
                }
            }
            if (layer + 1 >= L) break;
            __syncthreads();
            s.store(w_lds, LD);
            __syncthreads();
            if (layer + 2 < L) s.load(w_hidden + (size_t)(layer + 1) * W * W, W, W, W);
            acc.clear();
#pragma unroll
            for (int k = 0; k < MT; ++k) acc.add_rows(w_lds, LD, k, h[k]);
        }
        Sums<1> o;
        o.clear();
#pragma unroll
        for (int k = 0; k < MT; ++k) o.add_rows(out_lds, LD, k, h[k]);
        const floatx4 z = o.sum(0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * g + r < a.n_output && valid) out[(size_t)q * a.n_output + 4 * g + r] = act_fwd(a.out_act, z[r]);
    }
}

// Backward through the layers for a tile: delta_l (SoA [L][W][N], dL/d pre-activation),
// delta_out (SoA [n_out_padded][N]) and dL/d(enc) (SoA [K][N], optional).
template <int W>
__global__ __launch_bounds__(kThreads, W >= 128 ? 1 : 2) void mlp_bwd_delta_kernel(uint32_t N, MlpArgs a, const float* __restrict__ w,
                                                     const float* __restrict__ hidden, const float* __restrict__ out,
                                                     const float* __restrict__ d_out, float* __restrict__ delta,
                                                     float* __restrict__ delta_out, float* __restrict__ d_enc) {
    constexpr int MT = W / 16, LD = kLd<W>;
    extern __shared__ float4 smem4[];
    float* w_lds = reinterpret_cast<float*>(smem4);  // [W][LD]: the current matrix
    float* out_lds = w_lds + W * LD;                 // [16][LD]: the output matrix
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, n16 = lane & 15;
    const uint32_t K = a.n_input, L = a.n_hidden_layers;
    const float* w_hidden = w + (size_t)W * K;
    {
        Staged<16, W> so;
        so.load(w_hidden + (size_t)(L - 1) * W * W, a.n_output, W, W);
        so.store(out_lds, LD);
    }
    __syncthreads();
    const uint32_t n_tiles = (N + kTile - 1) / kTile;
    for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const uint32_t q = tile * kTile + wave * 16 + n16;
        const bool valid = q < N;
        floatx4 hv[MT];  // the layer's activations
        auto load_hidden = [&](uint32_t layer) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    hv[m][r] = valid ? hidden[((size_t)layer * W + 16 * m + 4 * g + r) * N + q] : 0.0f;
        };
        // output activation transfer (fully_fused_mlp.cu:757-760)
        floatx4 dz;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t row = 4 * g + r;
            dz[r] = 0.0f;
            if (valid && row < a.n_output)
                dz[r] = d_out[(size_t)q * a.n_output + row] * act_bwd(a.out_act, out[(size_t)q * a.n_output + row]);
            if (valid && row < a.n_output_padded) delta_out[(size_t)row * N + q] = dz[r];
        }
        load_hidden(L - 1);
        Staged<W, W> s;
        if (L > 1) s.load(w_hidden + (size_t)(L - 2) * W * W, W, W, W);
        Sums<MT> acc;
        acc.clear();
        acc.add_cols(out_lds, LD, 0, dz);
        floatx4 d[MT];
        for (uint32_t layer = L; layer-- > 0;) {
            // through the hidden activation: delta = acc * act'(h_layer)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const floatx4 z = acc.sum(m);
                float y[4], dv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = hv[m][r];
                act_bwd_n<4>(a.act, y, dv);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    d[m][r] = z[r] * dv[r];
                    if (valid) delta[((size_t)layer * W + 16 * m + 4 * g + r) * N + q] = d[m][r];
                }
            }
            if (layer == 0) break;
            __syncthreads();
            s.store(w_lds, LD);
            __syncthreads();
            load_hidden(layer - 1);
            if (layer > 1) s.load(w_hidden + (size_t)(layer - 2) * W * W, W, W, W);
            acc.clear();
#pragma unroll
            for (int k = 0; k < MT; ++k) acc.add_cols(w_lds, LD, k, d[k]);
        }
        if (!d_enc) continue;
        // dL/d(enc)[m][q] = sum_u W0[u][m] delta_0[u][q]
        for (uint32_t m0 = 0; m0 < K; m0 += kChunkK) {
            const uint32_t mc = min((uint32_t)kChunkK, K - m0);
            Staged<W, kChunkK> s0;
            s0.load(w + m0, W, mc, K);
            __syncthreads();
            s0.store(w_lds, LD);
            __syncthreads();
            for (uint32_t m = 0; m < mc; m += 16) {
                Sums<1> e;
                e.clear();
#pragma unroll
                for (int k = 0; k < MT; ++k) e.add_cols(w_lds + m, LD, k, d[k]);
                const floatx4 z = e.sum(0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (valid) d_enc[(size_t)(m0 + m + 4 * g + r) * N + q] = z[r];
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

template <int W>
constexpr size_t kSmemBytes = sizeof(float) * (W + 16) * kLd<W>;

template <int W, typename Kern>
uint32_t grid_for(Kern kern, uint32_t N) {
    const int occ = occupancy_blocks((const void*)kern, kThreads, kSmemBytes<W>);
    return std::min<uint32_t>(div_round_up(N, kTile), (uint32_t)(cu_count() * occ));
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
    by_width(net.width, [&](auto Wc) {
        constexpr int W = decltype(Wc)::value;
        auto kern = mlp_fwd_kernel<W>;
        const uint32_t blocks = grid_for<W>(kern, N);
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), kSmemBytes<W>, stream, N, a, weights, enc, out,
                           hidden);
    });
    NLOD_LAUNCH_CHECK();
}

void mlp_backward_delta_f32(hipStream_t stream, const NetShape& net, const float* weights, const float* hidden,
                            const float* out, const float* d_out, uint32_t N, float* delta, float* delta_out,
                            float* d_enc) {
    if (N == 0) return;
    const MlpArgs a = make_args(net);
    by_width(net.width, [&](auto Wc) {
        constexpr int W = decltype(Wc)::value;
        auto kern = mlp_bwd_delta_kernel<W>;
        const uint32_t blocks = grid_for<W>(kern, N);
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), kSmemBytes<W>, stream, N, a, weights, hidden, out,
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
