// FP16-MFMA training kernels of the fully fused MLP (gfx950): forward with
// saved activations, backward through the layers, and weight gradients.
// Semantics follow tiny-cuda-nn src/fully_fused_mlp.cu:706-833 (no biases).
//
// Saved tensors (per 16-query tile, "unit-major": [tile][unit][16 queries], FP16):
//   H_l   post-activation of hidden layer l (l = 0 .. L-1)
//   D_l   dL/d(pre-activation) of layer l (l = 0 .. L-1), D_L = output layer
// The encoded features X stay in the fragment layout of the encoding pass.
//
// Backward per 16-query tile (one wave): delta_out = dL/dy * act'(y) in the
// accumulator layout, then G_{l-1} = W_l^T delta_l on MFMA with the transposed
// weights pre-packed (columns permuted to the accumulator layout of delta_l),
// delta_{l-1} = G_{l-1} * act'(H_{l-1}); finally dL/d(enc) = W_0^T delta_0.
// Weight gradients dW_l = sum_q delta_l[u][q] H_{l-1}[k][q] have the queries as
// the reduction dimension, split over query chunks with a deterministic
// second-pass reduction.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"
#include "mfma_common.h"
#include "model.h"
#include "nlod_common.h"
#include "wgrad.h"

namespace nlod {
namespace {

constexpr int kBlock = 256;
constexpr size_t kMaxLds = 160 * 1024;  // LDS of one CU

__device__ __forceinline__ size_t unit_major(uint32_t tile, uint32_t units, uint32_t u, uint32_t n) {
    return ((size_t)tile * units + u) * 16 + n;
}

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// 4 x 4 transpose among the lanes of a quad: element j of lane i becomes element
// i of lane j.  A lane holds 4 consecutive units of its query; transposed, it
// holds one unit of the quad's 4 queries, 8 contiguous bytes of a unit-major
// tensor (2-byte accesses, four times as many, bound the kernels below).
__device__ __forceinline__ half4_t quad_transpose(half4_t v) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 w = __builtin_bit_cast(u32x2, v);
    const bool odd = threadIdx.x & 1, upper = threadIdx.x & 2;
    const uint32_t n0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[0], 0xB1, 0xF, 0xF, false);
    const uint32_t n1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[1], 0xB1, 0xF, 0xF, false);
    // 2 x 2 blocks of halves: even lanes keep the low halves, odd lanes the high ones
    const uint32_t a = odd ? __builtin_amdgcn_perm(w[0], n0, 0x07060302u) : __builtin_amdgcn_perm(n0, w[0], 0x05040100u);
    const uint32_t b = odd ? __builtin_amdgcn_perm(w[1], n1, 0x07060302u) : __builtin_amdgcn_perm(n1, w[1], 0x05040100u);
    // 2 x 2 blocks of those pairs
    const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)(upper ? a : b), 0x4E, 0xF, 0xF, false);
    const u32x2 o = {upper ? r : a, upper ? b : r};
    return __builtin_bit_cast(half4_t, o);
}

// Units u .. u + 3 of query n of a tile (n = lane % 16, u a multiple of 4 and
// equal in the lanes of a quad), from or to a unit-major tensor.
__device__ __forceinline__ half4_t load_units(const half_t* __restrict__ t, uint32_t tile, uint32_t units, uint32_t u,
                                              uint32_t n) {
    return quad_transpose(*reinterpret_cast<const half4_t*>(t + unit_major(tile, units, u + (n & 3), n & ~3u)));
}
__device__ __forceinline__ void store_units(half_t* __restrict__ t, uint32_t tile, uint32_t units, uint32_t u,
                                            uint32_t n, half4_t v) {
    *reinterpret_cast<half4_t*>(t + unit_major(tile, units, u + (n & 3), n & ~3u)) = quad_transpose(v);
}

struct TrainArgs {
    uint32_t N, n_output, n_hidden_layers, k_enc, k_padded, width;
    int32_t act, out_act;
    uint32_t packed_halves, packed_bwd_halves;
};

// Forward for training: like the inference MLP but stores every hidden
// activation (exactly the FP16 values fed to the next layer) and y.
template <int W>
constexpr int kFwdThreads = W == 128 ? 512 : kBlock;  // width 128: one block per CU (110 to 150 KB of weights)
template <int W>
__global__ __launch_bounds__(kFwdThreads<W>) void mlp_fwd_train_kernel(TrainArgs a, const half_t* __restrict__ packed,
                                                                       const half_t* __restrict__ feat,
                                                                       half_t* __restrict__ H,
                                                                       float* __restrict__ out) {
    constexpr int NT = kFwdThreads<W>;
    constexpr int MT = W / 16, KC = W / 32;
    extern __shared__ float4 smem4[];
    half_t* sw = reinterpret_cast<half_t*>(smem4);
    stage_weights<NT>(sw, packed, a.packed_halves);
    __syncthreads();
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const uint32_t kc0 = a.k_padded / 32, kp2 = a.k_padded / 2;
    const uint32_t n_tiles = (a.N + 15) / 16;
    const uint32_t n_waves = gridDim.x * (NT / 64);
    const size_t layer_stride = (size_t)n_tiles * W * 16;
    for (uint32_t tile = blockIdx.x * (NT / 64) + (threadIdx.x >> 6); tile < n_tiles; tile += n_waves) {
        floatx4 acc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t c = 0; c < kc0; ++c) {
            const half8 b = load_feat_frag(feat, tile, kp2, c, g, n);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const half8 w = *reinterpret_cast<const half8*>(sw + ((size_t)(mt * kc0 + c) * 64 + lane) * 8);
                acc[mt] = mfma16(w, b, acc[mt]);
            }
        }
        const half_t* frag = sw + (size_t)MT * kc0 * 512;
        half8 b[KC];
        for (uint32_t layer = 0;; ++layer) {
            half_t* Hl = H + layer * layer_stride;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                b[c] = pack_act(acc[2 * c], acc[2 * c + 1], a.act);
                store_units(Hl, tile, W, 32 * c + 4 * g, n, __builtin_shufflevector(b[c], b[c], 0, 1, 2, 3));
                store_units(Hl, tile, W, 32 * c + 16 + 4 * g, n, __builtin_shufflevector(b[c], b[c], 4, 5, 6, 7));
            }
            if (layer + 1 >= a.n_hidden_layers) break;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < KC; ++c) {
                    const half8 w = *reinterpret_cast<const half8*>(frag + ((size_t)(mt * KC + c) * 64 + lane) * 8);
                    s = mfma16(w, b[c], s);
                }
                acc[mt] = s;
            }
            frag += (size_t)MT * KC * 512;
        }
        floatx4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const half8 w = *reinterpret_cast<const half8*>(frag + ((size_t)c * 64 + lane) * 8);
            o = mfma16(w, b[c], o);
        }
        const uint32_t q = tile * 16 + n;
        if (q < a.N) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t oi = 4 * g + i;
                if (oi < a.n_output) out[(size_t)q * a.n_output + oi] = act_fwd(a.out_act, o[i]);
            }
        }
    }
}

// The weights are staged in LDS, where they always fit (see mfma_mlp_backward).
// 101003 queries of the 144-input 128 x 4 network: 134 us with weights from the
// caches and 2-byte accesses to H and D, 93 us now (forward with saved
// activations: 58 -> 42 us).
template <int W>
__global__ __launch_bounds__(kFwdThreads<W>) void mlp_bwd_kernel(TrainArgs a, const half_t* __restrict__ packed_bwd,
                                                                 const half_t* __restrict__ H,
                                                                 const float* __restrict__ y,
                                                                 const float* __restrict__ dy, half_t* __restrict__ D,
                                                                 float* __restrict__ d_enc) {
    constexpr int MT = W / 16, KC = W / 32, NT = kFwdThreads<W>;
    extern __shared__ float4 smem4[];
    half_t* sw = reinterpret_cast<half_t*>(smem4);
    stage_weights<NT>(sw, packed_bwd, a.packed_bwd_halves);
    __syncthreads();
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const uint32_t n_tiles = (a.N + 15) / 16;
    const uint32_t n_waves = gridDim.x * (NT / 64);
    const uint32_t L = a.n_hidden_layers;
    const size_t layer_stride = (size_t)n_tiles * W * 16;
    half_t* D_out = D + (size_t)L * layer_stride;
    for (uint32_t tile = blockIdx.x * (NT / 64) + (threadIdx.x >> 6); tile < n_tiles; tile += n_waves) {
        const uint32_t q = tile * 16 + n;
        const bool valid = q < a.N;
        // delta_out = dL/dy * act'(y) (fully_fused_mlp.cu:757-760), rows 4g+i = outputs
        half8 bo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t oi = 4 * g + i;
            float d = 0.0f;
            if (valid && oi < a.n_output)
                d = dy[(size_t)q * a.n_output + oi] * act_bwd(a.out_act, y[(size_t)q * a.n_output + oi]);
            bo[i] = (half_t)d;
            bo[i + 4] = (half_t)0.0f;
        }
        store_units(D_out, tile, 16, 4 * g, n, __builtin_shufflevector(bo, bo, 0, 1, 2, 3));
        floatx4 acc[MT];
        const half_t* frag = sw;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const half8 w = *reinterpret_cast<const half8*>(frag + ((size_t)mt * 64 + lane) * 8);
            acc[mt] = mfma16(w, bo, floatx4{0.f, 0.f, 0.f, 0.f});
        }
        frag += (size_t)MT * 512;
        half8 b[KC];
        for (int layer = (int)L - 1; layer >= 0; --layer) {
            const half_t* Hl = H + (size_t)layer * layer_stride;
            half_t* Dl = D + (size_t)layer * layer_stride;
            // delta_layer = G * act'(H_layer), stored unit-major, packed as next B fragments
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                float y[8], dv[8];  // units 32c + 4g + i (i < 4) and 16 above them
                const uint32_t u0 = 32 * c + 4 * g, u1 = u0 + 16;
                const half4_t y0 = load_units(Hl, tile, W, u0, n), y1 = load_units(Hl, tile, W, u1, n);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    y[i] = (float)y0[i];
                    y[i + 4] = (float)y1[i];
                }
                act_bwd_n<8>(a.act, y, dv);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    b[c][i] = (half_t)(acc[2 * c][i] * dv[i]);
                    b[c][i + 4] = (half_t)(acc[2 * c + 1][i] * dv[i + 4]);
                }
                store_units(Dl, tile, W, u0, n, __builtin_shufflevector(b[c], b[c], 0, 1, 2, 3));
                store_units(Dl, tile, W, u1, n, __builtin_shufflevector(b[c], b[c], 4, 5, 6, 7));
            }
            if (layer == 0) break;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < KC; ++c) {
                    const half8 w = *reinterpret_cast<const half8*>(frag + ((size_t)(mt * KC + c) * 64 + lane) * 8);
                    s = mfma16(w, b[c], s);
                }
                acc[mt] = s;
            }
            frag += (size_t)MT * KC * 512;
        }
        if (!d_enc) continue;
        // dL/d(enc) = W_0^T delta_0, rows = encoded features
        const uint32_t mt0 = a.k_padded / 16;
        for (uint32_t mt = 0; mt < mt0; ++mt) {
            floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const half8 w = *reinterpret_cast<const half8*>(frag + ((size_t)(mt * KC + c) * 64 + lane) * 8);
                s = mfma16(w, b[c], s);
            }
            if (valid) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t row = 16 * mt + 4 * g + i;
                    if (row < a.k_enc) d_enc[(size_t)row * a.N + q] = s[i];
                }
            }
        }
    }
}

// dW partials: grid (chunks, 64 x 64 tiles of all matrices), see wgrad.h.  The
// reduction dimension is the queries: one v_mfma_f32_16x16x32_f16 takes 32 of
// them, lane group g the 8 queries 8 (g & 1) of query tile 2 step + (g >> 1), so
// a fragment of the unit-major tensors is one 16-byte load a lane.  The next
// step's fragments load while the current step's MFMAs run.
// 101003 queries through the 144-input 128 x 4 network: one block per (1024
// queries, matrix), whose waves loaded two fragments per 16x16x16 MFMA, took
// 931 us of a 1.46 ms training step, which is 0.58 ms with this split.
template <int RT, int CT>
__device__ __forceinline__ void wgrad_tile(const TrainArgs& a, const WgradItem& it, uint32_t step0, uint32_t step1,
                                           const half_t* __restrict__ feat, const half_t* __restrict__ Hp,
                                           const half_t* __restrict__ Dl, uint32_t d_units, float* __restrict__ p,
                                           uint32_t ld, float4* lds) {
    const int lane = threadIdx.x & 63, g = lane >> 4, m16 = lane & 15, wave = threadIdx.x >> 6;
    const uint32_t n_tiles = (a.N + 15) / 16, W = a.width, kp2 = a.k_padded / 2;
    floatx4 acc[RT * CT];
#pragma unroll
    for (int t = 0; t < RT * CT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    const uint32_t half_sel = (m16 & 1) ? 0x07060302u : 0x05040100u;
    auto load = [&](uint32_t step, half8 (&d)[RT], half8 (&x)[CT]) {
        const uint32_t qt = 2 * step + (uint32_t)(g >> 1), q8 = 8u * (uint32_t)(g & 1);
        const uint32_t tile = min(qt, n_tiles - 1);
#pragma unroll
        for (int r = 0; r < RT; ++r)
            d[r] = *reinterpret_cast<const half8*>(Dl + unit_major(tile, d_units, it.row0 + 16 * r + m16, q8));
        if (it.layer == 0) {  // X in the pair layout: this lane's half of 8 queries' pairs
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const uint32_t k = it.col0 + 16 * c + m16;
                const uint4* w = reinterpret_cast<const uint4*>(feat + feat_pair_offset(tile, k >> 1, kp2, q8));
                const uint4 w0 = w[0], w1 = w[1];
                const uint4 v = {__builtin_amdgcn_perm(w0.y, w0.x, half_sel), __builtin_amdgcn_perm(w0.w, w0.z, half_sel),
                                 __builtin_amdgcn_perm(w1.y, w1.x, half_sel), __builtin_amdgcn_perm(w1.w, w1.z, half_sel)};
                x[c] = __builtin_bit_cast(half8, v);
            }
        } else {
#pragma unroll
            for (int c = 0; c < CT; ++c)
                x[c] = *reinterpret_cast<const half8*>(Hp + unit_major(tile, W, it.col0 + 16 * c + m16, q8));
        }
        if (2 * step + 1 >= n_tiles) {  // the last step of an odd number of query tiles
            const half8 zero = {};
#pragma unroll
            for (int r = 0; r < RT; ++r) d[r] = qt < n_tiles ? d[r] : zero;
#pragma unroll
            for (int c = 0; c < CT; ++c) x[c] = qt < n_tiles ? x[c] : zero;
        }
    };
    half8 nd[RT], nx[CT];
    uint32_t step = step0 + (uint32_t)wave;
    if (step < step1) load(step, nd, nx);
    for (; step < step1; step += 4) {
        half8 d[RT], x[CT];
#pragma unroll
        for (int r = 0; r < RT; ++r) d[r] = nd[r];
#pragma unroll
        for (int c = 0; c < CT; ++c) x[c] = nx[c];
        if (step + 4 < step1) load(step + 4, nd, nx);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[r * CT + c] = mfma16(d[r], x[c], acc[r * CT + c]);
    }
    wgrad_add_waves<RT * CT>(acc, lds);
    if (wave != 0) return;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = it.row0 + 16 * r + 4 * g + i, col = it.col0 + 16 * c + m16;
                if (col < ld) p[(size_t)row * ld + col] = acc[r * CT + c][i];
            }
}

__global__ __launch_bounds__(kBlock, 3) void wgrad_mfma_kernel(TrainArgs a, const half_t* __restrict__ feat,
                                                               const half_t* __restrict__ H,
                                                               const half_t* __restrict__ D,
                                                               float* __restrict__ partial, uint32_t partial_stride,
                                                               uint32_t chunk_steps) {
    __shared__ float4 lds[2 * 16 * 64];
    const uint32_t L = a.n_hidden_layers, W = a.width;
    const WgradItem it = wgrad_item(blockIdx.y, WgradShape{W, a.k_padded, L, 16});
    const uint32_t n_tiles = (a.N + 15) / 16, n_steps = (n_tiles + 1) / 2;
    const uint32_t step0 = min(n_steps, blockIdx.x * chunk_steps), step1 = min(n_steps, step0 + chunk_steps);
    const size_t layer_stride = (size_t)n_tiles * W * 16;
    const uint32_t rows = it.layer == L ? 16u : W, cols = it.layer == 0 ? a.k_padded : W;
    const uint32_t ld = it.layer == 0 ? a.k_enc : W;
    const half_t* Dl = D + (size_t)it.layer * layer_stride;  // layer L: the output deltas
    const half_t* Hp = it.layer == 0 ? nullptr : H + (size_t)(it.layer - 1) * layer_stride;
    float* p = partial + (size_t)blockIdx.x * partial_stride +
               (it.layer == 0 ? 0 : (size_t)W * a.k_enc + (size_t)(it.layer - 1) * W * W);
    auto run = [&](auto RTc, auto CTc) {
        wgrad_tile<decltype(RTc)::value, decltype(CTc)::value>(a, it, step0, step1, feat, Hp, Dl, rows, p, ld, lds);
    };
    auto run_rows = [&](auto RTc) {  // widths are multiples of 32, so a tile is 32 or 64 wide
        if (cols - it.col0 >= kWgradTile) run(RTc, std::integral_constant<int, 4>{});
        else run(RTc, std::integral_constant<int, 2>{});
    };
    const uint32_t rt = (rows - it.row0) / 16;
    if (rt >= 4) run_rows(std::integral_constant<int, 4>{});
    else if (rt >= 2) run_rows(std::integral_constant<int, 2>{});
    else run_rows(std::integral_constant<int, 1>{});
}

TrainArgs make_targs(const Layout& L, uint32_t N) {
    TrainArgs a{};
    a.N = N;
    a.n_output = L.net.n_output;
    a.n_hidden_layers = L.net.n_hidden_layers;
    a.k_enc = L.net.n_input;
    a.k_padded = k_padded_of(L.net);
    a.width = L.net.width;
    a.act = L.net.activation;
    a.out_act = L.net.output_activation;
    a.packed_halves = (uint32_t)packed_halves(L.net);
    a.packed_bwd_halves = (uint32_t)packed_bwd_halves(L.net);
    return a;
}

template <typename Fn>
void by_w(uint32_t W, Fn&& f) {
    switch (W) {
        case 32: f(std::integral_constant<int, 32>{}); break;
        case 64: f(std::integral_constant<int, 64>{}); break;
        case 128: f(std::integral_constant<int, 128>{}); break;
        default: fail(NLOD_ERR_UNSUPPORTED, "FP16 MFMA kernels support widths 32, 64 and 128");
    }
}

template <typename Kern>
uint32_t persistent_blocks(Kern kern, int threads, size_t smem, uint32_t n_tiles) {
    const int occ = occupancy_blocks((const void*)kern, threads, smem);
    return std::min<uint32_t>(div_round_up(n_tiles, threads / 64), (uint32_t)(cu_count() * occ));
}

}  // namespace

size_t mfma_packed_bwd_bytes(const NetShape& net) { return packed_bwd_halves(net) * sizeof(half_t); }


size_t mfma_hidden_bytes(const Layout& L, uint32_t N) {
    return sizeof(half_t) * (size_t)L.net.n_hidden_layers * div_round_up(N, 16) * L.net.width * 16;
}

size_t mfma_delta_bytes(const Layout& L, uint32_t N) {
    return mfma_hidden_bytes(L, N) + sizeof(half_t) * (size_t)div_round_up(N, 16) * 16 * 16;
}

void mfma_mlp_forward_train(hipStream_t stream, const Layout& L, const void* packed, const void* feat, uint32_t N,
                            void* hidden, float* out) {
    if (N == 0) return;
    const TrainArgs a = make_targs(L, N);
    const size_t smem = mfma_packed_bytes(L.net);
    by_w(L.net.width, [&](auto Wc) {
        constexpr int W = decltype(Wc)::value;
        auto kern = mlp_fwd_train_kernel<W>;
        const uint32_t blocks = persistent_blocks(kern, kFwdThreads<W>, smem, div_round_up(N, 16));
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kFwdThreads<W>), smem, stream, a, static_cast<const half_t*>(packed),
                           static_cast<const half_t*>(feat), static_cast<half_t*>(hidden), out);
    });
    NLOD_LAUNCH_CHECK();
}

void mfma_mlp_backward(hipStream_t stream, const Layout& L, const void* packed_bwd, const void* hidden,
                       const float* y, const float* dy, uint32_t N, void* delta, float* d_enc) {
    if (N == 0) return;
    const TrainArgs a = make_targs(L, N);
    // mfma_supported holds the forward packing to 160 KB, that is to 160 fragments
    // of 1 KB.  The backward packing has W / 32 fragments more (W / 16 for the
    // output matrix instead of W / 32); without the output matrix both have a
    // multiple of W / 16, so that at most 160 - W / 16 of the forward packing's 160
    // are the shared ones, and the backward packing fits as well.
    const size_t smem = mfma_packed_bwd_bytes(L.net);
    if (smem > kMaxLds) fail(NLOD_ERR_UNSUPPORTED, "the backward weights do not fit in LDS");
    by_w(L.net.width, [&](auto Wc) {
        constexpr int W = decltype(Wc)::value;
        auto kern = mlp_bwd_kernel<W>;
        const uint32_t blocks = persistent_blocks(kern, kFwdThreads<W>, smem, div_round_up(N, 16));
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kFwdThreads<W>), smem, stream, a, static_cast<const half_t*>(packed_bwd),
                           static_cast<const half_t*>(hidden), y, dy, static_cast<half_t*>(delta), d_enc);
    });
    NLOD_LAUNCH_CHECK();
}

static uint32_t wgrad_steps(uint32_t N) { return div_round_up(div_round_up(std::max<uint32_t>(N, 1), 16), 2); }
static uint32_t wgrad_chunks_of(const Layout& L, uint32_t N) {
    return wgrad_chunks(wgrad_items({L.net.width, k_padded_of(L.net), L.net.n_hidden_layers, 16}), wgrad_steps(N));
}

size_t mfma_wgrad_workspace_floats(const Layout& L, uint32_t N) {
    return (size_t)wgrad_chunks_of(L, N) * L.net.n_params();
}

void mfma_weight_grad(hipStream_t stream, const Layout& L, const void* feat, const void* hidden, const void* delta,
                      uint32_t N, float* grads, float* workspace, size_t workspace_floats, bool accumulate) {
    if (workspace_floats < mfma_wgrad_workspace_floats(L, N)) fail(NLOD_ERR_STATE, "weight-gradient workspace too small");
    const uint32_t n_net = (uint32_t)L.net.n_params();
    if (N == 0) {
        if (!accumulate) fill_f32(stream, grads, n_net, 0.0f);
        return;
    }
    const TrainArgs a = make_targs(L, N);
    const uint32_t chunks = wgrad_chunks_of(L, N);
    const uint32_t items = wgrad_items({a.width, a.k_padded, a.n_hidden_layers, 16});
    hipLaunchKernelGGL(wgrad_mfma_kernel, dim3(chunks, items), dim3(kBlock), 0, stream, a,
                       static_cast<const half_t*>(feat), static_cast<const half_t*>(hidden),
                       static_cast<const half_t*>(delta), workspace, n_net, div_round_up(wgrad_steps(N), chunks));
    NLOD_LAUNCH_CHECK();
    partial_reduce(stream, n_net, chunks, workspace, grads, accumulate);
}

}  // namespace nlod
