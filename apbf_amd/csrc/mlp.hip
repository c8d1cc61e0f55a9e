// Learned lambda warm start: a 16-64-64-1 ReLU network on the matrix cores.
//
// BF16 weights and activations feed the matrix cores with FP32 accumulation:
// gfx950's v_mfma_f32_16x16x32_bf16 for the 64-deep products (layer 2 and
// its input gradient), v_mfma_f32_16x16x16_bf16 for the 16-deep ones (layer
// 1, whose input has 16 features, and the weight gradients, summed over the
// 16 samples of a tile). Biases, the last layer and all reductions stay FP32.
// One 64-lane wavefront handles a tile of 16 samples, independent of the other
// waves of its block. In the 16x16x16 operand layout (A: lane l holds row l%16,
// k = 4(l/16)..+3; B: lane l holds column l%16, k = 4(l/16)..+3; D: lane l holds
// column l%16, rows 4(l/16)..+3) a product's output is the operand of the next
// one that contracts over its rows; which way round a product is done decides
// whether these are the hidden units (the next layer) or the samples (the weight
// gradients).
//
// Training keeps FP32 master weights and Adam moments; every step writes
// per-block gradient partials, and a second kernel sums them in a fixed order
// (deterministic) and applies Adam.
#include "apbf_internal.h"
#include "mlp.h"

namespace apbf {

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));  // a caller's row: aligned as a float

__device__ __forceinline__ bf16x4_t pack4(f32x4_t x) {  // round to nearest even (v_cvt_pk_bf16_f32)
    typedef __bf16 v4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(bf16x4_t, __builtin_convertvector(x, v4));
}
__device__ __forceinline__ bf16x8_t pack8(f32x4_t x, f32x4_t y) {
    return __builtin_convertvector(__builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7), bf16x8_t);
}
__device__ __forceinline__ f32x4_t relu4(f32x4_t x) {
    return f32x4_t{fmaxf(x[0], 0.0f), fmaxf(x[1], 0.0f), fmaxf(x[2], 0.0f), fmaxf(x[3], 0.0f)};
}
__device__ __forceinline__ f32x4_t load4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ f32x4_t mfma(bf16x4_t a, bf16x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// gfx950's 16x16x32 form for the 64-deep products (layer 2 and its input
// gradient): lane l holds row / column l%16 and k = 8(l/16) .. +7 of A / B;
// D as in the 16x16x16 form.
__device__ __forceinline__ f32x4_t mfma32(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// A wavefront's LDS tile written by some lanes and read by others (and the
// reverse before the next write): a wavefront-level fence, no block barrier.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int MLP_WAVES = 4;               // waves per block
constexpr int MLP_THREADS = 64 * MLP_WAVES;

// Tile t, place m of the products holds hidden unit mlp_unit(16t + m): with the
// units of two tiles dealt out four by four, the four rows that a lane gets of
// each tile are the eight consecutive units it has to hold of the next product's
// operand, so a layer's output is the next layer's input without leaving its lane.
__host__ __device__ constexpr int mlp_unit(int place) {
    return (place & 32) | ((place & 12) << 1) | ((place & 16) >> 2) | (place & 3);
}
__host__ __device__ constexpr int mlp_place(int unit) {
    return (unit & 32) | ((unit & 24) >> 1) | ((unit & 4) << 2) | (unit & 3);
}

// Inference: out[s] = network(features[s]) * out_scale for s < *d_len. A wave
// holds the whole network in registers and takes 16 samples at a time, hidden
// units down the rows and samples along the columns of every product, so nothing
// goes through LDS. Bound by memory (64 B in and 4 B out per sample); the features of
// the next MLP_INFER_AHEAD tiles are on their way while one is computed. 1.1 M
// samples: 38 us, where turning layer 1's output through LDS 16 samples at a time
// with strided reads of the weights took 83; 4 M: 126 us a call, 3.2 TB/s.
constexpr int MLP_INFER_AHEAD = 2;
__global__ __launch_bounds__(MLP_THREADS) void k_mlp_infer(const float* __restrict__ params,
                                                           const float* __restrict__ norm,
                                                           const float* __restrict__ x,
                                                           const uint32_t* __restrict__ d_len,
                                                           float* __restrict__ out) {
    const uint32_t n = *d_len;
    const int l = threadIdx.x & 63, lo = l & 15, hi = l >> 4;
    const uint64_t step = (uint64_t)gridDim.x * MLP_WAVES * 16;
    uint64_t s = ((uint64_t)blockIdx.x * MLP_WAVES + (threadIdx.x >> 6)) * 16 + lo;
    if (s - lo >= n) return;
    f32x4_any_t ahead[MLP_INFER_AHEAD];
    const auto load = [&](uint64_t at) {
        return at < n ? *reinterpret_cast<const f32x4_any_t*>(x + at * MLP_IN + 4 * hi) : f32x4_any_t{0, 0, 0, 0};
    };
#pragma unroll
    for (int u = 0; u < MLP_INFER_AHEAD; ++u) ahead[u] = load(s + u * step);
    const f32x4_any_t mean = *reinterpret_cast<const f32x4_any_t*>(norm + 4 * hi);
    const f32x4_any_t scale = *reinterpret_cast<const f32x4_any_t*>(norm + MLP_IN + 4 * hi);
    const float out_scale = norm[2 * MLP_IN], b3 = params[MLP_OFF_B3];
    bf16x4_t w1[4];
    bf16x8_t w2[4][2];
    f32x4_t b1[4], b2[4], w3[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        w1[t] = pack4(load4(params + MLP_OFF_W1 + mlp_unit(16 * t + lo) * MLP_IN + 4 * hi));
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            const float* w = params + MLP_OFF_W2 + (16 * t + lo) * MLP_H + 32 * kt + 8 * hi;
            w2[t][kt] = pack8(load4(w), load4(w + 4));
        }
        b1[t] = load4(params + MLP_OFF_B1 + mlp_unit(16 * t + 4 * hi));
        b2[t] = load4(params + MLP_OFF_B2 + 16 * t + 4 * hi);
        w3[t] = load4(params + MLP_OFF_W3 + 16 * t + 4 * hi);
    }
    while (s - lo < n) {
#pragma unroll
        for (int u = 0; u < MLP_INFER_AHEAD; ++u, s += step) {
            const f32x4_any_t v = ahead[u];
            ahead[u] = load(s + MLP_INFER_AHEAD * step);
            const bf16x4_t a =
                s < n ? pack4(f32x4_t{(v[0] - mean[0]) * scale[0], (v[1] - mean[1]) * scale[1],
                                      (v[2] - mean[2]) * scale[2], (v[3] - mean[3]) * scale[3]})
                      : bf16x4_t{0, 0, 0, 0};
            bf16x8_t h1[2];
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
                h1[kt] = pack8(relu4(mfma(w1[2 * kt], a, b1[2 * kt])), relu4(mfma(w1[2 * kt + 1], a, b1[2 * kt + 1])));
            // layer 3 (FP32): units 4hi + r of every tile, then the 16 sums pairwise
            float p[4] = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x4_t z2 = mfma32(w2[t][1], h1[1], mfma32(w2[t][0], h1[0], b2[t]));
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] += fmaxf(z2[r], 0.0f) * w3[t][r];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] += __shfl_xor(p[r], 32, 64);
                p[r] += __shfl_xor(p[r], 16, 64);
            }
            if (hi == 0 && s < n) out[s] = (((p[0] + p[2]) + (p[1] + p[3])) + b3) * out_scale;
        }
    }
}

// A block's gradient partial, in the order the lanes hold it: four floats per
// lane and tile of W1 (4 tiles) and W2 (16), then b1, b2, w3 and a float that is
// b3 in lane 0 and the loss in lane 1.
constexpr int MLP_FRAGS = 4 + 16 + 1;
constexpr int MLP_PARTIAL = MLP_FRAGS * 256;
// Parameter that float q of a partial belongs to: MLP_PARAMS is the loss, -1 none.
__device__ __forceinline__ int mlp_partial_param(int q) {
    const int f = q >> 8, l = (q >> 2) & 63, r = q & 3, lo = l & 15, row = 4 * (l >> 4) + r;
    if (f < 4) return MLP_OFF_W1 + mlp_unit(16 * f + lo) * MLP_IN + row;
    if (f < 20) {
        const int g = f - 4;  // tile of inputs g / 4, of outputs g % 4
        return MLP_OFF_W2 + mlp_unit(16 * (g & 3) + lo) * MLP_H + mlp_unit(16 * (g >> 2) + row);
    }
    if (r < 3) return (r == 0 ? MLP_OFF_B1 : r == 1 ? MLP_OFF_B2 : MLP_OFF_W3) + mlp_unit(l);
    return l == 0 ? MLP_OFF_B3 : l == 1 ? MLP_PARAMS : -1;
}

// The network in LDS for the gradient: rows in the order of their places,
// padded so that the 16 rows that a read takes lie in different banks.
constexpr int MLP_ROW1 = MLP_IN + 4, MLP_ROW2 = MLP_H + 8;
struct MlpShared {
    alignas(16) uint16_t w2[MLP_H * MLP_ROW2], w2t[MLP_H * MLP_ROW2];  // [n][k] and [k][n], first index by place
    alignas(16) uint16_t w1[MLP_H * MLP_ROW1];
    alignas(16) uint16_t xt[MLP_WAVES][16 * MLP_ROW1];  // a wave's features [sample][feature]
    alignas(16) float b1[MLP_H], b2[MLP_H], w3[MLP_H];  // by place
};
union MlpGradShared {
    MlpShared net;
    f32x4_t sum[2][MLP_FRAGS * 64];  // once the samples are done
};

__device__ void load_network(const float* __restrict__ p, MlpShared& sh) {
#pragma unroll
    for (int q = 0; q < MLP_H * MLP_H / 4 / MLP_THREADS; ++q) {
        const int i = 4 * (q * MLP_THREADS + (int)threadIdx.x), n = i / MLP_H, k = i % MLP_H;
        const bf16x4_t v = pack4(load4(p + MLP_OFF_W2 + i));
        *reinterpret_cast<bf16x4_t*>(&sh.w2[mlp_place(n) * MLP_ROW2 + k]) = v;
#pragma unroll
        for (int j = 0; j < 4; ++j) sh.w2t[mlp_place(k + j) * MLP_ROW2 + n] = (uint16_t)v[j];
    }
    {
        static_assert(MLP_H * MLP_IN == 4 * MLP_THREADS, "one load of W1 per thread");
        const int i = 4 * (int)threadIdx.x;
        *reinterpret_cast<bf16x4_t*>(&sh.w1[mlp_place(i / MLP_IN) * MLP_ROW1 + i % MLP_IN]) =
            pack4(load4(p + MLP_OFF_W1 + i));
    }
    if (threadIdx.x < MLP_H) {
        const int at = mlp_place((int)threadIdx.x);
        sh.b1[at] = p[MLP_OFF_B1 + threadIdx.x];
        sh.b2[at] = p[MLP_OFF_B2 + threadIdx.x];
        sh.w3[at] = p[MLP_OFF_W3 + threadIdx.x];
    }
    __syncthreads();
}

// One training step: gradient of 0.5 * mean((y - t/out_scale)^2) over the
// batch perm[start .. start+batch) (indices wrap modulo n), a partial per block.
//
// A wave takes 16 samples at a time. The weight gradients sum over samples and
// want a lane to hold one unit and four samples, the next layer wants it to hold
// one sample and eight units: each product is done both ways round (the second
// is a few cycles of an idle matrix core) instead of turning its result through
// LDS. The rows are read through perm, one tile ahead of their use. What bounds
// it is what a block does once: the network into LDS, and the sum of its waves
// and its partial out; two blocks per CU fill the registers, so the grid has no
// more than 512, and a partial is stored in the order the lanes hold it.
// 262 147 samples: 33 us, where the products turned through LDS, weights read from
// unpadded rows, 1 024 blocks and a serial sum of the waves took 171 and a gather of
// the rows before it 12.
__global__ __launch_bounds__(MLP_THREADS, 2) void k_mlp_grad(const float* __restrict__ params,
                                                             const float* __restrict__ norm,
                                                             const float* __restrict__ x,
                                                             const float* __restrict__ target,
                                                             const uint32_t* __restrict__ perm, uint32_t n,
                                                             uint32_t start, uint32_t batch,
                                                             float* __restrict__ partial) {
    __shared__ MlpGradShared shared;
    MlpShared& sh = shared.net;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, lo = l & 15, hi = l >> 4;
    const uint32_t step = gridDim.x * MLP_WAVES * 16;
    // the lane's sample of the current tile, its features 4hi .. +3 and target, and the next tile's row
    uint64_t b = ((uint64_t)blockIdx.x * MLP_WAVES + wave) * 16 + lo;
    const auto row_of = [&](uint64_t i) {
        const uint64_t at = start + i;
        return perm[at < n ? at : at - n];
    };
    uint32_t row = b < batch ? row_of(b) : 0u;
    uint32_t row_next = b + step < batch ? row_of(b + step) : 0u;
    f32x4_any_t x_next = {0, 0, 0, 0};
    float t_next = 0.0f;
    if (b < batch) {
        x_next = *reinterpret_cast<const f32x4_any_t*>(x + (size_t)row * MLP_IN + 4 * hi);
        t_next = target[row];
    }
    const f32x4_any_t mean = *reinterpret_cast<const f32x4_any_t*>(norm + 4 * hi);
    const f32x4_any_t scale = *reinterpret_cast<const f32x4_any_t*>(norm + MLP_IN + 4 * hi);
    const float out_scale = norm[2 * MLP_IN], b3 = params[MLP_OFF_B3];
    load_network(params, sh);
    const float inv_b = 1.0f / (float)batch;
    f32x4_t gw1[4], gw2[4][4];
    float gb1[4] = {0, 0, 0, 0}, gb2[4] = {0, 0, 0, 0}, gw3[4] = {0, 0, 0, 0}, gb3 = 0.0f, loss = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        gw1[t] = f32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < 4; ++u) gw2[t][u] = f32x4_t{0, 0, 0, 0};
    }
    uint16_t* xt = sh.xt[wave];
    for (; b - lo < batch; b += step) {
        const bool valid = b < batch;
        f32x4_t v = {0, 0, 0, 0};
        if (valid)
            v = f32x4_t{(x_next[0] - mean[0]) * scale[0], (x_next[1] - mean[1]) * scale[1],
                        (x_next[2] - mean[2]) * scale[2], (x_next[3] - mean[3]) * scale[3]};
        const float tgt = t_next;
        if (b + step < batch) {
            x_next = *reinterpret_cast<const f32x4_any_t*>(x + (size_t)row_next * MLP_IN + 4 * hi);
            t_next = target[row_next];
        }
        if (b + 2ull * step < batch) row_next = row_of(b + 2ull * step);
        const bf16x4_t a = pack4(v);
        *reinterpret_cast<bf16x4_t*>(&xt[lo * MLP_ROW1 + 4 * hi]) = a;
        wave_lds_sync();
        bf16x4_t xa;  // feature lo of samples 4hi .. +3
#pragma unroll
        for (int r = 0; r < 4; ++r) xa[r] = (short)xt[(4 * hi + r) * MLP_ROW1 + lo];
        wave_lds_sync();
        // Layer 1. z1: sample 4hi + r, unit lo of tile t; the turned product becomes the lane's own
        // sample's input of layer 2.
        f32x4_t z1[4];
        bf16x8_t h1[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            f32x4_t turned[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int t = 2 * kt + e;
                const bf16x4_t w = *reinterpret_cast<const bf16x4_t*>(&sh.w1[(16 * t + lo) * MLP_ROW1 + 4 * hi]);
                const float bias = sh.b1[16 * t + lo];
                z1[t] = mfma(a, w, f32x4_t{bias, bias, bias, bias});
                turned[e] = relu4(mfma(w, a, load4(&sh.b1[16 * t + 4 * hi])));
            }
            h1[kt] = pack8(turned[0], turned[1]);
        }
        // Layer 2, both ways round, and the output of sample lo
        f32x4_t z2[4], z2t[4];
        float p = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float bias = sh.b2[16 * t + lo];
            z2[t] = f32x4_t{bias, bias, bias, bias};
            z2t[t] = load4(&sh.b2[16 * t + 4 * hi]);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const bf16x8_t w =
                    *reinterpret_cast<const bf16x8_t*>(&sh.w2[(16 * t + lo) * MLP_ROW2 + 32 * kt + 8 * hi]);
                z2[t] = mfma32(h1[kt], w, z2[t]);
                z2t[t] = mfma32(w, h1[kt], z2t[t]);
            }
            const f32x4_t w3 = load4(&sh.w3[16 * t + 4 * hi]);
#pragma unroll
            for (int r = 0; r < 4; ++r) p += fmaxf(z2t[t][r], 0.0f) * w3[r];
        }
        p += __shfl_xor(p, 32, 64);
        p += __shfl_xor(p, 16, 64);
        const float d = valid ? (p + b3) - tgt / out_scale : 0.0f;
        const float dy = d * inv_b;
        if (hi == 0) {
            loss += 0.5f * d * d * inv_b;
            gb3 += dy;
        }
        float dys[4];  // of samples 4hi + r
#pragma unroll
        for (int r = 0; r < 4; ++r) dys[r] = __shfl(dy, 4 * hi + r, 64);
        // Layer 3 and layer 2's pre-activation gradient, both ways round
        bf16x4_t dz2b[4];
        bf16x8_t ad[2];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float w = sh.w3[16 * t + lo];
            f32x4_t g;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gw3[t] += fmaxf(z2[t][r], 0.0f) * dys[r];
                g[r] = z2[t][r] > 0.0f ? dys[r] * w : 0.0f;
                gb2[t] += g[r];
            }
            dz2b[t] = pack4(g);
            const f32x4_t w3 = load4(&sh.w3[16 * t + 4 * hi]);
#pragma unroll
            for (int r = 0; r < 4; ++r) z2t[t][r] = z2t[t][r] > 0.0f ? dy * w3[r] : 0.0f;
        }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) ad[kt] = pack8(z2t[2 * kt], z2t[2 * kt + 1]);
        // dW2[k][n] += sum_s relu(z1)[s][k] dz2[s][n]
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const bf16x4_t h = pack4(relu4(z1[mt]));
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) gw2[mt][nt] = mfma(h, dz2b[nt], gw2[mt][nt]);
        }
        // dh1 = dz2 . W2, then dW1[f][k] += sum_s x[s][f] dz1[s][k]
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4_t c = {0, 0, 0, 0};
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
                c = mfma32(ad[kt],
                           *reinterpret_cast<const bf16x8_t*>(&sh.w2t[(16 * t + lo) * MLP_ROW2 + 32 * kt + 8 * hi]), c);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                c[r] = z1[t][r] > 0.0f ? c[r] : 0.0f;
                gb1[t] += c[r];
            }
            gw1[t] = mfma(xa, pack4(c), gw1[t]);
        }
    }
    // the per-lane sums over the four row groups; lane l keeps place l
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        gb1[t] += __shfl_xor(gb1[t], 16, 64);
        gb1[t] += __shfl_xor(gb1[t], 32, 64);
        gb2[t] += __shfl_xor(gb2[t], 16, 64);
        gb2[t] += __shfl_xor(gb2[t], 32, 64);
        gw3[t] += __shfl_xor(gw3[t], 16, 64);
        gw3[t] += __shfl_xor(gw3[t], 32, 64);
    }
#pragma unroll
    for (int m = 8; m > 0; m >>= 1) {
        gb3 += __shfl_xor(gb3, m, 64);
        loss += __shfl_xor(loss, m, 64);
    }
    f32x4_t rest = {hi == 0 ? gb1[0] : hi == 1 ? gb1[1] : hi == 2 ? gb1[2] : gb1[3],
                    hi == 0 ? gb2[0] : hi == 1 ? gb2[1] : hi == 2 ? gb2[2] : gb2[3],
                    hi == 0 ? gw3[0] : hi == 1 ? gw3[1] : hi == 2 ? gw3[2] : gw3[3], l == 0 ? gb3 : loss};
    const auto each = [&](auto&& f) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f(64 * t + l, gw1[t]);
#pragma unroll
            for (int u = 0; u < 4; ++u) f(64 * (4 + 4 * t + u) + l, gw2[t][u]);
        }
        f(64 * 20 + l, rest);
    };
    // block sum: waves 0 + 1 and 2 + 3, then both (a fixed order)
    for (int m = 1; m < MLP_WAVES; m *= 2) {
        __syncthreads();  // the network, or the sums before, are done with
        f32x4_t* sum = shared.sum[wave / (2 * m)];
        if (wave % (2 * m) == m) each([&](int at, f32x4_t& v) { sum[at] = v; });
        __syncthreads();
        if (wave % (2 * m) == 0) each([&](int at, f32x4_t& v) { v += sum[at]; });
    }
    if (wave == 0) {
        f32x4_t* out = reinterpret_cast<f32x4_t*>(partial) + (size_t)blockIdx.x * (MLP_FRAGS * 64);
        each([&](int at, f32x4_t& v) { out[at] = v; });
    }
}

// Sums the block partials (a fixed order) into grad[0 .. MLP_PARAMS] and,
// when lr > 0, applies one Adam step to the FP32 master parameters. The step
// number for the bias corrections is *step_base + k + 1: the device keeps the
// count, so captured steps replay with the right corrections. A block takes 64
// places of the partials and each of its waves a piece of the blocks, so that
// the reads of all pieces are in flight together. 512
// partials: 6 us (a thread per parameter over 1 024 of them: 84).
constexpr int MLP_ADAM_THREADS = 1024;
__global__ __launch_bounds__(MLP_ADAM_THREADS) void k_mlp_adam(const float* __restrict__ partial, uint32_t blocks,
                                                               float* __restrict__ grad, float* __restrict__ params,
                                                               float* __restrict__ m1, float* __restrict__ m2,
                                                               float lr, float beta1, float beta2, float eps,
                                                               const uint32_t* __restrict__ step_base, uint32_t k,
                                                               float* __restrict__ loss_out) {
    constexpr uint32_t WAVES = MLP_ADAM_THREADS / 64;
    __shared__ float sum[WAVES][64];
    const uint32_t wave = threadIdx.x >> 6, l = threadIdx.x & 63u, q = blockIdx.x * 64u + l;
    const uint32_t piece = (blocks + WAVES - 1) / WAVES;
    const uint32_t last = min(blocks, (wave + 1) * piece);
    float g = 0.0f;
#pragma unroll 8
    for (uint32_t b = wave * piece; b < last; ++b) g += partial[(size_t)b * MLP_PARTIAL + q];
    sum[wave][l] = g;
    __syncthreads();
    if (wave) return;
    g = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < WAVES; ++w) g += sum[w][l];
    const int p = mlp_partial_param((int)q);
    if (p < 0) return;
    if (p == MLP_PARAMS) {
        if (loss_out) *loss_out = g;
        return;
    }
    grad[p] = g;
    if (lr > 0.0f) {
        const float t = (float)(*step_base + k + 1u);
        const float bc1 = 1.0f - powf(beta1, t), bc2 = 1.0f - powf(beta2, t);
        const float a = beta1 * m1[p] + (1.0f - beta1) * g;
        const float v = beta2 * m2[p] + (1.0f - beta2) * g * g;
        m1[p] = a;
        m2[p] = v;
        params[p] -= lr * (a / bc1) / (sqrtf(v / bc2) + eps);
    }
}

__global__ void k_mlp_steps_done(uint32_t* __restrict__ step_base, uint32_t steps) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *step_base += steps;
}

// ------------------------------------------------------------------- host
static uint32_t mlp_grid_tiles(uint32_t samples, uint32_t max_blocks) {
    const uint32_t tiles = samples / 16 + (samples % 16 ? 1u : 0u);
    const uint32_t g = (tiles + MLP_WAVES - 1) / MLP_WAVES;
    return g < max_blocks ? (g ? g : 1u) : max_blocks;
}
// As many blocks as the registers let the chip hold at once: three per CU for the
// inference (1 024 blocks with one tile ahead left a quarter of them for a second
// round: 43 us at 1.1 M samples, against 38), two for the gradient (one per CU is
// 161 us a call at 1 M samples, against 133).
constexpr uint32_t MLP_INFER_BLOCKS = 768;
constexpr uint32_t MLP_GRAD_BLOCKS = 512;

void launch_mlp_infer(const float* params, const float* norm, const float* x, const uint32_t* d_len, uint32_t cap,
                      float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_infer, dim3(mlp_grid_tiles(cap, MLP_INFER_BLOCKS)), dim3(MLP_THREADS), 0, s, params, norm, x, d_len, out);
}

}  // namespace apbf

using namespace apbf;


// The captured training launches hold the buffers' addresses: any
// reallocation drops them.
static void drop_training_graph(apbf_mlp* m) {
    if (m->graph) (void)hipGraphExecDestroy(m->graph);
    m->graph = nullptr;
}

static apbf_status mlp_reserve(apbf_mlp* m, uint32_t batch, uint32_t steps, uint32_t n) {
    const uint32_t blocks = mlp_grid_tiles(batch, MLP_GRAD_BLOCKS);
    if (blocks > m->max_blocks || steps > m->max_steps || n > m->max_n) drop_training_graph(m);
    if (blocks > m->max_blocks) {
        if (m->partial) (void)hipFree(m->partial);
        if (hipMalloc(&m->partial, (size_t)blocks * MLP_PARTIAL * 4) != hipSuccess) return APBF_ERR_HIP;
        m->max_blocks = blocks;
    }
    if (steps > m->max_steps) {
        if (m->loss) (void)hipFree(m->loss);
        if (hipMalloc(&m->loss, (size_t)steps * 4) != hipSuccess) return APBF_ERR_HIP;
        m->max_steps = steps;
    }
    if (n > m->max_n) {
        if (m->perm) (void)hipFree(m->perm);
        if (hipMalloc(&m->perm, (size_t)n * 4) != hipSuccess) return APBF_ERR_HIP;
        m->max_n = n;
    }
    return APBF_OK;
}

// The launches of one training call (steps of gradient and Adam,
// then the step counter), on stream s.
static void enqueue_training(apbf_mlp* m, const float* features, const float* targets, const uint32_t* perm,
                             uint32_t n, uint32_t batch, uint32_t steps, float lr, hipStream_t s) {
    const uint32_t blocks = mlp_grid_tiles(batch, MLP_GRAD_BLOCKS);
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    for (uint32_t k = 0; k < (steps ? steps : 1u); ++k) {
        const uint32_t start = (uint32_t)(((uint64_t)k * batch) % n);
        hipLaunchKernelGGL(k_mlp_grad, dim3(blocks), dim3(MLP_THREADS), 0, s, m->params, m->norm, features, targets,
                           perm, n, start, batch, m->partial);
        hipLaunchKernelGGL(k_mlp_adam, dim3(MLP_PARTIAL / 64), dim3(MLP_ADAM_THREADS), 0, s, m->partial, blocks,
                           m->grad, m->params, m->m1, m->m2, steps ? lr : 0.0f, beta1, beta2, eps, m->step_base, k,
                           m->loss + k);
    }
    if (steps) hipLaunchKernelGGL(k_mlp_steps_done, dim3(1), dim3(64), 0, s, m->step_base, steps);
}

extern "C" {

apbf_status apbf_mlp_create(apbf_mlp** out) {
    if (!out) return APBF_ERR_INVALID_ARGUMENT;
    int dev = 0;
    if (hipGetDeviceCount(&dev) != hipSuccess || dev <= 0) return APBF_ERR_NO_DEVICE;
    apbf_mlp* m = new apbf_mlp();
    if (hipMalloc(&m->params, MLP_PARAMS * 4) != hipSuccess || hipMalloc(&m->norm, (2 * MLP_IN + 1) * 4) != hipSuccess ||
        hipMalloc(&m->m1, MLP_PARAMS * 4) != hipSuccess || hipMalloc(&m->m2, MLP_PARAMS * 4) != hipSuccess ||
        hipMalloc(&m->grad, MLP_PARAMS * 4) != hipSuccess || hipMalloc(&m->step_base, 4) != hipSuccess) {
        apbf_mlp_destroy(m);
        return APBF_ERR_HIP;
    }
    (void)hipMemset(m->step_base, 0, 4);
    (void)hipMemset(m->m1, 0, MLP_PARAMS * 4);
    (void)hipMemset(m->m2, 0, MLP_PARAMS * 4);
    (void)hipMemset(m->params, 0, MLP_PARAMS * 4);
    *out = m;
    return hipDeviceSynchronize() == hipSuccess ? APBF_OK : APBF_ERR_HIP;
}

apbf_status apbf_mlp_destroy(apbf_mlp* m) {
    if (!m) return APBF_ERR_INVALID_ARGUMENT;
    drop_training_graph(m);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    float* ps[] = {m->params, m->norm, m->m1, m->m2, m->grad, m->partial, m->loss};
    for (float* p : ps)
        if (p) (void)hipFree(p);
    if (m->perm) (void)hipFree(m->perm);
    if (m->step_base) (void)hipFree(m->step_base);
    delete m;
    return APBF_OK;
}

apbf_status apbf_mlp_set_params(apbf_mlp* m, const float* host_params, const float* host_norm) {
    if (!m || !host_params || !host_norm) return APBF_ERR_INVALID_ARGUMENT;
    if (hipMemcpy(m->params, host_params, MLP_PARAMS * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m->norm, host_norm, (2 * MLP_IN + 1) * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(m->m1, 0, MLP_PARAMS * 4) != hipSuccess || hipMemset(m->m2, 0, MLP_PARAMS * 4) != hipSuccess ||
        hipMemset(m->step_base, 0, 4) != hipSuccess)
        return APBF_ERR_HIP;
    return APBF_OK;
}

apbf_status apbf_mlp_get_params(apbf_mlp* m, float* host_params, float* host_norm) {
    if (!m) return APBF_ERR_INVALID_ARGUMENT;
    if ((host_params && hipMemcpy(host_params, m->params, MLP_PARAMS * 4, hipMemcpyDeviceToHost) != hipSuccess) ||
        (host_norm && hipMemcpy(host_norm, m->norm, (2 * MLP_IN + 1) * 4, hipMemcpyDeviceToHost) != hipSuccess))
        return APBF_ERR_HIP;
    return APBF_OK;
}

apbf_status apbf_mlp_forward(apbf_mlp* m, const float* features, const uint32_t* d_len, uint32_t capacity,
                             float* out, apbf_stream stream) {
    if (!m || !features || !d_len || !out) return APBF_ERR_INVALID_ARGUMENT;
    launch_mlp_infer(m->params, m->norm, features, d_len, capacity, out, reinterpret_cast<hipStream_t>(stream));
    return hipGetLastError() == hipSuccess ? APBF_OK : APBF_ERR_HIP;
}

apbf_status apbf_mlp_train(apbf_mlp* m, const float* features, const float* targets, const uint32_t* perm,
                           uint32_t n, uint32_t batch, uint32_t steps, float lr, float* host_losses,
                           apbf_stream stream) {
    if (!m || !features || !targets || !perm || n == 0 || batch == 0 || batch > n) return APBF_ERR_INVALID_ARGUMENT;
    apbf_status st = mlp_reserve(m, batch, steps ? steps : 1, n);
    if (st != APBF_OK) return st;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // The steps read the sample order from the network's own copy, so the
    // same captured launches serve every call with the same arguments.
    if (hipMemcpyAsync(m->perm, perm, (size_t)n * 4, hipMemcpyDeviceToDevice, s) != hipSuccess) return APBF_ERR_HIP;
    if (steps < 16) {
        enqueue_training(m, features, targets, m->perm, n, batch, steps, lr, s);
    } else {
        // many steps: one graph of the call's launches on the network's own
        // stream (captured at the first call with these arguments), ordered
        // after the caller's stream and before its later work
        if (!m->stream && hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) return APBF_ERR_HIP;
        if (!(m->graph && m->g_features == features && m->g_targets == targets && m->g_n == n &&
              m->g_batch == batch && m->g_steps == steps && m->g_lr == lr)) {
            drop_training_graph(m);
            hipGraph_t g = nullptr;
            if (hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return APBF_ERR_HIP;
            enqueue_training(m, features, targets, m->perm, n, batch, steps, lr, m->stream);
            if (hipStreamEndCapture(m->stream, &g) != hipSuccess || !g) return APBF_ERR_HIP;
            const bool ok = hipGraphInstantiate(&m->graph, g, nullptr, nullptr, 0) == hipSuccess;
            (void)hipGraphDestroy(g);
            if (!ok) {
                m->graph = nullptr;
                return APBF_ERR_HIP;
            }
            m->g_features = features;
            m->g_targets = targets;
            m->g_n = n;
            m->g_batch = batch;
            m->g_steps = steps;
            m->g_lr = lr;
        }
        hipEvent_t before = nullptr, after = nullptr;
        if (hipEventCreateWithFlags(&before, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&after, hipEventDisableTiming) != hipSuccess)
            return APBF_ERR_HIP;
        const bool ok = hipEventRecord(before, s) == hipSuccess && hipStreamWaitEvent(m->stream, before, 0) == hipSuccess &&
                        hipGraphLaunch(m->graph, m->stream) == hipSuccess && hipEventRecord(after, m->stream) == hipSuccess &&
                        hipStreamWaitEvent(s, after, 0) == hipSuccess;
        (void)hipEventDestroy(before);
        (void)hipEventDestroy(after);
        if (!ok) return APBF_ERR_HIP;
    }
    if (hipGetLastError() != hipSuccess) return APBF_ERR_HIP;
    if (host_losses) {
        if (hipMemcpyAsync(host_losses, m->loss, (size_t)(steps ? steps : 1) * 4, hipMemcpyDeviceToHost, s) !=
                hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return APBF_ERR_HIP;
    }
    return APBF_OK;
}

apbf_status apbf_mlp_gradient(apbf_mlp* m, const float* features, const float* targets, const uint32_t* perm,
                              uint32_t n, float* host_grad, float* host_loss, apbf_stream stream) {
    if (!m || !host_grad) return APBF_ERR_INVALID_ARGUMENT;
    apbf_status st = apbf_mlp_train(m, features, targets, perm, n, n, 0, 0.0f, host_loss, stream);
    if (st != APBF_OK) return st;
    if (hipMemcpy(host_grad, m->grad, MLP_PARAMS * 4, hipMemcpyDeviceToHost) != hipSuccess) return APBF_ERR_HIP;
    return APBF_OK;
}

}  // extern "C"
