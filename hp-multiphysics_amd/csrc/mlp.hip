// Preconditioner MLP: training and inference kernels for gfx950.
//
// Network 11 -> 64 -> 64 -> 64 -> 9, GELU (tanh form) on the hidden layers.  The
// FP32 master weights are rounded to bfloat16 (nearest even) for every matrix
// product and activations are rounded to bfloat16 on input to a product;
// accumulation is FP32.  Inference runs on the matrix cores (bf16 MFMA, 16 samples
// per tile), and so does training (bf16 MFMA forward, FP32 MFMA deltas and weight
// gradients); per-block partial gradients are summed in a fixed order by the Adam
// kernel, so training is bitwise reproducible.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/hpgpu.h"
#include "mlp.h"
#include "host_copy.h"

namespace hpg {

constexpr int MI = MLP_IN, MH = 64, MO = MLP_OUT;
static_assert(MO <= 16, "the inference head is one 16-row MFMA tile");
constexpr int O_W1 = 0, O_B1 = O_W1 + MI * MH, O_W2 = O_B1 + MH, O_B2 = O_W2 + MH * MH, O_W3 = O_B2 + MH,
              O_B3 = O_W3 + MH * MH, O_W4 = O_B3 + MH, O_B4 = O_W4 + MH * MO, NPARAM = O_B4 + MO;
constexpr float C_GELU = 0.7978845608028654f;  // sqrt(2/pi)

__host__ __device__ inline float bf16r(float x) {
    unsigned u;
    std::memcpy(&u, &x, 4);
    u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
    float r;
    std::memcpy(&r, &u, 4);
    return r;
}
__device__ inline float gelu(float z) {
    const float t = tanhf(C_GELU * (z + 0.044715f * z * z * z));
    return 0.5f * z * (1.f + t);
}

// ---- inference on the matrix cores -------------------------------------------------
// v_mfma_f32_16x16x16_bf16 with the hidden units as rows and 16 samples as columns.
// Operand layout: lane l holds A[l%16][4(l/16)+j] and B[4(l/16)+j][l%16] (j = 0..3);
// accumulator register i of lane l holds D[4(l/16)+i][l%16] (checked on the device
// by hpg_selftest_mfma_bf16).  The accumulators of output tile mt of one layer are
// therefore the B operand of K-step kt = mt of the next layer, lane for lane: the
// activations never leave registers.  Each wave holds every weight as A fragments
// (80 VGPRs) and sweeps 16-sample tiles; products of bfloat16 operands are exact in
// FP32 and accumulate in FP32.
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ inline short bf16_bits(float x) {
    unsigned u;
    std::memcpy(&u, &x, 4);
    return (short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

__device__ inline f32x4_t mfma_bf16(bf16x4_t a, bf16x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// GELU of the accumulators, rounded to bfloat16: the B operands of the next layer
__device__ inline void gelu_fragments(const f32x4_t z[4], bf16x4_t h[4]) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j) h[kt][j] = bf16_bits(gelu(z[kt][j]));
}

__global__ __launch_bounds__(256) void k_mlp_forward_mfma(int n, const float* __restrict__ X,
                                                          const float* __restrict__ wq, float* __restrict__ Y) {
    const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
    bf16x4_t A1[4], A2[4][4], A3[4][4], A4[4];
    f32x4_t b1[4], b2[4], b3[4], b4;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 4 * q + j;
            A1[mt][j] = k < MI ? bf16_bits(wq[O_W1 + k * MH + 16 * mt + c]) : (short)0;
        }
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = 16 * kt + 4 * q + j;
                A2[mt][kt][j] = bf16_bits(wq[O_W2 + k * MH + 16 * mt + c]);
                A3[mt][kt][j] = bf16_bits(wq[O_W3 + k * MH + 16 * mt + c]);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            b1[mt][i] = wq[O_B1 + 16 * mt + 4 * q + i];
            b2[mt][i] = wq[O_B2 + 16 * mt + 4 * q + i];
            b3[mt][i] = wq[O_B3 + 16 * mt + 4 * q + i];
        }
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 16 * kt + 4 * q + j;
            A4[kt][j] = c < MO ? bf16_bits(wq[O_W4 + k * MO + c]) : (short)0;
        }
#pragma unroll
    for (int i = 0; i < 4; ++i) b4[i] = 4 * q + i < MO ? wq[O_B4 + 4 * q + i] : 0.f;

    const long ntile = ((long)n + 15) / 16;
    for (long tile = (long)blockIdx.x * 4 + (threadIdx.x >> 6); tile < ntile; tile += (long)gridDim.x * 4) {
        const long s = tile * 16 + c;
        bf16x4_t h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 4 * q + j;
            h[0][j] = (s < n && k < MI) ? bf16_bits(X[s * MI + k]) : (short)0;
        }
        f32x4_t z[4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) z[mt] = mfma_bf16(A1[mt], h[0], b1[mt]);
        gelu_fragments(z, h);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4_t acc = b2[mt];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) acc = mfma_bf16(A2[mt][kt], h[kt], acc);
            z[mt] = acc;
        }
        gelu_fragments(z, h);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4_t acc = b3[mt];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) acc = mfma_bf16(A3[mt][kt], h[kt], acc);
            z[mt] = acc;
        }
        gelu_fragments(z, h);
        f32x4_t y = b4;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) y = mfma_bf16(A4[kt], h[kt], y);
        // register i of lane group q holds output 4q + i of sample column c
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < MO && s < n) Y[s * MO + 4 * q + i] = y[i];
    }
}

// one v_mfma_f32_16x16x16_bf16 on A, B (16 x 16 row-major, rounded to bfloat16)
__global__ void k_mfma_probe_bf16(const float* A, const float* B, float* out) {
    const int l = threadIdx.x, q = l >> 4, c = l & 15;
    bf16x4_t a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a[j] = bf16_bits(A[c * 16 + 4 * q + j]);
        b[j] = bf16_bits(B[(4 * q + j) * 16 + c]);
    }
    f32x4_t d = {0.f, 0.f, 0.f, 0.f};
    d = mfma_bf16(a, b, d);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[l * 4 + i] = d[i];
}

// ---- training step on the matrix cores ----------------------------------------------
// Forward, backward and weight gradients of 16-sample tiles, one tile per wave at a time;
// a wave keeps its sums of all 9 673 gradient entries in registers over its tiles, the
// block adds its four waves in a fixed order and writes one partial, so a minibatch of
// 65 536 samples writes 256 partials (the card's CUs) instead of one per 64 samples.
//   forward: the tiles of k_mlp_forward_mfma (bf16 products, FP32 accumulation);
//   deltas:  dz_l = (W_{l+1} dz_{l+1}) * gelu'(z_l) on v_mfma_f32_16x16x4f32.  The deltas
//            stay FP32 (the bf16 weights are exact in FP32); register i of output tile mt
//            holds unit 16 mt + 4 q + i, which is K-step (mt, i) of the next product;
//   weight gradients h_l^T dz_{l+1} contract over the samples, which sit in the lane
//            columns, so h and dz go through a transposed copy in LDS (row = unit, 16
//            samples, padded to 20 words: a lane's four samples are one 16-byte read, no
//            bank conflicts); v_mfma_f32_16x16x4f32 again.
// A minibatch takes 48 us (the weights and fragments built in LDS from scattered loads, the
// block sums, 8 us of the update kernel) and 13 us for each tile of a wave: 65 536 samples,
// four tiles a wave, 100 us (1 903 us for the sample-per-lane form with a reduction per
// parameter before it).  Of a tile's 13 us the FP32 matrix instructions are 4 (304 of 32
// cycles); the rest is the 48 tanh a lane and one wave per SIMD (all 512 registers, 108 bytes
// a lane in scratch) between the LDS round trips of its phases.
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ inline f4_t mfma_f32(float a, float b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ inline float bf16_value(short b) {
    const unsigned u = (unsigned)(unsigned short)b << 16;
    return __uint_as_float(u);
}

constexpr int TRAIN_BLOCKS = 256;         // partials of a minibatch at most: one block per CU
constexpr int TW = 68, TS = 20;           // LDS row strides (words): weights, transposed tiles
constexpr int LW2 = 0, LW3 = LW2 + MH * TW, LW4 = LW3 + MH * TW;         // FP32 weights by row
constexpr int LFW = LW4 + MH * TS;                                      // bf16 A fragments, 2 words a lane
constexpr int NFRAG = 40;                                               // 4 + 16 + 16 + 4
constexpr int LWAVE = LFW + NFRAG * 64 * 2;                             // per-wave tiles from here
constexpr int WTILE = 2 * MH * TS + 2 * 16 * TS;                        // h, dz, x, dy
constexpr int TRAIN_LDS = LWAVE + 4 * WTILE;
static_assert(NPARAM <= LWAVE, "the block's gradient sums reuse the weights' LDS");
static_assert(TRAIN_LDS * 4 <= 160 * 1024, "LDS of one CU");
static_assert(LWAVE % 2 == 0, "the block's loss is a double there");

// gelu(z) as bfloat16 bits (the B operands of the next layer) and gelu'(z) in place of z
__device__ inline void gelu_and_slope(f32x4_t z[4], bf16x4_t h[4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float v = z[t][j];
            const float th = tanhf(C_GELU * (v + 0.044715f * v * v * v));
            const float du = C_GELU * (1.f + 3.f * 0.044715f * v * v);
            h[t][j] = bf16_bits(0.5f * v * (1.f + th));
            z[t][j] = 0.5f * (1.f + th) + 0.5f * v * (1.f - th * th) * du;
        }
}

// orders this wave's LDS writes before its reads of other lanes' values
__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(256) void k_mlp_train_mfma(int n, int nscale, const float* __restrict__ X,
                                                        const float* __restrict__ T, const float* __restrict__ wq,
                                                        float* __restrict__ partial, double* __restrict__ lossp) {
    __shared__ __align__(16) float sm[TRAIN_LDS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 15;
    for (int k = threadIdx.x; k < MH * MH; k += 256) {
        const int i = k / MH, j = k % MH;
        sm[LW2 + i * TW + j] = wq[O_W2 + k];
        sm[LW3 + i * TW + j] = wq[O_W3 + k];
    }
    for (int k = threadIdx.x; k < MH * 16; k += 256) {
        const int i = k >> 4, o = k & 15;
        sm[LW4 + i * TS + o] = o < MO ? wq[O_W4 + i * MO + o] : 0.f;
    }
    bf16x4_t* const frag = reinterpret_cast<bf16x4_t*>(sm + LFW);
    for (int k = threadIdx.x; k < NFRAG * 64; k += 256) {
        const int f = k >> 6, l = k & 63, lq = l >> 4, lc = l & 15;
        bf16x4_t v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x;
            if (f < 4) {
                const int i = 4 * lq + j;
                x = i < MI ? wq[O_W1 + i * MH + 16 * f + lc] : 0.f;
            } else if (f < 36) {
                const int g = (f - 4) & 15, i = 16 * (g & 3) + 4 * lq + j;
                x = wq[(f < 20 ? O_W2 : O_W3) + i * MH + 16 * (g >> 2) + lc];
            } else {
                const int i = 16 * (f - 36) + 4 * lq + j;
                x = lc < MO ? wq[O_W4 + i * MO + lc] : 0.f;
            }
            v[j] = bf16_bits(x);
        }
        frag[k] = v;
    }
    __syncthreads();

    float* const sh = sm + LWAVE + w * WTILE;   // h of a layer, then
    float* const sd = sh + MH * TS;             // deltas of the layer above it
    float* const sx = sd + MH * TS;             // bf16(x), rows 11.. zero
    float* const sy = sx + 16 * TS;             // output deltas, rows 9.. zero
    const f4_t z0 = {0.f, 0.f, 0.f, 0.f};
    f4_t g2[4][4], g3[4][4], g1[4], g4[4];
    float gb1[4], gb2[4], gb3[4], gb4 = 0.f;
    double loss = 0.0;  // of any number of samples: FP32 would lose a large minibatch's digits
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        g1[a] = z0; g4[a] = z0; gb1[a] = gb2[a] = gb3[a] = 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b) { g2[a][b] = z0; g3[a][b] = z0; }
    }
    // rows of unit 16 t + c, samples 4 q .. 4 q + 3 of a transposed tile
    auto row = [&](const float* s, int t) { return *reinterpret_cast<const f4_t*>(s + (16 * t + c) * TS + 4 * q); };
    auto put_h = [&](const bf16x4_t* h) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) sh[(16 * t + 4 * q + i) * TS + c] = bf16_value(h[t][i]);
    };
    auto put_d = [&](const f4_t* d) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) sd[(16 * t + 4 * q + i) * TS + c] = d[t][i];
    };
    // sum over the tile's samples of h (64 rows) x d (64 columns); bias sums of d
    auto outer = [&](f4_t g[4][4], float* gb) {
        f4_t d[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            d[b] = row(sd, b);
            gb[b] += (d[b][0] + d[b][1]) + (d[b][2] + d[b][3]);
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f4_t h = row(sh, a);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int b = 0; b < 4; ++b) g[a][b] = mfma_f32(h[k], d[b][k], g[a][b]);
        }
    };
    // (W d) * slope, W rows in LDS at lw: the deltas of the layer below
    auto back = [&](int lw, const f4_t* d, const f32x4_t* slope, f4_t* out) {
#pragma unroll
        for (int r = 0; r < 4; ++r) out[r] = z0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f4_t a[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                a[r] = *reinterpret_cast<const f4_t*>(sm + lw + (16 * r + c) * TW + 16 * t + 4 * q);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) out[r] = mfma_f32(a[r][i], d[t][i], out[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[r][i] *= slope[r][i];
    };

    const int ntile = (n + 15) / 16;
    for (int tile = blockIdx.x * 4 + w; tile < ntile; tile += gridDim.x * 4) {
        const int s = tile * 16 + c;
        const bool ok = s < n;
        bf16x4_t hx, h1[4], h2[4], h3[4];
        f32x4_t s1[4], s2[4], s3[4];   // pre-activations, then gelu'
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 4 * q + j;
            hx[j] = (ok && k < MI) ? bf16_bits(X[(size_t)s * MI + k]) : (short)0;
            sx[k * TS + c] = bf16_value(hx[j]);
        }
        auto bias = [&](int o, int t) {
            f32x4_t b;
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = wq[o + 16 * t + 4 * q + i];
            return b;
        };
#pragma unroll
        for (int t = 0; t < 4; ++t) s1[t] = mfma_bf16(frag[t * 64 + lane], hx, bias(O_B1, t));
        gelu_and_slope(s1, h1);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            s2[t] = bias(O_B2, t);
#pragma unroll
            for (int k = 0; k < 4; ++k) s2[t] = mfma_bf16(frag[(4 + 4 * t + k) * 64 + lane], h1[k], s2[t]);
        }
        gelu_and_slope(s2, h2);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            s3[t] = bias(O_B3, t);
#pragma unroll
            for (int k = 0; k < 4; ++k) s3[t] = mfma_bf16(frag[(20 + 4 * t + k) * 64 + lane], h2[k], s3[t]);
        }
        gelu_and_slope(s3, h3);
        f32x4_t y;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = 4 * q + i < MO ? wq[O_B4 + 4 * q + i] : 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) y = mfma_bf16(frag[(36 + k) * 64 + lane], h3[k], y);
        f4_t dy;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int o = 4 * q + i;
            const float d = (ok && o < MO) ? y[i] - T[(size_t)s * MO + o] : 0.f;
            loss += (double)(d * d);
            dy[i] = 2.f * d / (float)nscale;
            sy[o * TS + c] = dy[i];
        }
        // dz3 and the gradients of the output layer
        f4_t da[4], db[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f4_t a = *reinterpret_cast<const f4_t*>(sm + LW4 + (16 * r + c) * TS + 4 * q);
            f4_t t = z0;
#pragma unroll
            for (int i = 0; i < 4; ++i) t = mfma_f32(a[i], dy[i], t);
#pragma unroll
            for (int i = 0; i < 4; ++i) da[r][i] = t[i] * s3[r][i];
        }
        put_h(h3);
        wave_lds_sync();
        {
            const f4_t d = row(sy, 0);
            gb4 += (d[0] + d[1]) + (d[2] + d[3]);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f4_t h = row(sh, a);
#pragma unroll
                for (int k = 0; k < 4; ++k) g4[a] = mfma_f32(h[k], d[k], g4[a]);
            }
        }
        wave_lds_sync();
        put_h(h2);
        put_d(da);
        wave_lds_sync();
        outer(g3, gb3);
        back(LW3, da, s2, db);
        wave_lds_sync();
        put_h(h1);
        put_d(db);
        wave_lds_sync();
        outer(g2, gb2);
        back(LW2, db, s1, da);
        wave_lds_sync();
        put_d(da);
        wave_lds_sync();
        {
            const f4_t x = row(sx, 0);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const f4_t d = row(sd, b);
                gb1[b] += (d[0] + d[1]) + (d[2] + d[3]);
#pragma unroll
                for (int k = 0; k < 4; ++k) g1[b] = mfma_f32(x[k], d[k], g1[b]);
            }
        }
        wave_lds_sync();
    }
    // block sums: waves 0..3 in order, in the weights' LDS; accumulator register i of lane
    // (q, c) is row 4 q + i, column c of its tile
    auto quarter = [&](float v) {   // over the four lane groups (the samples of a tile)
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
#pragma unroll
    for (int a = 0; a < 4; ++a) { gb1[a] = quarter(gb1[a]); gb2[a] = quarter(gb2[a]); gb3[a] = quarter(gb3[a]); }
    gb4 = quarter(gb4);
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_down(loss, off, 64);
    double* const lsum = reinterpret_cast<double*>(sm + LWAVE);
    for (int turn = 0; turn < 4; ++turn) {
        __syncthreads();
        if (turn != w) continue;
        auto add = [&](int p, float v) { sm[p] = w == 0 ? v : sm[p] + v; };
#pragma unroll
        for (int a = 0; a < 4; ++a) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * a + 4 * q + i;
                if (4 * q + i < MI) add(O_W1 + (4 * q + i) * MH + 16 * a + c, g1[a][i]);
                if (c < MO) add(O_W4 + r * MO + c, g4[a][i]);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    add(O_W2 + r * MH + 16 * b + c, g2[a][b][i]);
                    add(O_W3 + r * MH + 16 * b + c, g3[a][b][i]);
                }
            }
            if (q == 0) {
                add(O_B1 + 16 * a + c, gb1[a]);
                add(O_B2 + 16 * a + c, gb2[a]);
                add(O_B3 + 16 * a + c, gb3[a]);
            }
        }
        if (q == 0 && c < MO) add(O_B4 + c, gb4);
        if (lane == 0) *lsum = w == 0 ? loss : *lsum + loss;
    }
    __syncthreads();
    float* const P = partial + (size_t)blockIdx.x * NPARAM;
    for (int p = threadIdx.x; p < NPARAM; p += 256) P[p] = sm[p];
    if (threadIdx.x == 0) lossp[blockIdx.x] = *lsum;
}

// gradient = sum of the block partials in a fixed order (four lanes a quarter of the
// partials each, then the quarters in order); optional Adam step on the masters.  64
// parameters per block: 151 blocks keep the 38 KB partials streaming (242 us for 1 024
// partials with one lane per parameter before, 8 us for 256 now).  lsum (may
// be null) accumulates the minibatch's loss sum.
__global__ __launch_bounds__(256) void k_mlp_reduce_adam(int nblocks, const float* __restrict__ partial,
                                                         float* __restrict__ grad, float* master, float* wq,
                                                         float* m1, float* m2, float lr, float bc1, float bc2,
                                                         int do_step, const double* __restrict__ lossp, double* lsum) {
    __shared__ float part[4][64];
    const int j = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + j;
    const int per = (nblocks + 3) / 4, b0 = w * per, b1 = min(nblocks, b0 + per);
    float s = 0.f;
    if (p < NPARAM) {
#pragma unroll 8
        for (int b = b0; b < b1; ++b) s += partial[(size_t)b * NPARAM + p];
    }
    part[w][j] = s;
    __syncthreads();
    if (lsum && blockIdx.x == 0 && threadIdx.x == 64) {
        double l = lsum[0];
        for (int b = 0; b < nblocks; ++b) l += lossp[b];
        lsum[0] = l;
    }
    if (w != 0 || p >= NPARAM) return;
    const float g = ((part[0][j] + part[1][j]) + part[2][j]) + part[3][j];
    grad[p] = g;
    if (!do_step) return;
    const float a = 0.9f * m1[p] + 0.1f * g;
    const float v = 0.999f * m2[p] + 0.001f * g * g;
    m1[p] = a;
    m2[p] = v;
    const float x = master[p] - lr * (a / bc1) / (sqrtf(v / bc2) + 1e-8f);
    master[p] = x;
    const bool is_bias = (p >= O_B1 && p < O_W2) || (p >= O_B2 && p < O_W3) || (p >= O_B3 && p < O_W4) || p >= O_B4;
    wq[p] = is_bias ? x : bf16r(x);
}

// mean-square loss from the block losses: the same double sum, in block order, and
// the same final division as the host side of hpg_mlp_loss_grad
__global__ void k_mlp_loss_sum(int nblocks, const double* __restrict__ lossp, int nscale, float* __restrict__ loss) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double s = 0.0;
    for (int b = 0; b < nblocks; ++b) s += lossp[b];
    loss[0] = (float)(s / (double)nscale);
}

// Scratch of the allocation-free loss/gradient entry point: the per-block partial
// gradients (NPARAM floats per block of k_mlp_train_mfma, room for one block per 64
// samples) followed by the block losses (doubles, from the next even word).  One
// copy per GPU, held until the process ends; host code uses the address that
// hipGetSymbolAddress returns for the current device, never the symbol itself.
// Every call overwrites what it reads (each block writes all of its partials and
// its loss), and calls that overlap on one GPU race on it.
constexpr int NOALLOC_FLOATS = 4 << 20;  // 16 MiB
constexpr int NOALLOC_MAX_BLOCKS = NOALLOC_FLOATS / (NPARAM + 1);
static __device__ __align__(256) float scratch[NOALLOC_FLOATS];
static_assert((TRAIN_BLOCKS * NPARAM + 1) / 2 * 2 + 2 * TRAIN_BLOCKS <= NOALLOC_FLOATS, "partials and losses of a minibatch");
static_assert(NOALLOC_MAX_BLOCKS * 64 == HPG_MLP_NOALLOC_MAX_SAMPLES, "header limit out of step with the scratch size");

}  // namespace hpg

using namespace hpg;

struct hpg_mlp {
    hipStream_t stream = nullptr;
    HostCopyUser staging;
    float *master = nullptr, *wq = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
    float *partial = nullptr, *X = nullptr, *T = nullptr, *Y = nullptr;
    double* lossp = nullptr;  // a minibatch's block losses
    double* lsum = nullptr;  // loss sum of a training run's last epoch
    int cap_blocks = 0, cap_n = 0, step = 0;
    int dev = 0;  // device the MLP was created on
    std::string err;
    ~hpg_mlp() {
        for (float* p : {master, wq, m1, m2, grad, partial, X, T, Y})
            if (p) hipFree(p);
        for (double* p : {lossp, lsum})
            if (p) hipFree(p);
        if (stream) hipStreamDestroy(stream);
    }
};

namespace {
void ck(hipError_t e, const char* w) {
    if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}
void quantise(hpg_mlp* m, const std::vector<float>& w) {
    std::vector<float> q(w);
    for (int p = 0; p < NPARAM; ++p) {
        const bool is_bias = (p >= O_B1 && p < O_W2) || (p >= O_B2 && p < O_W3) || (p >= O_B3 && p < O_W4) || p >= O_B4;
        if (!is_bias) q[p] = bf16r(w[p]);
    }
    ck(hipMemcpyAsync(m->master, w.data(), NPARAM * 4, hipMemcpyHostToDevice, m->stream), "H2D");
    ck(hipMemcpyAsync(m->wq, q.data(), NPARAM * 4, hipMemcpyHostToDevice, m->stream), "H2D");
    ck(hipStreamSynchronize(m->stream), "sync");
}
void ensure_n(hpg_mlp* m, int n) {
    if (n <= m->cap_n) return;
    for (float** p : {&m->X, &m->T, &m->Y})
        if (*p) { hipFree(*p); *p = nullptr; }
    ck(hipMalloc(&m->X, (size_t)n * MI * 4), "hipMalloc");
    ck(hipMalloc(&m->T, (size_t)n * MO * 4), "hipMalloc");
    ck(hipMalloc(&m->Y, (size_t)n * MO * 4), "hipMalloc");
    m->cap_n = n;
}
// the caller's samples (and targets) into X (and T)
void send_batch(hpg_mlp* m, const float* X, const float* T, int n) {
    const HostSeg seg[2] = {{const_cast<float*>(X), m->X, (size_t)n * MI * 4},
                            {const_cast<float*>(T), m->T, T ? (size_t)n * MO * 4 : 0}};
    copy_to_device(m->stream, seg, 2);
}
// device address of `scratch` per GPU, resolved once per device with that device
// current (each GPU holds its own copy of the array at its own address)
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float* g_scratch[MAX_DEVICES] = {};

void resolve_scratch(int dev) {
    if (dev < 0 || dev >= MAX_DEVICES) throw std::runtime_error("device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch[dev]) return;
    void* p = nullptr;
    ck(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    if (!p) throw std::runtime_error("hipGetSymbolAddress(scratch) returned null");
    g_scratch[dev] = static_cast<float*>(p);
}

// blocks (= partials) of a minibatch: at least one 16-sample tile per wave, one block per
// CU at most, so larger minibatches give each wave more tiles instead of more partials
int train_blocks(int n) { return std::max(1, std::min((n + 63) / 64, TRAIN_BLOCKS)); }

// enqueue the backward pass of n samples (block partials and block losses into
// partial / lossp) and the ordered gradient sum into grad, no weight update
void enqueue_loss_grad(hpg_mlp* m, const float* X, const float* T, int n, float* partial, double* lossp,
                       float* grad) {
    const int nb = train_blocks(n);
    hipLaunchKernelGGL(k_mlp_train_mfma, dim3(nb), dim3(256), 0, m->stream, n, n * MO, X, T, m->wq, partial, lossp);
    hipLaunchKernelGGL(k_mlp_reduce_adam, dim3((NPARAM + 63) / 64), dim3(256), 0, m->stream, nb, partial, grad,
                       m->master, m->wq, m->m1, m->m2, 0.f, 1.f, 1.f, 0, (const double*)nullptr, (double*)nullptr);
}

void ensure_blocks(hpg_mlp* m, int nb) {
    if (nb <= m->cap_blocks) return;
    if (m->partial) hipFree(m->partial);
    if (m->lossp) hipFree(m->lossp);
    ck(hipMalloc(&m->partial, (size_t)nb * NPARAM * 4), "hipMalloc");
    ck(hipMalloc(&m->lossp, (size_t)nb * 8), "hipMalloc");
    m->cap_blocks = nb;
}
}  // namespace

namespace hpg {
void mlp_forward_device(const hpg_mlp* m, const float* X, int n, float* Y, hipStream_t stream) {
    if (n <= 0) return;
    // four 16-sample tiles per block and pass; at most 2048 blocks, each wave loops
    const long tiles = ((long)n + 15) / 16;
    const long blocks = std::min<long>((tiles + 3) / 4, 2048);
    hipLaunchKernelGGL(k_mlp_forward_mfma, dim3((unsigned)blocks), dim3(256), 0, stream, n, X, m->wq, Y);
}
}  // namespace hpg

extern "C" {

int hpg_mlp_create(unsigned seed, hpg_mlp** out) {
    if (!out) return -2;
    std::unique_ptr<hpg_mlp> m(new hpg_mlp());
    try {
        ck(hipGetDevice(&m->dev), "hipGetDevice");
        resolve_scratch(m->dev);
        ck(hipStreamCreate(&m->stream), "hipStreamCreate");
        for (float** p : {&m->master, &m->wq, &m->m1, &m->m2, &m->grad}) ck(hipMalloc(p, NPARAM * 4), "hipMalloc");
        ck(hipMalloc(&m->lsum, sizeof(double)), "hipMalloc");
        ck(hipMemsetAsync(m->m1, 0, NPARAM * 4, m->stream), "memset");
        ck(hipMemsetAsync(m->m2, 0, NPARAM * 4, m->stream), "memset");
        // He-style uniform init from a fixed LCG, biases zero
        std::vector<float> w(NPARAM, 0.f);
        unsigned long long st = 0x9E3779B97F4A7C15ull ^ seed;
        auto rnd = [&]() {
            st = st * 6364136223846793005ull + 1442695040888963407ull;
            return ((st >> 40) & 0xFFFFFF) / 16777216.0f * 2.f - 1.f;
        };
        const int fan[4] = {MI, MH, MH, MH}, offs[4] = {O_W1, O_W2, O_W3, O_W4}, nout[4] = {MH, MH, MH, MO};
        for (int L = 0; L < 4; ++L) {
            const float a = std::sqrt(6.f / fan[L]) * (L == 3 ? 0.1f : 1.f);
            for (int k = 0; k < fan[L] * nout[L]; ++k) w[offs[L] + k] = a * rnd();
        }
        quantise(m.get(), w);
    } catch (const std::exception&) {
        return -1;
    }
    *out = m.release();
    return 0;
}

int hpg_mlp_destroy(hpg_mlp* m) {
    delete m;
    return 0;
}

int hpg_mlp_num_params(void) { return NPARAM; }

int hpg_mlp_get_weights(hpg_mlp* m, float* w) {
    if (!m || !w) return -2;
    try {
        ck(hipMemcpyAsync(w, m->master, NPARAM * 4, hipMemcpyDeviceToHost, m->stream), "D2H");
        ck(hipStreamSynchronize(m->stream), "sync");
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

int hpg_mlp_set_weights(hpg_mlp* m, const float* w) {
    if (!m || !w) return -2;
    try {
        quantise(m, std::vector<float>(w, w + NPARAM));
        m->step = 0;
        ck(hipMemsetAsync(m->m1, 0, NPARAM * 4, m->stream), "memset");
        ck(hipMemsetAsync(m->m2, 0, NPARAM * 4, m->stream), "memset");
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

// MFMA bf16 16x16x16 lane-layout probe (test support; A, B 16x16 row-major, out 64x4)
int hpg_selftest_mfma_bf16(const float* A, const float* B, float* out) {
    if (!A || !B || !out) return -2;
    float *dA = nullptr, *dB = nullptr, *dO = nullptr;
    if (hipMalloc(&dA, 256 * 4) != hipSuccess || hipMalloc(&dB, 256 * 4) != hipSuccess ||
        hipMalloc(&dO, 256 * 4) != hipSuccess) {
        hipFree(dA); hipFree(dB);
        return -1;
    }
    hipMemcpy(dA, A, 256 * 4, hipMemcpyHostToDevice);
    hipMemcpy(dB, B, 256 * 4, hipMemcpyHostToDevice);
    hipLaunchKernelGGL(k_mfma_probe_bf16, dim3(1), dim3(64), 0, 0, dA, dB, dO);
    const hipError_t e = hipMemcpy(out, dO, 256 * 4, hipMemcpyDeviceToHost);
    hipFree(dA); hipFree(dB); hipFree(dO);
    return e == hipSuccess ? 0 : -1;
}

int hpg_mlp_forward(hpg_mlp* m, const float* X, int n, float* Y) {
    if (!m || !X || !Y || n < 0) return -2;
    try {
        ensure_n(m, n);
        send_batch(m, X, nullptr, n);
        mlp_forward_device(m, m->X, n, m->Y, m->stream);
        const HostSeg seg{Y, m->Y, (size_t)n * MO * 4};
        copy_to_host(m->stream, &seg, 1);
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

// loss (mean square over samples and outputs) and its gradient for one batch, no update
int hpg_mlp_loss_grad(hpg_mlp* m, const float* X, const float* T, int n, float* loss, float* grad) {
    if (!m || !X || !T || n <= 0) return -2;
    try {
        ensure_n(m, n);
        const int nb = train_blocks(n);
        ensure_blocks(m, nb);
        send_batch(m, X, T, n);
        enqueue_loss_grad(m, m->X, m->T, n, m->partial, m->lossp, m->grad);
        std::vector<double> lp(nb);
        ck(hipMemcpyAsync(lp.data(), m->lossp, nb * 8, hipMemcpyDeviceToHost, m->stream), "D2H");
        if (grad) ck(hipMemcpyAsync(grad, m->grad, NPARAM * 4, hipMemcpyDeviceToHost, m->stream), "D2H");
        ck(hipStreamSynchronize(m->stream), "sync");
        double s = 0.0;
        for (double v : lp) s += v;
        if (loss) *loss = (float)(s / ((double)n * MO));
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

// Allocation-free form of hpg_mlp_loss_grad on device buffers: X (n x 11), T (n x 3),
// loss (1 float) and grad (NPARAM floats) are device pointers of the caller; the
// block partials live in the library's static scratch array.  Same kernels and
// summation order as hpg_mlp_loss_grad, so loss and gradient are bitwise equal.
int hpg_mlp_loss_grad_noalloc(hpg_mlp* m, const float* X, const float* T, int n, float* loss, float* grad) {
    if (!m || !X || !T || !loss || !grad || n <= 0) return -2;
    if ((n + 63) / 64 > NOALLOC_MAX_BLOCKS) {
        m->err = "hpg_mlp_loss_grad_noalloc: n exceeds the scratch capacity of " +
                 std::to_string(HPG_MLP_NOALLOC_MAX_SAMPLES) + " samples";
        return -2;
    }
    try {
        float* sp = (m->dev >= 0 && m->dev < MAX_DEVICES) ? g_scratch[m->dev] : nullptr;
        if (!sp) throw std::runtime_error("scratch address not resolved for this device");
        const int nb = train_blocks(n);
        double* lossp = reinterpret_cast<double*>(sp + ((size_t)nb * NPARAM + 1) / 2 * 2);
        enqueue_loss_grad(m, X, T, n, sp, lossp, grad);
        hipLaunchKernelGGL(k_mlp_loss_sum, dim3(1), dim3(64), 0, m->stream, nb, lossp, n * MO, loss);
        ck(hipGetLastError(), "loss_grad_noalloc launch");
        ck(hipStreamSynchronize(m->stream), "sync");
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

// Adam training: `epochs` passes over (X, T) in mini-batches of `batch` samples
// (taken in order), learning rate lr; returns the mean loss of the last epoch
int hpg_mlp_train(hpg_mlp* m, const float* X, const float* T, int n, int epochs, int batch, float lr, float* last) {
    if (!m || !X || !T || n <= 0 || batch <= 0 || epochs <= 0) return -2;
    try {
        ensure_n(m, n);
        batch = ((batch + 63) / 64) * 64;
        ensure_blocks(m, train_blocks(std::min(batch, n)));
        send_batch(m, X, T, n);
        double lsum = 0.0;
        ck(hipMemcpyAsync(m->lsum, &lsum, sizeof(double), hipMemcpyHostToDevice, m->stream), "H2D");
        for (int ep = 0; ep < epochs; ++ep) {
            for (int b0 = 0; b0 < n; b0 += batch) {
                const int nb_s = std::min(batch, n - b0), nb = train_blocks(nb_s);
                ++m->step;
                const float bc1 = 1.f - std::pow(0.9f, (float)m->step), bc2 = 1.f - std::pow(0.999f, (float)m->step);
                hipLaunchKernelGGL(k_mlp_train_mfma, dim3(nb), dim3(256), 0, m->stream, nb_s, nb_s * MO,
                                   m->X + (size_t)b0 * MI, m->T + (size_t)b0 * MO, m->wq, m->partial, m->lossp);
                // the last epoch's loss accumulates on the device: nothing waits between steps
                hipLaunchKernelGGL(k_mlp_reduce_adam, dim3((NPARAM + 63) / 64), dim3(256), 0, m->stream, nb,
                                   m->partial, m->grad, m->master, m->wq, m->m1, m->m2, lr, bc1, bc2, 1, m->lossp,
                                   ep == epochs - 1 ? m->lsum : nullptr);
            }
            ck(hipGetLastError(), "train launch");
        }
        ck(hipMemcpyAsync(&lsum, m->lsum, sizeof(double), hipMemcpyDeviceToHost, m->stream), "D2H");
        ck(hipStreamSynchronize(m->stream), "sync");
        if (last) *last = (float)(lsum / ((double)n * MO));
    } catch (const std::exception& e) { m->err = e.what(); return -1; }
    return 0;
}

}  // extern "C"
