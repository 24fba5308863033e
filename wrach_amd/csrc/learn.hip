// The learned warm start's network on gfx950: 64 -> 128 -> 128 -> 2 with
// SiLU, bf16 weights and activations into v_mfma_f32_16x16x32_bf16 with f32
// accumulation; inference, the training rows (forward + backward through the
// layers), the weight gradients and Adam.  No
// counterpart in the reference, whose separation is one Gauss-Seidel sweep
// per cell (shaders/physics/src/particles.rs:62-93); the network predicts
// the displacement that the plain separation passes produce, and those
// passes then start from its guess.
//
// MFMA layout (v_mfma_f32_16x16x32_bf16, wave64): D[i][j] = sum_k A[i][k]
// B[k][j] + C[i][j] over a 16 x 32 A, 32 x 16 B and 16 x 16 C.  Lane l
// supplies row l % 16 of A and column l % 16 of B, the 8 k entries of lane
// group g = l / 16 (k = 8g .. 8g + 7), and holds D[4g + r][l % 16],
// r = 0..3.
//
// The network runs transposed: a layer computes out^T = W^T . in^T, so the
// particles are the B/D columns.  Layer 1's B operand is then 16 bytes of a
// particle's feature row.  Layer 1's D registers hold, per lane, outputs
// 16t + 4g + r of one particle; two consecutive tiles give lane group g the
// 8 features {32s + 4g + 0..3, 32s + 16 + 4g + 0..3} -- exactly a B operand
// of layer 2's k-step s if the k order of that step is permuted the same way
// in A.  The weights are packed with that permutation (kmap below), so the
// layers chain in registers with no transpose.
#include <hip/hip_runtime.h>

#include "learn.h"

namespace wrach {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t lane_id() {
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// f32 -> bf16 bits, round to nearest even (NaN kept quiet).
__host__ __device__ __forceinline__ uint16_t bf16_bits(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ float bf16_float(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Feature of the permuted k order: slot e of lane group g in k-step s.
__host__ __device__ constexpr uint32_t kmap(uint32_t s, uint32_t g, uint32_t e) {
    return 32u * s + (e < 4u ? 4u * g + e : 16u + 4u * g + (e - 4u));
}

// SiLU and its derivative, in f32, from the hardware exp2 and reciprocal
// (v_exp_f32, v_rcp_f32: about 1 ulp each; the network is trained and run
// with the same function).
__device__ __forceinline__ float sigmoid(float z) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * 1.4426950408889634f));
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }
__device__ __forceinline__ float silu_grad(float z) {
    const float s = sigmoid(z);
    return s * (1.0f + z * (1.0f - s));
}

// Eight f32 to bf16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ bf16x8 pack8(const float (&v)[8]) {
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (__bf16)v[e];
    return r;
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Inference of NC column tiles (16 particles each) by one wavefront with few
// live registers: layer 1 a pair of output tiles at a time (one k-step of
// layer 2's B operands, its k order permuted), layer 2 one output tile at a
// time, folded straight into layer 3 (128 -> 2, on the vector ALUs: each
// lane group sums its 32 outputs, then the four groups are added).  xb[c][s]:
// layer-1 B operands (feature rows); frag: the packed fragments (global or
// LDS).  The same arithmetic in the same order as a training row's.
template <int NC, typename FragPtr>
__device__ __forceinline__ void mlp_infer(const bf16x8 (&xb)[NC][2], FragPtr frag, const float *b1,
                                          const float *b2, const float *w3, const float *b3,
                                          float (&y)[NC][2]) {
    const uint32_t l = lane_id(), g = l >> 4;
    bf16x8 h1[NC][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        f32x4 z[2][NC];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int t = 2 * s + h;
            f32x4 bias;
#pragma unroll
            for (int r = 0; r < 4; ++r) bias[r] = b1[16 * t + 4 * g + r];
#pragma unroll
            for (int c = 0; c < NC; ++c) z[h][c] = bias;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const bf16x8 a = frag[(kFragW1 + t * 2 + k) * 64 + l];
#pragma unroll
                for (int c = 0; c < NC; ++c) z[h][c] = mfma(a, xb[c][k], z[h][c]);
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float v[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = silu(z[0][c][r]);
                v[4 + r] = silu(z[1][c][r]);
            }
            h1[c][s] = pack8(v);
        }
    }
    float y0[NC], y1[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) y0[c] = y1[c] = 0.0f;
    // One output tile at a time (not unrolled): its 4 fragments and 8 W3
    // entries are the only weights live, which keeps the kernel at 4
    // wavefronts per SIMD without spilling.
#pragma unroll 1
    for (int t = 0; t < 8; ++t) {
        f32x4 bias;
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[r] = b2[16 * t + 4 * g + r];
        f32x4 z[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) z[c] = bias;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bf16x8 a = frag[(kFragW2F + t * 4 + k) * 64 + l];
#pragma unroll
            for (int c = 0; c < NC; ++c) z[c] = mfma(a, h1[c][k], z[c]);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t o = 16 * t + 4 * g + r;
                const float a2 = silu(z[c][r]);
                y0[c] = fmaf(a2, w3[2 * o], y0[c]);
                y1[c] = fmaf(a2, w3[2 * o + 1], y1[c]);
            }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        float u0 = y0[c], u1 = y1[c];
        u0 += __shfl_xor(u0, 16, 64);
        u1 += __shfl_xor(u1, 16, 64);
        u0 += __shfl_xor(u0, 32, 64);
        u1 += __shfl_xor(u1, 32, 64);
        y[c][0] = u0 + b3[0];
        y[c][1] = u1 + b3[1];
    }
}

// Layer-1 B operands of particles row0 + 16c + l % 16 (rows >= n: zeros).
template <int NC>
__device__ __forceinline__ void load_rows(const uint16_t *feat, const uint32_t *sel, uint32_t row0,
                                          uint32_t n, bf16x8 (&xb)[NC][2]) {
    const uint32_t l = lane_id(), g = l >> 4;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const uint32_t p = row0 + 16 * c + (l & 15);
        const uint32_t row = p < n ? (sel ? sel[p] : p) : 0u;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (p < n) {
                xb[c][s] = *reinterpret_cast<const bf16x8 *>(feat + (size_t)row * kFeat + 32 * s + 8 * g);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) xb[c][s][e] = __builtin_bit_cast(__bf16, (uint16_t)0);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Inference: persistent blocks of 4 wavefronts, weights staged in LDS once
// per block, 32 particles per wavefront per step.

constexpr int kInferBlock = 512;
constexpr int kInferCols = 2;  // 16-particle column tiles per wavefront step

__global__ __launch_bounds__(kInferBlock) __attribute__((amdgpu_waves_per_eu(4))) void learn_infer_kernel(MlpWeights w, InferArgs a) {
    __shared__ bf16x8 s_frag[(kW1Frags + kW2Frags) * 64];  // 48 KiB
    __shared__ __align__(16) float s_b1[kHid];
    __shared__ __align__(16) float s_b2[kHid];
    __shared__ __align__(16) float s_w3[kHid * kOutDim];
    __shared__ float s_b3[kOutDim];
    const bf16x8 *gfrag = reinterpret_cast<const bf16x8 *>(w.frag);
    for (uint32_t i = threadIdx.x; i < (kW1Frags + kW2Frags) * 64; i += kInferBlock) s_frag[i] = gfrag[i];
    for (uint32_t i = threadIdx.x; i < (uint32_t)kHid; i += kInferBlock) {
        s_b1[i] = w.params[kOffB1 + i];
        s_b2[i] = w.params[kOffB2 + i];
    }
    for (uint32_t i = threadIdx.x; i < (uint32_t)(kHid * kOutDim); i += kInferBlock) s_w3[i] = w.w3[i];
    if (threadIdx.x < (uint32_t)kOutDim) s_b3[threadIdx.x] = w.params[kOffB3 + threadIdx.x];
    __syncthreads();
    const uint32_t l = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t per_step = 16 * kInferCols;
    for (uint32_t row0 = (blockIdx.x * (kInferBlock / 64) + wave) * per_step; row0 < a.n;
         row0 += gridDim.x * (kInferBlock / 64) * per_step) {
        bf16x8 xb[kInferCols][2];
        load_rows<kInferCols>(a.feat, nullptr, row0, a.n, xb);
        float y[kInferCols][2];
        // The weights stay in LDS: an offset the optimiser cannot see
        // through keeps it from hoisting all 48 fragments into registers for
        // the whole loop (192 VGPRs, one wavefront per SIMD).  An offset, not
        // the addresses: those would lose their address space and turn every
        // LDS read into a flat load (111 us for 1M rows).
        uint32_t z = 0;
        asm volatile("" : "+v"(z));
        mlp_infer<kInferCols>(xb, s_frag + z, s_b1 + z, s_b2 + z, s_w3 + z, s_b3, y);
        if (l < 16) {
#pragma unroll
            for (int c = 0; c < kInferCols; ++c) {
                const uint32_t p = row0 + 16 * c + l;
                if (p < a.n) {
                    if (a.y_out) a.y_out[p] = make_float2(y[c][0], y[c][1]);
                    if (a.pout) {
                        const float2 q = a.pin[p];
                        const float dx = fminf(fmaxf(y[c][0], -kMaxWarm), kMaxWarm);
                        const float dy = fminf(fmaxf(y[c][1], -kMaxWarm), kMaxWarm);
                        a.pout[p] = make_float2(q.x + dx, q.y + dy);
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// A training step is three launches, none of them near a rate of the chip at
// 8,192 rows (1.1 GFLOP, 12 MB): each is a chain of latencies, so each
// spreads its chain over as many wavefronts as it can.
//
// learn_rows_kernel     16 batch rows a block of 4 wavefronts, wavefront w
//                       the output tiles 2w and 2w + 1 of every layer:
//                       forward, output error and backward.  All weights a
//                       wavefront needs (20 fragments) are on their way to
//                       registers before the first product; the layers'
//                       operands pass through LDS, a wavefront's two tiles
//                       being exactly one k-step of the next layer.
// learn_sums_kernel     the weight gradients, MFMA products over chunks of
//                       the batch, one 16 x 16 tile a wavefront, and beside
//                       them the column sums for b1, b2, W3, b3 and the loss.
// learn_update_kernel   sums the chunks in order and applies Adam and the
//                       packing of the new weights to each entry.
//
// Every sum keeps a fixed order (deterministic, and the same however the
// work is spread).  With one wavefront a row tile, two product launches, a
// reduction, Adam and the packing apart, a step of 8,192 rows took 26 + 2 * 6
// + 20 + 5 + 4 us and 75 us with the gaps; now 12.8 + 9.1 + 4.7 and 41 us.
// (One kernel for the rows and their products, partial gradients per block:
// 22 us, and sums in another order.)

// The activations and gradients the weight gradients read: for every 16
// batch rows a block of [feature][16 rows], so that a block of the rows
// kernel writes whole lines and an operand's 8 rows of a feature are 16
// bytes.
__device__ __forceinline__ size_t tiled(uint32_t features, uint32_t f, uint32_t row) {
    return ((size_t)(row >> 4) * features + f) * 16 + (row & 15);
}

__global__ __launch_bounds__(256, 2) void learn_rows_kernel(MlpWeights w, TrainArgs a) {
    __shared__ bf16x8 s_h1[4][64], s_d2[4][64];
    __shared__ f32x4 s_a2[8][64];
    const uint32_t l = lane_id(), g = l >> 4, col = l & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t p = blockIdx.x * 16 + col;
    const uint32_t row = a.sel[p];
    const bf16x8 *frag = reinterpret_cast<const bf16x8 *>(w.frag) + l;
    // Loads, all in flight together: this wavefront's weights, the rows.
    bf16x8 w1[2][2], w2f[2][4], w2b[2][4], xb[2];
    f32x4 bias1[2], bias2[2], w3a[8], w3b[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t t = 2 * wave + h;
#pragma unroll
        for (int s = 0; s < 2; ++s) w1[h][s] = frag[(kFragW1 + t * 2 + s) * 64];
#pragma unroll
        for (int s = 0; s < 4; ++s) w2f[h][s] = frag[(kFragW2F + t * 4 + s) * 64];
#pragma unroll
        for (int s = 0; s < 4; ++s) w2b[h][s] = frag[(kFragW2B + t * 4 + s) * 64];
        bias1[h] = *reinterpret_cast<const f32x4 *>(w.params + kOffB1 + 16 * t + 4 * g);
        bias2[h] = *reinterpret_cast<const f32x4 *>(w.params + kOffB2 + 16 * t + 4 * g);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {  // W3's rows of this lane group: outputs 16t + 4g ..
        w3a[t] = *reinterpret_cast<const f32x4 *>(w.w3 + 2 * (16 * t + 4 * g));
        w3b[t] = *reinterpret_cast<const f32x4 *>(w.w3 + 2 * (16 * t + 4 * g) + 4);
    }
    const float b30 = w.params[kOffB3], b31 = w.params[kOffB3 + 1];
#pragma unroll
    for (int s = 0; s < 2; ++s)
        xb[s] = *reinterpret_cast<const bf16x8 *>(a.feat + (size_t)row * kFeat + 32 * s + 8 * g);
    const float2 tg = a.target[row];

    f32x4 z1[2], z2[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        z1[h] = bias1[h];
#pragma unroll
        for (int s = 0; s < 2; ++s) z1[h] = mfma(w1[h][s], xb[s], z1[h]);
    }
    float v[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[r] = silu(z1[0][r]);
        v[4 + r] = silu(z1[1][r]);
    }
    const bf16x8 h1 = pack8(v);
    s_h1[wave][l] = h1;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        z2[h] = bias2[h];
#pragma unroll
        for (int s = 0; s < 4; ++s) z2[h] = mfma(w2f[h][s], s_h1[s][l], z2[h]);
    }
    f32x4 a2[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int r = 0; r < 4; ++r) a2[h][r] = silu(z2[h][r]);
        s_a2[2 * wave + h][l] = a2[h];
    }
    __syncthreads();
    // Layer 3, in every wavefront: each lane group sums its 32 outputs, then
    // the four groups are added.
    float y0 = 0.0f, y1 = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const f32x4 h = s_a2[t][l];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            y0 = fmaf(h[r], r < 2 ? w3a[t][2 * (r & 1)] : w3b[t][2 * (r & 1)], y0);
            y1 = fmaf(h[r], r < 2 ? w3a[t][2 * (r & 1) + 1] : w3b[t][2 * (r & 1) + 1], y1);
        }
    }
    y0 += __shfl_xor(y0, 16, 64);
    y1 += __shfl_xor(y1, 16, 64);
    y0 += __shfl_xor(y0, 32, 64);
    y1 += __shfl_xor(y1, 32, 64);
    const float e0 = (y0 + b30) - tg.x, e1 = (y1 + b31) - tg.y;
    const float dy0 = e0 * a.inv_bsz, dy1 = e1 * a.inv_bsz;
    // dL/dz2 = (W3 . dy) * SiLU'(z2) of this wavefront's tiles.
    f32x4 wa[2] = {w3a[0], w3a[1]}, wb[2] = {w3b[0], w3b[1]};
#pragma unroll
    for (int t = 2; t < 8; ++t) {
        const bool own = (uint32_t)(t >> 1) == wave;
        wa[t & 1] = own ? w3a[t] : wa[t & 1];
        wb[t & 1] = own ? w3b[t] : wb[t & 1];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float u0 = r < 2 ? wa[h][2 * (r & 1)] : wb[h][2 * (r & 1)];
            const float u1 = r < 2 ? wa[h][2 * (r & 1) + 1] : wb[h][2 * (r & 1) + 1];
            float da = u0 * dy0;
            da = da + u1 * dy1;
            v[4 * h + r] = da * silu_grad(z2[h][r]);
        }
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    const bf16x8 d2 = pack8(v);
    s_d2[wave][l] = d2;
    __syncthreads();
    // dL/da1 = W2 . dz2 (rows = layer-2 inputs), then dL/dz1.
    f32x4 acc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        acc[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[h] = mfma(w2b[h][s], s_d2[s][l], acc[h]);
    }
    // What the weight gradients read.  (Turned in LDS to store 16 bytes a
    // lane instead of 2: no faster, 12.8 us either way.)
    const u16x8 h1b = __builtin_bit_cast(u16x8, h1), d2b = __builtin_bit_cast(u16x8, d2);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const size_t at = tiled(kHid, 16 * (2 * wave + h) + 4 * g + r, p);
            a.a2t[at] = a2[h][r];
            a.dz2t[at] = d2b[4 * h + r];
            a.a1t[at] = h1b[4 * h + r];
            a.dz1t[at] = bf16_bits(acc[h][r] * silu_grad(z1[h][r]));
        }
    const u16x8 xw = __builtin_bit_cast(u16x8, wave < 2 ? xb[0] : xb[1]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        a.xt[tiled(kFeat, 32 * (wave >> 1) + 8 * g + 4 * (wave & 1) + e, p)] = wave & 1 ? xw[4 + e] : xw[e];
    if (wave == 0) {
        // Squared error of the tile (lane group 0 holds each row once).
        float se = g == 0 ? e0 * e0 + e1 * e1 : 0.0f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o, 64);
        if (l == 0) a.sqerr[blockIdx.x] = se;
        if (g == 0) {
            a.dyt[p] = dy0;
            a.dyt[a.bsz + p] = dy1;
        }
    }
}

// chunk c of in^T . dz: sum over its rows k of A[m][k] B[n][k], a 32 x 32
// output tile per block, one 16 x 16 MFMA tile per wavefront.
__device__ __forceinline__ void weight_tile(const uint16_t *A, uint32_t fa, const uint16_t *B, uint32_t m32,
                                            uint32_t n32, uint32_t first, uint32_t rows, float *out) {
    const uint32_t l = lane_id(), g = l >> 4, wave = threadIdx.x >> 6;
    const uint32_t m0 = m32 * 32 + (wave & 1) * 16, n0 = n32 * 32 + (wave >> 1) * 16;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t *ar = A + tiled(fa, m0 + (l & 15), first + 8 * g);
    const uint16_t *br = B + tiled(kHid, n0 + (l & 15), first + 8 * g);
    uint32_t k = 0;
    for (; k + 128 <= rows; k += 128) {  // four steps' operands in flight together
        bf16x8 x[4], y[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            x[s] = *reinterpret_cast<const bf16x8 *>(ar + (size_t)(k + 32 * s) * fa);
            y[s] = *reinterpret_cast<const bf16x8 *>(br + (size_t)(k + 32 * s) * kHid);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = mfma(x[s], y[s], acc);
    }
    for (; k < rows; k += 32)
        acc = mfma(*reinterpret_cast<const bf16x8 *>(ar + (size_t)k * fa),
                   *reinterpret_cast<const bf16x8 *>(br + (size_t)k * kHid), acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(size_t)(m0 + 4 * g + r) * kHid + n0 + (l & 15)] = acc[r];
}

// Sums of 256 per-thread partials, N of them at once, in a fixed order
// (halves added to halves); thread 0 has them.
template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N], float (*s)[256]) {
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < N; ++q) s[q][t] = v[q];
    __syncthreads();
    if (t < 128)
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = s[q][t] + s[q][t + 128];
    __syncthreads();
    if (t < 128)
#pragma unroll
        for (int q = 0; q < N; ++q) s[q][t] = v[q];
    __syncthreads();
    if (t < 64) {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            v[q] += s[q][t + 64];
#pragma unroll
            for (int h = 32; h > 0; h >>= 1) v[q] += __shfl_down(v[q], h, 64);
        }
    }
}

// Blocks: first the column sums, the longest, four columns a block (whole
// lines of the tiled arrays): b1, b2, W3's rows, then b3 and the loss; after
// them the chunks' tiles of dW1 (2 x 4) and dW2 (4 x 4).
constexpr uint32_t kColBlocks = 3 * kHid / 4 + 1;

__global__ __launch_bounds__(256) void learn_sums_kernel(TrainArgs a) {
    __shared__ float s[8][256];
    uint32_t blk = blockIdx.x;
    if (blk >= kColBlocks) {
        blk -= kColBlocks;
        // Blocks go to the 8 XCDs in turn: a chunk's 24 tiles on one of them,
        // whose L2 then fetches its rows once.
        const uint32_t c = blk % 8 + blk / 192 * 8, q = blk / 8 % 24, first = c * a.kc;
        if (c >= a.chunks) return;
        const uint32_t rows = min(a.kc, a.bsz - first);  // the last chunk may be shorter
        float *part = a.part + (size_t)c * kWeights;
        if (q < 8) weight_tile(a.xt, kFeat, a.dz1t, q / 4, q % 4, first, rows, part);
        else weight_tile(a.a1t, kHid, a.dz2t, (q - 8) / 4, q % 4, first, rows, part + kFeat * kHid);
        return;
    }
    float *cols = a.cols;
    if (blk < 2u * kHid / 4) {  // b1, b2
        const uint32_t o = blk % (kHid / 4) * 4;
        const uint16_t *d = blk < (uint32_t)kHid / 4 ? a.dz1t : a.dz2t;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
        for (uint32_t p = threadIdx.x; p < a.bsz; p += 256) {
            const uint16_t *e = d + tiled(kHid, o, p);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += bf16_float(e[16 * q]);
        }
        block_sums<4>(v, s);
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < 4; ++q) cols[(blk < (uint32_t)kHid / 4 ? 0 : kHid) + o + q] = v[q];
    } else if (blk < 3u * kHid / 4) {  // W3 rows o .. o + 3
        const uint32_t o = (blk - 2 * kHid / 4) * 4;
        float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
        for (uint32_t p = threadIdx.x; p < a.bsz; p += 256) {
            const float *e = a.a2t + tiled(kHid, o, p);
            const float d0 = a.dyt[p], d1 = a.dyt[a.bsz + p];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float h = e[16 * q];
                v[2 * q] = fmaf(h, d0, v[2 * q]);
                v[2 * q + 1] = fmaf(h, d1, v[2 * q + 1]);
            }
        }
        block_sums<8>(v, s);
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < 8; ++q) cols[2 * kHid + 2 * o + q] = v[q];
    } else {  // b3 and the squared error
        float v[3] = {0.0f, 0.0f, 0.0f};
        for (uint32_t p = threadIdx.x; p < a.bsz; p += 256) {
            v[0] += a.dyt[p];
            v[1] += a.dyt[a.bsz + p];
        }
        for (uint32_t t = threadIdx.x; t < a.bsz / 16; t += 256) v[2] += a.sqerr[t];
        block_sums<3>(v, s);
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < 3; ++q) cols[4 * kHid + q] = v[q];
    }
}

// Where entry (k, o) of a weight matrix lies in its fragments: rows of the A
// operand are `row`, its k-step entries `k`; natural or permuted k order
// (the inverse of kmap).
__device__ __forceinline__ uint32_t frag_index(uint32_t first, uint32_t steps, uint32_t row, uint32_t k,
                                               bool permuted) {
    const uint32_t s = k / 32, q = k % 32;
    const uint32_t g = permuted ? (q % 16) / 4 : q / 8, e = permuted ? q % 4 + (q < 16 ? 0u : 4u) : q % 8;
    return (first + row / 16 * steps + s) * kFragElems + (16 * g + row % 16) * 8 + e;
}

// One entry a thread (64-thread blocks, so that the 25,090 reach every CU):
// its gradient -- the chunks' sums in order, or the column sum -- and then
// that gradient out (u.grad), or Adam (Kingma & Ba, 2015) on the master
// vector, each step a rounded f32 operation in this order (no contraction),
// and the packing of the new value.
__global__ __launch_bounds__(64) void learn_update_kernel(UpdateArgs u) {
    const uint32_t i = blockIdx.x * 64 + threadIdx.x;
    if (i >= kParams) {
        if (i == kParams && u.loss) *u.loss = u.cols[4 * kHid + 2] * u.loss_scale;
        return;
    }
    float gr;
    if (u.given) {
        gr = u.given[i];
    } else if (i < kOffB1 || (i >= kOffW2 && i < kOffB2)) {
        const float *q = u.part + (i < kOffB1 ? i : i - kOffW2 + kFeat * kHid);
        gr = 0.0f;
#pragma unroll 32
        for (uint32_t c = 0; c < u.chunks; ++c) gr += q[(size_t)c * kWeights];
    } else {
        gr = u.cols[i < kOffW2 ? i - kOffB1 : i < kOffW3 ? i - kOffB2 + kHid : i - kOffW3 + 2 * kHid];
    }
    if (u.grad) {
        u.grad[i] = gr;
        return;
    }
    float m = u.beta1 * u.m[i];
    m = m + (1.0f - u.beta1) * gr;
    float q = u.beta2 * u.v[i];
    q = q + (1.0f - u.beta2) * (gr * gr);
    u.m[i] = m;
    u.v[i] = q;
    const float mh = m * u.c1;
    const float vh = q * u.c2;
    const float step = u.lr * mh / (sqrtf(vh) + u.eps);
    const float x = u.params[i] - step;
    u.params[i] = x;
    const uint16_t h = bf16_bits(x);
    if (i < kOffB1) {
        const uint32_t k = i / kHid, o = i % kHid;
        u.frag[frag_index(kFragW1, 2, o, k, false)] = h;
    } else if (i >= kOffW2 && i < kOffB2) {
        const uint32_t k = (i - kOffW2) / kHid, o = (i - kOffW2) % kHid;
        u.frag[frag_index(kFragW2F, 4, o, k, true)] = h;
        u.frag[frag_index(kFragW2B, 4, k, o, true)] = h;
    } else if (i >= kOffW3 && i < kOffB3) {
        u.w3[i - kOffW3] = bf16_float(h);
    }
}

// Fragments and the rounded W3 from the master vector: one thread per
// fragment entry (kFrags * 512), the first 256 also round W3.
__global__ __launch_bounds__(256) void learn_pack_kernel(const float *params, uint16_t *frag, float *w3) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < (uint32_t)(kHid * kOutDim)) w3[i] = bf16_float(bf16_bits(params[kOffW3 + i]));
    if (i >= kFrags * kFragElems) return;
    const uint32_t f = i / kFragElems, l = (i / 8) % 64, e = i % 8, g = l / 16, row = l % 16;
    float v;
    if (f < kFragW2F) {  // W1^T: rows = outputs, k = inputs (natural order)
        const uint32_t t = (f - kFragW1) / 2, s = (f - kFragW1) % 2;
        v = params[kOffW1 + (32 * s + 8 * g + e) * kHid + 16 * t + row];
    } else if (f < kFragW2B) {  // W2^T: rows = outputs, k = inputs (permuted)
        const uint32_t t = (f - kFragW2F) / 4, s = (f - kFragW2F) % 4;
        v = params[kOffW2 + kmap(s, g, e) * kHid + 16 * t + row];
    } else {  // W2: rows = inputs, k = outputs (permuted)
        const uint32_t t = (f - kFragW2B) / 4, s = (f - kFragW2B) % 4;
        v = params[kOffW2 + (16 * t + row) * kHid + kmap(s, g, e)];
    }
    frag[i] = bf16_bits(v);
}

__global__ __launch_bounds__(256) void learn_target_kernel(const float2 *pk, const float2 *p0, float2 *target,
                                                           uint32_t row0, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float2 a = pk[i], b = p0[i];
    target[row0 + i] = make_float2(a.x - b.x, a.y - b.y);
}

}  // namespace

uint32_t resident_blocks_infer() {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, learn_infer_kernel, kInferBlock, 0) != hipSuccess)
        return 0;
    return (uint32_t)(cus * (per > 0 ? per : 1));
}

hipError_t launch_learn_infer(const MlpWeights &w, const InferArgs &a, hipStream_t stream) {
    if (a.n == 0) return hipSuccess;
    static uint32_t resident = 0;
    if (!resident) resident = resident_blocks_infer();
    const uint32_t steps = (a.n + 16 * kInferCols - 1) / (16 * kInferCols);
    uint32_t grid = (steps + kInferBlock / 64 - 1) / (kInferBlock / 64);
    if (resident && grid > resident) grid = resident;
    hipLaunchKernelGGL(learn_infer_kernel, dim3(grid), dim3(kInferBlock), 0, stream, w, a);
    return hipGetLastError();
}

hipError_t launch_learn_grad(const MlpWeights &w, const TrainArgs &a, hipStream_t stream) {
    if (a.bsz == 0 || a.bsz % 64 || a.kc == 0 || a.kc % 32 || a.chunks == 0 ||
        (size_t)a.kc * (a.chunks - 1) >= a.bsz || (size_t)a.kc * a.chunks < a.bsz)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(learn_rows_kernel, dim3(a.bsz / 16), dim3(256), 0, stream, w, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(learn_sums_kernel, dim3((a.chunks + 7) / 8 * 8 * 24 + kColBlocks), dim3(256), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_learn_update(const UpdateArgs &u, hipStream_t stream) {
    if (!u.given && (!u.part || !u.cols || u.chunks == 0)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(learn_update_kernel, dim3((kParams + 64) / 64), dim3(64), 0, stream, u);
    return hipGetLastError();
}

hipError_t launch_learn_pack(const float *params, uint16_t *frag, float *w3, hipStream_t stream) {
    hipLaunchKernelGGL(learn_pack_kernel, dim3((kFrags * kFragElems + 255) / 256), dim3(256), 0, stream,
                       params, frag, w3);
    return hipGetLastError();
}

hipError_t launch_learn_target(const float2 *pk, const float2 *p0, float2 *target, uint32_t row0,
                               uint32_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(learn_target_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, pk, p0, target,
                       row0, n);
    return hipGetLastError();
}

}  // namespace wrach
