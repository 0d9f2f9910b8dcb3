// plis_mlp.hip -- the learned tau proposal on gfx950 matrix cores.
//
// MLP 12 -> 64 -> 64 -> 2 (GELU or ReLU), bfloat16 operands with fp32
// accumulation on v_mfma_f32_32x32x16_bf16.  One wavefront owns a tile of 64
// rows (subvolumes or training samples); activations are staged in LDS in
// both row- and column-major form so every MFMA fragment is a contiguous
// 16-byte LDS read.
//
// Parameter blob (fp32 master, shared with the host):
//   W1[16][64] | b1[64] | W2[64][64] | b2[64] | W3[64][2] | b3[2]
// (W[i][o] multiplies input i into output o; rows 12..15 of W1 stay zero).
// Packed bf16 copies for the MFMA B operand: Wt[o][i] (forward) and W[i][o]
// (backward), W3 padded to 32 outputs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plis_numerics.h"

namespace plis {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kNin = 16, kNh = 64, kNo = 2, kNoPad = 32;
constexpr int kPW1 = 0, kPB1 = kPW1 + kNin * kNh, kPW2 = kPB1 + kNh, kPB2 = kPW2 + kNh * kNh;
constexpr int kPW3 = kPB2 + kNh, kPB3 = kPW3 + kNh * kNo, kPTotal = kPB3 + kNo;  // 5378
// packed bf16 layout (element offsets)
constexpr int kQW1t = 0;                         // [64][16]
constexpr int kQW2t = kQW1t + kNh * kNin;        // [64][64]
constexpr int kQW3t = kQW2t + kNh * kNh;         // [32][64]
constexpr int kQW2 = kQW3t + kNoPad * kNh;       // [64][64]  W2[i][o]
constexpr int kQW3 = kQW2 + kNh * kNh;           // [64][32]  W3[i][o]
constexpr int kQTotal = kQW3 + kNh * kNoPad;
// LDS row strides (bf16 elements), padded against bank conflicts
constexpr int kLdX = 24, kLdH = 72;

struct MlpDev {
    const float* w32;        // fp32 master blob
    const __bf16* q;         // packed bf16
    const float* norm;       // fmu[12] fsig[12] y_mu y_sig
};

// Activations: ACT 0 = ReLU, 1 = GELU.  GELU(z) = z Phi(z) is evaluated as
//     max(z, 0) - |z| max(0, p(|z|)),  p(a) = 0.5 + a (C1 + a (C2 + a C3)),
// a cubic fitted minimax over the real line to the correction
// |z| Phi(-|z|) = relu(z) - GELU(z), with p(0) = 1/2 so that the slope at 0
// is GELU's 1/2: largest error 0.0058 against the erf form, 7 VALU
// instructions, no transcendental.
constexpr float kGeluC1 = -0.47735822f, kGeluC2 = 0.15120307f, kGeluC3 = -0.01585033f;

template <int ACT>
__device__ __forceinline__ float act_f(float z) {
    if constexpr (ACT == 0) {
        return fmaxf(z, 0.0f);
    } else {
        const float a = __builtin_fabsf(z);
        const float p = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(kGeluC3, a, kGeluC2), a, kGeluC1), a, 0.5f);
        return fmaxf(z, 0.0f) - a * fmaxf(p, 0.0f);
    }
}

// d act / dz (the backward pass keeps it from the forward pass)
template <int ACT>
__device__ __forceinline__ float act_d(float z) {
    if constexpr (ACT == 0) {
        return z > 0.0f ? 1.0f : 0.0f;
    } else {
        const float a = __builtin_fabsf(z);
        const float p = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(kGeluC3, a, kGeluC2), a, kGeluC1), a, 0.5f);
        const float dp = __builtin_fmaf(__builtin_fmaf(3.0f * kGeluC3, a, 2.0f * kGeluC2), a, kGeluC1);
        const float q = p > 0.0f ? __builtin_fmaf(a, dp, p) : 0.0f;
        return z > 0.0f ? 1.0f - q : q;
    }
}

// lane-layout of v_mfma_f32_32x32x16_bf16: A fragment = 8 consecutive k of
// row (l % 32) starting at k = 8*(l/32); B fragment = 8 consecutive k of
// column (l % 32); accumulator element i of lane l sits at
// row 8*(i/4) + 4*(l/32) + i%4, column l % 32.
__device__ __forceinline__ bf16x8 lds_frag(const __bf16* M, int ld, int row0, int k0,
                                           int l = threadIdx.x & 63) {
    return *reinterpret_cast<const bf16x8*>(M + (row0 + (l & 31)) * ld + k0 + 8 * (l >> 5));
}
__device__ __forceinline__ bf16x8 glb_frag(const __bf16* M, int ld, int row0, int k0,
                                           int l = threadIdx.x & 63) {
    return *reinterpret_cast<const bf16x8*>(M + (row0 + (l & 31)) * ld + k0 + 8 * (l >> 5));
}
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int acc_row(int i, int l = threadIdx.x & 63) { return 8 * (i >> 2) + 4 * (l >> 5) + (i & 3); }
__device__ __forceinline__ int acc_col(int l = threadIdx.x & 63) { return l & 31; }

// One training tile's staging: 39,680 bytes, so that four blocks share a CU.
// Row-major activations serve only the next layer of the forward pass; the
// backward pass stages its gradients in their place.
struct MlpLds {
    __bf16 xt[kNin * kLdH];    // standardised inputs, transposed [feature][row]
    __bf16 h1t[64 * kLdH];     // hidden activations, transposed [unit][row]
    union {
        __bf16 x[64 * kLdX];   // inputs [row][16] (until layer 1 is done)
        __bf16 h2t[64 * kLdH];
    };
    union {
        __bf16 h1[64 * kLdH];  // [row][unit] (until layer 2 is done)
        __bf16 dzt[64 * kLdH];
    };
    union {
        __bf16 h2[64 * kLdH];  // (until the output layer is done)
        __bf16 dz[64 * kLdH];
    };
    float out[64 * 2];
};
static_assert(4 * sizeof(MlpLds) <= 160 * 1024, "four blocks per CU");

// ---------------------------------------------------------------------------
// training: forward + backward over tiles of 64 samples, per-wave gradient
// partials (fixed summation order afterwards: deterministic)
// ---------------------------------------------------------------------------
struct TrainArgs {
    MlpDev m;
    const float* feats;      // [n][12]
    const float* ylog;       // [n] standardised log tau target
    const float* ycrit;      // [n] 0/1
    uint64_t n, n_inv;       // records; floor((2^64 - 1) / n)
    uint32_t batch;          // samples per step (multiple of 64)
    uint32_t step;           // selects the minibatch
    uint32_t seed_lo, seed_hi;
    int32_t full_pass;       // 1: use records 0..batch-1 in order (gradient checks)
    float* partial;          // [gridDim.x][kPTotal + 1] (last = loss sum)
};

// The 32x32 block (mb, nb) of in[64][K] . W, W given transposed as fragments.
template <int K>
__device__ __forceinline__ f32x16 mfma_block(const __bf16* in, int ldin, int mb, int l, const bf16x8 (&w)[K / 16]) {
    f32x16 c = {};
#pragma unroll
    for (int kb = 0; kb < K / 16; ++kb) c = mfma(lds_frag(in, ldin, mb * 32, kb * 16, l), w[kb], c);
    return c;
}

template <int K>
__device__ __forceinline__ void load_frags(const __bf16* wt, int nb, int l, bf16x8 (&w)[K / 16]) {
#pragma unroll
    for (int kb = 0; kb < K / 16; ++kb) w[kb] = glb_frag(wt, K, nb * 32, kb * 16, l);
}

// Four consecutive rows of a column at once (an accumulator holds them).
__device__ __forceinline__ void store4(__bf16* p, const bf16x4& v) { *reinterpret_cast<bf16x4*>(p) = v; }

// A hidden layer's block: bf16 activations (row-major and transposed); d
// keeps act'(z), rounded to bf16, for the backward pass of the same block.
template <int ACT>
__device__ __forceinline__ void activate_block(const f32x16& c, float bias, int mb, int nb, int l, __bf16* h, __bf16* ht,
                                               u32x8& d) {
    const int col = nb * 32 + acc_col(l);
    bf16x16 g;
    bf16x4 t;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = mb * 32 + acc_row(i, l);
        const float z = c[i] + bias;
        t[i & 3] = (__bf16)act_f<ACT>(z);
        h[row * kLdH + col] = t[i & 3];
        if ((i & 3) == 3) store4(ht + col * kLdH + row - 3, t);
        g[i] = (__bf16)act_d<ACT>(z);
    }
    // formed here: sunk to their use, they would keep z live instead
    d = __builtin_bit_cast(u32x8, g);
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(d[i]));
}

__device__ __forceinline__ void grad_block(const f32x16& c, const u32x8& d, int mb, int nb, int l, MlpLds& s) {
    const int col = nb * 32 + acc_col(l);
    const bf16x16 g = __builtin_bit_cast(bf16x16, d);
    bf16x4 t;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = mb * 32 + acc_row(i, l);
        t[i & 3] = (__bf16)(c[i] * (float)g[i]);
        s.dz[row * kLdH + col] = t[i & 3];
        if ((i & 3) == 3) store4(s.dzt + col * kLdH + row - 3, t);
    }
}

// One 64-sample tile per block of four wavefronts.  Wavefront (mb, nb) forms
// the same 32x32 block of every 64x64 product -- activations, their
// derivatives (which stay in its registers) and gradients -- so each layer is
// one MFMA chain deep; dW3, dW1 and the bias sums are shared out.  What
// bounds it is that chain of layers and barriers, not the matrix cores.  (One
// wavefront per tile with 79 KB of LDS put two wavefronts on a CU: 60 us for
// a batch of 65,536, in two rounds; four blocks of four now fit: 23 us.)
template <int ACT>
__global__ __launch_bounds__(256, 4) void mlp_train_kernel(TrainArgs a) {
    __shared__ MlpLds s;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int mb = w >> 1, nb = w & 1;
    f32x16 dw2 = {}, dw13 = {};  // dw13: dW3 rows 32w.. in wavefronts 0, 1; dW1 columns 32(w-2).. in 2, 3
    float db = 0.f, db3 = 0.f, loss = 0.f;  // db: b2 in wavefront 1, b1 in 0
    
    const uint32_t ntile = a.batch / 64u;
    for (uint32_t t = blockIdx.x; t < ntile; t += gridDim.x) {
        // (opaque: fragments and LDS addresses held over the loop would spill)
        const __bf16* wq = a.m.q;
        int l = lane;
        asm volatile("" : "+s"(wq), "+v"(l));
        const uint32_t sidx = t * 64u + (uint32_t)l;
        uint64_t rec;
        if (a.full_pass) {
            rec = sidx;
        } else {
            const U4 o = philox10(sidx, a.step, 0x4D4C50u, 0u, a.seed_lo, a.seed_hi);
            // x mod n: n_inv = floor((2^64 - 1) / n) gives a quotient at most 2 too small
            const uint64_t x = ((uint64_t)o.y << 32) | o.x;
            rec = x - __umul64hi(x, a.n_inv) * a.n;
            if (rec >= a.n) rec -= a.n;
            if (rec >= a.n) rec -= a.n;
        }
        // wavefront w standardises features 3w .. 3w+2 and clears input 12+w
        float y = 0.f, c = 0.f;
        if (w == 0) {
            y = a.ylog[rec];
            c = a.ycrit[rec];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = q < 3 ? 3 * w + q : 12 + w;
            float z = 0.0f;
            if (q < 3) z = (a.feats[rec * 12 + k] - a.m.norm[k]) * (1.0f / a.m.norm[12 + k]);
            const __bf16 b = (__bf16)z;
            s.x[l * kLdX + k] = b;
            s.xt[k * kLdH + l] = b;
        }
        u32x8 g1, g2;
        {
            bf16x8 w1[1];
            load_frags<16>(wq + kQW1t, nb, l, w1);
            __syncthreads();
            activate_block<ACT>(mfma_block<16>(s.x, kLdX, mb, l, w1), a.m.w32[kPB1 + nb * 32 + acc_col(l)], mb, nb, l, s.h1, s.h1t, g1);
            bf16x8 w2[4];
            load_frags<64>(wq + kQW2t, nb, l, w2);
            __syncthreads();
            activate_block<ACT>(mfma_block<64>(s.h1, kLdH, mb, l, w2), a.m.w32[kPB2 + nb * 32 + acc_col(l)], mb, nb, l, s.h2, s.h2t, g2);
        }
        {
            bf16x8 w3[4];
            if (w < 2) load_frags<64>(wq + kQW3t, 0, l, w3);
            __syncthreads();
            if (w < 2) {
                const f32x16 o = mfma_block<64>(s.h2, kLdH, w, l, w3);
                if (acc_col(l) < kNo) {
                    const float b3 = a.m.w32[kPB3 + acc_col(l)];
#pragma unroll
                    for (int i = 0; i < 16; ++i) s.out[(w * 32 + acc_row(i, l)) * 2 + acc_col(l)] = o[i] + b3;
                }
            }
        }
        bf16x8 w3[2];
        load_frags<32>(wq + kQW3, nb, l, w3);
        __syncthreads();
        // dO staged as bf16 [row][32] (columns 0, 1) and transposed
        float d0 = 0.f, d1 = 0.f;
        if (w == 0) {
            const float o0 = s.out[l * 2], o1 = s.out[l * 2 + 1];
            const float sp = fmaxf(o1, 0.f) + log1pf(expf(-fabsf(o1)));
            loss += (o0 - y) * (o0 - y) + sp - c * o1;
            const float inv_b = 1.0f / (float)a.batch;
            d0 = 2.0f * (o0 - y) * inv_b;
            d1 = (1.0f / (1.0f + expf(-o1)) - c) * inv_b;
        }
        bf16x8 dO = {};
        dO[0] = (__bf16)d0;
        dO[1] = (__bf16)d1;
        *reinterpret_cast<bf16x8*>(s.dz + l * kLdH + 8 * w) = dO;
#pragma unroll
        for (int q = 0; q < 8; ++q) s.dzt[(8 * w + q) * kLdH + l] = dO[q];
        __syncthreads();
        // dW3[hid][out] += H2^T . dO ; db3 ; dH2 = dO . W3^T
        f32x16 dh = mfma_block<32>(s.dz, kLdH, mb, l, w3);
        if (w < 2) {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                dw13 = mfma(lds_frag(s.h2t, kLdH, w * 32, kb * 16, l), lds_frag(s.dzt, kLdH, 0, kb * 16, l), dw13);
        } else if (w == 2 && l < kNo) {
#pragma unroll 8
            for (int r = 0; r < 64; ++r) db3 += (float)s.dz[r * kLdH + l];
        }
        __syncthreads();
        grad_block(dh, g2, mb, nb, l, s);
        bf16x8 w2[4];
        load_frags<64>(wq + kQW2, nb, l, w2);
        __syncthreads();
        // dW2[in][out] += H1^T . dZ2 ; db2 ; dH1 = dZ2 . W2^T
        dh = mfma_block<64>(s.dz, kLdH, mb, l, w2);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
            dw2 = mfma(lds_frag(s.h1t, kLdH, mb * 32, kb * 16, l), lds_frag(s.dzt, kLdH, nb * 32, kb * 16, l), dw2);
        if (w == 1) {
#pragma unroll 8
            for (int r = 0; r < 64; ++r) db += (float)s.dz[r * kLdH + l];
        }
        __syncthreads();
        grad_block(dh, g1, mb, nb, l, s);
        __syncthreads();
        // dW1[in][hid] += X^T . dZ1 (M = 16 inputs padded to 32 rows) ; db1
        if (w >= 2) {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                bf16x8 af;
                const int mrow = l & 31, k0 = kb * 16 + 8 * (l >> 5);
#pragma unroll
                for (int j = 0; j < 8; ++j) af[j] = mrow < kNin ? s.xt[mrow * kLdH + k0 + j] : (__bf16)0.0f;
                dw13 = mfma(af, lds_frag(s.dzt, kLdH, (w - 2) * 32, kb * 16, l), dw13);
            }
        } else if (w == 0) {
#pragma unroll 8
            for (int r = 0; r < 64; ++r) db += (float)s.dz[r * kLdH + l];
        }
        __syncthreads();
    }
    // write this block's partial gradient in blob order
    float* P = a.partial + (size_t)blockIdx.x * (kPTotal + 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        P[kPW2 + (mb * 32 + acc_row(i)) * kNh + nb * 32 + acc_col()] = dw2[i];
        const int row = acc_row(i), col = acc_col();
        if (w < 2) {
            if (col < kNo) P[kPW3 + (w * 32 + row) * kNo + col] = dw13[i];
        } else if (row < kNin) {
            P[kPW1 + row * kNh + (w - 2) * 32 + col] = dw13[i];
        }
    }
    if (w == 0) {
        P[kPB1 + lane] = db;
        // loss: wave sum
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
        if (lane == 0) P[kPTotal] = loss;
    } else if (w == 1) {
        P[kPB2 + lane] = db;
    } else if (w == 2 && lane < kNo) {
        P[kPB3 + lane] = db3;
    }
}

// Sum the per-block partials in a fixed order; optional Adam update.
struct AdamArgs {
    float* w32;
    float* m;
    float* v;
    float* grad;             // out: summed gradient (+ loss at [kPTotal])
    float* loss;             // out: the loss sum (nullptr: not wanted)
    __bf16* q;               // packed bf16 copies, updated with the parameters
    const float* partial;
    uint32_t nparts;
    int32_t t;               // Adam step (1-based); 0 = only reduce
    float lr, b1, b2, eps;
};

// Block b reduces parameters 64b..64b+63: wave w sums partials w, w+4, ...
// (coalesced rows), then the four sums are combined in a fixed order, so the
// gradient is deterministic.  22 MB of partials at a batch of 65,536: 128 loads
// in flight per lane hide their latency (8 us; 16 with 32 loads, 23 with 4).  Each updated
// parameter goes to its bf16 copies at once (a pass of its own took 5 us).
constexpr int kAdamParams = 64;
constexpr uint32_t kAdamLoads = 128;
static __global__ __launch_bounds__(256) void mlp_adam_kernel(AdamArgs a) {
    __shared__ float s_g[4][kAdamParams];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int p = blockIdx.x * kAdamParams + lane;
    float g = 0.f;
    if (p <= kPTotal) {
        const float* P = a.partial + p;
        uint32_t q = (uint32_t)w;
        for (; q + 4u * (kAdamLoads - 1u) < a.nparts; q += 4u * kAdamLoads) {
            float part[kAdamLoads];
#pragma unroll
            for (uint32_t i = 0; i < kAdamLoads; ++i) part[i] = P[(size_t)(q + 4u * i) * (kPTotal + 1)];
#pragma unroll
            for (uint32_t i = 0; i < kAdamLoads; ++i) g += part[i];
        }
#pragma unroll 4
        for (; q < a.nparts; q += 4u) g += P[(size_t)q * (kPTotal + 1)];
    }
    s_g[w][lane] = g;
    __syncthreads();
    if (w != 0 || p > kPTotal) return;
    g = (s_g[0][lane] + s_g[1][lane]) + (s_g[2][lane] + s_g[3][lane]);
    a.grad[p] = g;
    if (p == kPTotal && a.loss) *a.loss = g;
    if (p == kPTotal || a.t <= 0) return;
    if (p >= 12 * kNh && p < kNin * kNh) return;  // padding rows of W1 stay zero
    const float m = a.b1 * a.m[p] + (1.0f - a.b1) * g;
    const float v = a.b2 * a.v[p] + (1.0f - a.b2) * g * g;
    a.m[p] = m;
    a.v[p] = v;
    const float mh = m / (1.0f - powf(a.b1, (float)a.t));
    const float vh = v / (1.0f - powf(a.b2, (float)a.t));
    const float wn = a.w32[p] - a.lr * mh / (sqrtf(vh) + a.eps);
    a.w32[p] = wn;
    const __bf16 b = (__bf16)wn;
    if (p < kPB1) {
        a.q[kQW1t + (p % kNh) * kNin + p / kNh] = b;
    } else if (p >= kPW2 && p < kPB2) {
        const int e = p - kPW2;
        a.q[kQW2t + (e % kNh) * kNh + e / kNh] = b;
        a.q[kQW2 + e] = b;
    } else if (p >= kPW3 && p < kPB3) {
        const int e = p - kPW3;
        a.q[kQW3t + (e % kNo) * kNh + e / kNo] = b;
        a.q[kQW3 + (e / kNo) * kNoPad + e % kNo] = b;
    }
}

// fp32 master -> packed bf16 copies
static __global__ __launch_bounds__(256) void mlp_pack_kernel(const float* w32, __bf16* q) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= kQTotal) return;
    float v = 0.f;
    if (e < kQW2t) {  // W1t[o][i]
        const int o = (e - kQW1t) / kNin, i = (e - kQW1t) % kNin;
        v = w32[kPW1 + i * kNh + o];
    } else if (e < kQW3t) {  // W2t[o][i]
        const int o = (e - kQW2t) / kNh, i = (e - kQW2t) % kNh;
        v = w32[kPW2 + i * kNh + o];
    } else if (e < kQW2) {  // W3t[o][i], o < 32
        const int o = (e - kQW3t) / kNh, i = (e - kQW3t) % kNh;
        v = o < kNo ? w32[kPW3 + i * kNo + o] : 0.f;
    } else if (e < kQW3) {  // W2[i][o]
        v = w32[kPW2 + (e - kQW2)];
    } else {  // W3[i][o], o < 32
        const int i = (e - kQW3) / kNoPad, o = (e - kQW3) % kNoPad;
        v = o < kNo ? w32[kPW3 + i * kNo + o] : 0.f;
    }
    q[e] = (__bf16)v;
}

// ---------------------------------------------------------------------------
// inference: the three layers chained in registers
//
// Each layer runs in transposed form, out^T = W^T in^T: the A operand is a
// fragment of W^T (staged in LDS once per block), the B operand the tile's
// activations.  A lane's accumulator holds units 8(i/4) + 4(l/32) + i%4 of
// tile row l%32 (rows 32..63 in the second half-tile nb), and the next
// layer's B fragment wants 8 consecutive units of that row: lane l < 32
// already holds half of them, its partner l + 32 the other half, so one
// v_permlane32_swap per packed bf16 pair builds the fragment without any
// LDS round trip.  Input rows enter the same way (lane r holds row r).
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kLdW1 = 24, kLdW2 = 72;  // LDS row strides (bf16), padded against bank conflicts

// Weights of the inference path in LDS: W1^T [64][16], W2^T [64][64],
// W3^T [32][64] (rows 2..31 zero), biases.
struct MlpLdsW {
    __bf16 w1t[kNh * kLdW1];
    __bf16 w2t[kNh * kLdW2];
    __bf16 w3t[kNoPad * kLdW2];
    float b1[kNh], b2[kNh], b3[4];
};

// Whole block, 16-byte copies; the caller synchronises the block after it.
__device__ __forceinline__ void stage_weights(MlpLdsW& W, const MlpDev& m) {
    const uint32_t nt = blockDim.x;
    const uint4* q = reinterpret_cast<const uint4*>(m.q);
    for (uint32_t e = threadIdx.x; e < (uint32_t)kNh * 2u; e += nt)
        *reinterpret_cast<uint4*>(&W.w1t[(e >> 1) * kLdW1 + (e & 1u) * 8u]) = q[(kQW1t >> 3) + e];
    for (uint32_t e = threadIdx.x; e < (uint32_t)kNh * 8u; e += nt)
        *reinterpret_cast<uint4*>(&W.w2t[(e >> 3) * kLdW2 + (e & 7u) * 8u]) = q[(kQW2t >> 3) + e];
    for (uint32_t e = threadIdx.x; e < (uint32_t)kNoPad * 8u; e += nt)
        *reinterpret_cast<uint4*>(&W.w3t[(e >> 3) * kLdW2 + (e & 7u) * 8u]) = q[(kQW3t >> 3) + e];
    for (uint32_t e = threadIdx.x; e < (uint32_t)kNh; e += nt) {
        W.b1[e] = m.w32[kPB1 + e];
        W.b2[e] = m.w32[kPB2 + e];
    }
    if (threadIdx.x < (uint32_t)kNo) W.b3[threadIdx.x] = m.w32[kPB3 + threadIdx.x];
}

// The dword of lane l ^ 32 (v_permlane32_swap exchanges lanes 32..63 of its
// first operand with lanes 0..31 of its second).
__device__ __forceinline__ uint32_t xhalf(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32u) ? r[0] : r[1];
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    const bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// act(acc + bias) of one 32-unit accumulator block as 8 packed bf16 pairs
// (pair j = elements 2j, 2j + 1); bias points at the block's first unit.
template <int ACT>
__device__ __forceinline__ void act_pack(const f32x16& c, const float* bias, uint32_t (&P)[8]) {
    const uint32_t hi = (threadIdx.x >> 5) & 1u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(bias + 8 * j + 4 * (int)hi);
        P[2 * j] = pack_bf16(act_f<ACT>(c[4 * j] + b.x), act_f<ACT>(c[4 * j + 1] + b.y));
        P[2 * j + 1] = pack_bf16(act_f<ACT>(c[4 * j + 2] + b.z), act_f<ACT>(c[4 * j + 3] + b.w));
    }
}

// B fragment of the next layer for k block 2 mb + H from the packed
// activations P of accumulator block mb: lane l < 32 keeps units 16H + 0..3
// and receives 16H + 4..7 from its partner; lane l >= 32 receives
// 16H + 8..11 and keeps 16H + 12..15.
template <int H>
__device__ __forceinline__ bf16x8 next_frag(const uint32_t (&P)[8]) {
    const bool up = (threadIdx.x & 32u) != 0u;
    const uint32_t r0 = xhalf(up ? P[4 * H] : P[4 * H + 2]);
    const uint32_t r1 = xhalf(up ? P[4 * H + 1] : P[4 * H + 3]);
    const u32x4 f = up ? u32x4{r0, r1, P[4 * H + 2], P[4 * H + 3]} : u32x4{P[4 * H], P[4 * H + 1], r0, r1};
    return __builtin_bit_cast(bf16x8, f);
}

// Forward pass of one 64-row tile: lane r holds feature row r (valid: the
// row exists); returns row r's two outputs.  W holds the staged weights.
template <int ACT>
__device__ __forceinline__ void mlp_infer_regs(const MlpLdsW& W, const MlpDev& m, const float (&f)[12], bool valid,
                                               float& o0, float& o1) {
    const bool up = (threadIdx.x & 32u) != 0u;
    uint32_t q[8];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const float z0 = valid ? (f[2 * j] - m.norm[2 * j]) * (1.0f / m.norm[12 + 2 * j]) : 0.0f;
        const float z1 = valid ? (f[2 * j + 1] - m.norm[2 * j + 1]) * (1.0f / m.norm[13 + 2 * j]) : 0.0f;
        q[j] = pack_bf16(z0, z1);
    }
    q[6] = 0u;
    q[7] = 0u;
    // layer-1 B fragments: features 0..7 / 8..15 of rows 0..31 (nb 0) and 32..63 (nb 1)
    uint32_t r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = xhalf(up ? q[i] : q[4 + i]);
    bf16x8 B1[2];
    B1[0] = __builtin_bit_cast(bf16x8, up ? u32x4{r[0], r[1], r[2], r[3]} : u32x4{q[0], q[1], q[2], q[3]});
    B1[1] = __builtin_bit_cast(bf16x8, up ? u32x4{q[4], q[5], q[6], q[7]} : u32x4{r[0], r[1], r[2], r[3]});
    float out[2][2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
        bf16x8 B2[4];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            const f32x16 c = mfma(lds_frag(W.w1t, kLdW1, mb * 32, 0), B1[nb], f32x16{});
            uint32_t P[8];
            act_pack<ACT>(c, W.b1 + mb * 32, P);
            B2[2 * mb] = next_frag<0>(P);
            B2[2 * mb + 1] = next_frag<1>(P);
        }
        bf16x8 B3[4];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            f32x16 c = {};
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) c = mfma(lds_frag(W.w2t, kLdW2, mb * 32, kb * 16), B2[kb], c);
            uint32_t P[8];
            act_pack<ACT>(c, W.b2 + mb * 32, P);
            B3[2 * mb] = next_frag<0>(P);
            B3[2 * mb + 1] = next_frag<1>(P);
        }
        f32x16 c = {};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) c = mfma(lds_frag(W.w3t, kLdW2, 0, kb * 16), B3[kb], c);
        // units 0 and 1 of row nb 32 + l % 32 sit in lanes l < 32
        out[nb][0] = c[0];
        out[nb][1] = c[1];
    }
    const float t0 = __builtin_bit_cast(float, xhalf(__builtin_bit_cast(uint32_t, out[1][0])));
    const float t1 = __builtin_bit_cast(float, xhalf(__builtin_bit_cast(uint32_t, out[1][1])));
    o0 = (up ? t0 : out[0][0]) + W.b3[0];
    o1 = (up ? t1 : out[0][1]) + W.b3[1];
}

// Inference over given feature rows (parity checks and the host API):
// out[n][2].  One wavefront per block, grid-stride over tiles.
template <int ACT>
__global__ __launch_bounds__(64) void mlp_infer_kernel(MlpDev m, const float* feats, uint32_t n, float* out) {
    __shared__ MlpLdsW W;
    stage_weights(W, m);
    __syncthreads();
    const int l = threadIdx.x & 63;
    for (uint32_t t = blockIdx.x; t * 64u < n; t += gridDim.x) {
        const uint32_t r = t * 64u + (uint32_t)l;
        float f[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) f[k] = r < n ? feats[(size_t)r * 12 + k] : 0.f;
        float o0, o1;
        mlp_infer_regs<ACT>(W, m, f, r < n, o0, o1);
        if (r < n) {
            out[(size_t)r * 2] = o0;
            out[(size_t)r * 2 + 1] = o1;
        }
    }
}

}  // namespace plis
