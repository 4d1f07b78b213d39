// lps_mlp.hip -- the learned PCISPH warm start: a per-particle MLP
// 16 -> 64 -> 64 -> 1 (ReLU) on BF16 matrix cores with FP32 accumulation.
//
// The network is evaluated in transposed form, Y = W X, with particles along
// the N dimension of v_mfma_f32_16x16x16_bf16: a 16x16 accumulator tile
// (lane l holds rows 4*(l/16)..+3 of column l%16) is exactly the B operand of
// the next layer (lane l holds K rows 4*(l/16)..+3 of column l%16), so the
// forward pass needs no data movement between layers.  The weight-gradient
// products reduce over particles; for them each layer is also evaluated the
// other way round (k_mlp_grad).
//
// BF16: inputs (after normalisation), weights and hidden activations are
// rounded to BF16 (round to nearest even); biases, accumulators, the output
// layer's sum and all gradients accumulate in FP32.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>

#include "lps_common.h"
#include "lps_kernels.h"

using lps_dev::MlpArgs;
using lps_dev::RowMap;

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int IN = LPS_MLP_IN;       // 16
constexpr int HID = LPS_MLP_HIDDEN;  // 64
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + HID * IN;
constexpr int OFF_W2 = OFF_B1 + HID;
constexpr int OFF_B2 = OFF_W2 + HID * HID;
constexpr int OFF_W3 = OFF_B2 + HID;
constexpr int OFF_B3 = OFF_W3 + HID;
static_assert(OFF_B3 + 1 == LPS_MLP_PARAMS, "parameter layout");

// Round to nearest even bfloat16 (v_cvt_pk_bf16_f32; equal to rounding the bit
// pattern for every non-NaN float, a NaN stays a NaN: tests/bf16_check.hip).
__device__ __forceinline__ unsigned short f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef unsigned u32x2v __attribute__((ext_vector_type(2)));

// Two roundings in one instruction: a in the low half, b in the high half.
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{a, b}, bf16x2v));
}
__device__ __forceinline__ bf16x4 f2bf4(float a, float b, float c, float d) {
    return __builtin_bit_cast(bf16x4, u32x2v{f2bf2(a, b), f2bf2(c, d)});
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float rbf(float f) { return bf2f(f2bf(f)); }

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 load4(const unsigned short* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    bf16x4 r;
    r[0] = (short)(v.x & 0xFFFFu);
    r[1] = (short)(v.x >> 16);
    r[2] = (short)(v.y & 0xFFFFu);
    r[3] = (short)(v.y >> 16);
    return r;
}

// The inference weights in BF16, packed once per change of the FP32 master
// copy (k_mlp_pack) so that the seed kernel copies them instead of converting
// them in every block.  The weight matrices are stored as MFMA A-operand
// fragments: fragment t holds, for lane l, the four values the lane passes
// to v_mfma_f32_16x16x16_bf16 (row 16 m + l%16, columns 16 k + 4 (l/16)..+3),
// at [t][l][4].  A wave's fragment read is then 512 contiguous bytes, free of
// LDS bank conflicts (a [row][column] layout puts the 16 rows a lane group
// reads 128 bytes apart, all in one bank).
struct alignas(16) MlpPacked {
    unsigned short w1[HID * IN];    // fragments (m), m < 4: W1[16 m + l%16][4 (l/16) + r]
    unsigned short w2[HID * HID];   // fragments (4 m + k): W2[16 m + l%16][16 k + 4 (l/16) + r]
    float b1[HID], b2[HID], w3[HID];
    float mean[IN], istd[IN];
    float b3;
    float pad_[3];
};
static_assert(sizeof(MlpPacked) % 16 == 0, "packed weights are copied as uint4");

// Inference of one group of 16 samples (column l%16), the output only.
// xin holds features 4*(l/16)..+3 of the lane's sample.
__device__ __forceinline__ float infer(const MlpPacked& S, const float4& xin, bool valid) {
    const uint32_t l = threadIdx.x & 63u, g = l >> 4;
    const float xv[4] = {xin.x, xin.y, xin.z, xin.w};
    float v[4];
    for (int r = 0; r < 4; r++) {
        const uint32_t f = 4u * g + (uint32_t)r;
        v[r] = valid ? (xv[r] - S.mean[f]) * S.istd[f] : 0.f;
    }
    const bf16x4 x = f2bf4(v[0], v[1], v[2], v[3]);
    bf16x4 h1[4];
    for (int mt = 0; mt < 4; mt++) {
        const f32x4 y = mfma(load4(&S.w1[(mt * 64 + l) * 4]), x, f32x4{0.f, 0.f, 0.f, 0.f});
        const float* b1 = &S.b1[mt * 16 + 4 * g];
        h1[mt] = f2bf4(fmaxf(y[0] + b1[0], 0.f), fmaxf(y[1] + b1[1], 0.f), fmaxf(y[2] + b1[2], 0.f),
                       fmaxf(y[3] + b1[3], 0.f));
    }
    float part = 0.f;
    for (int mt = 0; mt < 4; mt++) {
        f32x4 acc{0.f, 0.f, 0.f, 0.f};
        for (int kt = 0; kt < 4; kt++) acc = mfma(load4(&S.w2[((mt * 4 + kt) * 64 + l) * 4]), h1[kt], acc);
        const float* b2 = &S.b2[mt * 16 + 4 * g];
        const float* w3 = &S.w3[mt * 16 + 4 * g];
        const uint32_t lo = f2bf2(fmaxf(acc[0] + b2[0], 0.f), fmaxf(acc[1] + b2[1], 0.f));
        const uint32_t hi = f2bf2(fmaxf(acc[2] + b2[2], 0.f), fmaxf(acc[3] + b2[3], 0.f));
        part += w3[0] * __uint_as_float(lo << 16);
        part += w3[1] * __uint_as_float(lo & 0xFFFF0000u);
        part += w3[2] * __uint_as_float(hi << 16);
        part += w3[3] * __uint_as_float(hi & 0xFFFF0000u);
    }
    part += __shfl_xor(part, 16, 64);
    part += __shfl_xor(part, 32, 64);
    return part + S.b3;
}

__global__ __launch_bounds__(LPS_BLOCK) void k_mlp_pack(const float* __restrict__ params,
                                                        const float* __restrict__ fscale, MlpPacked* __restrict__ out) {
    // element e of the fragment array: r = e % 4, lane l = (e / 4) % 64,
    // fragment t = e / 256
    for (uint32_t e = threadIdx.x; e < HID * IN; e += blockDim.x) {
        const uint32_t r = e & 3u, l = (e >> 2) & 63u, m = e >> 8;
        out->w1[e] = f2bf(params[OFF_W1 + (16u * m + (l & 15u)) * IN + 4u * (l >> 4) + r]);
    }
    for (uint32_t e = threadIdx.x; e < HID * HID; e += blockDim.x) {
        const uint32_t r = e & 3u, l = (e >> 2) & 63u, t = e >> 8, m = t >> 2, k = t & 3u;
        out->w2[e] = f2bf(params[OFF_W2 + (16u * m + (l & 15u)) * HID + 16u * k + 4u * (l >> 4) + r]);
    }
    for (uint32_t k = threadIdx.x; k < HID; k += blockDim.x) {
        out->b1[k] = params[OFF_B1 + k];
        out->b2[k] = params[OFF_B2 + k];
        out->w3[k] = rbf(params[OFF_W3 + k]);
    }
    for (uint32_t k = threadIdx.x; k < IN; k += blockDim.x) {
        out->mean[k] = fscale[k];
        out->istd[k] = fscale[IN + k];
    }
    if (threadIdx.x == 0) {
        out->b3 = params[OFF_B3];
        out->pad_[0] = out->pad_[1] = out->pad_[2] = 0.f;
    }
}

// Copy of the packed weights into LDS by a block of LPS_BLOCK threads: every
// load is issued before the first store, so the copy waits for one memory
// round trip rather than one per row of the block.
__device__ __forceinline__ void load_packed(MlpPacked& S, const MlpPacked* __restrict__ packed) {
    constexpr uint32_t N = sizeof(MlpPacked) / 16u;
    static_assert(N > 2u * LPS_BLOCK && N <= 3u * LPS_BLOCK, "three rows of uint4 per thread");
    const uint4* src = reinterpret_cast<const uint4*>(packed);
    uint4* dst = reinterpret_cast<uint4*>(&S);
    const uint32_t t = threadIdx.x;
    const bool third = t + 2u * LPS_BLOCK < N;
    const uint4 a = src[t], b = src[t + LPS_BLOCK];
    const uint4 c = third ? src[t + 2u * LPS_BLOCK] : make_uint4(0u, 0u, 0u, 0u);
    dst[t] = a;
    dst[t + LPS_BLOCK] = b;
    if (third) dst[t + 2u * LPS_BLOCK] = c;
}

// Network output (in units of the target scale) of n rows of x.
__global__ __launch_bounds__(LPS_BLOCK) void k_mlp_forward(const MlpPacked* __restrict__ packed,
                                                           const float* __restrict__ x, uint32_t n,
                                                           float* __restrict__ y) {
    __shared__ MlpPacked S;
    load_packed(S, packed);
    __syncthreads();
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63u;
    for (uint32_t bb = blockIdx.x * LPS_BLOCK; bb < n; bb += gridDim.x * LPS_BLOCK)
        for (uint32_t grp = 0; grp < 4; grp++) {
            const uint32_t p = bb + w * 64u + grp * 16u + (l & 15u);
            const float4 xin = *reinterpret_cast<const float4*>(x + (size_t)min(p, n - 1u) * IN + 4u * (l >> 4));
            const float v = infer(S, xin, p < n);
            if (p < n && (l >> 4) == 0u) y[p] = v;
        }
}

}  // namespace

// Seed of the PCISPH pressure: p_i = pscale * tscale * MLP(features_i) with
// pscale = delta * rho0 (the network works in units of delta * rho0, which
// makes it independent of particle size and time step), clamped at zero when
// negative pressures are disabled, non-finite values replaced by 0;
// q_i = p_i / rho*_i^2 for the pressure-force pass.
// Four waves per SIMD: the compiler keeps the layer weights and biases in
// registers across the four sample groups (128 VGPRs, no spills; five waves
// would spill).
__global__ __launch_bounds__(LPS_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_mlp_seed(const MlpPacked* __restrict__ packed, float tscale,
                                                        const float* __restrict__ feat, uint32_t fs, uint32_t n,
                                                        float* __restrict__ press, float4* __restrict__ xq,
                                                        float* __restrict__ seed, const float* __restrict__ rho_pred,
                                                        const float* __restrict__ pprev, float kappa,
                                                        float pscale, int clamp_nonneg, const DevGrid* g,
                                                        lps_dev::Scenes sc, LoopRule rule, float rest_density) {
    if (g->status != 0u) return;
    __shared__ MlpPacked S;
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63u;
    // one block per 256-slot chunk, which is one particle block and so belongs
    // to one scene; chunks of scenes that stopped at the first correction are
    // skipped.  The wave's four groups of 16 samples load their features
    // first, so that their latency overlaps the copy of the weights.
    const uint32_t bb = blockIdx.x * LPS_BLOCK;
    // features are feature-major (feature f of slot p at f * fs + p)
    float4 xin[4];
    for (uint32_t grp = 0; grp < 4; grp++) {
        const uint32_t p = min(bb + w * 64u + grp * 16u + (l & 15u), n - 1u);
        const float* fp = feat + (size_t)(4u * (l >> 4)) * fs + p;
        xin[grp] = make_float4(fp[0], fp[fs], fp[2 * (size_t)fs], fp[3 * (size_t)fs]);
    }
    load_packed(S, packed);
    {
        // the seed replaces the first correction's pressure unless the scene's
        // loop stops there (the loop rule at k = 1, which the pressure pass
        // applies: a non-finite error, the tolerance met with min <= 1, or max
        // <= 1; the stall rule cannot stop a loop at its first correction).
        // The test is uniform over the block, so the whole block leaves
        // before the barrier or none of it does.
        const uint32_t s = sc.count == 1u ? 0u : sc.block_scene[blockIdx.x];
        const uint32_t* err = lps_dev::err_slot(sc, s, 1u);
        uint32_t eb = 0u;
#pragma unroll
        for (uint32_t u = 0; u < LPS_ERR_SUBS; u++) eb = max(eb, err[u * LPS_ERR_STRIDE]);
        if (eb >= 0x7F800000u || (1u >= rule.min_iter && __uint_as_float(eb) / rest_density < rule.tol) ||
            1u >= rule.max_iter)
            return;
        const uint32_t end = min(n, sc.info[s].slot0 + sc.info[s].count);
        // the first correction's pressure buffer of this scene
        const size_t ob = (size_t)sc.grid[s].buf_of[1] * fs;
        __syncthreads();
        // lane l finishes slot l of the wave; its values load during the
        // inference (the groups' 16 first lanes finishing each group in turn
        // waited for them four times: 23.8 us, now 19.9 at 524,288 particles)
        const uint32_t p = bb + w * 64u + l;
        const bool own = p < end;
        const uint32_t q = own ? p : bb;
        const float p1 = clamp_nonneg ? press[ob + q] : 0.f, before = clamp_nonneg ? pprev[q] : 0.f;
        const float rp = rho_pred[ob + q];
        float y = 0.f;  // infer gives every row of lanes the group's outputs
        for (uint32_t grp = 0; grp < 4; grp++) {
            const float yg = infer(S, xin[grp], bb + w * 64u + grp * 16u + (l & 15u) < end);
            if (grp == l >> 4) y = yg;
        }
        if (!own) return;
        float v = y * tscale * pscale;
        if (!isfinite(v)) v = 0.f;
        seed[p] = v;
        if (clamp_nonneg) {
            // With negative pressures disabled the loop never lowers a
            // pressure, so the seed stays within an envelope: at least the
            // zero start's own first-correction pressure p1 (which the loop
            // would reach anyway), at most kappa times the particle's previous
            // applied pressure unless p1 is larger.  An over-prediction then
            // shrinks by kappa per step instead of feeding itself through the
            // previous-pressure feature.
            v = fmaxf(p1, fminf(v, kappa * before));
        }
        press[ob + p] = v;
        // the pressure pass reads p / rho*^2 from the w slot of the prediction copy
        reinterpret_cast<float*>(xq)[4u * p + 3u] = v / (rp * rp);
    }
}


// p[0..n) = 0 (clears accumulators without a memset node)
__global__ void k_fill_zero(float* __restrict__ p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

// Gradient of the weighted mean squared error mean(w d^2), d = y - t/tscale,
// w = over_weight where d > 0 and 1 elsewhere, over a batch of n rows of x / t
// (row of sample s given by rm) with respect to the FP32 parameters: each
// block's sums to its row of `part` (then the block's loss), which k_grad_sum
// or k_adam adds up.  The forward uses the BF16-rounded values
// (straight-through).
//
// Every product runs on the matrix cores without moving a value between lanes.
// A 16x16 result tile leaves its rows in 4 (l/16) + r and its columns in l%16,
// an operand its contracted index in the former and its free one in the
// latter, so a tile serves the next product only if that contracts the tile's
// rows.  Forward and backward contract neurons, the weight gradients samples.
// So each layer is evaluated both ways round, with the operands swapped:
// "P" tiles hold neurons in rows (they feed the next layer's product), "Q"
// tiles samples in rows (they feed the weight gradients, and a bias or output
// gradient is a sum over a lane's own four values).  32 samples at a time, so
// that every contraction is 32 long (16 features excepted).
//
// Bound by the latency of its one wave per SIMD and the fetch of its straight
// code: the weights live in registers (as fragments), the loop has no LDS
// traffic but the biases, and the blocks' sums leave without atomics.  19 us
// for 65,536 rows, and 4 us for the sums or Adam; with one orientation and
// transposes through LDS (weights in rows 128 bytes apart, all in one bank) and
// atomic sums it took 73 and 5.  The MFMA work alone is about 1 us.
struct alignas(16) GradSmem {
    // fp32 parameters, W2's rows padded to 68 floats (a fragment's 16 rows then
    // lie in different banks); after the loop the waves' sums in the same layout
    static constexpr int W2S = HID + 4;
    struct Copy {
        float w1[HID * IN], b1[HID], w2[HID * W2S], b2[HID], w3[HID], b3, loss;
        float pad_[2];
    } c[LPS_BLOCK / 64];
};

// Element k of the parameters (the loss after them) in a copy.
__device__ __forceinline__ uint32_t grad_at(uint32_t k) {
    if (k < OFF_W2) return k;
    if (k < OFF_B2) return OFF_W2 + (k - OFF_W2) / HID * GradSmem::W2S + (k - OFF_W2) % HID;
    return k + HID * (GradSmem::W2S - HID);
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// two 16-long halves of a contraction (in the same order on both operands)
__device__ __forceinline__ bf16x8 cat(bf16x4 lo, bf16x4 hi) {
    struct { bf16x4 a, b; } v{lo, hi};
    return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ float relu_bf(float f) { return rbf(fmaxf(f, 0.f)); }

__global__ __launch_bounds__(LPS_BLOCK) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mlp_grad(
    MlpArgs m, const float* __restrict__ x, const float* __restrict__ t, RowMap rm, uint32_t n, float inv_n,
    float over_weight, float* __restrict__ part) {
    __shared__ GradSmem S;
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63u, g = l >> 4, c = l & 15u;
    GradSmem::Copy& P = S.c[0];
    float* copy = reinterpret_cast<float*>(&P);
    {
        // every load before the first store (one memory round trip)
        constexpr uint32_t IT = (LPS_MLP_PARAMS + LPS_BLOCK - 1u) / LPS_BLOCK;
        float v[IT];
#pragma unroll
        for (uint32_t q = 0; q < IT; q++) v[q] = m.params[min(threadIdx.x + q * LPS_BLOCK, (uint32_t)LPS_MLP_PARAMS - 1u)];
#pragma unroll
        for (uint32_t q = 0; q < IT; q++) {
            const uint32_t k = threadIdx.x + q * LPS_BLOCK;
            if (k < LPS_MLP_PARAMS) copy[grad_at(k)] = k >= OFF_W3 && k < OFF_B3 ? rbf(v[q]) : v[q];
        }
    }
    __syncthreads();
    // fragments: W1 and W2 by row (A of the P products, B of the Q ones), W2
    // by column for the backward product
    bf16x4 w1f[4];
    bf16x8 w2f[4][2], w2t[4][2];
    for (int a = 0; a < 4; a++) {
        const float* q = &P.w1[(16 * a + c) * IN + 4 * g];
        w1f[a] = f2bf4(q[0], q[1], q[2], q[3]);
        for (int h = 0; h < 2; h++) {
            const float* u0 = &P.w2[(16 * a + c) * GradSmem::W2S + 32 * h + 4 * g];
            w2f[a][h] = cat(f2bf4(u0[0], u0[1], u0[2], u0[3]), f2bf4(u0[16], u0[17], u0[18], u0[19]));
            const float* v0 = &P.w2[(32 * h + 4 * g) * GradSmem::W2S + 16 * a + c];
            constexpr int R = GradSmem::W2S;
            w2t[a][h] = cat(f2bf4(v0[0], v0[R], v0[2 * R], v0[3 * R]),
                            f2bf4(v0[16 * R], v0[17 * R], v0[18 * R], v0[19 * R]));
        }
    }
    const float b3 = P.b3;
    float b1q[4], b2q[4], w3q[4];
    for (int a = 0; a < 4; a++) {
        b1q[a] = P.b1[16 * a + c];
        b2q[a] = P.b2[16 * a + c];
        w3q[a] = P.w3[16 * a + c];
    }
    float mean[4], istd[4];
    for (int r = 0; r < 4; r++) {
        mean[r] = m.fscale[4 * g + r];
        istd[r] = m.fscale[IN + 4 * g + r];
    }
    const float meanq = m.fscale[c], istdq = m.fscale[IN + c];
    const f32x4 zero{0.f, 0.f, 0.f, 0.f};
    f32x4 dw2[4][4], dw1[4];
    float gw3[4], gb2[4], gb1[4], gb3 = 0.f, lsum = 0.f;
    for (int a = 0; a < 4; a++) {
        dw1[a] = zero;
        gw3[a] = gb2[a] = gb1[a] = 0.f;
        for (int b = 0; b < 4; b++) dw2[a][b] = zero;
    }
    for (uint32_t s0 = (blockIdx.x * (LPS_BLOCK / 64) + w) * 32u; s0 < n; s0 += gridDim.x * (LPS_BLOCK / 64) * 32u) {
        // both groups' rows first: features by quad (P) and by feature (Q)
        float4 xin[2];
        float xq[2][4], tn[2];
        bool valid[2];
        for (int u = 0; u < 2; u++) {
            const uint32_t s = s0 + 16u * u + c;
            valid[u] = s < n;
            const uint32_t row = valid[u] ? rm.row(s) : 0u;
            xin[u] = *reinterpret_cast<const float4*>(x + (size_t)row * IN + 4u * g);
            tn[u] = t[row];
            for (int r = 0; r < 4; r++) {
                const uint32_t rq = (uint32_t)__shfl((int)row, 4 * (int)g + r, 64);
                xq[u][r] = x[(size_t)rq * IN + c];
            }
        }
        bf16x4 xb[2], h1q[2][4], dy2b[2][4], dy1b[2][4];
        for (int u = 0; u < 2; u++) {
            // samples past the end have zero features and no gradient
            const float xi[4] = {xin[u].x, xin[u].y, xin[u].z, xin[u].w};
            float v[4];
            for (int r = 0; r < 4; r++) v[r] = valid[u] ? (xi[r] - mean[r]) * istd[r] : 0.f;
            const bf16x4 xp = f2bf4(v[0], v[1], v[2], v[3]);
            for (int r = 0; r < 4; r++) v[r] = s0 + 16u * u + 4u * g + r < n ? (xq[u][r] - meanq) * istdq : 0.f;
            xb[u] = f2bf4(v[0], v[1], v[2], v[3]);
            // layer 1, P and Q
            bf16x4 h1p[4];
            f32x4 y1q[4];
            for (int a = 0; a < 4; a++) {
                const f32x4 y = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w1f[a], xp, zero, 0, 0, 0);
                const float* b1 = &P.b1[16 * a + 4 * g];
                h1p[a] = f2bf4(fmaxf(y[0] + b1[0], 0.f), fmaxf(y[1] + b1[1], 0.f), fmaxf(y[2] + b1[2], 0.f),
                               fmaxf(y[3] + b1[3], 0.f));
                y1q[a] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(xp, w1f[a], zero, 0, 0, 0);
                for (int r = 0; r < 4; r++) y1q[a][r] += b1q[a];
                h1q[u][a] = f2bf4(fmaxf(y1q[a][0], 0.f), fmaxf(y1q[a][1], 0.f), fmaxf(y1q[a][2], 0.f),
                                  fmaxf(y1q[a][3], 0.f));
            }
            const bf16x8 h1a = cat(h1p[0], h1p[1]), h1b = cat(h1p[2], h1p[3]);
            // layer 2 and the output, P
            f32x4 y2p[4];
            float y = 0.f;
            for (int a = 0; a < 4; a++) {
                y2p[a] = mfma32(w2f[a][1], h1b, mfma32(w2f[a][0], h1a, zero));
                const float* b2 = &P.b2[16 * a + 4 * g];
                const float* w3 = &P.w3[16 * a + 4 * g];
                for (int r = 0; r < 4; r++) {
                    y2p[a][r] += b2[r];
                    y += w3[r] * relu_bf(y2p[a][r]);
                }
            }
            y += __shfl_xor(y, 16, 64);
            y += __shfl_xor(y, 32, 64);
            const float d = valid[u] ? y + b3 - tn[u] / m.tscale : 0.f;
            const float wd = d > 0.f ? over_weight : 1.f;  // over-predictions weigh more
            const float dy = 2.f * wd * d * inv_n;
            if (g == 0u) {
                lsum += wd * d * d;
                gb3 += dy;
            }
            float dyq[4];
            for (int r = 0; r < 4; r++) dyq[r] = __shfl(dy, 4 * (int)g + r, 64);
            // dY2, P
            bf16x4 dy2p[4];
            for (int a = 0; a < 4; a++) {
                const float* w3 = &P.w3[16 * a + 4 * g];
                float q[4];
                for (int r = 0; r < 4; r++) q[r] = y2p[a][r] > 0.f ? w3[r] * dy : 0.f;
                dy2p[a] = f2bf4(q[0], q[1], q[2], q[3]);
            }
            const bf16x8 da = cat(dy2p[0], dy2p[1]), db = cat(dy2p[2], dy2p[3]);
            for (int a = 0; a < 4; a++) {
                // layer 2 and dY2, Q
                f32x4 y2 = mfma32(h1b, w2f[a][1], mfma32(h1a, w2f[a][0], zero));
                float q[4];
                for (int r = 0; r < 4; r++) {
                    const float v2 = y2[r] + b2q[a];
                    gw3[a] += dyq[r] * relu_bf(v2);
                    q[r] = v2 > 0.f ? w3q[a] * dyq[r] : 0.f;
                    gb2[a] += q[r];
                }
                dy2b[u][a] = f2bf4(q[0], q[1], q[2], q[3]);
                // dY1 = (W2^T dY2) relu'(Y1), Q
                const f32x4 e = mfma32(db, w2t[a][1], mfma32(da, w2t[a][0], zero));
                for (int r = 0; r < 4; r++) {
                    q[r] = y1q[a][r] > 0.f ? e[r] : 0.f;
                    gb1[a] += q[r];
                }
                dy1b[u][a] = f2bf4(q[0], q[1], q[2], q[3]);
            }
        }
        // weight gradients over the 32 samples
        bf16x8 hb[4];
        for (int a = 0; a < 4; a++) hb[a] = cat(h1q[0][a], h1q[1][a]);
        const bf16x8 xx = cat(xb[0], xb[1]);
        for (int a = 0; a < 4; a++) {
            const bf16x8 d2 = cat(dy2b[0][a], dy2b[1][a]);
            for (int b = 0; b < 4; b++) dw2[a][b] = mfma32(d2, hb[b], dw2[a][b]);
            dw1[a] = mfma32(cat(dy1b[0][a], dy1b[1][a]), xx, dw1[a]);
        }
    }
    __syncthreads();  // the parameters' copy becomes the first wave's sums
    GradSmem::Copy& G = S.c[w];
    for (int a = 0; a < 4; a++) {
        for (int r = 0; r < 4; r++) {
            const int o = 16 * a + 4 * (int)g + r;
            for (int b = 0; b < 4; b++) G.w2[o * GradSmem::W2S + 16 * b + (int)c] = dw2[a][b][r];
            G.w1[o * IN + (int)c] = dw1[a][r];
        }
        for (float* v : {&gw3[a], &gb2[a], &gb1[a]}) {
            *v += __shfl_xor(*v, 16, 64);
            *v += __shfl_xor(*v, 32, 64);
        }
        if (g == 0u) {
            G.w3[16 * a + c] = gw3[a];
            G.b2[16 * a + c] = gb2[a];
            G.b1[16 * a + c] = gb1[a];
        }
    }
    for (int off = 1; off < 16; off <<= 1) {
        gb3 += __shfl_xor(gb3, off, 64);
        lsum += __shfl_xor(lsum, off, 64);
    }
    if (l == 0u) {
        G.b3 = gb3;
        G.loss = lsum * inv_n;
    }
    __syncthreads();
    float* __restrict__ out = part + (size_t)blockIdx.x * LPS_GRAD_STRIDE;
    for (uint32_t k = threadIdx.x; k <= LPS_MLP_PARAMS; k += LPS_BLOCK) {
        float v = 0.f;
        for (uint32_t q = 0; q < LPS_BLOCK / 64; q++) v += reinterpret_cast<const float*>(&S.c[q])[grad_at(k)];
        out[k] = v;
    }
}

// Sum of element k over the blocks' rows of `part`: a workgroup takes 64
// elements, its 16 waves every sixteenth row each.  The sum on every wave's
// lane of the element; all 1024 threads call it.
constexpr uint32_t LPS_SUM_WAVES = 16u;
__device__ __forceinline__ float part_sum(const float* __restrict__ part, uint32_t nb) {
    __shared__ float s[LPS_SUM_WAVES][64];
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6;
    float v = 0.f;
#pragma unroll 8
    for (uint32_t b = w; b < nb; b += LPS_SUM_WAVES) v += part[(size_t)b * LPS_GRAD_STRIDE + blockIdx.x * 64u + l];
    s[w][l] = v;
    __syncthreads();
    v = 0.f;
    for (uint32_t q = 0; q < LPS_SUM_WAVES; q++) v += s[q][l];
    return v;
}

// The gradient, and the batch's loss added to loss.
__global__ __launch_bounds__(LPS_SUM_WAVES * 64) void k_grad_sum(const float* __restrict__ part, uint32_t nb,
                                                                 float* __restrict__ grad, float* __restrict__ loss) {
    const uint32_t k = blockIdx.x * 64u + (threadIdx.x & 63u);
    const float v = part_sum(part, nb);
    if (threadIdx.x >= 64u) return;
    if (k < LPS_MLP_PARAMS) grad[k] = v;
    else if (k == LPS_MLP_PARAMS) *loss += v;
}

// Adam on the FP32 master parameters (bias-corrected) with the blocks' sums of
// the batch; the batch's loss is added to loss.
__global__ __launch_bounds__(LPS_SUM_WAVES * 64) void k_adam(float* __restrict__ params,
                                                             const float* __restrict__ part, uint32_t nb,
                                                             float* __restrict__ loss, float* __restrict__ m1,
                                                             float* __restrict__ m2, float lr, float b1, float b2,
                                                             float eps, float c1, float c2) {
    const uint32_t k = blockIdx.x * 64u + (threadIdx.x & 63u);
    const float gk = part_sum(part, nb);
    if (threadIdx.x >= 64u) return;
    if (k == LPS_MLP_PARAMS) *loss += gk;
    if (k >= LPS_MLP_PARAMS) return;
    const float a = b1 * m1[k] + (1.f - b1) * gk;
    const float b = b2 * m2[k] + (1.f - b2) * gk * gk;
    m1[k] = a;
    m2[k] = b;
    params[k] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// Per-column sums of x and x^2 (double) over n rows of IN columns, added to
// acc[0..IN) and acc[IN..2 IN).  A lane takes four columns of a row (one
// 16-byte load), so a wave reads 16 whole rows; lanes of the same columns are
// added across the wave, waves in LDS.
__global__ __launch_bounds__(LPS_BLOCK) void k_feature_stats(const float* __restrict__ x, uint64_t n,
                                                             double* __restrict__ acc) {
    __shared__ double s[LPS_BLOCK / 64][2 * IN];
    static_assert(IN == 16, "four lanes per row");
    const uint32_t q = threadIdx.x & 3u, l = threadIdx.x & 63u;
    double a[4] = {0.0, 0.0, 0.0, 0.0}, b[4] = {0.0, 0.0, 0.0, 0.0};
    const uint64_t step = (uint64_t)gridDim.x * (LPS_BLOCK / 4);
#pragma unroll 4
    for (uint64_t i = (uint64_t)blockIdx.x * (LPS_BLOCK / 4) + threadIdx.x / 4u; i < n; i += step) {
        const float4 v = reinterpret_cast<const float4*>(x)[i * 4u + q];
        const double d[4] = {v.x, v.y, v.z, v.w};
        for (int f = 0; f < 4; f++) {
            a[f] += d[f];
            b[f] += d[f] * d[f];
        }
    }
    for (int f = 0; f < 4; f++)
        for (int off = 4; off < 64; off <<= 1) {
            a[f] += __shfl_xor(a[f], off, 64);
            b[f] += __shfl_xor(b[f], off, 64);
        }
    if (l < 4u)
        for (int f = 0; f < 4; f++) {
            s[threadIdx.x >> 6][4u * q + f] = a[f];
            s[threadIdx.x >> 6][IN + 4u * q + f] = b[f];
        }
    __syncthreads();
    if (threadIdx.x < 2 * IN) {
        double v = 0.0;
        for (int w = 0; w < LPS_BLOCK / 64; w++) v += s[w][threadIdx.x];
        atomicAdd(&acc[threadIdx.x], v);
    }
}

// Sums of t and t^2 (double) over n values, added to acc[0] and acc[1].
__global__ __launch_bounds__(LPS_BLOCK) void k_target_stats(const float* __restrict__ t, uint64_t n,
                                                            double* __restrict__ acc) {
    __shared__ double s[LPS_BLOCK / 64][2];
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (uint64_t i = (uint64_t)blockIdx.x * LPS_BLOCK + threadIdx.x; i < n; i += (uint64_t)gridDim.x * LPS_BLOCK) {
        const double v = t[i];
        a += v;
        b += v * v;
    }
    for (int off = 1; off < 64; off <<= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        s[threadIdx.x >> 6][0] = a;
        s[threadIdx.x >> 6][1] = b;
    }
    __syncthreads();
    if (threadIdx.x < 2u) {
        double v = 0.0;
        for (int w = 0; w < LPS_BLOCK / 64; w++) v += s[w][threadIdx.x];
        atomicAdd(&acc[threadIdx.x], v);
    }
}

// Training-set append: particle offset + r * stride (r < count) gives row
// base + r: its features (feature-major source, feature f at f * fs + i) and
// its final pressure divided by pscale.
__global__ void k_collect(const float* __restrict__ feat, uint32_t fs, const float* __restrict__ press,
                          float inv_pscale, uint32_t n, uint32_t stride, uint32_t offset, uint32_t count,
                          float* __restrict__ X, float* __restrict__ Tg, uint64_t base) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= count) return;
    const uint64_t i = (uint64_t)offset + (uint64_t)r * stride;
    if (i >= n) return;
    float* dst = X + (base + r) * IN;
    for (int f = 0; f < IN; f++) dst[f] = feat[(uint64_t)f * fs + i];
    Tg[base + r] = press[i] * inv_pscale;
}

namespace lps_dev {

namespace {
uint32_t mlp_grid(uint64_t n) {
    const uint64_t nb = (n + LPS_BLOCK - 1u) / LPS_BLOCK;
    return (uint32_t)(nb < 1024u ? (nb ? nb : 1u) : 1024u);
}
}  // namespace

size_t mlp_packed_bytes() { return sizeof(MlpPacked); }

void launch_mlp_pack(hipStream_t s, const MlpArgs& m, void* packed) {
    k_mlp_pack<<<1, LPS_BLOCK, 0, s>>>(m.params, m.fscale, static_cast<MlpPacked*>(packed));
}

void launch_mlp_seed(hipStream_t s, const void* packed, float tscale, const float* feat, uint32_t fs, uint32_t n,
                     float* press, float4* xq, float* seed, const float* rho_pred, const float* pprev,
                     float kappa, float pscale, int clamp_nonneg, const DevGrid* g, const Scenes& sc,
                     const LoopRule& rule, float rest_density) {
    // one block per particle block (n is a whole number of blocks)
    k_mlp_seed<<<(n + LPS_BLOCK - 1u) / LPS_BLOCK, LPS_BLOCK, 0, s>>>(static_cast<const MlpPacked*>(packed), tscale,
                                                                      feat, fs, n, press, xq, seed, rho_pred, pprev,
                                                                      kappa, pscale, clamp_nonneg, g, sc, rule,
                                                                      rest_density);
}

void launch_fill_zero(hipStream_t s, float* p, uint32_t n) {
    if (n == 0) return;
    k_fill_zero<<<(n + 255u) / 256u, 256, 0, s>>>(p, n);
}

void launch_mlp_forward(hipStream_t s, const void* packed, const float* x, uint32_t n, float* y) {
    k_mlp_forward<<<mlp_grid(n), LPS_BLOCK, 0, s>>>(static_cast<const MlpPacked*>(packed), x, n, y);
}

namespace {
// blocks of k_mlp_grad: 128 samples each (two rounds of 32 per wave for 65,536
// rows), one per CU at most
uint32_t grad_blocks(uint32_t n) {
    const uint32_t nb = n / 128u + (n % 128u ? 1u : 0u);
    return nb < LPS_GRAD_BLOCKS ? nb : LPS_GRAD_BLOCKS;
}
}  // namespace

void launch_mlp_grad(hipStream_t s, const MlpArgs& m, const float* x, const float* t, const RowMap& rm, uint32_t n,
                     float over_weight, float* part, float* grad, float* loss) {
    const uint32_t nb = grad_blocks(n);
    k_mlp_grad<<<nb, LPS_BLOCK, 0, s>>>(m, x, t, rm, n, 1.f / (float)n, over_weight, part);
    k_grad_sum<<<LPS_GRAD_STRIDE / 64, LPS_SUM_WAVES * 64, 0, s>>>(part, nb, grad, loss);
}

void launch_train_step(hipStream_t s, const MlpArgs& m, const float* x, const float* t, const RowMap& rm, uint32_t n,
                       float over_weight, float* part, float* loss, float* params, float* m1, float* m2, float lr,
                       float b1, float b2, float eps, uint32_t step) {
    const uint32_t nb = grad_blocks(n);
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    k_mlp_grad<<<nb, LPS_BLOCK, 0, s>>>(m, x, t, rm, n, 1.f / (float)n, over_weight, part);
    k_adam<<<LPS_GRAD_STRIDE / 64, LPS_SUM_WAVES * 64, 0, s>>>(params, part, nb, loss, m1, m2, lr, b1, b2, eps, c1,
                                                              c2);
}

void launch_feature_stats(hipStream_t s, const float* x, uint64_t n, double* acc) {
    k_feature_stats<<<512, LPS_BLOCK, 0, s>>>(x, n, acc);
}

void launch_target_stats(hipStream_t s, const float* t, uint64_t n, double* acc) {
    k_target_stats<<<256, LPS_BLOCK, 0, s>>>(t, n, acc);
}

void launch_collect(hipStream_t s, const float* feat, uint32_t fs, const float* press, float pscale, uint32_t n,
                    uint32_t stride, uint32_t offset, uint32_t count, float* X, float* T, uint64_t base) {
    if (count == 0) return;
    k_collect<<<(count + 255u) / 256u, 256, 0, s>>>(feat, fs, press, 1.f / pscale, n, stride, offset, count, X, T,
                                                    base);
}

}  // namespace lps_dev
