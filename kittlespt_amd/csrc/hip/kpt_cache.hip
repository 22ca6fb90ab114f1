// kpt_cache.hip — the radiance-cache MLP on gfx950 matrix cores.
//
// The reference renderer has no radiance cache; this is the learned part of
// the path tracer: a 6-layer, 64-wide ReLU MLP over a 32-feature frequency
// encoding of (position, direction, roughness), BF16 weights and activations
// on v_mfma_f32_16x16x32_bf16 with FP32 accumulation, trained online with
// Adam on the tracer's own path suffixes.
//
// MFMA operand layout (16x16x32, wave of 64 lanes, r = lane % 16,
// g = lane / 16): lane holds A[r][8g .. 8g+7], B[8g .. 8g+7][r] and
// D[4g .. 4g+3][r].  Every GEMM is arranged so the lane's 8 K-values are
// contiguous in memory (one 16-byte load):
//   forward        Y^T[out][q]  = W[out][in]      * X^T[in][q]   (X row-major [q][in])
//   input grad     dX^T[in][q]  = W^T[in][out]    * dY^T[out][q] (W^T kept as its own copy)
//   weight grad    dW[out][in]  = dY^T[out][q]    * X[q][in]     (X^T and dY^T kept in LDS)
// so D hands lane (r, g) the outputs 4g..4g+3 of query r of each 16-wide tile.
//
// Kernels
//   k_rc_infer<MODE>  inference over queries: MODE 0 adds throughput * radiance
//                     to the path's radiance, MODE 1 writes the raw outputs.
//                     Weights (40 KB BF16) staged once per workgroup in LDS,
//                     one 16-query tile per wave, activations in a per-wave
//                     LDS row buffer.
//   k_rc_train        forward + relative-L2 loss + backward for 64 samples per
//                     workgroup (8 waves); writes its weight-gradient partial.
//   k_rc_adam         adds the partials in a fixed order (deterministic), Adam
//                     step on the FP32 master weights, BF16 republish.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../common/kpt_dmath.h"
#include "kpt_cache.h"
#include "kpt_launch.h"

namespace kpt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float RC_PI = 3.14159265358979323846f;
constexpr float RC_HALF_PI = 1.57079632679489661923f;
constexpr int TRAIN_Q = 64;                 // samples per training workgroup
constexpr int TRAIN_BLOCK = 512;            // 8 waves: 4 groups of 16 samples x 2 halves of the outputs

// Row strides of the matrices in LDS, in BF16 values.  A wave reads 16 rows at
// once, 16 bytes each: at a stride of 64 or 32 values the rows start in two or
// four of the banks and queue eight or four deep, at 72 and 40 in all of them.
constexpr int PAD_IN = RC_IN + 8;
constexpr int PAD_HID = RC_HID + 8;
__host__ __device__ constexpr int pad_in(int l) { return l == 0 ? PAD_IN : PAD_HID; }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// two floats -> two bfloat16, round to nearest even (one instruction)
__device__ __forceinline__ uint32_t bf2(float lo, float hi) {
    const bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 zero4() { f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f}; return z; }
// lanes of one wave exchange data through LDS: order their accesses
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float comp(float x, float y, float z, int a) { return a == 0 ? x : (a == 1 ? y : z); }

// Input features 2i and 2i + 1 of a query (position xyz + roughness in pos,
// outgoing direction in dir): sin and cos of the normalised position at 1, 2,
// 4, 8 cycles per box (i < 12), of (pi/2) * direction (i < 15), then roughness
// and the constant 1.  As one BF16 pair.
__device__ __forceinline__ uint32_t rc_feature_pair(int i, float4 pos, float4 dir, const CacheEncode& e) {
    const int k = i / 3, a = i - 3 * k;
    const float ph = (comp(pos.x, pos.y, pos.z, a) - comp(e.bmin[0], e.bmin[1], e.bmin[2], a)) *
                     comp(e.binv[0], e.binv[1], e.binv[2], a);
    const float arg = i < 12 ? (RC_PI * (float)(1 << k)) * ph : RC_HALF_PI * comp(dir.x, dir.y, dir.z, a);
    float s, c;
    dm::sincosf(arg, &s, &c);
    return i < 15 ? bf2(s, c) : bf2(pos.w, 1.0f);
}

// ReLU + BF16 of one 16-wide output tile into a row-major [q][out] buffer
__device__ __forceinline__ void store_relu_row(uint16_t* row, int t, int g, f32x4 y) {
    uint2 v;
    v.x = bf2(fmaxf(y[0], 0.0f), fmaxf(y[1], 0.0f));
    v.y = bf2(fmaxf(y[2], 0.0f), fmaxf(y[3], 0.0f));
    *reinterpret_cast<uint2*>(row + 16 * t + 4 * g) = v;
}

// ------------------------------------------------------------------ inference
// Bound by vector instructions: about 250 (in double) of a tile's 450 are the
// encoding.  One reduction gives a sine and its cosine, and the padded rows
// keep the weights' reads, 38 of 1 KB per tile, free of bank conflicts (they
// queued eight deep).  862,139 queries: 256 -> 95 us.
constexpr int inf_off(int l) {   // layer l's first value in s_w
    return l == 0 ? 0 : RC_HID * PAD_IN + (l - 1) * RC_HID * PAD_HID;
}
constexpr int INF_W = inf_off(5) + 16 * PAD_HID;   // the output layer's first 16 rows (3 used)

template <int MODE>
__global__ __launch_bounds__(256) void k_rc_infer(CacheBuffers cb, CacheEncode enc, const float4* qpos,
                                                  const float4* qdir, const float4* qbeta, const int32_t* count_dev,
                                                  int64_t count_host, int64_t cap, float4* dst) {
    __shared__ __attribute__((aligned(16))) uint16_t s_w[INF_W];
    __shared__ __attribute__((aligned(16))) uint16_t s_act[4][16 * PAD_HID];
    for (int i = threadIdx.x; i < (rc_off(5) + 16 * RC_HID) / 8; i += 256) {
        // 16-byte pieces: 4 a row in layer 0, 8 in the others
        const int first = rc_off(1) / 8, j = i - first;
        const int at = i < first ? (i >> 2) * PAD_IN + (i & 3) * 8 : inf_off(1) + (j >> 3) * PAD_HID + (j & 7) * 8;
        *reinterpret_cast<uint4*>(s_w + at) = reinterpret_cast<const uint4*>(cb.wb)[i];
    }
    __syncthreads();
    const int64_t n = count_dev ? std::min<int64_t>((int64_t)*count_dev, cap) : count_host;
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63), r = lane & 15, g = lane >> 4;
    uint16_t* act = s_act[wave];
    uint16_t* row = act + r * PAD_HID;
    const int64_t tiles = (n + 15) / 16;
    const int64_t stride = (int64_t)gridDim.x * 4;
    const float4 z4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // the next tile's query (and, adding into paths, its throughput and the
    // path's radiance) is loaded while the current tile runs its layers
    int64_t tile = (int64_t)blockIdx.x * 4 + wave;
    float4 p4n = z4, d4n = z4, ben = z4, lpn = z4;
    if (tile < tiles && tile * 16 + r < n) {
        p4n = qpos[tile * 16 + r];
        d4n = qdir[tile * 16 + r];
        if (MODE == 0) {
            ben = qbeta[tile * 16 + r];
            lpn = dst[(int)__builtin_bit_cast(uint32_t, d4n.w)];
        }
    }
    for (; tile < tiles; tile += stride) {
        const int64_t qi = tile * 16 + r;
        const bool valid = qi < n;
        const float4 p4 = p4n, d4 = d4n, be = ben, lp = lpn;
        const int64_t ni = (tile + stride) * 16 + r;
        if (tile + stride < tiles && ni < n) {
            p4n = qpos[ni];
            d4n = qdir[ni];
            if (MODE == 0) {
                ben = qbeta[ni];
                lpn = dst[(int)__builtin_bit_cast(uint32_t, d4n.w)];
            }
        }
        uint4 f;
        f.x = rc_feature_pair(4 * g, p4, d4, enc);
        f.y = rc_feature_pair(4 * g + 1, p4, d4, enc);
        f.z = rc_feature_pair(4 * g + 2, p4, d4, enc);
        f.w = rc_feature_pair(4 * g + 3, p4, d4, enc);
        const bf16x8 x = __builtin_bit_cast(bf16x8, f);
        // layer 0 (K = 32)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 y = mfma(ld8(s_w + (16 * t + r) * PAD_IN + 8 * g), x, zero4());
            store_relu_row(row, t, g, y);
        }
        wave_lds_sync();
        // layers 1..4 (K = 64): the whole input row is loaded before it is overwritten
#pragma unroll
        for (int L = 1; L <= 4; ++L) {
            const bf16x8 b0 = ld8(row + 8 * g), b1 = ld8(row + 32 + 8 * g);
            wave_lds_sync();
            const uint16_t* wl = s_w + inf_off(L);
            f32x4 y[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                y[t] = mfma(ld8(wl + (16 * t + r) * PAD_HID + 8 * g), b0, zero4());
                y[t] = mfma(ld8(wl + (16 * t + r) * PAD_HID + 32 + 8 * g), b1, y[t]);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) store_relu_row(row, t, g, y[t]);
            wave_lds_sync();
        }
        // output layer: its first 16 rows
        const bf16x8 b0 = ld8(row + 8 * g), b1 = ld8(row + 32 + 8 * g);
        const uint16_t* w5 = s_w + inf_off(5);
        f32x4 o = mfma(ld8(w5 + r * PAD_HID + 8 * g), b0, zero4());
        o = mfma(ld8(w5 + r * PAD_HID + 32 + 8 * g), b1, o);
        wave_lds_sync();
        if (valid && g == 0) {
            if (MODE == 0) {
                const int p = (int)__builtin_bit_cast(uint32_t, d4.w);
                dst[p] = make_float4(lp.x + be.x * (enc.scale * fmaxf(o[0], 0.0f)),
                                     lp.y + be.y * (enc.scale * fmaxf(o[1], 0.0f)),
                                     lp.z + be.z * (enc.scale * fmaxf(o[2], 0.0f)), lp.w);
            } else {
                dst[qi] = make_float4(o[0], o[1], o[2], 0.0f);
            }
        }
    }
}

// ------------------------------------------------------------------ training
// Bound by latency: one workgroup of 64 samples per compute unit, a chain of
// 11 layer products.  So the weights a wave needs, forward and backward, are
// loaded into registers before the first of them, two waves share 16 samples
// (half of the outputs each), and the partial gradient, 75 KB, is written per
// 64 samples.  A step of 16,384 samples: 50 -> 24 us (32 samples in two
// waves, weights loaded layer by layer).
__host__ __device__ constexpr int xo(int l) { return l == 0 ? 0 : TRAIN_Q * PAD_IN + (l - 1) * TRAIN_Q * PAD_HID; }
__host__ __device__ constexpr int xt(int l) { return (l == 0 ? 0 : RC_IN + (l - 1) * RC_HID) * PAD_HID; }   // PAD_HID: TRAIN_Q + 8
static_assert(TRAIN_Q + 8 == PAD_HID, "transposed rows hold a workgroup's samples");
constexpr int XS = TRAIN_Q * (PAD_IN + 5 * PAD_HID);   // layer inputs [q][in]
constexpr int XT = (RC_IN + 5 * RC_HID) * PAD_HID;     // the same, [in][q]

__global__ __launch_bounds__(TRAIN_BLOCK) void k_rc_train(CacheBuffers cb, CacheEncode enc, const float4* qpos,
                                                          const float4* qdir, const float4* target,
                                                          const int32_t* count_dev, int64_t count_host, int64_t cap,
                                                          int64_t first, int32_t batch) {
    __shared__ __attribute__((aligned(16))) uint16_t sX[XS];
    __shared__ __attribute__((aligned(16))) uint16_t sXT[XT];
    __shared__ __attribute__((aligned(16))) uint16_t sdY[TRAIN_Q * PAD_HID];    // output gradients [q][out]
    __shared__ __attribute__((aligned(16))) uint16_t sdYT[RC_HID * PAD_HID];    // the same, [out][q]
    __shared__ float s_loss[4];
    const int64_t n = count_dev ? std::min<int64_t>((int64_t)*count_dev, cap) : count_host;
    const int64_t last = std::min<int64_t>(first + batch, n);
    const int64_t b_eff = last - first;
    if (b_eff <= 0) return;
    const float inv_norm = 1.0f / (3.0f * (float)b_eff);
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63), r = lane & 15, g = lane >> 4;
    const int half = wave & 1;                     // output tiles 2 * half, 2 * half + 1
    const int q = (wave >> 1) * 16 + r;
    const int64_t qi = first + (int64_t)blockIdx.x * TRAIN_Q + q;
    const bool valid = qi < last;
    float* part = cb.partial + (size_t)blockIdx.x * RC_PADDED;
    const float4 z4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 p4 = valid ? qpos[qi] : z4, d4 = valid ? qdir[qi] : z4, t4 = valid ? target[qi] : z4;

    // the wave's weights: w0 / wf / w5 forward, wb (transposed) backward
    bf16x8 w0[2], wf[4][2][2], w5[2], wb5[2], wb[4][2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int row = 16 * (2 * half + t) + r;
        w0[t] = ld8(cb.wb + rc_off(0) + row * RC_IN + 8 * g);
        wb5[t] = ld8(cb.wbt + rc_off(5) + row * 32 + 8 * g);
        w5[t] = ld8(cb.wb + rc_off(5) + r * RC_HID + 32 * t + 8 * g);
#pragma unroll
        for (int l = 0; l < 4; ++l)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                wf[l][t][k] = ld8(cb.wb + rc_off(l + 1) + row * RC_HID + 32 * k + 8 * g);
                wb[l][t][k] = ld8(cb.wbt + rc_off(l + 1) + row * RC_HID + 32 * k + 8 * g);
            }
    }
    // ---- forward, keeping every layer input (and its transpose) in LDS
    {
        uint32_t f[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) f[j] = rc_feature_pair(4 * g + 2 * half + j, p4, d4, enc);
        const int col = 8 * g + 4 * half;
        *reinterpret_cast<uint2*>(sX + q * PAD_IN + col) = make_uint2(f[0], f[1]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sXT[(col + j) * PAD_HID + q] = (uint16_t)(f[j >> 1] >> (16 * (j & 1)));
    }
    __syncthreads();
    f32x4 y[2];
    {
        const bf16x8 x = ld8(sX + q * PAD_IN + 8 * g);
#pragma unroll
        for (int t = 0; t < 2; ++t) y[t] = mfma(w0[t], x, zero4());
    }
#pragma unroll
    for (int L = 1; L <= 5; ++L) {
        // y holds layer L-1's pre-activations: ReLU -> layer L input
        uint16_t* xr = sX + xo(L) + q * PAD_HID;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = 16 * (2 * half + t) + 4 * g;
            const uint32_t lo = bf2(fmaxf(y[t][0], 0.0f), fmaxf(y[t][1], 0.0f)),
                           hi = bf2(fmaxf(y[t][2], 0.0f), fmaxf(y[t][3], 0.0f));
            *reinterpret_cast<uint2*>(xr + col) = make_uint2(lo, hi);
            uint16_t* xc = sXT + xt(L) + col * PAD_HID + q;
            xc[0] = (uint16_t)lo;
            xc[PAD_HID] = (uint16_t)(lo >> 16);
            xc[2 * PAD_HID] = (uint16_t)hi;
            xc[3 * PAD_HID] = (uint16_t)(hi >> 16);
        }
        __syncthreads();
        const bf16x8 b0 = ld8(xr + 8 * g), b1 = ld8(xr + 32 + 8 * g);
        if (L < 5) {
#pragma unroll
            for (int t = 0; t < 2; ++t) y[t] = mfma(wf[L - 1][t][1], b1, mfma(wf[L - 1][t][0], b0, zero4()));
        } else {
            y[0] = mfma(w5[1], b1, mfma(w5[0], b0, zero4()));   // in both halves
        }
    }
    // ---- relative L2 loss (o - t)^2 / (o^2 + 0.01), denominator held constant
    float loss = 0.0f;
    float dy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (g == 0 && valid) {
        const float tt[3] = {t4.x, t4.y, t4.z};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float o = y[0][c];
            const float d = o - tt[c];
            const float den = o * o + 0.01f;
            loss += d * d / den;
            dy[c] = (2.0f * d / den) * inv_norm;
        }
    }
    // output-layer gradient, padded to 32 columns (the second half writes the zeros)
    {
        const uint32_t lo = half ? 0u : bf2(dy[0], dy[1]), hi = half ? 0u : bf2(dy[2], dy[3]);
        const int col = 16 * half + 4 * g;
        *reinterpret_cast<uint2*>(sdY + q * PAD_HID + col) = make_uint2(lo, hi);
        uint16_t* yc = sdYT + col * PAD_HID + q;
        yc[0] = (uint16_t)lo;
        yc[PAD_HID] = (uint16_t)(lo >> 16);
        yc[2 * PAD_HID] = (uint16_t)hi;
        yc[3 * PAD_HID] = (uint16_t)(hi >> 16);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0 && half == 0) s_loss[wave >> 1] = loss;
    __syncthreads();

    // ---- backward
#pragma unroll
    for (int L = 5; L >= 0; --L) {
        constexpr int NW = TRAIN_BLOCK / 64;
        const int in = rc_in(L), ntn = in / 16, ntiles = (L == 5 ? 1 : 4) * ntn;   // layer 5: its first 16 rows
        // weight gradient tiles over the workgroup's 64 samples (K = 64)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int ti = wave + NW * i;
            if (ti < ntiles) {   // uniform in the wave
                const int tm = ti / ntn, tn = ti % ntn;
                const uint16_t* a = sdYT + (16 * tm + r) * PAD_HID + 8 * g;
                const uint16_t* b = sXT + xt(L) + (16 * tn + r) * PAD_HID + 8 * g;
                const f32x4 acc = mfma(ld8(a + 32), ld8(b + 32), mfma(ld8(a), ld8(b), zero4()));
#pragma unroll
                for (int j = 0; j < 4; ++j) part[rc_off(L) + (16 * tm + 4 * g + j) * in + 16 * tn + r] = acc[j];
            }
        }
        if (L == 0) break;
        // input gradient of the wave's own 16 samples, masked by the ReLU of layer L-1
        f32x4 dx[2];
        const bf16x8 d0 = ld8(sdY + q * PAD_HID + 8 * g);
        if (L == 5) {
#pragma unroll
            for (int t = 0; t < 2; ++t) dx[t] = mfma(wb5[t], d0, zero4());
        } else {
            const bf16x8 d1 = ld8(sdY + q * PAD_HID + 32 + 8 * g);
#pragma unroll
            for (int t = 0; t < 2; ++t) dx[t] = mfma(wb[L - 1][t][1], d1, mfma(wb[L - 1][t][0], d0, zero4()));
        }
        __syncthreads();   // every wave is done reading layer L's dY
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int col = 16 * (2 * half + t) + 4 * g;
            const uint2 xv = *reinterpret_cast<const uint2*>(sX + xo(L) + q * PAD_HID + col);   // ReLU outputs: not 0 is positive
            const uint32_t lo = bf2((xv.x & 0x7FFFu) ? dx[t][0] : 0.0f, (xv.x & 0x7FFF0000u) ? dx[t][1] : 0.0f),
                           hi = bf2((xv.y & 0x7FFFu) ? dx[t][2] : 0.0f, (xv.y & 0x7FFF0000u) ? dx[t][3] : 0.0f);
            *reinterpret_cast<uint2*>(sdY + q * PAD_HID + col) = make_uint2(lo, hi);
            uint16_t* yc = sdYT + col * PAD_HID + q;
            yc[0] = (uint16_t)lo;
            yc[PAD_HID] = (uint16_t)(lo >> 16);
            yc[2 * PAD_HID] = (uint16_t)hi;
            yc[3 * PAD_HID] = (uint16_t)(hi >> 16);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) cb.loss_partial[blockIdx.x] = (s_loss[0] + s_loss[1]) + (s_loss[2] + s_loss[3]);
}

// position of padded parameter i in the transposed [in][out_pad] copy
__device__ __forceinline__ int rc_transposed(int i) {
    int L = 5;
    while (L > 0 && i < rc_off(L)) --L;
    const int local = i - rc_off(L), in = rc_in(L);
    return rc_off(L) + (local % in) * rc_out_pad(L) + local / in;
}

struct AdamParams {
    float lr, beta1, beta2, eps;
    float bc1, bc2;       // 1 - beta^t
};

// The gradient sum and the Adam step, 64 parameters per workgroup: 16 waves
// each add a sixteenth of the workgroup partials (consecutive ones, in order),
// then the sixteen sums are added in order, so the total is the same for every
// launch.  The loss's partials are added the same way by one more workgroup
// (a single lane took 29 us over 512 of them).  Bound by the partials' reads
// (19 MB at 16,384 samples): with the sum as its own kernel 13 + 29 us a step,
// now 6.
constexpr int ADAM_GROUPS = 16;
__global__ __launch_bounds__(64 * ADAM_GROUPS) void k_rc_adam(CacheBuffers cb, int nwg, const int32_t* count_dev,
                                                              int64_t count_host, int64_t cap, int64_t first,
                                                              int32_t batch, AdamParams ap) {
    __shared__ float s_sum[ADAM_GROUPS][64];
    const int64_t n = count_dev ? std::min<int64_t>((int64_t)*count_dev, cap) : count_host;
    const int64_t b_eff = std::min<int64_t>(first + batch, n) - first;
    if (b_eff <= 0) return;
    const int lane = (int)(threadIdx.x & 63), grp = (int)(threadIdx.x >> 6);
    const bool of_loss = blockIdx.x * 64 >= (unsigned)RC_PARAMS;   // the last workgroup
    const int i = (int)(blockIdx.x * 64) + lane;
    const int per = (nwg + ADAM_GROUPS - 1) / ADAM_GROUPS;
    const int k0 = min(nwg, grp * per), k1 = min(nwg, k0 + per);
    float sum = 0.0f;
    if (of_loss) {
        for (int k = k0 + lane; k < k1; k += 64) sum += cb.loss_partial[k];
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    } else {
        const float* p = cb.partial + i;   // i < RC_PADDED: within each partial
#pragma unroll 8
        for (int k = k0; k < k1; ++k) sum += p[(size_t)k * RC_PADDED];
    }
    s_sum[grp][lane] = sum;
    __syncthreads();
    if (grp != 0) return;
    float gsum = 0.0f;
    for (int c = 0; c < ADAM_GROUPS; ++c) gsum += s_sum[c][lane];
    if (of_loss) {
        if (lane == 0) {
            cb.stats[0] = gsum / (3.0f * (float)b_eff);
            cb.stats[1] = (float)b_eff;
        }
        return;
    }
    if (i >= RC_PARAMS) return;
    cb.grad[i] = gsum;
    const float m = ap.beta1 * cb.adam_m[i] + (1.0f - ap.beta1) * gsum;
    const float v = ap.beta2 * cb.adam_v[i] + (1.0f - ap.beta2) * (gsum * gsum);
    cb.adam_m[i] = m;
    cb.adam_v[i] = v;
    const float mh = m / ap.bc1, vh = v / ap.bc2;
    const float w = cb.w[i] - ap.lr * mh / (__builtin_sqrtf(vh) + ap.eps);
    cb.w[i] = w;
    const uint16_t b = f2bf(w);
    cb.wb[i] = b;
    cb.wbt[rc_transposed(i)] = b;
}

// BF16 copies of the master weights (padding stays zero)
__global__ void k_rc_publish(CacheBuffers cb) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i >= RC_PADDED) return;
    const uint16_t b = (i < RC_PARAMS) ? f2bf(cb.w[i]) : (uint16_t)0;
    cb.wb[i] = b;
    cb.wbt[rc_transposed(i)] = b;
}

// suffix radiance of each training record in network units
__global__ __launch_bounds__(256) void k_rc_targets(CacheBuffers cb, const float4* L, float scale) {
    const int64_t n = std::min<int64_t>((int64_t)cb.counters[1], cb.train_cap);
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int p = (int)__builtin_bit_cast(uint32_t, cb.t_dir[i].w);
    const float4 l = L[p], b = cb.t_lbefore[i], be = cb.t_beta[i];
    auto suffix = [&](float lend, float lb, float bc) { return bc > 0.0f ? ((lend - lb) / bc) / scale : 0.0f; };
    cb.t_target[i] = make_float4(suffix(l.x, b.x, be.x), suffix(l.y, b.y, be.y), suffix(l.z, b.z, be.z), 0.0f);
}

// Start of a frame's cache records: this frame's training threshold into
// counters[2], then the query and record counts cleared.  With cf.adapt the
// previous frame's counts (same context and resolution) tell how many paths
// reached their cache vertex: when the cache rendered, each of them wrote a
// query or a record; when it only trained, the records were the threshold's
// share of them.  The threshold is then set so that about cf.train_samples
// paths train; otherwise cf.train_threshold (train_samples over the frame's
// paths) stands.
__global__ void k_rc_frame_start(CacheBuffers cb, CacheFrame cf) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    uint32_t thr = cf.train_threshold;
    if (cf.adapt) {
        const double q = (double)cb.counters[0], r = (double)cb.counters[1];
        const double prev = (double)(uint32_t)cb.counters[2];
        const double reach = cf.enabled ? q + r : (prev > 0.0 ? r * 16777216.0 / prev : 0.0);
        if (reach >= 1.0) thr = (uint32_t)fmin(16777216.0, ceil(16777216.0 * (double)cf.train_samples / reach));
    }
    cb.counters[2] = (int32_t)thr;
    cb.counters[0] = 0;
    cb.counters[1] = 0;
}

}  // namespace

int cache_train_workgroups(int32_t batch) { return (batch + TRAIN_Q - 1) / TRAIN_Q; }

hipError_t launch_cache_frame_start(hipStream_t s, const CacheBuffers& cb, const CacheFrame& cf) {
    hipLaunchKernelGGL(k_rc_frame_start, dim3(1), dim3(64), 0, s, cb, cf);
    return hipGetLastError();
}

hipError_t launch_cache_publish(hipStream_t s, const CacheBuffers& cb) {
    hipLaunchKernelGGL(k_rc_publish, dim3((RC_PADDED + 255) / 256), dim3(256), 0, s, cb);
    return hipGetLastError();
}

// Workgroups of k_rc_infer resident per CU (its 53 KB of LDS allow 3): the
// persistent grid is sized to what runs at once, so no workgroup waits for
// another to finish before it starts its share of the tiles.
int infer_blocks_per_cu() {
    static int nb = 0;
    if (nb == 0) {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, reinterpret_cast<const void*>(&k_rc_infer<0>), 256, 0) !=
                hipSuccess || v < 1)
            v = 1;
        nb = v;
    }
    return nb;
}

hipError_t launch_cache_infer_paths(hipStream_t s, const CacheBuffers& cb, const CacheEncode& enc, float4* L,
                                    int64_t max_queries, int num_cus) {
    const int64_t tiles = (max_queries + 15) / 16;
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((tiles + 3) / 4,
                                                                           (int64_t)num_cus * infer_blocks_per_cu()));
    hipLaunchKernelGGL(k_rc_infer<0>, dim3(grid), dim3(256), 0, s, cb, enc, cb.q_pos, cb.q_dir, cb.q_beta,
                       cb.counters, (int64_t)0, cb.query_cap, L);
    return hipGetLastError();
}

hipError_t launch_cache_infer_raw(hipStream_t s, const CacheBuffers& cb, const CacheEncode& enc, const float4* pos,
                                  const float4* dir, int64_t n, float4* out, int num_cus) {
    if (n <= 0) return hipSuccess;
    const int64_t tiles = (n + 15) / 16;
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((tiles + 3) / 4,
                                                                           (int64_t)num_cus * infer_blocks_per_cu()));
    hipLaunchKernelGGL(k_rc_infer<1>, dim3(grid), dim3(256), 0, s, cb, enc, pos, dir, (const float4*)nullptr,
                       (const int32_t*)nullptr, n, n, out);
    return hipGetLastError();
}

hipError_t launch_cache_targets(hipStream_t s, const CacheBuffers& cb, const float4* L, float scale) {
    const unsigned grid = (unsigned)((cb.train_cap + 255) / 256);
    hipLaunchKernelGGL(k_rc_targets, dim3(grid), dim3(256), 0, s, cb, L, scale);
    return hipGetLastError();
}

hipError_t launch_cache_train_step(hipStream_t s, const CacheBuffers& cb, const CacheEncode& enc, const float4* pos,
                                   const float4* dir, const float4* target, const int32_t* count_dev,
                                   int64_t count_host, int64_t cap, int64_t first, int32_t batch, float lr,
                                   int64_t step) {
    const int nwg = cache_train_workgroups(batch);
    if (nwg > cb.max_wg) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_rc_train, dim3(nwg), dim3(TRAIN_BLOCK), 0, s, cb, enc, pos, dir, target, count_dev,
                       count_host, cap, first, batch);
    AdamParams ap;
    ap.lr = lr;
    ap.beta1 = 0.9f;
    ap.beta2 = 0.99f;
    ap.eps = 1e-15f;
    ap.bc1 = (float)(1.0 - std::pow(0.9, (double)step));
    ap.bc2 = (float)(1.0 - std::pow(0.99, (double)step));
    hipLaunchKernelGGL(k_rc_adam, dim3((RC_PARAMS + 63) / 64 + 1), dim3(64 * ADAM_GROUPS), 0, s, cb, nwg, count_dev,
                       count_host, cap, first, batch, ap);
    return hipGetLastError();
}

}  // namespace kpt
