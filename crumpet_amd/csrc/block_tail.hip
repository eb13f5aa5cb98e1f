// The second half of a Swin block and the token-wise steps between stages
// (gfx950), over rows of channels (channels-last volumes):
//
//   swin_mlp_kernel  : x1 = x + a;  y = x1 + W2 gelu(W1 LN(x1) + b1) + b2
//   rows_norm_kernel : [x1 = x + a;] out = LN(x1), rows or 2x2x2 neighbourhoods
//   rows_linear_kernel : out = act(X W^T + b) [+ residual]
//
// MONAI runs the block's tail as an add, a LayerNorm, two Linears, a GELU
// and an add, each a pass over the tokens, with casts between them under
// autocast (SwinTransformerBlock.forward_part2 and forward, which the
// reference leaves to PyTorch: torch-ext/crumpet/monai_patch.py:235-261
// patches forward_part1 only).  At 48 channels those passes move about 60
// bytes per channel and token; the fused kernel moves 6.
//
// Numerics: x1 is rounded to the block's type (what the eager add stores),
// LayerNorm in fp32 in two passes, its result rounded once to the compute
// type, fp32 accumulation, the bias added and the GELU taken in fp32, its
// result rounded once to the compute type, and the last sum rounded once.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "crumpet_common.h"
#include "crumpet_hip.h"

namespace crumpet {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mma2;

template <>
struct Mma2<_Float16> {
    typedef _Float16 x4 __attribute__((ext_vector_type(4)));
    typedef _Float16 x8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x4 mma16(x4 a, x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 mma32(x8 a, x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

template <>
struct Mma2<__bf16> {
    typedef __bf16 x4 __attribute__((ext_vector_type(4)));
    typedef __bf16 x8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x4 mma16(x4 a, x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                         __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 mma32(x8 a, x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

template <typename T>
__device__ __forceinline__ f32x4 load4f(const T* p) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    const T4 v = *reinterpret_cast<const T4*>(p);
    f32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = static_cast<float>(v[e]);
    return r;
}

template <typename T>
__device__ __forceinline__ void store4f(T* p, f32x4 v) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    T4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = static_cast<T>(v[e]);
    *reinterpret_cast<T4*>(p) = o;
}

template <typename T>
__device__ __forceinline__ f32x4 rounded(f32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = static_cast<float>(static_cast<T>(v[e]));
    return v;
}

__device__ __forceinline__ f32x4 param4(const void* p, int32_t dtype, int c, float dflt) {
    if (p == nullptr) return f32x4{dflt, dflt, dflt, dflt};
    if (dtype == CRUMPET_DTYPE_F32) return load4f(static_cast<const float*>(p) + c);
    if (dtype == CRUMPET_DTYPE_F16) return load4f(static_cast<const _Float16*>(p) + c);
    return load4f(static_cast<const __bf16*>(p) + c);
}

// x Phi(x) for a 16-bit result.  Phi(x) = erfc(-x / sqrt 2) / 2 with erfc
// from formula 7.1.26 of Abramowitz & Stegun, Handbook of Mathematical
// Functions (|error| <= 1.5e-7): one reciprocal, one exponential and about
// ten multiply-adds, where erff takes both of its ranges in a wave.  The
// negative side uses erfc itself (no cancellation); +inf gives +inf and
// -inf NaN, as x * 0.5 * (1 + erf(x / sqrt 2)) does.
__device__ __forceinline__ float gelu(float x) {
    const float z = fabsf(x) * 0.70710678f;
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, z, 1.0f));
    float p = __builtin_fmaf(1.061405429f, t, -1.453152027f);
    p = __builtin_fmaf(p, t, 1.421413741f);
    p = __builtin_fmaf(p, t, -0.284496736f);
    p = __builtin_fmaf(p, t, 0.254829592f);
    const float half_erfc = 0.5f * p * t * __builtin_amdgcn_exp2f(z * z * -1.44269504f);
    return x * (x > 0.0f ? 1.0f - half_erfc : half_erfc);
}

// ---- the whole tail of a block, C = 16 KS up to 96 ---------------------------
//
// A wave owns 16 tokens (token = lane & 15, lane group g = lane >> 4 holds
// the channels [4 KS g, 4 KS (g+1)): the contraction order is free as long
// as A and B agree).  LayerNorm sums go over the 4 lanes of a token.  Per 16
// hidden features: KS 16x16x16 products W1 aT starting from b1, the GELU on
// the 4 results of the lane, and KS products W2 hT: the result layout of the
// first product is the B operand of the second, so the hidden layer never
// leaves registers.  Output feature rows are numbered so that a lane ends
// with the channels it loaded, next to its x1.
//
// Both weights live in LDS in fragment order (one conflict-free 8-byte read
// per lane and product), filled once per workgroup; waves are independent
// after that and take every waves-th tile.  What bounds it (fp16, counters of
// one encoder pass): at 48 channels and 110,592 tokens (33 us, 1.0 TB/s) the
// VALU is 43% busy, mostly with the GELU (4 per lane and hidden tile, about 60
// issue cycles each wave, against 2 KS products of 8 to 16), and the waves
// wait half of their cycles on the fill and the rows, for two tiles each.  At
// 96 channels and 13,824 tokens (24 us) the 146 KB of weights leave one
// workgroup a CU: one tile a wave behind the fill, one wave a SIMD, the VALU
// 18% busy and 60% of the cycles waits.
template <typename Tx, typename Tc, int KS>
__global__ void __launch_bounds__(256)
swin_mlp_kernel(Tx* __restrict__ y, const Tx* __restrict__ x, const Tc* __restrict__ add, const void* ln_w,
                const void* ln_b, int32_t ln_dtype, float eps, const Tc* __restrict__ w1,
                const Tc* __restrict__ b1, const Tc* __restrict__ w2, const Tc* __restrict__ b2, uint32_t T,
                int32_t HT, uint32_t tiles) {
    typedef Mma2<Tc> M;
    typedef typename M::x4 X4;
    constexpr int C = 16 * KS;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    X4* const w1l = reinterpret_cast<X4*>(smem);       // [HT][KS][64]
    X4* const w2l = w1l + HT * KS * 64;                // [HT][KS][64]
    f32x4* const b1l = reinterpret_cast<f32x4*>(w2l + HT * KS * 64);  // [HT][4]
    f32x4* const lnl = b1l + HT * 4;                   // [gamma | beta | b2][C / 4]
    const int H = 16 * HT;
    for (int i = threadIdx.x; i < HT * KS * 64; i += 256) {
        const int l = i & 63, col = l & 15, g = l >> 4;
        const int f = i >> 6, ht = f / KS, kk = f - ht * KS;
        // W1 row 16 ht + col, channels 4 KS g + 4 kk ..
        w1l[i] = *reinterpret_cast<const X4*>(w1 + (16 * ht + col) * C + 4 * KS * g + 4 * kk);
        // W2 row of output tile kk: feature 4 KS (col / 4) + 4 kk + col % 4,
        // hidden features 16 ht + 4 g ..
        w2l[i] = *reinterpret_cast<const X4*>(w2 + (4 * KS * (col >> 2) + 4 * kk + (col & 3)) * H + 16 * ht + 4 * g);
    }
    for (int i = threadIdx.x; i < HT * 4; i += 256)
        b1l[i] = b1 ? load4f(b1 + 4 * i) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (threadIdx.x < C / 4) {
        const int c = 4 * threadIdx.x;
        lnl[threadIdx.x] = param4(ln_w, ln_dtype, c, 1.0f);
        lnl[C / 4 + threadIdx.x] = param4(ln_b, ln_dtype, c, 0.0f);
        lnl[C / 2 + threadIdx.x] = b2 ? load4f(b2 + c) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int col = lane & 15;
    const int g = lane >> 4;
    const uint32_t waves = gridDim.x * 4;
    for (uint32_t tile = blockIdx.x * 4 + (threadIdx.x >> 6); tile < tiles; tile += waves) {
        const uint32_t t = tile * 16 + col;
        const int64_t row = int64_t(t < T ? t : T - 1) * C + 4 * KS * g;
        f32x4 x1[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) x1[k] = load4f(x + row + 4 * k);
        if (add != nullptr) {
            f32x4 av[KS];
#pragma unroll
            for (int k = 0; k < KS; ++k) av[k] = load4f(add + row + 4 * k);
#pragma unroll
            for (int k = 0; k < KS; ++k) x1[k] = rounded<Tx>(x1[k] + av[k]);
        }
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < KS; ++k) s += (x1[k][0] + x1[k][1]) + (x1[k][2] + x1[k][3]);
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        const float mean = s * (1.0f / C);
        float q = 0.0f;
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = x1[k][e] - mean;
                q = __builtin_fmaf(d, d, q);
            }
        q += __shfl_xor(q, 16);
        q += __shfl_xor(q, 32);
        const float rstd = rsqrtf(q * (1.0f / C) + eps);
        X4 a[KS];
        f32x4 acc[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const f32x4 gm = lnl[KS * g + k], bt = lnl[C / 4 + KS * g + k];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                a[k][e] = static_cast<Tc>(__builtin_fmaf((x1[k][e] - mean) * rstd, gm[e], bt[e]));
            acc[k] = lnl[C / 2 + KS * g + k];
        }
        // two hidden tiles at a time: the products of one cover the GELU of the
        // other
        for (int ht = 0; ht < HT; ht += 2) {
            f32x4 h[2];
            X4 hb[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                h[u] = b1l[(ht + u) * 4 + g];
#pragma unroll
                for (int k = 0; k < KS; ++k) h[u] = M::mma16(w1l[((ht + u) * KS + k) * 64 + lane], a[k], h[u]);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int e = 0; e < 4; ++e) hb[u][e] = static_cast<Tc>(gelu(h[u][e]));
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    acc[k] = M::mma16(w2l[((ht + u) * KS + k) * 64 + lane], hb[u], acc[k]);
            }
        }
        if (t < T) {
#pragma unroll
            for (int k = 0; k < KS; ++k) store4f(y + row + 4 * k, x1[k] + acc[k]);
        }
    }
}

// ---- fp32 parameters to the compute type ------------------------------------------

// Up to four fp32 arrays into one buffer, each at the next multiple of 8
// elements; a thread converts 8 (zeros past an array's end).  A launch and
// the bytes bound it: 4.1 us for the MLP of 384 channels (1.2 million weights
// and biases), where torch's foreach copy, in 20 workgroups of 64K elements,
// takes 12.
constexpr int kCastArrays = 4;
struct CastArrays {
    const float* src[kCastArrays];
    uint32_t n[kCastArrays];      // elements
    uint32_t first[kCastArrays];  // the array's first 8 elements in the buffer; unused ones past the end
};

template <typename Tc>
__global__ void __launch_bounds__(256) cast_arrays_kernel(Tc* __restrict__ out, const CastArrays a, uint32_t total) {
    typedef Tc T8 __attribute__((ext_vector_type(8)));
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    int k = 0;
#pragma unroll
    for (int j = 1; j < kCastArrays; ++j) k = i >= a.first[j] ? j : k;
    const float* src = a.src[0];
    uint32_t n = a.n[0], first = a.first[0];
#pragma unroll
    for (int j = 1; j < kCastArrays; ++j)
        if (k == j) {
            src = a.src[j];
            n = a.n[j];
            first = a.first[j];
        }
    const uint32_t e0 = (i - first) * 8;
    T8 v = {};
    if (e0 + 8 <= n && reinterpret_cast<uintptr_t>(src) % 16 == 0) {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(src + e0), hi = *reinterpret_cast<const f32x4*>(src + e0 + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = static_cast<Tc>(lo[e]);
            v[4 + e] = static_cast<Tc>(hi[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e0 + e < n) v[e] = static_cast<Tc>(src[e0 + e]);
    }
    *reinterpret_cast<T8*>(out + size_t(i) * 8) = v;
}

// ---- LayerNorm over rows or 2x2x2 neighbourhoods ---------------------------------

// Neighbourhood rows: row (b, d, h, w) of the halved grid holds 8 parts of
// Cp channels; part p is voxel (2d + od, 2h + oh, 2w + ow) with the offset
// bits of p in `order` (4 bits a part: od | oh << 1 | ow << 2); voxels past
// an odd axis are zeros.
struct MergeGeom {
    uint32_t D0, H0, W0;  // the unmerged volume
    uint32_t order;
    FastDiv f_W, f_H, f_D, f_part;  // halved axes; 4-channel chunks per part
};

// LPR lanes per row, kV 4-element chunks per lane (chunk lane + LPR j): the
// row stays in registers over the two passes of the LayerNorm.
template <typename Tx, typename To, int LPR, int kV, bool kMerge>
__global__ void __launch_bounds__(256)
rows_norm_kernel(To* __restrict__ out, Tx* __restrict__ sum_out, const Tx* __restrict__ x, const void* add,
                 int32_t add_dtype, const void* ln_w, const void* ln_b, int32_t ln_dtype, float eps, uint32_t T,
                 int32_t C, const MergeGeom m) {
    const uint32_t t = (blockIdx.y * gridDim.x + blockIdx.x) * (256 / LPR) + threadIdx.x / LPR;
    const int part = threadIdx.x % LPR;
    const int nch = C >> 2;
    const uint32_t tr = t < T ? t : T - 1;
    f32x4 v[kV];
    uint32_t d = 0, h = 0, w = 0, b = 0;
    if constexpr (kMerge) {
        uint32_t t1, t2;
        m.f_W.divmod(tr, t1, w);
        m.f_H.divmod(t1, t2, h);
        m.f_D.divmod(t2, b, d);
    }
#pragma unroll
    for (int j = 0; j < kV; ++j) {
        const int c = part + LPR * j;
        v[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (c < nch) {
            if constexpr (kMerge) {
                uint32_t p, e;
                m.f_part.divmod(c, p, e);
                const uint32_t o = m.order >> (4 * p);
                const uint32_t dd = 2 * d + (o & 1), hh = 2 * h + ((o >> 1) & 1), ww = 2 * w + ((o >> 2) & 1);
                if (dd < m.D0 && hh < m.H0 && ww < m.W0)
                    v[j] = load4f(x + (int64_t((b * m.D0 + dd) * m.H0 + hh) * m.W0 + ww) * (C >> 3) + 4 * e);
            } else {
                v[j] = load4f(x + int64_t(tr) * C + 4 * c);
            }
        }
    }
    if constexpr (!kMerge) {
        if (add != nullptr) {
#pragma unroll
            for (int j = 0; j < kV; ++j) {
                const int c = part + LPR * j;
                if (c < nch) {
                    const int64_t i = int64_t(tr) * C + 4 * c;
                    f32x4 av;
                    if (add_dtype == CRUMPET_DTYPE_F32) av = load4f(static_cast<const float*>(add) + i);
                    else if (add_dtype == CRUMPET_DTYPE_F16) av = load4f(static_cast<const _Float16*>(add) + i);
                    else av = load4f(static_cast<const __bf16*>(add) + i);
                    v[j] = rounded<Tx>(v[j] + av);
                    if (t < T) store4f(sum_out + i, v[j]);
                }
            }
        }
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kV; ++j) s += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) s += __shfl_xor(s, o, LPR);
    const float mean = s / static_cast<float>(C);
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < kV; ++j)
        if (part + LPR * j < nch) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float dv = v[j][e] - mean;
                q = __builtin_fmaf(dv, dv, q);
            }
        }
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) q += __shfl_xor(q, o, LPR);
    const float rstd = rsqrtf(q / static_cast<float>(C) + eps);
    if (t >= T) return;
    auto finish = [&](auto gamma, auto beta) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kV; ++j) {
            const int c = part + LPR * j;
            if (c < nch) {
                const f32x4 gm = gamma(4 * c), bt = beta(4 * c);
                f32x4 r;
#pragma unroll
                for (int e = 0; e < 4; ++e) r[e] = __builtin_fmaf((v[j][e] - mean) * rstd, gm[e], bt[e]);
                store4f(out + int64_t(t) * C + 4 * c, r);
            }
        }
    };
    if (ln_w == nullptr && ln_b == nullptr)
        finish([](int) { return f32x4{1.0f, 1.0f, 1.0f, 1.0f}; }, [](int) { return f32x4{0.0f, 0.0f, 0.0f, 0.0f}; });
    else if (ln_w != nullptr && ln_b != nullptr && ln_dtype == CRUMPET_DTYPE_F32)
        finish([&](int c) { return load4f(static_cast<const float*>(ln_w) + c); },
               [&](int c) { return load4f(static_cast<const float*>(ln_b) + c); });
    else
        finish([&](int c) { return param4(ln_w, ln_dtype, c, 1.0f); },
               [&](int c) { return param4(ln_b, ln_dtype, c, 0.0f); });
}

// ---- out = act(X W^T + b) [+ residual], X [T, K] in the compute type -------------
//
// A workgroup of 4 waves computes 64 features of BT tokens, K in 64-deep
// steps: a step's rows arrive as whole 128-byte lines (8 lanes a row) in
// registers, kAhead steps ahead, and pass through LDS, 16-byte chunks xor'ed
// with the row so that a fragment read (16 rows, one chunk) meets all banks.
// (Fragments loaded straight from memory, 16 rows of 64 bytes an instruction,
// move every line twice: 42 us against 14.7 for 13,824 x 768 -> 192 with the
// residual; hipBLASLt's plain product takes 11.5.)
//   S = 1, BT = 64: the waves take 2 x 2 quarters of the tile and share the
//     staged rows, double-buffered, one barrier a step;
//   S = 4, BT = 16: each wave stages and multiplies its own quarter of K (no
//     barrier), so that few tokens (the deep stages: 27 to 1,728, K = 384 ..
//     6144) fill the chip and the chain of dependent loads is a quarter as
//     long.
// Either way the tile is summed in LDS and leaves as whole lines of 64
// features, bias, GELU and residual on the way.  Workgroups of one XCD
// (xcd_chunk) take neighbouring tiles, features first, so that a row of X is
// fetched into one L2.
template <typename Tc, typename To, int BT, int S>
__global__ void __launch_bounds__(256)
rows_linear_kernel(To* __restrict__ out, const Tc* __restrict__ x, const Tc* __restrict__ w,
                   const Tc* __restrict__ bias, const To* __restrict__ res, int32_t act, uint32_t T, int32_t K,
                   int32_t n_out, uint32_t ftiles, uint32_t chunks) {
    typedef Mma2<Tc> M;
    typedef typename M::x8 X8;
    static_assert((S == 1 && BT == 64) || (S == 4 && BT == 16), "four accumulator tiles a wave");
    constexpr int kRows = 64 + BT;                   // staged rows: 64 of W, BT of X
    constexpr int kLoaders = S == 1 ? 256 : 64;      // threads that stage them
    constexpr int kLoads = kRows * 8 / kLoaders;     // 16-byte loads per thread and step
    constexpr int kAhead = S == 1 ? 3 : 2;           // steps in flight
    constexpr int kStage = kRows * 64;               // elements
    constexpr int kRow = 68;                         // floats per token in the final sum: rows 4 banks apart
    constexpr size_t kStageBytes = size_t(S == 1 ? 2 : 4) * kStage * 2;  // S = 4: one slice per wave
    constexpr size_t kSumBytes = size_t(S) * BT * kRow * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kStageBytes > kSumBytes ? kStageBytes : kSumBytes];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15;
    const int g = lane >> 4;
    uint32_t chunk;
    if (!xcd_chunk(blockIdx.x, gridDim.x, chunks, chunk)) return;
    const int f0 = static_cast<int>(chunk % ftiles) * 64;
    const uint32_t t0 = chunk / ftiles * BT;
    const int steps = (K + 63) >> 6;
    const int s0 = S == 1 ? 0 : steps * wave / S;
    const int s1 = S == 1 ? steps : steps * (wave + 1) / S;

    Tc* const stage = reinterpret_cast<Tc*>(smem) + (S == 1 ? 0 : wave * kStage);
    const int ltid = S == 1 ? threadIdx.x : lane;
    const int lrow = ltid >> 3, lchunk = ltid & 7;
    const Tc* src[kLoads];
    int dst[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = i * (kLoaders / 8) + lrow;
        // rows past the matrices repeat the last one; their results are not stored
        src[i] = (r < 64 ? w + int64_t(min(f0 + r, n_out - 1)) * K
                         : x + int64_t(min(t0 + uint32_t(r - 64), T - 1)) * K) + 8 * lchunk;
        dst[i] = r * 64 + ((lchunk ^ (r & 7)) << 3);
    }
    X8 regs[kAhead][kLoads];
    auto fetch = [&](int s, int buf) __attribute__((always_inline)) {
        const int k = 64 * s;
        const bool inside = s < s1 && k + 8 * lchunk < K;  // the last step may be half a step
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            X8 v = {};
            if (inside) v = *reinterpret_cast<const X8*>(src[i] + k);
            regs[buf][i] = v;
        }
    };
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int fa = S == 1 ? 32 * (wave & 1) : 0;    // the wave's features and tokens in the tile
    const int ta = S == 1 ? 32 * (wave >> 1) : 0;
    auto frag = [&](const Tc* st, int row, int u) __attribute__((always_inline)) {
        return *reinterpret_cast<const X8*>(st + row * 64 + (((4 * u + g) ^ (row & 7)) << 3));
    };
#pragma unroll
    for (int d = 0; d < kAhead; ++d) fetch(s0 + d, d);
    int buf = 0;
    for (int s = s0; s < s1; s += kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
            if (s + d < s1) {
                Tc* const st = stage + (S == 1 ? buf * kStage : 0);
#pragma unroll
                for (int i = 0; i < kLoads; ++i) *reinterpret_cast<X8*>(st + dst[i]) = regs[d][i];
                fetch(s + d + kAhead, d);
                if constexpr (S == 1) {
                    __syncthreads();
                } else {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if constexpr (S == 1) {
                        const X8 w0 = frag(st, fa + col, u), w1 = frag(st, fa + 16 + col, u);
                        const X8 x0 = frag(st, 64 + ta + col, u), x1 = frag(st, 64 + ta + 16 + col, u);
                        acc[0] = M::mma32(w0, x0, acc[0]);
                        acc[1] = M::mma32(w1, x0, acc[1]);
                        acc[2] = M::mma32(w0, x1, acc[2]);
                        acc[3] = M::mma32(w1, x1, acc[3]);
                    } else {
                        const X8 x0 = frag(st, 64 + col, u);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[i] = M::mma32(frag(st, 16 * i + col, u), x0, acc[i]);
                    }
                }
                if constexpr (S != 1) {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
                buf ^= 1;
            }
        }
    }

    __syncthreads();  // the sums reuse the staged rows' LDS
    float* const sum = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = fa + (S == 1 ? 16 * (i & 1) : 16 * i) + 4 * g;
        const int t = ta + (S == 1 ? 16 * (i >> 1) : 0) + col;
        *reinterpret_cast<f32x4*>(sum + ((S == 1 ? 0 : wave * BT) + t) * kRow + f) = acc[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BT / 16; ++i) {
        const int tok = i * 16 + (threadIdx.x >> 4), f = (threadIdx.x & 15) * 4;
        f32x4 v = *reinterpret_cast<const f32x4*>(sum + tok * kRow + f);
#pragma unroll
        for (int p = 1; p < S; ++p) v += *reinterpret_cast<const f32x4*>(sum + (p * BT + tok) * kRow + f);
        const uint32_t t = t0 + tok;
        if (f0 + f >= n_out || t >= T) continue;
        if (bias != nullptr) v += load4f(bias + f0 + f);
        if (act) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu(v[e]);
        }
        const int64_t at = int64_t(t) * n_out + f0 + f;
        if (res != nullptr) v += load4f(res + at);
        store4f(out + at, v);
    }
}

int esize_of(int32_t dtype) {
    return dtype == CRUMPET_DTYPE_F32 ? 4 : (dtype == CRUMPET_DTYPE_F16 || dtype == CRUMPET_DTYPE_BF16) ? 2 : 0;
}

bool aligned16(std::initializer_list<const void*> ps) {
    uintptr_t u = 0;
    for (const void* p : ps) u |= reinterpret_cast<uintptr_t>(p);
    return u % 16 == 0;
}

constexpr int kMlpMaxKS = 6;
constexpr size_t kMlpMaxLds = 160 * 1024;

size_t mlp_lds(int KS, int HT) {
    return size_t(HT) * KS * 64 * 8 * 2 + size_t(HT) * 4 * 16 + size_t(3) * KS * 4 * 16;
}

template <typename Tx, typename Tc, int KS>
int launch_mlp_k(const char* what, hipStream_t s, void* y, const void* x, const void* add, const void* ln_w,
                 const void* ln_b, int32_t ln_dtype, float eps, const void* w1, const void* b1, const void* w2,
                 const void* b2, uint32_t T, int HT) {
    const size_t lds = mlp_lds(KS, HT);
    const auto kernel = swin_mlp_kernel<Tx, Tc, KS>;
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(lds)) != hipSuccess)
        return check_launch(what);
    const uint32_t tiles = (T + 15) / 16;
    // as many workgroups as fit the LDS of 256 CUs (at most 4 each: 16
    // waves hide the loads), then the fewest that keep the number of rounds
    const uint32_t per_cu = static_cast<uint32_t>(std::min<size_t>(4, kMlpMaxLds / lds));
    const uint32_t cap = 256 * per_cu * 4;  // waves
    const uint32_t rounds = (tiles + cap - 1) / cap;
    const uint32_t grid = (tiles + rounds * 4 - 1) / (rounds * 4);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds, s, static_cast<Tx*>(y), static_cast<const Tx*>(x),
                       static_cast<const Tc*>(add), ln_w, ln_b, ln_dtype, eps, static_cast<const Tc*>(w1),
                       static_cast<const Tc*>(b1), static_cast<const Tc*>(w2), static_cast<const Tc*>(b2), T, HT,
                       tiles);
    return check_launch(what);
}

template <typename Tx, typename Tc>
int launch_mlp(const char* what, int KS, hipStream_t s, void* y, const void* x, const void* add, const void* ln_w,
               const void* ln_b, int32_t ln_dtype, float eps, const void* w1, const void* b1, const void* w2,
               const void* b2, uint32_t T, int HT) {
#define CRUMPET_MLP(K) \
    launch_mlp_k<Tx, Tc, K>(what, s, y, x, add, ln_w, ln_b, ln_dtype, eps, w1, b1, w2, b2, T, HT)
    switch (KS) {
        case 1: return CRUMPET_MLP(1);
        case 2: return CRUMPET_MLP(2);
        case 3: return CRUMPET_MLP(3);
        case 4: return CRUMPET_MLP(4);
        case 5: return CRUMPET_MLP(5);
        default: return CRUMPET_MLP(6);
    }
#undef CRUMPET_MLP
}

template <typename Tx, typename To, bool kMerge>
void launch_norm(hipStream_t s, void* out, void* sum_out, const void* x, const void* add, int32_t add_dtype,
                 const void* ln_w, const void* ln_b, int32_t ln_dtype, float eps, uint32_t T, int32_t C,
                 const MergeGeom& m) {
#define CRUMPET_NORM(L, V)                                                                                  \
    do {                                                                                                    \
        const GridXY g = grid_xy((T + 256 / L - 1) / (256 / L));                                            \
        hipLaunchKernelGGL((rows_norm_kernel<Tx, To, L, V, kMerge>), dim3(g.x, g.y), dim3(256), 0, s,       \
                           static_cast<To*>(out), static_cast<Tx*>(sum_out), static_cast<const Tx*>(x), add, \
                           add_dtype, ln_w, ln_b, ln_dtype, eps, T, C, m);                                  \
    } while (0)
    const int nch = C / 4;
    if (nch <= 4 * 3)
        CRUMPET_NORM(4, 3);
    else if (nch <= 16 * 3)
        CRUMPET_NORM(16, 3);
    else if (nch <= 64 * 3)
        CRUMPET_NORM(64, 3);
    else if (nch <= 64 * 6)
        CRUMPET_NORM(64, 6);
    else
        CRUMPET_NORM(64, 24);
#undef CRUMPET_NORM
}

template <bool kMerge>
int launch_norm_t(const char* what, hipStream_t s, void* out, int32_t out_dtype, void* sum_out, const void* x,
                  int32_t x_dtype, const void* add, int32_t add_dtype, const void* ln_w, const void* ln_b,
                  int32_t ln_dtype, float eps, uint32_t T, int32_t C, const MergeGeom& m) {
#define CRUMPET_NORM_T(X, O) \
    launch_norm<X, O, kMerge>(s, out, sum_out, x, add, add_dtype, ln_w, ln_b, ln_dtype, eps, T, C, m)
    constexpr int F = CRUMPET_DTYPE_F32, H = CRUMPET_DTYPE_F16, B = CRUMPET_DTYPE_BF16;
    if (x_dtype == F && out_dtype == F) CRUMPET_NORM_T(float, float);
    else if (x_dtype == F && out_dtype == H) CRUMPET_NORM_T(float, _Float16);
    else if (x_dtype == F && out_dtype == B) CRUMPET_NORM_T(float, __bf16);
    else if (x_dtype == H && out_dtype == F) CRUMPET_NORM_T(_Float16, float);
    else if (x_dtype == H && out_dtype == H) CRUMPET_NORM_T(_Float16, _Float16);
    else if (x_dtype == B && out_dtype == F) CRUMPET_NORM_T(__bf16, float);
    else if (x_dtype == B && out_dtype == B) CRUMPET_NORM_T(__bf16, __bf16);
    else
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: input and output dtypes must be equal, or one of them float32",
                    what);
#undef CRUMPET_NORM_T
    return check_launch(what);
}

constexpr int64_t kNormMaxC = 64 * 24 * 4;

int check_norm(const char* what, int64_t rows, int64_t C, int32_t x_dtype, int32_t out_dtype, int32_t ln_dtype,
               float eps) {
    if (esize_of(x_dtype) == 0 || esize_of(out_dtype) == 0 || esize_of(ln_dtype) == 0)
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: unsupported dtype", what);
    if (rows < 0 || C <= 0) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: negative size", what);
    if (C % 8 != 0 || C > kNormMaxC)
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: channels (%lld) must be a multiple of 8 up to %lld", what,
                    (long long)C, (long long)kNormMaxC);
    if (rows >= (int64_t(1) << 31) - 256) return fail(CRUMPET_ERR_UNSUPPORTED, "%s: too many rows", what);
    if (!(eps >= 0.0f)) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: eps must be non-negative", what);
    return CRUMPET_OK;
}

template <typename Tc, typename To>
void launch_linear(hipStream_t s, void* out, const void* x, const void* w, const void* bias, const void* res,
                   int32_t act, uint32_t T, int32_t K, int32_t n_out) {
    const auto up = [](uint32_t a, uint32_t b) { return (a + b - 1) / b; };
    const uint32_t ft = up(static_cast<uint32_t>(n_out), 64);
#define CRUMPET_LINEAR(BT, S)                                                                              \
    do {                                                                                                   \
        const uint32_t chunks = ft * up(T, BT);                                                            \
        hipLaunchKernelGGL((rows_linear_kernel<Tc, To, BT, S>), dim3(xcd_launch_count(chunks)), dim3(256), \
                           0, s, static_cast<To*>(out), static_cast<const Tc*>(x),                         \
                           static_cast<const Tc*>(w), static_cast<const Tc*>(bias),                        \
                           static_cast<const To*>(res), act, T, K, n_out, ft, chunks);                     \
    } while (0)
    // 64-token tiles once there are about three for every four CUs (216 x 768
    // -> 3072, 192 tiles: 8.5 us against 9.5 with 16-token tiles; 1,728 x
    // 1536 -> 384, 162 tiles: 13.0 against 12.0)
    if (ft * up(T, 64) >= 192)
        CRUMPET_LINEAR(64, 1);
    else
        CRUMPET_LINEAR(16, 4);
#undef CRUMPET_LINEAR
}

}  // namespace
}  // namespace crumpet

using namespace crumpet;

extern "C" int crumpet_swin_mlp(void* y, const void* x, int32_t x_dtype, const void* add, int32_t dtype,
                                int64_t rows, int64_t C, int64_t hidden, const void* ln_weight,
                                const void* ln_bias, int32_t ln_dtype, float eps, const void* w1, const void* b1,
                                const void* w2, const void* b2, void* stream) {
    const char* what = "crumpet_swin_mlp";
    int st = check_norm(what, rows, C, x_dtype, dtype, ln_dtype, eps);
    if (st != CRUMPET_OK) return st;
    if (esize_of(dtype) != 2 || (x_dtype != dtype && x_dtype != CRUMPET_DTYPE_F32))
        return fail(CRUMPET_ERR_UNSUPPORTED,
                    "%s: the compute type must be float16 or bfloat16, and the rows in it or in float32", what);
    if (C % 16 != 0 || C > 16 * kMlpMaxKS || hidden <= 0 || hidden % 32 != 0 || hidden > (1 << 16) ||
        mlp_lds(static_cast<int>(C / 16), static_cast<int>(hidden / 16)) > kMlpMaxLds)
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: %lld channels with %lld hidden features are not covered", what,
                    (long long)C, (long long)hidden);
    if (rows == 0) return CRUMPET_OK;
    if (!y || !x || !w1 || !w2) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: null pointer argument", what);
    if (!aligned16({y, x, add, ln_weight, ln_bias, w1, b1, w2, b2}))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: pointers must be 16-byte aligned", what);
    const int KS = static_cast<int>(C / 16), HT = static_cast<int>(hidden / 16);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t T = static_cast<uint32_t>(rows);
    const bool f32 = x_dtype == CRUMPET_DTYPE_F32;
    if (dtype == CRUMPET_DTYPE_F16)
        return f32 ? launch_mlp<float, _Float16>(what, KS, s, y, x, add, ln_weight, ln_bias, ln_dtype, eps, w1, b1,
                                                 w2, b2, T, HT)
                   : launch_mlp<_Float16, _Float16>(what, KS, s, y, x, add, ln_weight, ln_bias, ln_dtype, eps, w1,
                                                    b1, w2, b2, T, HT);
    return f32 ? launch_mlp<float, __bf16>(what, KS, s, y, x, add, ln_weight, ln_bias, ln_dtype, eps, w1, b1, w2,
                                           b2, T, HT)
               : launch_mlp<__bf16, __bf16>(what, KS, s, y, x, add, ln_weight, ln_bias, ln_dtype, eps, w1, b1, w2,
                                            b2, T, HT);
}

extern "C" int crumpet_swin_mlp_fits(int64_t C, int64_t hidden) {
    return C > 0 && C % 16 == 0 && C <= 16 * kMlpMaxKS && hidden > 0 && hidden % 32 == 0 && hidden <= (1 << 16) &&
           mlp_lds(static_cast<int>(C / 16), static_cast<int>(hidden / 16)) <= kMlpMaxLds;
}

extern "C" int crumpet_cast_arrays(void* out, int32_t dtype, const float* const* arrays, const int64_t* sizes,
                                   int32_t count, void* stream) {
    const char* what = "crumpet_cast_arrays";
    if (esize_of(dtype) != 2) return fail(CRUMPET_ERR_UNSUPPORTED, "%s: dtype must be float16 or bfloat16", what);
    if (count < 0 || count > kCastArrays || (count > 0 && (arrays == nullptr || sizes == nullptr)))
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: at most %d arrays", what, kCastArrays);
    CastArrays a;
    int64_t total = 0;
    for (int i = 0; i < kCastArrays; ++i) {
        a.src[i] = i < count ? arrays[i] : nullptr;
        const int64_t n = i < count ? sizes[i] : 0;
        if (n < 0 || (n > 0 && arrays[i] == nullptr))
            return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: negative size or null array", what);
        if (n >= (int64_t(1) << 31)) return fail(CRUMPET_ERR_UNSUPPORTED, "%s: an array of 2^31 elements", what);
        a.n[i] = static_cast<uint32_t>(n);
        a.first[i] = i < count ? static_cast<uint32_t>(total) : 0xffffffffu;
        total += (n + 7) / 8;
    }
    if (total == 0) return CRUMPET_OK;
    if (out == nullptr) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: null output", what);
    if (!aligned16({out})) return fail(CRUMPET_ERR_UNSUPPORTED, "%s: the output must be 16-byte aligned", what);
    const uint32_t t = static_cast<uint32_t>(total);  // below 2^30
    const dim3 grid((t + 255) / 256), block(256);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == CRUMPET_DTYPE_F16)
        hipLaunchKernelGGL((cast_arrays_kernel<_Float16>), grid, block, 0, s, static_cast<_Float16*>(out), a, t);
    else
        hipLaunchKernelGGL((cast_arrays_kernel<__bf16>), grid, block, 0, s, static_cast<__bf16*>(out), a, t);
    return check_launch(what);
}

extern "C" int crumpet_rows_norm(void* out, int32_t out_dtype, void* sum_out, const void* x, int32_t x_dtype,
                                 const void* add, int32_t add_dtype, int64_t rows, int64_t C,
                                 const void* ln_weight, const void* ln_bias, int32_t ln_dtype, float eps,
                                 void* stream) {
    const char* what = "crumpet_rows_norm";
    int st = check_norm(what, rows, C, x_dtype, out_dtype, ln_dtype, eps);
    if (st != CRUMPET_OK) return st;
    if (add != nullptr && (sum_out == nullptr || esize_of(add_dtype) == 0))
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: an addend needs a known dtype and a place for the sum", what);
    if (rows == 0) return CRUMPET_OK;
    if (!out || !x) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: null data pointer", what);
    if (!aligned16({out, sum_out, x, add, ln_weight, ln_bias}))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: pointers must be 16-byte aligned", what);
    return launch_norm_t<false>(what, static_cast<hipStream_t>(stream), out, out_dtype, sum_out, x, x_dtype, add,
                                add_dtype, ln_weight, ln_bias, ln_dtype, eps, static_cast<uint32_t>(rows),
                                static_cast<int32_t>(C), MergeGeom{});
}

extern "C" int crumpet_merge_norm_3d(void* out, int32_t out_dtype, const void* x, int32_t x_dtype, int64_t B,
                                     int64_t D, int64_t H, int64_t W, int64_t C, uint32_t order,
                                     const void* ln_weight, const void* ln_bias, int32_t ln_dtype, float eps,
                                     void* stream) {
    const char* what = "crumpet_merge_norm_3d";
    if (B < 0 || D <= 0 || H <= 0 || W <= 0)
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: B must be non-negative and D, H, W positive", what);
    if (C <= 0 || C % 4 != 0 || C > kNormMaxC / 8)
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: channels (%lld) must be a multiple of 4 up to %lld", what,
                    (long long)C, (long long)(kNormMaxC / 8));
    if (order & 0x88888888u)
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: every part's offset takes three bits", what);
    if (B * D * H * W >= (int64_t(1) << 31))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: more than 2^31 tokens", what);
    const int64_t D2 = (D + 1) / 2, H2 = (H + 1) / 2, W2 = (W + 1) / 2;
    const int64_t rows = B * D2 * H2 * W2;
    int st = check_norm(what, rows, 8 * C, x_dtype, out_dtype, ln_dtype, eps);
    if (st != CRUMPET_OK) return st;
    if (rows == 0) return CRUMPET_OK;
    if (!out || !x) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: null data pointer", what);
    if (!aligned16({out, x, ln_weight, ln_bias}))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: pointers must be 16-byte aligned", what);
    MergeGeom m;
    m.D0 = static_cast<uint32_t>(D);
    m.H0 = static_cast<uint32_t>(H);
    m.W0 = static_cast<uint32_t>(W);
    m.order = order;
    m.f_W.init(static_cast<uint32_t>(W2));
    m.f_H.init(static_cast<uint32_t>(H2));
    m.f_D.init(static_cast<uint32_t>(D2));
    m.f_part.init(static_cast<uint32_t>(C / 4));
    return launch_norm_t<true>(what, static_cast<hipStream_t>(stream), out, out_dtype, nullptr, x, x_dtype, nullptr,
                               CRUMPET_DTYPE_F32, ln_weight, ln_bias, ln_dtype, eps, static_cast<uint32_t>(rows),
                               static_cast<int32_t>(8 * C), m);
}

extern "C" int crumpet_rows_linear(void* out, int32_t out_dtype, const void* x, int32_t dtype, int64_t rows,
                                   int64_t K, const void* weight, const void* bias, int64_t n_out,
                                   int32_t activation, const void* residual, void* stream) {
    const char* what = "crumpet_rows_linear";
    if (esize_of(dtype) != 2 || (out_dtype != dtype && out_dtype != CRUMPET_DTYPE_F32))
        return fail(CRUMPET_ERR_UNSUPPORTED,
                    "%s: the operands must be float16 or bfloat16, and the result in that type or float32", what);
    if (rows < 0 || K <= 0 || n_out <= 0) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: negative size", what);
    if (K % 32 != 0 || n_out % 16 != 0 || K > (1 << 20) || n_out > (1 << 20))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: K must be a multiple of 32 and n_out of 16 (at most 2^20)", what);
    if (activation != 0 && activation != 1)
        return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: unknown activation %d", what, activation);
    if (rows >= (int64_t(1) << 31) - 256 || (rows + 31) / 32 * ((n_out + 31) / 32) >= (int64_t(1) << 31))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: too many rows", what);
    if (rows == 0) return CRUMPET_OK;
    if (!out || !x || !weight) return fail(CRUMPET_ERR_INVALID_ARGUMENT, "%s: null pointer argument", what);
    if (!aligned16({out, x, weight, bias, residual}))
        return fail(CRUMPET_ERR_UNSUPPORTED, "%s: pointers must be 16-byte aligned", what);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t T = static_cast<uint32_t>(rows);
    const int32_t k = static_cast<int32_t>(K), n = static_cast<int32_t>(n_out);
    const bool f32 = out_dtype == CRUMPET_DTYPE_F32;
    if (dtype == CRUMPET_DTYPE_F16) {
        if (f32) launch_linear<_Float16, float>(s, out, x, weight, bias, residual, activation, T, k, n);
        else launch_linear<_Float16, _Float16>(s, out, x, weight, bias, residual, activation, T, k, n);
    } else {
        if (f32) launch_linear<__bf16, float>(s, out, x, weight, bias, residual, activation, T, k, n);
        else launch_linear<__bf16, __bf16>(s, out, x, weight, bias, residual, activation, T, k, n);
    }
    return check_launch(what);
}
