// Fused window attention in key chunks for 16-bit types at head dims 32, 64
// and 128 (any N; at head dim 32 windows of more than 32 tokens, or 15 with a
// mask tensor, where the bias-stationary kernel has no form), rows 16-byte
// aligned.  Contract, mask modes and numerics of
// swin_attention_wide_kernel (attention_wide.hip): q scaled in fp32 and
// rounded to the input type, scores and softmax in fp32, P rounded to the
// input type for the P v product, the row sums accumulated from the unrounded
// fp32 P, one division at the end.
//
// Decomposition: a workgroup of 4 waves owns one (window, head) and 64 QT
// queries, QT 16-query tiles per wave, and walks the keys in chunks of 64.
//   - K and V rows arrive as 16-byte pieces, one chunk ahead in registers,
//     and pass through double-buffered LDS, row-major; V^T fragments come
//     from the LDS transpose read.  Pieces are xor'ed with the row so that
//     fragment reads meet distinct banks.
//   - Both products are v_mfma_f32_16x16x32; with QT = 2 every K and V
//     fragment feeds two of them.
//   - Bias (+ mask) words are the accumulators' start, requested a chunk
//     ahead, one 16-byte load (fp32) or the 3 dwords around 4 keys (16-bit).
//   - One online-softmax update per chunk, the row max exact: the largest P
//     is then 1 without rounding (a max that lags by up to 8 loses 20-30% of
//     accuracy at sharp rows: 2.06e-3 against 1.7e-3 in fp16 at head dim 128).
// VALU issue bounds it: 125 shifted windows of 343, 6 heads of 64, bf16 (84 us;
// the general kernel 139) keep the VALU 69% busy, the matrix cores 14%, LDS
// 22%, and the waves spend 29% of their cycles in waits; 128 windows of 512, 6
// heads of 32, fp16 (109 us; 146) 50%, 9%, 7% and 29%, with 43% waiting to
// issue.
// The general kernel at these shapes (16 queries per wave, 16-deep products, a
// transposing scalar store of V, one load per bias value) kept the matrix
// cores at 6-7% of their rate, stalled on LDS stores and on 4-byte loads.
#include <hip/hip_runtime.h>

#include <math.h>

#include "attention_kernel.h"
#include "crumpet_common.h"
#include "crumpet_hip.h"

namespace crumpet {
namespace attn {
namespace {

constexpr int kChunkKeys = 64;
constexpr int kChunkThreads = 256;
// The row max starts at the lowest float, so that keys at -inf have a P of 0.
constexpr float kLowestMax = -3.402823466e38f;
// Row maxima below this (rows masked wholly with the lowest value of fp32 or
// bf16): the product with log2 e would overflow, and keys that differ at all
// differ by more than 1e31, so that P is 1 at the max and 0 elsewhere.
constexpr float kScaledMax = -1e38f;
typedef uint32_t u32x3c __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4c __attribute__((ext_vector_type(4)));

// 16-byte piece of a K row, and 32-byte piece of a V row, in LDS (elements).
template <int D>
__device__ __forceinline__ int k_at(int row, int c) {
    const int sw = D == 32 ? (row >> 1) & 3 : row & 7;
    return row * D + ((c ^ sw) << 3);
}
template <int D>
__device__ __forceinline__ int v_at(int row, int b) {
    const int sw = D == 32 ? (row >> 2) & 1 : D == 64 ? (row >> 1) & 3 : row & 7;
    return row * D + ((b ^ sw) << 4);
}

// Four keys of a bias or mask row from its raw words.
template <int kDtype>
__device__ __forceinline__ f32x4 four_keys(u32x4c w, int shift) {
    f32x4 v;
    if constexpr (kDtype == CRUMPET_DTYPE_F32) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = __uint_as_float(w[r]);
    } else {
        const uint32_t hw[2] = {__builtin_amdgcn_alignbit(w[1], w[0], shift),
                                __builtin_amdgcn_alignbit(w[2], w[1], shift)};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t bits = (r & 1) ? hw[r >> 1] >> 16 : hw[r >> 1] & 0xffffu;
            if constexpr (kDtype == CRUMPET_DTYPE_BF16)
                v[r] = __uint_as_float(bits << 16);
            else
                v[r] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits)));
        }
    }
    return v;
}

// A lane's rows of a [N, N] bias or mask of one head or window.
struct RowWords {
    __amdgpu_buffer_rsrc_t rs;
    int es;
    __device__ __forceinline__ u32x4c load(int rowb, int key) const {
        // 16-bit rows: the dwords around the 4 keys (rowb is dword-aligned)
        if (es == 4) return __builtin_amdgcn_raw_buffer_load_b128(rs, rowb + key * 4, 0, 0);
        const u32x3c w = __builtin_amdgcn_raw_buffer_load_b96(rs, rowb + key * 2, 0, 0);
        return u32x4c{w[0], w[1], w[2], 0u};
    }
};

// Sum and max over the 4 lane groups (lanes l, l ^ 16, l ^ 32, l ^ 48).
__device__ __forceinline__ float sum_groups(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}
__device__ __forceinline__ float over_groups(float x) {
    uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    u = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
    r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Waves per SIMD that the registers are allotted for.
constexpr int chunk_waves(int D, int mode, int QT) {
    if (D == 32) return QT == 1 ? (mode == 1 ? 3 : 4) : (mode == 1 ? 2 : 3);
    return D == 64 ? (mode == 1 ? 3 : 4) : 2;
}

// kMode: 0 no mask, 1 mask tensor (mask[b mod mask_batch], skipped where a
// boundary flag is 0), 2 shifted-window regions.
template <typename T, int D, int kMode, int QT>
__global__ void __launch_bounds__(kChunkThreads) __attribute__((amdgpu_waves_per_eu(chunk_waves(D, kMode, QT))))
swin_attention_chunk_kernel(const Params p, int32_t mask_dtype, uint32_t qblocks, uint32_t chunks) {
    typedef Frag<T> F;
    typedef typename F::x4 X4;
    typedef typename F::x8 X8;
    constexpr int kKS = D / 32;                                  // 32-deep steps of the score product
    constexpr int kDT = D / 16;                                  // 16-dim output tiles
    constexpr int kLoads = kChunkKeys * (D / 8) / kChunkThreads; // 16-byte pieces per thread, of K and of V
    constexpr int kStage = kChunkKeys * D;
    __shared__ __attribute__((aligned(16))) T k_lds[2][kStage];
    __shared__ __attribute__((aligned(16))) T v_lds[2][kStage];
    __shared__ __attribute__((aligned(16))) uint8_t cls_lds[kMode == 2 ? kWideMaxRegionN + kChunkKeys : 4];

    uint32_t chunk;
    if (!xcd_chunk(blockIdx.x, gridDim.x, chunks, chunk)) return;
    const int qb = static_cast<int>(chunk % qblocks);
    const uint32_t bh = chunk / qblocks;
    // the workgroups of one XCD share a head's bias, or with a mask tensor a
    // window's mask
    const int h = static_cast<int>(kMode == 1 ? bh % uint32_t(p.H) : bh / uint32_t(p.B));
    const int b = static_cast<int>(kMode == 1 ? bh / uint32_t(p.H) : bh % uint32_t(p.B));
    const int N = p.N;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15;
    const int g = lane >> 4;

    int split = 0;  // region mode: axes along which this is the last window of a shifted axis
    if constexpr (kMode == 2) {
        const int wi = b % p.nW;
        const int ww = wi % p.nWw;
        const int wt = wi / p.nWw;
        const int wh = wt % p.nWh;
        const int wd = wt / p.nWh;
        split = ((wd == p.nWd - 1 && p.ss[0] > 0) ? 4 : 0) | ((wh == p.nWh - 1 && p.ss[1] > 0) ? 2 : 0) |
                ((ww == p.nWw - 1 && p.ss[2] > 0) ? 1 : 0);
        if (split != 0) {
            for (int j = threadIdx.x; j < N; j += kChunkThreads) {
                const int lw = j % p.ws[2];
                const int t = j / p.ws[2];
                const int lh = t % p.ws[1];
                const int ld = t / p.ws[1];
                cls_lds[j] = static_cast<uint8_t>(((ld >= p.ws[0] - p.ss[0]) ? 4 : 0) |
                                                  ((lh >= p.ws[1] - p.ss[1]) ? 2 : 0) |
                                                  ((lw >= p.ws[2] - p.ss[2]) ? 1 : 0));
            }
        }
    }

    // K and V rows of a chunk: thread unit e covers row e / (D / 8), piece
    // e mod (D / 8); keys past N repeat row N - 1 (their P is 0)
    const T* kbase = static_cast<const T*>(p.k) + int64_t(b) * p.ks[0] + int64_t(h) * p.ks[1];
    const T* vbase = static_cast<const T*>(p.v) + int64_t(b) * p.vs[0] + int64_t(h) * p.vs[1];
    X8 kr[kLoads], vr[kLoads];
    auto fetch_kv = [&](int kc0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int e = threadIdx.x + u * kChunkThreads;
            const int64_t row = min(kc0 + e / (D / 8), N - 1);
            const int d0 = (e % (D / 8)) * 8;
            kr[u] = *reinterpret_cast<const X8*>(kbase + row * p.ks[2] + d0);
            vr[u] = *reinterpret_cast<const X8*>(vbase + row * p.vs[2] + d0);
        }
    };
    auto stash_kv = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int e = threadIdx.x + u * kChunkThreads;
            const int row = e / (D / 8), c = e % (D / 8);
            *reinterpret_cast<X8*>(&k_lds[buf][k_at<D>(row, c)]) = kr[u];
            *reinterpret_cast<X8*>(&v_lds[buf][v_at<D>(row, c >> 1) + (c & 1) * 8]) = vr[u];
        }
    };
    fetch_kv(0);

    // bias and mask rows of the lane's queries
    RowWords bias_rows;
    RowWords mask_rows;
    bias_rows.es = p.bias_dtype == CRUMPET_DTYPE_F32 ? 4 : 2;
    int bias_rowb[QT], bias_shift[QT], mask_rowb[QT], mask_shift[QT], qi[QT];
    const AlignedRsrc br = aligned_rsrc(static_cast<const char*>(p.bias) + int64_t(h) * p.bsd[0] * bias_rows.es,
                                    (int64_t(N - 1) * p.bsd[1] + N) * bias_rows.es);
    bias_rows.rs = br.rs;
    mask_rows = bias_rows;
    bool use_mask = false;
    int mask_lead = 0;
    if constexpr (kMode == 1) {
        use_mask = p.boundary == nullptr || p.boundary[b] != 0;
        mask_rows.es = mask_dtype == CRUMPET_DTYPE_F32 ? 4 : 2;
        const AlignedRsrc mr =
            aligned_rsrc(static_cast<const char*>(p.mask) + int64_t(b % p.mask_batch) * p.ms[0] * mask_rows.es,
                       (int64_t(N - 1) * p.ms[1] + N) * mask_rows.es);
        mask_rows.rs = mr.rs;
        mask_lead = mr.lead;
    }
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        qi[i] = (qb * 4 + wave) * 16 * QT + 16 * i + col;
        const int qr = min(qi[i], N - 1);  // padded queries are computed, never stored
        const int rb = br.lead + static_cast<int>(int64_t(qr) * p.bsd[1]) * bias_rows.es;
        bias_rowb[i] = rb & ~3;
        bias_shift[i] = (rb & 2) * 8;
        mask_rowb[i] = mask_shift[i] = 0;
        if constexpr (kMode == 1) {
            const int mb = mask_lead + static_cast<int>(int64_t(qr) * p.ms[1]) * mask_rows.es;
            mask_rowb[i] = mb & ~3;
            mask_shift[i] = (mb & 2) * 8;
        }
    }
    u32x4c bw[QT][4], mw[kMode == 1 ? QT : 1][4];
    auto fetch_bias = [&](int kc0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < QT; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bw[i][t] = bias_rows.load(bias_rowb[i], kc0 + 16 * t + 4 * g);
                if constexpr (kMode == 1)
                    if (use_mask) mw[i][t] = mask_rows.load(mask_rowb[i], kc0 + 16 * t + 4 * g);
            }
    };
    fetch_bias(0);

    // B operand of S^T = K Q^T: Q[query][32 s + 8 g ..], scaled in fp32 and
    // rounded back to T
    X8 qf[QT][kKS];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const T* qrow = static_cast<const T*>(p.q) + int64_t(b) * p.qs[0] + int64_t(h) * p.qs[1] +
                        int64_t(min(qi[i], N - 1)) * p.qs[2];
#pragma unroll
        for (int s = 0; s < kKS; ++s) {
            const X8 qv = *reinterpret_cast<const X8*>(qrow + 32 * s + 8 * g);
#pragma unroll
            for (int e = 0; e < 8; ++e) qf[i][s][e] = static_cast<T>(static_cast<float>(qv[e]) * p.scale);
        }
    }

    f32x4 o[QT][kDT];  // o[i][dd][r] = O[query][16 dd + 4 g + r]
    float l[QT];       // this lane's share of the query's row sum (its keys), of the fp32 P
    float m_run[QT];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
#pragma unroll
        for (int dd = 0; dd < kDT; ++dd) o[i][dd] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        m_run[i] = kLowestMax;
        l[i] = 0.0f;
    }
    stash_kv(0);
    __syncthreads();  // chunk 0 and the class table are in LDS
    uint32_t my_cls[QT];
    if constexpr (kMode == 2) {
#pragma unroll
        for (int i = 0; i < QT; ++i) my_cls[i] = split ? cls_lds[min(qi[i], N - 1)] * 0x01010101u : 0u;
    }

    const int nchunks = (N + kChunkKeys - 1) / kChunkKeys;
    for (int c = 0; c < nchunks; ++c) {
        const int kc0 = c * kChunkKeys;
        const int buf = c & 1;
        const bool more = c + 1 < nchunks;
        f32x4 S[QT][4];  // S[i][t][r]: key kc0 + 16 t + 4 g + r
        auto start = [&](auto bias_dtype) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < QT; ++i)
#pragma unroll
                for (int t = 0; t < 4; ++t) S[i][t] = four_keys<decltype(bias_dtype)::value>(bw[i][t], bias_shift[i]);
        };
        auto add_mask = [&](auto dtype) __attribute__((always_inline)) {
            if constexpr (kMode == 1) {
#pragma unroll
                for (int i = 0; i < QT; ++i)
#pragma unroll
                    for (int t = 0; t < 4; ++t) S[i][t] += four_keys<decltype(dtype)::value>(mw[i][t], mask_shift[i]);
            }
        };
        using F32 = std::integral_constant<int, CRUMPET_DTYPE_F32>;
        using F16 = std::integral_constant<int, CRUMPET_DTYPE_F16>;
        using BF16 = std::integral_constant<int, CRUMPET_DTYPE_BF16>;
        if (p.bias_dtype == CRUMPET_DTYPE_F32) start(F32{});
        else if (p.bias_dtype == CRUMPET_DTYPE_F16) start(F16{});
        else start(BF16{});
        if constexpr (kMode == 1) {
            if (use_mask) {
                if (mask_dtype == CRUMPET_DTYPE_F32) add_mask(F32{});
                else if (mask_dtype == CRUMPET_DTYPE_F16) add_mask(F16{});
                else add_mask(BF16{});
            }
        }
        if constexpr (kMode == 2) {
            if (split != 0) {
                const uint32_t split4 = split * 0x01010101u;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint32_t kc = *reinterpret_cast<const uint32_t*>(&cls_lds[kc0 + 16 * t + 4 * g]);
#pragma unroll
                    for (int i = 0; i < QT; ++i) {
                        const uint32_t cut = (kc ^ my_cls[i]) & split4;
#pragma unroll
                        for (int r = 0; r < 4; ++r) S[i][t][r] += (cut & (0xffu << (8 * r))) ? -100.0f : 0.0f;
                    }
                }
            }
        }
        if (!more) {  // keys past N
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool past = kc0 + 16 * t + 4 * g + r >= N;
#pragma unroll
                    for (int i = 0; i < QT; ++i) S[i][t][r] = past ? -INFINITY : S[i][t][r];
                }
        }
        if (more) {
            fetch_kv(kc0 + kChunkKeys);
            fetch_bias(kc0 + kChunkKeys);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int s = 0; s < kKS; ++s) {
                const X8 kf = *reinterpret_cast<const X8*>(&k_lds[buf][k_at<D>(16 * t + col, 4 * s + g)]);
#pragma unroll
                for (int i = 0; i < QT; ++i) S[i][t] = F::mma32(kf, qf[i][s], S[i][t]);
            }

        float mb[QT], cm[QT];
        bool grow = false;
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            cm[i] = S[i][0][0];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) cm[i] = fmaxf(cm[i], S[i][t][r]);
            grow |= !(cm[i] <= m_run[i]);
        }
        if (__any(grow)) {
#pragma unroll
            for (int i = 0; i < QT; ++i) {
                const float m_new = fmaxf(m_run[i], over_groups(cm[i]));
                const float alpha = __builtin_amdgcn_exp2f((m_run[i] - m_new) * kLog2e);
                l[i] *= alpha;
#pragma unroll
                for (int dd = 0; dd < kDT; ++dd) o[i][dd] *= alpha;
                m_run[i] = m_new;
            }
        }
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            mb[i] = m_run[i] * kLog2e;
            if (__any(m_run[i] < kScaledMax)) {
                const bool low = m_run[i] < kScaledMax;
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float d = S[i][t][r] < m_run[i] ? -INFINITY : S[i][t][r] - m_run[i];
                        S[i][t][r] = low ? d : S[i][t][r];
                    }
                mb[i] = low ? 0.0f : mb[i];
            }
        }

#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
            X8 pb[QT];
#pragma unroll
            for (int i = 0; i < QT; ++i)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(S[i][2 * pr + u][r], kLog2e, -mb[i]));
                        l[i] += pv;
                        pb[i][4 * u + r] = static_cast<T>(pv);
                    }
            // O^T += V^T P^T: lane (col, g) holds V[keys 4 g .. of both tiles][16 dd + col]
            const int vrow = 32 * pr + 4 * g + (col >> 2);
#pragma unroll
            for (int dd = 0; dd < kDT; ++dd) {
                const X4 v0 = lds_read_tr<T>(&v_lds[buf][v_at<D>(vrow, dd) + 4 * (col & 3)]);
                const X4 v1 = lds_read_tr<T>(&v_lds[buf][v_at<D>(vrow + 16, dd) + 4 * (col & 3)]);
                const X8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int i = 0; i < QT; ++i) o[i][dd] = F::mma32(vf, pb[i], o[i][dd]);
            }
        }
        if (more) stash_kv(buf ^ 1);  // last read before the previous barrier
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const float sum = sum_groups(l[i]);
        if (qi[i] < N) {
            T* orow = static_cast<T*>(p.out) + int64_t(b) * p.os[0] + int64_t(h) * p.os[1] + int64_t(qi[i]) * p.os[2];
#pragma unroll
            for (int dd = 0; dd < kDT; ++dd) {
                X4 ov;
#pragma unroll
                for (int r = 0; r < 4; ++r) ov[r] = static_cast<T>(o[i][dd][r] / sum);
                *reinterpret_cast<X4*>(orow + 16 * dd + 4 * g) = ov;
            }
        }
    }
}

template <typename T, int D, int QT>
void launch_q(const Params& p, int mode, int32_t mask_dtype, hipStream_t s) {
    const uint32_t qblocks = static_cast<uint32_t>((p.N + 64 * QT - 1) / (64 * QT));
    const uint32_t chunks = static_cast<uint32_t>(uint64_t(p.B) * uint64_t(p.H) * qblocks);
    const dim3 grid(xcd_launch_count(chunks)), block(kChunkThreads);
    if (mode == 0)
        hipLaunchKernelGGL((swin_attention_chunk_kernel<T, D, 0, QT>), grid, block, 0, s, p, mask_dtype, qblocks,
                           chunks);
    else if (mode == 1)
        hipLaunchKernelGGL((swin_attention_chunk_kernel<T, D, 1, QT>), grid, block, 0, s, p, mask_dtype, qblocks,
                           chunks);
    else
        hipLaunchKernelGGL((swin_attention_chunk_kernel<T, D, 2, QT>), grid, block, 0, s, p, mask_dtype, qblocks,
                           chunks);
}

// Two query tiles per wave at head dim 32 without a mask tensor, for long
// windows that 128-query blocks do not pad more than 64-query blocks, or that
// are long enough for it not to matter.  fp16, 6 heads, us with one / two
// tiles: 128 windows of 512 108 to 113 / 106, 40 of 1,000 121 / 112, 24 of
// 1,536 199 / 177; but 336 of 128 26.6 / 29.2, 96 of 448 64 / 71, 72 of 576
// 80 / 84.  Elsewhere the second tile's registers cost more than the shared
// fragments give: 203 / 221 at 128 windows of 512 with a mask tensor, 129 /
// 184 at head dim 128 (125 windows of 343); at head dim 64 they spill.
template <typename T, int D>
void launch_dim(const Params& p, int mode, int32_t mask_dtype, hipStream_t s) {
    const bool even = (p.N + 63) / 64 % 2 == 0;
    if (D == 32 && mode != 1 && p.N >= (even ? 512 : 700))
        launch_q<T, D, D == 32 ? 2 : 1>(p, mode, mask_dtype, s);
    else
        launch_q<T, D, 1>(p, mode, mask_dtype, s);
}

template <typename T>
void launch_type(const Params& p, int Dh, int mode, int32_t mask_dtype, hipStream_t s) {
    if (Dh == 32)
        launch_dim<T, 32>(p, mode, mask_dtype, s);
    else if (Dh == 64)
        launch_dim<T, 64>(p, mode, mask_dtype, s);
    else
        launch_dim<T, 128>(p, mode, mask_dtype, s);
}

}  // namespace

void launch_chunk(const Params& p, int Dh, int kmask, int32_t dtype, int32_t mask_dtype, hipStream_t s) {
    const int mode = kmask == kMaskRegion ? 2 : kmask == kNoMask ? 0 : 1;
    if (dtype == CRUMPET_DTYPE_F16)
        launch_type<_Float16>(p, Dh, mode, mask_dtype, s);
    else
        launch_type<__bf16>(p, Dh, mode, mask_dtype, s);
}

}  // namespace attn
}  // namespace crumpet
