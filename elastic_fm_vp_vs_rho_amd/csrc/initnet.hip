// Kernels of the learned moment-tensor / location initializer (a 1-D
// convolutional network trained and run on the GPU).  No counterpart in the
// reference, whose inversions start from a fixed moment tensor.
//
// BF16 operands are uint16 upper halves of IEEE float32 (round to nearest
// even); products accumulate in FP32 on the matrix cores with gfx950's
// v_mfma_f32_16x16x32_bf16 (one 32-deep k step per instruction).
// Activations are (C, B, L).
#include "common.hpp"
#include "efm_initnet.h"

namespace efm {
namespace net {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                      // round to nearest even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((unsigned)h << 16); }

inline int blocks_for(long long n, int bs) {
    long long b = (n + bs - 1) / bs;
    return (int)(b > 65535LL * 8 ? 65535LL * 8 : b);
}

// ---- GEMM ---------------------------------------------------------------------
// Block tile 64 (m) x 64 (n), k-slab 32, 4 waves; wave w owns the 32 x 32
// quadrant (w/2, w%2) as 2 x 2 MFMA 16x16 tiles, one 16x16x32 instruction per
// tile and k-slab.  Operands are staged through LDS as [row][k] (A) and
// [col][k] (B) so that each lane reads its 8 consecutive k values as one
// 16-byte word.  MFMA 16x16x32 lane layout: lane l supplies A[l%16][8(l/16)+j]
// and B[8(l/16)+j][l%16], j < 8, and receives D[4(l/16)+j][l%16], j < 4.
constexpr int GBM = 64, GBN = 64, GBK = 32, GLD = GBK + 8;

__device__ __forceinline__ f32x4 mfma_1(const uint4 &a, const uint4 &b, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8 *>(&a),
                                                   *reinterpret_cast<const bf16x8 *>(&b), acc, 0, 0, 0);
}

// The 2 x 2 MFMA tiles of one k-slab from the LDS stages.
__device__ __forceinline__ void mfma_slab(const uint16_t *As, const uint16_t *Bs, int wm, int wn,
                                          int lane, f32x4 (&acc)[2][2]) {
    bf16x8 a[2], b[2];
    const int ko = 8 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        a[i] = *reinterpret_cast<const bf16x8 *>(&As[(wm + 16 * i + (lane & 15)) * GLD + ko]);
        b[i] = *reinterpret_cast<const bf16x8 *>(&Bs[(wn + 16 * i + (lane & 15)) * GLD + ko]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
}

__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const uint16_t *__restrict__ A,
                                              long long sam, long long sak,
                                              const uint16_t *__restrict__ B, long long sbk,
                                              long long sbn, float *__restrict__ C, long long ldc,
                                              const float *__restrict__ bias,
                                              uint16_t *__restrict__ Cb, int epi) {
    __shared__ __attribute__((aligned(16))) uint16_t As[GBM * GLD];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[GBN * GLD];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const bool a_kfast = (sak == 1);  // choose the staging order that coalesces
    const bool b_nfast = (sbn == 1);
    for (int k0 = 0; k0 < K; k0 += GBK) {
#pragma unroll
        for (int i = 0; i < (GBM * GBK) / 256; ++i) {
            const int idx = t + 256 * i;
            int r, k;
            if (a_kfast) { r = idx >> 5; k = idx & 31; } else { r = idx & 63; k = idx >> 6; }
            const int gm = m0 + r, gk = k0 + k;
            uint16_t v = 0;
            if (gm < M && gk < K) v = A[(long long)gm * sam + (long long)gk * sak];
            As[r * GLD + k] = v;
        }
#pragma unroll
        for (int i = 0; i < (GBN * GBK) / 256; ++i) {
            const int idx = t + 256 * i;
            int c, k;
            if (b_nfast) { c = idx & 63; k = idx >> 6; } else { c = idx >> 5; k = idx & 31; }
            const int gn = n0 + c, gk = k0 + k;
            uint16_t v = 0;
            if (gn < N && gk < K) v = B[(long long)gk * sbk + (long long)gn * sbn];
            Bs[c * GLD + k] = v;
        }
        __syncthreads();
        mfma_slab(As, Bs, wm, wn, lane, acc);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                const int col = n0 + wn + 16 * j + (lane & 15);
                if (row < M && col < N) {
                    float v = acc[i][j][r];
                    if (epi >= 1) v += bias[row];
                    if (epi == 1) v = fmaxf(v, 0.f);
                    const long long o = (long long)row * ldc + col;
                    C[o] = v;
                    if (Cb) Cb[o] = f2bf(v);
                }
            }
}

// Vectorised variant for operands whose contiguous dimension has unit stride
// (A: k-fast when AK, else m-fast; B: n-fast when BN, else k-fast) and whose
// other stride is a multiple of 8 elements: each thread moves one 16-byte
// vector (8 values) of each operand per k-slab, and the next slab is fetched
// into registers while the matrix cores work on the current one (two LDS
// stages).  Vectors that cross the M/N/K edge fall back to element loads.
template <bool AK, bool BN>
__device__ __forceinline__ void gemm_fetch(uint4 &va, uint4 &vb, int t, int m0, int n0, int k0,
                                           int M, int N, int K, const uint16_t *__restrict__ A,
                                           long long lda, const uint16_t *__restrict__ B,
                                           long long ldb) {
    // A: AK -> row m = t/4, k = 8(t%4); else k = t/8, m = 8(t%8)
    {
        const int r = AK ? (t >> 2) : ((t & 7) << 3), k = AK ? ((t & 3) << 3) : (t >> 3);
        const int gm = m0 + r, gk = k0 + k;
        if (AK ? (gm < M && gk + 7 < K) : (gk < K && gm + 7 < M)) {
            va = *reinterpret_cast<const uint4 *>(AK ? A + (long long)gm * lda + gk
                                                     : A + (long long)gk * lda + gm);
        } else {
            uint16_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int mm = AK ? gm : gm + i, kk = AK ? gk + i : gk;
                e[i] = (mm < M && kk < K) ? (AK ? A[(long long)mm * lda + kk] : A[(long long)kk * lda + mm])
                                          : (uint16_t)0;
            }
            va = make_uint4(e[0] | (unsigned)e[1] << 16, e[2] | (unsigned)e[3] << 16,
                            e[4] | (unsigned)e[5] << 16, e[6] | (unsigned)e[7] << 16);
        }
    }
    // B: BN -> k = t/8, n = 8(t%8); else n = t/4, k = 8(t%4)
    {
        const int c = BN ? ((t & 7) << 3) : (t >> 2), k = BN ? (t >> 3) : ((t & 3) << 3);
        const int gn = n0 + c, gk = k0 + k;
        if (BN ? (gk < K && gn + 7 < N) : (gn < N && gk + 7 < K)) {
            vb = *reinterpret_cast<const uint4 *>(BN ? B + (long long)gk * ldb + gn
                                                     : B + (long long)gn * ldb + gk);
        } else {
            uint16_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int nn = BN ? gn + i : gn, kk = BN ? gk : gk + i;
                e[i] = (nn < N && kk < K) ? (BN ? B[(long long)kk * ldb + nn] : B[(long long)nn * ldb + kk])
                                          : (uint16_t)0;
            }
            vb = make_uint4(e[0] | (unsigned)e[1] << 16, e[2] | (unsigned)e[3] << 16,
                            e[4] | (unsigned)e[5] << 16, e[6] | (unsigned)e[7] << 16);
        }
    }
}

template <bool AK, bool BN>
__device__ __forceinline__ void gemm_stage(uint16_t *As, uint16_t *Bs, const uint4 &va,
                                           const uint4 &vb, int t) {
    if (AK) {
        *reinterpret_cast<uint4 *>(&As[(t >> 2) * GLD + ((t & 3) << 3)]) = va;
    } else {
        const uint16_t *e = reinterpret_cast<const uint16_t *>(&va);
        const int m = (t & 7) << 3, k = t >> 3;
#pragma unroll
        for (int i = 0; i < 8; ++i) As[(m + i) * GLD + k] = e[i];
    }
    if (BN) {
        const uint16_t *e = reinterpret_cast<const uint16_t *>(&vb);
        const int n = (t & 7) << 3, k = t >> 3;
#pragma unroll
        for (int i = 0; i < 8; ++i) Bs[(n + i) * GLD + k] = e[i];
    } else {
        *reinterpret_cast<uint4 *>(&Bs[(t >> 2) * GLD + ((t & 3) << 3)]) = vb;
    }
}

constexpr int kGemmLds = 2 * (GBM + GBN) * GLD;      // 16-bit words
template <bool AK, bool BN>
__device__ __forceinline__ void gemm_tile(uint16_t *sm, int t, int m0, int n0, int M, int N, int K,
                                          const uint16_t *__restrict__ A, long long lda,
                                          const uint16_t *__restrict__ B, long long ldb, float *__restrict__ C,
                                          long long ldc, const float *__restrict__ bias, uint16_t *__restrict__ Cb,
                                          int epi) {
    const int lane = t & 63, w = t >> 6;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    uint4 va, vb;
    gemm_fetch<AK, BN>(va, vb, t, m0, n0, 0, M, N, K, A, lda, B, ldb);
    gemm_stage<AK, BN>(sm, sm + 2 * GBM * GLD, va, vb, t);
    __syncthreads();
    int cur = 0;
    for (int k0 = 0; k0 < K; k0 += GBK) {
        const bool more = k0 + GBK < K;
        if (more) gemm_fetch<AK, BN>(va, vb, t, m0, n0, k0 + GBK, M, N, K, A, lda, B, ldb);
        mfma_slab(sm + cur * GBM * GLD, sm + (2 * GBM + cur * GBN) * GLD, wm, wn, lane, acc);
        if (more) gemm_stage<AK, BN>(sm + (cur ^ 1) * GBM * GLD, sm + (2 * GBM + (cur ^ 1) * GBN) * GLD, va, vb, t);
        __syncthreads();
        cur ^= 1;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                const int col = n0 + wn + 16 * j + (lane & 15);
                if (row < M && col < N) {
                    float v = acc[i][j][r];
                    if (epi >= 1) v += bias[row];
                    if (epi == 1) v = fmaxf(v, 0.f);
                    const long long o = (long long)row * ldc + col;
                    C[o] = v;
                    if (Cb) Cb[o] = f2bf(v);
                }
            }
}

template <bool AK, bool BN>
__global__ __launch_bounds__(256) void k_gemm_vec(int M, int N, int K,
                                                  const uint16_t *__restrict__ A, long long lda,
                                                  const uint16_t *__restrict__ B, long long ldb,
                                                  float *__restrict__ C, long long ldc,
                                                  const float *__restrict__ bias,
                                                  uint16_t *__restrict__ Cb, int epi) {
    __shared__ __attribute__((aligned(16))) uint16_t sm[kGemmLds];
    gemm_tile<AK, BN>(sm, threadIdx.x, blockIdx.y * GBM, blockIdx.x * GBN, M, N, K, A, lda, B, ldb, C, ldc, bias, Cb, epi);
}

// ---- strided 1-D convolutions as implicit GEMMs ------------------------------------
// The forward pass and the weight gradient multiply against the im2col matrix
// without storing it: a lane owns one output sample (b, l) and reads the KS <= 9 taps of
// a channel with one 16-byte load and one of 2 bytes, from the place nearest to them
// inside the row (shifted afterwards where that is not their own), and the tile goes to
// LDS as [column][k].  A slab's loads are issued before the MFMAs of the slab before
// it.  Few wide loads also keep the kernels short: they run for one to six slabs, and
// unrolled over 72 two-byte loads they spent their time fetching instructions (the four
// layers of 64 examples, 192 channels of 1024: forward 33 + 3 x 13 us that way, 19 + 3 x 7.9
// now, against 192 us of im2col, GEMM and flatten over the stored matrix).
struct ConvShape {
    int C, B, L, M, ks, stride, pad, Lout;
};

__device__ __forceinline__ uint4 pack8(const uint16_t *e) {
    return make_uint4(e[0] | (unsigned)e[1] << 16, e[2] | (unsigned)e[3] << 16, e[4] | (unsigned)e[5] << 16,
                      e[6] | (unsigned)e[7] << 16);
}

// 8 consecutive k of row m of A (lda apart), zero past M and kend.
__device__ __forceinline__ uint4 conv_a8(const uint16_t *__restrict__ A, int lda, int M, int m, int k, int kend,
                                         bool avec) {
    if (avec && m < M && k + 7 < kend) return *reinterpret_cast<const uint4 *>(A + (long long)m * lda + k);
    unsigned long long h[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll 1
        for (int u = 0; u < 4; ++u)
            if (m < M && k + 4 * i + u < kend)
                h[i] |= (unsigned long long)A[(long long)m * lda + k + 4 * i + u] << 16 * u;
    return make_uint4((unsigned)h[0], (unsigned)(h[0] >> 32), (unsigned)h[1], (unsigned)(h[1] >> 32));
}

// The taps of output sample (b, l): pos = l·stride - pad is the input of tap 0.
struct Taps {
    int first;                     // offset in x's channel of the 8 samples read
    int shift;                     // pos - (sample of `first` in its row): 0 inside the row
    int ninth;                     // offset of tap 8, kept inside the row
    bool has9;
};
__device__ __forceinline__ Taps conv_taps(const ConvShape &q, int b, int l) {
    const int pos = l * q.stride - q.pad, start = min(max(pos, 0), q.L - 8);
    return Taps{b * q.L + start, pos - start, b * q.L + min(max(pos + 8, 0), q.L - 1),
                (unsigned)(pos + 8) < (unsigned)q.L};
}
// Taps 0-7 from the 8 samples read at Taps::first: element i moves to i - shift, zeros in.
__device__ __forceinline__ uint4 shift_taps(uint4 v, int shift) {
    unsigned long long lo = v.x | (unsigned long long)v.y << 32, hi = v.z | (unsigned long long)v.w << 32;
    if (shift <= -8 || shift >= 8) return make_uint4(0, 0, 0, 0);
    const int n = 16 * (shift < 0 ? -shift : shift);      // bits
    if (shift > 0) {
        const int m = n & 63;
        const unsigned long long a = n >= 64 ? hi : lo, b = n >= 64 ? 0 : hi;
        lo = m ? a >> m | b << (64 - m) : a;
        hi = b >> m;
    } else if (shift < 0) {
        const int m = n & 63;
        const unsigned long long a = n >= 64 ? lo : hi, b = n >= 64 ? 0 : lo;
        hi = m ? a << m | b >> (64 - m) : a;
        lo = b << m;
    }
    return make_uint4((unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32));
}
typedef unsigned u32x4u __attribute__((ext_vector_type(4), aligned(2)));
// Element k of 8 packed ones and a ninth.
__device__ __forceinline__ uint16_t tap_of(const uint4 &v, uint16_t n, int k) {
    const unsigned w = k < 2 ? v.x : k < 4 ? v.y : k < 6 ? v.z : v.w;
    return k == 8 ? n : (uint16_t)(k & 1 ? w >> 16 : w);
}

// y[m, b·Lout + l] = max(Σ W·x + bias, 0); yb = bf16(y) at the same place, or flattened
// for the dense head (yb[(m·Lout + l)·B + b]).  Block tile 64 x 64, slabs of 32
// channels: a multiple of 32 k for any KS, so that the MFMA steps and the bits are those
// of the GEMM over the stored matrix.  16 waves, two whole channels of a slab and one MFMA
// tile each: the kernel lasts two to six slabs, so it is the few hundred instructions and the
// loads' latency of a slab that it waits for (first layer and the others, us: 4 waves
// 22.7 and 10.7, 8 waves 19.6 and 8.7, 16 waves 18.8 and 7.9; with two slabs' loads in
// flight 19.2 and 8.4).
constexpr int kFwdWaves = 16, kFwdThreads = 64 * kFwdWaves;
template <int KS>
struct FwdSlab {
    static constexpr int NA = (64 * 4 * KS + kFwdThreads - 1) / kFwdThreads;
    uint4 a[NA], x[2];
    uint16_t x9[2];
};
template <int KS>
__global__ __launch_bounds__(kFwdThreads) void k_conv_fwd(ConvShape q, const uint16_t *__restrict__ x,
                                                          const uint16_t *__restrict__ W,
                                                          const float *__restrict__ bias, float *__restrict__ y,
                                                          uint16_t *__restrict__ yb, int flat, int avec) {
    constexpr int SLAB = 32 * KS, LD = SLAB + 8, NA = FwdSlab<KS>::NA;
    static_assert(kFwdWaves * 2 == 32, "two channels of a slab to a wave");
    __shared__ __attribute__((aligned(16))) uint16_t As[64 * LD], Bs[64 * LD];
    const int N = q.B * q.Lout, K = q.C * KS, BL = q.B * q.L;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = (w >> 2) * 16, wn = (w & 3) * 16;
    const int n = min(n0 + lane, N - 1), b = n / q.Lout;      // lanes past the last column repeat it
    const Taps tp = conv_taps(q, b, n - b * q.Lout);
    const bool edge = __any(tp.shift != 0 || !tp.has9);
    auto fetch = [&](FwdSlab<KS> &f, int c0) __attribute__((always_inline)) {
        if (c0 >= q.C) return;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint16_t *p = x + (long long)min(c0 + 2 * w + j, q.C - 1) * BL;
            const u32x4u v = *reinterpret_cast<const u32x4u *>(p + tp.first);
            f.x[j] = make_uint4(v.x, v.y, v.z, v.w);
            f.x9[j] = KS > 8 ? p[tp.ninth] : (uint16_t)0;
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int j = t + kFwdThreads * i, row = j / (4 * KS), kv = (j - row * (4 * KS)) * 8;
            if (row < 64) f.a[i] = conv_a8(W, K, q.M, m0 + row, c0 * KS + kv, K, avec);
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    FwdSlab<KS> f;
    fetch(f, 0);
#pragma unroll 1
    for (int c0 = 0; c0 < q.C; c0 += 32) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (edge) {
                f.x[j] = shift_taps(f.x[j], tp.shift);
                if (!tp.has9) f.x9[j] = 0;
            }
            if (c0 + 2 * w + j >= q.C) { f.x[j] = make_uint4(0, 0, 0, 0); f.x9[j] = 0; }
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int j = t + kFwdThreads * i, row = j / (4 * KS), kv = (j - row * (4 * KS)) * 8;
            if (row < 64) *reinterpret_cast<uint4 *>(&As[row * LD + kv]) = f.a[i];
        }
#pragma unroll
        for (int i = 0; i < KS; ++i)
            *reinterpret_cast<unsigned *>(&Bs[lane * LD + 2 * KS * w + 2 * i]) =
                tap_of(f.x[2 * i / KS], f.x9[2 * i / KS], 2 * i % KS) |
                (unsigned)tap_of(f.x[(2 * i + 1) / KS], f.x9[(2 * i + 1) / KS], (2 * i + 1) % KS) << 16;
        __syncthreads();
        fetch(f, c0 + 32);
        const int ko = 8 * (lane >> 4);
#pragma unroll 3
        for (int kk = 0; kk < SLAB; kk += 32)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                *reinterpret_cast<const bf16x8 *>(&As[(wm + (lane & 15)) * LD + kk + ko]),
                *reinterpret_cast<const bf16x8 *>(&Bs[(wn + (lane & 15)) * LD + kk + ko]), acc, 0, 0, 0);
        __syncthreads();
    }
    const int col = n0 + wn + (lane & 15);
    if (col >= N) return;
    const int bb = col / q.Lout, ll = col - bb * q.Lout;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 4 * (lane >> 4) + r;
        if (row >= q.M) continue;
        const float v = fmaxf(acc[r] + bias[row], 0.f);
        const long long o = (long long)row * N + col;
        y[o] = v;
        yb[flat ? ((long long)row * q.Lout + ll) * q.B + bb : o] = f2bf(v);
    }
}

// dW[m, c·ks + tap] = Σ_(b, l) dp[m, b·Lout + l]·x[c, b, l·stride + tap - pad].  A block makes
// 32 rows x 16 channels of one tap in one pass over (b, l), slabs of 256 samples: the sum
// of an entry stays one accumulator over rising 32-deep MFMA steps, as in the product with
// the stored matrix, since another order moves the last bit of a gradient, and Adam's
// first steps turn that into other BF16 weights.  Waves 0 and 1 multiply, a row tile each;
// 2 and 3 put the next slab's dp into the other of two LDS buffers, whole rows at a time,
// and 4 to 7 its 16 channels, a sample to a lane, so that every lane's tap is in the row or
// not for all channels at once.  Three slabs of loads are in flight.  What binds it is the
// vector memory path of a CU, the taps' 2-byte loads above all (0.4 of 0.8 us a slab): 32 rows
// a block for 64 (the first layer's chain of 64 slabs 92 -> 63 us on 216 CUs; blocks of 16
// rows go twice to a CU, 101), dp in whole rows instead of MFMA fragments 63 -> 56.  Four
// layers of 64 examples: 87 us against 278 of 64 x 64 tiles over the stored matrix, its
// im2col not counted.
constexpr int kDwSlab = 256, kDwLd = kDwSlab + 8, kDwThreads = 512, kDwRows = 32;
constexpr int kDwLds = 2 * (16 + kDwRows) * kDwLd;                // 16-bit words
template <bool AVEC>
__device__ __forceinline__ void conv_dw_tile(uint16_t *Bs, int c0, int tap, int m0, const ConvShape &q,
                                             const uint16_t *__restrict__ dp, int ldp,
                                             const uint16_t *__restrict__ x, float *__restrict__ out) {
    constexpr int AHEAD = AVEC ? 3 : 1, NK = kDwSlab / 32, NA = kDwRows * kDwSlab / 8 / 128;        // slabs of loads in flight
    const int K = q.B * q.Lout, BL = q.B * q.L;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    // slabs, whole rounds of AHEAD: those past the end add nothing, and with no condition on a
    // load the compiler can wait for the oldest one alone
    const int nslab = (K + kDwSlab * AHEAD - 1) / (kDwSlab * AHEAD) * AHEAD;
    if (w >= 4) {
        const int kl = t - 256;
        const uint16_t *px[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) px[j] = x + (long long)min(c0 + j, q.C - 1) * BL;
        uint16_t f[AHEAD][16];
        bool in[AHEAD];
        auto fetch = [&](uint16_t (&g)[16], bool &valid, int i) __attribute__((always_inline)) {
            const int k = min(i, nslab) * kDwSlab + kl, kc = min(k, K - 1), b = kc / q.Lout;
            const int pos = (kc - b * q.Lout) * q.stride - q.pad + tap;
            valid = k < K && (unsigned)pos < (unsigned)q.L;
            const unsigned off = (unsigned)(b * q.L + min(max(pos, 0), q.L - 1));
#pragma unroll
            for (int j = 0; j < 16; ++j) g[j] = px[j][off];
        };
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) fetch(f[d], in[d], d);
#pragma unroll 1
        for (int i = 0; i < nslab; i += AHEAD)
#pragma unroll
            for (int d = 0; d < AHEAD; ++d) {
                uint16_t *B = Bs + ((i + d) & 1) * 16 * kDwLd + kl;
#pragma unroll
                for (int j = 0; j < 16; ++j) B[j * kDwLd] = in[d] ? f[d][j] : (uint16_t)0;
                fetch(f[d], in[d], i + d + AHEAD);
                __syncthreads();
            }
        return;
    }
    uint16_t *As = Bs + 2 * 16 * kDwLd;
    if (w >= 2) {
        // rows of dp, 512 contiguous bytes each
        const int u = t - 128, kk = (u & 31) * 8;
        uint4 a[AHEAD][NA];
        auto load = [&](uint4 (&g)[NA], int i) __attribute__((always_inline)) {
            const int k = min(i, nslab) * kDwSlab + kk;
#pragma unroll
            for (int j = 0; j < NA; ++j) {
                const uint16_t *row = dp + (long long)min(m0 + (u >> 5) + 4 * j, q.M - 1) * ldp;     // past M: not stored
                // a row of whole vectors is in range or past the end as one
                g[j] = AVEC ? *reinterpret_cast<const uint4 *>(row + min(k, K - 8)) : conv_a8(row, K, 1, 0, k, K, false);
            }
        };
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) load(a[d], d);
#pragma unroll 1
        for (int i = 0; i < nslab; i += AHEAD)
#pragma unroll
            for (int d = 0; d < AHEAD; ++d) {
                const bool in = (i + d) * kDwSlab + kk < K;
#pragma unroll
                for (int j = 0; j < NA; ++j)
                    *reinterpret_cast<uint4 *>(As + (((i + d) & 1) * kDwRows + (u >> 5) + 4 * j) * kDwLd + kk) =
                        in ? a[d][j] : make_uint4(0, 0, 0, 0);
                load(a[d], i + d + AHEAD);
                __syncthreads();
            }
        return;
    }
    const int ko = 8 * (lane >> 4);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int i = 0; i < nslab; ++i) {
        __syncthreads();
        const uint16_t *A = As + ((i & 1) * kDwRows + 16 * w + (lane & 15)) * kDwLd + ko;
        const uint16_t *B = Bs + ((i & 1) * 16 + (lane & 15)) * kDwLd + ko;
        uint4 a[NK], v[NK];
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            a[k] = *reinterpret_cast<const uint4 *>(A + 32 * k);
            v[k] = *reinterpret_cast<const uint4 *>(B + 32 * k);
        }
        __builtin_amdgcn_sched_barrier(0);        // all reads before the first product
#pragma unroll
        for (int k = 0; k < NK; ++k) acc = mfma_1(a[k], v[k], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * w + 4 * (lane >> 4) + r, c = c0 + (lane & 15);
        if (m < q.M && c < q.C) out[((long long)m * q.C + c) * q.ks + tap] = acc[r];
    }
}

// The weight gradient's blocks, dw_blocks of them, and behind them those of dcol = Wᵀ·dp
// (its gn tiles along (b, l)): both wait for dp only, and each alone leaves much of the chip
// idle.  Row tiles and taps of 16 channels follow one another on an XCD, whose L2 then holds
// those channels.
__host__ __device__ inline int dw_rows(const ConvShape &q) { return (q.M + kDwRows - 1) / kDwRows; }
__host__ __device__ inline int dw_tiles(const ConvShape &q) { return (q.C + 15) / 16 * q.ks * dw_rows(q); }
template <bool AVEC>
__global__ __launch_bounds__(kDwThreads) void k_conv_back(ConvShape q, const uint16_t *__restrict__ dp, int ldp,
                                                          const uint16_t *__restrict__ x, float *__restrict__ dW,
                                                          int dw_blocks, const uint16_t *__restrict__ W,
                                                          float *__restrict__ dcol, int gn) {
    __shared__ __attribute__((aligned(16))) uint16_t sm[kDwLds > 2 * kGemmLds ? kDwLds : 2 * kGemmLds];
    int b = blockIdx.x;
    if (b < dw_blocks) {
        const int tile = b % 8 * (dw_blocks / 8) + b / 8, rows = dw_rows(q);
        if (tile < dw_tiles(q))
            conv_dw_tile<AVEC>(sm, tile / (rows * q.ks) * 16, tile / rows % q.ks, tile % rows * kDwRows, q, dp, ldp, x,
                               dW);
        return;
    }
    // two tiles of 256 threads; they walk the same number of slabs, so their barriers agree,
    // and waves without a tile leave before the first
    const int K = q.C * q.ks, N = q.B * q.Lout, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    b = 2 * (b - dw_blocks) + g;
    if (b >= gn * ((K + GBM - 1) / GBM)) return;
    gemm_tile<false, true>(sm + g * kGemmLds, threadIdx.x & 255, b / gn * GBM, b % gn * GBN, K, N, q.M, W, K, dp, ldp,
                           dcol, N, nullptr, nullptr, 0);
}

// ---- ReLU backward with the bias gradient --------------------------------------------
// A bias gradient is 256 chains (chain i: the row's values i, i + 256, ... in rising order)
// and a tree over them; the order is kept whatever computes it (see conv_dw_tile).
__device__ __forceinline__ float tree256(float *red, float v) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    return red[0];
}

// dp = dy·(y > 0) of row m = blockIdx.x; `value(m, n)` gives dy.  One block to a row
// (chains null): db[m].  Else gridDim.y = 16 blocks to a row, kChains chains each: their sums
// to chains[256·m ..], added up by k_bias_sums.  64 rows of 16384 / 4096 values through
// col2im: 30 / 25 us in one block a row, 10.8 / 7.4 in blocks of 16 chains (14.9 / 9.4 of
// 32, 23.7 / 14.2 of 64).
constexpr int kChains = 16;
template <typename F>
__device__ __forceinline__ void relu_bias_row(const float *__restrict__ y, uint16_t *__restrict__ dpb,
                                              float *__restrict__ db, float *__restrict__ chains, int N, int ldp,
                                              F value) {
    const int m = blockIdx.x, t = threadIdx.x;
    const long long row = (long long)m * N;
    dpb += (long long)m * ldp;
    if (!chains) {
        __shared__ float red[256];
        float s = 0.f;
#pragma unroll 4
        for (unsigned n = t; n < (unsigned)N; n += 256) {      // N may be within 256 of 2^31
            const float d = value(m, (int)n);
            const float v = y[row + n] > 0.f ? d : 0.f;
            dpb[n] = f2bf(v);
            s += v;
        }
        s = tree256(red, s);
        if (t == 0) db[m] = s;
        return;
    }
    __shared__ float v[64][kChains + 1];    // 64 values of each of the block's chains
    const int i = t % kChains, c = kChains * blockIdx.y + i;
    float s = 0.f;
    for (long long n0 = 0; n0 < N; n0 += 64 * 256) {
#pragma unroll
        for (int jj = 0; jj < kChains / 4; ++jj) {
            const int j = t / kChains + 256 / kChains * jj;
            const long long n = n0 + 256 * j + c;
            const int nc = (int)(n < N ? n : N - 1);         // past the end: computed, not kept
            const float d = value(m, nc);
            const float p = y[row + nc] > 0.f ? d : 0.f;
            v[j][i] = p;
            if (n < N) dpb[n] = f2bf(p);
        }
        __syncthreads();
        if (t < kChains)
#pragma unroll 8
            for (int j = 0; j < 64; ++j)
                if (n0 + 256 * j + c < N) s += v[j][i];
        __syncthreads();
    }
    if (t < kChains) chains[256LL * m + c] = s;
}

// db[m] from the chains of rows m < M, for every bias of the list.
struct BiasList {
    EfmNetBias s[EFM_NET_BIASES];
    int first[EFM_NET_BIASES];        // its first block, a row each
    int n;
};
__global__ __launch_bounds__(256) void k_bias_sums(BiasList l) {
    __shared__ float red[256];
    int j = 0;
    while (j + 1 < l.n && (int)blockIdx.x >= l.first[j + 1]) ++j;
    const int m = blockIdx.x - l.first[j];
    const float s = tree256(red, l.s[j].chains[256LL * m + threadIdx.x]);
    if (threadIdx.x == 0) l.s[j].db[m] = s;
}

// dy (M, N) row-major, or flattened (dy[(m·L + l)·B + b] for n = b·L + l) when L > 0.
__global__ __launch_bounds__(256) void k_relu_bias(const float *__restrict__ dy, const float *__restrict__ y,
                                                   uint16_t *__restrict__ dpb, float *__restrict__ db,
                                                   float *__restrict__ chains, int N, int B, int L, int ldp) {
    relu_bias_row(y, dpb, db, chains, N, ldp, [&](int m, int n) {
        if (L <= 0) return dy[(long long)m * N + n];
        const int b = n / L, l = n - b * L;
        return dy[((long long)m * L + l) * B + b];
    });
}

// dy = the transposed im2col of dcol (see k_col2im) at channel c, n = b·L + j: the taps with
// j + pad - k a multiple of the stride, in rising k, at most T of them (0: any number).
template <int T>
__global__ __launch_bounds__(256) void k_col2im_relu_bias(const float *__restrict__ dcol, const float *__restrict__ y,
                                                          uint16_t *__restrict__ dpb, float *__restrict__ db,
                                                          float *__restrict__ chains, ConvShape q, int ldp) {
    const unsigned ncol = (unsigned)q.B * q.Lout, L = q.L, stride = q.stride;
    relu_bias_row(y, dpb, db, chains, q.B * q.L, ldp, [&](int c, int n) __attribute__((always_inline)) {
        const unsigned b = (unsigned)n / L, j = n - b * L + q.pad;
        int l = j / stride, k = j - l * stride;
        const float *col = dcol + (long long)c * q.ks * ncol + b * q.Lout;
        float s = 0.f;
        if (T == 0) {
            for (; k < q.ks && l >= 0; k += stride, --l)
                if (l < q.Lout) s += col[(long long)k * ncol + l];
            return s;
        }
        // every tap loaded from a place inside the row, counted if it is its own
#pragma unroll
        for (int i = 0; i < T; ++i, k += stride, --l) {
            const float v = col[(long long)min(k, q.ks - 1) * ncol + min(max(l, 0), q.Lout - 1)];
            s += k < q.ks && (unsigned)l < (unsigned)q.Lout ? v : 0.f;
        }
        return s;
    });
}

// ---- the dense head --------------------------------------------------------------------
// Two small products forward and four backward, each a launch of 4 us or more whatever it
// holds: the two forward ones walked their sums slab by slab on one or two blocks (11.4 and
// 6.5 us for 128 x 256 by 64).  Here a block takes 16 examples through both layers,
// its waves 16 rows each, eight slabs of a row's sum in flight at once: 8.5 us; and one
// block takes the loss and the last layer back to the hidden layer: 10.3 us in place of six
// launches (25 us).  MFMA steps of 32 k in rising order, as the general product's.
__host__ __device__ constexpr int up32(int n) { return (n + 31) & ~31; }

__global__ __launch_bounds__(512) void k_head_fwd(int B, int flat, int hidden, int nout,
                                                  const uint16_t *__restrict__ X, const uint16_t *__restrict__ F1,
                                                  const float *__restrict__ c1, const uint16_t *__restrict__ F2,
                                                  const float *__restrict__ c2, float *__restrict__ z,
                                                  uint16_t *__restrict__ zb, float *__restrict__ out, int xvec,
                                                  int avec1, int avec2) {
    extern __shared__ __attribute__((aligned(16))) uint16_t sm[];
    const int LX = up32(flat) + 8, LZ = up32(hidden) + 8;
    uint16_t *Xs = sm, *Zs = sm + 16 * LX;                  // [example][k]
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, i = lane & 15, ko = 8 * (lane >> 4);
    const int n0 = blockIdx.x * 16, col = n0 + i;
    for (int k = t; k < 2 * up32(flat); k += 512) {
        const int kk = k >> 1, n = n0 + 8 * (k & 1);
        const uint4 v = kk < flat ? conv_a8(X, B, flat, kk, n, B, xvec) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 8; ++u) Xs[(8 * (k & 1) + u) * LX + kk] = tap_of(v, 0, u);
    }
    for (int k = t; k < 16 * LZ; k += 512) Zs[k] = 0;
    __syncthreads();
    for (int r0 = 16 * w; r0 < hidden; r0 += 128) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        int k0 = 0;
        for (; k0 + 256 <= up32(flat); k0 += 256) {
            uint4 a[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] = conv_a8(F1, flat, hidden, r0 + i, k0 + 32 * u + ko, flat, avec1);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                acc = mfma_1(a[u], *reinterpret_cast<const uint4 *>(&Xs[i * LX + k0 + 32 * u + ko]), acc);
        }
        for (; k0 < up32(flat); k0 += 32)
            acc = mfma_1(conv_a8(F1, flat, hidden, r0 + i, k0 + ko, flat, avec1),
                         *reinterpret_cast<const uint4 *>(&Xs[i * LX + k0 + ko]), acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 4 * (lane >> 4) + r;
            if (row >= hidden || col >= B) continue;
            const float v = fmaxf(acc[r] + c1[row], 0.f);
            z[(long long)row * B + col] = v;
            zb[(long long)row * B + col] = Zs[i * LZ + row] = f2bf(v);
        }
    }
    __syncthreads();
    for (int r0 = 16 * w; r0 < nout; r0 += 128) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int k0 = 0; k0 < up32(hidden); k0 += 32)
            acc = mfma_1(conv_a8(F2, hidden, nout, r0 + i, k0 + ko, hidden, avec2),
                         *reinterpret_cast<const uint4 *>(&Zs[i * LZ + k0 + ko]), acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 4 * (lane >> 4) + r;
            if (row < nout && col < B) out[(long long)row * B + col] = acc[r] + c2[row];
        }
    }
}

// loss = Σ (out - t)²/n and its way back: dF2, dc2, dc1 and bf16(dz·(z > 0)).  One block;
// at most kHeadB examples and 16 outputs.
constexpr int kHeadB = 128;
__global__ __launch_bounds__(512) void k_head_bwd(int B, int hidden, int nout, float inv_n,
                                                  const float *__restrict__ out, const float *__restrict__ tg,
                                                  const float *__restrict__ z, const uint16_t *__restrict__ zb,
                                                  const uint16_t *__restrict__ F2, float *__restrict__ dF2,
                                                  float *__restrict__ dc2, float *__restrict__ dc1,
                                                  uint16_t *__restrict__ dzpb, double *loss, int bvec) {
    constexpr int LM = kHeadB + 8, LN = 40;
    __shared__ __attribute__((aligned(16))) uint16_t Dm[16 * LM], Dn[kHeadB * LN];     // bf16(dout): [o][n], [n][o]
    __shared__ float Df[16][kHeadB];
    __shared__ double red[512];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, i = lane & 15, ko = 8 * (lane >> 4);
    for (int k = t; k < 16 * LM; k += 512) Dm[k] = 0;
    for (int k = t; k < kHeadB * LN; k += 512) Dn[k] = 0;
    __syncthreads();
    double s = 0.0;
    for (int k = t; k < nout * B; k += 512) {
        const int o = k / B, n = k - o * B;
        const float r = out[k] - tg[k];
        s += (double)r * (double)r;
        const float g = 2.f * r * inv_n;
        Df[o][n] = g;
        Dm[o * LM + n] = Dn[n * LN + o] = f2bf(g);
    }
    red[t] = s;
    __syncthreads();
    for (int o = 256; o > 0; o >>= 1) {
        if (t < o) red[t] += red[t + o];
        __syncthreads();
    }
    if (t == 0) *loss = red[0] * (double)inv_n;
    for (int o = w; o < nout; o += 8) {
        float v = (lane < B ? Df[o][lane] : 0.f) + (lane + 64 < B ? Df[o][lane + 64] : 0.f);
        for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
        if (lane == 0) dc2[o] = v;
    }
    for (int r0 = 16 * w; r0 < hidden; r0 += 128) {
        // dF2[:, r0 .. r0+15] = dout · zbᵀ
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int k0 = 0; k0 < up32(B); k0 += 32)
            acc = mfma_1(*reinterpret_cast<const uint4 *>(&Dm[i * LM + k0 + ko]),
                         conv_a8(zb, B, hidden, r0 + i, k0 + ko, B, bvec), acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 4 * (lane >> 4) + r;
            if (o < nout && r0 + i < hidden) dF2[o * hidden + r0 + i] = acc[r];
        }
        // rows r0 .. r0+15 of dz = F2ᵀ · dout
        uint16_t e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            e[u] = ko + u < nout && r0 + i < hidden ? F2[(ko + u) * hidden + r0 + i] : (uint16_t)0;
        const uint4 a = pack8(e);
        float p[kHeadB / 16][4];
#pragma unroll
        for (int j = 0; j < kHeadB / 16; ++j) {
            const int n = 16 * j + i;
            f32x4 dz = {0.f, 0.f, 0.f, 0.f};
            if (16 * j < B) dz = mfma_1(a, *reinterpret_cast<const uint4 *>(&Dn[n * LN + ko]), dz);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = r0 + 4 * (lane >> 4) + r, at = row * B + n;
                p[j][r] = 0.f;
                if (row >= hidden || n >= B) continue;
                p[j][r] = z[at] > 0.f ? dz[r] : 0.f;
                dzpb[at] = f2bf(p[j][r]);
            }
        }
        // the bias gradient's tree over examples: 64 apart, 32, 16, then within the 16 lanes
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = ((p[0][r] + p[4][r]) + (p[2][r] + p[6][r])) + ((p[1][r] + p[5][r]) + (p[3][r] + p[7][r]));
            for (int d = 8; d > 0; d >>= 1) v += __shfl_xor(v, d);
            const int row = r0 + 4 * (lane >> 4) + r;
            if (i == 0 && row < hidden) dc1[row] = v;
        }
    }
}

// ---- elementwise / layout kernels -----------------------------------------------
__global__ void k_cast(const float *__restrict__ x, uint16_t *__restrict__ y, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        y[i] = f2bf(x[i]);
}

__global__ void k_im2col(const uint16_t *__restrict__ x, uint16_t *__restrict__ col, int C, int B,
                         int L, int ks, int stride, int pad, int Lout) {
    const long long ncol = (long long)B * Lout;
    const long long n = (long long)C * ks * ncol;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const long long row = i / ncol, cc = i - row * ncol;
        const int c = (int)(row / ks), k = (int)(row - (long long)c * ks);
        const int b = (int)(cc / Lout), l = (int)(cc - (long long)b * Lout);
        const int p = l * stride + k - pad;
        col[i] = (p >= 0 && p < L) ? x[((long long)c * B + b) * L + p] : (uint16_t)0;
    }
}

__global__ void k_col2im(const float *__restrict__ dcol, float *__restrict__ dx, int C, int B, int L,
                         int ks, int stride, int pad, int Lout) {
    const long long n = (long long)C * B * L;
    const long long ncol = (long long)B * Lout;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int j = (int)(i % L);
        const long long cb = i / L;
        const int b = (int)(cb % B), c = (int)(cb / B);
        float s = 0.f;
        for (int k = 0; k < ks; ++k) {
            const int q = j + pad - k;
            if (q < 0 || q % stride) continue;
            const int l = q / stride;
            if (l >= Lout) continue;
            s += dcol[((long long)c * ks + k) * ncol + (long long)b * Lout + l];
        }
        dx[i] = s;
    }
}

__global__ void k_relu_bwd(const float *__restrict__ dy, const float *__restrict__ y,
                           float *__restrict__ dp, uint16_t *__restrict__ dpb, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const float v = y[i] > 0.f ? dy[i] : 0.f;
        dp[i] = v;
        if (dpb) dpb[i] = f2bf(v);
    }
}

__global__ __launch_bounds__(256) void k_bias_grad(const float *__restrict__ dp,
                                                   float *__restrict__ db, long long N) {
    __shared__ float red[256];
    const float *row = dp + (long long)blockIdx.x * N;
    float s = 0.f;
    for (long long i = threadIdx.x; i < N; i += 256) s += row[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ out,
                                             const float *__restrict__ tg, float *__restrict__ d,
                                             uint16_t *__restrict__ db, double *loss, long long n,
                                             float inv_n) {
    __shared__ double red[256];
    double s = 0.0;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const float r = out[i] - tg[i];
        s += (double)r * (double)r;
        const float g = 2.f * r * inv_n;
        d[i] = g;
        if (db) db[i] = f2bf(g);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0] * (double)inv_n);
}

__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, uint16_t *__restrict__ wb, long long n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
        w[i] = wi;
        if (wb) wb[i] = f2bf(wi);
    }
}

__global__ void k_flatten(const uint16_t *__restrict__ a, uint16_t *__restrict__ X, int C, int B,
                          int L) {
    const long long n = (long long)C * B * L;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        // i indexes X[(c*L + l), b]
        const int b = (int)(i % B);
        const long long f = i / B;
        const int c = (int)(f / L), l = (int)(f - (long long)c * L);
        X[i] = a[((long long)c * B + b) * L + l];
    }
}

__global__ void k_unflatten(const float *__restrict__ dX, float *__restrict__ da, int C, int B,
                            int L) {
    const long long n = (long long)C * B * L;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        // i indexes da[c, b, l]
        const int l = (int)(i % L);
        const long long cb = i / L;
        const int b = (int)(cb % B), c = (int)(cb / B);
        da[i] = dX[((long long)c * L + l) * B + b];
    }
}

// One block per shot: max |g| over the shot's gathers, then the normalised,
// channel-major copy.
__global__ __launch_bounds__(256) void k_pack(const float *__restrict__ g, int ncomp, int ntmax,
                                              int nrec, int L, uint16_t *__restrict__ data,
                                              long long s0) {
    __shared__ float red[256];
    const int s = blockIdx.x;
    const long long per = (long long)ncomp * ntmax * nrec;
    const float *gs = g + (long long)s * per;
    float mx = 0.f;
    for (long long i = threadIdx.x; i < per; i += 256) mx = fmaxf(mx, fabsf(gs[i]));
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    const float inv = red[0] > 0.f ? 1.f / red[0] : 0.f;
    const int C = ncomp * nrec;
    uint16_t *ds = data + (s0 + s) * (long long)C * L;
    const long long n = (long long)C * L;
    for (long long i = threadIdx.x; i < n; i += 256) {
        const int l = (int)(i % L);
        const int c = (int)(i / L);
        const int comp = c / nrec, r = c - comp * nrec;
        ds[i] = f2bf(gs[((long long)comp * ntmax + l) * nrec + r] * inv);
    }
}

// The same with 16-byte copies, for rows of a multiple of 8 samples on 16-byte bases.
__global__ void k_gather_batch8(const uint4 *__restrict__ data, const float *__restrict__ tg, long long ntotal,
                                const int *__restrict__ idx, unsigned B, unsigned C, unsigned L8, int nout,
                                uint4 *__restrict__ x, float *__restrict__ t) {
    const unsigned n = C * B * L8;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned row = i / L8, l = i - row * L8, c = row / B, b = row - c * B;
        const long long e = idx[b];
        x[i] = (e >= 0 && e < ntotal) ? data[(e * C + c) * L8 + l] : make_uint4(0, 0, 0, 0);
    }
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    for (unsigned i = g; i < nout * B; i += gridDim.x * blockDim.x) {
        const unsigned j = i / B, bb = i - j * B;
        const long long eb = idx[bb];
        t[i] = (eb >= 0 && eb < ntotal) ? tg[eb * nout + j] : 0.f;
    }
}

__global__ void k_gather_batch(const uint16_t *__restrict__ data, const float *__restrict__ tg,
                               long long ntotal, const int *__restrict__ idx, int B, int C, int L,
                               int nout, uint16_t *__restrict__ x, float *__restrict__ t) {
    const long long n = (long long)C * B * L;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int l = (int)(i % L);
        const long long cb = i / L;
        const int b = (int)(cb % B), c = (int)(cb / B);
        const long long e = idx[b];
        x[i] = (e >= 0 && e < ntotal) ? data[(e * C + c) * L + l] : (uint16_t)0;
        if (i < (long long)nout * B) {
            const int j = (int)(i / B), bb = (int)(i % B);
            const long long eb = idx[bb];
            t[i] = (eb >= 0 && eb < ntotal) ? tg[eb * nout + j] : 0.f;
        }
    }
}

}  // namespace net
}  // namespace efm

using namespace efm;
using namespace efm::net;

#define NET_CHECK(cond, msg) \
    if (!(cond)) return fail(EFM_E_ARG, msg)

extern "C" int efm_net_cast_bf16(const float *x, uint16_t *y, long long n, void *stream) {
    NET_CHECK(x && y && n >= 0, "efm_net_cast_bf16: bad arguments");
    if (n == 0) return EFM_OK;
    k_cast<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(x, y, n);
    return check_launch("efm_net_cast_bf16");
}

extern "C" int efm_net_gemm(int M, int N, int K, const uint16_t *A, long long sam, long long sak,
                            const uint16_t *B, long long sbk, long long sbn, float *C,
                            long long ldc, const float *bias, uint16_t *Cb, int epilogue,
                            void *stream) {
    NET_CHECK(A && B && C && M > 0 && N > 0 && K > 0, "efm_net_gemm: null pointer or empty shape");
    NET_CHECK(sam >= 0 && sak >= 0 && sbk >= 0 && sbn >= 0 && ldc >= N,
              "efm_net_gemm: bad strides");
    NET_CHECK(epilogue >= 0 && epilogue <= 2, "efm_net_gemm: epilogue must be 0, 1 or 2");
    NET_CHECK(epilogue == 0 || bias, "efm_net_gemm: bias epilogue needs a bias");
    NET_CHECK((M + GBM - 1) / GBM <= 65535, "efm_net_gemm: M too large");
    dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM);
    hipStream_t st = (hipStream_t)stream;
    // vectorised path: unit stride along one dimension of each operand, the
    // other stride a multiple of 8, 16-byte aligned bases
    const bool a_ok = ((sak == 1 && sam % 8 == 0) || (sam == 1 && sak % 8 == 0)) &&
                      ((uintptr_t)A % 16 == 0) && !(sak == 1 && sam == 1 && M > 1 && K > 1);
    const bool b_ok = ((sbn == 1 && sbk % 8 == 0) || (sbk == 1 && sbn % 8 == 0)) &&
                      ((uintptr_t)B % 16 == 0) && !(sbn == 1 && sbk == 1 && N > 1 && K > 1);
    if (a_ok && b_ok) {
        const bool ak = (sak == 1), bn = (sbn == 1);
        const long long lda = ak ? sam : sak, ldb = bn ? sbk : sbn;
        if (ak && bn)
            k_gemm_vec<true, true><<<grid, 256, 0, st>>>(M, N, K, A, lda, B, ldb, C, ldc, bias, Cb, epilogue);
        else if (ak)
            k_gemm_vec<true, false><<<grid, 256, 0, st>>>(M, N, K, A, lda, B, ldb, C, ldc, bias, Cb, epilogue);
        else if (bn)
            k_gemm_vec<false, true><<<grid, 256, 0, st>>>(M, N, K, A, lda, B, ldb, C, ldc, bias, Cb, epilogue);
        else
            k_gemm_vec<false, false><<<grid, 256, 0, st>>>(M, N, K, A, lda, B, ldb, C, ldc, bias, Cb, epilogue);
        return check_launch("efm_net_gemm");
    }
    k_gemm<<<grid, 256, 0, st>>>(M, N, K, A, sam, sak, B, sbk, sbn, C, ldc, bias, Cb, epilogue);
    return check_launch("efm_net_gemm");
}

static bool conv_ok(int C, int B, int L, int ks, int stride, int pad) {
    return C > 0 && B > 0 && L > 0 && ks > 0 && stride > 0 && pad >= 0 && L + 2 * pad >= ks;
}

extern "C" int efm_net_im2col(const uint16_t *x, uint16_t *col, int C, int B, int L, int ks,
                              int stride, int pad, void *stream) {
    NET_CHECK(x && col && conv_ok(C, B, L, ks, stride, pad), "efm_net_im2col: bad arguments");
    const int Lout = (L + 2 * pad - ks) / stride + 1;
    const long long n = (long long)C * ks * B * Lout;
    k_im2col<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(x, col, C, B, L, ks, stride, pad,
                                                                    Lout);
    return check_launch("efm_net_im2col");
}

extern "C" int efm_net_col2im(const float *dcol, float *dx, int C, int B, int L, int ks,
                              int stride, int pad, void *stream) {
    NET_CHECK(dcol && dx && conv_ok(C, B, L, ks, stride, pad), "efm_net_col2im: bad arguments");
    const int Lout = (L + 2 * pad - ks) / stride + 1;
    const long long n = (long long)C * B * L;
    k_col2im<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(dcol, dx, C, B, L, ks, stride,
                                                                    pad, Lout);
    return check_launch("efm_net_col2im");
}

// A convolution the implicit kernels take: at most 9 taps, rows of at least 8 samples,
// 32-bit offsets into x, and launches within a dispatch's limits.
#define EFM_CONV_SIZES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9)
constexpr long long kConvBlocks = 1LL << 22;
static long long dw_blocks(const ConvShape &q) {
    const long long tiles = (q.C + 15LL) / 16 * q.ks * ((q.M + kDwRows - 1) / kDwRows);
    return (tiles + 7) / 8 * 8;
}
static bool conv_shape(ConvShape &q, int C, int B, int L, int M, int ks, int stride, int pad) {
    if (!conv_ok(C, B, L, ks, stride, pad) || M <= 0 || ks > 9 || L < 8) return false;
    const long long lim = 1LL << 31, Lout = (L + 2LL * pad - ks) / stride + 1;
    q = ConvShape{C, B, L, M, ks, stride, pad, (int)Lout};
    return (long long)C * B * L < lim && (long long)C * ks < lim - 1024 && B * Lout < lim - 1024 &&
           L + 2LL * pad + ks < lim && (M + 63LL) / 64 <= 65535 &&
           (B * Lout + 63) / 64 * kFwdThreads <= (long long)UINT32_MAX && dw_blocks(q) < kConvBlocks;
}

extern "C" int efm_net_conv1d(const uint16_t *x, const uint16_t *W, const float *bias, float *y, uint16_t *yb,
                              int C, int B, int L, int M, int ks, int stride, int pad, int flat, void *stream) {
    ConvShape q;
    NET_CHECK(x && W && bias && y && yb && conv_shape(q, C, B, L, M, ks, stride, pad), "efm_net_conv1d: bad arguments");
    const int avec = (C * ks) % 8 == 0 && (uintptr_t)W % 16 == 0;
    const dim3 grid((B * q.Lout + 63) / 64, (M + 63) / 64);
    hipStream_t st = (hipStream_t)stream;
    switch (ks) {
#define EFM_CONV(KS) \
    case KS: k_conv_fwd<KS><<<grid, kFwdThreads, 0, st>>>(q, x, W, bias, y, yb, flat, avec); break;
        EFM_CONV_SIZES(EFM_CONV)
#undef EFM_CONV
    }
    return check_launch("efm_net_conv1d");
}

extern "C" int efm_net_conv1d_fits(int C, int B, int L, int M, int ks, int stride, int pad) {
    ConvShape q;
    return conv_shape(q, C, B, L, M, ks, stride, pad);
}

extern "C" int efm_net_conv1d_back(const uint16_t *dp, const uint16_t *x, const uint16_t *W, float *dW, float *dcol,
                                   int C, int B, int L, int M, int ks, int stride, int pad, int ldp, void *stream) {
    ConvShape q;
    NET_CHECK(dp && x && dW && (W || !dcol) && conv_shape(q, C, B, L, M, ks, stride, pad) && ldp >= B * q.Lout,
              "efm_net_conv1d_back: bad arguments");
    const int K = B * q.Lout, gn = (K + GBN - 1) / GBN;
    const bool avec = K % 8 == 0 && ldp % 8 == 0 && (uintptr_t)dp % 16 == 0;
    // dcol rides along where its product may take 16-byte loads and the launch holds both
    const long long dw = dw_blocks(q), with = dw + ((long long)gn * ((C * ks + GBM - 1) / GBM) + 1) / 2;
    const bool both = dcol && avec && C * ks % 8 == 0 && (uintptr_t)W % 16 == 0 && with < kConvBlocks;
    const long long blocks = both ? with : dw;
    (avec ? k_conv_back<true> : k_conv_back<false>)<<<(unsigned)blocks, kDwThreads, 0, (hipStream_t)stream>>>(
        q, dp, ldp, x, dW, (int)dw, W, dcol, gn);
    if (int rc = check_launch("efm_net_conv1d_back")) return rc;
    if (!dcol || both) return EFM_OK;
    return efm_net_gemm(C * ks, K, M, W, 1, C * ks, dp, ldp, 1, dcol, K, nullptr, nullptr, 0, stream);
}

// Rows of at least 1024 values, fewer of them than fill the chip a block to a row.
extern "C" int efm_net_bias_split(int M, int N) { return M <= 512 && N >= 1024; }

extern "C" int efm_net_bias_sums(const EfmNetBias *biases, int n, void *stream) {
    NET_CHECK(n >= 0 && (biases || n == 0), "efm_net_bias_sums: bad arguments");
    for (int j0 = 0; j0 < n; j0 += EFM_NET_BIASES) {
        BiasList l{};
        long long blocks = 0;
        for (; l.n < EFM_NET_BIASES && j0 + l.n < n; ++l.n) {
            const EfmNetBias &s = biases[j0 + l.n];
            NET_CHECK(s.chains && s.db && s.M > 0, "efm_net_bias_sums: bad bias");
            l.s[l.n] = s;
            l.first[l.n] = (int)blocks;
            blocks += s.M;
            NET_CHECK(blocks < (1LL << 22), "efm_net_bias_sums: too many rows");
        }
        k_bias_sums<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(l);
        if (int rc = check_launch("efm_net_bias_sums")) return rc;
    }
    return EFM_OK;
}

extern "C" int efm_net_relu_bias_backward(const float *dy, const float *y, uint16_t *dpb, float *db, float *chains,
                                          int M, int N, int B, int L, int ldp, void *stream) {
    NET_CHECK(dy && y && dpb && (db || chains) && M > 0 && N > 0 && ldp >= N && (L <= 0 || (B > 0 && (long long)B * L == N)),
              "efm_net_relu_bias_backward: bad arguments");
    k_relu_bias<<<dim3(M, chains ? 256 / kChains : 1), 256, 0, (hipStream_t)stream>>>(dy, y, dpb, db, chains, N, B, L, ldp);
    return check_launch("efm_net_relu_bias_backward");
}

extern "C" int efm_net_col2im_relu_bias(const float *dcol, const float *y, uint16_t *dpb, float *db, float *chains,
                                        int C, int B, int L, int ks, int stride, int pad, int ldp, void *stream) {
    NET_CHECK(dcol && y && dpb && (db || chains) && conv_ok(C, B, L, ks, stride, pad) &&
                  (long long)B * L < (1LL << 31) && ldp >= B * L,
              "efm_net_col2im_relu_bias: bad arguments");
    const ConvShape q{C, B, L, 1, ks, stride, pad, (L + 2 * pad - ks) / stride + 1};
    const int taps = (ks + stride - 1) / stride;
    const auto kernel = taps == 1   ? k_col2im_relu_bias<1>
                        : taps == 2 ? k_col2im_relu_bias<2>
                        : taps == 3 ? k_col2im_relu_bias<3>
                                    : k_col2im_relu_bias<0>;
    kernel<<<dim3(C, chains ? 256 / kChains : 1), 256, 0, (hipStream_t)stream>>>(dcol, y, dpb, db, chains, q, ldp);
    return check_launch("efm_net_col2im_relu_bias");
}

// 16 examples' inputs and hidden values in 64 KB of LDS.
static bool head_fits(int B, int flat, int hidden, int nout) {
    return B > 0 && flat > 0 && hidden > 0 && nout > 0 && (long long)flat + hidden <= 1968 && nout <= 4096 &&
           (long long)B * (hidden > flat ? hidden : flat) < (1LL << 31);
}

extern "C" int efm_net_head_fits(int B, int flat, int hidden, int nout) {
    if (!head_fits(B, flat, hidden, nout)) return 0;
    return B <= kHeadB && nout <= 16 ? 3 : 1;
}

extern "C" int efm_net_head_forward(const uint16_t *X, const uint16_t *F1, const float *c1, const uint16_t *F2,
                                    const float *c2, float *z, uint16_t *zb, float *out, int B, int flat, int hidden,
                                    int nout, void *stream) {
    NET_CHECK(X && F1 && c1 && F2 && c2 && z && zb && out && head_fits(B, flat, hidden, nout),
              "efm_net_head_forward: bad arguments");
    const auto vec = [](const void *p, int ld) { return (int)(ld % 8 == 0 && (uintptr_t)p % 16 == 0); };
    const int lds = 16 * (up32(flat) + 8 + up32(hidden) + 8) * 2;
    k_head_fwd<<<(B + 15) / 16, 512, lds, (hipStream_t)stream>>>(B, flat, hidden, nout, X, F1, c1, F2, c2, z, zb, out,
                                                                 vec(X, B), vec(F1, flat), vec(F2, hidden));
    return check_launch("efm_net_head_forward");
}

extern "C" int efm_net_head_backward(const float *out, const float *target, const float *z, const uint16_t *zb,
                                     const uint16_t *F2, float *dF2, float *dc2, float *dc1, uint16_t *dzpb,
                                     double *loss, int B, int hidden, int nout, float inv_n, void *stream) {
    NET_CHECK(out && target && z && zb && F2 && dF2 && dc2 && dc1 && dzpb && loss && head_fits(B, 1, hidden, nout) &&
              B <= kHeadB && nout <= 16, "efm_net_head_backward: bad arguments");
    k_head_bwd<<<1, 512, 0, (hipStream_t)stream>>>(B, hidden, nout, inv_n, out, target, z, zb, F2, dF2, dc2, dc1, dzpb,
                                                   loss, B % 8 == 0 && (uintptr_t)zb % 16 == 0);
    return check_launch("efm_net_head_backward");
}

extern "C" int efm_net_relu_backward(const float *dy, const float *y, float *dpre,
                                     uint16_t *dpre_b, long long n, void *stream) {
    NET_CHECK(dy && y && dpre && n >= 0, "efm_net_relu_backward: bad arguments");
    if (n == 0) return EFM_OK;
    k_relu_bwd<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(dy, y, dpre, dpre_b, n);
    return check_launch("efm_net_relu_backward");
}

extern "C" int efm_net_bias_grad(const float *dpre, float *db, int M, long long N, void *stream) {
    NET_CHECK(dpre && db && M > 0 && M <= 65535 * 8 && N > 0, "efm_net_bias_grad: bad arguments");
    k_bias_grad<<<M, 256, 0, (hipStream_t)stream>>>(dpre, db, N);
    return check_launch("efm_net_bias_grad");
}

extern "C" int efm_net_mse(const float *out, const float *target, float *dout, uint16_t *dout_b,
                           double *loss, long long n, float inv_n, void *stream) {
    NET_CHECK(out && target && dout && loss && n > 0, "efm_net_mse: bad arguments");
    k_mse<<<blocks_for(n, 256) < 1024 ? blocks_for(n, 256) : 1024, 256, 0, (hipStream_t)stream>>>(
        out, target, dout, dout_b, loss, n, inv_n);
    return check_launch("efm_net_mse");
}

extern "C" int efm_net_adam(float *w, const float *g, float *m, float *v, uint16_t *wb,
                            long long n, float lr, float b1, float b2, float eps, float c1,
                            float c2, void *stream) {
    NET_CHECK(w && g && m && v && n > 0, "efm_net_adam: bad arguments");
    k_adam<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(w, g, m, v, wb, n, lr, b1, b2, eps,
                                                                  c1, c2);
    return check_launch("efm_net_adam");
}

extern "C" int efm_net_flatten(const uint16_t *act, uint16_t *X, int C, int B, int L,
                               void *stream) {
    NET_CHECK(act && X && C > 0 && B > 0 && L > 0, "efm_net_flatten: bad arguments");
    const long long n = (long long)C * B * L;
    k_flatten<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(act, X, C, B, L);
    return check_launch("efm_net_flatten");
}

extern "C" int efm_net_unflatten(const float *dX, float *dact, int C, int B, int L, void *stream) {
    NET_CHECK(dX && dact && C > 0 && B > 0 && L > 0, "efm_net_unflatten: bad arguments");
    const long long n = (long long)C * B * L;
    k_unflatten<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(dX, dact, C, B, L);
    return check_launch("efm_net_unflatten");
}

extern "C" int efm_net_pack_gathers(const float *g, int S, int ncomp, int ntmax, int nrec, int L,
                                    uint16_t *data, long long s0, void *stream) {
    NET_CHECK(g && data && S > 0 && S <= 65535 * 8 && ncomp > 0 && nrec > 0 && L > 0 &&
                  L <= ntmax && s0 >= 0,
              "efm_net_pack_gathers: bad arguments");
    k_pack<<<S, 256, 0, (hipStream_t)stream>>>(g, ncomp, ntmax, nrec, L, data, s0);
    return check_launch("efm_net_pack_gathers");
}

extern "C" int efm_net_gather_batch(const uint16_t *data, const float *targets, long long ntotal,
                                    const int *idx, int B, int C, int L, int nout, uint16_t *x,
                                    float *t, void *stream) {
    NET_CHECK(data && targets && idx && x && t && ntotal > 0 && B > 0 && C > 0 && L > 0 &&
                  nout > 0 && (long long)nout * B <= (long long)C * B * L,
              "efm_net_gather_batch: bad arguments");
    const long long n = (long long)C * B * L;
    if (L % 8 == 0 && (uintptr_t)data % 16 == 0 && (uintptr_t)x % 16 == 0 && n <= (1LL << 31)) {
        // 16 bytes a thread: 31 -> 8.7 us for 64 examples of 192 x 1024
        k_gather_batch8<<<blocks_for(n / 8, 256), 256, 0, (hipStream_t)stream>>>(
            reinterpret_cast<const uint4 *>(data), targets, ntotal, idx, B, C, L / 8, nout,
            reinterpret_cast<uint4 *>(x), t);
        return check_launch("efm_net_gather_batch");
    }
    k_gather_batch<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(data, targets, ntotal, idx,
                                                                          B, C, L, nout, x, t);
    return check_launch("efm_net_gather_batch");
}
