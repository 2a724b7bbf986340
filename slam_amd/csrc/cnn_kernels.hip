// cnn_kernels.hip -- the learned warm start: a small BF16 convnet on MFMA.
//
// Input: 2 x (80x60) depth + intensity, NHWC [N][60][80][4] bf16 in [0, 1]
// (model depth, model intensity, current depth, current intensity).
// Six 3x3 stride-2 convolutions (pad 1) with ReLU, 4 -> 32 -> 64 -> 96 ->
// 128 -> 128 -> 128 channels (60x80 -> 30x40 -> 15x20 -> 8x10 -> 4x5 -> 2x3
// -> 1x2), global average pooling, FC 128 -> 3840 (ReLU) -> 6: a scaled se(3)
// increment (1.0 M parameters).  No counterpart in the reference (its only network is the
// unrelated YOLACT segmenter); the tracker uses the prediction as the initial
// increment of a Gauss-Newton solve.
//
// Every convolution and linear layer is a matrix product on MFMA (bf16
// operands, fp32 accumulation) that gathers its im2col operand as it runs:
// forward Y = im2col(X) W, weight gradient dW = im2col(X)^T dY (split over
// the reduction and summed in a fixed order), input gradient dX =
// col2im(dY W^T).  Master weights and Adam moments are fp32; the products
// read bf16 copies.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "slam_cnn.h"

namespace cnn {

typedef uint16_t bf16;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

__host__ __device__ inline bf16 f2bf(float x)
{
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)(u >> 16);  // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);                              // round to nearest even
    return (bf16)(u >> 16);
}

__host__ __device__ inline float bf2f(bf16 h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// ============================================================= training
// Layers as matrix products on MFMA (bf16 operands, fp32 sums), without
// im2col or col2im in memory: a lane's fragment is 4 consecutive channels of
// one tap, loaded from the activations (or gradients) themselves, which the
// caches hold.  The first operand of a product is the weights, so a lane's
// four results are four consecutive channels of one position: an 8-byte bf16
// store.  Every sum has one order, in 16-deep products ascending through parts
// of a stated length: a rounding that moves a bf16 activation moves a ReLU's
// mask and, through Adam, whole weights (other orders of any sum, the weight
// gradients' too, moved the gradients four steps on by 1 to 8 % in some runs),
// so the order of the sums is part of what a training run reproduces.
//
// Bound by latency and launches: a training step of 256 samples is 23 GFLOP
// (10 us at the card's dense rate) and about 150 MB.  With im2col and col2im
// buffers, 64x64 LDS-staged products, one-thread-per-column sums and 75
// launches it took 2.1 ms, 0.9 ms of it in the sums over partial results; now
// 0.43 ms in 27 launches, with the same bits.
__device__ __forceinline__ v4f mma16(uint2 a, uint2 b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4s, a), __builtin_bit_cast(v4s, b), c, 0, 0,
                                                     0);
}

__device__ __forceinline__ uint2 pack4(const float (&v)[4])
{
    return make_uint2((uint32_t)f2bf(v[0]) | (uint32_t)f2bf(v[1]) << 16,
                      (uint32_t)f2bf(v[2]) | (uint32_t)f2bf(v[3]) << 16);
}

__device__ __forceinline__ float bf_at(uint2 p, int r)
{
    const uint32_t w = r < 2 ? p.x : p.y;
    return bf2f((bf16)((r & 1) ? w >> 16 : w & 0xffffu));
}

// One layer: a 3x3 / stride 2 / pad 1 convolution (TAPS 9) or a linear layer
// (TAPS 1, sizes 1).  Reduction index k = tap * CIN + channel, padded with
// zeros to KP, a multiple of 32.
template <int TAPS_, int CIN_, int COUT_, int HI_ = 1, int WI_ = 1, int HO_ = 1, int WO_ = 1>
struct Layer {
    static constexpr int TAPS = TAPS_, CIN = CIN_, COUT = COUT_, HI = HI_, WI = WI_, HO = HO_, WO = WO_;
    static constexpr int K = TAPS * CIN, KP = (K + 31) / 32 * 32;
};

// Where row m of a layer's im2col matrix starts: sample n, upper left tap (h, w).
struct RowPos {
    int n, h, w;
};

template <class L>
__device__ __forceinline__ RowPos row_pos(int m)
{
    const int n = m / (L::HO * L::WO), p = m - n * (L::HO * L::WO);
    return {n, 2 * (p / L::WO) - 1, 2 * (p % L::WO) - 1};
}

// Elements k..k+7 (k a multiple of 8) of a row of im2col(X), 0 outside the
// image and the reduction.  Loads go to a valid address and are selected
// after, so that several are in flight.
template <class L>
__device__ __forceinline__ uint4 patch8(const bf16* __restrict__ X, const RowPos& r, int k, bool live)
{
    if constexpr (L::TAPS == 1) {
        const uint4 v = *(const uint4*)(X + (size_t)r.n * L::CIN + k);
        return live ? v : make_uint4(0, 0, 0, 0);
    } else if constexpr (L::CIN % 8 == 0) {
        const int tap = k / L::CIN, c = k - tap * L::CIN;
        const int h = r.h + tap / 3, w = r.w + tap % 3;
        const bool ok = live && k < L::K && h >= 0 && h < L::HI && w >= 0 && w < L::WI;
        const uint4 v = *(const uint4*)(X + (ok ? ((size_t)(r.n * L::HI + h) * L::WI + w) * L::CIN + c : 0));
        return ok ? v : make_uint4(0, 0, 0, 0);
    } else {
        static_assert(L::CIN == 4, "channels come in groups of 4 or 8");
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int tap = k / 4 + q;
            const int h = r.h + tap / 3, w = r.w + tap % 3;
            const bool ok = live && tap < L::TAPS && h >= 0 && h < L::HI && w >= 0 && w < L::WI;
            const uint2 v = *(const uint2*)(X + (ok ? ((size_t)(r.n * L::HI + h) * L::WI + w) * 4 : 0));
            o[2 * q] = ok ? v.x : 0u;
            o[2 * q + 1] = ok ? v.y : 0u;
        }
        return make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// The same for k..k+3 (k a multiple of 4).
template <class L>
__device__ __forceinline__ uint2 patch4(const bf16* __restrict__ X, const RowPos& r, int k)
{
    if constexpr (L::TAPS == 1) return *(const uint2*)(X + (size_t)r.n * L::CIN + k);
    const int tap = k / L::CIN, c = k - tap * L::CIN;
    const int h = r.h + tap / 3, w = r.w + tap % 3;
    const bool ok = k < L::K && h >= 0 && h < L::HI && w >= 0 && w < L::WI;
    const uint2 v = *(const uint2*)(X + (ok ? ((size_t)(r.n * L::HI + h) * L::WI + w) * L::CIN + c : 0));
    return ok ? v : make_uint2(0, 0);
}

// Forward: Y = relu(im2col(X) W + b) as bf16, and for the last convolution the
// mean over its two positions (GAP); or fp32 sums without ReLU, eight columns
// per row and the first kHeadOut of them to `user` (HEAD).
//   Wf: the weights in fragment order (store_weight): k step s, column tile j, lane
//   L hold W[16 s + 4 (L >> 4) + q][16 j + (L & 15)], q = 0..3.
// A wave forms RT row tiles x CT column tiles, in chunks of `chunk` (an even
// number of) k steps whose sums are added in order.  KS = 1: a workgroup is
// four waves of different rows; KS > 1, for the layers with few rows, long
// reductions and several chunks: the KS waves share the chunks, of which there
// are at most PARTS.  A row's sums do not depend on the rows beside it.
enum Out { kRelu, kReluGap, kHead };
constexpr int kHeadOut = 6, kHeadPad = 8;

template <class L, int RT, int CT, int KS, Out OUT, int PARTS>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS) void k_fwd(const bf16* __restrict__ X,
                                                                 const bf16* __restrict__ Wf,
                                                                 const float* __restrict__ bias, int M, int chunk,
                                                                 bf16* __restrict__ Y, bf16* __restrict__ gap,
                                                                 float* __restrict__ out, float* __restrict__ user)
{
    constexpr int NT = (L::COUT + 15) / 16, STEPS = L::KP / 16, UNROLL = STEPS % 6 == 0 ? 6 : (STEPS % 4 == 0 ? 4 : 2);
    static_assert(NT % CT == 0 && STEPS % 2 == 0, "whole column groups and pairs of steps");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (KS == 1 ? (int)blockIdx.x * 4 + wave : (int)blockIdx.x) * RT * 16, col0 = blockIdx.y * CT;
    RowPos pos[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) pos[i] = row_pos<L>(min(row0 + 16 * i + (lane & 15), M - 1));
    v4f acc[RT][CT];
    const auto clear = [&] {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    // U steps from s: all their loads are issued before the first product
    const auto steps = [&](int s, auto U) {
        uint2 w[U.value][CT], x[U.value][RT];
#pragma unroll
        for (int q = 0; q < U.value; ++q) {
#pragma unroll
            for (int j = 0; j < CT; ++j)
                w[q][j] = *(const uint2*)(Wf + ((size_t)((s + q) * NT + col0 + j) * 64 + lane) * 4);
#pragma unroll
            for (int i = 0; i < RT; ++i) x[q][i] = patch4<L>(X, pos[i], 16 * (s + q) + 4 * (lane >> 4));
        }
#pragma unroll
        for (int q = 0; q < U.value; ++q)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = mma16(w[q][j], x[q][i], acc[i][j]);
    };
    const auto run = [&](int s, int end) {
        for (; s + UNROLL <= end; s += UNROLL) steps(s, std::integral_constant<int, UNROLL>{});
        for (; s < end; s += 2) steps(s, std::integral_constant<int, 2>{});
    };
    const auto store = [&](int i, int j, v4f a) {
        const int m = row0 + 16 * i + (lane & 15), n = (col0 + j) * 16 + 4 * (lane >> 4);
        if constexpr (OUT == kHead) {
            if (m >= M) return;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (n + r >= kHeadPad) break;
                const float v = a[r] + bias[n + r];
                out[(size_t)m * kHeadPad + n + r] = v;
                if (user && n + r < kHeadOut) user[(size_t)m * kHeadOut + n + r] = v;
            }
        } else {
            const float4 b = *(const float4*)(bias + n);
            const float v[4] = {fmaxf(a[0] + b.x, 0.0f), fmaxf(a[1] + b.y, 0.0f), fmaxf(a[2] + b.z, 0.0f),
                                fmaxf(a[3] + b.w, 0.0f)};
            const uint2 y = pack4(v);
            if (m < M) *(uint2*)(Y + (size_t)m * L::COUT + n) = y;
            if constexpr (OUT == kReluGap) {
                static_assert(L::HO * L::WO == 2, "a sample's positions are two neighbouring lanes");
                float g[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float f = bf_at(y, r);
                    g[r] = (f + __shfl_xor(f, 1, 64)) / 2.0f;
                }
                if (m < M && (lane & 1) == 0) *(uint2*)(gap + (size_t)(m >> 1) * L::COUT + n) = pack4(g);
            }
        }
    };
    if constexpr (KS == 1) {
        v4f sum[RT][CT];
        for (int s = 0; s < STEPS; s += chunk) {
            clear();
            run(s, min(STEPS, s + chunk));
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) sum[i][j] = s ? sum[i][j] + acc[i][j] : acc[i][j];
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) store(i, j, sum[i][j]);
    } else {
        __shared__ v4f part[PARTS][RT * CT][64];
        const int parts = (STEPS + chunk - 1) / chunk;
        for (int p = wave; p < parts; p += KS) {
            clear();
            run(p * chunk, min(STEPS, (p + 1) * chunk));
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) part[p][i * CT + j][lane] = acc[i][j];
        }
        __syncthreads();
        for (int t = wave; t < RT * CT; t += KS) {
            v4f a = part[0][t][lane];
            for (int p = 1; p < parts; ++p) a += part[p][t][lane];
            store(t / CT, t % CT, a);
        }
    }
}

constexpr int kLayers = 8;

// The bf16 weights in every form that a kernel reads: as they lie in the
// parameter vector, in k_fwd's (and the inference's) fragment order, and for
// the layers with an input gradient in k_dgrad's (the same for the transposed
// weights: row tile r, k step s, lane L hold W[16 r + (L & 15)][16 s + 4 (L >> 4)
// + q]).  Whoever writes a weight writes them all, so no call has to know
// whether they are up to date, and a captured graph stays right when its
// weights change.  first, n: a layer's weights [n / ld][ld] in the vector,
// multiples of 64, so a wave's 64 parameters lie in one tensor.  k_fwd's
// columns from ld to the tile's end stay 0.
struct WeightForms {
    bf16* flat;
    bf16 *fwd[kLayers], *dgrad[kLayers];        // dgrad: null without an input gradient
    int first[kLayers], n[kLayers], ld[kLayers];
};

// Whole waves of consecutive i, the first a multiple of 64.
__device__ __forceinline__ void store_weight(const WeightForms& F, int i, bf16 b)
{
    F.flat[i] = b;
    const int base = __builtin_amdgcn_readfirstlane(i & ~63);
#pragma unroll
    for (int l = 0; l < kLayers; ++l) {
        if ((unsigned)(base - F.first[l]) >= (unsigned)F.n[l]) continue;
        const int e = i - F.first[l], ld = F.ld[l], k = e / ld, c = e - k * ld, tile = (k >> 4) * ((ld + 15) >> 4) + (c >> 4);
        F.fwd[l][(tile * 64 + ((k >> 2) & 3) * 16 + (c & 15)) * 4 + (k & 3)] = b;
        if (F.dgrad[l]) F.dgrad[l][(tile * 64 + ((c >> 2) & 3) * 16 + (k & 15)) * 4 + (c & 3)] = b;
    }
}

// A copy of the input, which backward needs (the caller's may be gone by then)
// and which gives it the loads' alignment.  n: fragments of 8.
__global__ __launch_bounds__(256) void k_copy_input(const bf16* __restrict__ x, int n, bf16* __restrict__ to)
{
    const bool wide = ((uintptr_t)x & 15) == 0;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        const bf16* p = x + (size_t)e * 8;
        uint4 v;
        if (wide) v = *(const uint4*)p;
        else v = make_uint4(p[0] | (uint32_t)p[1] << 16, p[2] | (uint32_t)p[3] << 16,
                            p[4] | (uint32_t)p[5] << 16, p[6] | (uint32_t)p[7] << 16);
        *(uint4*)(to + (size_t)e * 8) = v;
    }
}

// Input gradient, through the ReLU of the layer below: dZl = (Yl > 0) ? dX : 0
// with dX[h][w] = sum over the taps (kh, kw) with h = 2 ho - 1 + kh, w = 2 wo
// - 1 + kw of dZ[ho][wo] W[tap]^T; dZl as bf16 for the products and as fp32
// (dZf) for the bias gradient.  Positions of one
// parity of (h, w) meet the same 1, 2, 2 or 4 taps, so each parity is a
// product of its own (blockIdx.z, the longest first).  For the linear layer
// above the average pooling (TAPS 1) both of a sample's two positions take
// half its gradient; it has few tiles and a long reduction, so its waves are
// workgroups of their own, on as many CUs.  A wave forms RT row tiles x CT
// column tiles; each tap's product is summed by itself, then the taps in order.
//   Wp: the weights in k_dgrad's fragment order (store_weight).
template <class L, int RT, int CT>
__global__ __launch_bounds__(L::TAPS == 1 ? 64 : 256) void k_dgrad(const bf16* __restrict__ dZ,
                                                                   const bf16* __restrict__ Wp,
                                                                   const bf16* __restrict__ Yl, int N,
                                                                   bf16* __restrict__ dZl, float* __restrict__ dZf)
{
    constexpr int WAVES = L::TAPS == 1 ? 1 : 4;
    constexpr int NT = L::CIN / 16, STEPS = L::COUT / 16, U = STEPS > 8 ? 24 : STEPS;
    static_assert(L::CIN % 16 == 0 && NT % CT == 0 && STEPS % U == 0, "whole tiles");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = ((int)blockIdx.x * WAVES + wave) * RT * 16, col0 = blockIdx.y * CT;
    const int ph = L::TAPS == 1 ? 0 : 1 - (int)(blockIdx.z >> 1), pw = L::TAPS == 1 ? 0 : 1 - (int)(blockIdx.z & 1);
    const int hc = (L::HI - ph + 1) / 2, wc = (L::WI - pw + 1) / 2;
    const int M = L::TAPS == 1 ? N : N * hc * wc;
    int n[RT], hh[RT], ww[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int m = min(row0 + 16 * i + (lane & 15), M - 1);
        if (L::TAPS == 1) {
            n[i] = m;
            hh[i] = ww[i] = 0;
        } else {
            n[i] = m / (hc * wc);
            const int p = m - n[i] * (hc * wc);
            hh[i] = p / wc;
            ww[i] = p - hh[i] * wc;
        }
    }
    v4f sum[RT][CT];
    for (int a = 0; a <= ph; ++a)
        for (int b = 0; b <= pw; ++b) {
            // kh = 1 (even rows) or 0, 2; the output row it meets
            const int kh = ph ? 2 * a : 1, kw = pw ? 2 * b : 1;
            const int tap = L::TAPS == 1 ? 0 : 3 * kh + kw;
            const int dh = ph && a == 0, dw = pw && b == 0;
            size_t at[RT];
            bool ok[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int ho = hh[i] + dh, wo = ww[i] + dw;
                ok[i] = ho < L::HO && wo < L::WO;
                at[i] = ok[i] ? ((size_t)(n[i] * L::HO + ho) * L::WO + wo) * L::COUT : 0;
            }
            const bf16* wt = Wp + ((size_t)(tap * NT + col0) * STEPS * 64 + lane) * 4;
            v4f acc[RT][CT];
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
            for (int s = 0; s < STEPS; s += U) {
                uint2 w[U][CT], x[U][RT];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    const int c = 16 * (s + q) + 4 * (lane >> 4);
#pragma unroll
                    for (int j = 0; j < CT; ++j) w[q][j] = *(const uint2*)(wt + (size_t)(j * STEPS + s + q) * 256);
#pragma unroll
                    for (int i = 0; i < RT; ++i) {
                        const uint2 v = *(const uint2*)(dZ + at[i] + c);
                        x[q][i] = ok[i] ? v : make_uint2(0, 0);
                    }
                }
#pragma unroll
                for (int q = 0; q < U; ++q)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
#pragma unroll
                        for (int j = 0; j < CT; ++j) acc[i][j] = mma16(w[q][j], x[q][i], acc[i][j]);
            }
            // a tap beyond the image adds nothing
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) sum[i][j] = a + b ? sum[i][j] + acc[i][j] : acc[i][j];
        }
    // mask and store
    const auto store = [&](int i, int j, v4f a) {
        const bool live = row0 + 16 * i + (lane & 15) < M;
        const int ch = (col0 + j) * 16 + 4 * (lane >> 4);
        constexpr int POS = L::TAPS == 1 ? 2 : 1;
#pragma unroll
        for (int p = 0; p < POS; ++p) {
            const size_t o = L::TAPS == 1
                                 ? (size_t)(2 * n[i] + p) * L::CIN + ch
                                 : ((size_t)(n[i] * L::HI + 2 * hh[i] + ph) * L::WI + 2 * ww[i] + pw) * L::CIN + ch;
            const uint2 y = *(const uint2*)(Yl + o);
            float g[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                g[r] = live && bf_at(y, r) > 0.0f ? (L::TAPS == 1 ? a[r] / 2.0f : a[r]) : 0.0f;
            }
            if (live) {
                *(uint2*)(dZl + o) = pack4(g);
                *(float4*)(dZf + o) = make_float4(g[0], g[1], g[2], g[3]);
            }
        }
    };
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) store(i, j, sum[i][j]);
}

// Weight gradient: dW = im2col(X)^T dZ over the rows of split blockIdx.z
// (rows_per of them), to out[split][KP][COUT].  The reduction runs over rows,
// so both operands go through LDS transposed: a thread loads 4 rows x 8
// channels and writes 8 four-row columns of 8 bytes; the next chunk's loads
// fly behind the products.  A workgroup forms 64 reduction rows x BN columns,
// each wave 16 rows.
constexpr int kWgTile = 64, kWgChunk = 64, kWgLd = kWgChunk + 8;

__device__ __forceinline__ void transpose_store(const uint4 (&v)[4], bf16* to)
{
    const uint32_t r[4][4] = {{v[0].x, v[0].y, v[0].z, v[0].w},
                              {v[1].x, v[1].y, v[1].z, v[1].w},
                              {v[2].x, v[2].y, v[2].z, v[2].w},
                              {v[3].x, v[3].y, v[3].z, v[3].w}};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const uint32_t sel = (q & 1) ? 0x07060302u : 0x05040100u;
        *(uint2*)(to + q * kWgLd) = make_uint2(__builtin_amdgcn_perm(r[1][q >> 1], r[0][q >> 1], sel),
                                               __builtin_amdgcn_perm(r[3][q >> 1], r[2][q >> 1], sel));
    }
}

template <class L, int BN>
__global__ __launch_bounds__(256) void k_wgrad(const bf16* __restrict__ X, const bf16* __restrict__ dZ, int M,
                                               int rows_per, float* __restrict__ out)
{
    constexpr int NT = BN / 16, XU = kWgChunk / 4 * (kWgTile / 8), ZU = kWgChunk / 4 * (BN / 8);
    static_assert(L::COUT % BN == 0 && ZU <= 256 && XU <= 256, "a thread stages one unit of each operand");
    __shared__ __align__(16) bf16 Xs[kWgTile][kWgLd];
    __shared__ __align__(16) bf16 Zs[BN][kWgLd];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int k0 = blockIdx.x * kWgTile, n0 = blockIdx.y * BN;
    const int mbeg = blockIdx.z * rows_per, mend = min(M, mbeg + rows_per);
    const int xk = (t % (kWgTile / 8)) * 8, xm = t / (kWgTile / 8) * 4;
    const int u = 255 - t;                              // the other end's threads stage dZ
    const int zn = (u % (BN / 8)) * 8, zm = u / (BN / 8) * 4;
    uint4 xv[4], zv[4];
    const auto load = [&](int m0) {
        if (t < XU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + xm + r;
                xv[r] = patch8<L>(X, row_pos<L>(min(m, M - 1)), k0 + xk, m < mend && k0 + xk < L::KP);
            }
        }
        if (u < ZU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + zm + r;
                const uint4 v = *(const uint4*)(dZ + (size_t)min(m, M - 1) * L::COUT + n0 + zn);
                zv[r] = m < mend ? v : make_uint4(0, 0, 0, 0);
            }
        }
    };
    v4f acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    load(mbeg);
    for (int m0 = mbeg; m0 < mend; m0 += kWgChunk) {
        if (t < XU) transpose_store(xv, &Xs[xk][xm]);
        if (u < ZU) transpose_store(zv, &Zs[zn][zm]);
        __syncthreads();
        if (m0 + kWgChunk < mend) load(m0 + kWgChunk);
#pragma unroll
        for (int s = 0; s < kWgChunk; s += 16) {
            const int q = s + 4 * (lane >> 4);
            const uint2 x = *(const uint2*)&Xs[wave * 16 + (lane & 15)][q];
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = mma16(*(const uint2*)&Zs[j * 16 + (lane & 15)][q], x, acc[j]);
        }
        __syncthreads();
    }
    const int k = k0 + wave * 16 + (lane & 15);
    if (k >= L::KP) return;
    float* o = out + ((size_t)blockIdx.z * L::KP + k) * L::COUT + n0 + 4 * (lane >> 4);
#pragma unroll
    for (int j = 0; j < NT; ++j) *(v4f*)(o + 16 * j) = acc[j];
}

// The head's gradients: the weighted squared error over the first kHeadOut
// outputs, loss = sum_j w_j (O - T)^2 and dO = 2 w_j (O - T) / N; and dZ1 =
// (H1 > 0) ? dO W2^T : 0; both as bf16 and, for the biases, fp32.  A workgroup
// takes 16 samples (blockIdx.y) x 256 hidden units, four tiles a wave.
constexpr int kHeadChunk = 16;
struct LossWeights {
    float w[kHeadOut];
};

__global__ __launch_bounds__(256) void k_head_bwd(const float* __restrict__ O, const float* __restrict__ T,
                                                  LossWeights lw, int N, int H, const bf16* __restrict__ h1,
                                                  const bf16* __restrict__ W2, float* __restrict__ loss,
                                                  bf16* __restrict__ dob, float* __restrict__ dof,
                                                  bf16* __restrict__ dz1, float* __restrict__ dz1f)
{
    __shared__ __align__(8) bf16 db[kHeadChunk][kHeadPad];
    const int r0 = blockIdx.y * kHeadChunk, rows = min(kHeadChunk, N - r0);
    if (threadIdx.x < kHeadChunk)
        for (int q = 0; q < kHeadPad; ++q) db[threadIdx.x][q] = 0;
    if ((int)threadIdx.x < rows) {
        const int n = r0 + threadIdx.x;
        float l = 0.0f;
        for (int q = 0; q < kHeadPad; ++q) {
            float g = 0.0f;
            if (q < kHeadOut) {
                const float e = O[(size_t)n * kHeadPad + q] - T[(size_t)n * kHeadOut + q];
                l += lw.w[q] * e * e;
                g = 2.0f * lw.w[q] * e / (float)N;
                db[threadIdx.x][q] = f2bf(g);
            }
            if (blockIdx.x == 0) {
                dob[(size_t)n * kHeadPad + q] = f2bf(g);
                dof[(size_t)n * kHeadPad + q] = g;
            }
        }
        if (loss && blockIdx.x == 0) loss[n] = l;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, g4 = lane >> 4;
    const int n = r0 + (lane & 15);
    const uint2 x = g4 < 2 ? *(const uint2*)&db[lane & 15][4 * g4] : make_uint2(0, 0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int unit0 = (int)blockIdx.x * 256 + ((threadIdx.x >> 6) * 4 + q) * 16;
        if (unit0 >= H) break;                            // whole tiles: H is a multiple of 16
        const uint2 v = *(const uint2*)(W2 + (size_t)(unit0 + (lane & 15)) * kHeadPad + 4 * (g4 & 1));
        const v4f a = mma16(g4 < 2 ? v : make_uint2(0, 0), x, v4f{0.f, 0.f, 0.f, 0.f});
        if (n >= N) continue;
        const size_t o = (size_t)n * H + unit0 + 4 * g4;
        const uint2 y = *(const uint2*)(h1 + o);
        float g[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) g[r] = bf_at(y, r) > 0.0f ? a[r] : 0.0f;
        *(uint2*)(dz1 + o) = pack4(g);
        *(float4*)(dz1f + o) = make_float4(g[0], g[1], g[2], g[3]);
    }
}

// The head's weight gradient H1^T dO: 16 hidden units a wave, the samples in
// chunks of `chunk` (a multiple of 16) whose sums are added in order.
__global__ __launch_bounds__(256) void k_head_wgrad(const bf16* __restrict__ h1, const bf16* __restrict__ dob, int N,
                                                    int H, int chunk, float* __restrict__ out)
{
    const int lane = threadIdx.x & 63, col = lane & 15, g4 = lane >> 4;
    const int unit0 = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * 16;
    if (unit0 >= H) return;
    v4f sum = v4f{0.f, 0.f, 0.f, 0.f};
    for (int n0 = 0; n0 < N; n0 += chunk) {
        const int end = min(N, n0 + chunk);
        v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
        for (int n = n0; n < end; n += 16) {
            uint32_t a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int m = n + 4 * g4 + q, mc = min(m, N - 1);
                const uint32_t h = h1[(size_t)mc * H + unit0 + col], d = dob[(size_t)mc * kHeadPad + (col & 7)];
                a[q] = m < end ? h : 0u;
                b[q] = m < end && col < kHeadPad ? d : 0u;
            }
            acc = mma16(make_uint2(a[0] | a[1] << 16, a[2] | a[3] << 16),
                        make_uint2(b[0] | b[1] << 16, b[2] | b[3] << 16), acc);
        }
        sum = n0 ? sum + acc : acc;
    }
    if (col < kHeadPad)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(size_t)(unit0 + 4 * g4 + r) * kHeadPad + col] = sum[r];
}

// Column sums of every layer's fp32 gradients (the biases'), in one launch: a
// thread adds the rows of one chunk and column in order, 32 loads in flight.
constexpr int kSumJobs = 2 * kLayers;
struct ColJobs {
    const float* G[kLayers];
    float* part[kLayers];                       // [chunks][N]
    int M[kLayers], N[kLayers], rows[kLayers], chunks[kLayers], first[kLayers];
    int count;
};

__global__ __launch_bounds__(64) void k_colsum(ColJobs J)
{
    int s = 0;
    while (s + 1 < J.count && (int)blockIdx.x >= J.first[s + 1]) ++s;
    const int i = ((int)blockIdx.x - J.first[s]) * 64 + threadIdx.x, N = J.N[s];
    if (i >= J.chunks[s] * N) return;
    const int c = i / N, n = i - c * N;
    const int r0 = c * J.rows[s], r1 = min(J.M[s], r0 + J.rows[s]);
    const float* G = J.G[s] + n;
    float a = 0.0f;
    for (int r = r0; r < r1; r += 32) {
        float v[32];
#pragma unroll
        for (int q = 0; q < 32; ++q) v[q] = G[(size_t)min(r + q, r1 - 1) * N];
#pragma unroll
        for (int q = 0; q < 32; ++q) a = r + q < r1 ? a + v[q] : a;
    }
    J.part[s][i] = a;
}

// Every gradient's sum over its partial results, in order, in one launch: a
// value a thread, 16 loads in flight.
struct SumJobs {
    const float* part[kSumJobs];
    float* dst[kSumJobs];
    int parts[kSumJobs], n[kSumJobs], first[kSumJobs];   // values per part; first workgroup
    int count;
};

__global__ __launch_bounds__(64) void k_sum_parts(SumJobs J)
{
    int s = 0;
    while (s + 1 < J.count && (int)blockIdx.x >= J.first[s + 1]) ++s;
    const int i = ((int)blockIdx.x - J.first[s]) * 64 + threadIdx.x, n = J.n[s], parts = J.parts[s];
    if (i >= n) return;
    const float* p = J.part[s] + i;
    float a = 0.0f;
    for (int z = 0; z < parts; z += 16) {
        float v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = p[(size_t)min(z + q, parts - 1) * n];
#pragma unroll
        for (int q = 0; q < 16; ++q) a = z + q < parts ? a + v[q] : a;
    }
    J.dst[s][i] = a;
}

// Adam with decoupled weight decay on fp32 master weights; writes the bf16
// copies that the products read.  Entries with mask 0 (reduction padding)
// stay 0.  n: a multiple of 64.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, WeightForms F,
                                              const uint8_t* __restrict__ mask, int n, float lr, float b1, float b2,
                                              float eps, float bc1, float bc2, float wd)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float pi = 0.0f;
    if (!mask || mask[i]) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float upd = (mi / bc1) / (sqrtf(vi / bc2) + eps);
        pi = p[i] * (1.0f - lr * wd) - lr * upd;
    }
    p[i] = pi;
    store_weight(F, i, f2bf(pi));
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ a, int n, WeightForms F)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) store_weight(F, i, f2bf(a[i]));
}

// Network input from frame data at twice the input resolution (2W x 2H):
// each channel is the mean of the valid values of a 2x2 block (depth valid
// when positive and finite), depth in metres / 5 clamped to [0, 1], intensity
// / 255.  Channels: model depth (float metres), model intensity, current
// depth (uint16 millimetres), current intensity.
__global__ __launch_bounds__(256) void k_prepare(const float* __restrict__ dA, const uint8_t* __restrict__ iA,
                                                 const uint16_t* __restrict__ dB, const uint8_t* __restrict__ iB,
                                                 int Nb, int W, int H, size_t frame_stride, bf16* __restrict__ X)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= Nb * W * H) return;
    const int n = i / (W * H), p = i - n * (W * H);
    const int y = p / W, x = p - y * W;
    const int W2 = 2 * W;
    const size_t base = (size_t)n * frame_stride;
    float sa = 0.f, sb = 0.f, ia = 0.f, ib = 0.f;
    int ca = 0, cb = 0;
    for (int dy = 0; dy < 2; ++dy)
        for (int dx = 0; dx < 2; ++dx) {
            const size_t q = base + (size_t)(2 * y + dy) * W2 + (2 * x + dx);
            const float za = dA[q];
            if (za > 0.0f && za < 1e30f) { sa += za; ++ca; }
            const float zb = (float)dB[q] * 0.001f;
            if (zb > 0.0f) { sb += zb; ++cb; }
            ia += (float)iA[q];
            ib += (float)iB[q];
        }
    float v[4];
    v[0] = ca ? fminf(sa / (float)ca / 5.0f, 1.0f) : 0.0f;
    v[1] = ia / (4.0f * 255.0f);
    v[2] = cb ? fminf(sb / (float)cb / 5.0f, 1.0f) : 0.0f;
    v[3] = ib / (4.0f * 255.0f);
    for (int c = 0; c < 4; ++c) X[(size_t)i * 4 + c] = f2bf(v[c]);
}

}  // namespace cnn

namespace slam {
void cnn_launch_prepare(const float* depth_a, const uint8_t* image_a, const uint16_t* depth_b, const uint8_t* image_b,
                        int n, size_t frame_stride, void* x, hipStream_t s)
{
    hipLaunchKernelGGL(cnn::k_prepare, dim3((unsigned)((n * 80 * 60 + 255) / 256)), dim3(256), 0, s, depth_a, image_a,
                       depth_b, image_b, n, 80, 60, frame_stride, (cnn::bf16*)x);
}
}  // namespace slam

namespace cnn {

// ============================================================= network
struct ConvSpec {
    int cin, cout, hi, wi, ho, wo;
};
constexpr int kConvs = 6;
const ConvSpec kSpec[kConvs] = {{4, 32, 60, 80, 30, 40},  {32, 64, 30, 40, 15, 20},  {64, 96, 15, 20, 8, 10},
                                {96, 128, 8, 10, 4, 5},   {128, 128, 4, 5, 2, 3},  {128, 128, 2, 3, 1, 2}};
constexpr int kFc1In = 128, kFc1Out = 3840, kOut = 6, kOutPad = 8;

struct Param {
    size_t off, n;
};

}  // namespace cnn

using namespace cnn;

struct cnn_net_s {
    int max_batch = 0;
    hipStream_t stream = nullptr;    // null: the legacy default stream
    // parameters (flat): per conv W [Kp][Cout] + b [Cout]; fc1 W [128][3840] + b; fc2 W [3840][8] + b [8]
    Param convW[kConvs], convB[kConvs], fc1W, fc1B, fc2W, fc2B;
    int Kp[kConvs];
    size_t nparam = 0;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    bf16* pb = nullptr;
    WeightForms forms{};             // where the bf16 weights go
    // the split inference head: pooled features, per-workgroup FC2 partials
    // and the per-sample arrival tickets (back to 0 after every launch)
    int infer_split = 1;
    float *infer_gap = nullptr, *infer_part = nullptr;
    unsigned int* infer_ticket = nullptr;
    uint8_t* mask = nullptr;
    int step = 0;
    // a copy of the last forward's input (the caller's may be gone before
    // cnn_backward) and its activations, sized for max_batch
    bf16* x = nullptr;
    bf16* y[kConvs] = {};
    bf16 *gap = nullptr, *h1 = nullptr;
    float* out = nullptr;            // [N][8]
    // backward scratch: gradients before the activations, partial sums
    bf16 *dz[kConvs] = {}, *dz1 = nullptr, *dob = nullptr;
    float *dzf[kConvs] = {}, *dz1f = nullptr, *dof = nullptr, *part = nullptr;
    std::vector<void*> allocs;
};

namespace {

int fail(hipError_t e, const char* what)
{
    fprintf(stderr, "slam_cnn: %s failed: %s\n", what, hipGetErrorString(e));
    return CNN_ERR_HIP;
}

#define CK(x)                                \
    do {                                     \
        hipError_t e_ = (x);                 \
        if (e_ != hipSuccess) return fail(e_, #x); \
    } while (0)

template <class T>
int dalloc(cnn_net_s* c, T** p, size_t n)
{
    CK(hipMalloc((void**)p, n * sizeof(T) + 16));
    c->allocs.push_back(*p);
    return CNN_OK;
}

int launch_check(const char* what)
{
    hipError_t e = hipPeekAtLastError();
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(e, what);
    }
    return CNN_OK;
}

inline dim3 g1(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

// ---- the layers of the training pass, and their tiles
using Conv0 = Layer<9, 4, 32, 60, 80, 30, 40>;
using Conv1 = Layer<9, 32, 64, 30, 40, 15, 20>;
using Conv2 = Layer<9, 64, 96, 15, 20, 8, 10>;
using Conv3 = Layer<9, 96, 128, 8, 10, 4, 5>;
using Conv4 = Layer<9, 128, 128, 4, 5, 2, 3>;
using Conv5 = Layer<9, 128, 128, 2, 3, 1, 2>;
using Fc1 = Layer<1, kFc1In, kFc1Out>;
using Fc2 = Layer<1, kFc1Out, kOutPad>;
static_assert(kOut == kHeadOut && kOutPad == kHeadPad, "the head's outputs");

// The rows of a weight gradient's parts: up to 512 of 512 rows or more over
// the layer's 64x64 output tiles.
constexpr int wgrad_max_splits(int kp, int cout) { return std::max(1, 512 / std::max(1, kp * cout / 4096)); }

inline int wgrad_rows(int M, int kp, int cout)
{
    const int splits = std::min(wgrad_max_splits(kp, cout), std::max(1, M / 512));
    return cdiv(cdiv(M, splits), 32) * 32;
}

template <class L>
constexpr size_t wgrad_part_elems()
{
    return (size_t)wgrad_max_splits(L::KP, L::COUT) * L::KP * L::COUT;
}

// The chunks of a bias gradient's rows.
inline int col_chunks(int M) { return std::min(256, std::max(1, M / 64)); }

// Workgroups along the rows of k_dgrad's largest parity class.
template <class L, int RT>
int dgrad_blocks(int N)
{
    return L::TAPS == 1 ? cdiv(N, 16 * RT) : cdiv(N * ((L::HI + 1) / 2) * ((L::WI + 1) / 2), 64 * RT);
}

// The chunks of a forward layer's reduction (k steps of 16 each; an even
// number): one, unless the layer has few 64x64 output tiles, then at most
// K / 128, aiming at 64 tiles and chunks.  For inference-sized batches (N <=
// 64) it is chosen from one sample's rows, so a sample's output, bit for bit,
// does not depend on the batch the sample runs in; training batches choose
// from all rows.
template <class L>
int fwd_chunk(int N)
{
    const int rows = L::HO * L::WO, tiles = cdiv(N <= 64 ? rows : N * rows, 64) * cdiv(L::COUT, 64);
    const int splits = tiles >= 64 ? 1 : std::max(1, std::min(64 / tiles, L::KP / 128));
    return cdiv(cdiv(L::KP, splits), 32) * 2;
}

template <class L, int RT, int CT, int KS, Out OUT, int PARTS = 1>
void launch_fwd(cnn_net_s* c, int layer, const bf16* X, int N, const float* bias, bf16* Y, bf16* gap = nullptr,
                float* out = nullptr, float* user = nullptr)
{
    static_assert(KS == 1 || L::KP / 128 <= PARTS, "fwd_chunk's chunks fit the kernel's LDS");
    const int M = N * L::HO * L::WO;
    const dim3 grid(cdiv(M, (KS == 1 ? 64 : 16) * RT), cdiv(L::COUT, 16) / CT);
    hipLaunchKernelGGL((k_fwd<L, RT, CT, KS, OUT, PARTS>), grid, dim3(KS == 1 ? 256 : 64 * KS), 0, c->stream, X,
                       c->forms.fwd[layer], bias, M, fwd_chunk<L>(N), Y, gap, out, user);
}

// The partial sums of one backward pass, taken from c->part in order.
struct Parts {
    cnn_net_s* c;
    SumJobs jobs{};
    ColJobs cols{};
    size_t used = 0;
    int blocks = 0, col_blocks = 0;

    float* take(size_t n)
    {
        float* p = c->part + used;
        used += n;
        return p;
    }
    // dst = the sum of `parts` parts of n values at p
    void sum(const float* p, int parts, int n, float* dst)
    {
        const int q = jobs.count++;
        jobs.part[q] = p;
        jobs.dst[q] = dst;
        jobs.parts[q] = parts;
        jobs.n[q] = n;
        jobs.first[q] = blocks;
        blocks += cdiv(n, 64);
    }
    // dst = the column sums of G [M][N]
    void columns(const float* G, int M, int N, float* dst)
    {
        const int q = cols.count++, chunks = col_chunks(M);
        cols.G[q] = G;
        cols.part[q] = take((size_t)chunks * N);
        cols.M[q] = M;
        cols.N[q] = N;
        cols.rows[q] = cdiv(M, chunks);
        cols.chunks[q] = chunks;
        cols.first[q] = col_blocks;
        col_blocks += cdiv(chunks * N, 64);
        sum(cols.part[q], chunks, N, dst);
    }
};

template <class L, int BN>
void launch_wgrad(Parts& w, const bf16* X, const bf16* dZ, int M, float* dst)
{
    const int kt = cdiv(L::K, kWgTile), rows_per = wgrad_rows(M, L::KP, L::COUT), splits = cdiv(M, rows_per);
    float* out = splits == 1 ? dst : w.take((size_t)splits * L::KP * L::COUT);
    hipLaunchKernelGGL((k_wgrad<L, BN>), dim3(kt, L::COUT / BN, splits), dim3(256), 0, w.c->stream, X, dZ, M,
                       rows_per, out);
    if (splits > 1) w.sum(out, splits, L::KP * L::COUT, dst);
}

template <class L, int RT, int CT>
void launch_dgrad(Parts& w, const bf16* dZ, const bf16* W, const bf16* Yl, int N, bf16* dZl, float* dZf, float* dbias)
{
    const int classes = L::TAPS == 1 ? 1 : 4, blocks = dgrad_blocks<L, RT>(N);
    hipLaunchKernelGGL((k_dgrad<L, RT, CT>), dim3(blocks, L::CIN / 16 / CT, classes), dim3(L::TAPS == 1 ? 64 : 256), 0,
                       w.c->stream, dZ, W, Yl, N, dZl, dZf);
    w.columns(dZf, L::TAPS == 1 ? 2 * N : N * L::HI * L::WI, L::CIN, dbias);
}

// Room for the partial sums of a batch of N (all of cnn_backward's takes).
size_t part_elems(int N)
{
    size_t n = wgrad_part_elems<Conv0>() + wgrad_part_elems<Conv1>() + wgrad_part_elems<Conv2>() +
               wgrad_part_elems<Conv3>() + wgrad_part_elems<Conv4>() + wgrad_part_elems<Conv5>() +
               wgrad_part_elems<Fc1>();
    for (const auto& c : kSpec) n += (size_t)col_chunks(N * c.ho * c.wo) * c.cout;
    return n + (size_t)col_chunks(N) * (kFc1Out + kOutPad);
}

}  // namespace

// ============================================================= fused inference
// The whole forward pass of one sample in one workgroup: the activations stay
// in LDS (at most 76.8 KB + 38.4 KB, the first layer's output and input), every
// convolution is an implicit-GEMM on MFMA (the im2col operand is gathered
// from the LDS activations as it is consumed, 4 consecutive channels of one
// input pixel per lane), the weights are read from the bf16 copy, and the
// epilogue (bias, ReLU, bf16) writes the next layer's input.  The rounding
// points are those of cnn_forward (bf16 activations, fp32 accumulation), and a
// sample's result does not depend on the other samples of the launch.  One
// launch for the whole network; no activations are kept.
constexpr int kInferThreads = 1024;
constexpr int kHeadGroups = kInferThreads / 64;   // k_cnn_head's groups per sample: one per head wave
// Activations in LDS are [H][W][C + kActPad] (the input: [H][W][4]): a pixel
// stride of C + 4 elements puts the 16 pixels of a stride-2 fragment load
// 16 bytes apart modulo the 128-byte bank period (2-way), where C alone
// (a multiple of 32 from layer 2 on) would put all of them on one bank.
constexpr int kActPad = 4;
constexpr int kInferBufA = 30 * 40 * (32 + kActPad);   // elements: the largest output (layer 1)
constexpr int kInferBufB = 15 * 20 * (64 + kActPad);   // layer 2's output; also holds the input
constexpr int kInferIn = 60 * 80 * 4;                  // the input sample
// One LDS array holds both buffers and four zeros, which a tap outside the
// image reads.
constexpr int kInferZero = kInferBufA + kInferBufB;
static_assert(kInferIn <= kInferBufB, "the input fits its buffer");

struct InferParams {
    const bf16* W[kConvs];                   // k_fwd's fragment order
    const float* b[kConvs];
    const bf16* fc1W;                        // [128][3840]
    const float* fc1b;
    const bf16* fc2W;                        // [3840][8]
    const float* fc2b;
};

// One convolution layer (3x3, stride 2, pad 1) from X (LDS, [HI][WI][CIN])
// into Y (LDS, [HO][WO][COUT]).  Each wave takes (column tile, up to four row
// tiles) work items.  The weight fragments of up to kGroup consecutive
// 16-deep k steps are loaded together before their MFMAs, so an item waits
// for one memory latency per group rather than per step; each fragment serves
// all the item's row tiles.  W is in fragment order: step ks, column tile nt,
// lane L hold W[16 ks + 4 (L >> 4) + q][16 nt + (L & 15)], q = 0..3.
constexpr int kGroup = 24;

// The k steps [k0, k1) of one work item (column tile nt, row tiles from
// ch * CH) into acc.  S: the LDS of the kernel, X its input's offset.  A step
// lies in one tap (with 4 input channels: four of a lane's group each), so a
// fragment's address is the row's base plus an offset that is the same in the
// whole wave, and whether the tap lies in the image is a bit of the row's
// mask; a tap outside reads zeros.  With the tap and the bounds formed per
// lane and step the launch took 37.6 us, so 31.0 (the same bits).
template <int CIN, int COUT, int HI, int WI, int HO, int WO, int XS, int CH, int GR, int k0, int k1>
__device__ __forceinline__ void infer_conv_item(const bf16* __restrict__ S, int X, const bf16* __restrict__ W, int nt,
                                                int ch, v4f (&acc)[CH])
{
    constexpr int M = HO * WO, MT = (M + 15) / 16, NT = COUT / 16;
    const int lane = threadIdx.x & 63;
    const int grp = lane >> 4;                // this lane's k offset within a 16-deep step: 4 grp
    // the rows of this lane's A fragments (one per row tile of the chunk)
    int base[CH], taps[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int m = (ch * CH + i) * 16 + (lane & 15);
        const int h = 2 * (m / WO) - 1, w = 2 * (m % WO) - 1;
        base[i] = X + (h * WI + w) * XS + (CIN == 4 ? 0 : 4 * grp);
        const int cols = (w >= 0 ? 1 : 0) | (w + 1 < WI ? 2 : 0) | (w + 2 < WI ? 4 : 0);
        taps[i] = (h >= 0 ? cols : 0) | (h + 1 < HI ? cols << 3 : 0) | (h + 2 < HI ? cols << 6 : 0);
        if ((ch * CH + i) >= MT || m >= M) taps[i] = 0;
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int g0 = k0; g0 < k1; g0 += GR) {
        // one 8-byte fragment per lane and step (the wave reads 512
        // contiguous bytes), all of the group's steps in flight together
        v4s b[GR];
#pragma unroll
        for (int g = 0; g < GR; ++g)
            if (g0 + g < k1) b[g] = *(const v4s*)(W + ((size_t)((g0 + g) * NT + nt) * 64 + lane) * 4);
#pragma unroll
        for (int g = 0; g < GR; ++g) {
            if (g0 + g >= k1) break;
            int tap, c;
            if constexpr (CIN == 4) {
                tap = 4 * (g0 + g) + grp;
                c = 0;
            } else {
                static_assert(CIN % 16 == 0, "a step lies in one tap");
                tap = (g0 + g) / (CIN / 16);
                c = ((g0 + g) % (CIN / 16)) * 16;
            }
            const int kh = tap / 3, off = (kh * WI + tap - 3 * kh) * XS + c;
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const v4s a = *(const v4s*)&S[(taps[i] >> tap) & 1 ? base[i] + off : kInferZero];
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[g], acc[i], 0, 0, 0);
            }
        }
    }
}

// Bias, ReLU and the bf16 store of one work item.
template <int COUT, int HO, int WO, int YS, int CH>
__device__ __forceinline__ void infer_conv_store(bf16* __restrict__ Y, const float* __restrict__ bias, int nt, int ch,
                                                 const v4f (&acc)[CH])
{
    constexpr int M = HO * WO, MT = (M + 15) / 16;
    const int lane = threadIdx.x & 63;
    const int rq = 4 * (lane >> 4);
    const int n = nt * 16 + (lane & 15);
    const float bn = bias[n];
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = (ch * CH + i) * 16 + rq + r;
            if ((ch * CH + i) >= MT || m >= M) continue;
            float v = acc[i][r] + bn;
            v = fmaxf(v, 0.0f);
            Y[m * YS + n] = f2bf(v);
        }
}

// XS, YS: the pixel strides (elements) of X and Y.  ROWS: row tiles per work
// item (fewer when the layer has fewer, so no MFMA runs on an all-padding
// tile), such that the items come out even over the 16 waves: 75 x 2 tiles in
// 30 items of 5, 19 x 4 in 16 of 5, 5 x 6 in 12 of 3 (31.0 -> 29.0 us against
// items of 4).  Layers with at most half as many work items as waves (the deep,
// small ones) split each item's k steps in two halves on two waves; the
// second half's sums go through LDS past the layer's output in Y (at
// kKPartOff elements; Y is larger than the small outputs that split) and are
// added to the first half's, in that order.
constexpr int kKPartOff = 4096;

template <int CIN, int COUT, int HI, int WI, int HO, int WO, int XS, int YS, int ROWS>
__device__ __forceinline__ void infer_conv(bf16* __restrict__ S, int X, int yoff, const bf16* __restrict__ W,
                                           const float* __restrict__ bias)
{
    constexpr int M = HO * WO, MT = (M + 15) / 16, NT = COUT / 16, CH = MT < ROWS ? MT : ROWS;
    constexpr int KREAL = 9 * CIN, KP = (KREAL + 31) / 32 * 32, KS = KP / 16;
    static_assert(COUT % 16 == 0 && CIN % 4 == 0 && KP % 16 == 0, "tile shapes");
    bf16* Y = S + yoff;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int WAVES = kInferThreads / 64;
    constexpr int CHUNKS = (MT + CH - 1) / CH, ITEMS = NT * CHUNKS;
    constexpr bool SPLIT = 2 * ITEMS <= WAVES && KS >= 2 * kGroup;
    if constexpr (!SPLIT) {
        constexpr int GR = KS < kGroup ? KS : kGroup;
        for (int item = wave; item < ITEMS; item += WAVES) {
            const int nt = item % NT, ch = item / NT;
            v4f acc[CH];
            infer_conv_item<CIN, COUT, HI, WI, HO, WO, XS, CH, GR, 0, KS>(S, X, W, nt, ch, acc);
            infer_conv_store<COUT, HO, WO, YS, CH>(Y, bias, nt, ch, acc);
        }
    } else {
        constexpr int KH = (KS + 1) / 2;
        constexpr int GR = KH < kGroup ? KH : kGroup;
        static_assert(M * YS <= kKPartOff && kKPartOff * 2 + ITEMS * CH * 256 * 4 <= kInferBufB * 2 &&
                          kKPartOff * 2 + ITEMS * CH * 256 * 4 <= kInferBufA * 2,
                      "the second-half sums fit past the output");
        const int lane = threadIdx.x & 63;
        const bool live = wave < 2 * ITEMS;
        const int item = wave % ITEMS, half = wave / ITEMS;
        const int nt = item % NT, ch = item / NT;
        v4f acc[CH];
        if (!live) {
#pragma unroll
            for (int i = 0; i < CH; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
        } else if (half == 0) {
            infer_conv_item<CIN, COUT, HI, WI, HO, WO, XS, CH, GR, 0, KH>(S, X, W, nt, ch, acc);
        } else {
            infer_conv_item<CIN, COUT, HI, WI, HO, WO, XS, CH, GR, KH, KS>(S, X, W, nt, ch, acc);
        }
        float* kp = (float*)(Y + kKPartOff) + ((size_t)item * CH * 64 + lane) * 4;
        if (live && half == 1)
#pragma unroll
            for (int i = 0; i < CH; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) kp[i * 256 + r] = acc[i][r];
        __syncthreads();
        if (live && half == 0) {
#pragma unroll
            for (int i = 0; i < CH; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][r] = acc[i][r] + kp[i * 256 + r];
            infer_conv_store<COUT, HO, WO, YS, CH>(Y, bias, nt, ch, acc);
        }
    }
}

__global__ __launch_bounds__(kInferThreads) void k_cnn_infer(const bf16* __restrict__ x, InferParams P,
                                                             float* __restrict__ out, float* __restrict__ gap_out)
{
    __shared__ __align__(16) bf16 S[kInferZero + 4];
    constexpr int A = 0, B = kInferBufA;
    static_assert(kInferBufA % 8 == 0 && kInferZero % 4 == 0, "16-byte rows, 8-byte fragments");
    bf16* bufB = S + B;
    __shared__ float s_h1[kFc1Out];
    __shared__ float s_gap[kFc1In];
    __shared__ float s_fc2[kInferThreads / 64][kOut];
    const int t = threadIdx.x;
    // the input, 16 bytes per thread and step
    const uint4* src = (const uint4*)(x + (size_t)blockIdx.x * kInferIn);
    for (int i = t; i < kInferIn / 8; i += kInferThreads) ((uint4*)bufB)[i] = src[i];
    if (t < 4) S[kInferZero + t] = 0;
    __syncthreads();
    constexpr int P4 = 4 + 0, P32 = 32 + kActPad, P64 = 64 + kActPad, P96 = 96 + kActPad, P128 = 128 + kActPad;
    infer_conv<4, 32, 60, 80, 30, 40, P4, P32, 5>(S, B, A, P.W[0], P.b[0]);
    __syncthreads();
    infer_conv<32, 64, 30, 40, 15, 20, P32, P64, 5>(S, A, B, P.W[1], P.b[1]);
    __syncthreads();
    infer_conv<64, 96, 15, 20, 8, 10, P64, P96, 3>(S, B, A, P.W[2], P.b[2]);
    __syncthreads();
    infer_conv<96, 128, 8, 10, 4, 5, P96, P128, 2>(S, A, B, P.W[3], P.b[3]);
    __syncthreads();
    infer_conv<128, 128, 4, 5, 2, 3, P128, P128, 1>(S, B, A, P.W[4], P.b[4]);
    __syncthreads();
    infer_conv<128, 128, 2, 3, 1, 2, P128, P128, 1>(S, A, B, P.W[5], P.b[5]);
    __syncthreads();
    // global average pooling over the 1 x 2 output (the arithmetic of
    // k_fwd's kReluGap)
    if (t < kFc1In) {
        const float sgap = bf2f(bufB[t]) + bf2f(bufB[P128 + t]);
        s_gap[t] = bf2f(f2bf(sgap / 2.0f));
        if (gap_out) gap_out[(size_t)blockIdx.x * kFc1In + t] = s_gap[t];
    }
    if (gap_out) return;   // the FC layers run in k_cnn_head
    __syncthreads();
    // fc1 (ReLU, bf16 output) and fc2, fp32 accumulation of bf16 operands.
    // fc1 is a matrix-vector product over 983 KB of weights: each thread
    // forms 4 consecutive hidden units from 8-byte weight loads, 32 rows of
    // them in flight at a time; every unit sums its 128 terms in row order.
    static_assert(kFc1Out % 4 == 0 && kFc1Out / 4 <= kInferThreads && kFc1In % 32 == 0, "fc1 blocking");
    if (t < kFc1Out / 4) {
        constexpr int G = kFc1Out / 4;
        const uint2* Wv = (const uint2*)P.fc1W;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int k0 = 0; k0 < kFc1In; k0 += 32) {
            uint2 wv[32];
#pragma unroll
            for (int kk = 0; kk < 32; ++kk) wv[kk] = Wv[(size_t)(k0 + kk) * G + t];
#pragma unroll
            for (int kk = 0; kk < 32; ++kk) {
                const float g = s_gap[k0 + kk];
                acc[0] += g * bf2f((bf16)(wv[kk].x & 0xffffu));
                acc[1] += g * bf2f((bf16)(wv[kk].x >> 16));
                acc[2] += g * bf2f((bf16)(wv[kk].y & 0xffffu));
                acc[3] += g * bf2f((bf16)(wv[kk].y >> 16));
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) s_h1[4 * t + q] = bf2f(f2bf(fmaxf(acc[q] + P.fc1b[4 * t + q], 0.0f)));
    }
    __syncthreads();
    // fc2: every wave sums its slice of the hidden units for all six outputs
    // (one 16-byte weight row per lane and step, all of a lane's rows in
    // flight together), then the waves' sums in wave order
    {
        constexpr int NW = kInferThreads / 64, RPW = kFc1Out / NW, STEPS = (RPW + 63) / 64;
        static_assert(kFc1Out % NW == 0 && kOutPad == 8 && kOut <= 8, "fc2 blocking");
        const int wv = t >> 6, lane = t & 63;
        const uint4* W8 = (const uint4*)P.fc2W;   // row k: the 8 (padded) outputs' bf16 weights
        uint4 w[STEPS];
#pragma unroll
        for (int q = 0; q < STEPS; ++q) {
            const int r = lane + 64 * q;
            w[q] = W8[wv * RPW + (r < RPW ? r : 0)];
        }
        float acc[kOut];
#pragma unroll
        for (int j = 0; j < kOut; ++j) acc[j] = 0.0f;
#pragma unroll
        for (int q = 0; q < STEPS; ++q) {
            const int r = lane + 64 * q;
            if (r < RPW) {
                const float h = s_h1[wv * RPW + r];
                const uint32_t wq[4] = {w[q].x, w[q].y, w[q].z, w[q].w};
#pragma unroll
                for (int j = 0; j < kOut; ++j)
                    acc[j] += h * bf2f((bf16)((j & 1) ? (wq[j >> 1] >> 16) : (wq[j >> 1] & 0xffffu)));
            }
        }
#pragma unroll
        for (int j = 0; j < kOut; ++j) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) acc[j] += __shfl_xor(acc[j], off, 64);
        }
        if (lane == 0)
#pragma unroll
            for (int j = 0; j < kOut; ++j) s_fc2[wv][j] = acc[j];
        __syncthreads();
        if (t < kOut) {
            float o = 0.0f;
            for (int q = 0; q < NW; ++q) o += s_fc2[q][t];
            out[(size_t)blockIdx.x * kOut + t] = o + P.fc2b[t];
        }
    }
}

extern "C" {

int cnn_create(int max_batch, cnn_net* out)
{
    if (!out || max_batch < 1 || max_batch > 4096) return CNN_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return CNN_ERR_NODEV;
    cnn_net_s* c = new cnn_net_s();
    c->max_batch = max_batch;
    size_t off = 0;
    auto take = [&](Param& p, size_t n) {
        p.off = off;
        p.n = n;
        off += (n + 63) & ~(size_t)63;
    };
    for (int l = 0; l < kConvs; ++l) {
        c->Kp[l] = (9 * kSpec[l].cin + 31) / 32 * 32;
        take(c->convW[l], (size_t)c->Kp[l] * kSpec[l].cout);
        take(c->convB[l], kSpec[l].cout);
    }
    take(c->fc1W, (size_t)kFc1In * kFc1Out);
    take(c->fc1B, kFc1Out);
    take(c->fc2W, (size_t)kFc1Out * kOutPad);
    take(c->fc2B, kOutPad);
    c->nparam = off;
    const int N = max_batch;
    int rc = CNN_OK;
    rc = rc ? rc : dalloc(c, &c->p, off);
    rc = rc ? rc : dalloc(c, &c->g, off);
    rc = rc ? rc : dalloc(c, &c->m, off);
    rc = rc ? rc : dalloc(c, &c->v, off);
    rc = rc ? rc : dalloc(c, &c->pb, off);
    rc = rc ? rc : dalloc(c, &c->mask, off);
    rc = rc ? rc : dalloc(c, &c->infer_gap, (size_t)N * kFc1In);
    rc = rc ? rc : dalloc(c, &c->infer_part, (size_t)N * kHeadGroups * kOutPad);
    rc = rc ? rc : dalloc(c, &c->infer_ticket, (size_t)N);
    for (int l = 0; l < kConvs && !rc; ++l) {
        const size_t n = (size_t)N * kSpec[l].ho * kSpec[l].wo * kSpec[l].cout;
        rc = dalloc(c, &c->y[l], n);
        rc = rc ? rc : dalloc(c, &c->dz[l], n);
        rc = rc ? rc : dalloc(c, &c->dzf[l], n);
    }
    size_t form_n[2 * kLayers] = {}, form_total = 0;
    c->forms.flat = c->pb;
    for (int l = 0; l < kLayers; ++l) {
        const Param& w = l < kConvs ? c->convW[l] : (l == kConvs ? c->fc1W : c->fc2W);
        const int ld = l < kConvs ? kSpec[l].cout : (l == kConvs ? kFc1Out : kOutPad);
        c->forms.first[l] = (int)w.off;
        c->forms.n[l] = (int)w.n;
        c->forms.ld[l] = ld;
        form_n[l] = w.n / ld * (cdiv(ld, 16) * 16);
        form_n[kLayers + l] = l > 0 && l <= kConvs ? w.n : 0;   // conv 1..5 and fc1 have input gradients
        form_total += form_n[l] + form_n[kLayers + l];
    }
    bf16* form = nullptr;
    rc = rc ? rc : dalloc(c, &form, form_total);
    for (size_t q = 0, at = 0; q < 2 * kLayers && !rc; at += form_n[q++])
        (q < kLayers ? c->forms.fwd[q] : c->forms.dgrad[q - kLayers]) = form_n[q] ? form + at : nullptr;
    rc = rc ? rc : dalloc(c, &c->x, (size_t)N * 60 * 80 * 4);
    rc = rc ? rc : dalloc(c, &c->gap, (size_t)N * kFc1In);
    rc = rc ? rc : dalloc(c, &c->h1, (size_t)N * kFc1Out);
    rc = rc ? rc : dalloc(c, &c->dz1, (size_t)N * kFc1Out);
    rc = rc ? rc : dalloc(c, &c->dz1f, (size_t)N * kFc1Out);
    rc = rc ? rc : dalloc(c, &c->dob, (size_t)N * kOutPad);
    rc = rc ? rc : dalloc(c, &c->dof, (size_t)N * kOutPad);
    rc = rc ? rc : dalloc(c, &c->out, (size_t)N * kOutPad);
    rc = rc ? rc : dalloc(c, &c->part, part_elems(N));
    if (rc) {
        cnn_destroy(c);
        return rc;
    }
    // parameter mask: 0 on the reduction padding rows of each conv weight and
    // on the padding columns of fc2
    std::vector<uint8_t> mk(off, 1);
    for (int l = 0; l < kConvs; ++l)
        for (int k = 9 * kSpec[l].cin; k < c->Kp[l]; ++k)
            for (int n = 0; n < kSpec[l].cout; ++n) mk[c->convW[l].off + (size_t)k * kSpec[l].cout + n] = 0;
    for (int k = 0; k < kFc1Out; ++k)
        for (int n = kOut; n < kOutPad; ++n) mk[c->fc2W.off + (size_t)k * kOutPad + n] = 0;
    for (int n = kOut; n < kOutPad; ++n) mk[c->fc2B.off + n] = 0;
    if (hipMemcpy(c->mask, mk.data(), off, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(c->p, 0, off * 4) != hipSuccess || hipMemset(c->g, 0, off * 4) != hipSuccess ||
        hipMemset(c->m, 0, off * 4) != hipSuccess || hipMemset(c->v, 0, off * 4) != hipSuccess ||
        hipMemset(c->pb, 0, off * 2) != hipSuccess || hipMemset(form, 0, form_total * 2) != hipSuccess ||
        hipMemset(c->infer_ticket, 0, (size_t)N * sizeof(unsigned int)) != hipSuccess) {
        cnn_destroy(c);
        return CNN_ERR_HIP;
    }
    *out = c;
    return CNN_OK;
}

int cnn_destroy(cnn_net c)
{
    if (!c) return CNN_ERR_ARG;
    (void)hipDeviceSynchronize();
    for (void* p : c->allocs) (void)hipFree(p);
    delete c;
    return CNN_OK;
}

int cnn_set_stream(cnn_net c, void* stream)
{
    if (!c) return CNN_ERR_ARG;
    c->stream = (hipStream_t)stream;
    return CNN_OK;
}

int cnn_num_params(cnn_net c, size_t* n)
{
    if (!c || !n) return CNN_ERR_ARG;
    *n = c->nparam;
    return CNN_OK;
}

int cnn_param_layout(cnn_net c, size_t* offsets, size_t* sizes, int cap)
{
    if (!c || !offsets || !sizes || cap < 2 * kConvs + 4) return CNN_ERR_ARG;
    int q = 0;
    for (int l = 0; l < kConvs; ++l) {
        offsets[q] = c->convW[l].off; sizes[q++] = c->convW[l].n;
        offsets[q] = c->convB[l].off; sizes[q++] = c->convB[l].n;
    }
    offsets[q] = c->fc1W.off; sizes[q++] = c->fc1W.n;
    offsets[q] = c->fc1B.off; sizes[q++] = c->fc1B.n;
    offsets[q] = c->fc2W.off; sizes[q++] = c->fc2W.n;
    offsets[q] = c->fc2B.off; sizes[q++] = c->fc2B.n;
    return q;
}

int cnn_set_params(cnn_net c, const float* host, size_t n)
{
    if (!c || !host || n != c->nparam) return CNN_ERR_ARG;
    CK(hipMemcpy(c->p, host, n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_to_bf16, g1(n), dim3(256), 0, c->stream, c->p, (int)n, c->forms);
    CK(hipMemset(c->m, 0, n * 4));
    CK(hipMemset(c->v, 0, n * 4));
    c->step = 0;
    CK(hipDeviceSynchronize());
    return launch_check("set_params");
}

int cnn_get_params(cnn_net c, float* host, size_t n)
{
    if (!c || !host || n != c->nparam) return CNN_ERR_ARG;
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(host, c->p, n * 4, hipMemcpyDeviceToHost));
    return CNN_OK;
}

int cnn_get_grads(cnn_net c, float* host, size_t n)
{
    if (!c || !host || n != c->nparam) return CNN_ERR_ARG;
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(host, c->g, n * 4, hipMemcpyDeviceToHost));
    return CNN_OK;
}

int cnn_prepare_input(cnn_net c, const float* depth_a, const uint8_t* image_a, const uint16_t* depth_b,
                      const uint8_t* image_b, int n, size_t frame_stride, void* x)
{
    if (!c || !depth_a || !image_a || !depth_b || !image_b || !x || n < 1) return CNN_ERR_ARG;
    hipLaunchKernelGGL(k_prepare, g1((size_t)n * 80 * 60), dim3(256), 0, c->stream, depth_a, image_a, depth_b,
                       image_b, n, 80, 60, frame_stride, (bf16*)x);
    return launch_check("prepare_input");
}

// Forward of N samples (x: NHWC bf16 [N][60][80][4], device); out (device,
// fp32 [N][6]) may be null.  Keeps the activations for cnn_backward.
int cnn_forward(cnn_net c, const void* x, int N, float* out)
{
    if (!c || !x || N < 1 || N > c->max_batch) return CNN_ERR_ARG;
    const int frags = N * (60 * 80 * 4 / 8);
    hipLaunchKernelGGL(k_copy_input, dim3(std::min(cdiv(frags, 256), 2048)), dim3(256), 0, c->stream, (const bf16*)x,
                       frags, c->x);
    const auto b = [&](const Param& p) { return c->p + p.off; };
    launch_fwd<Conv0, 4, 2, 1, kRelu>(c, 0, c->x, N, b(c->convB[0]), c->y[0]);
    launch_fwd<Conv1, 2, 4, 1, kRelu>(c, 1, c->y[0], N, b(c->convB[1]), c->y[1]);
    launch_fwd<Conv2, 1, 3, 1, kRelu>(c, 2, c->y[1], N, b(c->convB[2]), c->y[2]);
    launch_fwd<Conv3, 1, 4, 1, kRelu>(c, 3, c->y[2], N, b(c->convB[3]), c->y[3]);
    launch_fwd<Conv4, 1, 1, 1, kRelu>(c, 4, c->y[3], N, b(c->convB[4]), c->y[4]);
    launch_fwd<Conv5, 1, 1, 4, kReluGap, 9>(c, 5, c->y[4], N, b(c->convB[5]), c->y[5], c->gap);
    launch_fwd<Fc1, 1, 4, 1, kRelu>(c, 6, c->gap, N, b(c->fc1B), c->h1);
    launch_fwd<Fc2, 1, 1, 16, kHead, 30>(c, 7, c->h1, N, b(c->fc2B), nullptr, nullptr, c->out, out);
    return launch_check("forward");
}

// The FC layers of the split inference: kHeadGroups workgroups per sample
// (blockIdx.x = sample * kHeadGroups + group).  Group g forms the 240 hidden
// units [240 g, 240 g + 240) with all 128 of a unit's weights in flight at
// once, each unit summing its terms in row order, and their FC2 sums exactly
// as wave g of k_cnn_infer's head does (so the same bits); the group that
// arrives last at the sample's ticket adds the groups' sums in group order and
// the bias, and sets the ticket back to 0.
__global__ __launch_bounds__(256) void k_cnn_head(const float* __restrict__ gap, InferParams P,
                                                  float* __restrict__ part, unsigned int* __restrict__ ticket,
                                                  float* __restrict__ out)
{
    constexpr int RPW = kFc1Out / kHeadGroups, STEPS = (RPW + 63) / 64;
    static_assert(kFc1Out % kHeadGroups == 0 && RPW <= 256 && kOutPad == 8 && kOut <= 8, "head blocking");
    __shared__ float s_gap[kFc1In];
    __shared__ float s_h1[RPW];
    __shared__ unsigned int s_last;
    const int t = threadIdx.x;
    const int smp = blockIdx.x / kHeadGroups, grp = blockIdx.x - smp * kHeadGroups;
    const int unit = grp * RPW + t;
    // the unit's 128 fc1 weights (coalesced over the units) and the group's
    // fc2 rows, all loads issued before the first wait
    bf16 w[kFc1In];
    if (t < RPW) {
#pragma unroll
        for (int k = 0; k < kFc1In; ++k) w[k] = P.fc1W[(size_t)k * kFc1Out + unit];
    }
    const int lane = t & 63;
    uint4 w2[STEPS];
    const uint4* W8 = (const uint4*)P.fc2W;
    if (t < 64) {
#pragma unroll
        for (int q = 0; q < STEPS; ++q) {
            const int r = lane + 64 * q;
            w2[q] = W8[grp * RPW + (r < RPW ? r : 0)];
        }
    }
    if (t < kFc1In) s_gap[t] = gap[(size_t)smp * kFc1In + t];
    __syncthreads();
    if (t < RPW) {
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kFc1In; ++k) acc += s_gap[k] * bf2f(w[k]);
        s_h1[t] = bf2f(f2bf(fmaxf(acc + P.fc1b[unit], 0.0f)));
    }
    __syncthreads();
    if (t < 64) {
        float acc[kOut];
#pragma unroll
        for (int j = 0; j < kOut; ++j) acc[j] = 0.0f;
#pragma unroll
        for (int q = 0; q < STEPS; ++q) {
            const int r = lane + 64 * q;
            if (r < RPW) {
                const float h = s_h1[r];
                const uint32_t wq[4] = {w2[q].x, w2[q].y, w2[q].z, w2[q].w};
#pragma unroll
                for (int j = 0; j < kOut; ++j)
                    acc[j] += h * bf2f((bf16)((j & 1) ? (wq[j >> 1] >> 16) : (wq[j >> 1] & 0xffffu)));
            }
        }
#pragma unroll
        for (int j = 0; j < kOut; ++j) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) acc[j] += __shfl_xor(acc[j], off, 64);
        }
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < kOut; ++j) part[((size_t)smp * kHeadGroups + grp) * kOutPad + j] = acc[j];
            // the partial sums first, then the arrival (release); the last
            // arrival reads every group's sums (acquire)
            s_last = __hip_atomic_fetch_add(ticket + smp, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
                     (unsigned)(kHeadGroups - 1);
        }
    }
    __syncthreads();
    if (s_last && t < kOut) {
        const float* ps = part + (size_t)smp * kHeadGroups * kOutPad;
        float o = 0.0f;
        for (int q = 0; q < kHeadGroups; ++q)
            o += __hip_atomic_load(ps + (size_t)q * kOutPad + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        out[(size_t)smp * kOut + t] = o + P.fc2b[t];
        if (t == 0) __hip_atomic_store(ticket + smp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Inference of N samples in one launch (k_cnn_infer): out (device, fp32
// [N][6]).  Keeps no activations.
int cnn_infer(cnn_net c, const void* x, int N, float* out)
{
    if (!c || !x || !out || N < 1 || N > c->max_batch) return CNN_ERR_ARG;
    if ((uintptr_t)x % 16 != 0) return CNN_ERR_ARG;
    InferParams P;
    for (int l = 0; l < kConvs; ++l) {
        P.W[l] = c->forms.fwd[l];
        P.b[l] = c->p + c->convB[l].off;
    }
    P.fc1W = c->pb + c->fc1W.off;
    P.fc1b = c->p + c->fc1B.off;
    P.fc2W = c->pb + c->fc2W.off;
    P.fc2b = c->p + c->fc2B.off;
    if (c->infer_split) {
        hipLaunchKernelGGL(k_cnn_infer, dim3(N), dim3(kInferThreads), 0, c->stream, (const bf16*)x, P, out,
                           c->infer_gap);
        hipLaunchKernelGGL(k_cnn_head, dim3(N * kHeadGroups), dim3(256), 0, c->stream, c->infer_gap, P,
                           c->infer_part, c->infer_ticket, out);
    } else {
        hipLaunchKernelGGL(k_cnn_infer, dim3(N), dim3(kInferThreads), 0, c->stream, (const bf16*)x, P, out,
                           (float*)nullptr);
    }
    return launch_check("infer");
}

// The inference head's layout: 1 (default) the FC layers in k_cnn_head's
// workgroups, 0 in the convolution workgroup; the same bits either way.
int cnn_set_infer_split(cnn_net c, int split)
{
    if (!c || (split != 0 && split != 1)) return CNN_ERR_ARG;
    c->infer_split = split;
    return CNN_OK;
}

// Gradients of the weighted squared error against target (device fp32
// [N][6]) with weights w (host, 6) for the last forward of N samples: loss
// per sample into loss_n (device, optional), parameter gradients into the
// net's gradient buffer.
int cnn_backward(cnn_net c, int N, const float* target, const float* w, float* loss_n)
{
    if (!c || !target || !w || N < 1 || N > c->max_batch) return CNN_ERR_ARG;
    LossWeights lw;
    for (int j = 0; j < kOut; ++j) lw.w[j] = w[j];
    Parts P{c};
    const auto g = [&](const Param& p) { return c->g + p.off; };
    const auto wd = [&](int l) { return (const bf16*)c->forms.dgrad[l]; };   // conv l, or fc1 as 6
    hipLaunchKernelGGL(k_head_bwd, dim3(cdiv(kFc1Out, 256), cdiv(N, kHeadChunk)), dim3(256), 0, c->stream, c->out,
                       target, lw, N, kFc1Out, c->h1, c->pb + c->fc2W.off, loss_n, c->dob, c->dof, c->dz1, c->dz1f);
    hipLaunchKernelGGL(k_head_wgrad, dim3(cdiv(kFc1Out, 64)), dim3(256), 0, c->stream, c->h1, c->dob, N, kFc1Out,
                       wgrad_rows(N, kFc1Out, kOutPad), g(c->fc2W));
    P.columns(c->dof, N, kOutPad, g(c->fc2B));
    P.columns(c->dz1f, N, kFc1Out, g(c->fc1B));
    launch_wgrad<Fc1, 128>(P, c->gap, c->dz1, N, g(c->fc1W));
    launch_dgrad<Fc1, 1, 1>(P, c->dz1, wd(6), c->y[5], N, c->dz[5], c->dzf[5], g(c->convB[5]));
    launch_wgrad<Conv5, 32>(P, c->y[4], c->dz[5], N * 2, g(c->convW[5]));
    launch_dgrad<Conv5, 1, 1>(P, c->dz[5], wd(5), c->y[4], N, c->dz[4], c->dzf[4], g(c->convB[4]));
    launch_wgrad<Conv4, 32>(P, c->y[3], c->dz[4], N * 6, g(c->convW[4]));
    launch_dgrad<Conv4, 1, 1>(P, c->dz[4], wd(4), c->y[3], N, c->dz[3], c->dzf[3], g(c->convB[3]));
    launch_wgrad<Conv3, 64>(P, c->y[2], c->dz[3], N * 20, g(c->convW[3]));
    launch_dgrad<Conv3, 1, 3>(P, c->dz[3], wd(3), c->y[2], N, c->dz[2], c->dzf[2], g(c->convB[2]));
    launch_wgrad<Conv2, 96>(P, c->y[1], c->dz[2], N * 80, g(c->convW[2]));
    launch_dgrad<Conv2, 2, 4>(P, c->dz[2], wd(2), c->y[1], N, c->dz[1], c->dzf[1], g(c->convB[1]));
    launch_wgrad<Conv1, 64>(P, c->y[0], c->dz[1], N * 300, g(c->convW[1]));
    launch_dgrad<Conv1, 2, 2>(P, c->dz[1], wd(1), c->y[0], N, c->dz[0], c->dzf[0], g(c->convB[0]));
    launch_wgrad<Conv0, 32>(P, c->x, c->dz[0], N * 1200, g(c->convW[0]));
    hipLaunchKernelGGL(k_colsum, dim3(P.col_blocks), dim3(64), 0, c->stream, P.cols);
    hipLaunchKernelGGL(k_sum_parts, dim3(P.blocks), dim3(64), 0, c->stream, P.jobs);
    return launch_check("backward");
}

int cnn_adam_step(cnn_net c, float lr, float wd)
{
    if (!c || !(lr >= 0.0f)) return CNN_ERR_ARG;
    c->step++;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float bc1 = 1.0f - powf(b1, (float)c->step), bc2 = 1.0f - powf(b2, (float)c->step);
    hipLaunchKernelGGL(k_adam, g1(c->nparam), dim3(256), 0, c->stream, c->p, c->g, c->m, c->v, c->forms, c->mask,
                       (int)c->nparam, lr, b1, b2, eps, bc1, bc2, wd);
    return launch_check("adam");
}

}  // extern "C"
