// Layer norm over the channel dimension of (N, C, M) tensors on gfx950 (csrc/layer_norm.cu:53-257).
//   forward   out = (x - mean) * rsqrt(var + eps),  mean / var (population) over C per (n, m)   (:102-129)
//   backward  res = -rsqrt(v) * (1/C + (x - mean) * (x - 1/C) * mean * v) * grad,  v = var + eps  (:200-216)
// The backward is the reference's expression, kept as it is (it is not the derivative of the forward).
//
// The op has to see a slice twice (statistics, then the normalised values), and a slice of C
// channels times a wavefront's pixels is far more than caches keep per wave, so the slice stays in
// REGISTERS between the two uses: lanes run along pixels (8 bytes per lane and channel), and for
// C > 32 the four (C > 64: eight) waves of a block split the channels of one pixel group between
// them and exchange per-wave (mean, centred square sum) pairs through LDS, merged by the
// pairwise-variance rule. A wave holds at most 96 packed channels, which covers C <= 768; C <= 1024
// runs one pixel per lane; anything larger, and m_size == 1 (rows contiguous), takes a two-sweep
// kernel whose second sweep is served by cache.
#pragma once
#include <type_traits>
#include "plh_common.hpp"

namespace plh {

struct LnParams {
    int64_t P;          // n_size * m_size
    int64_t m_size;
    int C;
    int per_wave;       // channels per wave when the waves of a block share a pixel group
    float eps;
    // affine forms only: per-channel weight and bias (elements of x's type; the backward has no use for the bias),
    // the number of pixel groups, and the backward's per-block sums [blocks][C][2] (nullptr: not wanted)
    const void *weight, *bias;
    int64_t groups;
    float *partials;
};

constexpr int kLnBlock = 256;

// Wavefronts per SIMD that a kernel's registers have to leave room for: the affine backward's sums would take the slices
// of up to 32 slots past 128 registers, and a CU would hold one block of 512 threads where it holds two. Measured on fp32 and
// aligned planes. Blocks of 256 threads (up to 32 channels) share the limit without that reason, and tiles per image and
// 16-bit elements spill under it (17..32 channels up to 908 bytes per lane): (30,32,129,129) fp32 takes 149 us for the
// module's step where (30,32,128,128) takes 75; with torch's operations they took 511 and 453.
constexpr int ln_waves(int slots, bool sums) { return (sums && slots <= 32) ? 4 : 1; }

// The affine forms' parameters and where the backward leaves their gradients (partials = nullptr: not wanted).
template <class T>
struct LnAffine {
    const T *weight = nullptr, *bias = nullptr;
    float *partials = nullptr;
    T *grad_weight = nullptr, *grad_bias = nullptr;
};

// Sums of N values (8 or 16) over the 64 lanes of a wave: every step adds two values at once, each half of the lanes
// keeping one of them, so that N values cost 2 N + 2 instructions where N separate sums would cost 7 N.
// Lane i returns the sum of value i / (64 / N).
template <int N>
__device__ __forceinline__ float ln_transpose_sum(float (&v)[N], int lane) {
    static_assert(N == 8 || N == 16, "chunks of 4 or 8 channels");
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {                  // lanes 32..63 go on with the upper half of the values
        const auto s = __builtin_amdgcn_permlane32_swap(f32_bits(v[i]), f32_bits(v[i + N / 2]), false, false);
        v[i] = bits_f32(s[0]) + bits_f32(s[1]);
    }
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {                  // odd rows of 16 lanes with the upper half of what is left
        const auto s = __builtin_amdgcn_permlane16_swap(f32_bits(v[i]), f32_bits(v[i + N / 4]), false, false);
        v[i] = bits_f32(s[0]) + bits_f32(s[1]);
    }
#pragma unroll
    for (int i = 0; i < N / 8; ++i) {
        const bool up = lane & 8;
        const float keep = up ? v[i + N / 8] : v[i], give = up ? v[i] : v[i + N / 8];
        v[i] = keep + dpp_move<0x128>(give);           // row_ror:8
    }
    float r = v[0];
    if constexpr (N == 16) {
        const bool up = lane & 4;
        const float keep = up ? v[1] : v[0], give = up ? v[0] : v[1];
        r = keep + dpp_move<0x141>(give);              // row_half_mirror: lane ^ 7
    } else {
        r += dpp_move<0x141>(r);
    }
    r += dpp_move<0xB1>(r);                            // quad_perm [1,0,3,2]
    r += dpp_move<0x4E>(r);                            // quad_perm [2,3,0,1]
    return r;
}

// KW = channel slots per wave (>= the channels it holds), V = pixels per lane, WS = waves sharing a
// pixel group (1: each of a block's four waves has its own group and all channels; 4 or 8: the block
// is WS waves with 1/WS of the channels each).
// PerImage: pixel groups that never straddle two images (groups = images x groups per image), for channel planes
// that start on element boundaries only (odd lengths): a lane's V pixels are moved with accesses of the same
// width from element boundaries; the last lane of an image may hold fewer and goes pixel by pixel.
// Affine: out = weight * normalised + bias in the forward; in the backward the upstream gradient is multiplied by the
// weight on its way in, and the sums of grad * normalised and of grad over the pixels (the gradients of weight and bias)
// are left per block. HBM-bound like the plain forms: the module's two torch passes over the tensor after the forward
// and six before the backward fall away. The backward's blocks loop over pixel groups (ln_grid) so that there are
// few rows of sums; the cross-lane sums of a chunk of channels cost about 5 vector instructions per channel and group
// (ln_transpose_sum), against some 25 for the gradient itself. Module step at (16,256,128,128) fp32: 0.849 -> 0.241 ms
// (its four tensor passes of the plain forms, 5.6 TB/s).
template <class T, int KW, int V, int WS, bool Bwd, bool PerImage = false, bool Affine = false>
__global__ __launch_bounds__(WS > 4 ? 64 * WS : kLnBlock, ln_waves(KW, Affine && Bwd)) void ln_regs(const T *__restrict__ x, const T *__restrict__ g,
                                                    T *__restrict__ out, const LnParams p) {
    using PK = Pack<T, V>;
    constexpr bool kSums = Affine && Bwd;
    constexpr int kChunk = KW % 8 == 0 ? 8 : 4;        // channels of the backward in flight per trip
    // the blocks that loop write the next group's statistics while a slower wave may still read this one's
    __shared__ float ex[kSums ? 2 : 1][WS][2][V][64];
    __shared__ float wb[Affine ? (Bwd ? 1 : 2) : 1][Affine ? 1024 : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = WS > 1 ? wave * p.per_wave : 0;
    int cnt = WS > 1 ? p.C - c0 : p.C;
    cnt = cnt < 1 ? 1 : (WS > 1 && cnt > p.per_wave ? p.per_wave : cnt);   // a split always leaves every wave >= 1 channel
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    if constexpr (Affine) {
        for (int i = threadIdx.x; i < p.C; i += blockDim.x) {
            wb[0][i] = load_one(static_cast<const T *>(p.weight) + i);
            if constexpr (!Bwd) wb[1][i] = load_one(static_cast<const T *>(p.bias) + i);
        }
        __syncthreads();
    }
    float sums[kSums ? KW / kChunk : 1] = {};
    int turn = 0;
    for (int64_t group = WS > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
         !kSums || group < p.groups; group += WS > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * 4) {
    int held = cnt;
    int64_t plane = p.m_size;
    // hidden from the loop: every slot's test and plane offset, taken out of it, would be 300 spilled scalar registers
    if constexpr (kSums) asm volatile("" : "+s"(held), "+s"(plane));
    bool live;
    int nv = V;                                        // pixels this lane has
    int64_t pc, n;
    if constexpr (PerImage) {
        const int64_t per_image = ceil_div_dev(plane, (int64_t)64 * V);
        n = group / per_image;
        const int64_t local = ((group - n * per_image) * 64 + lane) * V;
        const int64_t left = plane - local;
        nv = left >= V ? V : (left > 0 ? (int)left : 0);
        live = nv > 0 && n * plane < p.P;
        if (!live) { n = 0; nv = V; }                  // dead lanes read pixel 0 and store nothing
        pc = live ? n * plane + local : 0;
    } else {
        const int64_t pix = (group * 64 + lane) * V;
        live = pix < p.P;
        pc = live ? pix : 0;                           // dead lanes read pixel 0 and store nothing
        n = pc / plane;
    }
    const int64_t base = pc + n * (int64_t)(p.C - 1) * plane + (int64_t)c0 * plane;
    auto fetch = [&](const T *at) {
        if constexpr (PerImage) {
            if (nv < V) {
                float one[V];
#pragma unroll
                for (int k = 0; k < V; ++k) one[k] = k < nv ? load_one(at + k) : 0.f;
                return PK::put(one);
            }
            return PK::load_unaligned(at);
        } else {
            return PK::load(at);
        }
    };
    auto put_back = [&](T *at, const float (&r)[V]) {
        if constexpr (PerImage) {
            if (nv < V) {
#pragma unroll
                for (int k = 0; k < V; ++k)
                    if (k < nv) store_one(at + k, r[k]);
                return;
            }
            PK::store_unaligned(at, PK::put(r));
        } else {
            PK::store(at, PK::put(r));
        }
    };

    // Slots past the wave's last channel re-read that channel (same address, served by cache) and are
    // weighted out of the sums: straight-line code, no per-slot control flow.
    typename PK::Raw raw[KW];
#pragma unroll
    for (int j = 0; j < KW; ++j) raw[j] = fetch(x + base + (int64_t)(j < held ? j : held - 1) * plane);

    const float inv_c = 1.f / (float)p.C;
    float mean[V], v[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < KW; ++j) s += j < held ? PK::get(raw[j], k) : 0.f;
        const float mw = s / (float)held;
        // every sweep widens the packed slice again: kept apart for the optimiser, which would
        // otherwise hold all widened values of the first sweep in registers for the later ones
#pragma unroll
        for (int j = 0; j < KW; ++j) forget_origin(raw[j]);
        float q = 0.f;
#pragma unroll
        for (int j = 0; j < KW; ++j) {
            const float d = j < held ? PK::get(raw[j], k) - mw : 0.f;
            q = __builtin_fmaf(d, d, q);
        }
        if constexpr (WS > 1) {
            ex[turn][wave][0][k][lane] = mw;
            ex[turn][wave][1][k][lane] = q;
        } else {
            mean[k] = mw;
            v[k] = q * inv_c + p.eps;
        }
    }
    if constexpr (WS > 1) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < V; ++k) {
            float mw[WS], cw[WS], tot = 0.f;
#pragma unroll
            for (int w = 0; w < WS; ++w) {
                int c = p.C - w * p.per_wave;
                c = c < 0 ? 0 : (c > p.per_wave ? p.per_wave : c);
                cw[w] = (float)c;
                mw[w] = ex[turn][w][0][k][lane];
                tot = __builtin_fmaf(cw[w], mw[w], tot);
            }
            const float m = tot * inv_c;
            float m2 = 0.f;
#pragma unroll
            for (int w = 0; w < WS; ++w) {
                const float d = mw[w] - m;
                m2 += ex[turn][w][1][k][lane] + cw[w] * d * d;
            }
            mean[k] = m;
            v[k] = m2 * inv_c + p.eps;
        }
    }
    float rstd[V], mv[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        rstd[k] = 1.f / sqrtf(v[k]);
        mv[k] = mean[k] * v[k];
    }
#pragma unroll
    for (int j = 0; j < KW; ++j) forget_origin(raw[j]);

    if constexpr (!Bwd) {
#pragma unroll
        for (int j = 0; j < KW; ++j) {
            float r[V];
#pragma unroll
            for (int k = 0; k < V; ++k) {
                r[k] = (PK::get(raw[j], k) - mean[k]) * rstd[k];
                if constexpr (Affine) r[k] = __builtin_fmaf(wb[0][c0 + (j < held ? j : 0)], r[k], wb[1][c0 + (j < held ? j : 0)]);
            }
            if (live && j < held) put_back(out + base + (int64_t)j * plane, r);
        }
    } else {
#pragma unroll
        for (int j0 = 0; j0 < KW; j0 += kChunk) {
            typename PK::Raw graw[kChunk];
            float part[2 * kChunk];                    // per channel: grad * normalised, grad (this lane's pixels)
#pragma unroll
            for (int jj = 0; jj < kChunk; ++jj)
                graw[jj] = fetch(g + base + (int64_t)(j0 + jj < held ? j0 + jj : held - 1) * plane);
#pragma unroll
            for (int jj = 0; jj < kChunk; ++jj) {
                float r[V];
                float sg = 0.f, sgy = 0.f;
                const float w = Affine ? wb[0][c0 + (j0 + jj < held ? j0 + jj : 0)] : 1.f;
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float val = PK::get(raw[j0 + jj], k);
                    float gv = PK::get(graw[jj], k);
                    const float inner = __builtin_fmaf((val - mean[k]) * (val - inv_c), mv[k], inv_c);
                    if constexpr (Affine) {
                        sg += gv;
                        // a partly filled lane's missing pixels are zeros, normalised to NaN where eps is 0
                        const float y = (val - mean[k]) * rstd[k];
                        sgy = __builtin_fmaf(PerImage && k >= nv ? 0.f : y, gv, sgy);
                        gv *= w;
                    }
                    r[k] = -rstd[k] * inner * gv;
                }
                if (live && j0 + jj < held) put_back(out + base + (int64_t)(j0 + jj) * plane, r);
                if constexpr (kSums) {
                    part[2 * jj] = live ? sgy : 0.f;
                    part[2 * jj + 1] = live ? sg : 0.f;
                }
            }
            if constexpr (kSums) {
                if (p.partials) sums[j0 / kChunk] += ln_transpose_sum<2 * kChunk>(part, lane);
            }
        }
    }
    if constexpr (!kSums) return;
    turn ^= 1;
    }
    if constexpr (kSums) {
        if (!p.partials) return;                       // grid-uniform
        // lane i of a wave holds value i / (64 / (2 * kChunk)) of every chunk; rows of sums are [C][2]
        constexpr int kSpan = 64 / (2 * kChunk);
        float *row = p.partials + (int64_t)blockIdx.x * 2 * p.C;
        if constexpr (WS > 1) {
#pragma unroll
            for (int h = 0; h < KW / kChunk; ++h) {
                const int ch = h * kChunk + lane / kSpan / 2;
                if (lane % kSpan == 0 && ch < cnt) row[2 * (c0 + ch) + ((lane / kSpan) & 1)] = sums[h];
            }
        } else {
            __shared__ float all[4][2 * KW];           // the four waves of the block hold all channels each
#pragma unroll
            for (int h = 0; h < KW / kChunk; ++h)
                if (lane % kSpan == 0) all[wave][h * 2 * kChunk + lane / kSpan] = sums[h];
            __syncthreads();
            for (int i = threadIdx.x; i < 2 * p.C; i += kLnBlock) row[i] = (all[0][i] + all[1][i]) + (all[2][i] + all[3][i]);
        }
    }
}

// Any C: G lanes share one slice and stride over it (G = 64: a wavefront per contiguous row;
// G = 1: a lane per slice). Statistics from sums shifted by the mean of the slice's first elements, which keeps
// the one-pass variance well conditioned; the second sweep re-reads the slice through cache.
template <class T, int G, bool Bwd>
__global__ __launch_bounds__(256) void ln_group(const T *__restrict__ x, const T *__restrict__ g, T *__restrict__ out,
                                                const LnParams p) {
    constexpr int kPix = 256 / G;
    const int sub = threadIdx.x % G, grp = threadIdx.x / G;
    const float inv_c = 1.f / (float)p.C;
    const int64_t rounds = ceil_div_dev(p.P, (int64_t)gridDim.x * kPix);
    for (int64_t rd = 0; rd < rounds; ++rd) {
        const int64_t pix = (rd * gridDim.x + blockIdx.x) * kPix + grp;
        const bool live = pix < p.P;
        const int64_t pc = live ? pix : 0;
        const int64_t n = pc / p.m_size;
        const int64_t base = pc + n * (int64_t)(p.C - 1) * p.m_size;
        // The shift is the mean of the slice's first (up to) 8 elements: a single element can sit several standard
        // deviations from the mean, and E[d^2] - E[d]^2 then cancels digits (shifted by its first element, a slice
        // of 1317 channels missed 1e-5 by a factor of 4). Four independent partial sums per lane keep the rounding
        // of the long sums down and eight loads in flight.
        const int n_shift = p.C < 8 ? p.C : 8;
        float shift = 0.f;
        for (int j = 0; j < n_shift; ++j) shift += load_one(x + base + (int64_t)j * p.m_size);
        shift *= 1.f / (float)n_shift;
        float a1[4] = {0.f, 0.f, 0.f, 0.f}, a2[4] = {0.f, 0.f, 0.f, 0.f};
        int j = sub;
#pragma unroll 2
        for (; j + 3 * G < p.C; j += 4 * G) {
            float d[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) d[u] = load_one(x + base + (int64_t)(j + u * G) * p.m_size) - shift;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a1[u] += d[u];
                a2[u] = __builtin_fmaf(d[u], d[u], a2[u]);
            }
        }
        for (; j < p.C; j += G) {
            const float d = load_one(x + base + (int64_t)j * p.m_size) - shift;
            a1[0] += d;
            a2[0] = __builtin_fmaf(d, d, a2[0]);
        }
        float s1 = (a1[0] + a1[1]) + (a1[2] + a1[3]), s2 = (a2[0] + a2[1]) + (a2[2] + a2[3]);
        s1 = group_reduce<G>(s1, OpSum());
        s2 = group_reduce<G>(s2, OpSum());
        const float dm = s1 * inv_c;
        const float mean = shift + dm;
        const float var = fmaxf(s2 * inv_c - dm * dm, 0.f);
        const float v = var + p.eps;
        const float rstd = 1.f / sqrtf(v), mv = mean * v;
        if (!live) continue;
#pragma unroll 8
        for (int j = sub; j < p.C; j += G) {
            const int64_t at = base + (int64_t)j * p.m_size;
            const float val = load_one(x + at);
            if constexpr (Bwd) {
                const float inner = __builtin_fmaf((val - mean) * (val - inv_c), mv, inv_c);
                store_one(out + at, -rstd * inner * load_one(g + at));
            } else {
                store_one(out + at, (val - mean) * rstd);
            }
        }
    }
}

// Rows of sums in the affine backward: column by column in a fixed order, in the parameters' type. A block takes 16
// columns (64 bytes of every row) with 64 rows in flight.
template <class T>
__global__ __launch_bounds__(1024) void ln_finish_sums(const float *__restrict__ partials, int rows, int C,
                                                       T *__restrict__ grad_weight, T *__restrict__ grad_bias) {
    __shared__ float part[64][17];
    const int col = blockIdx.x * 16 + (threadIdx.x & 15), first = threadIdx.x >> 4;
    float s = 0.f;
    if (col < 2 * C) {
#pragma unroll 8
        for (int r = first; r < rows; r += 64) s += partials[(int64_t)r * 2 * C + col];
    }
    part[first][threadIdx.x & 15] = s;
    __syncthreads();
#pragma unroll
    for (int half = 32; half > 0; half >>= 1) {
        if (first < half) part[first][threadIdx.x & 15] += part[first + half][threadIdx.x & 15];
        __syncthreads();
    }
    if (first == 0 && col < 2 * C) store_one((col & 1 ? grad_bias : grad_weight) + (col >> 1), part[0][threadIdx.x & 15]);
}

// The shapes that have an affine form: what ln_regs serves.
inline bool ln_has_affine(int64_t dimsize, int64_t m_size) { return m_size > 1 && dimsize <= 1024; }

// Blocks of the affine backward, which loop over the pixel groups: enough to fill the chip with the blocks that fit it
// at once (two of 512 threads per CU, eight of 256), twice over.
inline unsigned ln_sum_blocks(int64_t dimsize, int64_t blocks) {
    const int64_t cap = dimsize > 64 ? 1024 : 2048;
    return (unsigned)(blocks < cap ? blocks : cap);
}

template <class T, bool Bwd, bool Affine>
void ln_launch(const T *x, const T *g, T *out, int64_t n_size, int64_t dimsize, int64_t m_size, float eps,
               const LnAffine<T> &af, hipStream_t st) {
    constexpr int VT = ElemTraits<T>::kVec;
    LnParams p = {};
    p.weight = af.weight;
    p.bias = af.bias;
    p.P = n_size * m_size;
    p.m_size = m_size;
    p.C = (int)dimsize;
    p.eps = eps;
    // Channels per wave: all of them up to 32, a quarter up to 64, an eighth beyond (smaller register
    // chunks in more waves measured better: they overlap one wave's loads with another's stores).
    // With 4 waves and C > 32, or 8 waves and C > 64, every wave holds at least one channel.
    const int ws = dimsize > 64 ? 8 : (dimsize > 32 ? 4 : 1);
    p.per_wave = (int)ceil_div(dimsize, ws);
    if (!ln_has_affine(dimsize, m_size)) {
        if constexpr (Affine) return;
        if (m_size == 1) {
            hipLaunchKernelGGL((ln_group<T, 64, Bwd>), dim3(group_grid(p.P, 4)), dim3(256), 0, st, x, g, out, p);
        } else {
            hipLaunchKernelGGL((ln_group<T, 1, Bwd>), dim3(group_grid(p.P, 256)), dim3(256), 0, st, x, g, out, p);
        }
        return;
    }
    const bool vec = dimsize <= 768 && m_size % VT == 0 && !misaligned(x, VT * sizeof(T)) &&
                     !misaligned(out, VT * sizeof(T)) && !(Bwd && misaligned(g, VT * sizeof(T)));
    // planes that start on element boundaries only (odd lengths, misaligned tensors) and are long enough that
    // the partly filled last group of every image is a small share: the same pixels per lane in groups per image
    const bool image = !vec && dimsize <= 768 && m_size >= 4096;
    const int slots = p.per_wave;
    // 16-bit elements, more than 48 slots per wave: 64 and 96 slots of four pixels are 256 and 384 values per lane, and
    // where the kernel spills them (up to 1168 bytes per lane: the per-image form, and fp16 with 96 slots) two pixels per
    // lane are faster: fp16 (32,768,4098) forward 0.565 -> 0.174 ms, backward 0.739 -> 0.271; (32,768,4096) 0.109 -> 0.092
    // and 0.180 -> 0.172. (bf16 on aligned planes keeps four: 0.129 against 0.192 ms backward at (32,768,4096).)
    constexpr int VN = (sizeof(T) == 2) ? 2 : VT;
    const bool narrow = sizeof(T) == 2 && ws == 8 && slots > 48 && slots <= 96 &&
                        (image || (vec && std::is_same<T, f16>::value && slots > 64));
    const int vv = narrow ? VN : VT;
    const int64_t groups = image ? n_size * ceil_div(m_size, 64 * vv) : ceil_div(p.P, 64 * (vec ? vv : 1));
    p.groups = groups;
    unsigned grid = (unsigned)(ws > 1 ? groups : ceil_div(groups, 4));
    if constexpr (Affine && Bwd) {
        grid = ln_sum_blocks(dimsize, grid);
        p.partials = af.partials;
    }
#define PLH_LN(KW, VV, WS) \
    hipLaunchKernelGGL((ln_regs<T, KW, VV, WS, Bwd, false, Affine>), dim3(grid), dim3(WS > 4 ? 64 * WS : kLnBlock), 0, st, x, g, out, p)
#define PLH_LN_IMAGE(KW, WS) \
    hipLaunchKernelGGL((ln_regs<T, KW, VT, WS, Bwd, true, Affine>), dim3(grid), dim3(WS > 4 ? 64 * WS : kLnBlock), 0, st, x, g, out, p)
#define PLH_LN_V(KW, WS) do { if (vec) PLH_LN(KW, VT, WS); else if (image) PLH_LN_IMAGE(KW, WS); else PLH_LN(KW, 1, WS); } while (0)
#define PLH_LN_NARROW(KW, WS)                                                                                              \
    do {                                                                                                                   \
        if (vec) PLH_LN(KW, VN, WS);                                                                                       \
        else if (image)                                                                                                    \
            hipLaunchKernelGGL((ln_regs<T, KW, VN, WS, Bwd, true, Affine>), dim3(grid), dim3(64 * WS), 0, st, x, g, out, p);       \
        else PLH_LN(KW, 1, WS);                                                                                            \
    } while (0)
    // Slot counts in steps of about 1.5x: a wave whose channels fall short of its slots re-reads its last
    // channel for the rest, and at 12 channels in 16 slots that cost a third of the bandwidth.
    if (ws == 1) {
        if (slots <= 8) PLH_LN_V(8, 1);
        else if (slots <= 12) PLH_LN_V(12, 1);
        else if (slots <= 16) PLH_LN_V(16, 1);
        else if (slots <= 24) PLH_LN_V(24, 1);
        else PLH_LN_V(32, 1);
    } else if (ws == 4) {
        if (slots <= 12) PLH_LN_V(12, 4);
        else PLH_LN_V(16, 4);
    } else if (slots <= 12) PLH_LN_V(12, 8);
    else if (slots <= 16) PLH_LN_V(16, 8);
    else if (slots <= 24) PLH_LN_V(24, 8);
    else if (slots <= 32) PLH_LN_V(32, 8);
    else if (slots <= 48) PLH_LN_V(48, 8);
    else if (slots <= 64) { if (narrow) PLH_LN_NARROW(64, 8); else PLH_LN_V(64, 8); }
    else if (slots <= 96) { if (narrow) PLH_LN_NARROW(96, 8); else PLH_LN_V(96, 8); }      // C <= 768
    else PLH_LN(128, 1, 8);                            // 768 < C <= 1024: one pixel per lane
#undef PLH_LN_NARROW
#undef PLH_LN_V
#undef PLH_LN_IMAGE
#undef PLH_LN
    if constexpr (Affine && Bwd) {
        if (af.partials)
            hipLaunchKernelGGL(ln_finish_sums<T>, dim3((unsigned)ceil_div(2 * dimsize, 16)), dim3(1024), 0, st, af.partials, (int)grid,
                               p.C, af.grad_weight, af.grad_bias);
    }
}

// Per-dtype entries, instantiated in layernorm_{f32,f16,bf16}.hip (plain) and layernorm_{f32,f16,bf16}_affine.hip.
template <class T>
void ln_run_typed(bool bwd, const T *x, const T *g, T *out, int64_t n_size, int64_t dimsize, int64_t m_size, float eps,
                  hipStream_t st) {
    if (bwd) ln_launch<T, true, false>(x, g, out, n_size, dimsize, m_size, eps, LnAffine<T>{}, st);
    else ln_launch<T, false, false>(x, g, out, n_size, dimsize, m_size, eps, LnAffine<T>{}, st);
}
template <class T>
void ln_run_affine(bool bwd, const T *x, const T *g, T *out, int64_t n_size, int64_t dimsize, int64_t m_size, float eps,
                   const LnAffine<T> &af, hipStream_t st) {
    if (bwd) ln_launch<T, true, true>(x, g, out, n_size, dimsize, m_size, eps, af, st);
    else ln_launch<T, false, true>(x, g, out, n_size, dimsize, m_size, eps, af, st);
}

#define PLH_LN_SIGNATURE(T) void ln_run_typed<T>(bool, const T *, const T *, T *, int64_t, int64_t, int64_t, float, hipStream_t);
#define PLH_LN_AFFINE_SIGNATURE(T) \
    void ln_run_affine<T>(bool, const T *, const T *, T *, int64_t, int64_t, int64_t, float, const LnAffine<T> &, hipStream_t);
#define PLH_LN_EXTERN(T) extern template PLH_LN_SIGNATURE(T) extern template PLH_LN_AFFINE_SIGNATURE(T)
#define PLH_LN_INSTANTIATE(T) template PLH_LN_SIGNATURE(T)
#define PLH_LN_INSTANTIATE_AFFINE(T) template PLH_LN_AFFINE_SIGNATURE(T)

}  // namespace plh
