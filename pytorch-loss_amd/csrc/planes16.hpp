// Backward of 16-bit channel planes that do not start on 128-byte lines (513 x 513 crops) from what the forward left per pixel
// (LSR: the largest logit and the sum of exponentials; Taylor cross entropy: S), plane by plane: included by lsr_kernels.hpp and
// taylor_kernels.hpp.
//
// With that at hand an element's gradient needs no other channel, so a block takes 2048 pixels of an image and in
// every plane its 256 threads move the 32 whole lines that begin at the tile's first pixel shifted back by the plane's offset
// into its line: 16 aligned bytes per lane, loads and stores alike, four planes in flight. The pixels' values and labels are
// staged in LDS, transposed by pixel mod 8, so that a lane's window of 8 pixels reads without bank conflicts from one
// address and constants per plane. Bound by memory: the walk alone, a copy, takes 148 of the 150 us at (16,19,769,769) bf16
// (5.5 TB/s; a copy in the order of the addresses 6.2), with LSR's 6 bytes per pixel 168.
#pragma once
#include "plh_common.hpp"

namespace plh {

// Where the pair runs. Steps with the kernels that recompute -> with it, bf16, us: LSR, which keeps 6 bytes per pixel,
// (16,19,769,769) 269 -> 260, (9,32,770,766) 251 -> 229, (8,150,513,513) 509 -> 440, (6,200,513,513) 684 -> 510; Taylor, 4,
// (30,40,513,513) 483 -> 459, (8,150,513,513) 483 -> 396.
// Below 16 channels the forward's float weighs more than the backward gains (2 channels of 769 x 769: 452 -> 576), and on
// planes of whole lines the kernels that recompute are the faster ones (LSR (8,150,512,512) 398 -> 414, Taylor 356 -> 373).
inline bool planes16_apply(size_t elem_bytes, int64_t dimsize, int64_t m_size) {
    if (elem_bytes != 2 || dimsize < 16 || m_size < 4096 || m_size * 2 % 128 == 0) return false;
    return dimsize <= kMaxRegsChannels ? image_form_pays<bf16>((int)dimsize, m_size) : dimsize <= kMaxSplitChannels;
}

template <class T, class Op>
__global__ __launch_bounds__(256) void planes16_bwd(const T *__restrict__ x, const int64_t *__restrict__ lab,
                                                    const Upstream up, T *__restrict__ grad, Op op, int64_t M, int C, int64_t ignore, int tiles, int planes_per_block) {
    using G = PlaneGeom<T>;
    constexpr int kPer = G::kPer, kTile = G::kTile, kHalo = G::kHalo, kCols = (kTile + kHalo) / kPer;
    static_assert(sizeof(T) == 2 && kPer == 8, "8 elements of 16 bits per lane");
    using Pixel = typename Op::Pixel;
    static_assert(sizeof(Pixel) == 8, "a lane's window without bank conflicts");
    __shared__ Pixel pairs[kPer][kCols];            // entry i at [i % kPer][i / kPer]
    const int64_t n = blockIdx.x / tiles;
    const int t = (int)(blockIdx.x - n * tiles), l = threadIdx.x;
    float gk = up.gout ? *up.gout * up.scale : up.scale;
    if (up.divide_by) gk = gk / (float)(*up.divide_by);
    op.begin(gk);
    auto pixel = [&](int64_t q) { return q >= 0 && q < M ? op.pixel(n * M + q, lab[n * M + q], ignore, C) : Op::nothing(); };
    auto shift_of = [&](const T *plane) { return (int)((reinterpret_cast<uintptr_t>(plane) / 2) & (unsigned)(G::kLine - 1)); };
    const int64_t first = (int64_t)t * kTile - kHalo;
    for (int i = l; i < kTile + kHalo; i += 256) pairs[i % kPer][i / kPer] = pixel(first + i);
    __syncthreads();
    constexpr int U = 4;                            // planes in flight per thread
    const int c_begin = blockIdx.y * planes_per_block;
    const int c_end = c_begin + planes_per_block < C ? c_begin + planes_per_block : C;
    for (int c0 = c_begin; c0 < c_end; c0 += U) {
        plh_u4 xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const T *plane = x + (n * C + (c0 + u < c_end ? c0 + u : c_end - 1)) * M;
            const int64_t q = (int64_t)t * kTile - shift_of(plane) + kPer * l;
            // (the ends of a plane: its first aligned chunk, not used)
            xv[u] = __builtin_nontemporal_load(reinterpret_cast<const plh_u4 *>(plane + (q >= 0 && q + kPer <= M ? q : -shift_of(plane) & (kPer - 1))));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u;
            if (c >= c_end) break;
            const int64_t at = (n * C + c) * M;
            const int shift = shift_of(x + at);
            const int64_t q = (int64_t)t * kTile - shift + kPer * l;
            // staged entry kHalo + 8 l - shift + d: row (s + d) % 8, column l and a constant of the plane
            const int s = -shift & (kPer - 1), col = (kHalo - shift - s) / kPer;
            auto px = [&](int d) { return pairs[(s + d) & (kPer - 1)][l + col + ((s + d) >> 3)]; };
            if (q >= 0 && q + kPer <= M) {
                const unsigned in[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
                unsigned out[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const Pixel a = px(2 * d), b = px(2 * d + 1);
                    const float ga = op.grad(widen_lo(in[d], T{}), a, c), gb = op.grad(widen_hi(in[d], T{}), b, c);
                    out[d] = narrow2(a.dropped() ? 0.f : ga, b.dropped() ? 0.f : gb, T{});
                }
                __builtin_nontemporal_store(plh_u4{out[0], out[1], out[2], out[3]}, reinterpret_cast<plh_u4 *>(grad + at + q));
            } else {                                // the two ends of a plane, element by element
#pragma unroll
                for (int d = 0; d < kPer; ++d)
                    if (q + d >= 0 && q + d < M) {
                        const Pixel a = px(d);
                        float g = op.grad(load_one(x + at + q + d), a, c);
                        asm("" : "+v"(g));          // rounded to fp32 first, as above: not one v_fma_mixlo_f16
                        store_one(grad + at + q + d, a.dropped() ? 0.f : g);
                    }
            }
        }
    }
}

// Planes that a block walks: its share of a tile's, so that the last wave of blocks is short. us of the backward with 8, 12, 16,
// 28 and 40 planes: (16,19,769,769) 159 150 150 154 -, (9,32,769,769) 147 142 146 156 -, (8,150,513,513) 237 241 246 259 269,
// (6,200,513,513) 268 253 254 269 288, (2,40,513,513) 30 33 36 51 65, (1,150,257,257) 20 26 30 44 60.
inline int planes16_per_block(int64_t tiles, int C) {
    if (C <= kMaxRegsChannels) return 16;
    return tiles * ceil_div(C, 12) < 4096 ? 8 : 12;
}

// Logits and gradient at the same offset into a 128-byte line (whole lines of the one are whole lines of the other), one scalar
// upstream gradient. False: nothing was launched.
template <class T, class Op>
inline bool planes16_launch(const T *x, const int64_t *lab, const Upstream &up, T *grad, const Op &op, int64_t P, int64_t M, int C,
                            int64_t ignore, hipStream_t st) {
    const int64_t tiles = ceil_div(M + PlaneGeom<T>::kHalo - 1, (int64_t)PlaneGeom<T>::kTile), all = P / M * tiles;
    if (((reinterpret_cast<uintptr_t>(x) ^ reinterpret_cast<uintptr_t>(grad)) & 127) != 0 || misaligned(x, 2) || all >= ((int64_t)1 << 31))
        return false;
    const int per = planes16_per_block(all, C);
    hipLaunchKernelGGL((planes16_bwd<T, Op>), dim3((unsigned)all, (unsigned)ceil_div(C, per)), dim3(256), 0, st, x, lab, up, grad, op, M, C,
                       ignore, (int)tiles, per);
    return true;
}

}  // namespace plh
