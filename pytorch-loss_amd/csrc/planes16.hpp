// Backward of 16-bit channel planes that do not start on 128-byte lines (513 x 513 crops) from what the forward left per pixel
// (LSR: the largest logit and the sum of exponentials; Taylor cross entropy: S), plane by plane: included by lsr_kernels.hpp and
// taylor_kernels.hpp.
//
// With that at hand an element's gradient needs no other channel, so a block takes 2048 pixels of an image and in
// every plane its 256 threads move the 32 whole lines that begin at the tile's first pixel shifted back by the plane's offset
// into its line: 16 aligned bytes per lane, loads and stores alike, four planes in flight. The pixels' values and labels are
// staged in LDS, transposed by pixel mod 8, so that a lane's window of 8 pixels reads without bank conflicts from one
// address and constants per plane. Bound by memory: of LSR's 160 us at (16,19,769,769) bf16 the walk alone, a copy with nothing
// staged, takes 122 (5.9 TB/s; a copy in the order of the addresses 113), with labels and 4 bytes per pixel staged 149, with
// LSR's 6 bytes 154.
#pragma once
#include "plh_common.hpp"

namespace plh {

// Where the pair can run: from 16 channels on (2 channels of 769 x 769: 452 -> 576 us), and not on planes of whole lines (LSR
// (8,150,512,512) 398 -> 414, Taylor 356 -> 373).
inline bool planes16_apply(size_t elem_bytes, int64_t dimsize, int64_t m_size) {
    if (elem_bytes != 2 || dimsize < 16 || m_size < 4096 || m_size * 2 % 128 == 0) return false;
    return dimsize <= kMaxRegsChannels ? image_form_pays<bf16>((int)dimsize, m_size) : dimsize <= kMaxSplitChannels;
}

// Where a step with the pair is no slower than one with the kernels that recompute. What it gains are the lines that planes
// share, which come from HBM twice; what it costs are 4 (Taylor) or 6 bytes per pixel and a block that waits for its stage. Under
// the 256 MiB of the cache in front of HBM there is little to gain: graph-timed steps recomputed -> with the pair, bf16, us
//   (2,16,257,257) LSR 25 -> 45, (8,20,513,513) 81 -> 92, (8,32,513,513) 113 -> 130, (4,40,129,129) 29 -> 35; Taylor (28,16,129,129) 30 -> 54
// and above it the gain grows with the planes:
//   16..32 channels: (16,19,769,769) 360 MB LSR 262 -> 258, Taylor 275 -> 252; of 340..640 MB on 769 x 769 LSR +2..-10 %,
//     Taylor -1..-11, on 1021 x 1021 +3..-5, -1..-10, on 1281 x 1281 -1..-8, -3..-13; of 500 MB on 513 x 513 +4..-2, -3..-5, on
//     129 x 129 +3..+8, +4..-3
//   33..128: of 315..500 MB on 513 x 513 LSR -2..-11 %, Taylor -7..-25; on 129 x 129 +4..-9, 0..-18; on 65 x 67 Taylor up to +4
// The kernels that recompute hold 33 and more channels in slots of 8 wavefronts (split_slots), and lose by what they hold: with
// more slots than channels by a whole wavefront, or a few wavefronts per CU, the pair gains from some 32 MB on:
//   LSR 97..104 channels +3..-24 %, 129..256 +2..-36 (two sizes of 160 +5 and +7); 105..128: +7..-20
//   Taylor 97..128 +1..-26 %, 161..256 +4..-34; 129..160: +10..-19
// and with fewer bytes (129..256 channels of 129 x 129, 4 MB) +8, Taylor +19.
inline bool planes16_pays(bool lsr, size_t elem_bytes, int64_t n_size, int64_t dimsize, int64_t m_size) {
    if (!planes16_apply(elem_bytes, dimsize, m_size)) return false;
    const int64_t bytes = n_size * dimsize * m_size * (int64_t)elem_bytes;
    if (dimsize > 96 && (lsr ? dimsize <= 104 || dimsize > 128 : dimsize <= 128 || dimsize > 160)) return bytes >= (int64_t)1 << 25;
    const int64_t plane = dimsize <= kMaxRegsChannels ? 768 * 768 : (lsr ? 1 << 18 : 1 << 14);
    return m_size >= plane && bytes >= (int64_t)5 << 26;
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
