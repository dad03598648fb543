// The sort of the Lovasz forward by value buckets (included by lovasz.hip, after the keys and the rank primitives).
//
// A radix sort moves every (key, pixel) pair three times before its rank is known. Here a key moves inside its tile only: the
// class row is cut into buckets of neighbouring key values, every tile is put in the order of the buckets, and what lies in a
// few neighbouring buckets, a segment of every tile, is sorted in a block's LDS.
//   bk_sample     the classes' limits, and a sample of their keys
//   bk_split      a block per class sorts the sample; every n-th key of it starts a bucket
//   bk_cut        every tile's keys in the order of their buckets, in pixel order inside one (stable ranks), in the keys' place
//   bk_sum        the tiles' counts by bucket: where every bucket starts in the row
//   bk_group      runs of buckets that a block can sort at once
//   bk_rank       a block per run of buckets: its segments sorted in LDS, Jaccard difference of every key in its place
//   bk_rank_rest  the same for runs whose values crowd, and for buckets that outgrew the LDS (wide)
//   bk_restore    Jaccard differences back to pixel order, tile by tile, with those of single values that fill more than a block
// Sampled bounds follow any distribution; a value that fills several buckets by itself gets one of its own, which
// needs no sort (flat: its keys are ranked as they stand), and a bucket that outgrew the LDS all the same is cut into value
// ranges that fit.
// A key moves 28 bytes: read and written by bk_cut, bk_rank and bk_restore, and a place of 2 bytes. The form before this one
// wrote the buckets out one after the other: that takes a histogram first (6 bytes a key more, buckets kept for the second
// pass) and writes of some 10 keys, where a segment of a run has 24 here. (4,19,512,1024) fp32: histogram and scatter
// 67 + 117 us against 93 now, rank 119 against 105, gather 72 against 56, step 557 -> 437 us; (8,21,513,513) bf16 trained
// 77 + 154 against 130, 217 against 231, 116 against 70, step 792 -> 618. Which rows come here: bk_pays.
#pragma once

namespace plh {

constexpr int kBkThreads = 512;
constexpr int kBkItems = 15;
constexpr int kBkCap = kBkThreads * kBkItems;       // keys a block sorts at once: 8 bytes each, two blocks per CU
constexpr int kBkTileItems = 16;
constexpr int kBkTile = kBkThreads * kBkTileItems;  // keys of a tile
constexpr int kBkWaves = kBkThreads / kWave;
constexpr int kBkChunk = 16;                        // neighbours in the order that one thread sorts
constexpr int kBkBins = 4096;                       // bins of a run's value range
constexpr int kBkFineBits = 13;                     // table from a key's top bits to the first bucket it can be in
constexpr int kBkFine = 1 << kBkFineBits;
constexpr int kBkTarget = 2560;                     // mean keys per bucket: sampled bounds leave few above kBkCap
constexpr int kBkSlab = 6144;                       // buckets that start in one such part of the row are sorted together
constexpr int kBkMax = 1024;                        // buckets per class
constexpr int64_t kBkMaxRow = (int64_t)kBkTarget * kBkMax;
constexpr uint32_t kBkCrowd = 257;                  // keys in one bin up to which merges between chunks put them in order: 97 left
                                                    // lumps of bf16 logits to the crowded path (227 + 37 -> 231 + 9 us)
constexpr uint16_t kBkNowhere = 0xFFFFu;            // place of a pixel that takes no part

struct BucketArgs {
    uint32_t *keys;             // [C][P] in pixel order; bk_cut leaves every tile's keys by bucket, the rank kernels a key's Jaccard
                                // difference in its place, bk_restore those in pixel order (jacc's memory)
    uint32_t *pos_max;          // pos_max[C], kept[C], all_min[C], key_bits[C] (see keep_key, publish_class); not for a row of one block
    const uint32_t *block_table;        // [C][key_blocks] largest positive key plus 1 that a block of lov_keys_* met
    uint16_t *place;            // [C][P] every pixel's place in its tile's order
    uint32_t *sorted, *dj;      // [C][P] keys and differences of the wide buckets; in dj's memory first the
                                // sample, [C][kBkCap]
    uint32_t *tile_start;       // [C][tiles][stride + 1] in the tile's order: keys | positives << 16 before the bucket
    uint32_t *start;            // [C][stride + 1][tiles] the same
    uint32_t *base, *hot_base;  // [C][stride + 1] keys and positives before the bucket
    uint32_t *bounds;           // [C][stride] least key of buckets 1, 2, ...
    uint32_t *runs;             // [C][stride + 1] first bucket of every run, and the end
    uint32_t *large;            // [C][stride] buckets of more keys than kBkCap: the wide ones, then the flat ones
    uint32_t *crowded;          // [C][stride] runs whose values crowd, in any order
    uint32_t *numbers;          // [9][C]: buckets, runs, positives, least key of the sample, largest one below the limit,
                                // first step of the search in `bounds`, wide buckets, flat buckets, crowded runs
    uint16_t *fine;             // [C][kBkFine] bucket of the least key with these top bits
    double *loss_part;          // [C][2 * stride]: runs, from `stride` on large buckets
    int P, C, tiles, stride, key_blocks;
};

__device__ __forceinline__ uint32_t bk_limit(const BucketArgs &a, int c) {
    const uint32_t m = a.pos_max[c];
    if (m) return m - 1u;
    const uint32_t lowest = a.pos_max[2 * a.C + c];
    return lowest <= kOne ? lowest : kOne;
}

// A class's loss with one term more. The product of two floats is exact in double, and the terms are added in a fixed order:
// small losses keep their digits, and a loss is the same on every call. Another order of the terms (radix passes, buckets)
// moves the sum by a few 2^-53 of it, which its rounding to float all but never shows.
__device__ __forceinline__ double add_loss(double sum, float e, float dj) {
    return __builtin_fma((double)e, (double)dj, sum);
}
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// a / b as the division operator rounds it, for whole numbers 0 <= a <= b <= kBkMaxRow, b > 0: Newton's step on the reciprocal
// leaves it 2^-24 of its value off, the product 2 units in its last place, the residual's correction 2^-23 of a unit. No
// quotient of such numbers is nearer than 1 / 2b > 2^-23 of a unit to where the rounding changes (2a / unit and b times an odd
// number are whole and differ). The operator's second residual and its scaling are for other operands.
__device__ __forceinline__ float whole_ratio(float a, float b) {
    float y = __builtin_amdgcn_rcpf(b);
    y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.f), y, y);
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
static_assert(kBkMaxRow < 1 << 22, "2b < 2^23");

// Jaccard index of a class's first k keys, cs of its npos positives among them: a multiple of 2^-24, whatever the division
// gives (a quotient from 1/2 on is one, and its difference from 1 is exact; one below leaves a difference from 1/2 on).
__device__ __forceinline__ float jaccard(float npos, uint32_t k, uint32_t cs) {
    const float inter = npos - (float)cs;
    return k == 0 ? 0.f : 1.f - whole_ratio(inter, inter + (float)k);
}

// Jaccard difference of the key at rank `pos`, with `cs` of the class's npos positives before it. kAnyRow: rows of more than
// kBkMaxRow pixels too, by all of the division operator's steps (whole numbers below 2^31 need none of its scaling).
template <bool kAnyRow = false>
__device__ __forceinline__ float jaccard_step(float npos, uint32_t pos, uint32_t cs, uint32_t hot) {
    auto ratio = [](float a, float b) { return kAnyRow ? DivideBy(b)(a) : whole_ratio(a, b); };
    const float inter_prev = npos - (float)cs;                             // csrc/lovasz_softmax.cu:124-127
    const float inter = npos - (float)(cs + hot);
    const float j_now = 1.f - ratio(inter, inter + (float)(pos + 1));
    const float j_prev = (pos == 0) ? 0.f : 1.f - ratio(inter_prev, inter_prev + (float)pos);
    return j_now - j_prev;                                                 // csrc/lovasz_softmax.cu:141-147
}

// A key, its place among the block's items and its positive flag, ordered as the stable sort orders them, as a double in
// [1, 2): the smaller and the larger of two are one instruction each.
typedef double BkPair;
__device__ __forceinline__ BkPair bk_pair(uint32_t key, uint32_t item) {
    const uint32_t hi = __builtin_amdgcn_alignbit(0x3FF00000u >> 14, key & 0x7FFFFFFFu, 18);       // exponent | key >> 18
    const uint32_t lo = key << 14 | __builtin_amdgcn_alignbit(item, key, 31);                      // item << 1 | key >> 31
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ uint32_t bk_item_of(BkPair p) { return ((uint32_t)__builtin_bit_cast(uint64_t, p) >> 1) & 0x1FFFu; }
__device__ __forceinline__ uint32_t bk_hot_of(BkPair p) { return (uint32_t)__builtin_bit_cast(uint64_t, p) & 1u; }
__device__ __forceinline__ uint32_t bk_key_of(BkPair p) {              // below 2^30: the exponent's bits fall out
    return (uint32_t)(__builtin_bit_cast(uint64_t, p) >> 14);
}
__device__ __forceinline__ BkPair bk_last() { return __builtin_bit_cast(double, (uint64_t)0x3FFFFFFFFFFFFFFEull); }   // no positive
static_assert(kBkCap <= 1 << 13 && kOne < 1u << 30, "13 bits of a pair name the item, 30 hold the key");

__device__ __forceinline__ void bk_order(BkPair &a, BkPair &b) {
    double lo, hi;                              // asm: fmin and fmax would quiet signalling NaNs first
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}
// Batcher's odd-even merges of a chunk's runs of kFrom, 2 kFrom, ... pairs (kFrom = 1: the sort, 63 pairs ordered;
// kFrom = 8: the merge of its halves, 25).
template <int kFrom>
__device__ __forceinline__ void bk_merge(BkPair (&v)[kBkChunk]) {
#pragma unroll
    for (int p = kFrom; p < kBkChunk; p *= 2)
#pragma unroll
        for (int k = p; k >= 1; k /= 2)
#pragma unroll
            for (int i = 0; i < kBkChunk; ++i) {
                // i and i + k: not across the runs being merged, and only the pairs of this step
                const bool pair = i >= k % p && ((i - k % p) / k) % 2 == 0 && i + k < kBkChunk && i / (2 * p) == (i + k) / (2 * p);
                if (pair) bk_order(v[i], v[i + k]);
            }
}

// Where the keys of a few neighbouring buckets stand: in every tile a segment of its order. The segments one after the other are
// the keys in the order that the sort keeps among equals; places from..from + kBkCap - 1 of it are covered.
constexpr int kBkWords = kBkCap / kWave;
constexpr int kBkGroup = 3;                     // rounds whose LDS accesses are waited for together
static_assert(kBkItems % kBkGroup == 0, "groups of rounds");
struct BkSegments {
    struct alignas(16) Word {
        uint64_t starts;                        // bit i: a segment starts at place 64 k + i + 1
        uint32_t segment, unused;               // that of place 64 k
    };
    Word word[kBkWords + kBkGroup - 1];         // the last ones are looked at, and not used
    uint32_t shift[kBkMaxRow / kBkTile + 1];    // where the segment starts in the row less its first place
    // The thread's tile: first key of the buckets from b0 to before b1 in its order, and their number.
    struct Tile {
        uint32_t first, keys;
        __device__ __forceinline__ Tile() : first(0), keys(0) {}
        __device__ __forceinline__ Tile(const BucketArgs &a, int c, uint32_t b0, uint32_t b1) : first(0), keys(0) {
            const int64_t cell = (int64_t)c * (a.stride + 1);
            if ((int)threadIdx.x < a.tiles) {
                first = a.start[(cell + b0) * a.tiles + threadIdx.x] & 0xFFFFu;
                keys = (a.start[(cell + b1) * a.tiles + threadIdx.x] & 0xFFFFu) - first;
            }
        }
    };
    // Every thread of the block calls it; ends with a barrier. The memory is free before, with a barrier in between.
    __device__ __forceinline__ void collect(const Tile tile, uint32_t from, uint32_t *scan) {
        uint32_t *words = reinterpret_cast<uint32_t *>(word);
        if (threadIdx.x < 4 * (kBkWords + kBkGroup - 1)) words[threadIdx.x] = 0;
        const uint32_t n = tile.keys;
        uint32_t place, all, index, segments;
        block_excl_scan2(n, n ? 1u : 0u, scan, place, all, index, segments);
        if (n && place + n > from && place < from + kBkCap) {
            shift[index] = threadIdx.x * kBkTile + tile.first - place;
            const uint32_t first = place > from ? place - from : 0u, end = min(place + n - from, (uint32_t)kBkCap);
            if (first & 63u) atomicOr(&words[((first - 1u) >> 6) * 4u + (((first - 1u) >> 5) & 1u)], 1u << ((first - 1u) & 31u));
            for (uint32_t k = (first + 63u) / 64u; k * 64u < end; ++k) word[k].segment = index;
        }
        __syncthreads();
    }
    // Where the keys at places from + p, from + p + 64, ... stand in the row (lane i of a wave: a place p = 64 k + i), and any
    // place up to `most` for a key that is not there. The words of all, then their segments, so that LDS is waited for twice.
    template <int N>
    __device__ __forceinline__ void where(uint32_t p, uint32_t most, uint32_t (&at)[N], uint32_t from = 0) const {
        const Word *words = word + (p >> 6);
        Word w[N];
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = words[i];
#pragma unroll
        for (int i = 0; i < N; ++i)
            at[i] = shift[__builtin_amdgcn_mbcnt_hi((uint32_t)(w[i].starts >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)w[i].starts, w[i].segment))];
#pragma unroll
        for (int i = 0; i < N; ++i) at[i] = min(at[i] + (from + p + (uint32_t)i * kWave), most);
    }
};
static_assert(kBkMaxRow / kBkTile < kBkThreads && 4 * (kBkWords + kBkGroup - 1) <= kBkThreads, "a thread per tile and per word");

struct BkShared {
    // the pairs, 16 neighbours in the order of thread t in row t; the crowded path's keys and items; the results by item
    __align__(16) BkPair pair[kBkCap + kBkChunk];
    __align__(16) uint32_t bin[kBkBins];
    uint32_t scan[2 * kSortWaves];
    uint32_t least[kBkWaves], most[kBkWaves], crowd[kBkWaves];
    __device__ uint32_t *key() { return reinterpret_cast<uint32_t *>(pair); }
    __device__ uint16_t *src() { return reinterpret_cast<uint16_t *>(pair) + 2 * kBkCap; }
    // place p of the order: the 16 pairs of a row are turned by half the row's number, so that the rows of 32 lanes
    // reading one column each fall into different banks
    __device__ __forceinline__ BkPair &at(uint32_t p) { return pair[p ^ ((p >> 5) & 15u)]; }
};

// Least and largest of the block's valid keys (least > largest: none).
__device__ __forceinline__ void bk_range(BkShared &s, const uint32_t (&key)[kBkItems], uint32_t valid, uint32_t &least,
                                         uint32_t &most) {
    uint32_t lo = 0xFFFFFFFFu, hi = 0;
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) {
        if (!((valid >> r) & 1u)) continue;
        const uint32_t k = key[r] & 0x7FFFFFFFu;
        lo = min(lo, k);
        hi = max(hi, k);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, off, 64));
    }
    __syncthreads();                            // an earlier use of the words is over
    if ((threadIdx.x & 63) == 0) {
        s.least[threadIdx.x >> 6] = lo;
        s.most[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    least = s.least[0];
    most = s.most[0];
#pragma unroll
    for (int w = 1; w < kBkWaves; ++w) {
        least = min(least, s.least[w]);
        most = max(most, s.most[w]);
    }
}

// Where item r of this thread stands in the block's order of `rounds` x 512 items: a wave's items are neighbours.
__device__ __forceinline__ int bk_item(int rounds, int r) {
    return ((int)(threadIdx.x >> 6) * rounds + r) * kWave + (int)(threadIdx.x & 63);
}

// The bins of the values from..to: one width for all, or another below `knee`, which then gets the first `share` of them.
// Monotone in the key, and below kBkBins.
struct BkBinning {
    uint32_t from, knee;
    float below, above, start;
    bool bent;                                  // wave-uniform
    __device__ BkBinning(uint32_t from_, uint32_t knee_, uint32_t to, float share) : from(from_), knee(knee_) {
        bent = __builtin_amdgcn_readfirstlane(knee > from && knee <= to);
        start = bent ? share * kBkBins : 0.f;
        below = bent ? (start - 1.f) / (float)(knee - from) : 0.f;
        above = ((float)(kBkBins - 1) - start) / (float)(to - (bent ? knee : from) + 1u);
    }
    __device__ __forceinline__ uint32_t of(uint32_t key) const {
        const uint32_t k = key & 0x7FFFFFFFu;               // not below `from`, or not looked at
        const float last = (float)(kBkBins - 1);
        if (!bent) return (uint32_t)fminf((float)(k - from) * above, last);
        return (uint32_t)fminf(k < knee ? (float)(k - from) * below : __builtin_fmaf((float)(k - knee), above, start), last);
    }
};

// Sorts the block's valid keys (n of them in all, in `rounds` x 512 items): v[e] becomes the pair at place 16 t + e of the
// order for thread t, bk_last() past the end. False (block-uniform) where values crowd: then bk_ranks_crowded has to do it.
//
// Counting the keys into 4096 bins of their range puts them in order but for the one or two per bin; those are sorted by
// the threads, 16 places each, then across the chunks' borders (8 places of either side) and within the chunks in turn:
// odd-even transposition of halves of 8, of which a bin of L keys touches at most 2 + (L - 2) / 8.
struct BkMask {                                 // which of a thread's items are keys: any
    uint32_t bits;
    __device__ __forceinline__ bool operator()(int r) const { return (bits >> r) & 1u; }
};
struct BkFirst {                                // or the first ones
    int count;
    __device__ __forceinline__ bool operator()(int r) const { return r < count; }
};
template <class Valid>
__device__ __forceinline__ bool bk_sort(BkShared &s, const uint32_t (&key)[kBkItems], Valid valid, int rounds,
                                        const BkBinning bins, uint32_t &n, BkPair (&v)[kBkChunk]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    {
        uint4 *b4 = reinterpret_cast<uint4 *>(s.bin);
#pragma unroll
        for (int i = 0; i < kBkBins / 4 / kBkThreads; ++i) b4[i * kBkThreads + threadIdx.x] = make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
    uint32_t slot[kBkItems];                    // bin << 16 | arrival
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                // block-uniform
        uint32_t arrival[kBkGroup];
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) {
            const int r = r0 + i;
            slot[r] = bins.of(key[r]);
            arrival[i] = 0;
            if (valid(r)) arrival[i] = atomicAdd(&s.bin[slot[r]], 1u);
        }
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) slot[r0 + i] = slot[r0 + i] << 16 | arrival[i];
    }
    __syncthreads();
    constexpr int kPer = kBkBins / kBkThreads;
    uint32_t mine[kPer], sum = 0, crowd = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        mine[i] = s.bin[threadIdx.x * kPer + i];
        sum += mine[i];
        crowd = max(crowd, mine[i]);
    }
    const float wave_crowd = group_reduce<64>((float)crowd, OpMax());
    if (lane == 0) s.crowd[wave] = (uint32_t)wave_crowd;
    uint32_t run = block_excl_scan(sum, s.scan, n);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        s.bin[threadIdx.x * kPer + i] = run;
        run += mine[i];
    }
#pragma unroll
    for (int w = 0; w < kBkWaves; ++w) crowd = max(crowd, s.crowd[w]); // written before the scan's barriers
    crowd = (uint32_t)__builtin_amdgcn_readfirstlane((int)crowd);
    __syncthreads();
    if (crowd > kBkCrowd) return false;
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                // block-uniform
        uint32_t to[kBkGroup];
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) to[i] = s.bin[slot[r0 + i] >> 16] + (slot[r0 + i] & 0xFFFFu);
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) {
            const int r = r0 + i;
            if (valid(r)) s.at(to[i]) = bk_pair(key[r], (uint32_t)bk_item(rounds, r));
        }
    }
    if (threadIdx.x < kBkChunk) s.at(n + threadIdx.x) = bk_last();
    __syncthreads();
    const uint32_t p0 = threadIdx.x * kBkChunk;
    const bool busy = p0 < n;
    if (busy) {
#pragma unroll
        for (int e = 0; e < kBkChunk; ++e) v[e] = s.at(p0 + e);
        bk_merge<1>(v);
    }
    const bool next = p0 + kBkChunk < n;        // the thread above holds places too
    int left = crowd < 2u ? 0 : 1 + (int)(crowd - 2u) / 8;             // steps after the first
#pragma unroll 1
    while (left > 0) {                          // block-uniform
        uint32_t p0 = threadIdx.x * kBkChunk;
        asm volatile("" : "+v"(p0));            // the places' addresses stay in the loop, not in 24 registers
        if (busy) {
#pragma unroll
            for (int e = 0; e < kBkChunk / 2; ++e) s.at(p0 + e) = v[e];
        }
        __syncthreads();
        if (next) {
            BkPair w[kBkChunk];
#pragma unroll
            for (int e = 0; e < kBkChunk / 2; ++e) {
                w[e] = v[kBkChunk / 2 + e];
                w[kBkChunk / 2 + e] = s.at(p0 + kBkChunk + e);
            }
            bk_merge<kBkChunk / 2>(w);
#pragma unroll
            for (int e = 0; e < kBkChunk / 2; ++e) {
                v[kBkChunk / 2 + e] = w[e];
                s.at(p0 + kBkChunk + e) = w[kBkChunk / 2 + e];
            }
        }
        __syncthreads();
        if (busy && p0) {
#pragma unroll
            for (int e = 0; e < kBkChunk / 2; ++e) v[e] = s.at(p0 + e);
        }
        if (busy && left > 1) bk_merge<kBkChunk / 2>(v);
        left -= 2;
    }
    __syncthreads();                            // s.pair is free again
    return true;
}

// Lanes of the wave with the same digit.
template <int kBits>
__device__ __forceinline__ uint64_t bk_peers(uint32_t digit, bool valid) {
    uint32_t diff_lo = 0, diff_hi = 0;
#pragma unroll
    for (int b = 0; b < kBits; ++b) {
        uint32_t splat = (uint32_t)((int32_t)(digit << (31 - b)) >> 31);
        asm("" : "+v"(splat));
        const uint64_t vote = __builtin_amdgcn_ballot_w64(splat != 0u);
        diff_lo |= (uint32_t)vote ^ splat;
        diff_hi |= (uint32_t)(vote >> 32) ^ splat;
    }
    const uint64_t diff = ((uint64_t)diff_hi << 32) | diff_lo;
    return __builtin_amdgcn_ballot_w64(valid) & ~diff;
}

constexpr int kBkDigitBits = 7;                   // of a pass of the crowded path
constexpr int kBkDigitWords = (kBkWaves << kBkDigitBits) / 2;     // its counters, at the start of the bins' memory

// rank[r] = valid keys of the block that sort before key[r] (equal keys in item order) | positives among them << 16, for
// values that crowd (ties, clusters): a stable radix sort in LDS, 7 bits a pass over the bits of the range least..most.
// Few blocks run it, so that it is latency that counts: 7 bits in place of 6 are a pass less, votes over a fixed number of bits let
// rounds overlap, and a crowded run's keys are fetched three rounds at a time. Steps, logits of the right class 20 above the others:
// (1,18,384,384) 177 -> 167 us, (1,14,512,512) 197 -> 187; 14 above: (8,8,512,512) 381 -> 360, (4,19,512,1024) 698 -> 669.
__device__ __forceinline__ void bk_ranks_crowded(BkShared &s, const uint32_t (&key)[kBkItems], uint32_t valid, int rounds, uint32_t least,
                                 uint32_t most, uint32_t (&rank)[kBkItems]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t span = most - least + 1u;    // valid keys exist; keys are below 2^30
    uint32_t slot[kBkItems];
    // items without a key take the value after the largest
    uint32_t k2[kBkItems], it[kBkItems];
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) {
        const bool v = r < rounds && ((valid >> r) & 1u);
        k2[r] = v ? (key[r] & 0x80000000u) | ((key[r] & 0x7FFFFFFFu) - least) : span;
        it[r] = (uint32_t)bk_item(rounds, r);
    }
    constexpr int kDigits = 1 << kBkDigitBits;
    constexpr int kThreadsPerDigit = kBkThreads / kDigits, kWavesPerThread = kBkWaves / kThreadsPerDigit;
    uint16_t *counts = reinterpret_cast<uint16_t *>(s.bin);        // [kBkWaves][kDigits], then their exclusive sums
    const int bits = 32 - __builtin_clz(span);
    auto digit_of = [&](uint32_t k, int shift) { return ((k & 0x7FFFFFFFu) >> shift) & (uint32_t)(kDigits - 1); };
    for (int shift = 0; shift < bits; shift += kBkDigitBits) {
        __syncthreads();
        for (int i = threadIdx.x; i < kBkDigitWords; i += kBkThreads) s.bin[i] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            slot[r] = 0;
            if (r < rounds) {
                const uint32_t digit = digit_of(k2[r], shift);
                uint32_t unused;
                wave_rank_of<false>(bk_peers<kBkDigitBits>(digit, true), digit, true, false, counts + wave * kDigits, nullptr, slot[r], unused);
                if (r % kBkGroup == kBkGroup - 1) __builtin_amdgcn_sched_barrier(0);        // more rounds at once spill
            }
        }
        __syncthreads();
        const int d = (int)threadIdx.x / kThreadsPerDigit, w = (int)threadIdx.x % kThreadsPerDigit * kWavesPerThread;   // order: digit, then wave
        uint32_t n[kWavesPerThread], mine = 0, all;
#pragma unroll
        for (int i = 0; i < kWavesPerThread; ++i) mine += n[i] = counts[(w + i) * kDigits + d];
        uint32_t start = block_excl_scan(mine, s.scan, all);
#pragma unroll
        for (int i = 0; i < kWavesPerThread; ++i) {
            counts[(w + i) * kDigits + d] = (uint16_t)start;
            start += n[i];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            if (r < rounds) {
                const uint32_t at = counts[wave * kDigits + digit_of(k2[r], shift)] + slot[r];
                s.key()[at] = k2[r];
                s.src()[at] = (uint16_t)it[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            if (r < rounds) {
                k2[r] = s.key()[bk_item(rounds, r)];
                it[r] = s.src()[bk_item(rounds, r)];
            }
        }
    }
    // positives before each place, then back to the items
    uint32_t hot_here[kBkItems], wave_hot = 0;
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) {
        hot_here[r] = 0;
        if (r < rounds) {
            const uint64_t vote = __builtin_amdgcn_ballot_w64(k2[r] >> 31);
            hot_here[r] = wave_hot + peers_below(vote);
            wave_hot += (uint32_t)__builtin_popcountll(vote);
        }
    }
    __syncthreads();
    uint32_t all;
    const uint32_t before = block_excl_scan(lane == 0 ? wave_hot : 0u, s.scan, all);
    const uint32_t wave_before = (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
#pragma unroll
    for (int r = 0; r < kBkItems; ++r)
        if (r < rounds) s.key()[it[r]] = (uint32_t)bk_item(rounds, r) | (wave_before + hot_here[r]) << 16;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) rank[r] = r < rounds ? s.key()[bk_item(rounds, r)] : 0u;
    __syncthreads();
}

// A class's limit, and kBkCap sampled keys, one from each of as many equal parts of the row. The sample lies anywhere in memory:
// by 15 blocks beside the one for the limit 3 us, by the one that sorts it 10.
__global__ __launch_bounds__(kBkThreads) void bk_sample(const BucketArgs a) {
    __shared__ uint32_t wave_max[kBkWaves];
    const int c = blockIdx.y;
    if (blockIdx.x == 0) {                                  // block-uniform
        const uint32_t top = class_top<kBkThreads>(a.block_table, a.key_blocks, c, wave_max);
        if (threadIdx.x == 0) publish_class(a.pos_max, a.C, c, top);
        return;
    }
    const uint32_t part = (uint32_t)a.P / kBkCap;           // >= 1: shorter rows are not cut
    const uint32_t i = (blockIdx.x - 1u) * kBkThreads + threadIdx.x;
    uint32_t h = i * 0x9E3779B1u;                           // somewhere in the part, so that no stride meets the image's
    h = (h ^ (h >> 15)) * 0x85EBCA6Bu;
    a.dj[(int64_t)c * kBkCap + i] = a.keys[(int64_t)c * a.P + (uint32_t)((uint64_t)i * (uint32_t)a.P / kBkCap) + __umulhi(h, part)];
}

// Bounds of a class's buckets from the sample: every (sample / buckets)-th key in its order. A value that would bound two
// buckets gets one to itself: (v, v + 1). A class without positives, whose keys that take part are equal, has one bucket; the
// blocks behind the first C look for their value.
__global__ __launch_bounds__(kBkThreads) void bk_split(const BucketArgs a) {
    __shared__ BkShared s;
    const int c = (int)blockIdx.x % a.C, turn = (int)blockIdx.x / a.C;
    const bool absent = a.pos_max[c] == 0u;
    if (turn > 0) {                                         // block-uniform
        if (absent) absent_min<kBkThreads>(a.keys, a.pos_max + 2 * a.C, a.P, c, turn - 1, s.least);
        return;
    }
    const uint32_t limit = a.pos_max[c] - 1u;               // not for an absent class
    uint32_t key[kBkItems], valid = 0, mine = 0;
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) key[r] = a.dj[(int64_t)c * kBkCap + bk_item(kBkItems, r)];
#pragma unroll
    for (int r = 0; r < kBkItems; ++r)
        if (!absent && keep_key(key[r], limit)) {
            valid |= 1u << r;
            ++mine;
        }
    uint32_t n;
    block_excl_scan(mine, s.scan, n);
    uint32_t want = 1, least, most;
    bk_range(s, key, valid, least, most);
    uint32_t *sorted = s.key();
    if (n > 0) {                                            // block-uniform
        BkPair v[kBkChunk];
        uint32_t m;
        // errors near 1 crowd in classes that the network misses: a quarter of the bins for the first 64th of the range
        if (bk_sort(s, key, BkMask{valid}, kBkItems, BkBinning(least, least + (most - least) / 64u, most, 0.25f), m, v)) {
#pragma unroll
            for (int e = 0; e < kBkChunk; ++e)
                if (threadIdx.x * kBkChunk + e < n) sorted[threadIdx.x * kBkChunk + e] = bk_key_of(v[e]);
        } else {
            uint32_t rank[kBkItems];
            bk_ranks_crowded(s, key, valid, kBkItems, least, most, rank);
#pragma unroll
            for (int r = 0; r < kBkItems; ++r)
                if ((valid >> r) & 1u) sorted[rank[r] & 0xFFFFu] = key[r] & 0x7FFFFFFFu;
        }
        const uint64_t keys = (uint64_t)n * (uint32_t)a.P / kBkCap;
        want = (uint32_t)((keys + kBkTarget - 1) / kBkTarget);
        want = min(max(want, 1u), (uint32_t)a.stride - 1u);
    }
    __syncthreads();
    // candidates 1..want-1, a run of neighbours per thread; the bounds are collected where the bins were
    const int per = kBkMax / kBkThreads;
    auto candidate = [&](uint32_t j) { return sorted[j * n / want]; };         // below 2^24
    uint32_t out = 0;
    for (int u = 0; u < per; ++u) {
        const uint32_t j = 1u + threadIdx.x * per + u;
        if (j >= want) break;
        const uint32_t v = candidate(j);
        if (j > 1 && candidate(j - 1) == v) continue;
        out += (j + 1 < want && candidate(j + 1) == v) ? 2u : 1u;
    }
    uint32_t bounds;
    uint32_t at = block_excl_scan(out, s.scan, bounds);
    for (int u = 0; u < per; ++u) {
        const uint32_t j = 1u + threadIdx.x * per + u;
        if (j >= want) break;
        const uint32_t v = candidate(j);
        if (j > 1 && candidate(j - 1) == v) continue;
        s.bin[at++] = v;
        if (j + 1 < want && candidate(j + 1) == v) s.bin[at++] = v + 1u;
    }
    __syncthreads();
    // The largest key that takes part, the lowest-ranked positive's, has a bucket too: where the network is sure, that is an
    // error of exactly 0, shared by many and far from the next.
    if (n > 0 && limit > (bounds ? s.bin[bounds - 1] : 0u)) {
        __syncthreads();
        if (threadIdx.x == 0) s.bin[bounds] = limit;
        ++bounds;
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < bounds; i += kBkThreads) a.bounds[(int64_t)c * a.stride + i] = s.bin[i];
    for (uint32_t i = threadIdx.x; i < n; i += kBkThreads)  // the last one below the limit
        if (sorted[i] < limit && (i + 1u == n || sorted[i + 1u] >= limit)) a.numbers[4 * a.C + c] = sorted[i];
    if (threadIdx.x == 0) {
        a.numbers[c] = bounds + 1u;
        a.numbers[3 * a.C + c] = n ? least : 0u;
        if (n == 0u || sorted[0] >= limit) a.numbers[4 * a.C + c] = 0u;
    }
    __syncthreads();                                        // the sample is done with: the cells of the top bits take its place
    // the bucket of the least key with each pattern of the top bits, and the most bounds that one pattern's keys can lie between
    const int bits = (int)a.pos_max[3 * a.C + c], shift = bits > kBkFineBits ? bits - kBkFineBits : 0;
    constexpr int kPerFine = kBkFine / kBkThreads;
    uint32_t *above = s.key();                              // [kBkFine + 1] bounds above the least key of the pattern before
    for (int f = threadIdx.x; f <= kBkFine; f += kBkThreads) above[f] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < bounds; i += kBkThreads)
        atomicAdd(&above[min((s.bin[i] + (1u << shift) - 1u) >> shift, (uint32_t)kBkFine)], 1u);
    __syncthreads();
    uint32_t here[kPerFine], sum = 0, width = 0, all;
#pragma unroll
    for (int u = 0; u < kPerFine; ++u) {
        here[u] = above[threadIdx.x * kPerFine + u];
        sum += here[u];
        width = max(width, above[threadIdx.x * kPerFine + u + 1]);
    }
    uint32_t bucket = block_excl_scan(sum, s.scan, all);
#pragma unroll
    for (int u = 0; u < kPerFine; ++u) {
        bucket += here[u];
        a.fine[(int64_t)c * kBkFine + threadIdx.x * kPerFine + u] = (uint16_t)bucket;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) width = max(width, (uint32_t)__shfl_xor((int)width, off, 64));
    if ((threadIdx.x & 63) == 0) s.crowd[threadIdx.x >> 6] = width;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 0; w < kBkWaves; ++w) width = max(width, s.crowd[w]);
        a.numbers[5 * a.C + c] = width ? 0x80000000u >> __builtin_clz(width) : 0u;
    }
}

// The bounds and the table in LDS.
template <int kStride>
struct BkLookup {
    uint32_t bounds[2 * kStride];
    uint16_t fine[kBkFine];
    // first_step: 2^k of which 2^(k+1) - 1 is no less than the bounds in any cell of `fine`
    __device__ void fetch(const BucketArgs &a, int c, uint32_t buckets, uint32_t first_step) {
        for (uint32_t i = threadIdx.x; i + 1 < buckets; i += kBkThreads) bounds[i] = a.bounds[(int64_t)c * kStride + i];
        for (uint32_t i = threadIdx.x; i < 2 * first_step; i += kBkThreads)
            if (buckets - 1 + i < 2 * kStride) bounds[buckets - 1 + i] = 0xFFFFFFFFu;
        const uint32_t *from = reinterpret_cast<const uint32_t *>(a.fine + (int64_t)c * kBkFine);
        uint32_t *to = reinterpret_cast<uint32_t *>(fine);
#pragma unroll
        for (int i = 0; i < kBkFine / 2 / kBkThreads; ++i) to[i * kBkThreads + threadIdx.x] = from[i * kBkThreads + threadIdx.x];
    }
    // buckets of N keys (kStride for one that takes no part): a step of all their searches at a time. Bounds behind a cell's
    // are above its keys, so the search needs no end.
    template <int N>
    __device__ __forceinline__ void find(const uint32_t *key, uint32_t limit, int shift, uint32_t first_step, uint32_t *bucket) const {
        uint32_t at[N];
#pragma unroll
        for (int i = 0; i < N; ++i) at[i] = fine[min(key[i] & 0x7FFFFFFFu, limit) >> shift];
        for (uint32_t step = first_step; step; step >>= 1) {        // block-uniform
#pragma unroll
            for (int i = 0; i < N; ++i) at[i] += bounds[at[i] + step - 1u] <= (key[i] & 0x7FFFFFFFu) ? step : 0u;
        }
#pragma unroll
        for (int i = 0; i < N; ++i) bucket[i] = keep_key(key[i], limit) ? at[i] : (uint32_t)kStride;
    }
};

// The tile's keys in the order of their buckets (in pixel order inside one), in the place of its keys, and every pixel's place
// in that order.
// Bound by vector and LDS instructions, 68 and 13 per 64 keys (two thirds of the time at 24 waves per CU). Match masks of 10
// votes for every key were 126 (149 -> 102 us at (4,19,512,1024) fp32, 177 -> 137 at (8,21,513,513) bf16 trained); a wave's 64 keys
// lie in up to 1024 buckets, so that some 5 of them meet another. A look-up table of 13 bits instead of 11 leaves two steps
// less to the search (100 -> 96, 133 -> 127).
template <int kBits>
__global__ __launch_bounds__(kBkThreads, 6) void bk_cut(const BucketArgs a) {
    constexpr int kStride = 1 << kBits, kPer = (kStride + kBkThreads - 1) / kBkThreads, kChunks = kBkTile / kWave;
    // 49 KiB, three blocks per CU: the look-up's tables are done with when the tile is put in order
    union Tile {
        BkLookup<kStride> look;
        uint32_t key[kBkTile];
    };
    __shared__ Tile s;
    __shared__ __align__(16) uint16_t counts[kBkWaves][kStride + 2];        // a wave's keys so far; the last of those that take no part
    __shared__ uint64_t hot_mask[kChunks + 1];
    __shared__ uint32_t hot_before[kChunks + 1];
    __shared__ uint32_t scan_tmp[kSortWaves];
    const int c = blockIdx.y, tile = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int begin = tile * kBkTile, n = min(kBkTile, a.P - begin);
    uint32_t *row = a.keys + (int64_t)c * a.P + begin;
    uint32_t key[kBkTileItems], b[kBkTileItems], rank[kBkTileItems];
    if (n == kBkTile) {
#pragma unroll
        for (int r = 0; r < kBkTileItems; ++r) key[r] = row[bk_item(kBkTileItems, r)];
    } else {
#pragma unroll
        for (int r = 0; r < kBkTileItems; ++r) {
            const int li = bk_item(kBkTileItems, r);
            key[r] = li < n ? row[li] : kIgnoredKey;
        }
    }
    const uint32_t buckets = a.numbers[c], first_step = a.numbers[5 * a.C + c], limit = bk_limit(a, c);
    const int bits = (int)a.pos_max[3 * a.C + c], shift = bits > kBkFineBits ? bits - kBkFineBits : 0;
    s.look.fetch(a, c, buckets, first_step);
    for (int i = threadIdx.x; i < kBkWaves * (kStride + 2) / 2; i += kBkThreads) reinterpret_cast<uint32_t *>(counts)[i] = 0;
    __syncthreads();
    constexpr int kFind = 8;
#pragma unroll
    for (int r = 0; r < kBkTileItems; r += kFind) s.look.template find<kFind>(key + r, limit, shift, first_step, b + r);
    // A key's rank among the wave's keys of its bucket: the counter tells what came in earlier rounds, and whether every key of
    // this one moved it on from there. LDS takes a wave's operations in their order, so the rounds of a group wait for nothing.
    // The few that meet others of their round (whichever of them LDS took first) find their place by a vote per bucket met
    // twice; many, by a vote per bit.
    constexpr int kGroup = 2;
    constexpr uint32_t kFew = 16;
    uint16_t *mine_of = counts[wave];
#pragma unroll
    for (int r0 = 0; r0 < kBkTileItems; r0 += kGroup) {
        uint32_t moved[kGroup];
#pragma unroll
        for (int h = 0; h < kGroup; ++h) {
            const uint32_t d = b[r0 + h];
            rank[r0 + h] = mine_of[d];
            asm volatile("" ::: "memory");
            moved[h] = 0;
            if (d != (uint32_t)kStride)         // additions to one address take their turns
                moved[h] = atomicAdd(reinterpret_cast<uint32_t *>(mine_of) + (d >> 1), 1u << (16u * (d & 1u)));
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int h = 0; h < kGroup; ++h) {
            const uint32_t d = b[r0 + h], seen = rank[r0 + h];
            uint64_t met = __builtin_amdgcn_ballot_w64(d != (uint32_t)kStride && ((moved[h] >> (16u * (d & 1u))) & 0xFFFFu) != seen);
            bool first = true;
            while (met && (first || __builtin_popcountll(met) <= kFew)) {   // wave-uniform
                const uint32_t one = (uint32_t)__builtin_amdgcn_readlane((int)d, __builtin_ctzll(met));
                const uint64_t peers = __builtin_amdgcn_ballot_w64(d == one);
                if (d == one) rank[r0 + h] = seen + peers_below(peers);
                met &= ~peers;
                first = false;
            }
            if (met) {
                const uint64_t peers = bk_peers<kBits>(d, d != (uint32_t)kStride);
                rank[r0 + h] = seen + peers_below(peers);
            }
        }
    }
    __syncthreads();
    uint32_t mine[kPer], n_mine = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t d = threadIdx.x * kPer + i;
        mine[i] = 0;
        if (d < buckets) {
#pragma unroll
            for (int w = 0; w < kBkWaves; ++w) {
                const uint32_t t = counts[w][d];
                counts[w][d] = (uint16_t)mine[i];
                mine[i] += t;
            }
        }
        n_mine += mine[i];
    }
    uint32_t n_here;
    const uint32_t first = block_excl_scan(n_mine, scan_tmp, n_here);
    uint32_t at = first;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t d = threadIdx.x * kPer + i;
        if (d < buckets) {
#pragma unroll
            for (int w = 0; w < kBkWaves; ++w) counts[w][d] = (uint16_t)(counts[w][d] + at);
        }
        at += mine[i];
    }
    __syncthreads();
    uint16_t *place = a.place + (int64_t)c * a.P + begin;
#pragma unroll
    for (int r = 0; r < kBkTileItems; ++r) {
        asm volatile("" : "+v"(b[r]));                      // the counter's address again, not held in a register each
        const bool valid = b[r] != (uint32_t)kStride;       // not past the end: those keys take no part
        rank[r] = valid ? mine_of[b[r]] + rank[r] : (uint32_t)kBkNowhere;
        if (valid) s.key[rank[r]] = key[r];
    }
    if (n == kBkTile) {
#pragma unroll
        for (int r = 0; r < kBkTileItems; ++r) place[bk_item(kBkTileItems, r)] = (uint16_t)rank[r];
    } else {
#pragma unroll
        for (int r = 0; r < kBkTileItems; ++r) {
            const int li = bk_item(kBkTileItems, r);
            if (li < n) place[li] = (uint16_t)rank[r];
        }
    }
    __syncthreads();
    // out in order; the positives before a place from masks of 64 places each
#pragma unroll
    for (int r = 0; r < kBkTileItems; ++r) {
        const uint32_t i = (uint32_t)r * kBkThreads + threadIdx.x;
        const uint32_t k = i < n_here ? s.key[i] : 0u;
        const uint64_t hot = __builtin_amdgcn_ballot_w64(k >> 31);
        if (i < n_here) row[i] = k;
        if (lane == 0) hot_mask[i >> 6] = hot;
    }
    __syncthreads();
    if (wave == 0) {
        static_assert(kChunks == 2 * kWave, "two masks a lane");
        const uint32_t h0 = (uint32_t)__builtin_popcountll(hot_mask[2 * lane]), h1 = (uint32_t)__builtin_popcountll(hot_mask[2 * lane + 1]);
        const uint32_t incl = wave_incl_scan(h0 + h1);
        hot_before[2 * lane] = incl - h0 - h1;
        hot_before[2 * lane + 1] = incl - h1;
        if (lane == kWave - 1) {
            hot_before[kChunks] = incl;
            hot_mask[kChunks] = 0;
        }
    }
    __syncthreads();
    uint32_t *out = a.tile_start + ((int64_t)c * a.tiles + tile) * (kStride + 1);
    at = first;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t d = threadIdx.x * kPer + i;
        const uint32_t hot = hot_before[at >> 6] + (uint32_t)__builtin_popcountll(hot_mask[at >> 6] & ((1ull << (at & 63u)) - 1ull));
        if (d < buckets) out[d] = at | hot << 16;
        at += mine[i];
    }
    if (threadIdx.x == 0) out[buckets] = n_here | hot_before[kChunks] << 16;
}

// Keys and positives before each bucket in the row: the sums of the tiles', which are left by bucket for the rank kernels.
// 64 buckets x 64 tiles at a time, the next ones' loads under way. (With the work of bk_group done by the last block of a class,
// which has to see what the others wrote, 37 us instead of 7 + 5: every block's fence writes its L2 back.)
__global__ __launch_bounds__(1024) void bk_sum(const BucketArgs a) {
    __shared__ uint32_t part[64][65];
    __shared__ uint32_t sums[16][64], hots[16][64];
    const int c = blockIdx.y, first = blockIdx.x * 64, lane = threadIdx.x & 63, group = threadIdx.x >> 6;
    const int entries = (int)a.numbers[c] + 1;
    if (first >= entries) return;                           // block-uniform
    const int pitch = a.stride + 1;
    const uint32_t *in = a.tile_start + (int64_t)c * a.tiles * pitch;
    uint32_t *out = a.start + (int64_t)c * pitch * a.tiles;
    uint32_t n = 0, h = 0, v[2][4];
    auto fetch = [&](uint32_t (&to)[4], int t0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + i * 16 + group;
            to[i] = t < a.tiles && first + lane < entries ? in[(int64_t)t * pitch + first + lane] : 0u;
        }
    };
    fetch(v[0], 0);
    fetch(v[1], 64);
    for (int t0 = 0; t0 < a.tiles; t0 += 64) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            n += v[0][i] & 0xFFFFu;
            h += v[0][i] >> 16;
            part[i * 16 + group][lane] = v[0][i];
            v[0][i] = v[1][i];
        }
        fetch(v[1], t0 + 128);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int b = first + i * 16 + group;
            if (b < entries && t0 + lane < a.tiles) out[(int64_t)b * a.tiles + t0 + lane] = part[lane][i * 16 + group];
        }
        __syncthreads();
    }
    sums[group][lane] = n;
    hots[group][lane] = h;
    __syncthreads();
    if (group != 0 || first + lane >= entries) return;
    uint32_t total = 0, hot = 0;
#pragma unroll
    for (int g = 0; g < 16; ++g) {
        total += sums[g][lane];
        hot += hots[g][lane];
    }
    a.base[(int64_t)c * pitch + first + lane] = total;
    a.hot_base[(int64_t)c * pitch + first + lane] = hot;
}

// The runs of buckets that one block sorts: neighbours that start in the same kBkSlab keys of the row, unless they come to
// more than kBkCap, or lie so differently dense that bins of one width would not do.
__global__ __launch_bounds__(kBkThreads) void bk_group(const BucketArgs a) {
    __shared__ uint32_t base[kBkMax + 1], bound[kBkMax + 1], scan_tmp[2 * kSortWaves];
    constexpr int kPer = kBkMax / kBkThreads;
    const int c = blockIdx.x, buckets = (int)a.numbers[c], b0 = threadIdx.x * kPer;
    const bool absent = a.pos_max[c] == 0u;                 // one bucket of one value
    const int64_t row = (int64_t)c * (a.stride + 1);
    for (int b = threadIdx.x; b <= buckets; b += kBkThreads) {
        base[b] = a.base[row + b];
        bound[b] = b + 1 < buckets ? a.bounds[(int64_t)c * a.stride + b] : bk_limit(a, c) + 1u;     // of the next bucket
    }
    __syncthreads();
    const uint32_t least = a.numbers[3 * a.C + c];
    auto width = [&](int b) { return (float)(bound[b] - (b ? bound[b - 1] : min(least, bound[0]))) / (float)(base[b + 1] - base[b] + 1u); };
    bool start[kPer];
    uint32_t starts = 0, wide = 0, flat = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int b = b0 + i;
        start[i] = false;
        if (b >= buckets) continue;
        if (base[b + 1] - base[b] > (uint32_t)kBkCap) ((absent || (b && bound[b] - bound[b - 1] == 1u)) ? flat : wide) |= 1u << i;
        const uint32_t slab = base[b] / kBkSlab;
        start[i] = b == 0 || base[b - 1] / kBkSlab != slab;
        if (!start[i]) {
            int f = b - 1;                      // first bucket of the slab: few are empty or small
            while (f > 0 && base[f - 1] / kBkSlab == slab) --f;
            const float w = width(b), w1 = width(b - 1);
            // only a slab's last bucket can take it past kBkCap, or past it alone
            start[i] = base[b + 1] - base[f] > (uint32_t)kBkCap || w > 4.f * w1 || w1 > 4.f * w;
        }
        starts += start[i] ? 1u : 0u;
    }
    uint32_t runs;
    uint32_t k = block_excl_scan(starts, scan_tmp, runs);
#pragma unroll
    for (int i = 0; i < kPer; ++i)
        if (start[i]) a.runs[row + k++] = (uint32_t)(b0 + i);
    uint32_t w, f, wides, flats;
    block_excl_scan2((uint32_t)__builtin_popcount(wide), (uint32_t)__builtin_popcount(flat), scan_tmp, w, wides, f, flats);
    const float npos = (float)a.hot_base[row + buckets];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int b = b0 + i;
        if ((wide >> i) & 1u) a.large[(int64_t)c * a.stride + w++] = (uint32_t)b;
        if (!((flat >> i) & 1u)) continue;
        // one error, and the differences, exact as multiples of 2^-24, add up to that of the ends
        const float rise = jaccard(npos, base[b + 1], a.hot_base[row + b + 1]) - jaccard(npos, base[b], a.hot_base[row + b]);
        a.large[(int64_t)c * a.stride + wides + f] = (uint32_t)b;
        a.loss_part[(2 * (int64_t)c + 1) * a.stride + wides + f++] = add_loss(0.0, key_error(bound[b] - 1u), rise);
    }
    if (threadIdx.x == 0) {
        a.numbers[6 * a.C + c] = wides;
        a.numbers[7 * a.C + c] = flats;
        a.numbers[8 * a.C + c] = 0;
        a.runs[row + runs] = (uint32_t)buckets;
        a.numbers[a.C + c] = runs;
        a.numbers[2 * a.C + c] = a.hot_base[row + buckets];
    }
}

// n keys, a few times kBkCap at most, from rank `rank0` on, with hot0 positives before them: ranges of values [from, end)
// with at most kBkCap keys, one after the other, collected in order by sweeps over all n; a single value that more keys share
// is ranked by position.
__device__ __forceinline__ double bk_wide_keys(BkShared &s, const BucketArgs &a, int c, uint32_t rank0, uint32_t hot0, int n) {
    const uint32_t *kin = a.sorted + (int64_t)c * a.P + rank0;
    float *out = reinterpret_cast<float *>(a.dj) + (int64_t)c * a.P + rank0;
    const float npos = (float)a.numbers[2 * a.C + c];
    double part = 0.0;
    uint32_t key[kBkItems], rank[kBkItems], valid = 0, least, most;
    uint32_t lo = 0xFFFFFFFFu, hi = 0;
    for (int i = threadIdx.x; i < n; i += kBkThreads) {
        const uint32_t k = kin[i] & 0x7FFFFFFFu;
        lo = min(lo, k);
        hi = max(hi, k);
    }
    key[0] = lo;
    bk_range(s, key, 1u, least, most);
    uint32_t unused;
    key[0] = hi;
    bk_range(s, key, 1u, unused, most);
    uint32_t from = least, done = 0;
    int shift = 32 - (int)__builtin_clz((most - from) | 1u);
    shift = shift > 12 ? shift - 12 : 0;
    while (done < (uint32_t)n) {                        // a turn takes keys or narrows the bins (shift falls)
        __syncthreads();
        for (int i = threadIdx.x; i < kBkBins; i += kBkThreads) s.bin[i] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kBkThreads) {
            const uint32_t k = kin[i] & 0x7FFFFFFFu;
            if (k >= from && ((k - from) >> shift) < (uint32_t)kBkBins) atomicAdd(&s.bin[(k - from) >> shift], 1u);
        }
        __syncthreads();
        constexpr int kPer = kBkBins / kBkThreads;
        uint32_t sum = 0, total;
        for (int i = 0; i < kPer; ++i) sum += s.bin[threadIdx.x * kPer + i];
        uint32_t run = block_excl_scan(sum, s.scan, total);
        uint32_t bins = 0, keys = 0;                    // leading bins that fit together, and their keys
        for (int i = 0; i < kPer; ++i) {
            run += s.bin[threadIdx.x * kPer + i];
            if (run <= (uint32_t)kBkCap) {
                ++bins;
                keys = run;
            }
        }
        uint32_t take, take_keys, d0, d1;
        block_excl_scan2(bins, 0u, s.scan, d0, take, d1, unused);
        {
            uint32_t m = keys;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
            if ((threadIdx.x & 63) == 0) s.crowd[threadIdx.x >> 6] = m;
            __syncthreads();
            take_keys = 0;
            for (int w = 0; w < kBkWaves; ++w) take_keys = max(take_keys, s.crowd[w]);
            __syncthreads();
        }
        if (take_keys == 0 && take < (uint32_t)kBkBins && shift > 0) {       // the first bin with keys is too full
            from += take << shift;
            shift = shift > 12 ? shift - 12 : 0;
            continue;
        }
        const bool single = take_keys == 0;             // ... and holds a single value
        // 64 bits: the last range may end past 2^32
        const uint64_t first = (uint64_t)from + (single ? take : 0u);
        const uint64_t end = single ? first + 1u : first + ((uint64_t)take << shift);
        const int turns = (n + kBkCap - 1) / kBkCap;
        uint32_t seen = 0, seen_hot = 0;
        uint32_t place[kBkItems];
        // keys of the range in their order: into LDS, or (single) ranked as they come; then their places the same way
        for (int what = 0; what < (single ? 1 : 2); ++what) {
            seen = 0;
            for (int t = 0; t < turns; ++t) {
                uint32_t k[kBkItems], mine = 0, hot = 0;
#pragma unroll
                for (int r = 0; r < kBkItems; ++r) {    // a thread's keys are neighbours here
                    const int i = t * kBkCap + (int)threadIdx.x * kBkItems + r;
                    k[r] = i < n ? kin[i] : kIgnoredKey;
                    const uint32_t bits = k[r] & 0x7FFFFFFFu;
                    if (i < n && bits >= first && bits < end) {
                        ++mine;
                        hot += k[r] >> 31;
                    }
                }
                uint32_t at, all, at_hot, all_hot;
                block_excl_scan2(mine, hot, s.scan, at, all, at_hot, all_hot);
                at += seen;
                at_hot += seen_hot;
#pragma unroll
                for (int r = 0; r < kBkItems; ++r) {
                    const int i = t * kBkCap + (int)threadIdx.x * kBkItems + r;
                    const uint32_t bits = k[r] & 0x7FFFFFFFu;
                    if (i < n && bits >= first && bits < end) {
                        if (single) {
                            const float dj = jaccard_step(npos, rank0 + at, hot0 + at_hot, k[r] >> 31);
                            part = add_loss(part, key_error(k[r]), dj);
                            out[i] = dj;
                        } else {
                            s.key()[at] = what == 0 ? k[r] : (uint32_t)i;
                        }
                        ++at;
                        at_hot += k[r] >> 31;
                    }
                }
                seen += all;
                seen_hot += what == 0 ? all_hot : 0u;
            }
            if (single) break;
            __syncthreads();
            const int rounds = (int)(take_keys + kBkThreads - 1) / kBkThreads;
            valid = 0;
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                const int li = bk_item(rounds, r);
                if (r < rounds && li < (int)take_keys) {
                    if (what == 0) key[r] = s.key()[li];
                    else place[r] = s.key()[li];
                    valid |= 1u << r;
                }
            }
            __syncthreads();
            if (what == 1) {
                bk_range(s, key, valid, least, unused);
                uint32_t largest;
                bk_range(s, key, valid, unused, largest);
                bk_ranks_crowded(s, key, valid, rounds, least, largest, rank);
#pragma unroll
                for (int r = 0; r < kBkItems; ++r) {
                    if ((valid >> r) & 1u) {
                        const float dj = jaccard_step(npos, rank0 + (rank[r] & 0xFFFFu), hot0 + (rank[r] >> 16), key[r] >> 31);
                        part = add_loss(part, key_error(key[r]), dj);
                        out[place[r]] = dj;
                    }
                }
            }
        }
        done += seen;
        rank0 += seen;
        hot0 += seen_hot;
        if (done >= (uint32_t)n || seen == 0) break;        // every turn takes keys
        from = (uint32_t)end;                           // keys are left, so it is below 2^31
        shift = 32 - (int)__builtin_clz((most - from) | 1u);
        shift = shift > 12 ? shift - 12 : 0;
    }
    return part;
}

// What bk_huge_keys keeps in the block's memory: first, where the pairs are, the bounds of up to kBkIntervals value intervals
// and their keys; then, per group, in what the crowded path leaves free behind its counters and behind its keys
// and items.
constexpr int kBkIntervals = 4096, kBkGroups = 1100;
struct BkIntervals {
    uint32_t bound[2][kBkIntervals];
    uint32_t count[kBkIntervals];
};
struct BkGroups {
    uint32_t *least, *first;                    // [groups], [groups + 1]: least key, first rank
    uint32_t *next, *start;                     // the next place of one of its keys, its start in the tile
    __device__ explicit BkGroups(BkShared &s)
        : least(s.bin + kBkDigitWords), first(least + kBkGroups), next(reinterpret_cast<uint32_t *>(s.src() + kBkCap)),
          start(next + kBkGroups) {}
};
static_assert(kBkIntervals % kBkThreads == 0 && 3 * (kBkMaxRow / kBkCap + 2) < kBkGroups, "groups, see bk_huge_groups");
static_assert(sizeof(BkIntervals) <= sizeof(BkPair) * (kBkCap + kBkChunk) && kBkDigitWords + 2 * kBkGroups + 1 <= kBkBins &&
              6 * kBkCap + 8 * kBkGroups <= (int)sizeof(BkPair) * (kBkCap + kBkChunk), "they fit");

// The intervals of the thread's keys: the last of m ascending bounds that is not above a key. All keys a step at a time: one
// after the other, each waiting for LDS at every step, a tile took 12 us.
__device__ __forceinline__ void bk_intervals(const uint32_t *bound, uint32_t m, const uint32_t (&key)[kBkItems],
                                             uint32_t (&at)[kBkItems]) {
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) at[r] = 0;
    for (uint32_t step = m > 1u ? 0x80000000u >> __builtin_clz(m - 1u) : 0u; step; step >>= 1) {
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            const uint32_t to = at[r] + step, least = bound[min(to, m - 1u)];
            at[r] = to < m && least <= (key[r] & 0x7FFFFFFFu) ? to : at[r];
        }
    }
}

// Cuts the n keys of the values lo..hi - 1 into groups of at most kBkCap keys, or of one value: intervals that hold more are
// split, by a third at least, until none is left, and neighbours that come to no more than kBkCap are one again (those in one
// of the n / kBkCap slabs of the order; those that lie across two stand alone). Every turn reads the keys once; the
// values are 30 bits wide, so there are 19 at most, and 1 to 6 for what was tried. Returns the number of groups.
__device__ __forceinline__ uint32_t bk_huge_groups(BkShared &s, const BkGroups &out, const uint32_t *kin, uint32_t n, uint32_t lo, uint32_t hi) {
    constexpr uint32_t kPer = kBkIntervals / kBkThreads, kCap = kBkCap;
    BkIntervals &w = *reinterpret_cast<BkIntervals *>(s.pair);
    uint32_t m = 1, cur = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        w.bound[0][0] = lo;
        w.count[0] = n;
    }
    __syncthreads();
    for (;;) {
        const uint32_t *bound = w.bound[cur];
        uint32_t *next = w.bound[cur ^ 1u];
        const uint32_t j0 = threadIdx.x * kPer;
        uint32_t cnt[kPer], sum = 0, all;
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            cnt[u] = j0 + u < m ? w.count[j0 + u] : 0u;
            sum += cnt[u];
        }
        const uint32_t cnt_before = j0 > 0u && j0 <= m ? w.count[j0 - 1u] : 0u;
        const uint32_t first = block_excl_scan(sum, s.scan, all);
        auto alone = [&](uint32_t at, uint32_t c) { return c > 0u && (at + c - 1u) / kCap != at / kCap; };
        uint32_t at = first, keep = 0, split = 0;
        bool was_alone = alone(first - cnt_before, cnt_before);
        uint32_t slab = (first - cnt_before) / kCap;
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            const uint32_t j = j0 + u;
            const bool is_alone = alone(at, cnt[u]);
            if (j < m) {
                const uint32_t width = (j + 1u < m ? bound[j + 1u] : hi) - bound[j];
                if (cnt[u] > kCap && width > 1u) split |= 1u << u;
                else if (j == 0 || is_alone || was_alone || at / kCap != slab) keep |= 1u << u;
            }
            was_alone = is_alone;
            slab = at / kCap;
            at += cnt[u];
        }
        uint32_t k, kept, d, splits;
        block_excl_scan2((uint32_t)__builtin_popcount(keep), (uint32_t)__builtin_popcount(split), s.scan, k, kept, d, splits);
        if (splits == 0) {                                  // block-uniform
            at = first;
#pragma unroll
            for (uint32_t u = 0; u < kPer; ++u) {
                if ((keep >> u) & 1u) {
                    out.least[k] = bound[j0 + u];
                    out.first[k++] = at;
                }
                at += cnt[u];
            }
            if (threadIdx.x == 0) out.first[kept] = n;
            __syncthreads();
            return kept;
        }
        const uint32_t parts = (kBkIntervals - kept) / splits;          // 3 or more: see the bound on groups
        auto width_of = [&](uint32_t j) { return (j + 1u < m ? bound[j + 1u] : hi) - bound[j]; };
        auto step_of = [&](uint32_t width) { return (width + parts - 1u) / parts; };
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            if ((keep >> u) & 1u) ++mine;
            if ((split >> u) & 1u) {
                const uint32_t width = width_of(j0 + u), step = step_of(width);
                mine += (width + step - 1u) / step;
            }
        }
        uint32_t total;
        uint32_t to = block_excl_scan(mine, s.scan, total);
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            if ((keep >> u) & 1u) next[to++] = bound[j0 + u];
            if ((split >> u) & 1u) {                        // a list for all threads: the parts of one may be thousands
                const uint32_t width = width_of(j0 + u), step = step_of(width);
                out.least[d] = j0 + u;
                out.first[d++] = to;
                to += (width + step - 1u) / step;
            }
        }
        __syncthreads();
        for (uint32_t i = 0; i < splits; ++i) {
            const uint32_t j = out.least[i], width = width_of(j), step = step_of(width);
            for (uint32_t q = threadIdx.x; q * step < width; q += kBkThreads) next[out.first[i] + q] = bound[j] + q * step;
        }
        m = total;
        cur ^= 1u;
        for (uint32_t j = threadIdx.x; j < m; j += kBkThreads) w.count[j] = 0;
        __syncthreads();
        for (uint32_t i0 = 0; i0 < n; i0 += kBkCap) {
            uint32_t key[kBkItems], at_key[kBkItems];
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                const uint32_t i = i0 + (uint32_t)bk_item(kBkItems, r);
                key[r] = i < n ? kin[i] : 0u;
            }
            bk_intervals(next, m, key, at_key);
#pragma unroll
            for (int r = 0; r < kBkItems; ++r)
                if (i0 + (uint32_t)bk_item(kBkItems, r) < n) atomicAdd(&w.count[at_key[r]], 1u);
        }
        __syncthreads();
    }
}

// A bucket of n keys of the values lo..hi - 1, from rank `rank0` on, with hot0 positives before them, many times what a block
// holds: its keys are moved to their groups (bk_huge_groups), in order inside each, a group at a time is ranked in LDS,
// and the differences come back through the places left where the keys were. Every key is read and moved a bounded number
// of times: bounds that the sample misses by far ((1,32,1,500000), all keys in one bucket) cost 6.5 ms, where a sweep over
// the bucket per 7680 keys cost 56 (radix passes 0.23); twice the keys 14 and 262.
__device__ __forceinline__ double bk_huge_keys(BkShared &s, const BucketArgs &a, int c, uint32_t rank0, uint32_t hot0, uint32_t n,
                               uint32_t lo, uint32_t hi) {
    uint32_t *kin = a.sorted + (int64_t)c * a.P + rank0;   // the keys, then every key's place, then its difference
    uint32_t *moved = a.dj + (int64_t)c * a.P + rank0;
    const float npos = (float)a.numbers[2 * a.C + c];
    const BkGroups of(s);
    const uint32_t groups = bk_huge_groups(s, of, kin, n, lo, hi);
    uint32_t *next = of.next, *start = of.start;
    for (uint32_t g = threadIdx.x; g < groups; g += kBkThreads) next[g] = of.first[g];
    uint32_t key[kBkItems], rank[kBkItems];
    for (uint32_t i0 = 0; i0 < n; i0 += kBkCap) {           // to their groups
        const int here = (int)min((uint32_t)kBkCap, n - i0), rounds = (here + kBkThreads - 1) / kBkThreads;
        uint32_t group[kBkItems], valid = 0;
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            const int li = bk_item(rounds, r);
            key[r] = 0;
            if (r < rounds && li < here) {
                key[r] = kin[i0 + li];
                valid |= 1u << r;
            }
        }
        bk_intervals(of.least, groups, key, group);
        bk_ranks_crowded(s, group, valid, rounds, 0u, groups - 1u, rank);
        uint32_t *order = s.key();                          // groups in the tile's order
#pragma unroll
        for (int r = 0; r < kBkItems; ++r)
            if ((valid >> r) & 1u) order[rank[r] & 0xFFFFu] = group[r];
        __syncthreads();
        for (int p = threadIdx.x; p < here; p += kBkThreads)
            if (p == 0 || order[p - 1] != order[p]) start[order[p]] = (uint32_t)p;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            if (!((valid >> r) & 1u)) continue;
            const uint32_t place = next[group[r]] + (rank[r] & 0xFFFFu) - start[group[r]];
            moved[place] = key[r];
            kin[i0 + bk_item(rounds, r)] = place;
        }
        __syncthreads();
        for (int p = threadIdx.x; p < here; p += kBkThreads)
            if (p == here - 1 || order[p + 1] != order[p]) next[order[p]] += (uint32_t)p + 1u - start[order[p]];
        __syncthreads();
    }
    double part = 0.0;
    for (uint32_t g = 0; g < groups; ++g) {
        const uint32_t from = of.first[g], end = of.first[g + 1u];
        // more than fit: one value, in order as it stands, a block's fill at a time
        const bool single = end - from > (uint32_t)kBkCap;
        for (uint32_t i0 = from; i0 < end; i0 += kBkCap) {
            const int here = (int)min((uint32_t)kBkCap, end - i0), rounds = (here + kBkThreads - 1) / kBkThreads;
            uint32_t valid = 0, hot = 0, least, most;
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                const int li = bk_item(rounds, r);
                key[r] = 0;
                if (r < rounds && li < here) {
                    key[r] = moved[i0 + li];
                    valid |= 1u << r;
                    hot += key[r] >> 31;
                }
            }
            uint32_t hots;
            block_excl_scan(hot, s.scan, hots);
            bk_range(s, key, valid, least, most);
            if (single) most = least;
            bk_ranks_crowded(s, key, valid, rounds, least, most, rank);
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                if (!((valid >> r) & 1u)) continue;
                const float dj = jaccard_step(npos, rank0 + i0 + (rank[r] & 0xFFFFu), hot0 + (rank[r] >> 16), key[r] >> 31);
                part = add_loss(part, key_error(key[r]), dj);
                moved[i0 + bk_item(rounds, r)] = __builtin_bit_cast(uint32_t, dj);
            }
            hot0 += hots;
        }
    }
    __syncthreads();
    for (int copy = 0; copy < 2; ++copy) {                  // the reads of a tile before its writes, not one after the other
        const uint32_t *at = copy ? kin : moved;
        uint32_t *to = copy ? moved : kin;
        for (uint32_t i0 = 0; i0 < n; i0 += kBkCap) {
            if (!copy) {
#pragma unroll
                for (int r = 0; r < kBkItems; ++r) {
                    const uint32_t i = i0 + (uint32_t)bk_item(kBkItems, r);
                    rank[r] = i < n ? kin[i] : 0u;
                }
            }
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                const uint32_t i = i0 + (uint32_t)bk_item(kBkItems, r);
                key[r] = i < n ? at[copy ? i : rank[r]] : 0u;
            }
#pragma unroll
            for (int r = 0; r < kBkItems; ++r) {
                const uint32_t i = i0 + (uint32_t)bk_item(kBkItems, r);
                if (i < n) to[i] = key[r];
            }
        }
        __syncthreads();
    }
    return part;
}

// The n keys of bucket b to a row of their own from rank0 on, or the differences found there back to their places.
__device__ __forceinline__ void bk_wide_copy(BkShared &s, BkSegments &segments, const BucketArgs &a, int c, int b, uint32_t rank0, uint32_t n, bool back) {
    const int64_t row = (int64_t)c * a.P;
    const BkSegments::Tile tile(a, c, (uint32_t)b, (uint32_t)b + 1u);
    for (uint32_t from = 0; from < n; from += kBkCap) {
        uint32_t v[kBkItems], at[kBkItems];
        __syncthreads();
        segments.collect(tile, from, s.scan);
#pragma unroll
        for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
            uint32_t to[kBkGroup];
            segments.where((uint32_t)bk_item(kBkItems, r0), (uint32_t)a.P - 1u, to, from);
#pragma unroll
            for (int i = 0; i < kBkGroup; ++i) at[r0 + i] = to[i];
        }
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            const uint32_t li = min((uint32_t)bk_item(kBkItems, r), n - from - 1u);
            v[r] = back ? a.dj[row + rank0 + from + li] : a.keys[row + at[r]];
        }
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            const uint32_t li = (uint32_t)bk_item(kBkItems, r);
            if (from + li < n) (back ? a.keys[row + at[r]] : a.sorted[row + rank0 + from + li]) = v[r];
        }
    }
    __syncthreads();
}

// One run of buckets (or, Direct: a whole row of at most kBkCap pixels, straight from the keys in pixel order, with the
// Jaccard differences left in their place and the loss complete).
// Time goes into vector instructions, 118 per 64 keys (69 % of it at 16 waves per CU): a thread's places of the order are
// neighbours, so that a difference is one new quotient less the one before, and the positives before a place are a sum over
// the block's threads. The rounds of a group of three wait for LDS once where each waited by itself, and what tells a key's place
// lies at constant offsets: with the quotients' fewer steps and scans by DPP 149 -> 118 instructions, (8,21,513,513) bf16 trained 270 -> 227 us,
// (4,19,512,1024) fp32 134 -> 111.
template <bool Direct>
__global__ __launch_bounds__(kBkThreads, 4) void bk_rank(const BucketArgs a, float *__restrict__ losses) {
    __shared__ BkShared s;
    __shared__ BkSegments at;                               // not for a whole row
    __shared__ double wave_loss[kBkWaves];
    const int c = Direct ? blockIdx.x : blockIdx.y;
    const int64_t row = (int64_t)c * a.P, cells = (int64_t)c * (a.stride + 1);
    const int runs = Direct ? 1 : (int)a.numbers[a.C + c];
    if (!Direct && (int)blockIdx.x >= runs) return;                    // block-uniform
    // neighbouring runs on one XCD: a tile's segments of theirs share cache lines
    const int g = Direct ? 0 : xcd_chunk((int)blockIdx.x, runs);
    const uint32_t b0 = Direct ? 0u : a.runs[cells + g], b1 = Direct ? 0u : a.runs[cells + g + 1];
    const uint32_t rank0 = Direct ? 0u : a.base[cells + b0], hot0 = Direct ? 0u : a.hot_base[cells + b0];
    const int n = Direct ? a.P : (int)(a.base[cells + b1] - rank0);
    const BkSegments::Tile tile = Direct ? BkSegments::Tile() : BkSegments::Tile(a, c, b0, b1);
    if (!Direct && (n > kBkCap || n == 0)) {                // block-uniform; too many: a large bucket
        if (threadIdx.x == 0) a.loss_part[2 * (int64_t)c * a.stride + g] = 0.0;
        return;
    }
    uint32_t *kin = a.keys + row;                           // the differences take the keys' places
    uint32_t limit = Direct ? 0u : bk_limit(a, c);
    float npos = Direct ? 0.f : (float)a.numbers[2 * a.C + c];
    if constexpr (!Direct) at.collect(tile, 0u, s.scan);

    uint32_t key[kBkItems], valid = 0, least, most, knee = 0;
    float share = 0.25f;
    bool flat = false;                                      // block-uniform: one value, in order as it stands
    const int rounds = (n + kBkThreads - 1) / kBkThreads;
    int first = bk_item(rounds, 0);
    // the thread's items: first, first + 64, ... inside the wave's part
    const int count = max(0, (min(n, first - (int)(threadIdx.x & 63) + rounds * kWave) - first + kWave - 1) / kWave);
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) key[r] = 0;
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                            // block-uniform
        uint32_t from[kBkGroup];
        if constexpr (!Direct) {
            at.where((uint32_t)(first + r0 * kWave), (uint32_t)a.P - 1u, from);
        } else {
#pragma unroll
            for (int i = 0; i < kBkGroup; ++i) from[i] = (uint32_t)min(first + (r0 + i) * kWave, n - 1);
        }
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) key[r0 + i] = kin[from[i]];
    }
    if constexpr (Direct) {
        const uint32_t top = class_top<kBkThreads>(a.block_table, a.key_blocks, c, s.crowd);
        limit = top - 1u;
        if (top == 0u) {                                    // block-uniform: a class without positives, see absent_min
            bk_range(s, key, (1u << count) - 1u, least, most);
            limit = min(least, kOne);
        }
#pragma unroll
        for (int r = 0; r < kBkItems; ++r)
            if (r < count && keep_key(key[r], limit)) valid |= 1u << r;
    } else {
        valid = (1u << count) - 1u;
    }
    if constexpr (Direct) {
        bk_range(s, key, valid, least, most);
        uint32_t hot = 0, all;
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) hot += ((valid >> r) & 1u) ? key[r] >> 31 : 0u;
        block_excl_scan(hot, s.scan, all);
        npos = (float)all;
        most = max(least, most);                            // no valid key: nothing below looks at the range
    } else {
        const uint32_t *bound = a.bounds + (int64_t)c * a.stride;
        const uint32_t buckets = a.numbers[c];
        most = b1 < buckets ? bound[b1 - 1] - 1u : limit;
        least = b0 ? bound[b0 - 1] : 0u;
        flat = least == most || npos == 0.f;                // a class without positives: the one value of its limit
        if (!flat && (b0 == 0 || b1 + 1u >= buckets)) {
            // beyond the sample lie a few more, far apart: their own bins
            bk_range(s, key, valid, least, most);
            knee = b0 ? a.numbers[4 * a.C + c] + 1u : a.numbers[3 * a.C + c];
            // Nor do the first keys lie evenly: errors near 1 crowd in classes that the network misses, as in bk_split. A
            // knee right at the first key left 260 keys in one bin ((1,32,256,256), soft: bk_rank and the crowded path 34 + 36 -> 19 + 4 us).
            if (!b0) knee = max(knee, least + (most - least) / 64u);
            share = b0 ? 0.75f : 0.25f;
        }
    }
    double part = 0.0;
    BkPair v[kBkChunk];
    uint32_t kept;
    float *result = reinterpret_cast<float *>(s.pair);      // by item
    bool in_order = flat;
    if (flat) {
        kept = (uint32_t)n;
#pragma unroll
        for (int r = 0; r < kBkItems; ++r)
            if ((valid >> r) & 1u) s.at((uint32_t)bk_item(rounds, r)) = bk_pair(key[r], (uint32_t)bk_item(rounds, r));
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kBkChunk; ++e) {
            const uint32_t p = threadIdx.x * kBkChunk + e;
            v[e] = p < kept ? s.at(p) : bk_last();
        }
        __syncthreads();
    } else {
        const BkBinning bins(least, knee, most, share);
        if constexpr (Direct) in_order = bk_sort(s, key, BkMask{valid}, rounds, bins, kept, v);
        else in_order = bk_sort(s, key, BkFirst{count}, rounds, bins, kept, v);
    }
    if (in_order) {                                         // block-uniform
        const uint32_t p0 = threadIdx.x * kBkChunk;
        uint32_t hot = 0, all;
        if (p0 < kept) {
#pragma unroll
            for (int e = 0; e < kBkChunk; ++e) hot += bk_hot_of(v[e]);
        }
        const uint32_t cs = hot0 + block_excl_scan(hot, s.scan, all);
        const uint32_t pos = rank0 + p0;
        // whole numbers: the positives that are left, and those and the keys so far
        float inter = npos - (float)cs, both = inter + (float)pos;                     // csrc/lovasz_softmax.cu:124-127
        float j_prev = pos == 0 ? 0.f : 1.f - whole_ratio(inter, both);
        auto step = [&](int e) {
            const float now = (float)bk_hot_of(v[e]);
            inter -= now;
            both = (both + 1.f) - now;
            const float j_now = 1.f - whole_ratio(inter, both);
            const float dj = j_now - j_prev;                                           // csrc/lovasz_softmax.cu:141-147
            j_prev = j_now;
            part = add_loss(part, key_error(bk_key_of(v[e])), dj);
            result[bk_item_of(v[e])] = dj;
        };
        if (p0 + kBkChunk <= kept) {
#pragma unroll
            for (int e = 0; e < kBkChunk; ++e) step(e);
        } else {
#pragma unroll
            for (int e = 0; e < kBkChunk; ++e)
                if (p0 + e < kept) step(e);
        }
    } else if constexpr (!Direct) {                         // values crowd: bk_rank_rest's
        if (threadIdx.x == 0) a.crowded[(int64_t)c * a.stride + atomicAdd(&a.numbers[8 * a.C + c], 1u)] = (uint32_t)g;
        return;
    } else {
        bk_range(s, key, valid, least, most);
        uint32_t rank[kBkItems];
        bk_ranks_crowded(s, key, valid, rounds, least, most, rank);
#pragma unroll
        for (int r = 0; r < kBkItems; ++r) {
            if (!((valid >> r) & 1u)) continue;
            const float dj = jaccard_step(npos, rank[r] & 0xFFFFu, rank[r] >> 16, key[r] >> 31);
            part = add_loss(part, key_error(key[r]), dj);
            result[bk_item(rounds, r)] = dj;
        }
    }
    part = wave_sum_f64(part);
    if ((threadIdx.x & 63) == 0) wave_loss[threadIdx.x >> 6] = part;
    __syncthreads();
    asm volatile("" : "+v"(first));                         // looked up again, not held across the sort
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                            // block-uniform
        uint32_t to[kBkGroup];
        float dj[kBkGroup];
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) dj[i] = result[first + (r0 + i) * kWave];   // past the last: inside the pairs
        if constexpr (!Direct) {
            at.where((uint32_t)(first + r0 * kWave), (uint32_t)a.P - 1u, to);
        } else {
#pragma unroll
            for (int i = 0; i < kBkGroup; ++i) to[i] = (uint32_t)(first + (r0 + i) * kWave);
        }
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i)
            if (r0 + i < count)
                kin[to[i]] = __builtin_bit_cast(uint32_t, (!Direct || ((valid >> (r0 + i)) & 1u)) ? dj[i] : 0.f);
    }
    if (threadIdx.x == 0) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < kBkWaves; ++w) sum += wave_loss[w];
        if constexpr (Direct) losses[c] = (float)sum;
        else a.loss_part[2 * (int64_t)c * a.stride + g] = sum;
    }
}

// A run whose values crowd.
__device__ __forceinline__ double bk_crowded_keys(BkShared &s, BkSegments &at, const BucketArgs &a, int c, int g) {
    const int64_t cells = (int64_t)c * (a.stride + 1);
    const uint32_t b0 = a.runs[cells + g], b1 = a.runs[cells + g + 1];
    const uint32_t rank0 = a.base[cells + b0], hot0 = a.hot_base[cells + b0];
    const int n = (int)(a.base[cells + b1] - rank0), rounds = (n + kBkThreads - 1) / kBkThreads;
    uint32_t *kin = a.keys + (int64_t)c * a.P;
    uint32_t key[kBkItems], rank[kBkItems], valid = 0, least, most;
    __syncthreads();
    at.collect(BkSegments::Tile(a, c, b0, b1), 0u, s.scan);
    // three rounds at a time, waited for together, and a key somewhere in the row for what is past the last
    auto fetch = [&](int r0, uint32_t (&to)[kBkGroup], uint32_t (&k)[kBkGroup]) {
        at.where((uint32_t)bk_item(rounds, r0), (uint32_t)a.P - 1u, to);
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) k[i] = kin[to[i]];
    };
#pragma unroll
    for (int r = 0; r < kBkItems; ++r) key[r] = 0;
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                            // block-uniform
        uint32_t to[kBkGroup], k[kBkGroup];
        fetch(r0, to, k);
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) {
            key[r0 + i] = k[i];
            if (r0 + i < rounds && bk_item(rounds, r0 + i) < n) valid |= 1u << (r0 + i);
        }
    }
    bk_range(s, key, valid, least, most);
    bk_ranks_crowded(s, key, valid, rounds, least, most, rank);
    const float npos = (float)a.numbers[2 * a.C + c];
    double part = 0.0;
#pragma unroll
    for (int r0 = 0; r0 < kBkItems; r0 += kBkGroup) {
        if (r0 >= rounds) break;                            // block-uniform
        uint32_t to[kBkGroup], k[kBkGroup];
        fetch(r0, to, k);                                   // read again: not held across the sort
#pragma unroll
        for (int i = 0; i < kBkGroup; ++i) {
            const uint32_t place = rank[r0 + i];
            if (!((valid >> (r0 + i)) & 1u)) continue;
            const float dj = jaccard_step(npos, rank0 + (place & 0xFFFFu), hot0 + (place >> 16), k[i] >> 31);
            part = add_loss(part, key_error(k[i]), dj);
            kin[to[i]] = __builtin_bit_cast(uint32_t, dj);
        }
    }
    return part;
}

// A bucket that outgrew the LDS.
__device__ __forceinline__ double bk_wide_bucket(BkShared &s, BkSegments &at, const BucketArgs &a, int c, int b) {
    const int buckets = (int)a.numbers[c];
    const int64_t cells = (int64_t)c * (a.stride + 1), row = (int64_t)c * a.stride;
    const uint32_t lo = b ? a.bounds[row + b - 1] : 0u, hi = b + 1 < buckets ? a.bounds[row + b] : bk_limit(a, c) + 1u;
    const uint32_t rank0 = a.base[cells + b], n = a.base[cells + b + 1] - rank0, hot0 = a.hot_base[cells + b];
    bk_wide_copy(s, at, a, c, b, rank0, n, false);
    // Sampled bounds leave a bucket of 7700 to 9000 keys in every other step or so: by ranges 30 us, by groups 45.
    const double part = n <= 4u * kBkCap ? bk_wide_keys(s, a, c, rank0, hot0, (int)n) : bk_huge_keys(s, a, c, rank0, hot0, n, lo, hi);
    bk_wide_copy(s, at, a, c, b, rank0, n, true);
    return part;
}

constexpr int kBkWideBlocks = 8;                // per class: a wide bucket at a time each; then as many as there are for crowded runs

// What bk_rank leaves: the wide buckets and the crowded runs. 256 registers, one block per CU: with two, a wide bucket's code
// spills (a bucket of (8,8,512,512) bf16 logits 94 -> 235 us, against the crowded runs of a sure network 107 -> 98).
__global__ __launch_bounds__(kBkThreads) void bk_rank_rest(const BucketArgs a) {
    __shared__ BkShared s;
    __shared__ BkSegments at;
    __shared__ double wave_loss[kBkWaves];
    const int c = blockIdx.y;
    const bool wide = blockIdx.x < kBkWideBlocks;           // block-uniform
    const int todo = (int)a.numbers[(wide ? 6 : 8) * a.C + c];
    const uint32_t *list = (wide ? a.large : a.crowded) + (int64_t)c * a.stride;
    double *loss_part = a.loss_part + 2 * (int64_t)c * a.stride;
    for (int i = wide ? blockIdx.x : blockIdx.x - kBkWideBlocks; i < todo; i += wide ? kBkWideBlocks : gridDim.x - kBkWideBlocks) {
        const int what = (int)list[i];
        double part = wide ? bk_wide_bucket(s, at, a, c, what) : bk_crowded_keys(s, at, a, c, what);
        part = wave_sum_f64(part);
        __syncthreads();
        if ((threadIdx.x & 63) == 0) wave_loss[threadIdx.x >> 6] = part;
        __syncthreads();
        if (threadIdx.x == 0) {
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < kBkWaves; ++w) sum += wave_loss[w];
            loss_part[wide ? a.stride + i : what] = sum;
        }
    }
}

// The tile's part of a class's flat bucket b, in `tile` (LDS) in order: the keys become their Jaccard differences. (A value that
// many share is mostly the positives' or the others' alone.)
__device__ __forceinline__ void bk_flat_keys(uint32_t *keys, uint32_t *scan, const BucketArgs &a, int c, int tile, int b) {
    constexpr uint32_t kPer = 8, kStep = kPer * kBkThreads;
    const int64_t cells = (int64_t)c * (a.stride + 1) + b, cell = cells * a.tiles;
    const uint32_t start = a.start[cell + tile], end = a.start[cell + a.tiles + tile];
    const uint32_t first = start & 0xFFFFu, n = (end & 0xFFFFu) - first, hots = (end >> 16) - (start >> 16);
    const float npos = (float)a.numbers[2 * a.C + c];
    if (n == 0) return;                                     // block-uniform
    uint32_t before = 0, hot_before = 0, rank0, hot0, unused;
    if ((int)threadIdx.x < tile) {
        const uint32_t from = a.start[cell + threadIdx.x], to = a.start[cell + a.tiles + threadIdx.x];
        before = (to & 0xFFFFu) - (from & 0xFFFFu);
        hot_before = (to >> 16) - (from >> 16);
    }
    block_excl_scan2(before, hot_before, scan, unused, rank0, unused, hot0);
    rank0 += a.base[cells];
    hot0 += a.hot_base[cells];
    const bool mixed = hots != 0u && hots != n;
    for (uint32_t i0 = 0; i0 < n; i0 += kStep) {
        const uint32_t p0 = i0 + threadIdx.x * kPer;
        uint32_t flags = hots ? 0xFFu : 0u;
        uint32_t cs = hot0 + (hots ? p0 : 0u);
        if (mixed) {
            flags = 0;
#pragma unroll
            for (uint32_t e = 0; e < kPer; ++e) flags |= (p0 + e < n ? keys[first + p0 + e] >> 31 : 0u) << e;
            uint32_t all;
            cs = hot0 + block_excl_scan((uint32_t)__builtin_popcount(flags), scan, all);
            hot0 += all;
        }
        float j_prev = jaccard(npos, rank0 + p0, cs);
#pragma unroll
        for (uint32_t e = 0; e < kPer; ++e) {
            cs += (flags >> e) & 1u;
            const float j_now = jaccard(npos, rank0 + p0 + e + 1u, cs);
            if (p0 + e < n) keys[first + p0 + e] = __builtin_bit_cast(uint32_t, j_now - j_prev);       // csrc/lovasz_softmax.cu:141-147
            j_prev = j_now;
        }
    }
}

// The tile's Jaccard differences in pixel order. The first block of a class adds up its loss.
__global__ __launch_bounds__(kBkThreads) void bk_restore(const BucketArgs a, float *__restrict__ losses) {
    __shared__ uint32_t dj[kBkTile];
    __shared__ uint32_t scan_tmp[2 * kSortWaves];
    const int c = blockIdx.y, tile = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int begin = tile * kBkTile, n = min(kBkTile, a.P - begin);
    uint32_t *row = a.keys + (int64_t)c * a.P + begin;
    const uint16_t *places = a.place + (int64_t)c * a.P + begin;
    uint32_t place[kBkTileItems], v[kBkTileItems];
#pragma unroll
    for (int r = 0; r < kBkTileItems; ++r) {
        const int li = bk_item(kBkTileItems, r);
        v[r] = li < n ? row[li] : 0u;                       // past the keys that take part: not used
        place[r] = li < n ? places[li] : kBkNowhere;
    }
#pragma unroll
    for (int r = 0; r < kBkTileItems; ++r) dj[bk_item(kBkTileItems, r)] = v[r];
    const int wides = (int)a.numbers[6 * a.C + c], flats = (int)a.numbers[7 * a.C + c];
    __syncthreads();
    if (flats > 0) {                                        // block-uniform
        for (int i = 0; i < flats; ++i)
            bk_flat_keys(dj, scan_tmp, a, c, tile, (int)a.large[(int64_t)c * a.stride + wides + i]);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < kBkTileItems; ++r) {
        const int li = bk_item(kBkTileItems, r);
        if (li < n) row[li] = place[r] != kBkNowhere ? dj[place[r]] : 0u;
    }
    if (tile != 0) return;
    __shared__ double wave_sum[kBkWaves];
    const int runs = (int)a.numbers[a.C + c];
    const double *sums = a.loss_part + 2 * (int64_t)c * a.stride;
    double sum = 0.0;
    for (int i = threadIdx.x; i < runs; i += kBkThreads) sum += sums[i];
    for (int i = threadIdx.x; i < wides + flats; i += kBkThreads) sum += sums[a.stride + i];
    sum = wave_sum_f64(sum);
    if (lane == 0) wave_sum[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double all = 0.0;
#pragma unroll
        for (int w = 0; w < kBkWaves; ++w) all += wave_sum[w];
        losses[c] = (float)all;
    }
}

}  // namespace plh
