// recombine.hpp — recombination, mutation and free-space partials of one
// generation by groups of 64 gametes (device code of pipeline.hip): of single
// populations and replicates but those with few events in many rows, and narrow
// rows of the largest batches (recombine_by_event, batch_recombine_shape).
//
// A child word is a select between the two words of its parent individual by
// the crossover mask {slots j : odd #{events e <= key_j}} (block_crossover with
// region_classifier's upper_bound).  Positions are unordered across slots, so
// the mask needs a position test per slot.  Testing a word's slots for one
// gamete costs a lookup per event; here 64 gametes are tested at once, with
// the roles of slots and gametes exchanged: the events of a group of 64
// gametes are sorted, px[r] is the XOR of the gamete bits of the r smallest,
// and a slot of position key takes px[#{events <= key}] — bit g says whether
// gamete g crosses an odd number of times up to that slot.  A lane per slot
// makes that one lookup per slot for 64 gametes, whatever the event count, and
// a 64 x 64 bit transpose across the wave turns a word's 64 lookups into its 64
// gametes' masks.  Per 64 (gamete, word) pairs the masks and the row select are
// about 70 vector instructions, where a lookup per event took 123 at rho = 5 and
// grew with rho.
//
// Measured against that form (1024-thread blocks over 64-word column tiles,
// per-word order statistics in LDS): N = 250,000, 2072 words, rho = 10: 5.70 -> 3.68
// ms; N = 100,000, 816 words, rho = 5: 0.551 -> 0.539 ms; N = 12,345, 336 words:
// 50 -> 39 us; N = 1000, 496 words: 35 -> 17 us; N = 200, 56 words: 24 -> 16 us.
// What bounds it: memory (2.4 GB at N = 100,000: 0.43 ms at the copy rate), with
// the vector, LDS and L1 address units each at 45-60% of that time.  The width
// of a row access matters most: 16 bytes per lane (8 bytes: 0.74 ms at N =
// 100,000; the L1 takes a quad of lanes per cycle whatever their width) on whole
// 128-byte lines (64 bytes: 0.82 ms; 512 bytes, with barriers between the
// waves that share such a tile: 0.58 ms).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pipeline.hpp"
#include "traits_f6.hpp"

namespace clotho {
namespace rec {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kWaves = kThreads / 64;
constexpr uint32_t kGroup = 64;  // gametes of a group: one bit each of a mask column
// Position buckets of the sorted events: 0.16 (rho = 5) and 0.3 (rho = 10)
// events per bucket, so that three comparisons almost always place a slot.
constexpr uint32_t kBucketBits = 11, kBuckets = 1u << kBucketBits;
// New mutations of a group: one with more is cut after the gametes that fit (a
// gamete has at most 127).
constexpr uint32_t kMutations = 192;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

// The two forms of a block.  Rows of more than kNarrowWords words: each wave
// makes and uses mask tiles of its own, kTile words (a 128-byte line) of all 64
// gametes.  Narrower rows: the waves share one mask tile of whole rows, and each
// produces a quarter of the group's rows.  kEvents: a group with more is cut, like
// one with many mutations; at rho = 10 a full group has 640 on average.
constexpr uint32_t kNarrowWords = 32;
struct Wide {
    static constexpr uint32_t kEvents = 768;
    static constexpr uint32_t kTile = 16;
    static constexpr uint32_t kPitch = kTile + 2;  // words per gamete row of a mask tile
    static constexpr uint32_t kMaskTiles = kWaves;
};
struct Narrow {
    static constexpr uint32_t kEvents = 576;
    static constexpr uint32_t kTile = kNarrowWords;
    static constexpr uint32_t kPitch = kTile + 2;
    static constexpr uint32_t kMaskTiles = 1;
};

template <class Form>
struct Shared {
    // mask tiles (mask_at); scratch while a table is built
    alignas(16) uint64_t mask[Form::kMaskTiles * kGroup * Form::kPitch];
    uint64_t px[Form::kEvents + 4];      // XOR of the gamete bits of the r smallest events
    uint32_t sorted[Form::kEvents + 4];  // the group's event keys, ascending
    uint32_t start[kBuckets / 2];  // first event of each bucket, two 16-bit counts per word
    u64x2 ptr[kGroup];             // addresses of each gamete's parent pair and child row
    uint32_t mut_off[kGroup + 1];  // first staged mutation of each gamete
    uint32_t mut[kMutations];      // the group's new mutations: slot | gamete << 24
    uint64_t scan[kWaves];
    uint32_t count;                // gametes of the group
    uint32_t total;                // their events
};
// What the table build keeps in the mask tiles.
template <class Form>
struct BuildScratch {
    uint32_t key_in[Form::kEvents];  // keys by gamete
    uint32_t rank_g[Form::kEvents];  // rank in the bucket | gamete << 16
    uint32_t key_b[Form::kEvents];   // keys and gametes in bucket order
    uint32_t g_b[Form::kEvents];
    uint64_t bits[Form::kEvents];    // gamete bits in key order
    f6::u32x4 rec[kGroup];           // {child row, top row, events | mutations << 8, first mutation}
    uint32_t ev_off[kGroup + 1];     // first event of each gamete in key_in
    static __device__ __forceinline__ BuildScratch& of(Shared<Form>& S) {
        static_assert(sizeof(BuildScratch) <= sizeof(S.mask), "scratch of the table build");
        return *reinterpret_cast<BuildScratch*>(S.mask);
    }
};

template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gl(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}
__device__ __forceinline__ uint32_t uni(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ uint32_t lane_of(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

// Exchange of lane bits with the dword index d of a lane's 64 bits (x0, x1):
// the element at (lane bit = a, d = b) moves to (lane bit = b, d = a).
template <int kShift, int kBanks>
__device__ __forceinline__ void swap_rows(uint32_t& x0, uint32_t& x1) {
    // lanes of the banks with the bit clear read kShift up, the others down
    const uint32_t n1 =
        (uint32_t)__builtin_amdgcn_update_dpp((int)x1, (int)x0, 0x100 + kShift, 0xF, kBanks, false);
    x0 = (uint32_t)__builtin_amdgcn_update_dpp((int)x0, (int)x1, 0x110 + kShift, 0xF,
                                               0xF & ~kBanks, false);
    x1 = n1;
}
template <int kQuad>
__device__ __forceinline__ void swap_quad(uint32_t& x0, uint32_t& x1, bool bit) {
    const uint32_t send = bit ? x0 : x1;
    const uint32_t recv = (uint32_t)__builtin_amdgcn_mov_dpp((int)send, kQuad, 0xF, 0xF, true);
    x0 = bit ? recv : x0;
    x1 = bit ? x1 : recv;
}
// Exchange of a register index with the bit-index bit of weight S: bits of x0
// with it set against bits of x1 with it clear (M = the bits with it clear).
template <int S, uint32_t M>
__device__ __forceinline__ void swap_bits(uint32_t& x0, uint32_t& x1) {
    if constexpr (S == 16 || S == 8) {
        constexpr uint32_t lo = S == 16 ? 0x05040100u : 0x06020400u;
        constexpr uint32_t hi = S == 16 ? 0x07060302u : 0x07030501u;
        const uint32_t y0 = __builtin_amdgcn_perm(x1, x0, lo);
        x1 = __builtin_amdgcn_perm(x1, x0, hi);
        x0 = y0;
    } else {
        const uint32_t y0 = (x0 & M) | ((x1 << S) & ~M);
        x1 = ((x0 >> S) & M) | (x1 & ~M);
        x0 = y0;
    }
}

// The masks of four words are made together.  Lane l looks up four slots,
// 4 chunk_of_lane(l) + i, of word l / 16 (one 16-byte load of keys); its column
// of slot i is x[0][i] (gametes 0 .. 31) and x[1][i].  The transpose exchanges
// the five gamete bits of the bit index for slot bits, three of them from the
// lane by way of the dword index and two from i, in 26 instructions a word:
// x[d][i] of lane l ends as half l & 1 (slots 32 (l & 1) .. + 31) of the row
// of gamete 8 (l / 2 mod 8) + 4 d + i.  (Lanes are numbered so that the half is
// the lane bit that is not exchanged and the two cheaper row shifts are used.)
__device__ __forceinline__ uint32_t chunk_of_lane(uint32_t lane) {
    return ((lane & 1u) << 3) | ((lane >> 1) & 7u);
}
__device__ __forceinline__ void transpose(uint32_t (&x)[2][4], uint32_t lane) {
#define CLOTHO_EACH _Pragma("unroll") for (int i = 0; i < 4; ++i)
    CLOTHO_EACH swap_rows<8, 0x3>(x[0][i], x[1][i]);
    CLOTHO_EACH swap_bits<16, 0x0000FFFFu>(x[0][i], x[1][i]);
    CLOTHO_EACH swap_rows<4, 0x5>(x[0][i], x[1][i]);
    CLOTHO_EACH swap_bits<8, 0x00FF00FFu>(x[0][i], x[1][i]);
    CLOTHO_EACH swap_quad<0x4E>(x[0][i], x[1][i], lane & 2);
    CLOTHO_EACH swap_bits<4, 0x0F0F0F0Fu>(x[0][i], x[1][i]);
#undef CLOTHO_EACH
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        swap_bits<2, 0x33333333u>(x[d][0], x[d][2]);
        swap_bits<2, 0x33333333u>(x[d][1], x[d][3]);
        swap_bits<1, 0x55555555u>(x[d][0], x[d][1]);
        swap_bits<1, 0x55555555u>(x[d][2], x[d][3]);
    }
}

// Dword of a mask tile with half h of its word w, gamete g: 16 bytes
// hold two words, low halves first (what the two words of a lane read at
// once).  The pitch and the exchanged pairs spread a store of the transpose (64
// dwords: eight gametes 8 apart, four words, two halves) over all 64 banks.
template <class Form>
__device__ __forceinline__ uint32_t mask_at(uint32_t g, uint32_t w, uint32_t h) {
    return g * (2 * Form::kPitch) + 4 * ((w >> 1) ^ (((g >> 4) & 3u) << 1)) + 2 * h + (w & 1u);
}

// Inclusive scan of v over the wave.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, uint32_t lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)v, d, 64);
        if ((int)lane >= d) v += y;
    }
    return v;
}

// The group's records, positions [p0, p0 + n) of the chunk (n <= 64, at least
// one), cut to the gametes whose events and mutations fit.  Ends with a block barrier.
template <class Form>
__device__ __forceinline__ void load_records(const Params& P, const Buffers& B, Shared<Form>& S,
                                             uint32_t sel, uint32_t wc, uint32_t wp, uint32_t p0,
                                             uint32_t n) {
    BuildScratch<Form>& T = BuildScratch<Form>::of(S);
    const uint32_t tid = threadIdx.x;
    if (tid < 64) {
        const uint32_t pos = p0 + min(tid, n - 1);
        f6::u32x4 r;
        if (B.by_parent) {
            r = ((const __attribute__((address_space(1))) f6::u32x4*)B.by_parent)[pos];
        } else {
            r.x = pos;
            r.y = gl(B.top)[pos];
            r.z = gl(B.n_events)[pos] | (gl(B.mut_count)[pos] << 8);
            r.w = gl(B.mut_local)[pos] + gl(B.mut_bsum)[pos / kScanBlock];
        }
        const uint32_t ne = tid < n ? r.z & 0xFFu : 0u;
        const uint32_t nm = tid < n ? r.z >> 8 : 0u;
        const uint32_t ei = wave_scan(ne, tid), mi = wave_scan(nm, tid);
        const uint64_t fits = __ballot(tid < n && ei <= Form::kEvents && mi <= kMutations);
        const uint32_t count = (uint32_t)__popcll(fits);  // a prefix of the lanes
        // lanes past the group repeat its last gamete, into a spare row
        const int src = (int)min(tid, count - 1);
        r.x = (uint32_t)__shfl((int)r.x, src, 64);
        r.y = (uint32_t)__shfl((int)r.y, src, 64);
        T.rec[tid] = r;
        const uint64_t* const spare = B.fix_part + (size_t)P.max_chunks * P.w_cap;
        S.ptr[tid] =
            u64x2{(uint64_t)(B.rows[sel] + (size_t)(r.y & ~1u) * wp),
                  (uint64_t)(tid < count ? B.rows[1 - sel] + (size_t)r.x * wc : spare)};
        T.ev_off[tid + 1] = ei;
        S.mut_off[tid + 1] = mi;
        if (tid == 0) T.ev_off[0] = S.mut_off[0] = 0;
        if (tid == count - 1) {
            S.count = count;
            S.total = ei;
        }
    } else {
        for (uint32_t i = tid - 64; i < kBuckets / 2; i += kThreads - 64) S.start[i] = 0;
    }
    __syncthreads();
}

// The group's sorted events, bucket starts and prefix XORs (px), and the slots
// of its new mutations.  Needs load_records; ends with a block barrier.
template <class Form>
__device__ __forceinline__ void build_table(const Params& P, const Buffers& B, Shared<Form>& S,
                                            uint32_t tid) {
    constexpr uint32_t kEvents = Form::kEvents;
    BuildScratch<Form>& T = BuildScratch<Form>::of(S);
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63;
    const uint32_t nb = uni(S.count), total = uni(S.total);
    // 1: kPerG threads per gamete read its events and count them into buckets
    constexpr uint32_t kPerG = kThreads / kGroup;
    const uint32_t g = tid / kPerG;
    if (g < nb) {
        const f6::u32x4 r = T.rec[g];
        const uint32_t ne = r.z & 0xFFu, off = T.ev_off[g];
        const auto ev = gl(B.events) + (size_t)r.x * P.ev_cap;
        for (uint32_t e = tid & (kPerG - 1); e < ne; e += kPerG) {
            const uint32_t key = ev[e], b = key >> (32 - kBucketBits);
            const uint32_t old = atomicAdd(&S.start[b >> 1], 1u << (16 * (b & 1)));
            T.key_in[off + e] = key;
            T.rank_g[off + e] = ((old >> (16 * (b & 1))) & 0xFFFFu) | (g << 16);
        }
        const uint32_t nm = r.z >> 8, mo = S.mut_off[g];
        if (nm) {
            const auto st = gl(B.state);
            const uint32_t F = st->free_count, A = st->alleles, fb = st->free_base;
            for (uint32_t j = tid & (kPerG - 1); j < nm; j += kPerG) {
                const uint32_t k = r.w + j;
                const uint32_t slot = k < F ? gl(B.free_list)[fb + k] : A + (k - F);
                S.mut[mo + j] = slot < st->all_size ? slot | (g << 24) : ~0u;
            }
        }
    }
    __syncthreads();
    // 2: bucket counts to starts, eight buckets per thread
    {
        static_assert(kBuckets == 8 * kThreads, "eight buckets per thread");
        f6::u32x4* const mine = reinterpret_cast<f6::u32x4*>(S.start) + tid;
        const f6::u32x4 c = *mine;
        uint32_t s[8] = {c.x & 0xFFFFu, c.x >> 16, c.y & 0xFFFFu, c.y >> 16,
                         c.z & 0xFFFFu, c.z >> 16, c.w & 0xFFFFu, c.w >> 16};
        uint32_t sum = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t n = s[i];
            s[i] = sum;
            sum += n;
        }
        const uint32_t inc = wave_scan(sum, lane);
        if (lane == 63) S.scan[tid >> 6] = inc;
        __syncthreads();
        uint32_t off = inc - sum;
        for (uint32_t w = 0; w < (tid >> 6); ++w) off += (uint32_t)S.scan[w];
        *mine = f6::u32x4{(s[0] + off) | ((s[1] + off) << 16), (s[2] + off) | ((s[3] + off) << 16),
                          (s[4] + off) | ((s[5] + off) << 16), (s[6] + off) | ((s[7] + off) << 16)};
    }
    __syncthreads();
    const uint16_t* const start = reinterpret_cast<const uint16_t*>(S.start);
    // 3: bucket order, then key order within the bucket (a bucket seldom
    // holds more than one)
    for (uint32_t i = tid; i < total; i += kThreads) {
        const uint32_t key = T.key_in[i], rg = T.rank_g[i];
        const uint32_t at = start[key >> (32 - kBucketBits)] + (rg & 0xFFFFu);
        T.key_b[at] = key;
        T.g_b[at] = rg >> 16;
    }
    __syncthreads();
    for (uint32_t i = tid; i < total; i += kThreads) {
        const uint32_t key = T.key_b[i], b = key >> (32 - kBucketBits);
        const uint32_t s0 = start[b], s1 = b + 1 < kBuckets ? start[b + 1] : total;
        uint32_t at = s0;
        for (uint32_t j = s0; j < s1; ++j) {
            const uint32_t o = T.key_b[j];
            at += (o < key || (o == key && j < i)) ? 1u : 0u;
        }
        S.sorted[at] = key;
        // the last gamete stands for the missing ones of a short group, too
        T.bits[at] = (T.g_b[i] + 1 == nb ? ~(uint64_t)0 : (uint64_t)1) << T.g_b[i];
    }
    __syncthreads();
    // 4: prefix XORs, kPer events per thread.  px[0]: the gametes whose top
    // strand is their parent's second row.  Entries past the last event repeat
    // it, so that a slot at the largest key may count the sentinels.
    {
        constexpr uint32_t kPer = (kEvents + kThreads - 1) / kThreads;
        uint64_t x[kPer], run = 0;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) {
            const uint32_t e = kPer * tid + i;
            run ^= e < total ? T.bits[e] : 0;
            x[i] = run;
        }
        uint32_t lo = (uint32_t)run, hi = (uint32_t)(run >> 32);
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t yl = (uint32_t)__shfl_up((int)lo, d, 64);
            const uint32_t yh = (uint32_t)__shfl_up((int)hi, d, 64);
            if ((int)lane >= d) {
                lo ^= yl;
                hi ^= yh;
            }
        }
        const uint64_t inc = ((uint64_t)hi << 32) | lo;
        if (lane == 63) S.scan[tid >> 6] = inc;
        const uint64_t swapped = __ballot(T.rec[lane].y & 1u);
        __syncthreads();
        uint64_t off = inc ^ run ^ swapped;
        for (uint32_t w = 0; w < (tid >> 6); ++w) off ^= S.scan[w];
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i)
            if (kPer * tid + i < kEvents) S.px[kPer * tid + i + 1] = off ^ x[i];
        if (tid == 0) S.px[0] = swapped;
        if (tid < 3) {
            uint64_t all = swapped;
            for (uint32_t w = 0; w < kWaves; ++w) all ^= S.scan[w];
            if (total + 1 + tid > kEvents) S.px[total + 1 + tid] = all;
            S.sorted[total + tid] = 0xFFFFFFFFu;
        }
    }
    __syncthreads();
}

// Masks of kQuads quads of words of a tile for the group's gametes; quad q has
// the words word(q) .. + 3, and is left out where they are past the tile's
// words.  A lookup is a chain of three LDS reads (bucket start, the bucket's first
// events, prefix mask): the quads go through it staggered, so that the reads
// of one are in flight while another is compared or transposed.
template <class Form, int kQuads, class Word>
__device__ __forceinline__ void quad_masks(const Shared<Form>& S, uint32_t* tile,
                                           const f6::u32x4 (&key)[kQuads], uint32_t words,
                                           uint32_t lane, Word word) {
    const uint16_t* const start = reinterpret_cast<const uint16_t*>(S.start);
    const uint32_t total = uni(S.total);
    uint32_t r[kQuads][4], e[kQuads][4][3], x[kQuads][2][4];
    auto find = [&](int q) {
#pragma unroll
        for (int i = 0; i < 4; ++i) r[q][i] = start[key[q][i] >> (32 - kBucketBits)];
    };
    auto read = [&](int q) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 3; ++u) e[q][i][u] = S.sorted[r[q][i] + u];
    };
    auto count = [&](int q) {
        bool any = false, more[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t k = key[q][i];
            more[i] = e[q][i][2] <= k;
            r[q][i] += (e[q][i][0] <= k ? 1u : 0u) + (e[q][i][1] <= k ? 1u : 0u) + (more[i] ? 1u : 0u);
            any = any || more[i];
        }
        if (__ballot(any)) {  // three or more events of a bucket at or below a slot: rare
#pragma unroll
            for (int i = 0; i < 4; ++i)
                while (more[i] && r[q][i] < total && S.sorted[r[q][i]] <= key[q][i]) ++r[q][i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint64_t v = S.px[r[q][i]];
            x[q][0][i] = (uint32_t)v;
            x[q][1][i] = (uint32_t)(v >> 32);
        }
    };
    auto turn = [&](int q) {
        transpose(x[q], lane);
        const uint32_t at = mask_at<Form>((lane & 14u) << 2, word(q) + (lane >> 4), lane & 1u);
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[at + (4 * d + i) * (2 * Form::kPitch)] = x[q][d][i];
    };
#pragma unroll
    for (int s = 0; s < kQuads + 3; ++s) {
        if (s < kQuads && word(s) < words) find(s);
        if (s >= 1 && s - 1 < kQuads && word(s - 1) < words) read(s - 1);
        __builtin_amdgcn_sched_barrier(0);
        if (s >= 2 && s - 2 < kQuads && word(s - 2) < words) count(s - 2);
        if (s >= 3 && word(s - 3) < words) turn(s - 3);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// (t & ~m) | (b & m) in one instruction
__device__ __forceinline__ uint32_t select32(uint32_t m, uint32_t b, uint32_t t) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)m, (int)b, (int)t, 0xCA);
}

// The rows of a step combined by op: lane l returns dword (l / 8 & 2) | l / 32 of
// its two words over all rows.
template <class Op>
__device__ __forceinline__ uint32_t fold_rows(f6::u32x4 x, Op op) {
    const auto r01 = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
    const auto r23 = __builtin_amdgcn_permlane32_swap(x[2], x[3], false, false);
    const auto r = __builtin_amdgcn_permlane16_swap(op(r01[0], r01[1]), op(r23[0], r23[1]), false, false);
    uint32_t y = op(r[0], r[1]);
    y = op(y, (uint32_t)__builtin_amdgcn_mov_dpp((int)y, 0x128, 0xF, 0xF, true));  // row_ror:8
    return y;
}

// A lane of a row access holds two words: the addresses of the pair (t, b) of a
// parent individual and of the child.
typedef __attribute__((address_space(1))) uint64_t g_u64;
__device__ __forceinline__ void load_pair(uint64_t pair, uint32_t wp, uint32_t col, f6::u32x4& t,
                                          f6::u32x4& b) {
    t = *(const f6::g_u32x4*)((const g_u64*)pair + col);
    b = *(const f6::g_u32x4*)((const g_u64*)pair + (size_t)wp + col);
}
// first word of the lane's pair in the parent row: in bounds for words past it
__device__ __forceinline__ uint32_t parent_column(uint32_t w, uint32_t wp) {
    return wp ? min(w, wp - 2) : 0u;
}
// Words are (low, high) pairs in rows, low and high pairs in masks.
__device__ __forceinline__ f6::u32x4 child_words(f6::u32x4 m, f6::u32x4 b, f6::u32x4 t,
                                                 f6::u32x4 keep) {
    return f6::u32x4{select32(m.x, b.x, t.x), select32(m.z, b.y, t.y), select32(m.y, b.z, t.z),
                     select32(m.w, b.w, t.w)} &
           keep;
}
__device__ __forceinline__ f6::u32x4 keep_words(const Buffers& B, uint32_t w, uint32_t wp) {
    const f6::u32x4 fixed = *(const f6::g_u32x4*)(gl(B.fixed_bits) + w);
    const uint32_t in_parent = w < wp ? ~0u : 0u;
    return f6::u32x4{~fixed.x & in_parent, ~fixed.y & in_parent, ~fixed.z & in_parent,
                     ~fixed.w & in_parent};
}
__device__ __forceinline__ void store_words(uint64_t row, uint32_t w, f6::u32x4 c) {
    __builtin_nontemporal_store(c, (f6::g_u32x4*)((g_u64*)row + w));
}
// The staged mutations m0 .. m1 - 1 whose word inside(word) takes: the lane that
// stored the word (owner(gamete, word)) flips the bit there, and every lane that
// holds it adds the bit to its OR.  The slot was free, so no other row of the
// population has the bit: the column's AND is zero without it, too.
template <class Form, class Inside, class Owner>
__device__ __forceinline__ void flip_mutations(const Shared<Form>& S, uint32_t m0, uint32_t m1,
                                               uint32_t lane, uint32_t w, f6::u32x4& acc_or,
                                               Inside inside, Owner owner) {
    for (uint32_t j = m0; j < m1; j += 64) {
        const uint32_t e = S.mut[min(j + lane, kMutations - 1)];
        uint64_t q = __ballot(j + lane < m1 && e != ~0u && inside((e & 0xFFFFFFu) >> 6));
        for (; q; q &= q - 1) {
            const uint32_t x = lane_of(e, (uint32_t)__builtin_ctzll(q));
            const uint32_t g = x >> 24, xw = (x >> 6) & 0x3FFFFu;
            const uint32_t bit = 1u << (x & 31u), at = (x >> 5) & 3u;
#pragma unroll
            for (uint32_t d = 0; d < 4; ++d) acc_or[d] |= w == (xw & ~1u) && at == d ? bit : 0u;
            if (lane == owner(g, xw))
                (void)__hip_atomic_fetch_xor((uint64_t*)S.ptr[g].y + xw, (uint64_t)1 << (x & 63),
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}
// the lane's 16 bytes of keys for quad words from w on (in bounds past the last word)
__device__ __forceinline__ f6::u32x4 load_keys(const Params& P, const Buffers& B, uint32_t w,
                                               uint32_t lane) {
    const uint32_t at = uni(min(w, P.w_cap - 4)) * 64u;
    return *(const f6::g_u32x4*)(gl(B.keys) + at + (lane >> 4) * 64 + 4 * chunk_of_lane(lane));
}

// Positions [c0, c1) of a row chunk: whole groups of gametes but for the last.
__device__ __forceinline__ void chunk_range(const Params& P, uint32_t chunk, uint32_t& c0,
                                            uint32_t& c1) {
    const uint32_t groups = (P.h + kGroup - 1) / kGroup;
    c0 = kGroup * (uint32_t)((uint64_t)groups * chunk / P.chunks);
    c1 = min(P.h, kGroup * (uint32_t)((uint64_t)groups * (chunk + 1) / P.chunks));
}
__device__ __forceinline__ void neutral_partials(const Params& P, const Buffers& B, uint32_t chunk,
                                                 uint32_t w0, uint32_t w1) {
    for (uint32_t w = w0 + threadIdx.x; w < w1; w += kThreads) {
        gl(B.var_part)[(size_t)chunk * P.w_cap + w] = 0;
        gl(B.fix_part)[(size_t)chunk * P.w_cap + w] = ~(uint64_t)0;
    }
}

// Rows of up to kNarrowWords words.  A row access has FW / 2 lanes per row (FW:
// the width rounded up to 8, 16 or 32 words), and the wave's kWaveRows rows take
// FW / 8 steps; their parent words load before the table is built.  The keys of
// a wave's words are the same for every group.
__device__ __forceinline__ void narrow_rows(const Params& P, const Buffers& B, Shared<Narrow>& S,
                                            uint32_t sel, uint32_t chunk, uint32_t wc,
                                            uint32_t wp) {
    constexpr uint32_t kWaveRows = kGroup / kWaves, kMaxSteps = kNarrowWords / 8;
    uint32_t c0, c1;
    chunk_range(P, chunk, c0, c1);
    if (c0 >= c1) return neutral_partials(P, B, chunk, 0, wc);
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63, wave = uni(tid >> 6);
    const uint32_t lg = wc <= 8 ? 2u : wc <= 16 ? 3u : 4u;  // lanes per row: 4, 8, 16
    const uint32_t step_rows = 64u >> lg, steps = kWaveRows >> (6 - lg);
    const uint32_t pair = 2 * (lane & ((1u << lg) - 1)), w = pair < wc ? pair : pair - 8;
    const uint32_t col = parent_column(w, wp), g0 = wave * kWaveRows + (lane >> lg);
    uint32_t* const tile = reinterpret_cast<uint32_t*>(S.mask);
    auto word = [&](int q) { return 4 * (wave + kWaves * (uint32_t)q); };
    f6::u32x4 key[kMaxSteps / 2];
#pragma unroll
    for (int q = 0; q < (int)kMaxSteps / 2; ++q) key[q] = load_keys(P, B, word(q), lane);
    const f6::u32x4 keep = keep_words(B, w, wp);
    f6::u32x4 acc_or = {0, 0, 0, 0}, acc_and = {~0u, ~0u, ~0u, ~0u};
    for (uint32_t p0 = c0; p0 < c1;) {
        load_records(P, B, S, sel, wc, wp, p0, min(kGroup, c1 - p0));
        const uint32_t nb = uni(S.count);
        f6::u32x4 t[kMaxSteps], b[kMaxSteps];
#pragma unroll
        for (uint32_t k = 0; k < kMaxSteps; ++k)
            if (k < steps) load_pair(S.ptr[g0 + step_rows * k].x, wp, col, t[k], b[k]);
        build_table(P, B, S, tid);
        quad_masks(S, tile, key, wc, lane, word);
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kMaxSteps; ++k) {
            if (k >= steps) break;
            const uint32_t g = g0 + step_rows * k;
            const f6::u32x4 m = *(const f6::u32x4*)(tile + mask_at<Narrow>(g, w, 0));
            const f6::u32x4 c = child_words(m, b[k], t[k], keep);
            store_words(S.ptr[g].y, w, c);
            acc_or |= c;
            acc_and &= c;
        }
        const uint32_t r0 = min(nb, wave * kWaveRows), r1 = min(nb, (wave + 1) * kWaveRows);
        flip_mutations(
            S, uni(S.mut_off[r0]), uni(S.mut_off[r1]), lane, w, acc_or,
            [](uint32_t) { return true; },
            [&](uint32_t g, uint32_t xw) { return ((g & (step_rows - 1)) << lg) | (xw >> 1); });
        p0 += nb;
        __syncthreads();  // the tables are free for the next group
    }
    // columns over the block's rows
    uint32_t* const red = tile;  // ORs, then ANDs
    for (uint32_t i = tid; i < 4 * kNarrowWords; i += kThreads) red[i] = i < 2 * kNarrowWords ? 0u : ~0u;
    __syncthreads();
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) {
        atomicOr(&red[2 * w + d], acc_or[d]);
        atomicAnd(&red[2 * kNarrowWords + 2 * w + d], acc_and[d]);
    }
    __syncthreads();
    if (tid < 2 * wc) {
        gl((uint32_t*)B.var_part)[2 * (size_t)chunk * P.w_cap + tid] = red[tid];
        gl((uint32_t*)B.fix_part)[2 * (size_t)chunk * P.w_cap + tid] = red[2 * kNarrowWords + tid];
    }
}

// Wider rows, column tiles [t0, t1).  The waves of a block share the tables and
// take column tiles of kTile words in turn, each on its own: no barrier in the
// tile loop, so that the waves of a compute unit drift apart and the lookups of
// some overlap the row loads and stores of others.
//
// A tile: the masks of its words go through the wave's LDS tile; then lane =
// (row, word pair), kStepRows rows per step, each a full 128-byte line.  The
// parent pairs of a whole tile are in registers: the loads of the next tile are
// issued as each step's words are consumed and stay in flight while the next
// tile's masks are made.  Siblings are adjacent: the second load of a pair hits
// the line of the first.  Every memory operation of the row loop is
// unconditional (lanes past the row repeat its last eight words, rows past a
// short group go to a spare row), so that the compiler's wait counts are exact.
__device__ __forceinline__ void wide_rows(const Params& P, const Buffers& B, Shared<Wide>& S,
                                          uint32_t sel, uint32_t chunk, uint32_t wc, uint32_t wp,
                                          uint32_t t0, uint32_t t1) {
    constexpr uint32_t kTile = Wide::kTile, kQuads = kTile / 4;
    constexpr uint32_t kStepRows = 128 / kTile, kSteps = kGroup / kStepRows;
    uint32_t c0, c1;
    chunk_range(P, chunk, c0, c1);
    if (c0 >= c1) return neutral_partials(P, B, chunk, kTile * t0, min(wc, kTile * t1));
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63, wave = uni(tid >> 6);
    const uint32_t f = lane / (kTile / 2);
    uint32_t* const tile_mask =
        reinterpret_cast<uint32_t*>(S.mask) + wave * (2 * kGroup * Wide::kPitch);
    bool first = true;
    for (uint32_t p0 = c0; p0 < c1; first = false) {
        load_records(P, B, S, sel, wc, wp, p0, min(kGroup, c1 - p0));
        const uint32_t nb = uni(S.count);
        f6::u32x4 t[kSteps], b[kSteps], key[kQuads];
        auto tile_keys = [&](uint32_t tile) {
#pragma unroll
            for (uint32_t i = 0; i < kQuads; ++i) key[i] = load_keys(P, B, kTile * tile + 4 * i, lane);
        };
        // the lane's two words of a tile
        auto word_of = [&](uint32_t tile) {
            const uint32_t w = kTile * tile + 2 * (lane & (kTile / 2 - 1));
            return w < wc ? w : w - 8;
        };
        const uint32_t my0 = t0 + wave;
        {
            const uint32_t col = parent_column(word_of(min(my0, t1 - 1)), wp);
#pragma unroll
            for (uint32_t k = 0; k < kSteps; ++k)
                load_pair(S.ptr[kStepRows * k + f].x, wp, col, t[k], b[k]);
            tile_keys(min(my0, t1 - 1));
        }
        build_table(P, B, S, tid);
        const uint32_t nm = uni(S.mut_off[nb]);
        const uint32_t my_mut = S.mut[min(lane, kMutations - 1)];
        for (uint32_t tile = my0; tile < t1; tile += kWaves) {
            uint32_t lane = tid & 63;  // opaque: nothing per lane is hoisted out and held
            asm volatile("" : "+v"(lane));
            const uint32_t fold_dword = ((lane >> 3) & 2u) | (lane >> 5);
            const uint32_t w = word_of(tile);
            const size_t part = 2 * ((size_t)chunk * P.w_cap + w) + fold_dword;
            const f6::u32x4 keep = keep_words(B, w, wp);
            const uint32_t old_or = gl((const uint32_t*)B.var_part)[part];
            const uint32_t old_and = gl((const uint32_t*)B.fix_part)[part];
            quad_masks(S, tile_mask, key, kTile, lane, [](int q) { return 4u * (uint32_t)q; });
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            f6::u32x4 acc_or = {0, 0, 0, 0}, acc_and = {~0u, ~0u, ~0u, ~0u};
            const bool mutated =
                nm > 64 || __ballot(lane < nm && (my_mut & 0xFFFFFFu) / (64 * kTile) == tile) != 0;
            // the next tile's loads; after the last tile, one word pair per row
            const bool next = tile + kWaves < t1;
            const uint32_t ntile = next ? tile + kWaves : tile;
            tile_keys(ntile);
            const uint32_t ncol = next ? parent_column(word_of(ntile), wp) : 0u;
            f6::u32x4 mask[2];
            u64x2 ptr[2];
            auto read_step = [&](uint32_t k) {
                const uint32_t g = kStepRows * k + f;
                mask[k & 1] = *(const f6::u32x4*)(tile_mask + mask_at<Wide>(g, w - kTile * tile, 0));
                ptr[k & 1] = S.ptr[g];
            };
            read_step(0);
#pragma unroll
            for (uint32_t k = 0; k < kSteps; ++k) {
                if (k + 1 < kSteps) read_step(k + 1);
                const u64x2 p = ptr[k & 1];
                const f6::u32x4 c = child_words(mask[k & 1], b[k], t[k], keep);
                store_words(p.y, w, c);
                acc_or |= c;
                acc_and &= c;
                load_pair(p.x, wp, ncol, t[k], b[k]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (mutated)
                flip_mutations(
                    S, 0, nm, lane, w, acc_or, [&](uint32_t xw) { return xw / kTile == tile; },
                    [](uint32_t g, uint32_t xw) {
                        return (g % kStepRows) * (kTile / 2) + (xw % kTile) / 2;
                    });
            // lanes of one dword store the same value
            const uint32_t col_or = fold_rows(acc_or, [](uint32_t x, uint32_t y) { return x | y; });
            const uint32_t col_and = fold_rows(acc_and, [](uint32_t x, uint32_t y) { return x & y; });
            gl((uint32_t*)B.var_part)[part] = first ? col_or : col_or | old_or;
            gl((uint32_t*)B.fix_part)[part] = first ? col_and : col_and & old_and;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        p0 += nb;
        __syncthreads();  // the tables are free for the next group
    }
}

// Blocks: P.chunks ranges of groups x P.splits ranges of column tiles (more
// than one where the row chunks alone do not fill the chip; every split builds
// the tables of its chunk); narrow rows have no column tiles.
struct Recombine {
    static constexpr int kThreads = (int)rec::kThreads;
    static constexpr int kMinWaves = 3;  // three blocks per compute unit (LDS)
    __host__ __device__ static uint32_t blocks(const Params& P) { return P.chunks * P.splits; }
    // blocks with work at a child width of wc words
    __host__ __device__ static uint32_t live(const Params& P, uint32_t wc) {
        return !wc ? 0u : wc <= kNarrowWords ? P.chunks : P.chunks * P.splits;
    }
    __device__ static __forceinline__ void run(const Params& P, const Buffers& B, uint32_t sel,
                                               uint32_t blk) {
        static_assert(sizeof(Shared<Wide>) >= sizeof(Shared<Narrow>), "one allocation for both");
        __shared__ alignas(16) char memory[sizeof(Shared<Wide>)];
        const auto st = gl(B.state);
        const uint32_t wc = uni(st->wc), wp = uni(st->wp);  // multiples of eight
        if (blk >= live(P, wc)) return;
        if (wc <= kNarrowWords)
            return narrow_rows(P, B, *reinterpret_cast<Shared<Narrow>*>(memory), sel, uni(blk), wc,
                               wp);
        const uint32_t chunk = uni(blk / P.splits), split = uni(blk % P.splits);
        const uint32_t tiles = (wc + Wide::kTile - 1) / Wide::kTile;
        const uint32_t t0 = split * tiles / P.splits, t1 = (split + 1) * tiles / P.splits;
        if (t0 < t1)
            wide_rows(P, B, *reinterpret_cast<Shared<Wide>*>(memory), sel, chunk, wc, wp, t0, t1);
    }
};

}  // namespace rec
}  // namespace clotho
