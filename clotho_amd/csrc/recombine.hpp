// recombine.hpp — recombination, mutation and free-space partials of one
// generation of a single population (device code of pipeline.hip).
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
// Events of a group: a group with more is cut after the gametes that fit (a
// gamete has at most 127).  At rho = 10 a full group has 640 on average.
constexpr uint32_t kEvents = 768;
// Position buckets of the sorted events: 0.16 (rho = 5) and 0.3 (rho = 10)
// events per bucket, so that three comparisons almost always place a slot.
constexpr uint32_t kBucketBits = 11, kBuckets = 1u << kBucketBits;
// New mutations of a group, likewise (a gamete has at most 127).
constexpr uint32_t kMutations = 192;
constexpr int kMinWaves = 3;           // three blocks per compute unit (LDS)
constexpr uint32_t kTile = 16;         // words of a wave's tile: one 128-byte line per row
constexpr uint32_t kPitch = kTile + 2;  // words per gamete row of the mask tile
constexpr uint32_t kStepRows = 64 * 2 / kTile;       // rows of a step, two words per lane
constexpr uint32_t kSteps = kGroup / kStepRows;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

struct Shared {
    // each wave's mask tile (mask_at); scratch while a table is built
    alignas(16) uint64_t mask[kWaves][kGroup * kPitch];
    uint64_t px[kEvents + 4];      // XOR of the gamete bits of the r smallest events
    uint32_t sorted[kEvents + 4];  // the group's event keys, ascending
    uint32_t start[kBuckets / 2];  // first event of each bucket, two 16-bit counts per word
    u64x2 ptr[kGroup];             // addresses of each gamete's parent pair and child row
    f6::u32x4 rec[kGroup];         // {child row, top row, events | mutations << 8, first mutation}
    uint32_t ev_off[kGroup + 1];   // first event of each gamete, unsorted
    uint32_t mut_off[kGroup + 1];  // first staged mutation of each gamete
    uint32_t mut[kMutations];      // the group's new mutations: slot | gamete << 24
    uint64_t scan[kWaves];
    uint32_t count;                // gametes of the group
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

// Dword of the mask tile with half h of word w (mod kTile), gamete g: 16 bytes
// hold two words, low halves first (what the two words of a lane read at
// once).  The pitch and the exchanged pairs spread a store of the transpose (64
// dwords: eight gametes 8 apart, four words, two halves) over all 64 banks.
__device__ __forceinline__ uint32_t mask_at(uint32_t g, uint32_t w, uint32_t h) {
    return g * (2 * kPitch) + 4 * ((w >> 1) ^ (((g >> 4) << 1) & (kTile / 2 - 1))) + 2 * h + (w & 1u);
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
__device__ __forceinline__ void load_records(const Buffers& B, Shared& S, uint32_t sel, uint32_t wc,
                                             uint32_t wp, uint32_t p0, uint32_t n) {
    const uint32_t tid = threadIdx.x;
    if (tid < 64) {
        const uint32_t pos = p0 + min(tid, n - 1);  // lanes past the end repeat the last gamete
        f6::u32x4 r = ((const __attribute__((address_space(1))) f6::u32x4*)B.by_parent)[pos];
        const uint32_t ne = tid < n ? r.z & 0xFFu : 0u;
        const uint32_t nm = tid < n ? r.z >> 8 : 0u;
        const uint32_t ei = wave_scan(ne, tid), mi = wave_scan(nm, tid);
        const uint64_t fits = __ballot(tid < n && ei <= kEvents && mi <= kMutations);
        const uint32_t count = (uint32_t)__popcll(fits);  // a prefix of the lanes
        // lanes past the group repeat its last gamete
        const int src = (int)min(tid, count - 1);
        r.x = (uint32_t)__shfl((int)r.x, src, 64);
        r.y = (uint32_t)__shfl((int)r.y, src, 64);
        S.rec[tid] = r;
        S.ptr[tid] = u64x2{(uint64_t)(B.rows[sel] + (size_t)(r.y & ~1u) * wp),
                           (uint64_t)(B.rows[1 - sel] + (size_t)r.x * wc)};
        S.ev_off[tid + 1] = ei;
        S.mut_off[tid + 1] = mi;
        if (tid == 0) {
            S.ev_off[0] = S.mut_off[0] = 0;
            S.count = count;
        }
    } else {
        for (uint32_t i = tid - 64; i < kBuckets / 2; i += kThreads - 64) S.start[i] = 0;
    }
    __syncthreads();
}

// The group's sorted events, bucket starts and prefix XORs (px), and the slots
// of its new mutations.  Needs load_records; ends with a block barrier.
__device__ __forceinline__ void build_table(const Params& P, const Buffers& B, Shared& S,
                                            uint32_t tid) {
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid & 63;
    const uint32_t nb = uni(S.count), total = uni(S.ev_off[nb]);
    // scratch in the mask tile: unsorted keys, then the keys and gametes in
    // bucket order, and the gamete bits in key order
    uint32_t* const key_in = reinterpret_cast<uint32_t*>(&S.mask[0][0]);
    uint32_t* const rank_g = key_in + kEvents;   // rank in the bucket | gamete << 16
    uint32_t* const key_b = rank_g + kEvents;
    uint32_t* const g_b = key_b + kEvents;
    uint64_t* const bits = reinterpret_cast<uint64_t*>(g_b + kEvents);
    static_assert(sizeof(S.mask) >= kEvents * (16 + 8), "scratch of the table build");
    // 1: kPerG threads per gamete read its events and count them into buckets
    constexpr uint32_t kPerG = kThreads / kGroup;
    const uint32_t g = tid / kPerG;
    if (g < nb) {
        const f6::u32x4 r = S.rec[g];
        const uint32_t ne = r.z & 0xFFu, off = S.ev_off[g];
        const auto ev = gl(B.events) + (size_t)r.x * P.ev_cap;
        for (uint32_t e = tid & (kPerG - 1); e < ne; e += kPerG) {
            const uint32_t key = ev[e], b = key >> (32 - kBucketBits);
            const uint32_t old = atomicAdd(&S.start[b >> 1], 1u << (16 * (b & 1)));
            key_in[off + e] = key;
            rank_g[off + e] = ((old >> (16 * (b & 1))) & 0xFFFFu) | (g << 16);
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
        const uint32_t key = key_in[i], rg = rank_g[i];
        const uint32_t at = start[key >> (32 - kBucketBits)] + (rg & 0xFFFFu);
        key_b[at] = key;
        g_b[at] = rg >> 16;
    }
    __syncthreads();
    for (uint32_t i = tid; i < total; i += kThreads) {
        const uint32_t key = key_b[i], b = key >> (32 - kBucketBits);
        const uint32_t s0 = start[b], s1 = b + 1 < kBuckets ? start[b + 1] : total;
        uint32_t at = s0;
        for (uint32_t j = s0; j < s1; ++j) {
            const uint32_t o = key_b[j];
            at += (o < key || (o == key && j < i)) ? 1u : 0u;
        }
        S.sorted[at] = key;
        // the last gamete stands for the missing ones of a short group, too
        bits[at] = (g_b[i] + 1 == nb ? ~(uint64_t)0 : (uint64_t)1) << g_b[i];
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
            run ^= e < total ? bits[e] : 0;
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
        const uint64_t swapped = __ballot(S.rec[lane].y & 1u);
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

// Masks of the tile's words for the group's gametes, four words at a time.  A
// lookup is a chain of three LDS reads (bucket start, the bucket's first events,
// prefix mask): the quads go through it staggered, so that the reads of one are
// in flight while another is compared or transposed.
__device__ __forceinline__ void tile_masks(const Shared& S, uint32_t* tile,
                                           const f6::u32x4 (&key)[kTile / 4], uint32_t total,
                                           uint32_t lane) {
    constexpr int kQuads = kTile / 4;
    const uint16_t* const start = reinterpret_cast<const uint16_t*>(S.start);
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
        const uint32_t at = mask_at((lane & 14u) << 2, 4 * q + (lane >> 4), lane & 1u);
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[at + (4 * d + i) * (2 * kPitch)] = x[q][d][i];
    };
#pragma unroll
    for (int s = 0; s < kQuads + 3; ++s) {
        if (s < kQuads) find(s);
        if (s >= 1 && s - 1 < kQuads) read(s - 1);
        __builtin_amdgcn_sched_barrier(0);
        if (s >= 2 && s - 2 < kQuads) count(s - 2);
        if (s >= 3) turn(s - 3);
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

// Blocks: P.chunks ranges of groups x P.splits ranges of column tiles (more
// than one where the row chunks alone do not fill the chip; every split builds
// the tables of its chunk).  The waves of a block share the tables and take
// column tiles of kTile words in turn, each on its own: no barrier in the tile
// loop, so that the waves of a compute unit drift apart and the lookups of some
// overlap the row loads and stores of others.
//
// A tile: the masks of its words go through the wave's LDS tile; then lane =
// (row, word), kStepRows rows per step, each a full 128-byte line.  The
// parent pairs of a whole tile are in registers: the loads of the next tile are
// issued as each step's words are consumed and stay in flight while the next
// tile's masks are made.  Siblings are adjacent: the second load of a pair hits
// the line of the first.  Every memory operation of the row loop is
// unconditional (lanes past the row repeat its last eight words, rows past a
// short group its last row), so that the compiler's wait counts are exact.
struct Recombine {
    static constexpr int kThreads = (int)rec::kThreads;
    __host__ __device__ static uint32_t blocks(const Params& P) { return P.chunks * P.splits; }
    __device__ static __forceinline__ void run(const Params& P, const Buffers& B, uint32_t sel,
                                               uint32_t blk) {
        __shared__ Shared S;
        const auto st = gl(B.state);
        const uint32_t wc = uni(st->wc), wp = uni(st->wp);  // multiples of eight
        if (!wc) return;
        const uint32_t chunk = uni(blk / P.splits), split = uni(blk % P.splits);
        const uint32_t tiles = (wc + kTile - 1) / kTile;
        const uint32_t t0 = split * tiles / P.splits, t1 = (split + 1) * tiles / P.splits;
        if (t0 == t1) return;
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const uint32_t lane = tid & 63, wave = uni(tid >> 6);
        // positions [c0, c1): whole groups of gametes but for the last
        const uint32_t groups = (P.h + kGroup - 1) / kGroup;
        const uint32_t c0 = kGroup * (uint32_t)((uint64_t)groups * chunk / P.chunks);
        const uint32_t c1 =
            min(P.h, kGroup * (uint32_t)((uint64_t)groups * (chunk + 1) / P.chunks));
        if (c0 >= c1) {  // no rows: neutral partials
            for (uint32_t w = kTile * t0 + tid; w < min(wc, kTile * t1); w += kThreads) {
                gl(B.var_part)[(size_t)chunk * P.w_cap + w] = 0;
                gl(B.fix_part)[(size_t)chunk * P.w_cap + w] = ~(uint64_t)0;
            }
            return;
        }
        const auto keys = gl(B.keys);
        const uint32_t f = lane / (kTile / 2);
        uint32_t* const tile_mask = reinterpret_cast<uint32_t*>(S.mask[wave]);
        bool first = true;
        for (uint32_t p0 = c0; p0 < c1; first = false) {
            load_records(B, S, sel, wc, wp, p0, min(kGroup, c1 - p0));
            const uint32_t nb = uni(S.count), total = uni(S.ev_off[nb]);
            f6::u32x4 t[kSteps], b[kSteps], key[kTile / 4];
            const uint32_t lane_key = (lane >> 4) * 64 + 4 * chunk_of_lane(lane);
            auto load_keys = [&](uint32_t tile) {
#pragma unroll
                for (uint32_t i = 0; i < kTile / 4; ++i) {
                    const uint32_t w = uni(min(kTile * tile + 4 * i, P.w_cap - 4));
                    key[i] = *(const f6::g_u32x4*)(keys + w * 64u + lane_key);
                }
            };
            // the lane's two words of a tile
            auto word_of = [&](uint32_t tile) {
                const uint32_t w = kTile * tile + 2 * (lane & (kTile / 2 - 1));
                return w < wc ? w : w - 8;
            };
            auto load_pair = [&](uint32_t k, uint64_t pair, uint32_t col) {
                const auto row = (const __attribute__((address_space(1))) uint64_t*)pair;
                t[k] = *(const f6::g_u32x4*)(row + col);
                b[k] = *(const f6::g_u32x4*)(row + (size_t)wp + col);
            };
            auto column = [&](uint32_t w) { return wp ? min(w, wp - 2) : 0u; };
            const uint32_t my0 = t0 + wave;
            {
                const uint32_t col = column(word_of(min(my0, t1 - 1)));
#pragma unroll
                for (uint32_t k = 0; k < kSteps; ++k) load_pair(k, S.ptr[kStepRows * k + f].x, col);
                load_keys(min(my0, t1 - 1));
            }
            build_table(P, B, S, tid);
            const uint32_t nm = uni(S.mut_off[nb]);
            const uint32_t my_mut = S.mut[min(lane, kMutations - 1)];
            for (uint32_t tile = my0; tile < t1; tile += kWaves) {
                uint32_t lane = tid & 63;  // opaque: nothing per lane is hoisted out and held
                asm volatile("" : "+v"(lane));
                const uint32_t fold_dword = ((lane >> 3) & 2u) | (lane >> 5);
                const uint32_t w = word_of(tile);
                const size_t part = (size_t)chunk * P.w_cap + w;
                const f6::u32x4 fixed = *(const f6::g_u32x4*)(gl(B.fixed_bits) + w);
                const uint32_t old_or = gl((const uint32_t*)B.var_part)[2 * part + fold_dword];
                const uint32_t old_and = gl((const uint32_t*)B.fix_part)[2 * part + fold_dword];
                tile_masks(S, tile_mask, key, total, lane);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const uint32_t in_parent = w < wp ? ~0u : 0u;
                f6::u32x4 keep, acc_or = {0, 0, 0, 0}, acc_and = {~0u, ~0u, ~0u, ~0u};
#pragma unroll
                for (int e = 0; e < 4; ++e) keep[e] = ~fixed[e] & in_parent;
                const bool mutated =
                    nm > 64 ||
                    __ballot(lane < nm && (my_mut & 0xFFFFFFu) / (64 * kTile) == tile) != 0;
                // the next tile's loads; after the last tile, one word pair per row
                const bool next = tile + kWaves < t1;
                const uint32_t ntile = next ? tile + kWaves : tile;
                load_keys(ntile);
                const uint32_t ncol = next ? column(word_of(ntile)) : 0u;
                f6::u32x4 mask[2];
                u64x2 ptr[2];
                auto read_step = [&](uint32_t k) {
                    const uint32_t g = kStepRows * k + f;
                    mask[k & 1] = *(const f6::u32x4*)(tile_mask + mask_at(g, w - kTile * tile, 0));
                    ptr[k & 1] = S.ptr[g];
                };
                read_step(0);
#pragma unroll
                for (uint32_t k = 0; k < kSteps; ++k) {
                    if (k + 1 < kSteps) read_step(k + 1);
                    const f6::u32x4 m = mask[k & 1];
                    const u64x2 p = ptr[k & 1];
                    // words are (low, high) pairs in rows, low and high pairs in masks
                    f6::u32x4 c = {select32(m.x, b[k].x, t[k].x), select32(m.z, b[k].y, t[k].y),
                                   select32(m.y, b[k].z, t[k].z), select32(m.w, b[k].w, t[k].w)};
                    c &= keep;
                    __builtin_nontemporal_store(
                        c, (f6::g_u32x4*)((__attribute__((address_space(1))) uint64_t*)p.y + w));
                    acc_or |= c;
                    acc_and &= c;
                    load_pair(k, p.x, ncol);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // New mutations of the tile (few): the lane that stored the word
                // flips the bit there.  The slot was free, so no other row of the
                // population has the bit: the column's AND is zero without it, too.
                if (mutated) {
                    // rows of a short group were stored by several lanes: vmcnt(0)
                    if (nb < kGroup) __builtin_amdgcn_s_waitcnt(0x0F70);
                    for (uint32_t j = 0; j < nm; j += 64) {
                        const uint32_t e = S.mut[min(j + lane, kMutations - 1)];
                        uint64_t q = __ballot(j + lane < nm && e != ~0u &&
                                              (e & 0xFFFFFFu) / (64 * kTile) == tile);
                        for (; q; q &= q - 1) {
                            const uint32_t x = lane_of(e, (uint32_t)__builtin_ctzll(q));
                            const uint32_t g = x >> 24, xw = (x >> 6) & 0x3FFFFu;
                            const uint32_t bit = 1u << (x & 31u), at = (x >> 5) & 3u;
#pragma unroll
                            for (uint32_t e4 = 0; e4 < 4; ++e4)
                                acc_or[e4] |= w == (xw & ~1u) && at == e4 ? bit : 0u;
                            if (lane == (g % kStepRows) * (kTile / 2) + (xw % kTile) / 2)
                                (void)__hip_atomic_fetch_xor((uint64_t*)S.ptr[g].y + xw,
                                                             (uint64_t)1 << (x & 63),
                                                             __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                }
                // lanes of one dword store the same value
                const uint32_t col_or = fold_rows(acc_or, [](uint32_t x, uint32_t y) { return x | y; });
                const uint32_t col_and =
                    fold_rows(acc_and, [](uint32_t x, uint32_t y) { return x & y; });
                gl((uint32_t*)B.var_part)[2 * part + fold_dword] = first ? col_or : col_or | old_or;
                gl((uint32_t*)B.fix_part)[2 * part + fold_dword] =
                    first ? col_and : col_and & old_and;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            p0 += nb;
            __syncthreads();  // the tables are free for the next group
        }
    }
};

}  // namespace rec
}  // namespace clotho
