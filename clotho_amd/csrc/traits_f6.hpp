// traits_f6.hpp — exact genome traits on the FP4 x FP6 matrix instructions
// (v_mfma_scale_f32_16x16x128_f8f6f4; device code shared by the pipeline's
// single-population and batched launches and the standalone contraction).
//
// Quantised int32 effects are written as balanced base-32 digits in
// [-16, 15]; a digit is exact in FP6 (E2M3: integers up to 16 in units of
// 1/8 or 1/4), a genotype bit is exact in FP4 (E2M1), and the products
// accumulate in FP32 as multiples of 1/8 that stay below 2^23 of them, so
// every sum is exact; the digit planes recombine in int64, and the results
// equal the sequential FP64 sums of the reference bit for bit
// (common_phenotype_accumulator,
// include/clotho/data_spaces/phenotype_evaluator/common_phenotype_accumulator_row_block_alignment.hpp:47-66).
//
// Why FP4 x FP6: an FP4 operand holds eight elements per dword, and since
// the site order inside a K block is free, a dword of 32 genotype bits
// becomes the 32 elements of a lane with four ANDs and one shift (bits 4 p
// and 4 p + 1 of a nibble read as 0.5 and 1.0).  The int8 path it replaced
// spread every genotype byte to 8 bytes through an LDS table, whose lookups
// (10 GB of LDS reads at 2e5 x 50,176 sites, with bank conflicts) bounded the
// one-trait pass.  Measured, int8 against this: one trait at 2e5 x 816 words
// 281 -> 241 us (5.4 TB/s of rows; copies run at 5.8), 16 traits at 5e5 x 2,072
// words 3.35 -> 2.17 ms, 16 traits of the full 31-bit range at 2e5 x 65,536
// sites 844 -> 656 us, 2,000 rows of 496 words 97 -> 10 us (Balance, below).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace clotho {
namespace f6 {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // 16-byte loads and stores
typedef __attribute__((address_space(1))) u32x4 g_u32x4;
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Callers may hold these buffers as generic pointers read from device memory;
// viewing them in the global address space keeps every access a global (not
// FLAT) instruction.
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* as_global(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}

// Digits per effect: P balanced base-32 digits hold |k| <= 15 (32^P - 1) / 31.
// The effects' bound is kept beside them (GenState::eff_max), so the passes
// multiply by no more planes than the population's effects have: four for
// |k| < 507,376 (e.g. N(0, 0.002^2) effects in units of 2^-24), seven for the
// whole range |k| < 2^30.
constexpr uint32_t kMaxPlanes = 7;
__host__ __device__ inline uint32_t digit_planes(uint32_t max_abs) {
    uint64_t bound = 15;
    uint32_t p = 1;
    while (p < kMaxPlanes && bound < max_abs) {
        bound = bound * 32 + 15;
        ++p;
    }
    return p;
}

// Trait classes: one kernel each, with a body per possible number of
// 16-column tiles.  Up to two traits (class 0) take eight columns per trait, so
// that a trait's planes sum over aligned lanes; more traits take P adjacent
// columns per trait (three and four in eights, where that takes no more tiles: 57
// -> 61 us at 60,000 rows x 256 words x 4, as an eighth of the lanes store).  Measured against the 32x32x64 instruction (same layout,
// rows paired by v_permlane16_swap), which alone runs twice as fast: with real
// operands both are held back by the card's power limit (1.7-1.9 GHz), and its
// coarser tiles multiply more padding (16 traits, seven planes, 2e5 x 65,536:
// 847 against 695 us; four planes, 5e5 x 2,136 words: 2,355 against 2,338).
constexpr int kClasses = 5;
__host__ __device__ constexpr int trait_class(uint32_t traits) {
    return traits <= 2 ? 0 : traits <= 4 ? 1 : traits <= 8 ? 2 : traits <= 16 ? 3 : 4;
}
__host__ __device__ inline uint32_t column_stride(uint32_t traits, uint32_t planes) {
    return traits <= 2 ? 8u : planes;
}
// Column tiles the kernel of the class multiplies by: the digit planes are
// packed (zeros past the last column) for this many tiles.
__host__ __device__ constexpr uint32_t kernel_tiles(uint32_t traits, uint32_t planes) {
    const uint32_t cols = traits * planes;
    switch (trait_class(traits)) {
        case 0: return 1u;
        case 1: return cols <= 16 ? 1u : 2u;
        case 2: return cols <= 32 ? 2u : cols <= 48 ? 3u : 4u;
        case 3: return cols <= 64 ? 4u : cols <= 80 ? 5u : 7u;
        default: return cols <= 128 ? 8u : cols <= 160 ? 10u : 14u;
    }
}

// Rows are read 16 words (one 128-byte line) at a time per row, a group of
// 1,024 sites: lane group g = lane / 16 holds words 4 g .. 4 g + 3 of row
// lane % 16 (two 16-byte loads), and K block q (of 8 per group, 128 sites)
// takes dword q of the lane's eight.  Element i = 8 r + p of a lane (nibble p
// of register r) is bit 4 p + r of its dword.
constexpr uint32_t kGroupWords = 16;
constexpr uint32_t kGroupBlocks = 8;  // K blocks of a group
constexpr int kRawBuffer = 0x00020000;  // dword 3 of a raw buffer resource
// A B fragment: 32 six-bit digits per lane, stored as dwords 0-3 of every
// lane (1 KB), then dwords 4-5 (512 bytes).
constexpr uint32_t kFragVecs = 96;  // in 16-byte pieces

__device__ inline uint32_t site_of(uint32_t G, uint32_t q, uint32_t lane, uint32_t i) {
    return 64 * kGroupWords * G + 256 * (lane >> 4) + 32 * q + 4 * (i & 7) + (i >> 3);
}

// FP6 E2M3 code of digit d: d/8 for elements whose FP4 one reads as 1.0
// (odd register), d/4 where it reads as 0.5 (even register); the products are
// d/8 either way.
__device__ inline uint32_t digit_code(int32_t d, bool odd) {
    const uint32_t a = (uint32_t)(d < 0 ? -d : d);
    return (odd ? a : a < 8 ? 2 * a : a + 8) | (d < 0 ? 32u : 0u);
}

// B fragments: fragment (G * K blocks + q) * NT + nt, column c of the lane
// (trait c / stride, plane c % stride), for rows of W words, A alleles and
// effects of at most `most`.  A block packs four fragments, one per wave.  Bound
// by the latency of its gathers: 32 at once, 12,288 sites x 2 traits 8.1 -> 7.0 us,
// 4,000 x 16 7.2 -> 5.9.
__device__ __forceinline__ void pack_block(const int32_t* __restrict__ eff_in, uint32_t T, uint32_t W,
                                           uint32_t A, uint32_t most,
                                           uint4* __restrict__ packed_in, uint32_t block) {
    const auto eff = as_global(eff_in);
    const uint32_t P = digit_planes(most);
    const uint32_t NT = kernel_tiles(T, P), stride = column_stride(T, P);
    const uint32_t NG = (W + kGroupWords - 1) / kGroupWords;
    constexpr uint32_t KB = kGroupBlocks;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t f = block * 4 + (threadIdx.x >> 6);  // fragment
    if (f >= NG * KB * NT) return;
    const uint32_t nt = f % NT, gq = f / NT, G = gq / KB, q = gq % KB;
    const uint32_t c = 16 * nt + (lane & 15);
    const uint32_t t = c / stride, p = c % stride;
    const bool live = t < T && p < P;
    // every load unconditional and ahead of its use, so that all are in flight
    int32_t v[32];
    const auto column = eff + min(t, T - 1);
#pragma unroll
    for (uint32_t i = 0; i < 32; ++i)
        v[i] = A ? column[(size_t)min(site_of(G, q, lane, i), A - 1) * T] : 0;
    // digit p of k: bits 5 p .. 5 p + 4 of k + 16 (32^7 - 1) / 31, less 16 (a
    // balanced digit does not depend on how many planes lie above it)
    uint32_t d[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (uint32_t i = 0; i < 32; ++i) {
        const int32_t k = site_of(G, q, lane, i) < A ? v[i] : 0;
        const uint64_t u = (uint64_t)((int64_t)k + 16ll * (((1ll << 35) - 1) / 31));
        const int32_t dg = (int32_t)((u >> (5 * p)) & 31u) - 16;
        const uint32_t code = live ? digit_code(dg, (i >> 3) & 1) : 0u;
        constexpr uint32_t kBits = 6;
        const uint32_t at = kBits * i;
        d[at / 32] |= code << (at % 32);
        if (at % 32 > 32 - kBits) d[at / 32 + 1] |= code >> (32 - at % 32);
    }
    const auto out = as_global(packed_in) + (size_t)f * kFragVecs;
    *((g_u32x4*)out + lane) = u32x4{d[0], d[1], d[2], d[3]};
    *((__attribute__((address_space(1))) u32x2*)(out + 64) + lane) = u32x2{d[4], d[5]};
}
// blocks of pack_block for rows of W words, at up to `planes` digit planes
__host__ __device__ inline uint32_t pack_blocks(uint32_t traits, uint32_t planes, uint32_t W) {
    return (W + kGroupWords - 1) / kGroupWords * (kGroupBlocks / 4) *
           kernel_tiles(traits, planes);
}

// Rows of a wave's row tile.
constexpr uint32_t kTileRows = 16;

// End of a stage: wait until at most N vector-memory loads are in flight,
// then (kLds) until the wave's LDS accesses are done, then meet the block;
// without kLds the caller has used everything it read from the buffers that
// the block overwrites next.  The builtin wait tells the compiler which loads have landed (so that it adds
// no wait of its own before the next stage's LDS reads); the asm statement
// repeats it with the barrier, and its memory clobber keeps the compiler
// from moving a memory access across.  __syncthreads instead waits for every
// load in flight (its fences cover global memory, and a fence restricted to
// LDS counts direct-to-LDS loads as pending LDS writes), so loads of the next
// group could not stay in flight across it.  The caller pins its loads with
// compiler barriers right after issuing them, so that none is issued
// between the wait and the barrier.
template <int N, bool kLds = true>
__device__ __forceinline__ void stage_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt immediate");
    __builtin_amdgcn_s_waitcnt((kLds ? 0x0070 : 0x0F70) | (N & 15) | ((N >> 4) << 14));
    if constexpr (kLds)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(N)
                     : "memory");
    else
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The B fragments are staged in LDS by direct-to-LDS loads in stages of QS K
// blocks and a ring of NB buffers, each an LDS object of its own and, as the
// stages per group are a multiple of the ring, the buffer of every stage a
// constant: a read of one buffer is then known not to touch another, which
// loads are filling, and needs no wait for those loads.  Classes 1-4 have four
// buffers, so that a stage's loads have three stages of products to
// land in (with two, every stage waited for the round trip it had just
// started; the digit planes of wide rows, past the L2's 4 MB, come from the
// Infinity Cache).
constexpr int kNarrowBlocks = 4;  // class 0: 6 KB stages, two buffers
__host__ __device__ constexpr int stage_blocks(int nt) { return nt <= 4 ? 2 : 1; }
__host__ __device__ constexpr int stage_vecs(int nt) { return stage_blocks(nt) * nt * (int)kFragVecs; }

// Groups whose digit sums stay exact in FP32: 16 (largest |digit|) x 2^19
// sites = 2^23 units of 1/8.  Longer rows are summed in segments of this many
// groups, each added to the output in int64.
constexpr uint32_t kSegGroups = 512;

// Stages of VECS 16-byte vectors from a segment's first fragment on into LDS
// buffers, each wave moving its share in 1 KB pieces (a loop of known trip
// count over a wave-uniform index: otherwise the compiler cannot count the
// loads in flight; the clamped last pieces are moved twice, with the same
// bytes).  As buffer loads: the compiler counts a global (FLAT) load to LDS as
// an access to either memory, and while one is in flight turns every wait for
// an LDS read or a row into a wait for everything.  The buffer starts at the
// segment's first fragment: the planes of a contraction's rows may take more
// than the 4 GB that an offset reaches, those of a segment take 88 MB at most.
template <int VECS>
struct Stager {
    static constexpr int kPieces = (VECS + 63) / 64;
    static constexpr int kPerWave = (kPieces + 3) / 4;
    __amdgpu_buffer_rsrc_t planes;
    uint32_t wave, lane;
    __device__ Stager(const uint4* packed, uint32_t first_stage, uint32_t w, uint32_t l)
        : planes(__builtin_amdgcn_make_buffer_rsrc((void*)(packed + (size_t)first_stage * VECS), 0, -1,
                                                   kRawBuffer)),
          wave(w),
          lane(l) {}
    __device__ __forceinline__ void operator()(uint32_t k, u32x4* buf) const {
        const uint32_t src = k * (VECS * 16u);
#pragma unroll
        for (int j = 0; j < kPerWave; ++j) {
            const uint32_t at = min((wave + 4 * j) * 64, (uint32_t)(VECS - 64));
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                planes, (__attribute__((address_space(3))) void*)(buf + at), 16, lane * 16,
                src + at * 16, 0, 0);
        }
    }
};

// A lane's 32 genotype bits as FP4 elements.  Opaque: expanded where it is
// multiplied, not stages ahead (the expanded operands of a group would cost
// the kernel its waves per SIMD).
__device__ __forceinline__ i32x8 expand_bits(uint32_t d) {
    asm volatile("" : "+v"(d));
    const uint32_t e = d >> 2;
    return i32x8{(int)(d & 0x11111111u), (int)(d & 0x22222222u), (int)(e & 0x11111111u),
                 (int)(e & 0x22222222u), 0, 0, 0, 0};
}
__device__ __forceinline__ void read_frag(const u32x4* fr, uint32_t lane, u32x4& b0, u32x2& b1) {
    b0 = fr[lane];
    b1 = reinterpret_cast<const u32x2*>(fr + 64)[lane];
}
__device__ __forceinline__ i32x8 frag_of(const u32x4& b0, const u32x2& b1) {
    return i32x8{(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, 0, 0};
}
// keeps a step's LDS reads and products where they are written: reading a
// whole stage's fragments up front would cost the waves per SIMD
__device__ __forceinline__ void step_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
constexpr int kScaleOne = 0x7F7F7F7F;  // E8M0 scales of 1
constexpr int kFp4 = 4, kFp6 = 2;      // operand formats: E2M1, E2M3

template <int N>
struct Int {
    static constexpr int value = N;
};

// The sum of v over the eight lanes of an aligned group, in each of them: quads,
// then their mirror images.
template <int kCtrl>
__device__ __forceinline__ int64_t add_dpp(int64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)v, kCtrl, 0xF, 0xF, true);
    const uint32_t hi =
        (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), kCtrl, 0xF, 0xF, true);
    return v + (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int64_t sum_eight(int64_t v) {
    v = add_dpp<0xB1>(v);      // quad_perm [1, 0, 3, 2]
    v = add_dpp<0x4E>(v);      // quad_perm [2, 3, 0, 1]
    return add_dpp<0x141>(v);  // row_half_mirror
}

// A wave's sums, of rows base .. base + 16 RT - 1, from its accumulators (eighths
// of integers): register i of lane (m, g) holds row 4 g + i of column m.
// Opaque indices: the output addresses of every segment are the same, and hoisted
// out of the segment loop they would be held, in scratch memory, through the
// products.
//
// Eight columns per trait: shift by 5 p and sum over the lanes (with shuffles by
// way of LDS, a generation's traits of 256 replicates took 245 us, in row shifts
// 224).
template <int RT>
__device__ __forceinline__ void store_eights(const f32x4 (&acc)[RT][1], uint32_t lane, uint32_t h,
                                             uint32_t T, int64_t* __restrict__ out_in,
                                             uint32_t row0, uint32_t base, bool add) {
    const auto out = as_global(out_in);
    uint32_t ol = lane, ob = base;
    asm volatile("" : "+v"(ol), "+s"(ob));
    const uint32_t om = ol & 15, og = ol >> 4, p = om & 7, t = om >> 3;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t v = sum_eight((int64_t)(int32_t)(acc[r][0][i] * 8.0f) << (5 * p));
            const uint32_t row = ob + 16 * r + 4 * og + i;
            if (p == 0 && row < h && t < T) {
                const size_t o = (size_t)(row - row0) * T + t;
                out[o] = add ? out[o] + v : v;
            }
        }
}
// Adjacent columns: through s_w, LDS of the wave's own, TILES row tiles at a time
// (in two parts half of one: rows 4 g and 4 g + 1, then 4 g + 2 and 4 g + 3).
template <int RT, int NT, int PARTS, int TILES>
__device__ __forceinline__ void store_adjacent(const f32x4 (&acc)[RT][NT], int32_t* s_w,
                                               uint32_t lane, uint32_t h, uint32_t T, uint32_t P,
                                               int64_t* __restrict__ out_in, uint32_t row0,
                                               uint32_t base, bool add) {
    static_assert(RT % TILES == 0 && (PARTS == 1 || TILES == 1), "whole passes");
    constexpr int REGS = 4 / PARTS;
    const auto out = as_global(out_in);
    uint32_t ol = lane, ob = base;
    asm volatile("" : "+v"(ol), "+s"(ob));
#pragma unroll
    for (int r = 0; r < RT; r += TILES) {
        const uint32_t first = ob + 16 * r;
        if (first >= h) break;
#pragma unroll
        for (int part = 0; part < PARTS; ++part) {
#pragma unroll
            for (int q = 0; q < TILES; ++q)
#pragma unroll
                for (int i = 0; i < REGS; ++i)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        s_w[(16 * q + REGS * (ol >> 4) + i) * (16 * NT) + 16 * nt + (ol & 15)] =
                            (int32_t)(acc[r + q][nt][REGS * part + i] * 8.0f);
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            for (uint32_t e = ol; e < 4 * REGS * TILES * T; e += 64) {
                const uint32_t pr = e / T, t = e % T;  // row of the part, of the pass
                const uint32_t lr = PARTS == 1 ? pr : 4 * (pr / REGS) + REGS * part + pr % REGS;
                const int32_t* const src = s_w + pr * (16 * NT) + t * P;
                int64_t v = 0;
#pragma unroll
                for (uint32_t p = 0; p < kMaxPlanes; ++p)  // all reads in flight at once
                    v += (int64_t)(src[p] & (p < P ? -1 : 0)) << (5 * p);
                if (first + lr < h) {
                    const size_t o = (size_t)(first - row0 + lr) * T + t;
                    out[o] = add ? out[o] + v : v;
                }
            }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
}
// int32 elements that a pass takes of a wave's LDS, and `past` more that the last
// trait's reads past its planes reach
constexpr int pass_elems(int nt, int parts, int tiles, int past) { return 256 / parts * tiles * nt + past; }
// row tiles per pass: as many as `share` elements hold
constexpr int pass_tiles(int rt, int nt, int parts, int past, int share) {
    int n = parts == 1 ? rt : 1;
    while (n > 1 && (rt % n != 0 || pass_elems(nt, parts, n, past) > share)) --n;
    return n;
}

// The products stay where they are written: otherwise they are sunk into the
// branch of the row tile that needs them, their operands spilled.
template <int RT, int NT>
__device__ __forceinline__ void pin(f32x4 (&acc)[RT][NT]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[r][nt]));
}

// One or two column tiles in stages of four K blocks, two buffers (class 0, and class
// 1 in batches, whose rows are mostly one group: 256 replicates x 3 / 4 traits
// 290 / 338 us in wave_wide's four stages and four row tiles, 239 / 275 here in three),
// one wave's share of groups [Ga, Gb) (at least
// one): rows base .. base + 16 RT - 1 (those below h; base wave-uniform).
// The next group's rows load into registers of their own at the group's first
// stage, after the stage's fragment loads, and stay in flight across its
// barrier (loads complete in issue order).  Site bits past the alleles meet
// zero digits, so loads past the row re-read its last words.  The last group,
// which loads no further rows or fragments, is a body of its own: under a
// run-time condition the compiler could not count what is in flight and would
// wait for everything before the first LDS read of a stage.
template <int RT, int NT, bool kEights>
__device__ __forceinline__ void wave_narrow(const uint64_t* __restrict__ rows_in, uint32_t h,
                                            uint32_t W, uint32_t T, uint32_t P,
                                            const uint4* __restrict__ packed_in,
                                            int64_t* __restrict__ out_in, uint32_t row0,
                                            uint32_t base, uint32_t Ga, uint32_t Gb,
                                            bool add, u32x4* const (&s_b)[4]) {
    constexpr int QS = kNarrowBlocks, SPG = 8 / QS;
    static_assert(SPG == 2, "two stages per group, two buffers");
    const auto rows = as_global(rows_in);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t m = lane & 15, g = lane >> 4;
    constexpr int VECS = QS * NT * (int)kFragVecs;
    const Stager<VECS> stage_b(packed_in, Ga * SPG, wave, lane);
    f32x4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __attribute__((address_space(1))) uint64_t* rp[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const uint32_t row = base + 16 * r + m;
        rp[r] = rows + (size_t)(row < h ? row : 0) * W;
    }
    auto load_rows = [&](uint32_t G, u32x4 (&x)[RT][2]) {
        const uint32_t w = min(kGroupWords * G + 4 * g, W - 4);  // W is a multiple of 8
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const g_u32x4* src = (const g_u32x4*)(rp[r] + w);
            x[r][0] = src[0];
            x[r][1] = src[1];
        }
    };
    u32x4 x[RT][2];
    stage_b(0, s_b[0]);
    load_rows(Ga, x);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    auto group = [&](uint32_t G, auto is_last) {
        constexpr bool last = decltype(is_last)::value != 0;
        u32x4 xn[RT][2];
#pragma unroll
        for (int s = 0; s < SPG; ++s) {
            u32x4* const cur = s_b[s];
            if (!last || s + 1 < SPG) stage_b((G - Ga) * SPG + s + 1, s_b[1 - s]);
            asm volatile("" ::: "memory");
            if (!last && s == 0) load_rows(G + 1, xn);
            asm volatile("" ::: "memory");
            u32x4 b0, c0;
            u32x2 b1, c1;
            i32x8 a[RT];
            read_frag(cur, lane, b0, b1);
#pragma unroll
            for (int j = 0; j < QS * NT; ++j) {
                const int q = s * QS + j / NT, nt = j % NT;
                if (j + 1 < QS * NT) read_frag(cur + (j + 1) * (int)kFragVecs, lane, c0, c1);
                const i32x8 b = frag_of(b0, b1);
                if (nt == 0) {
#pragma unroll
                    for (int r = 0; r < RT; ++r) a[r] = expand_bits(x[r][q >> 2][q & 3]);
                }
#pragma unroll
                for (int r = 0; r < RT; ++r)
                    acc[r][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        a[r], b, acc[r][nt], kFp4, kFp6, 0, kScaleOne, 0, kScaleOne);
                step_barrier();
                b0 = c0;
                b1 = c1;
            }
            // the next stage complete, this one's buffer free
            if (!last && s == 0)
                stage_barrier<2 * RT>();
            else
                stage_barrier<0>();
        }
        if constexpr (!last) {
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                x[r][0] = xn[r][0];
                x[r][1] = xn[r][1];
            }
        }
    };
    for (uint32_t G = Ga; G + 1 < Gb; ++G) group(G, Int<0>{});
    group(Gb - 1, Int<1>{});
    pin(acc);
    if constexpr (kEights) {
        store_eights<RT>(acc, lane, h, T, out_in, row0, base, add);
    } else {
        // a wave's quarter of the two buffers; up to four traits' reads end within two tiles
        constexpr int PAST = NT == 2 ? 0 : 8, TILES = pass_tiles(RT, NT, 1, PAST, 2 * VECS);
        static_assert(2 * VECS >= pass_elems(NT, 1, TILES, PAST), "a pass fits");
        u32x4* const s_q = (wave < 2 ? s_b[0] : s_b[1]) + (wave & 1) * (VECS / 2);
        store_adjacent<RT, NT, 1, TILES>(acc, reinterpret_cast<int32_t*>(s_q), lane, h, T, P, out_in,
                                         row0, base, add);
    }
}

// Loads of classes 1-4 that may be in flight at the end of stage s of a group:
// those issued after the fragments of the stage after the next (whose first
// fragments are read before the next barrier).  A stage issues the PPW
// fragment loads of the stage three ahead; stage 0 then 2 RT row loads.
template <int SPG, int RT, int PPW>
constexpr int stage_in_flight(int s) {
    return PPW + (s == 0 || s == 1 ? 2 * RT : 0);
}

// Classes 1-4, one wave's share of groups [Ga, Gb): rows base .. base + 16 RT -
// 1, NT column tiles, NB stage buffers.  The next group's rows load into registers of their own
// at the group's first stage (whole lines at a time: loading each half line
// in place once its registers were free saved registers, but four traits'
// rows took 0.37 instead of 0.29 ms).  Fragments are read from LDS two steps
// ahead of their products, across the stage barriers too: every barrier waits
// for one stage more than the next.  Up to two row tiles the last group is a
// body of its own, which loads nothing further and has nothing to wait for at its
// end (with the digit sums' reads in flight at once, 3,000 rows x 1,024 sites x 8
// traits: two row tiles 12.3 -> 11.3 us, one 10.5 -> 10.2).  With four row
// tiles that body would spill accumulators, and the last group loads its rows and
// the last stages once more.
// With two buffers (class 4, one row tile) a stage's loads have one stage of
// products to land in and its fragments are read from its own barrier on: three
// blocks per compute unit hide what four buffers, for which LDS holds one block,
// hid within the wave.
template <int RT, int NT, int NB>
__device__ __forceinline__ void wave_wide(const uint64_t* __restrict__ rows_in, uint32_t h,
                                          uint32_t W, uint32_t T, uint32_t P,
                                          const uint4* __restrict__ packed_in,
                                          int64_t* __restrict__ out_in, uint32_t row0,
                                          uint32_t base, uint32_t Ga, uint32_t Gb,
                                          bool add, u32x4* const (&s_b)[4]) {
    constexpr int QS = stage_blocks(NT), SPG = 8 / QS, VECS = stage_vecs(NT);
    static_assert(SPG % NB == 0, "every group starts in buffer 0");
    static_assert(NB == 4 || (NB == 2 && RT <= 2), "with two buffers the last group has its own body");
    constexpr bool kAhead = NB == 4;
    const auto rows = as_global(rows_in);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t m = lane & 15, g = lane >> 4;
    using Stage = Stager<VECS>;
    const Stage stage_b(packed_in, Ga * SPG, wave, lane);
    f32x4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[r][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __attribute__((address_space(1))) uint64_t* rp[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const uint32_t row = base + 16 * r + m;
        rp[r] = rows + (size_t)(row < h ? row : 0) * W;
    }
    using Rows = u32x4[RT][2];
    auto load_rows = [&](uint32_t G, Rows& x) {
        const uint32_t w = min(kGroupWords * G + 4 * g, W - 4);  // W is a multiple of 8
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const g_u32x4* const src = (const g_u32x4*)(rp[r] + w);
            x[r][0] = src[0];
            x[r][1] = src[1];
        }
    };
    const uint32_t n_stages = (Gb - Ga) * SPG;
    Rows x;
#pragma unroll
    for (int j = 0; j < NB - 1; ++j) stage_b(min((uint32_t)j, n_stages - 1), s_b[j]);
    load_rows(Ga, x);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    // fragment j of the stage in buffer s, later stages in the next buffers
    constexpr int STEPS = QS * NT;
    auto read = [&](int s, int j, u32x4& f0, u32x2& f1) {
        read_frag(s_b[(s + j / STEPS) % NB] + (j % STEPS) * (int)kFragVecs, lane, f0, f1);
    };
    u32x4 f0[3];
    u32x2 f1[3];
    if constexpr (kAhead) {
        read(0, 0, f0[0], f1[0]);
        read(0, 1, f0[1], f1[1]);
    }
    auto group = [&](uint32_t G, auto is_last) __attribute__((always_inline)) {
        constexpr bool last = decltype(is_last)::value != 0;
        Rows xn;
#pragma unroll
        for (int s = 0; s < SPG; ++s) {
            const uint32_t k = (G - Ga) * SPG + s;
            // NB - 1 stages ahead, into the buffer of the stage before this
            // one, which every wave is done with
            if (!last || s + NB - 1 < SPG)
                stage_b(min(k + NB - 1, n_stages - 1), s_b[(s + NB - 1) % NB]);
            asm volatile("" ::: "memory");
            if (!last && s == 0) load_rows(min(G + 1, Gb - 1), xn);
            asm volatile("" ::: "memory");
            i32x8 a[RT];
            if constexpr (!kAhead) {
                read(s, 0, f0[0], f1[0]);
                read(s, 1, f0[1], f1[1]);
            }
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                const int q = s * QS + j / NT, nt = j % NT, at = kAhead ? s * STEPS + j : j;
                if (kAhead ? !last || at + 2 < SPG * STEPS : j + 2 < STEPS)
                    read(s, j + 2, f0[(at + 2) % 3], f1[(at + 2) % 3]);
                if (nt == 0) {
#pragma unroll
                    for (int r = 0; r < RT; ++r) a[r] = expand_bits(x[r][q >> 2][q & 3]);
                }
                const i32x8 b = frag_of(f0[at % 3], f1[at % 3]);
#pragma unroll
                for (int r = 0; r < RT; ++r)
                    acc[r][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        a[r], b, acc[r][nt], kFp4, kFp6, 0, kScaleOne, 0, kScaleOne);
                step_barrier();
            }
            if constexpr (!kAhead) {
                // the next stage complete, this one's buffer free
                if (!last && s == 0)
                    stage_barrier<2 * RT>();
                else if (!last || s + 1 < SPG)
                    stage_barrier<0>();
            } else if constexpr (last) {
                // the stage after the next complete, where there is one
                if (s + NB - 1 < SPG)
                    stage_barrier<Stage::kPerWave, false>();
                else if (s + 2 < SPG)
                    stage_barrier<0, false>();
            } else {
                switch (s) {
                    case 0: stage_barrier<stage_in_flight<SPG, RT, Stage::kPerWave>(0), false>(); break;
                    case 1: stage_barrier<stage_in_flight<SPG, RT, Stage::kPerWave>(1), false>(); break;
                    default: stage_barrier<stage_in_flight<SPG, RT, Stage::kPerWave>(2), false>(); break;
                }
            }
        }
        if constexpr (!last) {
            // the fragment registers rotate by three: move the two read ahead
            // back to the front
            constexpr int off = kAhead ? (SPG * STEPS) % 3 : 0;
            if constexpr (off != 0) {
                const u32x4 a0 = f0[off], a1 = f0[(off + 1) % 3];
                const u32x2 c0 = f1[off], c1 = f1[(off + 1) % 3];
                f0[0] = a0;
                f0[1] = a1;
                f1[0] = c0;
                f1[1] = c1;
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                x[r][0] = xn[r][0];
                x[r][1] = xn[r][1];
            }
        }
    };
    constexpr bool kOwnLast = RT <= 2;
    for (uint32_t G = Ga; G + (kOwnLast ? 1 : 0) < Gb; ++G) group(G, Int<0>{});
    if constexpr (kOwnLast) {
        group(Gb - 1, Int<1>{});
        pin(acc);
    }
    stage_barrier<0>();  // every wave, and any repeated last stage, is done with the buffers
    constexpr int PARTS = 4 / NB, TILES = pass_tiles(RT, NT, PARTS, 8, VECS * NB);
    static_assert(VECS * NB >= pass_elems(NT, PARTS, TILES, 8), "a wave's quarter of the buffers holds a pass");
    u32x4* const s_q = NB == 2     ? (wave < 2 ? s_b[0] : s_b[1]) + (wave & 1) * (VECS / 2)
                       : wave == 0 ? s_b[0]
                       : wave == 1 ? s_b[1]
                       : wave == 2 ? s_b[2]
                                   : s_b[3];
    store_adjacent<RT, NT, PARTS, TILES>(acc, reinterpret_cast<int32_t*>(s_q), lane, h, T, P, out_in,
                                         row0, base, add);
}

// Groups [Ga, Gb) of the wave's rows, kSegGroups at a time: sums of row r into
// out[r - row0][T].  NB: wave_wide's stage buffers, 0 for wave_narrow; kEights: eight
// columns per trait (class 0).
template <int RT, int NT, int NB, bool kEights>
__device__ __forceinline__ void wave_rows(const uint64_t* rows, uint32_t h, uint32_t W, uint32_t T,
                                          uint32_t P, const uint4* packed, int64_t* out,
                                          uint32_t row0, uint32_t base, uint32_t Ga,
                                          uint32_t Gb, u32x4* const (&s_b)[4]) {
    for (uint32_t g0 = Ga; g0 < Gb; g0 += kSegGroups) {
        const uint32_t g1 = min(Gb, g0 + kSegGroups);
        if (g0 != Ga) __syncthreads();  // the previous segment's sums are out of the buffers
        if constexpr (NB == 0)
            wave_narrow<RT, NT, kEights>(rows, h, W, T, P, packed, out, row0, base, g0, g1, g0 != Ga,
                                         s_b);
        else
            wave_wide<RT, NT, NB>(rows, h, W, T, P, packed, out, row0, base, g0, g1, g0 != Ga,
                              s_b);
    }
}

// Waves per SIMD that the accumulators, the rows and one step's operands of a
// kernel, and its LDS, leave room for (its register limit).
constexpr int kBatchTiles = 3;  // row tiles of class 1's blocks in batches (wave_narrow)
constexpr int min_waves(int rt, int cls) {
    if (cls == 0) return rt >= 5 ? 3 : 4;
    if (cls == 1) return rt <= kBatchTiles ? 4 : 3;
    if (cls == 4) return rt == 1 ? 3 : 1;
    return rt <= 2 ? 3 : 2;
}

// The work of a balanced launch of B blocks over h rows: row blocks of
// block_rows rows (four waves of RT tiles).  Whole rounds first: block b takes
// the row blocks b, b + B, ... of the first `full` rounds; the R = RB - full B
// left are cut along K too, their R NG (row block, group) units spread evenly
// over the first B' = min(B, R NG) blocks.  A block's share of units is at
// most NG, so it touches at most two row blocks; a row block that lies in one
// block's share is written directly, the others as pieces (two slots per
// block) that k_trait_reduce sums.  So one round of resident blocks is full to
// its end whatever H is, and a small population fills the chip: 2,000 rows of
// 496 words are 8 row blocks but 248 units.
struct Balance {
    uint32_t B, RB, full, R;
    __host__ __device__ Balance(uint32_t h, uint32_t block_rows, uint32_t blocks)
        : B(blocks),
          RB((h + block_rows - 1) / block_rows),
          full(RB / blocks),
          R(RB - (RB / blocks) * blocks) {}
    // units over NG > 0 groups
    __host__ __device__ uint64_t units(uint32_t NG) const { return (uint64_t)R * NG; }
    __host__ __device__ uint32_t sharing(uint32_t NG) const {
        return units(NG) < B ? (uint32_t)units(NG) : B;
    }
    // first unit of sharing block b (b <= sharing)
    __host__ __device__ uint64_t first(uint32_t b, uint32_t NG) const {
        return units(NG) * b / sharing(NG);
    }
    // the sharing block that holds unit u
    __host__ __device__ uint32_t owner(uint64_t u, uint32_t NG) const {
        return (uint32_t)(((u + 1) * sharing(NG) - 1) / units(NG));
    }
};

// Rows of at most this many groups of a population are not cut: their pieces, sums
// and second prologues take longer than the units even out, and blocks of two row
// tiles per wave in turn reach more compute units (traits and free space of
// a generation, us: 40,000 rows x 48 words x 8 traits 34.9 -> 25.6, 200,000 x 16 x 6
// 44.3 -> 34.8, 400 x 16 x 4 16.7 -> 13.8).  With few row blocks only the shortest
// rows, as units along K then reach more compute units than row blocks do (3,000
// rows x 1 trait, 48 / 96 words: cut 17.6 / 17.9, whole 16.3 / 19.1; 40,000 rows
// 22.4 / 25.5, 19.6 / 25.5; 10,000 rows x 8, 96 words 21.7, 22.1; 200 rows x 20, 64
// words 17.4, 25.8).
__host__ __device__ constexpr uint32_t few_groups(uint32_t h, uint32_t traits) {
    const int cls = trait_class(traits);
    if (cls == 4) return h > 20480 ? 8u : 1u;
    return h > 16384 ? 8u : cls == 1 ? 3u : 4u;
}

// The sums of element e = (row, trait) of the rows past the whole rounds,
// where its row block was cut into pieces (rows of more than `few` groups).
__device__ __forceinline__ void reduce_pieces(const int64_t* __restrict__ part_in, uint32_t h,
                                              uint32_t W, uint32_t T, const Balance& bal,
                                              uint32_t block_rows, uint32_t few, uint64_t e,
                                              int64_t* __restrict__ out_in) {
    const uint32_t NG = (W + kGroupWords - 1) / kGroupWords;
    const uint32_t row0 = bal.full * bal.B * block_rows;
    const uint32_t local = (uint32_t)(e / T), row = row0 + local;
    if (row >= h || NG <= few) return;
    const uint32_t rb = local / block_rows;
    const uint32_t b0 = bal.owner((uint64_t)rb * NG, NG);
    const uint32_t b1 = bal.owner((uint64_t)(rb + 1) * NG - 1, NG);
    if (b0 == b1) return;  // written directly
    const auto part = as_global(part_in);
    const size_t slot = (size_t)block_rows * T;
    const size_t at = (size_t)(local - rb * block_rows) * T + (size_t)(e % T);
    // a block's first row block is in its slot 0; only b0 can have started
    // with the row block before
    int64_t v = part[(2 * (size_t)b0 + (bal.first(b0, NG) < (uint64_t)rb * NG ? 1 : 0)) * slot + at];
    uint32_t b = b0 + 1;
    for (; b + 7 <= b1; b += 8) {  // eight independent loads in flight
        int64_t x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = part[2 * (size_t)(b + j) * slot + at];
#pragma unroll
        for (int j = 0; j < 8; ++j) v += x[j];
    }
    for (; b <= b1; ++b) v += part[2 * (size_t)b * slot + at];
    as_global(out_in)[(size_t)row * T + (size_t)(e % T)] = v;
}

// Forms of a launch: one row block per block; a balanced launch; a balanced
// launch that takes rows of few groups in whole blocks.
enum class Form { kRowBlock, kBalanced, kBalancedFew };

// A block's shared buffers and the body for the population's tile count.
template <int RT, int CLS, Form kForm>
struct TraitsBlock {
    static constexpr uint32_t kWaveRows = RT * kTileRows, kBlockRows = 4 * kWaveRows;
    // stage buffers of wave_wide, 0 for wave_narrow and its two: two of class 4's
    // leave LDS for three blocks of one row tile (with two row tiles registers leave one)
    static constexpr bool kNarrow = CLS == 0 || (CLS == 1 && RT == kBatchTiles);
    static constexpr int kBuffers = kNarrow ? 0 : CLS == 4 && RT == 1 ? 2 : 4;
    static constexpr int kVecs = kNarrow    ? (CLS + 1) * kNarrowBlocks * (int)kFragVecs
                                 : CLS == 1 ? stage_vecs(2)
                                 : CLS <= 3 ? stage_vecs(4)  // the largest of 2 to 7 tiles
                                            : stage_vecs(14);
    static constexpr bool kRing = kBuffers == 4;
    static_assert(stage_vecs(4) >= stage_vecs(5) && stage_vecs(4) >= stage_vecs(7),
                  "the stage buffers hold every body's stage");

    // blocks: the balanced launch's count (W, most: wave-uniform, as given to
    // pack_block)
    __device__ static __forceinline__ void run(const uint64_t* __restrict__ rows, uint32_t h,
                                               uint32_t W, uint32_t most, uint32_t T,
                                               const uint4* __restrict__ packed,
                                               int64_t* __restrict__ out,
                                               int64_t* __restrict__ part, uint32_t block,
                                               uint32_t blocks) {
        const uint32_t blk = (uint32_t)__builtin_amdgcn_readfirstlane((int)block);
        __shared__ u32x4 s_b0[kVecs];
        __shared__ u32x4 s_b1[kVecs];
        __shared__ u32x4 s_b2[kRing ? kVecs : 1];
        __shared__ u32x4 s_b3[kRing ? kVecs : 1];
        u32x4* const s_b[4] = {s_b0, s_b1, s_b2, s_b3};
        const uint32_t P = digit_planes(most);
        const uint32_t NG = (W + kGroupWords - 1) / kGroupWords, NT = kernel_tiles(T, P);
        const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if (W == 0) {  // no words: every sum is zero
            const uint64_t n = (uint64_t)h * T;
            if constexpr (kForm != Form::kRowBlock)
                for (uint64_t e = blk * 256ull + threadIdx.x; e < n; e += blocks * 256ull)
                    as_global(out)[e] = 0;
            else
                for (uint32_t e = threadIdx.x; e < kBlockRows * T; e += 256)
                    if ((uint64_t)blk * kBlockRows * T + e < n)
                        as_global(out)[(size_t)blk * kBlockRows * T + e] = 0;
            return;
        }
        // a wave's rows from base on, `tiles` row tiles
        auto piece = [&](auto tiles, uint32_t base, uint32_t Ga, uint32_t Gb, int64_t* dst,
                         uint32_t row0) __attribute__((always_inline)) {
            constexpr int rt = decltype(tiles)::value;
#define CLOTHO_F6_BODY(n) \
    wave_rows<rt, n, kBuffers, CLS == 0>(rows, h, W, T, P, packed, dst, row0, base, Ga, Gb, s_b)
            if constexpr (CLS == 0) {
                CLOTHO_F6_BODY(1);
            } else if constexpr (CLS == 1) {
                if (NT == 1) CLOTHO_F6_BODY(1);
                else CLOTHO_F6_BODY(2);
            } else if constexpr (CLS == 2) {
                if (NT == 2) CLOTHO_F6_BODY(2);
                else if (NT == 3) CLOTHO_F6_BODY(3);
                else CLOTHO_F6_BODY(4);
            } else if constexpr (CLS == 3) {
                if (NT == 4) CLOTHO_F6_BODY(4);
                else if (NT == 5) CLOTHO_F6_BODY(5);
                else CLOTHO_F6_BODY(7);
            } else {
                if (NT == 8) CLOTHO_F6_BODY(8);
                else if (NT == 10) CLOTHO_F6_BODY(10);
                else CLOTHO_F6_BODY(14);
            }
#undef CLOTHO_F6_BODY
        };
        if constexpr (kForm == Form::kRowBlock) {
            piece(Int<RT>{}, blk * kBlockRows + wave * kWaveRows, 0, NG, out, 0);
            return;
        }
        if constexpr (kForm == Form::kBalancedFew) {
            if (NG <= few_groups(h, T)) {
                constexpr int kFewTiles = RT < 2 ? RT : 2;
                constexpr uint32_t few_rows = 4 * kFewTiles * kTileRows;
                for (uint64_t row = (uint64_t)blk * few_rows; row < h; row += (uint64_t)blocks * few_rows) {
                    const uint32_t base = (uint32_t)row + wave * (kFewTiles * kTileRows);
                    piece(Int<kFewTiles>{}, (uint32_t)__builtin_amdgcn_readfirstlane((int)base), 0, NG,
                          out, 0);
                    __syncthreads();  // the stage buffers are free for the next row block
                }
                return;
            }
        }
        // One loop over the block's row blocks, whole ones and then its share
        // of the units, so that the bodies are inlined once.
        const Balance bal(h, kBlockRows, blocks);
        uint64_t u = 0, u1 = 0;
        if (bal.R && blk < bal.sharing(NG)) {
            u = bal.first(blk, NG);
            u1 = bal.first(blk + 1, NG);
        }
        uint32_t round = 0, slot = 0;
        while (round < bal.full || u < u1) {
            uint32_t rb, Ga = 0, Gb = NG, row0 = 0;
            int64_t* dst = out;
            if (round < bal.full) {
                rb = round * blocks + blk;
                ++round;
            } else {
                const uint32_t r = (uint32_t)(u / NG);
                rb = bal.full * blocks + r;
                Ga = (uint32_t)(u - (uint64_t)r * NG);
                Gb = (uint32_t)min((uint64_t)NG, Ga + (u1 - u));
                u += Gb - Ga;
                if (Ga != 0 || Gb != NG) {
                    dst = part + (2 * (size_t)blk + slot) * kBlockRows * T;
                    row0 = rb * kBlockRows;
                }
                ++slot;
            }
            piece(Int<RT>{},
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)(rb * kBlockRows + wave * kWaveRows)),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)Ga),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)Gb), dst,
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)row0));
            __syncthreads();  // the stage buffers are free for the next row block
        }
    }
};

// The balanced launches: row tiles per wave of each class (as many as the
// registers of the class's resident waves hold) and the int64 elements of piece
// slots a launch of B blocks of block_rows rows needs.
__host__ __device__ constexpr int balanced_tiles(int cls) {
    return cls == 0 ? 5 : cls <= 3 ? 4 : 2;
}
__host__ __device__ constexpr uint32_t tile_block_rows(int tiles) { return 4u * tiles * kTileRows; }
__host__ __device__ constexpr uint32_t balanced_block_rows(int cls) {
    return tile_block_rows(balanced_tiles(cls));
}
__host__ __device__ inline size_t piece_elems(uint32_t traits, uint32_t block_rows, uint32_t blocks) {
    return 2 * (size_t)blocks * block_rows * traits;
}

}  // namespace f6
}  // namespace clotho
