// traits_mfma.hip — genotype x effect contraction on CDNA4 matrix cores.
//
// z[h][t] = sum_j bit(h, j) * effect[j][t] over bit-packed rows (the
// population-wide common_phenotype_accumulator,
// include/clotho/data_spaces/phenotype_evaluator/common_phenotype_accumulator_row_block_alignment.hpp:47-66).
//
// Exact path (v_mfma_scale_f32_16x16x128_f8f6f4): quantised int32 effects are
// written as balanced base-32 digits in FP6, genotype bits as FP4 0/1; every
// FP32 sum is exact and the digit planes recombine in int64, so the sums equal
// the FP64 sequential sums of the reference bit for bit (effects are multiples
// of 2^q).  Kernel bodies: traits_f6.hpp.
//
// Split-BF16 path (v_mfma_f32_16x16x32_bf16): bits expand to BF16 0/1 (exact),
// effects split into 1-3 BF16 terms hi + mid + lo, FP32 accumulation per
// 64-word K chunk, chunks reduced in FP64.
//
// Operand layouts (16x16xK, wave64): lane l supplies A row (l % 16) and B
// column (l % 16) for K elements [K/4 * (l / 16), K/4 * (l / 16 + 1)); the
// accumulator lane l holds column (l % 16), rows 4 * (l / 16) + i.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "pipeline.hpp"
#include "traits.hpp"
#include "traits_f6.hpp"

namespace clotho {
namespace {

using f6::kGroupWords;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));


// two genotype bits -> two BF16 0/1 halves (1.0 = 0x3F80)
__device__ inline uint32_t bits2_bf16(uint32_t two) {
    return ((two * 0x8001u) & 0x10001u) * 0x3F80u;
}


// Exact-path kernels: bodies in traits_f6.hpp.
__global__ void __launch_bounds__(256) k_pack_digits_of(const int32_t* __restrict__ eff, uint32_t T,
                                                        uint32_t words, uint32_t sites,
                                                        uint32_t most,
                                                        uint4* __restrict__ packed) {
    f6::pack_block(eff, T, words, sites, most, packed, blockIdx.x);
}

template <int CLS>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(f6::min_waves(f6::balanced_tiles(CLS), CLS))))
    k_traits_exact(const uint64_t* __restrict__ rows, uint32_t h, uint32_t words, uint32_t most,
                   uint32_t T, const uint4* __restrict__ packed, int64_t* __restrict__ traits,
                   int64_t* __restrict__ part, uint32_t blocks) {
    f6::TraitsBlock<f6::balanced_tiles(CLS), CLS, f6::Form::kBalanced>::run(
        rows, h, words, most, T, packed, traits, part, blockIdx.x, blocks);
}

// one row block of RT row tiles per wave and block
template <int RT, int CLS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f6::min_waves(RT, CLS))))
    k_traits_rows(const uint64_t* __restrict__ rows, uint32_t h, uint32_t words, uint32_t most,
                  uint32_t T, const uint4* __restrict__ packed, int64_t* __restrict__ traits) {
    f6::TraitsBlock<RT, CLS, f6::Form::kRowBlock>::run(rows, h, words, most, T, packed, traits,
                                                       nullptr, blockIdx.x, 0);
}

__global__ void __launch_bounds__(256) k_exact_reduce(uint32_t h, uint32_t words, uint32_t T,
                                                      uint32_t blocks,
                                                      const int64_t* __restrict__ part,
                                                      int64_t* __restrict__ traits) {
    const uint32_t rows = f6::balanced_block_rows(f6::trait_class(T));
    f6::reduce_pieces(part, h, words, T, f6::Balance(h, rows, blocks), rows, 0,
                      (uint64_t)blockIdx.x * 256 + threadIdx.x, traits);
}


// Split-BF16 contraction, K chunked: block = 4 waves x RT row tiles, one
// chunk of kChunkGroups 16-word groups.  K block q (of 32 per group) takes
// byte q % 8 of the lane's word q / 8, i.e. sites bf_site(G, q, lane / 16, i);
// bits expand to BF16 0/1 through a 256-entry LDS table (byte -> 8 BF16).
// The B fragments (TERMS per K block, 1 KB each) are staged in LDS for the
// whole block, kStageBlocks K blocks at a time, double buffered and moved by
// direct global-to-LDS loads while the previous stage is multiplied: every
// wave reads its B operands from LDS instead of each wave fetching them from
// L2.  The FP32 accumulators are flushed into FP64 after every stage (256
// sites), so FP32 rounding acts only on short partial sums; FP64
// partial[chunk][row][t].
constexpr uint32_t kChunkGroups = 16;
constexpr uint32_t kStageBlocks = 8;

__host__ __device__ inline uint32_t bf_site(uint32_t G, uint32_t q, uint32_t g, uint32_t i) {
    return 64 * (16 * G + 4 * g + q / 8) + 8 * (q & 7) + i;
}

template <int RT, int TERMS>
__global__ void __launch_bounds__(256) k_traits_bf16(const uint64_t* __restrict__ rows_in,
                                                     uint32_t h, uint32_t W, uint32_t T,
                                                     const uint4* __restrict__ packed_in,
                                                     double* __restrict__ partial) {
    constexpr uint32_t QS = kStageBlocks;
    constexpr uint32_t FR = QS * TERMS;       // 1 KB fragments per stage
    constexpr uint32_t SPG = 32 / QS;         // stages per group
    static_assert(FR % 4 == 0 && SPG % 2 == 0, "stage pieces per wave, stage parity per group");
    // the two stage buffers are two LDS objects, not halves of one: a read of
    // one is then known not to touch the other, which direct-to-LDS loads are
    // filling, and needs no wait for those loads (SPG is even, so the buffer
    // of every stage is a constant)
    __shared__ uint4 s_b0[FR * 64];
    __shared__ uint4 s_b1[FR * 64];
    __shared__ uint4 s_lut[256];
    const auto rows = f6::as_global(rows_in);
    const auto packed = f6::as_global(packed_in);
    const uint32_t NG = (W + 15) / 16;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t m = lane & 15, g = lane >> 4;
    const uint32_t base = (blockIdx.x * 4 + wave) * (16 * RT);
    const uint32_t G0 = blockIdx.y * kChunkGroups;
    const uint32_t G1 = min(NG, G0 + kChunkGroups);
    {
        const uint32_t b8 = threadIdx.x;
        s_lut[b8] = make_uint4(bits2_bf16(b8 & 3), bits2_bf16((b8 >> 2) & 3),
                               bits2_bf16((b8 >> 4) & 3), bits2_bf16(b8 >> 6));
    }
    double acc64[RT][4];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc64[r][i] = 0.0;
    const __attribute__((address_space(1))) uint64_t* rp[RT];
    bool rv[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const uint32_t row = base + 16 * r + m;
        rv[r] = row < h;
        rp[r] = rows + (size_t)(rv[r] ? row : 0) * W;
    }
    auto load_rows = [&](uint32_t G, f6::u32x4 (&x)[RT][2]) {
        const uint32_t w = 16 * G + 4 * g;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            if (rv[r] && w < W) {
                const f6::g_u32x4* src = (const f6::g_u32x4*)(rp[r] + w);
                x[r][0] = src[0];
                x[r][1] = src[1];
            } else {
                x[r][0] = f6::u32x4{0, 0, 0, 0};
                x[r][1] = f6::u32x4{0, 0, 0, 0};
            }
        }
    };
    // stage k of the chunk: group G0 + k / SPG, K blocks (k % SPG) QS ..
    // + QS - 1, every term: FR contiguous 1 KB fragments, wave v moving
    // fragments v, v + 4, ...
    const uint32_t n_stages = (G1 > G0 ? G1 - G0 : 0) * SPG;
    // FR / 4 pieces per wave in a loop of known trip count over a
    // wave-uniform index (a loop of unknown length leaves the compiler unable
    // to count the loads in flight)
    const uint32_t wave_s = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
    auto stage_b = [&](uint32_t k) {
        if (k < n_stages) {
            const uint32_t G = G0 + k / SPG, qb = (k % SPG) * QS;
            const auto src = packed + (((size_t)G * 32 + qb) * TERMS) * 64 + lane;
#pragma unroll
            for (uint32_t j = 0; j < FR / 4; ++j) {
                const uint32_t i = wave_s + 4 * j;
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void*)(src + (size_t)i * 64),
                    (__attribute__((address_space(3))) void*)(((k & 1) ? s_b1 : s_b0) + i * 64),
                    16, 0, 0);
            }
        }
    };
    // vmcnt(0) only: the direct-to-LDS loads and the next group's rows have landed
    auto wait_loads = [] { __builtin_amdgcn_s_waitcnt(0x0F70); };
    f6::u32x4 x[RT][2];
    if (n_stages) load_rows(G0, x);
    stage_b(0);
    wait_loads();
    __syncthreads();
    for (uint32_t G = G0; G < G1; ++G) {
        f6::u32x4 xn[RT][2];
        if (G + 1 < G1) load_rows(G + 1, xn);
#pragma unroll
        for (uint32_t st = 0; st < SPG; ++st) {
            const uint32_t k = (G - G0) * SPG + st;
            stage_b(k + 1);
            v4f acc[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[r] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t qq = 0; qq < QS; ++qq) {
                const uint32_t q = st * QS + qq;
                v8bf a[RT];
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const f6::u32x4 v = x[r][q >> 4];
                    const uint32_t sel = (q >> 2) & 3;
                    const uint32_t dw = sel == 0 ? v.x : sel == 1 ? v.y : sel == 2 ? v.z : v.w;
                    const uint32_t b8 = (dw >> (8 * (q & 3))) & 0xFFu;
                    const uint4 u = s_lut[b8];
                    __builtin_memcpy(&a[r], &u, 16);
                }
#pragma unroll
                for (int tm = 0; tm < TERMS; ++tm) {
                    const uint4 bq = ((k & 1) ? s_b1 : s_b0)[(qq * TERMS + tm) * 64 + lane];
                    v8bf bv;
                    __builtin_memcpy(&bv, &bq, 16);
#pragma unroll
                    for (int r = 0; r < RT; ++r)
                        acc[r] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], bv, acc[r], 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc64[r][i] += (double)acc[r][i];
            wait_loads();
            __syncthreads();  // stage k + 1 complete; buffer k & 1 free
        }
        if (G + 1 < G1) {
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                x[r][0] = xn[r][0];
                x[r][1] = xn[r][1];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = base + 16 * r + 4 * g + i;
            if (row < h && m < T)
                partial[((size_t)blockIdx.y * h + row) * T + m] = acc64[r][i];
        }
}

__global__ void __launch_bounds__(256) k_reduce_chunks(const double* __restrict__ partial,
                                                       uint32_t chunks, size_t n,
                                                       double* __restrict__ z) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (uint32_t c = 0; c < chunks; ++c) s += partial[(size_t)c * n + i];
    z[i] = s;
}

uint16_t bf16_rne(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    const uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(r >> 16);
}
float bf16_to_f(uint16_t b) {
    const uint32_t u = (uint32_t)b << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

}  // namespace

// ---- exact path (used by the pipeline) -------------------------------------
size_t trait_digit_elems(uint32_t traits, uint32_t w_cap) {
    const size_t ng = (w_cap + kGroupWords - 1) / kGroupWords;
    return f6::kernel_tiles(traits, f6::kMaxPlanes) * ng *
           f6::kGroupBlocks * f6::kFragVecs;
}

hipError_t launch_pack_digits(const int32_t* eff, uint32_t traits, uint32_t words, uint32_t sites,
                              uint32_t most, uint4* packed, hipStream_t s) {
    const uint32_t blocks = f6::pack_blocks(traits, f6::digit_planes(most), words);
    hipLaunchKernelGGL(k_pack_digits_of, dim3(blocks), dim3(256), 0, s, eff, traits, words, sites,
                       most, packed);
    return hipGetLastError();
}

size_t trait_piece_elems(uint32_t traits, uint32_t block_rows, uint32_t h, uint32_t w_cap,
                         uint32_t round) {
    // a launch cuts fewer than `round` row blocks into units, and no more
    // blocks than units write pieces
    const uint64_t ng = std::max<uint32_t>(1, (w_cap + kGroupWords - 1) / kGroupWords);
    const uint64_t rb = std::min<uint64_t>(round, (h + block_rows - 1) / block_rows);
    return f6::piece_elems(traits, block_rows,
                           (uint32_t)std::min<uint64_t>(round, std::max<uint64_t>(1, rb * ng)));
}

namespace {
// The contraction takes at most 16 traits: classes 0-3.
typedef void (*ExactKernel)(const uint64_t*, uint32_t, uint32_t, uint32_t, uint32_t, const uint4*, int64_t*,
                            int64_t*, uint32_t);
typedef void (*RowsKernel)(const uint64_t*, uint32_t, uint32_t, uint32_t, uint32_t, const uint4*, int64_t*);
ExactKernel exact_kernel(int cls) {
    const ExactKernel kernels[4] = {k_traits_exact<0>, k_traits_exact<1>, k_traits_exact<2>,
                                    k_traits_exact<3>};
    return kernels[cls];
}
RowsKernel rows_kernel(int cls, uint32_t row_tiles) {
    const RowsKernel one[4] = {k_traits_rows<1, 0>, k_traits_rows<1, 1>, k_traits_rows<1, 2>,
                               k_traits_rows<1, 3>};
    const RowsKernel two[4] = {k_traits_rows<2, 0>, k_traits_rows<2, 1>, k_traits_rows<2, 2>,
                               k_traits_rows<2, 3>};
    return row_tiles == 1 ? one[cls] : two[cls];
}

// The launch over h rows of ng groups and nt column tiles: row tiles per wave, or 0 and
// the blocks of the balanced launch; the least expected time past the launch itself, in us.  A launch of one row block per block takes its groups' latency
// or the rows of its fullest compute unit, whichever is longer: small blocks
// reach every compute unit and have the shorter latency, larger ones read each
// fragment from LDS for more rows.  The balanced launch divides rows evenly
// and pays for its pieces, their sums and a second launch.  Constants fitted to
// launches of 1 to 16 traits, 500 to 65,536 sites and 500 to 200,000 rows, of which
// the rule takes the fastest form or one within 3%, with few exceptions.  Measured,
// int8 kernel of a fixed 64 to 256 rows per block (which this path replaced)
// against one / two row tiles / balanced, whole calls in us: 3,000 rows x
// 1,024 sites x 8 traits: 12.8 against 10.2 / 11.3 / -; 20,000 x 5,120 x 8: 19.1
// against 16.3 / 16.3 / -; 80,000 x 2,048 x 5: 20.0 against 16.8 / 16.0 / -;
// 200,000 x 1,024 x 8: 24.9 against 25.7 / 23.3 / -; 8,000 x 20,000 x 16: 99.9 against
// 48.5 / 57.7 / 37.8; 200,000 x 65,536 x 16: 816 against 1103 / 808 / 675.
// One column tile is bound by memory, and row blocks for most of a round reach its
// rate without being cut: a balanced launch of as many blocks has no pieces
// (200,000 x 12,288 x 2: 72 us, cut 77).
struct ExactShape {
    uint32_t tiles, blocks;
};
ExactShape exact_shape(uint32_t h, uint32_t ng, uint32_t nt, uint32_t traits, const ExactRound& round) {
    const auto rows = [&](uint32_t tiles, double latency, double per_row) {
        const uint32_t block = 64 * tiles, blocks = (h + block - 1) / block;
        const uint32_t most = (blocks + round.cus - 1) / round.cus * block;  // of one compute unit
        return ng * std::max(latency, most * per_row);
    };
    const double one = rows(1, 0.45 + 0.19 * nt, 5.0e-3 + 2.2e-3 * nt);
    const double two = rows(2, 0.50 + 0.24 * nt, 5.0e-3 + 1.4e-3 * nt);
    const uint32_t direct = one <= two ? 1 : 2;
    if (h >> 30) return {0, round.blocks};  // a grid of fewer than 2^32 threads
    if (ng <= 8) return {direct, 0};        // the balanced launch's own cost is as long
    const f6::Balance bal(h, f6::balanced_block_rows(f6::trait_class(traits)), round.blocks);
    const double even = (double)ng * h / round.cus * (5.0e-3 + 1.3e-3 * nt);
    const double pieces = bal.R ? 7.0 + 0.8 / 512 * traits * bal.sharing(ng) : 0.0;
    if (even + pieces >= std::min(one, two)) return {direct, 0};
    if (nt == 1 && bal.RB <= bal.B && 4 * bal.RB >= 3 * bal.B && 0.05 * even < pieces)
        return {0, bal.RB};
    return {0, bal.B};
}
}  // namespace

uint32_t exact_block_rows(uint32_t traits) { return f6::balanced_block_rows(f6::trait_class(traits)); }

ExactRound exact_round(uint32_t traits) {
    int device = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void*>(exact_kernel(f6::trait_class(traits))), 256, 0) !=
            hipSuccess)
        return {};
    const uint32_t n = (uint32_t)std::max(1, cus);
    return {n * (uint32_t)std::max(1, per_cu), n};
}

hipError_t launch_traits_exact(const uint64_t* rows, uint32_t h, uint32_t words, uint32_t most,
                               uint32_t traits, const uint4* packed, int64_t* out, int64_t* part,
                               const ExactRound& round, hipStream_t s) {
    const int cls = f6::trait_class(traits);
    const uint32_t ng = (words + kGroupWords - 1) / kGroupWords;
    const uint32_t nt = f6::kernel_tiles(traits, f6::digit_planes(most));
    const ExactShape shape = exact_shape(h, ng, nt, traits, round);
    if (shape.tiles) {
        const uint32_t block_rows = 64 * shape.tiles;
        hipLaunchKernelGGL(rows_kernel(cls, shape.tiles), dim3((h + block_rows - 1) / block_rows),
                           dim3(256), 0, s, rows, h, words, most, traits, packed, out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(exact_kernel(cls), dim3(shape.blocks), dim3(256), 0, s, rows, h, words, most,
                       traits, packed, out, part, shape.blocks);
    hipError_t e = hipGetLastError();
    const uint32_t block_rows = f6::balanced_block_rows(cls);
    const f6::Balance bal(h, block_rows, shape.blocks);
    if (e != hipSuccess || !bal.R) return e;
    const uint64_t n = (uint64_t)(h - bal.full * bal.B * block_rows) * traits;
    hipLaunchKernelGGL(k_exact_reduce, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, h, words,
                       traits, bal.B, part, out);
    return hipGetLastError();
}

// ---- split-BF16 path (standalone contraction) -----------------------------
// The packed effects cover whole 16-word groups of the padded row width
// (sites >= `sites` are 0): packed[((G * 32 + q) * terms + term) * 64 + lane]
// = 8 BF16 of column lane % 16 (trait) at sites bf_site(G, q, lane / 16, i).
size_t mfma_effect_elems(uint32_t words, int terms) {
    const size_t ng = (words + 15) / 16;
    return ng * 32 * (size_t)terms * 64 * 8;  // bf16 elements
}

void mfma_pack_effects(const double* effects, uint32_t sites, uint32_t traits, uint32_t words,
                       int terms, uint16_t* packed) {
    const uint32_t ng = (words + 15) / 16;
    for (uint32_t G = 0; G < ng; ++G)
        for (uint32_t q = 0; q < 32; ++q)
            for (uint32_t lane = 0; lane < 64; ++lane) {
                const uint32_t n = lane & 15, g = lane >> 4;
                for (uint32_t i = 0; i < 8; ++i) {
                    const size_t site = bf_site(G, q, g, i);
                    double x = (site < sites && n < traits) ? effects[site * traits + n] : 0.0;
                    for (int tm = 0; tm < terms; ++tm) {
                        const uint16_t hb = bf16_rne((float)x);
                        packed[((((size_t)G * 32 + q) * terms + tm) * 64 + lane) * 8 + i] = hb;
                        x -= (double)bf16_to_f(hb);
                    }
                }
            }
}

size_t mfma_partial_elems(uint32_t h, uint32_t w, uint32_t traits) {
    const size_t chunks = ((w + 15) / 16 + kChunkGroups - 1) / kChunkGroups;
    return chunks * h * traits;
}

hipError_t launch_traits_mfma(const uint64_t* rows, uint32_t h, uint32_t w,
                              const uint16_t* packed, uint32_t sites, uint32_t traits, int terms,
                              double* partial, double* z, hipStream_t s) {
    (void)sites;
    const uint32_t chunks = ((w + 15) / 16 + kChunkGroups - 1) / kChunkGroups;
    const dim3 grid((h + 4 * 64 - 1) / (4 * 64), chunks);
    const uint4* pk = reinterpret_cast<const uint4*>(packed);
    if (terms == 1)
        hipLaunchKernelGGL((k_traits_bf16<4, 1>), grid, dim3(256), 0, s, rows, h, w, traits, pk,
                           partial);
    else if (terms == 2)
        hipLaunchKernelGGL((k_traits_bf16<4, 2>), grid, dim3(256), 0, s, rows, h, w, traits, pk,
                           partial);
    else
        hipLaunchKernelGGL((k_traits_bf16<4, 3>), grid, dim3(256), 0, s, rows, h, w, traits, pk,
                           partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t n = (size_t)h * traits;
    hipLaunchKernelGGL(k_reduce_chunks, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s,
                       partial, chunks, n, z);
    return hipGetLastError();
}

}  // namespace clotho
