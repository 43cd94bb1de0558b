// traits_noalloc.hip — the exact trait contraction for callers that cannot
// allocate device memory (code under HIP graph capture, serving loops,
// harnesses that forbid hipMalloc).  No counterpart in the reference.
//
// The effect digit planes the exact MFMA path multiplies by and the partial
// sums of the row blocks it cuts along the sites live in `scratch`, a file-scope
// device array of fixed size.  Each GPU holds its own copy until the process
// ends; host code reaches it only through the address hipGetSymbolAddress
// returns for the current device (the array's name on the host is a stand-in,
// not a device address).  Every call on one GPU shares that GPU's array: calls
// that overlap on one GPU race, and a call overwrites everything of the
// previous call that it reads (every plane it multiplies by and every piece it
// sums), so nothing needs to be cleared between calls.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/clotho_amd.h"
#include "pipeline.hpp"
#include "traits.hpp"
#include "traits_f6.hpp"

namespace clotho {
namespace {

constexpr size_t kPlanesBytes =
    (size_t)f6::kernel_tiles(CLOTHO_NOALLOC_MAX_TRAITS, f6::kMaxPlanes) *
    (CLOTHO_NOALLOC_MAX_SITES / 64 / f6::kGroupWords) * f6::kGroupBlocks * f6::kFragVecs *
    sizeof(uint4);
// pieces of the row blocks a launch cuts along K (512 blocks at 16 traits)
constexpr size_t kPiecesBytes = (size_t)33554432;
constexpr size_t kScratchBytes = kPlanesBytes + kPiecesBytes;
static_assert(kScratchBytes == CLOTHO_NOALLOC_SCRATCH_BYTES, "scratch size as declared");

__device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_lock;
struct DeviceEntry {
    uint8_t* scratch = nullptr;
    ExactRound round[f6::kClasses];  // of each trait class's kernel
};
DeviceEntry g_devices[kMaxDevices];

// the device address of `scratch` on `device` (current) and the resident
// round of the kernel for `traits`, each looked up once
int entry_of(int device, uint32_t traits, uint8_t** out, ExactRound* round) {
    std::lock_guard<std::mutex> guard(g_lock);
    DeviceEntry& e = g_devices[device];
    if (!e.scratch) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
            return CLOTHO_ERR_HIP;
        e.scratch = static_cast<uint8_t*>(p);
    }
    ExactRound& r = e.round[f6::trait_class(traits)];
    if (!r.blocks) r = exact_round(traits);
    if (!r.blocks) return CLOTHO_ERR_HIP;
    *out = e.scratch;
    *round = r;
    return CLOTHO_OK;
}

}  // namespace
}  // namespace clotho

using namespace clotho;

extern "C" int clotho_trait_contract_exact_noalloc(const uint64_t* rows, uint32_t haplotypes,
                                                   uint32_t words, const int32_t* effects,
                                                   uint32_t sites, uint32_t traits, int64_t* sums,
                                                   void* stream) {
    if (traits == 0 || words == 0 || words % 8 || (size_t)words * 64 < sites)
        return CLOTHO_ERR_ARG;
    if (traits > CLOTHO_NOALLOC_MAX_TRAITS || (size_t)words * 64 > CLOTHO_NOALLOC_MAX_SITES)
        return CLOTHO_ERR_CAPACITY;
    if (haplotypes == 0) return CLOTHO_OK;
    if (!rows || !sums || (sites && !effects)) return CLOTHO_ERR_ARG;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices)
        return CLOTHO_ERR_HIP;
    uint8_t* base = nullptr;
    ExactRound round;
    const int rc = entry_of(device, traits, &base, &round);
    if (rc != CLOTHO_OK) return rc;
    const size_t fit = kPiecesBytes / (sizeof(int64_t) * f6::piece_elems(traits, f6::balanced_block_rows(f6::trait_class(traits)), 1));
    if (round.blocks > fit) round.blocks = (uint32_t)fit;
    uint4* planes = reinterpret_cast<uint4*>(base);
    int64_t* pieces = reinterpret_cast<int64_t*>(base + kPlanesBytes);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    // the effects are not read before they are packed: their bound is the API's
    const uint32_t most = (uint32_t)kEffectLimit;
    if (launch_pack_digits(effects, traits, words, sites, most, planes, s) != hipSuccess)
        return CLOTHO_ERR_HIP;
    if (launch_traits_exact(rows, haplotypes, words, most, traits, planes, sums, pieces, round, s) !=
        hipSuccess)
        return CLOTHO_ERR_HIP;
    return CLOTHO_OK;
}
