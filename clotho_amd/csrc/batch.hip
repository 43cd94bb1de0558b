// batch.hip — replicate batches: R independent populations advanced together.
//
// Each replicate is an ordinary context (own buffers, GenState and Philox
// streams keyed by its replicate number).  A batched generation launches every
// kernel of the generation once for all replicates (pipeline.hip,
// launch_batch_generation): the kernels read each replicate's Params and
// Buffers from a device array and walk per-kernel block-offset tables, so
// replicates of uneven size share one persistent grid.  All replicates of a
// batch advance in lockstep (same parent/child parity).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "pipeline.hpp"

using namespace clotho;

struct clotho_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<clotho_ctx*> reps;
    std::vector<RepView> host_views;  // last uploaded copy
    RepView* d_views = nullptr;
    uint32_t* d_offs = nullptr;
    uint32_t* d_live_offs = nullptr;  // [kLiveKinds][R + 1], written on the device each generation
    BatchLaunch L;
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    int cur = 0;
    Timing timing;
    std::string err;
};

namespace {

#define BATCH_TRY(b, expr)                                                   \
    do {                                                                     \
        const hipError_t e_ = (expr);                                        \
        if (e_ != hipSuccess) {                                              \
            (b)->err = std::string(#expr) + ": " + hipGetErrorString(e_);   \
            return CLOTHO_ERR_HIP;                                           \
        }                                                                    \
    } while (0)

void drop_graphs(clotho_batch* b) {
    for (hipGraphExec_t& g : b->exec)
        if (g) {
            (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
}

// Launch shape of a replicate's recombination within a batch of `groups` groups
// of 64 gametes: chunks of 16 groups (a block's offset search, tables and
// partials are paid per chunk; half and twice as many chunks measured 1.12 and
// 1.20 ms on the 256-replicate workload at generation 200; eight groups in a batch of
// 26,000 by event 234 us, 16 210).  A replicate that may recombine by groups takes
// fewer where that would not give every resident block four chunks (64 x 6,000, 392
// words, rho = 5: 2334 us, with 16 2699), and column ranges where the chunks alone
// do not give it one.  Row chunks that were set or tuned for a
// replicate are taken for it, two per block.  rho: events per gamete, filled: the
// part of the rows' column tiles of 64 words that they fill, over all rows.
void batch_recombine_shape(Params& P, bool chunks_set, uint64_t groups, double rho, double filled,
                           uint32_t resident) {
    if (groups <= (uint64_t)kGroupBatch * resident)
        P.group_words = 0;
    else if (rho <= (filled < kEventFill ? kEventRho : kWideEventRho))
        P.group_words = kNeverPerGroup;
    else
        P.group_words = groups <= (uint64_t)kSmallBatch * resident ? 0 : kWidePerGroup;
    const uint32_t own = (P.h + 63) / 64;
    const uint64_t fill = std::min<uint64_t>(16, std::max<uint64_t>(1, groups / (4ull * resident)));
    const uint64_t per = P.w_cap > P.group_words ? fill : 16;
    P.chunks = std::min<uint32_t>(
        P.max_chunks, chunks_set ? (P.chunks + 1) / 2 : (uint32_t)((own + per - 1) / per));
    const uint64_t turns = (P.w_cap + 63) / 64;
    P.splits = (uint32_t)std::max<uint64_t>(1, std::min(turns, resident / std::max<uint64_t>(1, groups)));
}

// Upload each replicate's Params/Buffers and the per-kernel block offsets
// when they changed (a replicate's launch shape may have been retuned).
int sync_views(clotho_batch* b) {
    const uint32_t R = (uint32_t)b->reps.size();
    std::vector<RepView> v(R);
    uint64_t groups = 0;
    double rho = 0.0, words = 0.0, tiles = 0.0;
    for (const clotho_ctx* c : b->reps) {
        const uint32_t own = (c->p.h + 63) / 64;
        groups += own;
        rho += own * c->cfg.rho;
        words += (double)own * c->live_words;
        tiles += (double)own * (64 * ((c->live_words + 63) / 64));
    }
    rho /= (double)groups;
    const double filled = tiles > 0.0 ? words / tiles : 0.0;
    const uint32_t resident = b->reps[0]->recombine_round;
    for (uint32_t r = 0; r < R; ++r) {
        std::memset(&v[r], 0, sizeof(RepView));
        v[r].P = b->reps[r]->p;
        v[r].B = b->reps[r]->b;
        v[r].B.by_parent = nullptr;  // replicates recombine in child order
        v[r].B.trait_part = nullptr;  // and sum their traits in whole row blocks
        batch_recombine_shape(v[r].P, b->reps[r]->chunks_set, groups, rho, filled,
                              resident);
        // a replicate with many chunks has its partials folded as in a single population
        v[r].P.free_words = v[r].P.chunks > 64 ? 16 : 64;
        v[r].P.word_blocks = (v[r].P.w_cap + v[r].P.free_words - 1) / v[r].P.free_words;
    }
    if (b->d_views && b->host_views.size() == R &&
        std::memcmp(v.data(), b->host_views.data(), sizeof(RepView) * R) == 0)
        return CLOTHO_OK;
    drop_graphs(b);
    std::vector<uint32_t> offs((size_t)kOpCount * (R + 1), 0);
    for (uint32_t r = 0; r < R; ++r) {
        uint32_t blocks[kOpCount];
        batch_op_blocks(v[r].P, blocks);
        for (int k = 0; k < kOpCount; ++k)
            offs[(size_t)k * (R + 1) + r + 1] = offs[(size_t)k * (R + 1) + r] + blocks[k];
    }
    if (!b->d_views) {
        BATCH_TRY(b, hipMalloc((void**)&b->d_views, sizeof(RepView) * R));
        BATCH_TRY(b, hipMalloc((void**)&b->d_offs, sizeof(uint32_t) * offs.size()));
        BATCH_TRY(b, hipMalloc((void**)&b->d_live_offs, sizeof(uint32_t) * kLiveKinds * (R + 1)));
    }
    BATCH_TRY(b, hipMemcpy(b->d_views, v.data(), sizeof(RepView) * R, hipMemcpyHostToDevice));
    BATCH_TRY(b, hipMemcpy(b->d_offs, offs.data(), sizeof(uint32_t) * offs.size(),
                           hipMemcpyHostToDevice));
    b->host_views = v;
    BatchLaunch& L = b->L;
    L.views = b->d_views;
    L.offs = b->d_offs;
    L.live_offs = b->d_live_offs;
    L.R = R;
    for (int k = 0; k < kOpCount; ++k) L.total[k] = offs[(size_t)k * (R + 1) + R];
    L.traits = v[0].P.traits;
    L.by_group = L.by_event = false;
    for (const RepView& x : v) {
        L.by_group = L.by_group || x.P.w_cap > x.P.group_words;
        L.by_event = L.by_event || x.P.group_words;
    }
    L.wide_events = false;
    for (const RepView& x : v) L.wide_events = L.wide_events || x.P.ev_cap > 64;
    L.cus = (uint32_t)std::max(1, b->reps[0]->prop.multiProcessorCount);
    return CLOTHO_OK;
}

int capture_batch(clotho_batch* b) {
    for (int k = 0; k < 2; ++k) {
        if (b->exec[k]) continue;
        hipGraph_t g = nullptr;
        BATCH_TRY(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        const hipError_t e1 = launch_batch_generation(b->L, (uint32_t)k, b->stream, nullptr);
        const hipError_t e2 = hipStreamEndCapture(b->stream, &g);
        if (e1 != hipSuccess || e2 != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            b->err = std::string("batch capture: ") +
                     hipGetErrorString(e1 != hipSuccess ? e1 : e2);
            return CLOTHO_ERR_HIP;
        }
        const hipError_t e3 = hipGraphInstantiate(&b->exec[k], g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e3 != hipSuccess) {
            b->err = std::string("batch instantiate: ") + hipGetErrorString(e3);
            return CLOTHO_ERR_HIP;
        }
    }
    return CLOTHO_OK;
}

// The views and, where the mode replays them, the captured launches, at the
// replicates' widths when last looked at (replicates one by one, 256 of 8-72 words:
// 19.8 -> 17.8 ms per generation against the shapes for their capacity).
int ready_launches(clotho_batch* b, int mode) {
    int rc = sync_views(b);
    if (rc == CLOTHO_OK && mode == CLOTHO_BATCH_GRAPH) rc = capture_batch(b);
    if (rc != CLOTHO_OK || mode != CLOTHO_BATCH_SEQUENTIAL) return rc;
    for (clotho_ctx* c : b->reps) {
        if (refresh_shapes(c)) destroy_graphs(c);
        rc = capture_graphs(c);
        if (rc != CLOTHO_OK) {
            b->err = "replicate graph: " + c->err;
            return rc;
        }
    }
    return CLOTHO_OK;
}

}  // namespace

extern "C" {

int clotho_batch_create(const clotho_config* cfgs, uint32_t count, int device,
                        clotho_batch** out) {
    if (!cfgs || !out || count == 0) return CLOTHO_ERR_ARG;
    *out = nullptr;
    for (uint32_t r = 0; r < count; ++r)
        if (cfgs[r].trait_count != cfgs[0].trait_count || cfgs[r].compact_every)
            return CLOTHO_ERR_ARG;
    clotho_batch* b = new (std::nothrow) clotho_batch();
    if (!b) return CLOTHO_ERR_ARG;
    b->device = device;
    auto bail = [&](int rc) {
        clotho_batch_destroy(b);
        return rc;
    };
    if (hipSetDevice(device) != hipSuccess) return bail(CLOTHO_ERR_HIP);
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(CLOTHO_ERR_HIP);
    for (uint32_t r = 0; r < count; ++r) {
        clotho_ctx* c = nullptr;
        const int rc = create_context(&cfgs[r], device, true, &c);
        if (rc != CLOTHO_OK) return bail(rc);
        b->reps.push_back(c);
    }
    const int rc = sync_views(b);
    if (rc != CLOTHO_OK) return bail(rc);
    *out = b;
    return CLOTHO_OK;
}

void clotho_batch_destroy(clotho_batch* b) {
    if (!b) return;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    drop_graphs(b);
    if (b->d_views) (void)hipFree(b->d_views);
    if (b->d_offs) (void)hipFree(b->d_offs);
    if (b->d_live_offs) (void)hipFree(b->d_live_offs);
    for (clotho_ctx* c : b->reps) clotho_destroy(c);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

const char* clotho_batch_last_error(const clotho_batch* b) { return b ? b->err.c_str() : ""; }

uint32_t clotho_batch_size(const clotho_batch* b) { return b ? (uint32_t)b->reps.size() : 0u; }

clotho_ctx* clotho_batch_replicate(clotho_batch* b, uint32_t r) {
    return (b && r < b->reps.size()) ? b->reps[r] : nullptr;
}

int clotho_batch_autotune(clotho_batch* b, uint32_t* percent) {
    if (!b) return CLOTHO_ERR_ARG;
    BATCH_TRY(b, hipSetDevice(b->device));
    for (clotho_ctx* c : b->reps) BATCH_TRY(b, hipStreamSynchronize(c->stream));
    int rc = sync_views(b);
    if (rc != CLOTHO_OK) return rc;
    const uint32_t par = (uint32_t)b->cur;
    const uint32_t nums[3] = {1, 1, 2}, dens[3] = {2, 1, 1};
    EventSet events;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    BATCH_TRY(b, events.add(&e0));
    BATCH_TRY(b, events.add(&e1));
    float best[3] = {1e30f, 1e30f, 1e30f};
    for (int pass = 0; pass < 2; ++pass)
        for (int i = 0; i < 3; ++i) {
            b->L.grid_scale_num = nums[i];
            b->L.grid_scale_den = dens[i];
            BATCH_TRY(b, launch_batch_replay(b->L, par, b->stream));  // warm-up
            BATCH_TRY(b, hipEventRecord(e0, b->stream));
            for (int r = 0; r < 3; ++r) BATCH_TRY(b, launch_batch_replay(b->L, par, b->stream));
            BATCH_TRY(b, hipEventRecord(e1, b->stream));
            BATCH_TRY(b, hipEventSynchronize(e1));
            float ms = 0.f;
            BATCH_TRY(b, hipEventElapsedTime(&ms, e0, e1));
            best[i] = std::min(best[i], ms);
        }
    int bi = 1;
    for (int i = 0; i < 3; ++i)
        if (best[i] < best[bi]) bi = i;
    b->L.grid_scale_num = nums[bi];
    b->L.grid_scale_den = dens[bi];
    drop_graphs(b);  // captured launches bake the grid in
    if (percent) *percent = 100u * nums[bi] / dens[bi];
    return CLOTHO_OK;
}

void clotho_batch_set_timing(clotho_batch* b, int enabled) {
    if (b) b->timing.enabled = enabled != 0;
}

int clotho_batch_timings(clotho_batch* b, double* ms, int cap) {
    if (!b || !ms) return CLOTHO_ERR_ARG;
    for (int i = 0; i < cap && i < 6; ++i) ms[i] = b->timing.ms[i];
    return b->timing.generations;
}

int clotho_batch_run(clotho_batch* b, uint32_t n, int mode, double* elapsed_ms) {
    if (!b) return CLOTHO_ERR_ARG;
    if (mode < CLOTHO_BATCH_GRAPH || mode > CLOTHO_BATCH_SEQUENTIAL) {
        b->err = "batch_run: unknown mode";
        return CLOTHO_ERR_ARG;
    }
    BATCH_TRY(b, hipSetDevice(b->device));
    for (clotho_ctx* c : b->reps) {
        if (c->cur != b->cur) {
            b->err = "batch_run: a replicate was advanced outside the batch";
            return CLOTHO_ERR_STATE;
        }
        if ((c->next_n && c->next_n != c->p.n) || c->p.n_par != c->p.n) {
            b->err = "batch_run: replicate population sizes are fixed inside a batch";
            return CLOTHO_ERR_ARG;
        }
        BATCH_TRY(b, hipStreamSynchronize(c->stream));  // uploads done
    }
    int rc = ready_launches(b, mode);
    if (rc != CLOTHO_OK) return rc;
    Timing& tm = b->timing;
    for (double& v : tm.ms) v = 0.0;
    tm.generations = 0;
    const bool phase_timing = tm.enabled && mode == CLOTHO_BATCH_EAGER;
    std::vector<std::vector<hipEvent_t>> marks;
    EventSet events;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    BATCH_TRY(b, events.add(&e0));
    BATCH_TRY(b, events.add(&e1));
    BATCH_TRY(b, hipEventRecord(e0, b->stream));
    for (uint32_t g = 0; g < n; ++g) {
        const uint32_t par = (uint32_t)b->cur;
        // Batched launches keep their shapes within a run: reading 256 replicates' widths
        // takes as long as eight generations of 3,000 individuals.
        if (mode == CLOTHO_BATCH_SEQUENTIAL && width_due(g)) {
            BATCH_TRY(b, hipStreamSynchronize(b->stream));
            for (clotho_ctx* c : b->reps) {
                GenState seen;
                if ((rc = read_state(c, &seen)) != CLOTHO_OK) {
                    b->err = c->err;
                    return rc;
                }
            }
            if ((rc = ready_launches(b, mode)) != CLOTHO_OK) return rc;
        }
        if (mode == CLOTHO_BATCH_GRAPH) {
            BATCH_TRY(b, hipGraphLaunch(b->exec[par], b->stream));
        } else if (mode == CLOTHO_BATCH_EAGER) {
            hipEvent_t* mk = nullptr;
            if (phase_timing) {
                marks.emplace_back(6);
                for (hipEvent_t& e : marks.back()) BATCH_TRY(b, events.add(&e));
                mk = marks.back().data();
            }
            BATCH_TRY(b, launch_batch_generation(b->L, par, b->stream, mk));
        } else {
            for (clotho_ctx* c : b->reps) BATCH_TRY(b, hipGraphLaunch(c->graphs.exec[par], b->stream));
        }
        b->cur = 1 - b->cur;
        for (clotho_ctx* c : b->reps) c->cur = b->cur;
    }
    BATCH_TRY(b, hipEventRecord(e1, b->stream));
    BATCH_TRY(b, hipEventSynchronize(e1));
    float ms = 0.f;
    BATCH_TRY(b, hipEventElapsedTime(&ms, e0, e1));
    if (elapsed_ms) *elapsed_ms = ms;
    if (phase_timing) {
        for (auto& mk : marks) {
            float t = 0.f;
            BATCH_TRY(b, hipEventElapsedTime(&t, mk[0], mk[5]));
            tm.ms[0] += t;
            for (int q = 0; q < 5; ++q) {
                BATCH_TRY(b, hipEventElapsedTime(&t, mk[q], mk[q + 1]));
                tm.ms[1 + q] += t;
            }
        }
        tm.generations = (int)n;
    }
    for (uint32_t r = 0; r < b->reps.size(); ++r) {
        clotho_ctx* c = b->reps[r];
        GenState st;
        rc = read_state(c, &st);
        if (rc != CLOTHO_OK) {
            b->err = c->err;
            return rc;
        }
        c->has_population = true;
        if (st.error) {
            b->err = "replicate " + std::to_string(r) + ": allele capacity exceeded at generation " +
                     std::to_string(st.error_gen);
            return CLOTHO_ERR_CAPACITY;
        }
    }
    return CLOTHO_OK;
}

}  // extern "C"
