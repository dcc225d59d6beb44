// ftdx_grouped.cpp -- grouped HERK over many problems of uneven N and K in one
// persistent launch (optionally replayed from a captured hipGraph).
//
// The reference runs one uniform (N, K, batch) HERK per call
// (cutlass_interface/cutlass_gemm_api.cu:1707-1878); its callers loop over
// sub-arrays.  Here a plan holds, in device memory, the problem descriptors and
// a static schedule: every lower-triangle tile of every problem is one item;
// items are sorted by cost (K rounded to the stage, less for diagonal tiles)
// and assigned longest-first to the least-loaded persistent workgroup.  Ties go
// to workgroups of the same XCD first, so items that share input rows run on
// one XCD and meet in its L2.
//
// Problems whose rows 16-byte loads cannot take (K % 16 != 0, or A not 16-byte aligned)
// are run on zero-padded copies of their rows (K rounded up to 16) in a buffer the plan
// owns, refreshed by one pad launch before the HERK launch on every run (captured in the
// same graph), so the HERK kernel is built with the 16-byte load path only.  If that
// buffer cannot be allocated, the plan runs the kernel that holds both load paths.
//
// A plan of no stated tile configuration may run the pipelined kernel instead: every run
// converts the problems' rows (any K and alignment) to E3M2 fragment rows in a buffer of
// the plan, then multiplies from there, one launch each.  No two problems share rows, so
// runs of one plan on two streams only write the same bytes twice.  The tiles, problems by
// descending K, are split over the XCDs in eight runs of equal cost, so that one XCD's L2
// serves the tiles of few problems; inside a run the hardware hands out tiles as workgroups
// finish.  512 problems of N, K up to 4096: 9.50 ms (persistent, 256 x 128 tiles) to 7.01;
// in chunks of 160, 320 and 640 MB of rows that stay in the memory-side cache: 7.07, 7.16
// and 7.02, so the rows go in one piece.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

#include "ftdx.h"
#include "ftdx_host.h"
#include "ftdx_internal.h"
#include "herk_fp8.h"
#include "herk_pipe.h"
#include "stages.h"

struct ftdx_grouped_plan {
    int device = 0;
    int cfg = 0;
    int out_fp16 = 0;
    int num_wg = 0;
    int count = 0;
    bool all_vec = false;  // every problem takes 16-byte loads
    int64_t items = 0;
    double max_load = 0, mean_load = 0;
    ftdx::GroupProblemDev* d_probs = nullptr;
    ftdx::GroupItemDev* d_items = nullptr;
    int* d_wg_begin = nullptr;
    uint8_t* d_pad = nullptr;             // padded rows of the problems that need them
    ftdx::PadRowsJob* d_pad_jobs = nullptr;
    ftdx::PadBlock* d_pad_blocks = nullptr;
    int pad_blocks = 0;
    uint8_t* d_rows = nullptr;  // fragment rows of the pipelined kernel; none: not used
    ftdx::PipeProblem* d_pipe = nullptr;
    ftdx::ConvBlock* d_conv = nullptr;
    ftdx::GroupItemDev* d_tiles = nullptr;
    int conv_blocks = 0;
    bool use_graph = false;
    hipStream_t cap_stream = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace ftdx {

namespace {

int stage_samples(int cfg) { return cfg == TILE_128x128_K128 ? 128 : 64; }

}  // namespace

int grouped_build(ftdx_grouped_plan* P, const ftdx_herk_problem* problems, int count, int cfg,
                  int out_fp16, int cu_count) {
    std::vector<int> Ns(count), Ks(count);
    for (int p = 0; p < count; ++p) {
        Ns[p] = problems[p].N;
        Ks[p] = problems[p].K;
    }
    GroupSchedule sch;
    const int rc = build_group_schedule(Ns.data(), Ks.data(), count, tile_config_rows(cfg), tile_config_cols(cfg),
                                        stage_samples(cfg), tile_config_wg_per_cu(cfg), cu_count, sch);
    if (rc == -2) return fail(FTDX_ERR_INVALID_ARG, "grouped: too many tiles");
    if (rc != 0) return fail(FTDX_ERR_INVALID_ARG, "grouped: invalid problem list");
    std::vector<GroupProblemDev> probs(count);
    bool all_vec = true;
    size_t pad_bytes = 0;
    for (int p = 0; p < count; ++p) {
        const ftdx_herk_problem& q = problems[p];
        GroupProblemDev& d = probs[p];
        d.A = static_cast<const uint8_t*>(q.A);
        d.C = q.C;
        d.N = q.N;
        d.K = q.K;
        d.alpha = q.alpha;
        d.beta = q.beta;
        // (N = 0 or K = 0: no loads at all)
        d.vec = q.N <= 0 || q.K <= 0 || ((q.K % 16 == 0) && ((reinterpret_cast<uintptr_t>(q.A) & 15u) == 0));
        d.tiles = sch.tiles[p];
        all_vec = all_vec && d.vec;
        if (!d.vec) pad_bytes += (size_t)q.N * precast_row_samples(q.K);
    }
    hipError_t e;
    if (pad_bytes > 0 && hipMalloc(&P->d_pad, pad_bytes) == hipSuccess) {
        // every problem that needs it reads its padded copy; the plan then takes 16-byte loads only
        std::vector<PadRowsJob> jobs;
        std::vector<PadBlock> blocks;
        size_t off = 0;
        for (int p = 0; p < count; ++p) {
            GroupProblemDev& d = probs[p];
            if (d.vec) continue;
            const int Kq = precast_row_samples(d.K);
            const int64_t segs = (int64_t)d.N * (Kq / 16);
            for (int64_t g = 0; g < segs; g += kPadBlockSegments) blocks.push_back({(int)jobs.size(), g});
            jobs.push_back({d.A, P->d_pad + off, (int64_t)d.N, d.K, Kq});
            d.A = P->d_pad + off;
            d.K = Kq;
            d.vec = 1;
            off += (size_t)d.N * Kq;
        }
        if ((e = hipMalloc(&P->d_pad_jobs, sizeof(PadRowsJob) * jobs.size())) != hipSuccess)
            return hip_fail(e, "grouped plan: hipMalloc");
        if ((e = hipMemcpy(P->d_pad_jobs, jobs.data(), sizeof(PadRowsJob) * jobs.size(),
                           hipMemcpyHostToDevice)) != hipSuccess)
            return hip_fail(e, "grouped plan: upload");
        if (blocks.size() > 0x7FFFFFFF) return fail(FTDX_ERR_INVALID_ARG, "grouped plan: too many rows to pad");
        if ((e = hipMalloc(&P->d_pad_blocks, sizeof(PadBlock) * blocks.size())) != hipSuccess)
            return hip_fail(e, "grouped plan: hipMalloc");
        if ((e = hipMemcpy(P->d_pad_blocks, blocks.data(), sizeof(PadBlock) * blocks.size(),
                           hipMemcpyHostToDevice)) != hipSuccess)
            return hip_fail(e, "grouped plan: upload");
        P->pad_blocks = (int)blocks.size();
        all_vec = true;
    } else if (pad_bytes > 0) {
        (void)hipGetLastError();  // out of memory for the copies: both load paths instead
    }
    static_assert(sizeof(GroupItemDev) == sizeof(ScheduleItem), "schedule items are uploaded as they are");
    const std::vector<ScheduleItem>& flat = sch.items;
    const std::vector<int>& begin = sch.begin;
    const int G = sch.num_wg;
    P->items = (int64_t)flat.size();
    P->max_load = sch.max_load;
    P->mean_load = sch.mean_load;

    if ((e = hipMalloc(&P->d_probs, sizeof(GroupProblemDev) * std::max(count, 1))) != hipSuccess)
        return hip_fail(e, "grouped plan: hipMalloc");
    if ((e = hipMalloc(&P->d_items, sizeof(GroupItemDev) * std::max<size_t>(flat.size(), 1))) !=
        hipSuccess)
        return hip_fail(e, "grouped plan: hipMalloc");
    if ((e = hipMalloc(&P->d_wg_begin, sizeof(int) * (G + 1))) != hipSuccess)
        return hip_fail(e, "grouped plan: hipMalloc");
    if ((e = hipMemcpy(P->d_probs, probs.data(), sizeof(GroupProblemDev) * count,
                       hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "grouped plan: upload");
    if (!flat.empty() &&
        (e = hipMemcpy(P->d_items, flat.data(), sizeof(GroupItemDev) * flat.size(),
                       hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "grouped plan: upload");
    if ((e = hipMemcpy(P->d_wg_begin, begin.data(), sizeof(int) * (G + 1),
                       hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "grouped plan: upload");
    P->num_wg = G;
    P->all_vec = all_vec;
    P->cfg = cfg;
    P->out_fp16 = out_fp16;
    P->count = count;
    return FTDX_OK;
}

namespace {

// The most fragment rows a plan holds (beyond that, or half of what is free, it runs the
// persistent kernel).
constexpr size_t kGroupRowsMax = size_t(8) << 30;

template <typename T>
hipError_t upload(T** dst, const std::vector<T>& v) {
    hipError_t e = hipMalloc(dst, sizeof(T) * std::max<size_t>(v.size(), 1));
    if (e == hipSuccess && !v.empty()) e = hipMemcpy(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
    return e;
}

// Cost of a tile in 64-sample stages: its stages and the share of its stores and its start.
double pipe_cost(const PipeProblem& p) { return p.steps / 2 + 6.0; }

}  // namespace

// The plan over fragment rows.  FTDX_ERR_UNSUPPORTED: sizes or memory that it does not take (the
// caller builds the fused plan).
int grouped_build_pipe(ftdx_grouped_plan* P, const ftdx_herk_problem* problems, int count, int cfg, int out_fp16) {
    std::vector<PipeProblem> probs;
    size_t total = 0;
    int64_t items = 0;
    for (int i = 0; i < count; ++i) {
        const ftdx_herk_problem& q = problems[i];
        if (q.N <= 0) continue;
        const int kq = std::max(q.K, 16);
        if (!pipe_supported(q.N, kq)) return FTDX_ERR_UNSUPPORTED;
        PipeProblem p;
        p.A = static_cast<const uint8_t*>(q.A);
        p.rows = nullptr;
        p.C = q.C;
        p.N = q.N;
        p.K = q.K;
        p.steps = frag_steps(kq);
        p.nt = pipe_nontemporal(q.N, q.K, out_fp16 != 0);
        p.alpha = q.alpha;
        p.beta = q.beta;
        probs.push_back(p);
        total += (size_t)frag_rows_bytes(q.N, kq);
        items += pipe_tiles(q.N);
    }
    size_t free_bytes = 0, all_bytes = 0;
    if (probs.empty() || items > 0x07FFFFFF || total > kGroupRowsMax) return FTDX_ERR_UNSUPPORTED;
    if (hipMemGetInfo(&free_bytes, &all_bytes) != hipSuccess || total > free_bytes / 2 ||
        hipMalloc(&P->d_rows, total) != hipSuccess) {
        (void)hipGetLastError();
        P->d_rows = nullptr;
        return FTDX_ERR_UNSUPPORTED;
    }
    std::stable_sort(probs.begin(), probs.end(),
                     [](const PipeProblem& a, const PipeProblem& b) { return a.steps > b.steps; });
    std::vector<ConvBlock> conv;
    std::vector<GroupItemDev> run[8], tiles;
    uint8_t* at = P->d_rows;
    double cost = 0.0, done = 0.0, load[8] = {};
    for (size_t p = 0; p < probs.size(); ++p) {
        PipeProblem& q = probs[p];
        q.rows = at;
        at += (size_t)frag_groups(q.N) * q.steps * kFragBytes;
        cost += pipe_cost(q) * pipe_tiles(q.N);
        const int64_t segs = (int64_t)frag_groups(q.N) * 64 * q.steps;  // < 2^31: its rows' bytes / 24
        for (int64_t f = 0; f < segs; f += kConvThreads) conv.push_back({(int)p, (uint32_t)f});
    }
    for (size_t p = 0; p < probs.size(); ++p) {
        const double one = pipe_cost(probs[p]);
        const int n = pipe_tiles(probs[p].N);
        for (int t = 0; t < n; ++t, done += one) {
            const int x = std::min(7, (int)(8.0 * done / cost));
            run[x].push_back({(int)p, t});
            load[x] += one;
        }
    }
    size_t len = 0;
    for (const auto& r : run) len = std::max(len, r.size());
    for (size_t k = 0; k < len; ++k)
        for (const auto& r : run) tiles.push_back(k < r.size() ? r[k] : GroupItemDev{-1, 0});
    hipError_t e;
    if ((e = upload(&P->d_pipe, probs)) != hipSuccess || (e = upload(&P->d_conv, conv)) != hipSuccess ||
        (e = upload(&P->d_tiles, tiles)) != hipSuccess) {
        (void)hipGetLastError();
        return FTDX_ERR_UNSUPPORTED;
    }
    P->items = items;
    P->max_load = *std::max_element(load, load + 8);
    P->mean_load = cost / 8.0;
    P->num_wg = (int)tiles.size();  // at most 8 per item: < 2^31
    P->conv_blocks = (int)conv.size();
    P->cfg = cfg;
    P->out_fp16 = out_fp16;
    P->count = count;
    return FTDX_OK;
}

hipError_t grouped_launch(ftdx_grouped_plan* P, hipStream_t s) {
    if (P->d_rows) {
        hipError_t e = launch_qc_frag_rows_multi(P->d_pipe, P->d_conv, P->conv_blocks, s);
        if (e != hipSuccess) return e;
        return launch_herk_pipe_grouped(P->d_pipe, P->d_tiles, P->num_wg, P->out_fp16 != 0, s);
    }
    if (P->pad_blocks > 0) {
        hipError_t e = launch_pad_qc_rows_multi(P->d_pad_jobs, P->d_pad_blocks, P->pad_blocks, s);
        if (e != hipSuccess) return e;
    }
    return launch_herk_int4_grouped(P->d_probs, P->d_items, P->d_wg_begin, P->num_wg, P->cfg,
                                    P->out_fp16 != 0, P->all_vec, s);
}

void grouped_release(ftdx_grouped_plan* P) {
    if (!P) return;
    if (P->exec) (void)hipGraphExecDestroy(P->exec);
    if (P->cap_stream) (void)hipStreamDestroy(P->cap_stream);
    if (P->d_probs) (void)hipFree(P->d_probs);
    if (P->d_items) (void)hipFree(P->d_items);
    if (P->d_wg_begin) (void)hipFree(P->d_wg_begin);
    if (P->d_pad) (void)hipFree(P->d_pad);
    if (P->d_pad_jobs) (void)hipFree(P->d_pad_jobs);
    if (P->d_pad_blocks) (void)hipFree(P->d_pad_blocks);
    if (P->d_rows) (void)hipFree(P->d_rows);
    if (P->d_pipe) (void)hipFree(P->d_pipe);
    if (P->d_conv) (void)hipFree(P->d_conv);
    if (P->d_tiles) (void)hipFree(P->d_tiles);
    P->d_rows = nullptr;
    P->d_pipe = nullptr;
    P->d_conv = nullptr;
    P->d_tiles = nullptr;
    P->d_pad = nullptr;
    P->d_pad_jobs = nullptr;
    P->d_pad_blocks = nullptr;
    P->pad_blocks = 0;
    P->exec = nullptr;
    P->cap_stream = nullptr;
    P->d_probs = nullptr;
    P->d_items = nullptr;
    P->d_wg_begin = nullptr;
}

int grouped_capture(ftdx_grouped_plan* P) {
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&P->cap_stream, hipStreamNonBlocking)) != hipSuccess)
        return hip_fail(e, "grouped plan: hipStreamCreate");
    if ((e = hipStreamBeginCapture(P->cap_stream, hipStreamCaptureModeRelaxed)) != hipSuccess)
        return hip_fail(e, "grouped plan: hipStreamBeginCapture");
    hipError_t le = grouped_launch(P, P->cap_stream);
    hipGraph_t graph = nullptr;
    e = hipStreamEndCapture(P->cap_stream, &graph);
    if (le != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return hip_fail(le, "grouped plan: captured launch");
    }
    if (e != hipSuccess) return hip_fail(e, "grouped plan: hipStreamEndCapture");
    e = hipGraphInstantiate(&P->exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return hip_fail(e, "grouped plan: hipGraphInstantiate");
    P->use_graph = true;
    return FTDX_OK;
}

// Times each tile configuration's plan, and the pipelined one, on the problems' own buffers
// (outputs are overwritten: only used when every beta is 0): the fastest tile configuration,
// and whether the pipelined plan beat it.
int grouped_autotune(const ftdx_herk_problem* problems, int count, int out16, int cus, int& best, bool& pipe) {
    hipEvent_t t0, t1;
    (void)hipEventCreate(&t0);
    (void)hipEventCreate(&t1);
    float best_ms = 1e30f;
    pipe = false;
    for (int cfg = 0; cfg <= NUM_TILE_CONFIGS; ++cfg) {
        ftdx_grouped_plan P;
        const bool rows = cfg == NUM_TILE_CONFIGS;
        int rc = rows ? grouped_build_pipe(&P, problems, count, best, out16)
                      : grouped_build(&P, problems, count, cfg, out16, cus);
        if (rc != FTDX_OK) {
            grouped_release(&P);
            continue;
        }
        float ms = 1e30f;
        if (grouped_launch(&P, nullptr) == hipSuccess) {
            (void)hipEventRecord(t0, nullptr);
            const int reps = 2;
            for (int r = 0; r < reps; ++r) (void)grouped_launch(&P, nullptr);
            (void)hipEventRecord(t1, nullptr);
            if (hipEventSynchronize(t1) == hipSuccess) {
                (void)hipEventElapsedTime(&ms, t0, t1);
                ms /= reps;
            }
        }
        (void)hipGetLastError();
        grouped_release(&P);
        if (ms < best_ms) {
            best_ms = ms;
            if (rows) pipe = true;
            else best = cfg;
        }
    }
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    if (best_ms >= 1e30f) return fail(FTDX_ERR_HIP, "grouped autotune: no configuration ran");
    return FTDX_OK;
}

}  // namespace ftdx

using ftdx::fail;
using ftdx::hip_fail;

extern "C" {

int ftdx_herk_grouped_plan_create(ftdx_context* ctx, const ftdx_herk_problem* problems, int count,
                                  int output, int tile_config, int use_graph,
                                  ftdx_grouped_plan** plan) {
    if (!ctx || !plan) return fail(FTDX_ERR_INVALID_ARG, "grouped plan: NULL context or plan");
    *plan = nullptr;
    if (count < 0 || (count > 0 && !problems))
        return fail(FTDX_ERR_INVALID_ARG, "grouped plan: bad problem list");
    if (output != FTDX_OUTPUT_FP32 && output != FTDX_OUTPUT_FP16)
        return fail(FTDX_ERR_INVALID_ARG, "grouped plan: unknown output precision");
    if (tile_config < -1 || tile_config >= ftdx::NUM_TILE_CONFIGS)
        return fail(FTDX_ERR_INVALID_ARG, "grouped plan: unknown tile configuration");
    for (int p = 0; p < count; ++p) {
        const ftdx_herk_problem& q = problems[p];
        if (q.N < 0 || q.K < 0) return fail(FTDX_ERR_INVALID_ARG, "grouped plan: negative size");
        if (q.N > 0 && ((!q.A && q.K > 0) || !q.C))
            return fail(FTDX_ERR_INVALID_ARG, "grouped plan: NULL data pointer");
        if (q.C && reinterpret_cast<uintptr_t>(q.C) % (output == FTDX_OUTPUT_FP32 ? 8u : 4u))
            return fail(FTDX_ERR_INVALID_ARG, "grouped plan: C must be aligned to one element");
    }
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "grouped plan: hipGetDevice");
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess)
        return hip_fail(e, "grouped plan: device attribute");
    const int out16 = output == FTDX_OUTPUT_FP16 ? 1 : 0;
    int cfg = tile_config >= 0 ? tile_config : ftdx::TILE_128x128_K64;
    bool all_beta0 = true;
    for (int p = 0; p < count; ++p) all_beta0 = all_beta0 && problems[p].beta == 0.0f;
    bool pipe = false;
    if (tile_config < 0 && all_beta0 && count > 0) {
        int rc = ftdx::grouped_autotune(problems, count, out16, cus, cfg, pipe);
        if (rc != FTDX_OK) return rc;
    }
    auto* P = new ftdx_grouped_plan();
    P->device = dev;
    int rc = pipe ? ftdx::grouped_build_pipe(P, problems, count, cfg, out16) : FTDX_ERR_UNSUPPORTED;
    if (rc != FTDX_OK) {  // also when the rows' memory went to someone else meanwhile
        ftdx::grouped_release(P);
        rc = ftdx::grouped_build(P, problems, count, cfg, out16, cus);
    }
    if (rc == FTDX_OK && use_graph && P->items > 0) rc = ftdx::grouped_capture(P);
    if (rc != FTDX_OK) {
        ftdx::grouped_release(P);
        delete P;
        return rc;
    }
    *plan = P;
    return FTDX_OK;
}

int ftdx_herk_grouped_plan_run(ftdx_grouped_plan* plan, void* stream) {
    if (!plan) return fail(FTDX_ERR_INVALID_ARG, "grouped run: NULL plan");
    if (plan->items == 0) return FTDX_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e = plan->use_graph ? hipGraphLaunch(plan->exec, s) : ftdx::grouped_launch(plan, s);
    if (e != hipSuccess) return hip_fail(e, "grouped run: launch");
    return FTDX_OK;
}

int ftdx_herk_grouped_plan_info(const ftdx_grouped_plan* plan, int* num_workgroups,
                                int64_t* num_items, int* tile_config, double* imbalance) {
    if (!plan) return fail(FTDX_ERR_INVALID_ARG, "grouped info: NULL plan");
    if (num_workgroups) *num_workgroups = plan->num_wg;
    if (num_items) *num_items = plan->items;
    if (tile_config) *tile_config = plan->cfg;
    if (imbalance) *imbalance = plan->mean_load > 0 ? plan->max_load / plan->mean_load : 1.0;
    return FTDX_OK;
}

int ftdx_herk_grouped_plan_destroy(ftdx_grouped_plan* plan) {
    if (!plan) return FTDX_OK;
    ftdx::grouped_release(plan);
    delete plan;
    return FTDX_OK;
}

}  // extern "C"
