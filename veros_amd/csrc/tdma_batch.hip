// Batched TDMA over many independent grids of different shapes and depths.
//
// A plan is built once from the list of systems (the arrays of every grid
// stay where they are): systems are grouped by 16-level nz bucket (8 lanes per
// column in the segmented solve: S = bucket / 8 levels per lane) and cut into
// tiles of up to 8 columns; each bucket's tiles form one sequence.
// vx_tdma_plan_run launches one persistent grid-stride kernel per non-empty
// bucket; a wave takes one tile at a time, finds its system by binary search
// over the systems' first tiles, and runs the single-grid kernels' solve in
// float64 (mode 0) or in mixed precision with one refinement step (mode 1).
// vx_tdma_plan_tune times block-size / grid-size candidates per bucket on the
// plan's own data and keeps the fastest (a process-wide cache keyed by bucket,
// mode, kernel and size reuses earlier choices); vx_tdma_plan_graph_launch captures
// run() once into a hipGraph and replays it.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "tdma_tile.hpp"

struct vx_tdma_plan;

namespace vx {

struct SysDesc {
    TdmaArgs args;
    TdmaTiling tiling;
    int64_t tile0;  // first tile of this system in its bucket
    int32_t vec;    // its arrays allow 16-byte copies into LDS
};

// How a bucket's systems are solved: on flat loads (tdma_tile.hpp; any depth, alignment and
// strides), with 16-byte copies straight into LDS, or each as its arrays allow.
enum BatchKind { kFlat = 0, kCopies = 1, kEither = 2 };

// Whether a bucket of which only the systems with vec_tiles of its tiles allow the copies
// takes those system by system, the others with each lane's own loads, which lose against
// the flat loads by more than the copies win. Six systems of one size, us, all on flat loads /
// by system, float64 and mixed:
//   resident tiles, 4 of 6 allowing: nz 32 1878 tiles 5.1 and 5.0 / 4.8 and 4.7; 48, 2700 8.3 and
//   8.3 / 7.9 and 7.6; 64, 2274 9.1 and 9.1 / 8.8 and 8.7; 80, 1806 9.9 and 9.9 / 9.1 and 9.2; 96, 1392
//   9.2 and 9.1 / 9.0 and 8.9. With 3 of 6: nz 64 9.2 / 11.6, 80 9.3 / 9.6. Fewer than two tiles per CU:
//   nz 80, 432 5.6 / 5.9; more than 16: nz 32, 4686 8.5 / 8.9. 14 and 16 levels per lane: no difference.
//   any size: nz 80, 67500 tiles, mixed, 5 of 6 257 / 241, 4 of 6 259 / 268; float64 235 / 240; nz 96 304 / 307.
inline bool batch_either(int S, bool mixed, int64_t vec_tiles, int64_t tiles) {
    const int64_t cus = cu_count();
    if (S == 10 && mixed && 6 * vec_tiles >= 5 * tiles) return true;
    return S <= 12 && 3 * vec_tiles >= 2 * tiles && tiles > 2 * cus && tiles <= 16 * cus && tdma_lds_resident(S, tiles);
}

// LDS doubles of a wave
template <int S, int KIND>
__host__ __device__ constexpr int batch_lds() {
    return KIND == kFlat ? tdma_tile_lds<S>() : seg_lds_wave_bytes(S) / 8;
}

// One launch per bucket: S levels per lane, MODE -1 = float64, else mixed with
// MODE refinement steps. On flat loads at S = 2 each lane loads its own levels
// (tdma_own_levels).
template <int S, int MODE, int KIND>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2))) void tdma_seg_batch_kernel(const SysDesc* __restrict__ sys, int nsys,
                                                             int64_t ntiles) {
    extern __shared__ double seg_lds[];
    double* lds = seg_lds + (threadIdx.x / 64) * batch_lds<S, KIND>();
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / 64);
    // the tile index is the same in every lane of a wave: keep it (and so
    // the system search and descriptor loads) in scalar registers
    const int64_t w0 = (int64_t)blockIdx.x * (blockDim.x / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    for (int64_t w = w0; w < ntiles; w += wstride) {
        int lo = 0, hi = nsys - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sys[mid].tile0 <= w) lo = mid;
            else hi = mid - 1;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        const SysDesc& sd = sys[lo];
        const TdmaArgs p = sd.args;
        SegLane L;
        const Tile<S, kTdmaP> t = tdma_tile_of<S>(p, sd.tiling, w - sd.tile0, L);
        if constexpr (KIND == kFlat && tdma_own_levels(S)) {
            if constexpr (MODE < 0) seg_f64<S, false>(p, L);
            else seg_mixed<S, false, MODE>(p, L);
        } else if constexpr (KIND == kFlat) {
            tdma_tile<S, MODE>(p, t, L, lds);
        } else {
            const bool copies = KIND == kCopies || sd.vec;
            double va[S], vb[S], vc[S], vd[S], x[S];
            if (copies) seg_rows_lds<S>(p, L, lds, va, vb, vc, vd);
            else seg_rows<S, false>(p, L, va, vb, vc, vd);
            if constexpr (MODE < 0) {
                seg_solve_f64<S>(L, va, vb, vc, vd);
#pragma unroll
                for (int q = 0; q < S; ++q) x[q] = vd[q];
            } else {
                seg_mixed_core<S, MODE>(L, va, vb, vc, vd, x);
            }
            if (copies) seg_store_lds<S>(p, L, lds, x);
            else if (L.valid) seg_store<S, false>(p.x + L.base, L.lo, p.nz, x);
        }
    }
}

namespace {

constexpr int kBuckets[] = {16, 32, 48, 64, 80, 96, 112, 128};
constexpr int kNumBuckets = 8;
constexpr int kBlockSizes[] = {64, 128};  // one or two waves (LDS: seg_lds_wave_bytes(S) per wave)
constexpr int kGridFactors[] = {1, 2, 4, 8, 0};  // blocks per CU; 0 = one tile per wave

struct Bucket {
    int nzb = 0;
    int first = 0;       // index of the first system of this bucket in the device table
    int nsys = 0;
    int64_t tiles = 0;   // tiles of up to 8 columns
    int64_t cols = 0;    // columns
    int kind = kFlat;    // BatchKind
    int bs = 128;
    int factor = 0;
};

// nzb, mode, kind (each has other LDS and registers), log2(columns), CUs
using TuneKey = std::tuple<int, int, int, int, int>;
std::mutex g_tune_mutex;
std::map<TuneKey, std::pair<int, int>> g_tune_cache;

int ilog2(int64_t v) {
    int r = 0;
    while (v > 1) {
        v >>= 1;
        ++r;
    }
    return r;
}

TuneKey tune_key(const Bucket& b, int mode, int num_cu) {
    return {b.nzb, mode, b.kind, ilog2(b.tiles * kSegCols), num_cu};
}

template <int S, int MODE, int KIND>
void launch_kind(int bs, const SysDesc* d, int nsys, int64_t tiles, unsigned grid, hipStream_t s) {
    const size_t lds = (size_t)batch_lds<S, KIND>() * 8 * (bs / 64);
    hipLaunchKernelGGL((tdma_seg_batch_kernel<S, MODE, KIND>), dim3(grid), dim3(bs), lds, s, d, nsys, tiles);
}
template <int S, int MODE>
void launch_bs(int bs, int kind, const SysDesc* d, int nsys, int64_t tiles, unsigned grid, hipStream_t s) {
    if constexpr (S <= 12) {
        if (kind == kEither) return launch_kind<S, MODE, kEither>(bs, d, nsys, tiles, grid, s);
    }
    if (kind == kCopies) launch_kind<S, MODE, kCopies>(bs, d, nsys, tiles, grid, s);
    else launch_kind<S, MODE, kFlat>(bs, d, nsys, tiles, grid, s);
}

template <int MODE>
void launch_mode(int nzb, int bs, int kind, const SysDesc* d, int nsys, int64_t tiles, unsigned grid, hipStream_t s) {
    switch (nzb) {
        case 16: launch_bs<2, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 32: launch_bs<4, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 48: launch_bs<6, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 64: launch_bs<8, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 80: launch_bs<10, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 96: launch_bs<12, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        case 112: launch_bs<14, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
        default: launch_bs<16, MODE>(bs, kind, d, nsys, tiles, grid, s); break;
    }
}

}  // namespace
}  // namespace vx

struct vx_tdma_plan {
    int mode = 0;
    int num_cu = 0;
    std::vector<vx::Bucket> buckets;
    vx::SysDesc* d_sys = nullptr;
    hipStream_t capture_stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // every non-empty system (tune checks that none solves in place)
    std::vector<vx_tdma_system> all;
};

namespace vx {
namespace {

unsigned grid_for(const vx_tdma_plan* P, const Bucket& b, int bs, int factor) {
    const int64_t full = (b.tiles * 64 + bs - 1) / bs;  // one tile per wave
    if (factor == 0) return (unsigned)std::max<int64_t>(1, full);
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(full, (int64_t)factor * P->num_cu));
}

void launch_bucket(const vx_tdma_plan* P, const Bucket& b, int bs, int factor, hipStream_t s) {
    const SysDesc* d = P->d_sys + b.first;
    const unsigned grid = grid_for(P, b, bs, factor);
    if (P->mode == 0) launch_mode<-1>(b.nzb, bs, b.kind, d, b.nsys, b.tiles, grid, s);
    else launch_mode<1>(b.nzb, bs, b.kind, d, b.nsys, b.tiles, grid, s);
}

}  // namespace
}  // namespace vx

extern "C" int vx_tdma_plan_create(const vx_tdma_system* systems, int32_t nsys, int32_t mode,
                                   vx_tdma_plan** out) {
    using namespace vx;
    const char* who = "vx_tdma_plan_create";
    if (!out) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null output handle", who);
    *out = nullptr;
    if (!systems || nsys < 1) return fail(VX_ERR_INVALID_ARGUMENT, "%s: need at least one system", who);
    if (mode < 0 || mode > 1)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: mode must be 0 (fp64) or 1 (mixed, one refinement step)", who);
    std::vector<std::vector<SysDesc>> per(kNumBuckets);
    std::vector<vx_tdma_system> all;
    for (int q = 0; q < nsys; ++q) {
        const vx_tdma_system& y = systems[q];
        if (y.nz < 1 || y.nx < 0 || y.ny < 0)
            return fail(VX_ERR_INVALID_ARGUMENT, "%s: system %d has an invalid shape", who, q);
        if (y.nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: system %d has nz=%d > %d", who, q, y.nz, kMaxNz);
        if (y.nx * y.ny == 0) continue;
        if (!y.a || !y.b || !y.c || !y.d || !y.kbot || !y.x)
            return fail(VX_ERR_INVALID_ARGUMENT, "%s: system %d has a null array", who, q);
        if (y.sy < y.nz || y.sx < (y.ny - 1) * y.sy + y.nz)
            return fail(VX_ERR_INVALID_ARGUMENT, "%s: system %d strides overlap columns", who, q);
        SysDesc sd{};
        TdmaArgs& p = sd.args;
        p.a = y.a, p.b = y.b, p.c = y.c, p.d = y.d, p.b_edge = y.b_edge, p.d_edge = y.d_edge;
        p.kbot = y.kbot, p.x = y.x;
        p.ny = y.ny, p.ncol = y.nx * y.ny, p.sx = y.sx, p.sy = y.sy, p.kx = y.kbot_sx, p.ky = y.kbot_sy;
        p.nz = y.nz;
        per[(y.nz + 15) / 16 - 1].push_back(sd);
        all.push_back(y);
    }
    auto* P = new vx_tdma_plan();
    P->mode = mode;
    P->all = std::move(all);
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
        delete P;
        return fail(VX_ERR_LAUNCH, "%s: cannot query the device", who);
    }
    P->num_cu = prop.multiProcessorCount;
    std::vector<SysDesc> table;
    for (int bk = 0; bk < kNumBuckets; ++bk) {
        if (per[bk].empty()) continue;
        Bucket b;
        b.nzb = kBuckets[bk];
        b.first = (int)table.size();
        b.nsys = (int)per[bk].size();
        int64_t vec_tiles = 0;
        for (SysDesc& sd : per[bk]) {
            sd.tiling = tdma_tiling(sd.args);
            sd.tile0 = b.tiles;
            b.tiles += sd.tiling.ntiles;
            b.cols += sd.args.ncol;
            sd.vec = tdma_vec_ok(sd.args) ? 1 : 0;
            vec_tiles += sd.vec ? sd.tiling.ntiles : 0;
            table.push_back(sd);
        }
        const int S = b.nzb / kTdmaP;
        if (vec_tiles == b.tiles && (tdma_lds_wins(S, mode != 0, true) || tdma_lds_resident(S, b.tiles)))
            b.kind = kCopies;
        else if (vec_tiles < b.tiles && batch_either(S, mode != 0, vec_tiles, b.tiles))
            b.kind = kEither;
        {
            std::lock_guard<std::mutex> lk(g_tune_mutex);
            auto it = g_tune_cache.find(tune_key(b, mode, P->num_cu));
            if (it != g_tune_cache.end()) {
                b.bs = it->second.first;
                b.factor = it->second.second;
            }
        }
        P->buckets.push_back(b);
    }
    if (!table.empty()) {
        if (hipMalloc(&P->d_sys, table.size() * sizeof(SysDesc)) != hipSuccess) {
            delete P;
            return fail(VX_ERR_LAUNCH, "%s: hipMalloc of the system table failed", who);
        }
        if (hipMemcpy(P->d_sys, table.data(), table.size() * sizeof(SysDesc), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(P->d_sys);
            delete P;
            return fail(VX_ERR_LAUNCH, "%s: copying the system table failed", who);
        }
    }
    *out = P;
    return VX_OK;
}

namespace vx {
namespace {
// Byte range [lo, hi) spanned by one (nx, ny, nz) float64 array of a system.
std::pair<uintptr_t, uintptr_t> span_of(const double* p, const vx_tdma_system& y) {
    const uintptr_t lo = reinterpret_cast<uintptr_t>(p);
    const int64_t last = (y.nx - 1) * y.sx + (y.ny - 1) * y.sy + y.nz;
    return {lo, lo + (uintptr_t)last * sizeof(double)};
}

// True when some system's x overlaps one of its (or another system's) inputs.
bool solves_in_place(const std::vector<vx_tdma_system>& sys) {
    for (const vx_tdma_system& y : sys) {
        const auto xs = span_of(y.x, y);
        for (const vx_tdma_system& z : sys) {
            for (const double* in : {z.a, z.b, z.c, z.d, z.b_edge, z.d_edge}) {
                if (!in) continue;
                const auto r = span_of(in, z);
                if (xs.first < r.second && r.first < xs.second) return true;
            }
        }
    }
    return false;
}

int run_plan(vx_tdma_plan* plan, hipStream_t s, const char* who) {
    for (const Bucket& b : plan->buckets) launch_bucket(plan, b, b.bs, b.factor, s);
    return check_launch(who);
}
}  // namespace
}  // namespace vx

extern "C" int vx_tdma_plan_run(vx_tdma_plan* plan, void* stream) {
    using namespace vx;
    if (!plan) return fail(VX_ERR_INVALID_ARGUMENT, "vx_tdma_plan_run: null plan");
    return run_plan(plan, (hipStream_t)stream, "vx_tdma_plan_run");
}

extern "C" int vx_tdma_plan_tune(vx_tdma_plan* plan, void* stream) {
    using namespace vx;
    const char* who = "vx_tdma_plan_tune";
    if (!plan) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null plan", who);
    // tuning solves every bucket many times over: an in-place system (x
    // overlapping an input) would solve its own previous result
    if (solves_in_place(plan->all))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: a system's x overlaps an input (in-place solve); tuning would "
                    "overwrite that input", who);
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
        return fail(VX_ERR_LAUNCH, "%s: hipEventCreate failed", who);
    int rc = VX_OK;
    for (Bucket& b : plan->buckets) {
        float best = 1e30f;
        int best_bs = b.bs, best_f = b.factor;
        for (int bs : kBlockSizes) {
            for (int f : kGridFactors) {
                launch_bucket(plan, b, bs, f, s);  // warm-up
                float ms = 1e30f;
                for (int r = 0; r < 3; ++r) {
                    (void)hipEventRecord(e0, s);
                    launch_bucket(plan, b, bs, f, s);
                    (void)hipEventRecord(e1, s);
                    if (hipEventSynchronize(e1) != hipSuccess) {
                        rc = fail(VX_ERR_LAUNCH, "%s: %s", who, hipGetErrorString(hipGetLastError()));
                        break;
                    }
                    float t = 0.f;
                    (void)hipEventElapsedTime(&t, e0, e1);
                    ms = std::min(ms, t);
                }
                if (rc) break;
                if (ms < best) {
                    best = ms;
                    best_bs = bs;
                    best_f = f;
                }
            }
            if (rc) break;
        }
        if (rc) break;
        b.bs = best_bs;
        b.factor = best_f;
        std::lock_guard<std::mutex> lk(g_tune_mutex);
        g_tune_cache[tune_key(b, plan->mode, plan->num_cu)] = {b.bs, b.factor};
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    // a graph captured before tuning used the old launch shapes
    if (plan->exec) {
        (void)hipGraphExecDestroy(plan->exec);
        plan->exec = nullptr;
    }
    if (plan->graph) {
        (void)hipGraphDestroy(plan->graph);
        plan->graph = nullptr;
    }
    return check_launch(who);
}

extern "C" int vx_tdma_plan_graph_launch(vx_tdma_plan* plan, void* stream) {
    using namespace vx;
    const char* who = "vx_tdma_plan_graph_launch";
    if (!plan) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null plan", who);
    if (!plan->exec) {
        // capture on a private stream (the legacy default stream cannot be captured)
        if (!plan->capture_stream &&
            hipStreamCreateWithFlags(&plan->capture_stream, hipStreamNonBlocking) != hipSuccess)
            return fail(VX_ERR_LAUNCH, "%s: hipStreamCreate failed", who);
        if (hipStreamBeginCapture(plan->capture_stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
            return fail(VX_ERR_LAUNCH, "%s: hipStreamBeginCapture failed", who);
        const int rc = run_plan(plan, plan->capture_stream, who);
        hipGraph_t g = nullptr;
        if (hipStreamEndCapture(plan->capture_stream, &g) != hipSuccess || !g)
            return fail(VX_ERR_LAUNCH, "%s: capture failed", who);
        if (rc) {
            (void)hipGraphDestroy(g);
            return rc;
        }
        if (hipGraphInstantiate(&plan->exec, g, nullptr, nullptr, 0) != hipSuccess) {
            (void)hipGraphDestroy(g);
            return fail(VX_ERR_LAUNCH, "%s: hipGraphInstantiate failed", who);
        }
        plan->graph = g;
    }
    if (hipGraphLaunch(plan->exec, (hipStream_t)stream) != hipSuccess)
        return fail(VX_ERR_LAUNCH, "%s: hipGraphLaunch failed: %s", who, hipGetErrorString(hipGetLastError()));
    return VX_OK;
}

extern "C" int vx_tdma_plan_info(const vx_tdma_plan* plan, int32_t* nbuckets, int64_t* total_columns,
                                 int32_t* choices, int32_t max_choices) {
    using namespace vx;
    if (!plan) return fail(VX_ERR_INVALID_ARGUMENT, "vx_tdma_plan_info: null plan");
    int64_t tot = 0;
    int q = 0;
    for (const Bucket& b : plan->buckets) {
        tot += b.cols;
        if (choices && q < max_choices) {
            choices[3 * q + 0] = b.nzb;
            choices[3 * q + 1] = b.bs;
            choices[3 * q + 2] = b.factor;
        }
        ++q;
    }
    if (nbuckets) *nbuckets = (int32_t)plan->buckets.size();
    if (total_columns) *total_columns = tot;
    return VX_OK;
}

extern "C" void vx_tdma_plan_destroy(vx_tdma_plan* plan) {
    if (!plan) return;
    if (plan->exec) (void)hipGraphExecDestroy(plan->exec);
    if (plan->graph) (void)hipGraphDestroy(plan->graph);
    if (plan->capture_stream) (void)hipStreamDestroy(plan->capture_stream);
    if (plan->d_sys) (void)hipFree(plan->d_sys);
    delete plan;
}
