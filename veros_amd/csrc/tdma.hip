// Batched kbot-masked tridiagonal (Thomas) solves for gfx950.
//
// Semantics follow solve_implicit / solve_tridiagonal (veros/core/utilities.py:51-59,
// veros/core/operators.py:60-77,133-156): per column the wet suffix
// k in [kbot-1, nz) is one system, the sub-diagonal is 0 at the edge row
// k = kbot-1 (where b, d may be replaced by b_edge, d_edge) and the
// super-diagonal is 0 at the top row; x is 0 outside the wet suffix.
//
// Layout: (x, y, z) with z contiguous. Eight lanes own a column (tdma_seg.hpp);
// a wave brings its eight columns in either flat through registers
// (tdma_tile.hpp: any alignment, stride and depth) or with 16-byte copies
// straight into LDS. The lane-per-column kernels at the end of the file walk
// their column bottom-up with the elimination factors in VGPRs.
#include "tdma_tile.hpp"

#include <cstdlib>

namespace vx {

template <int S, bool VEC>
__global__ __launch_bounds__(kSegBlock) void tdma_seg_f64_kernel(TdmaArgs p) {
    seg_f64<S, VEC>(p, seg_lane_of(p, S));
}

template <int S, bool VEC, int REFINE>
__global__ __launch_bounds__(kSegBlock) void tdma_seg_mixed_kernel(TdmaArgs p) {
    seg_mixed<S, VEC, REFINE>(p, seg_lane_of(p, S));
}

// LDS-staged segmented kernels (16-byte aligned operands only). Dynamic LDS:
// seg_lds_wave_bytes(S) per wave.
template <int S, bool VEC>
__global__ __launch_bounds__(kSegLdsBlock) void tdma_segl_f64_kernel(TdmaArgs p) {
    extern __shared__ double seg_lds[];
    double* lds = seg_lds + (threadIdx.x / 64) * (seg_lds_wave_bytes(S) / 8);
    seg_f64_lds<S>(p, seg_lane_of(p, S), lds);
}

template <int S, bool VEC, int REFINE>
__global__ __launch_bounds__(kSegLdsBlock) void tdma_segl_mixed_kernel(TdmaArgs p) {
    extern __shared__ double seg_lds[];
    double* lds = seg_lds + (threadIdx.x / 64) * (seg_lds_wave_bytes(S) / 8);
    seg_mixed_lds<S, REFINE>(p, seg_lane_of(p, S), lds);
}

// Column tiles, one per wave (two waves per SIMD at least: the mixed form at
// 16 levels per lane would take the registers of one).
template <int S, int MODE>
__global__ __launch_bounds__(kSegLdsBlock) __attribute__((amdgpu_waves_per_eu(2))) void tdma_tile_kernel(TdmaArgs p, TdmaTiling g) {
    __shared__ double img[kSegLdsBlock / 64][tdma_tile_lds<S>()];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    SegLane L;
    const Tile<S, kTdmaP> t = tdma_tile_of<S>(p, g, (int64_t)blockIdx.x * (kSegLdsBlock / 64) + wave, L);
    tdma_tile<S, MODE>(p, t, L, img[wave]);
}

template <int NZB, bool VEC>
__global__ __launch_bounds__(kTdmaBlock) void tdma_f64_kernel(TdmaArgs p) {
    ColumnRef cr;
    if (column_of(p, cr)) solve_f64_column<NZB, VEC>(p, cr);
}

template <int NZB, bool VEC, int REFINE>
__global__ __launch_bounds__(kTdmaBlock) void tdma_mixed_kernel(TdmaArgs p) {
    ColumnRef cr;
    if (column_of(p, cr)) solve_mixed_column<NZB, VEC, REFINE>(p, cr);
}

// ---------------------------------------------------------------------------
// Adjoint of the float64 solve: given x = A^-1 d and g = dL/dx, the
// transposed system A^T lam = g (sub-diagonal c[k-1], super-diagonal a[k+1]
// on the wet rows) is solved by Thomas, re-deriving the elimination from a, b,
// c instead of storing forward factors; then dL/dd = lam, dL/db = -lam*x,
// dL/da[k] = -lam[k]*x[k-1] (k above the edge), dL/dc[k] = -lam[k]*x[k+1]
// (k below the top). Entries the forward solve ignores (a at the edge, c at
// the top, dry cells, b/d at the edge when b_edge/d_edge replace them) get 0.
// ---------------------------------------------------------------------------
struct TdmaAdjArgs {
    TdmaArgs f;       // forward inputs; f.x is the forward solution
    const double* g;  // dL/dx
    double *ga, *gb, *gc, *gd;
    double *gbe, *gde;  // dL/db_edge, dL/dd_edge (nullable; used when b_edge / d_edge were given)
};

// On column tiles (tdma_tile.hpp): the transposed rows take c from the level
// below and a from the level above out of the images, lam comes back flat, and
// every gradient is formed and stored cell by cell. One lane per column with
// the column's factors in registers (16,200 columns of 180x90x40: 63 blocks)
// took 72 us there, the tiles 11 us.
template <int S>
__global__ __launch_bounds__(kSegLdsBlock) __attribute__((amdgpu_waves_per_eu(2))) void tdma_adjoint_kernel(TdmaAdjArgs q, TdmaTiling g) {
    __shared__ double lds[kSegLdsBlock / 64][2][tdma_tile_lds<S>()];
    const TdmaArgs& p = q.f;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    double* const img = lds[wave][0];
    double* const ximg = lds[wave][1];
    SegLane L;
    const Tile<S, kTdmaP> t = tdma_tile_of<S>(p, g, (int64_t)blockIdx.x * (kSegLdsBlock / 64) + wave, L);
    const int nz = p.nz;
    uint32_t wet[S];
#pragma unroll
    for (int r = 0; r < S; ++r) wet[r] = t.k[r] >= __shfl(L.k0, t.c[r] * kTdmaP) ? t.off[r] : kNoAccess;
    double sub[S], diag[S], sup[S], z[S], x[S], be, de;
    {
        double fa[S], fc[S];
        tile_load(tile_buf(t, p.c), wet, 1, fc);
        tile_load(tile_buf(t, p.a), wet, 1, fa);
        tile_load(tile_buf(t, p.b), wet, 1, diag);
        tile_load(tile_buf(t, q.g), wet, 1, z);
        tile_load(tile_buf(t, (const double*)p.x), wet, 1, x);
        seg_edge_values(p, L, S, be, de);
        double v[S];
        tile_put(t, img, fc);
        seg_get(t, img, v);
        sub[0] = seg_below(t, img);
#pragma unroll
        for (int r = 1; r < S; ++r) sub[r] = v[r - 1];
        tile_put(t, img, fa);
        seg_get(t, img, v);
        sup[S - 1] = seg_above(t, img);
#pragma unroll
        for (int r = 0; r < S - 1; ++r) sup[r] = v[r + 1];
        tile_put(t, img, diag);
        seg_get(t, img, diag);
        tile_put(t, img, z);
        seg_get(t, img, z);
        tile_put(t, ximg, x);
    }
    seg_mask_rows<S>(p, L, be, 0.0, sub, diag, sup, z, false);
    if constexpr (S <= 8) {
        // lam shares x's pivots, so that in gb = -lam x their roundings add up (nz 9 to 60:
        // 1.09 to 1.02 times the error of a sequential lam): one step of refinement
        double a[S], c[S], d[S];
#pragma unroll
        for (int r = 0; r < S; ++r) a[r] = sub[r], c[r] = sup[r], d[r] = z[r];
        seg_solve_f64<S, 2>(L, sub, diag, sup, z);
        const double zm = grp_prev(L.s, z[S - 1]), zp = grp_next(L.s, z[0]);
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const double m = r > 0 ? z[r > 0 ? r - 1 : 0] : zm, p = r < S - 1 ? z[r < S - 1 ? r + 1 : 0] : zp;
            d[r] = fma(-a[r], m, fma(-c[r], p, fma(-diag[r], z[r], d[r])));
        }
        seg_solve_f64<S>(L, a, diag, c, d);
#pragma unroll
        for (int r = 0; r < S; ++r) z[r] += fabs(d[r]) < HUGE_VAL ? d[r] : 0.0;
    } else {
        seg_solve_f64<S, 2>(L, sub, diag, sup, z);
    }
    seg_put(t, img, z);
    double lam[S], ga[S], gb[S], gc[S], gd[S];
    tile_get(t, img, lam);
    const bool has_be = p.b_edge != nullptr, has_de = p.d_edge != nullptr;
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const int k = t.k[r], k0 = __shfl(L.k0, t.c[r] * kTdmaP);
        const bool w = k >= k0, edge = k == k0;
        int below, above;
        flat_neighbours<S, kTdmaP>({k, t.c[r], t.pos[r], t.off[r]}, k0, nz, below, above);
        const double xm = ximg[below], xp = ximg[above];
        const double l = w ? lam[r] : 0.0;
        ga[r] = edge ? 0.0 : -l * xm;
        gb[r] = -l * x[r];
        gc[r] = k < nz - 1 ? -l * xp : 0.0;
        gd[r] = l;
    }
    tile_store(tile_buf(t, q.ga), t.off, 1, ga);
    tile_store(tile_buf(t, q.gc), t.off, 1, gc);
    // the edge row's derivatives go to the edge arrays when those were given
    auto split = [&](const double(&v)[S], double* inner, double* at_edge, bool has) {
        double e[S], i[S];
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const bool edge = has && t.k[r] == __shfl(L.k0, t.c[r] * kTdmaP);
            e[r] = edge ? v[r] : 0.0;
            i[r] = edge ? 0.0 : v[r];
        }
        tile_store(tile_buf(t, inner), t.off, 1, i);
        if (at_edge) tile_store(tile_buf(t, at_edge), t.off, 1, e);
    };
    split(gb, q.gb, q.gbe, has_be);
    split(gd, q.gd, q.gde, has_de);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

int validate_tdma(const TdmaArgs& p, int64_t nx, int64_t ny, int32_t nz, const char* who) {
    if (nx < 0 || ny < 0) return fail(VX_ERR_INVALID_ARGUMENT, "%s: negative shape (%lld, %lld)", who, (long long)nx, (long long)ny);
    if (nz < 1) return fail(VX_ERR_INVALID_ARGUMENT, "%s: nz must be >= 1 (got %d)", who, nz);
    if (nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d exceeds the compiled maximum %d", who, nz, kMaxNz);
    if (nx * ny == 0) return VX_OK;
    if (!p.a || !p.b || !p.c || !p.d || !p.kbot || !p.x)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if (p.sy < nz || p.sx < (ny - 1) * p.sy + nz)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: strides (sx=%lld, sy=%lld) overlap columns of depth %d", who,
                    (long long)p.sx, (long long)p.sy, nz);
    return VX_OK;
}

template <template <int, bool> class K>
int launch_bucket(const TdmaArgs& p, hipStream_t s, const char* who) {
    const int nzb = ((p.nz + 15) / 16) * 16;
    const bool vec = tdma_vec_ok(p);
    const dim3 grid((unsigned)((p.ncol + kTdmaBlock - 1) / kTdmaBlock));
    const dim3 block(kTdmaBlock);
#define VX_TDMA_CASE(N)                                                                      \
    case N:                                                                                  \
        if (vec) hipLaunchKernelGGL((K<N, true>::fn), grid, block, 0, s, p);       \
        else hipLaunchKernelGGL((K<N, false>::fn), grid, block, 0, s, p);          \
        break;
    switch (nzb) {
        VX_TDMA_CASE(16)
        VX_TDMA_CASE(32)
        VX_TDMA_CASE(48)
        VX_TDMA_CASE(64)
        VX_TDMA_CASE(80)
        VX_TDMA_CASE(96)
        VX_TDMA_CASE(112)
        VX_TDMA_CASE(128)
        default:
            return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, p.nz);
    }
#undef VX_TDMA_CASE
    return check_launch(who);
}

// Segmented kernels (kSegP lanes per column), instantiated per levels-per-lane S.
template <template <int, bool> class K>
int launch_seg(const TdmaArgs& p, hipStream_t s, const char* who) {
    const int S = seg_levels(p.nz);
    const bool vec = tdma_vec_ok(p);
    const int64_t threads = p.ncol * kSegP;
    const dim3 grid((unsigned)((threads + kSegBlock - 1) / kSegBlock));
    const dim3 block(kSegBlock);
#define VX_SEG_CASE(N)                                                            \
    case N:                                                                       \
        if (vec) hipLaunchKernelGGL((K<N, true>::fn), grid, block, 0, s, p);    \
        else hipLaunchKernelGGL((K<N, false>::fn), grid, block, 0, s, p);       \
        break;
    switch (S) {
        VX_SEG_CASE(2)
        VX_SEG_CASE(4)
        VX_SEG_CASE(6)
        VX_SEG_CASE(8)
        VX_SEG_CASE(10)
        VX_SEG_CASE(12)
        VX_SEG_CASE(14)
        VX_SEG_CASE(16)
        default:
            return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, p.nz);
    }
#undef VX_SEG_CASE
    return check_launch(who);
}

// LDS-staged segmented kernels: only with 16-byte aligned operands.
template <template <int, bool> class K>
int launch_segl(const TdmaArgs& p, hipStream_t s, const char* who) {
    const int S = seg_levels(p.nz);
    const int64_t threads = p.ncol * kSegP;
    const dim3 grid((unsigned)((threads + kSegLdsBlock - 1) / kSegLdsBlock));
    const dim3 block(kSegLdsBlock);
    const size_t lds = (size_t)seg_lds_wave_bytes(S) * (kSegLdsBlock / 64);
#define VX_SEGL_CASE(N)                                                     \
    case N:                                                                 \
        hipLaunchKernelGGL((K<N, true>::fn), grid, block, lds, s, p);       \
        break;
    switch (S) {
        VX_SEGL_CASE(2)
        VX_SEGL_CASE(4)
        VX_SEGL_CASE(6)
        VX_SEGL_CASE(8)
        VX_SEGL_CASE(10)
        VX_SEGL_CASE(12)
        VX_SEGL_CASE(14)
        VX_SEGL_CASE(16)
        default:
            return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, p.nz);
    }
#undef VX_SEGL_CASE
    return check_launch(who);
}

template <int MODE>
int launch_tile(const TdmaArgs& p, hipStream_t s, const char* who) {
    const TdmaTiling g = tdma_tiling(p);
    const int waves = kSegLdsBlock / 64;
    const dim3 grid((unsigned)((g.ntiles + waves - 1) / waves)), block(kSegLdsBlock);
#define VX_TILE_CASE(N) \
    case N: hipLaunchKernelGGL((tdma_tile_kernel<N, MODE>), grid, block, 0, s, p, g); break;
    switch (seg_levels(p.nz)) {  // not 2: tdma_own_levels
        VX_TILE_CASE(4)
        VX_TILE_CASE(6)
        VX_TILE_CASE(8)
        VX_TILE_CASE(10)
        VX_TILE_CASE(12)
        VX_TILE_CASE(14)
        VX_TILE_CASE(16)
        default:
            return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, p.nz);
    }
#undef VX_TILE_CASE
    return check_launch(who);
}

template <int N, bool V>
struct SeglF64K {
    static constexpr auto fn = tdma_segl_f64_kernel<N, V>;
};
template <int N, bool V>
struct SeglMixK0 {
    static constexpr auto fn = tdma_segl_mixed_kernel<N, V, 0>;
};
template <int N, bool V>
struct SeglMixK1 {
    static constexpr auto fn = tdma_segl_mixed_kernel<N, V, 1>;
};
template <int N, bool V>
struct SeglMixK2 {
    static constexpr auto fn = tdma_segl_mixed_kernel<N, V, 2>;
};

template <int N, bool V>
struct SegF64K {
    static constexpr auto fn = tdma_seg_f64_kernel<N, V>;
};
template <int N, bool V>
struct SegMixK0 {
    static constexpr auto fn = tdma_seg_mixed_kernel<N, V, 0>;
};
template <int N, bool V>
struct SegMixK1 {
    static constexpr auto fn = tdma_seg_mixed_kernel<N, V, 1>;
};
template <int N, bool V>
struct SegMixK2 {
    static constexpr auto fn = tdma_seg_mixed_kernel<N, V, 2>;
};

// Kernel family of the single-grid solves (VX_TDMA_KERNEL, read once):
// default: column tiles, or the LDS-staged kernels where they are faster (see
// tdma_lds_wins); "segment": segmented, register loads; "column": lane per
// column.
int tdma_kernel_family() {
    static const int fam = [] {
        const char* e = std::getenv("VX_TDMA_KERNEL");
        if (e != nullptr && std::string(e) == "column") return 0;
        if (e != nullptr && std::string(e) == "segment") return 1;
        return 2;
    }();
    return fam;
}
bool use_column_kernels() { return tdma_kernel_family() == 0; }
bool use_segment_kernels() { return tdma_kernel_family() == 1; }

bool lds_kernel_wins(const TdmaArgs& p, bool mixed) {
    const int S = seg_levels(p.nz);
    return tdma_vec_ok(p) && (tdma_lds_wins(S, mixed, false) || tdma_lds_resident(S, tdma_tiling(p).ntiles));
}

// the segmented kernels with register loads
bool own_levels(const TdmaArgs& p) {
    return use_segment_kernels() || (tdma_own_levels(seg_levels(p.nz)) && !tdma_vec_ok(p));
}

template <int N, bool V>
struct F64K {
    static constexpr auto fn = tdma_f64_kernel<N, V>;
};
template <int N, bool V>
struct MixK0 {
    static constexpr auto fn = tdma_mixed_kernel<N, V, 0>;
};
template <int N, bool V>
struct MixK1 {
    static constexpr auto fn = tdma_mixed_kernel<N, V, 1>;
};
template <int N, bool V>
struct MixK2 {
    static constexpr auto fn = tdma_mixed_kernel<N, V, 2>;
};

TdmaArgs make_args(const double* a, const double* b, const double* c, const double* d, const double* b_edge,
                   const double* d_edge, const int32_t* kbot, int64_t kbot_sx, int64_t kbot_sy, double* x,
                   int64_t nx, int64_t ny, int32_t nz, int64_t sx, int64_t sy) {
    TdmaArgs p;
    p.a = a;
    p.b = b;
    p.c = c;
    p.d = d;
    p.b_edge = b_edge;
    p.d_edge = d_edge;
    p.kbot = kbot;
    p.x = x;
    p.ny = ny;
    p.ncol = nx * ny;
    p.sx = sx;
    p.sy = sy;
    p.kx = kbot_sx;
    p.ky = kbot_sy;
    p.nz = nz;
    return p;
}

}  // namespace
}  // namespace vx

extern "C" int vx_tdma_f64(void* stream, const double* a, const double* b, const double* c, const double* d,
                           const double* b_edge, const double* d_edge, const int32_t* kbot, int64_t kbot_sx,
                           int64_t kbot_sy, double* x, int64_t nx, int64_t ny, int32_t nz, int64_t sx, int64_t sy) {
    using namespace vx;
    TdmaArgs p = make_args(a, b, c, d, b_edge, d_edge, kbot, kbot_sx, kbot_sy, x, nx, ny, nz, sx, sy);
    int rc = validate_tdma(p, nx, ny, nz, "vx_tdma_f64");
    if (rc != VX_OK || p.ncol == 0) return rc;
    if (use_column_kernels()) return launch_bucket<F64K>(p, (hipStream_t)stream, "vx_tdma_f64");
    if (own_levels(p)) return launch_seg<SegF64K>(p, (hipStream_t)stream, "vx_tdma_f64");
    if (lds_kernel_wins(p, false)) return launch_segl<SeglF64K>(p, (hipStream_t)stream, "vx_tdma_f64");
    return launch_tile<-1>(p, (hipStream_t)stream, "vx_tdma_f64");
}

extern "C" int vx_tdma_mixed(void* stream, const double* a, const double* b, const double* c, const double* d,
                             const double* b_edge, const double* d_edge, const int32_t* kbot, int64_t kbot_sx,
                             int64_t kbot_sy, double* x, int64_t nx, int64_t ny, int32_t nz, int64_t sx, int64_t sy,
                             int32_t refine_steps) {
    using namespace vx;
    if (refine_steps < 0 || refine_steps > 2)
        return fail(VX_ERR_INVALID_ARGUMENT, "vx_tdma_mixed: refine_steps must be 0, 1 or 2 (got %d)", refine_steps);
    TdmaArgs p = make_args(a, b, c, d, b_edge, d_edge, kbot, kbot_sx, kbot_sy, x, nx, ny, nz, sx, sy);
    int rc = validate_tdma(p, nx, ny, nz, "vx_tdma_mixed");
    if (rc != VX_OK || p.ncol == 0) return rc;
    hipStream_t s = (hipStream_t)stream;
    const char* who = "vx_tdma_mixed";
    if (use_column_kernels()) {
        switch (refine_steps) {
            case 0: return launch_bucket<MixK0>(p, s, who);
            case 1: return launch_bucket<MixK1>(p, s, who);
            default: return launch_bucket<MixK2>(p, s, who);
        }
    }
    if (own_levels(p)) {
        switch (refine_steps) {
            case 0: return launch_seg<SegMixK0>(p, s, who);
            case 1: return launch_seg<SegMixK1>(p, s, who);
            default: return launch_seg<SegMixK2>(p, s, who);
        }
    }
    if (lds_kernel_wins(p, true)) {
        switch (refine_steps) {
            case 0: return launch_segl<SeglMixK0>(p, s, who);
            case 1: return launch_segl<SeglMixK1>(p, s, who);
            default: return launch_segl<SeglMixK2>(p, s, who);
        }
    }
    switch (refine_steps) {
        case 0: return launch_tile<0>(p, s, who);
        case 1: return launch_tile<1>(p, s, who);
        default: return launch_tile<2>(p, s, who);
    }
}

extern "C" int vx_tdma_adjoint_f64(void* stream, const double* a, const double* b, const double* c,
                                   const double* b_edge, const double* d_edge, const int32_t* kbot,
                                   int64_t kbot_sx, int64_t kbot_sy, const double* x, const double* gx,
                                   double* ga, double* gb, double* gc, double* gd, double* gb_edge,
                                   double* gd_edge, int64_t nx, int64_t ny, int32_t nz, int64_t sx, int64_t sy) {
    using namespace vx;
    const char* who = "vx_tdma_adjoint_f64";
    TdmaArgs p = make_args(a, b, c, gx, b_edge, d_edge, kbot, kbot_sx, kbot_sy, const_cast<double*>(x), nx, ny,
                           nz, sx, sy);
    int rc = validate_tdma(p, nx, ny, nz, who);
    if (rc != VX_OK || p.ncol == 0) return rc;
    if (!gx || !ga || !gb || !gc || !gd) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null gradient array", who);
    if ((b_edge != nullptr) != (gb_edge != nullptr) || (d_edge != nullptr) != (gd_edge != nullptr))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: gb_edge/gd_edge must be given exactly when b_edge/d_edge are",
                    who);
    TdmaAdjArgs q{p, gx, ga, gb, gc, gd, gb_edge, gd_edge};
    const TdmaTiling g = tdma_tiling(p);
    const int waves = kSegLdsBlock / 64;
    const dim3 grid((unsigned)((g.ntiles + waves - 1) / waves)), block(kSegLdsBlock);
    hipStream_t s = (hipStream_t)stream;
#define VX_ADJ_CASE(N) \
    case N: hipLaunchKernelGGL(tdma_adjoint_kernel<N>, grid, block, 0, s, q, g); break;
    switch (seg_levels(nz)) {
        VX_ADJ_CASE(2)
        VX_ADJ_CASE(4)
        VX_ADJ_CASE(6)
        VX_ADJ_CASE(8)
        VX_ADJ_CASE(10)
        VX_ADJ_CASE(12)
        VX_ADJ_CASE(14)
        VX_ADJ_CASE(16)
        default: return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, nz);
    }
#undef VX_ADJ_CASE
    return check_launch(who);
}
