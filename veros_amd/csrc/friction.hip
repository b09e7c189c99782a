// Implicit vertical friction of the horizontal velocity for gfx950 (float64):
// implicit_vert_friction, veros/core/friction.py:90-205.
//
// For each velocity face column of [1, X-2) x [1, Y-2) the reference builds a
// tridiagonal system from kappaM averaged onto the face (delta = dt_mom / dzw
// * fxa * maskU[k+1] * maskU[k], a = -delta[k-1] / dzt, b = 1 + delta[k-1] /
// dzt + delta[k] / dzt, c = -delta / dzt, the edge row b_edge = 1 + delta /
// dzt), solves it with solve_implicit over the wet suffix k >= max(kbot,
// kbot_next) - 1, stores the result at taup1, forms du_mix / dv_mix = (new -
// tau) / dt_mom over the face range, and adds the dissipation of the solve,
// interpolated onto the T grid, to K_diss_v.
//
// Here a group of 8 or 16 lanes owns a face column (col_tile.hpp): it forms its
// rows in registers from the face viscosity, solves, and the wave writes the new
// velocity on the wet levels and the tendency on every level; the face's
// dissipation is formed from the velocities still in registers (the level above
// from the next lane). A T cell's dissipation needs the u faces i-1 and i and the
// v faces j-1 and j, so a block owns a strip of T columns and walks a chunk of
// rows in order: the u faces of the previous row are kept in registers, and the v
// faces of the row pass through LDS. No face dissipation goes through memory.
#include "col_tile.hpp"

namespace vx {
namespace {

struct FricArgs {
    const int32_t* kbot;      // (X, Y)
    const double* dzt;        // (nz)
    const double* dzw;        // (nz)
    const double* dxt;        // (X)
    const double* dxu;        // (X)
    const double* area_t;     // (X, Y)
    const double* area_v;     // (X, Y)
    const double* kappaM;     // (X, Y, nz)
    double* vel[2];           // u, v (X, Y, nz, 3)
    double* dmix[2];          // du_mix, dv_mix (X, Y, nz)
    double* K_diss_v;         // (X, Y, nz)
    int64_t X, Y;
    int32_t nz, tau, taup1;
    double dt;
    // time levels of u, v: level l of cell c at l * ls + c * cs (cs = 3,
    // ls = 1: levels innermost; cs = 1, ls = X*Y*nz: levels outermost)
    int64_t cs, ls;
};

// The face of component t (0: u, between T columns i and i+1; 1: v, between
// rows j and j+1) is wet at level k iff both T columns are wet there:
// k >= max(kbot, kbot_next) - 1 with both kbot > 0 (maskU / maskV as
// veros/core/numerics.py:195-221 builds them from kbot). The solve runs over
// k >= max(kbot, kbot_next) - 1 whenever that maximum is positive
// (create_water_masks of the max, veros/core/friction.py:108-109, 158-159), so
// a face with one dry side is solved with delta = 0 and keeps tau's value.
struct Face {
    int k0;      // first level of the solve (nz: no solve)
    bool both;   // both T columns wet somewhere: the face mask is k >= k0
};

__device__ inline Face face_of(int kb0, int kb1, int nz) {
    const int kss = kb0 > kb1 ? kb0 : kb1;
    Face f;
    f.k0 = (kss >= 1 && kss <= nz) ? kss - 1 : nz;
    f.both = kb0 > 0 && kb1 > 0;
    return f;
}

// First wet level of a T column (nz: none).
__device__ __forceinline__ int first_wet_level(int kb, int nz) { return kb >= 1 && kb <= nz ? kb - 1 : nz; }

// The rows, the solve and the dissipation of a tile's faces of one component.
// In: flat, the face viscosity fx and tau's velocity x0 (on the solved levels); the
// lane's column: its first solved level k0, whether both T columns are wet. Out: flat,
// the solution x1 and the tendency dm; the lane's segment of the face's dissipation
// (:137-153, 189-201): fxa * (x1[k+1] - x1[k]) / dzw[k] * mask[k+1] * mask[k] times
// (x0[k+1] - x0[k]) / dzw[k], x0 at tau and x1 at taup1, 0 on the top level. The
// masks are 0 or 1, so the products are taken as selects. rzt, rztl, dtw, rzw2, rzw2l:
// 1 / dzt, dt / dzw and 1 / dzw^2, the reciprocals with what their rounding cuts off,
// in LDS: rows, tendency and dissipation are then rounded no more often than by the
// reference's divisions.
template <int S, int P>
__device__ __forceinline__ void fric_face(const Tile<S, P>& t, double* img, int nz, const double* __restrict__ rzt,
                                          const double* __restrict__ rztl, const double* __restrict__ dtw,
                                          const double* __restrict__ rzw2, const double* __restrict__ rzw2l, int k0,
                                          bool both, const Recip& rdt, const double (&fx)[S], const double (&x0)[S],
                                          double (&x1)[S], double (&dm)[S], double (&ds)[S]) {
    double f[S], o[S], va[S], vb[S], vc[S], z[1][S];
    tile_put(t, img, fx);
    seg_get(t, img, f);
    const double fm = seg_below(t, img);
    tile_put(t, img, x0);
    seg_get(t, img, o);
    // rows (veros/core/friction.py:111-126, 161-176)
    double dlm = (both && t.lo > k0 && t.lo < nz) ? dtw[t.lo - 1] * fm : 0.0;
#pragma unroll
    for (int q = 0; q < S; ++q) {
        const int k = t.lo + q;
        const bool wet = k >= k0 && k < nz;
        const int kc = k < nz ? k : nz - 1;
        const double rz = rzt[kc], rl = rztl[kc];
        const double dl = (both && wet && k < nz - 1) ? dtw[kc] * f[q] : 0.0;
        const double below = scaled(dlm, rz, rl), above = scaled(dl, rz, rl);
        va[q] = (wet && k != k0) ? -below : 0.0;
        vb[q] = wet ? (k == k0 ? 1 + above : (1 + below) + above) : 1.0;
        vc[q] = wet ? -above : 0.0;
        z[0][q] = wet ? o[q] : 0.0;
        dlm = dl;
    }
    col_solve<S, 1>(t, va, vb, vc, z);
    seg_put(t, img, z[0]);
    // level lo+S from the lane above (every lane takes part in the moves)
    const double zn = col_next<P>(t.s, z[0][0]), on = col_next<P>(t.s, o[0]);
#pragma unroll
    for (int q = 0; q < S; ++q) {
        const int k = t.lo + q;
        const double z1 = q < S - 1 ? z[0][q < S - 1 ? q + 1 : 0] : zn;
        const double o1 = q < S - 1 ? o[q < S - 1 ? q + 1 : 0] : on;
        const bool d = both && k >= k0 && k < nz - 1;
        ds[q] = d ? scaled((o1 - o[q]) * (f[q] * (z1 - z[0][q])), rzw2[d ? k : 0], rzw2l[d ? k : 0]) : 0.0;
    }
    tile_get(t, img, x1);
#pragma unroll
    for (int q = 0; q < S; ++q) z[0][q] = scaled(z[0][q] - o[q], rdt.h, rdt.l);
    seg_put(t, img, z[0]);
    tile_get(t, img, dm);
}

// A block owns a strip of T columns j and walks the rows of a chunk [ib, ie) in
// order, starting one row early for the u faces west of the chunk. Half of its
// waves solve the row's v faces, the other half its u faces, four or eight columns each, on
// column tiles (col_tile.hpp); the strip's first column is solved for its v face
// only. The v faces' dissipation goes through LDS to the u waves (two images per
// wave, one barrier per row), which keep that of the previous row's u faces and
// update K_diss_v. Each face is stored by exactly one block.
// K_diss_v += ugrid_to_tgrid(diss_u), then += vgrid_to_tgrid(diss_v)
// (veros/core/friction.py:154-155, 203-204; veros/core/numerics.py:313-336): at T cell
// (i, j) the u faces i and i-1 weighted dxu / (2 dxt) for 2 <= i < X-2 (face i alone
// for i = 1), the v faces j and j-1 weighted area_v / (2 area_t) for 2 <= j < Y-2
// (face j alone for j = 1), on the wet levels below the top one (no face of a dry
// cell dissipates). Blocks are XCD-contiguous, strips fastest.
//
// A row's chain (kbot, the loads, the solve through LDS) is what bounds it, with
// 5.1 GB on 1440x720x80 at 3.1 TB/s. What lies below the solve is loaded and stored
// before it, so that no flat value but the operands lives across it. Blocks of
// four waves: with eight, one block fills a CU's registers and nothing runs
// while it waits at its barrier (2.22 -> 2.68 ms for the vertical step there).
// Loading the next row ahead took the registers that hold a second block's waves
// (2.55 ms). Eight lanes per column, each loading and storing its own levels,
// and every row's divisions in the lane: friction 1.94 ms there, now 1.60; 163
// us on 360x160x60, levels innermost, now 92.
constexpr int kFricGroups = 2;                                // column groups of a block
constexpr int kFricBlock = 2 * 64 * kFricGroups;              // a u and a v wave for each
template <int P>
constexpr int kFricCols = kFricGroups * (64 / P) - 1;         // T columns of a strip
// waves per SIMD (and blocks per CU): what the registers allow, but two for four
// levels on 8 lanes (1435x896x32 849 us with three, 813 with two; 360x160x60, 16
// lanes, 92 with three, 104 with two)
template <int S, int P>
constexpr int kFricWaves = S <= 3 ? 4 : S == 4 && P == kTileP ? 3 : 2;
template <int S, int P>
__global__ __launch_bounds__(kFricBlock) __attribute__((amdgpu_waves_per_eu(kFricWaves<S, P>))) void friction_walk_kernel(
    FricArgs p, int rows, int64_t nstrips, int64_t nblocks, uint32_t rnz) {
    using T = Tile<S, P>;
    constexpr int G = kFricGroups;
    __shared__ double work[2 * G][T::IMG];
    __shared__ double dsv[2][G][T::IMG];
    __shared__ double sdz[5][kMaxNz];
    const int64_t b = xcd_contiguous_block();
    if (b >= nblocks) return;
    const int nz = p.nz;
    for (int k = threadIdx.x; k < nz; k += kFricBlock) {
        const double zw = p.dzw[k];
        const Recip rzt = recip(p.dzt[k]);
        sdz[0][k] = rzt.h;
        sdz[4][k] = rzt.l;
        sdz[1][k] = p.dt / zw;
        const double sq = zw * zw, r = 1.0 / sq;
        sdz[2][k] = r;
        sdz[3][k] = r * fma(-r, fma(zw, zw, -sq), fma(-r, sq, 1.0));
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const bool vface = wave < G;
    const int grp = vface ? wave : wave - G, comp = vface ? 1 : 0;
    double* const img = work[wave];
    const int64_t strip = b % nstrips, chunk = b / nstrips;
    const int64_t ib = 1 + (int64_t)rows * chunk;
    const int64_t ie = ib + rows < p.X - 2 ? ib + rows : p.X - 2;
    const int64_t j0 = kFricCols<P> * strip + T::C * grp;  // the wave's columns
    const int64_t left = p.Y - 2 - j0;
    const int n = left >= T::C ? T::C : (left > 0 ? (int)left : 0);
    const int64_t next = vface ? 1 : p.Y;  // the face's other column
    const uint32_t cs = (uint32_t)p.cs;
    const Recip rdt = recip(p.dt);
    double* const vel = p.vel[comp];
    T t = make_tile<S, P>(0, n, nz, (uint32_t)nz, rnz);
    const int64_t j = t.q < n ? j0 + t.q : (n > 0 ? j0 : 0);  // the lane's column
    const bool jlive = t.q < n && j >= 1, jown = jlive && (grp > 0 || t.q > 0);
    // the block's own elements: not the strip's first column, nor j = 0
    auto own = [&](int r) { return t.off[r] != kNoAccess && (grp > 0 || t.c[r] > 0); };
    double du[S];  // the previous row's u faces' dissipation
#pragma unroll
    for (int r = 0; r < S; ++r) du[r] = 0.0;
#pragma unroll 1
    for (int64_t i = ib >= 2 ? ib - 1 : ib; i < ie; ++i) {
        const bool pre = i < ib;
        const int64_t col = i * p.Y + j;
        t.cell0 = (i * p.Y + j0) * nz;
        double ds[S];
        int kb = 0;
        if (n > 0 && !(pre && vface)) {
            kb = p.kbot[col];
            const bool live = vface ? jlive : jown;
            const Face f = face_of(live ? kb : 0, live ? p.kbot[col + next] : 0, nz);
            const BufRsrc b0 = tile_buf(t, vel + p.tau * p.ls, 0, (int)cs);
            const BufRsrc b1 = tile_buf(t, vel + p.taup1 * p.ls, 0, (int)cs);
            const BufRsrc bd = tile_buf(t, p.dmix[comp]);
            double fx[S], kn[S], x0[S], x1[S];
            uint32_t on[S];  // the solved levels
#pragma unroll
            for (int r = 0; r < S; ++r) on[r] = t.k[r] >= __shfl(f.k0, t.c[r] * P) ? t.off[r] : kNoAccess;
            tile_load(tile_buf(t, p.kappaM), on, 1, fx);
            tile_load(tile_buf(t, p.kappaM, next * nz), on, 1, kn);
            tile_load(b0, on, cs, x0);
#pragma unroll
            for (int r = 0; r < S; ++r) on[r] = own(r) && !pre ? on[r] : kNoAccess;
            if (!pre) {  // below the solve taup1 keeps its value
                double y0[S], dm[S];
                uint32_t below[S];
#pragma unroll
                for (int r = 0; r < S; ++r) below[r] = own(r) && on[r] == kNoAccess ? t.off[r] : kNoAccess;
                tile_load(b0, below, cs, y0);
                tile_load(b1, below, cs, dm);
#pragma unroll
                for (int r = 0; r < S; ++r) dm[r] = scaled(dm[r] - y0[r], rdt.h, rdt.l);
                tile_store(bd, below, 1, dm);
            }
#pragma unroll
            for (int r = 0; r < S; ++r) fx[r] = 0.5 * (fx[r] + kn[r]);
            fric_face<S, P>(t, img, nz, sdz[0], sdz[4], sdz[1], sdz[2], sdz[3], f.k0, f.both, rdt, fx, x0, x1, kn, ds);
            if (vface) seg_put(t, dsv[i & 1][grp], ds);
            tile_store(b1, on, cs, x1);
            tile_store(bd, on, 1, kn);
        }
        if (vface || n == 0) {
            if (!pre) __syncthreads();
            continue;
        }
        double bu[S];
        {
            const double wi = p.dxu[i], wm = p.dxu[i - 1];
            const Recip rden = recip(2 * p.dxt[i]);
#pragma unroll
            for (int r = 0; r < S; ++r) {
                bu[r] = i >= 2 ? scaled(wi * ds[r] + wm * du[r], rden.h, rden.l) : ds[r];
                du[r] = ds[r];
            }
        }
        if (pre) continue;  // uniform in the block
        // K_diss_v and the weights are loaded before the barrier, which their
        // latency then overlaps
        const BufRsrc bK = tile_buf(t, p.K_diss_v);
        double K[S], wj = 1.0, wjm = 0.0;
        Recip rden{1.0, 0.0};
        uint32_t ow[S];
        const int wc = jown ? first_wet_level(kb, nz) : nz;
#pragma unroll
        for (int r = 0; r < S; ++r)
            ow[r] = t.k[r] >= __shfl(wc, t.c[r] * P) && t.k[r] < nz - 1 ? t.off[r] : kNoAccess;
        tile_load(bK, ow, 1, K);
        const bool south = jown && j >= 2;
        if (south) {
            rden = recip(2 * p.area_t[col]);
            wj = p.area_v[col];
            wjm = p.area_v[col - 1];
        }
        __syncthreads();
        // the v faces of the lane's column and of the column south, which may be
        // the last of the wave before
        const double* vn = dsv[i & 1][grp];
        const double* vs = t.q > 0 ? vn - T::CS : dsv[i & 1][grp > 0 ? grp - 1 : 0] + (T::C - 1) * T::CS;
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const double dn = vn[t.seg + r], dd = vs[t.seg + r];
            bu[r] = bu[r] + (south ? scaled(wj * dn + wjm * dd, rden.h, rden.l) : dn);
        }
        seg_put(t, img, bu);
        tile_get(t, img, bu);
#pragma unroll
        for (int r = 0; r < S; ++r) buf_store(bK, ow[r], K[r] + bu[r]);
    }
}

// Rows per block of the walk kernel. A block walks `rows` rows and one extra row of
// u faces, and a launch of n blocks takes about ceil(n / slots) passes of rows + 1
// rows; the row count with the cheapest product is taken (at most 24: longer
// chunks leave the last pass emptier than the row they save). With 24 rows
// whatever the grid, an earlier form of the kernel launched 96 blocks for 256 CUs
// on 360x160x60: 459 us, 163 us with the rows chosen here.
int fric_rows(int64_t nrows, int64_t nstrips, int blocks_per_cu) {
    const int64_t slots = (int64_t)blocks_per_cu * cu_count();
    int best = 1;
    int64_t best_cost = INT64_MAX;
    for (int rows = 1; rows <= 24; ++rows) {
        const int64_t nblocks = nstrips * ((nrows + rows - 1) / rows);
        const int64_t cost = (nblocks + slots - 1) / slots * (rows + 1);
        if (cost <= best_cost) {
            best_cost = cost;
            best = rows;
        }
    }
    return best;
}

template <int S, int P>
void launch_fric_walk(const FricArgs& p, hipStream_t s) {
    const int64_t nstrips = (p.Y - 3 + kFricCols<P> - 1) / kFricCols<P>;
    const int rows = fric_rows(p.X - 3, nstrips, kFricWaves<S, P>);
    const int64_t nblocks = nstrips * ((p.X - 3 + rows - 1) / rows);
    hipLaunchKernelGGL((friction_walk_kernel<S, P>), dim3((unsigned)((nblocks + 7) / 8 * 8)), dim3(kFricBlock), 0, s, p,
                       rows, nstrips, nblocks, depth_reciprocal(p.nz));
}

}  // namespace
}  // namespace vx

extern "C" int vx_implicit_vert_friction_f64(void* stream, const vx_grid* grid, double dt_mom, double* u, double* v,
                                             int32_t tau, int32_t taup1, const double* kappaM, const double* area_t,
                                             const double* area_v, double* du_mix, double* dv_mix,
                                             double* K_diss_v) {
    using namespace vx;
    const char* who = "vx_implicit_vert_friction_f64";
    if (!grid) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid", who);
    if (grid->nx < 1 || grid->ny < 1 || grid->nz < 1)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: bad shape nx=%lld ny=%lld nz=%d", who, (long long)grid->nx,
                    (long long)grid->ny, grid->nz);
    if (grid->nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d too deep (max %d)", who, grid->nz, kMaxNz);
    if (!grid->kbot || !grid->dzt || !grid->dzw || !grid->dxt || !grid->dxu)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid array", who);
    if (tau < 0 || tau > 2 || taup1 < 0 || taup1 > 2 || tau == taup1)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: tau and taup1 must be distinct levels in 0..2", who);
    if (!u || !v || !kappaM || !area_t || !area_v || !du_mix || !dv_mix || !K_diss_v)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if (u == v || du_mix == dv_mix || (const double*)K_diss_v == kappaM || K_diss_v == du_mix || K_diss_v == dv_mix)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: u/v, du_mix/dv_mix and K_diss_v must be distinct arrays", who);
    if (!(dt_mom > 0.0)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: dt_mom must be positive", who);
    FricArgs p{};
    p.kbot = grid->kbot;
    p.dzt = grid->dzt;
    p.dzw = grid->dzw;
    p.dxt = grid->dxt;
    p.dxu = grid->dxu;
    p.area_t = area_t;
    p.area_v = area_v;
    p.kappaM = kappaM;
    p.vel[0] = u;
    p.vel[1] = v;
    p.dmix[0] = du_mix;
    p.dmix[1] = dv_mix;
    p.K_diss_v = K_diss_v;
    p.X = grid->nx + 4;
    p.Y = grid->ny + 4;
    p.nz = grid->nz;
    p.tau = tau;
    p.taup1 = taup1;
    p.dt = dt_mom;
    if (grid->time_layout != VX_LEVELS_INNER && grid->time_layout != VX_LEVELS_OUTER)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: time_layout must be VX_LEVELS_INNER or VX_LEVELS_OUTER", who);
    const bool outer = grid->time_layout == VX_LEVELS_OUTER;
    p.cs = outer ? 1 : 3;
    p.ls = outer ? p.X * p.Y * p.nz : 1;
    hipStream_t s = (hipStream_t)stream;
    if (col_lanes(p.nz) == kSegP) {
        switch (col_levels(p.nz)) {
            case 2: launch_fric_walk<2, kSegP>(p, s); break;
            case 3: launch_fric_walk<3, kSegP>(p, s); break;
            default: launch_fric_walk<4, kSegP>(p, s); break;
        }
    } else {
        switch (col_levels(p.nz)) {
            case 3: launch_fric_walk<3, kTileP>(p, s); break;
            case 4: launch_fric_walk<4, kTileP>(p, s); break;
            case 5: launch_fric_walk<5, kTileP>(p, s); break;
            case 6: launch_fric_walk<6, kTileP>(p, s); break;
            case 7: launch_fric_walk<7, kTileP>(p, s); break;
            default: launch_fric_walk<8, kTileP>(p, s); break;
        }
    }
    return check_launch(who);
}
