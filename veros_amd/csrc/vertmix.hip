// Implicit vertical mixing of temperature and salinity for gfx950 (float64):
// vertmix_tempsalt, veros/core/thermodynamics.py:248-300.
//
// The reference builds the tridiagonal system of each interior column from
// kappaH and the vertical grid (delta = dt / dzw * kappaH, a = -delta[k-1] /
// dzt, b = 1 + (delta[k] + delta[k-1]) / dzt, c = -delta / dzt, the edge row
// b_edge = 1 + delta / dzt), adds the surface forcing to the top level of the
// right-hand side, solves it with solve_implicit for temp and for salt, and
// then forms the tendencies (new - old) / dt over the whole array and copies
// the cyclic x halos.
//
// Here a group of 8 or 16 lanes owns a column (col_tile.hpp): it forms the rows in
// registers, solves temperature and salinity with one factorisation, and the
// wave writes the new tracers on the wet levels and both tendencies on every
// level. The coefficients never touch memory: the kernel reads kappaH and the
// two tracer columns once and writes them and the tendencies once.
#include "col_tile.hpp"

namespace vx {
namespace {

struct VmixArgs {
    const int32_t* kbot;      // (X, Y)
    const double* dzt;        // (nz)
    const double* dzw;        // (nz)
    const double* kappaH;     // (X, Y, nz)
    double* tr[2];            // temp, salt (X, Y, nz, 3)
    const double* forc[2];    // forc_temp_surface, forc_salt_surface (X, Y)
    double* dvmix[2];         // dtemp_vmix, dsalt_vmix (X, Y, nz)
    int64_t X, Y;
    int32_t nz, taup1;
    double dt;
    // time levels of temp/salt: level l of cell c at l * ls + c * cs (cs = 3,
    // ls = 1: levels innermost; cs = 1, ls = X*Y*nz: levels outermost)
    int64_t cs, ls;
};

// 1 / dzt (s[0, nz)), the rest of its rounding (from kMaxNz on) and dt / dzw (from
// 2 kMaxNz on) in LDS; every thread of the block calls it. The rows read them
// inside per-level selects, where a global load is waited for at once, level after level.
__device__ __forceinline__ void vmix_stage_dz(const VmixArgs& p, double* s) {
    for (int k = threadIdx.x; k < p.nz; k += blockDim.x) {
        const Recip r = recip(p.dzt[k]);
        s[k] = r.h;
        s[kMaxNz + k] = r.l;
        s[2 * kMaxNz + k] = p.dt / p.dzw[k];
    }
    __syncthreads();
}

// The rows of the lane's levels (veros/core/thermodynamics.py:267-277),
// identity rows off the wet suffix. KM(k) is kappaH at level k of the column, for
// k in [lo-1, lo+S); its value matters for k0 <= k < nz-1 only. rzt, rztl, dtw:
// 1 / dzt with its rest and dt / dzw (in LDS): every entry rounds as with the
// reference's divisions.
template <int S, class KMF>
__device__ __forceinline__ void vmix_rows(const VmixArgs& p, const double* __restrict__ rzt,
                                          const double* __restrict__ rztl, const double* __restrict__ dtw,
                                          const SegLane& L, KMF KM, double (&va)[S], double (&vb)[S], double (&vc)[S]) {
    const int nz = p.nz;
    const int kp = L.lo - 1;  // delta at the level below the segment
    double dlm = (kp >= L.k0 && kp < nz - 1) ? dtw[kp > 0 ? kp : 0] * KM(kp) : 0.0;
#pragma unroll
    for (int t = 0; t < S; ++t) {
        const int k = L.lo + t;
        const bool wet = k >= L.k0 && k < nz;
        const int kc = k < nz ? k : nz - 1;
        const double rz = rzt[kc], rl = rztl[kc];
        const double dl = (wet && k < nz - 1) ? dtw[kc] * KM(k) : 0.0;
        const bool edge = k == L.k0;
        va[t] = (wet && !edge) ? -scaled(dlm, rz, rl) : 0.0;
        vb[t] = wet ? 1 + scaled(edge ? dl : dl + dlm, rz, rl) : 1.0;
        vc[t] = (wet && k < nz - 1) ? -scaled(dl, rz, rl) : 0.0;
        dlm = dl;
    }
}

// Column tiles (any layout, depth and alignment): a wave's columns are loaded
// flat, the two tracers' old values stay with the lanes that loaded them, and
// everything goes back flat. Bound by HBM: on 1440x720x80, levels outermost, 2.6 GB
// in 0.60 ms (8 lanes per column with 16-byte copies into LDS: 0.60); 360x160x60,
// levels innermost, 71 -> 46 us against each lane loading its own levels.
constexpr int kVmixBlock = 128;
template <int S, int P>
__global__ __launch_bounds__(kVmixBlock) void vertmix_tile_kernel(VmixArgs p, uint32_t rnz) {
    using T = Tile<S, P>;
    __shared__ double sdz[3 * kMaxNz];
    __shared__ double lds[kVmixBlock / 64][T::IMG];
    vmix_stage_dz(p, sdz);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), nz = p.nz;
    double* const img = lds[wave];
    const int64_t col0 = ((int64_t)blockIdx.x * (kVmixBlock / 64) + wave) * T::C;
    const int64_t left = p.X * p.Y - col0;
    if (left <= 0) return;  // uniform in the wave; no barrier follows
    const int n = left >= T::C ? T::C : (int)left;
    const T t = make_tile<S, P>(col0 * nz, n, nz, (uint32_t)nz, rnz);
    SegLane L;
    L.s = t.s;
    L.lo = t.lo;
    L.valid = t.q < n;
    L.base = 0;
    const int64_t col = L.valid ? col0 + t.q : col0;
    const int64_t i = col / p.Y, j = col - i * p.Y;
    const bool interior = L.valid && i >= 2 && i < p.X - 2 && j >= 2 && j < p.Y - 2;
    const int kb = p.kbot[col];
    const double fT = p.forc[0][col], fS = p.forc[1][col];
    L.k0 = interior && kb >= 1 && kb <= nz ? kb - 1 : nz;
    const uint32_t cs = (uint32_t)p.cs;
    const BufRsrc bT = tile_buf(t, p.tr[0] + p.taup1 * p.ls, 0, (int)cs);
    const BufRsrc bS = tile_buf(t, p.tr[1] + p.taup1 * p.ls, 0, (int)cs);
    uint32_t wet[S];
    double oT[S], oS[S], nT[S], nS[S];
#pragma unroll
    for (int r = 0; r < S; ++r) {
        wet[r] = t.k[r] >= __shfl(L.k0, t.c[r] * P) ? t.off[r] : kNoAccess;
        nT[r] = nS[r] = 0.0;
    }
    // a tracer's right-hand sides: its old values and the surface forcing (:277, :284)
    auto rhs = [&](const double(&old)[S], double forc, double(&z)[S]) {
        const double ftop = scaled(p.dt * forc, sdz[nz - 1], sdz[kMaxNz + nz - 1]);
        double x[S];
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const double f = __shfl(ftop, t.c[r] * P);
            x[r] = t.k[r] == nz - 1 ? old[r] + f : old[r];
        }
        tile_put(t, img, x);
        seg_get(t, img, z);
#pragma unroll
        for (int r = 0; r < S; ++r) z[r] = L.lo + r >= L.k0 && L.lo + r < nz ? z[r] : 0.0;
    };
    if (__any(L.k0 < nz)) {
        double km[S + 1], va[S], vb[S], vc[S], z[2][S];
        {
            double kv[S];
            tile_load(tile_buf(t, p.kappaH), wet, 1, kv);
            tile_load(bT, wet, cs, oT);
            tile_load(bS, wet, cs, oS);
            tile_put(t, img, kv);
            seg_get(t, img, kv);
            km[0] = seg_below(t, img);
#pragma unroll
            for (int r = 0; r < S; ++r) km[r + 1] = kv[r];
        }
        vmix_rows<S>(p, sdz, sdz + kMaxNz, sdz + 2 * kMaxNz, L, [&](int k) { return km[k - L.lo + 1]; }, va, vb, vc);
        rhs(oT, fT, z[0]);
        rhs(oS, fS, z[1]);
        col_solve<S, 2>(t, va, vb, vc, z);
        seg_put(t, img, z[0]);
        tile_get(t, img, nT);
        seg_put(t, img, z[1]);
        tile_get(t, img, nS);
        tile_store(bT, wet, cs, nT);
        tile_store(bS, wet, cs, nS);
        const Recip rdt = recip(p.dt);
#pragma unroll
        for (int r = 0; r < S; ++r) {  // (new - old) / dt; 0 where unchanged
            nT[r] = wet[r] != kNoAccess ? scaled(nT[r] - oT[r], rdt.h, rdt.l) : 0.0;
            nS[r] = wet[r] != kNoAccess ? scaled(nS[r] - oS[r], rdt.h, rdt.l) : 0.0;
        }
    }
    tile_store(tile_buf(t, p.dvmix[0]), t.off, 1, nT);
    tile_store(tile_buf(t, p.dvmix[1]), t.off, 1, nS);
}

// enforce_boundaries on one process (veros/core/utilities.py:7-21): the x
// halos of level taup1, arr[-2:] = arr[2:4] and arr[:2] = arr[-4:-2].
__global__ __launch_bounds__(256) void vertmix_cyclic_kernel(VmixArgs p) {
    const int64_t plane = p.Y * p.nz;  // one x row of a level
    const int64_t n = 2 * 4 * plane;   // tracers x halo rows x row
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int t = (int)(e / (4 * plane));
    const int64_t r = e - (int64_t)t * 4 * plane;
    const int h = (int)(r / plane);  // halo row 0, 1, X-2, X-1
    const int64_t off = r - (int64_t)h * plane;
    const int64_t dst = h < 2 ? h : p.X - 4 + h;
    const int64_t src = h < 2 ? p.X - 4 + h : 2 + (h - 2);
    double* __restrict__ tr = p.tr[t] + p.taup1 * p.ls;
    tr[p.cs * (dst * plane + off)] = tr[p.cs * (src * plane + off)];
}

template <int S, int P>
void launch_vmix(const VmixArgs& p, hipStream_t s) {
    const int64_t threads = (p.X * p.Y + 64 / P - 1) / (64 / P) * 64;
    hipLaunchKernelGGL((vertmix_tile_kernel<S, P>), dim3((unsigned)((threads + kVmixBlock - 1) / kVmixBlock)),
                       dim3(kVmixBlock), 0, s, p, depth_reciprocal(p.nz));
}

}  // namespace
}  // namespace vx

extern "C" int vx_vertmix_tempsalt_f64(void* stream, const vx_grid* grid, double dt_tracer, double* temp,
                                       double* salt, int32_t taup1, const double* kappaH,
                                       const double* forc_temp_surface, const double* forc_salt_surface,
                                       double* dtemp_vmix, double* dsalt_vmix, int32_t enable_cyclic_x) {
    using namespace vx;
    const char* who = "vx_vertmix_tempsalt_f64";
    if (!grid) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid", who);
    if (grid->nx < 1 || grid->ny < 1 || grid->nz < 1)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: bad shape nx=%lld ny=%lld nz=%d", who, (long long)grid->nx,
                    (long long)grid->ny, grid->nz);
    if (grid->nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d too deep (max %d)", who, grid->nz, kMaxNz);
    if (!grid->kbot || !grid->dzt || !grid->dzw) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid array", who);
    if (taup1 < 0 || taup1 > 2) return fail(VX_ERR_INVALID_ARGUMENT, "%s: taup1 must be 0..2", who);
    if (!temp || !salt || !kappaH || !forc_temp_surface || !forc_salt_surface || !dtemp_vmix || !dsalt_vmix)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if (temp == salt || dtemp_vmix == dsalt_vmix)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: temp/salt and their tendencies must be distinct arrays", who);
    if (!(dt_tracer > 0.0)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: dt_tracer must be positive", who);
    // the halo copy runs as one parallel pass; its source and destination rows
    // are disjoint from nx = 4 on (the reference copies them one after the other)
    if (enable_cyclic_x && grid->nx < 4)
        return fail(VX_ERR_UNSUPPORTED, "%s: cyclic x needs nx >= 4 (nx=%lld)", who, (long long)grid->nx);
    VmixArgs p{};
    p.kbot = grid->kbot;
    p.dzt = grid->dzt;
    p.dzw = grid->dzw;
    p.kappaH = kappaH;
    p.tr[0] = temp;
    p.tr[1] = salt;
    p.forc[0] = forc_temp_surface;
    p.forc[1] = forc_salt_surface;
    p.dvmix[0] = dtemp_vmix;
    p.dvmix[1] = dsalt_vmix;
    p.X = grid->nx + 4;
    p.Y = grid->ny + 4;
    p.nz = grid->nz;
    p.taup1 = taup1;
    p.dt = dt_tracer;
    if (grid->time_layout != VX_LEVELS_INNER && grid->time_layout != VX_LEVELS_OUTER)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: time_layout must be VX_LEVELS_INNER or VX_LEVELS_OUTER", who);
    const bool outer = grid->time_layout == VX_LEVELS_OUTER;
    p.cs = outer ? 1 : 3;
    p.ls = outer ? p.X * p.Y * p.nz : 1;
    hipStream_t s = (hipStream_t)stream;
    if (col_lanes(p.nz) == kSegP) {
        switch (col_levels(p.nz)) {
            case 2: launch_vmix<2, kSegP>(p, s); break;
            case 3: launch_vmix<3, kSegP>(p, s); break;
            default: launch_vmix<4, kSegP>(p, s); break;
        }
    } else {
        switch (col_levels(p.nz)) {
            case 3: launch_vmix<3, kTileP>(p, s); break;
            case 4: launch_vmix<4, kTileP>(p, s); break;
            case 5: launch_vmix<5, kTileP>(p, s); break;
            case 6: launch_vmix<6, kTileP>(p, s); break;
            case 7: launch_vmix<7, kTileP>(p, s); break;
            default: launch_vmix<8, kTileP>(p, s); break;
        }
    }
    int rc = check_launch(who);
    if (rc) return rc;
    if (enable_cyclic_x) {
        const int64_t n = 2 * 4 * p.Y * p.nz;
        hipLaunchKernelGGL(vertmix_cyclic_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p);
        rc = check_launch(who);
    }
    return rc;
}
