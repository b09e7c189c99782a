// Implicit vertical integration of TKE, EKE and internal-wave energy on
// gfx950: integrate_tke_kernel (veros/core/tke.py:123-321),
// integrate_eke_kernel (veros/core/eke.py:93-255) and integrate_idemix_kernel
// (veros/core/idemix.py:47-265), without their advection branches.
//
// One kernel per model. A wave owns a tile of four or eight columns of the whole (X, Y)
// grid (col_tile.hpp): it loads its cells flat and coalesced, sums the forcing
// terms and forms the right-hand side and the dissipation coefficient cell by
// cell, passes those and the diffusivity through LDS to the segment layout,
// where the rows of the implicit system are formed (delta from the diffusivity
// at k and k+1, the edge row at kbot-1) and the columns solved, and takes the
// solution back through LDS to store, cell by cell, the new energy at taup1 on
// the wet levels of the interior columns, the dissipation diagnostic over the
// whole array and the lateral diffusion of the tau level on top (its fluxes
// read the four neighbouring columns, cells whose face is wet only). Halo
// columns only produce the diagnostics. Masks come from kbot (maskT = maskW =
// wet suffix, maskU / maskV the products of the two adjacent maskT).
//
// What bounds the three: the chain of memory round trips of a wave (kbot, the
// arrays, the lateral neighbours), behind it HBM. The earlier kernels (8 lanes
// per column, each lane loading its own levels, two waves per SIMD, a scalar
// variant for odd nz or levels innermost) took, TKE + EKE + IDEMIX together,
// 4.91 ms on 1440x720x80 (levels outermost), these 4.13; on 360x160x45 (odd,
// levels innermost) 336 -> 189 us; 700x400x75, innermost, 2.55 -> 1.28 ms. Of
// the 4.1 ms the lateral terms cost 1.1, the forcing terms 0.8, the solve 0.2.
#include "col_tile.hpp"

namespace vx {

constexpr int kMaxTerms = 12;
// threads per block of the three kernels; a constant, since reading the
// block size at run time costs a memory round trip at the start of every wave
constexpr int kTurbBlock = 256;

struct TurbGrid {
    const int32_t* kbot;
    const double *dxt, *dxu, *dyt, *dyu, *cost, *cosu, *dzt, *dzw;
    int32_t X, Y, nz;
    int64_t cs, ls;  // time levels: level l of cell c at l * ls + c * cs
};

// forcing = sgn[0] * p[0] + sgn[1] * p[1] + ... , summed left to right
struct Terms {
    const double* p[kMaxTerms];
    double sgn[kMaxTerms];
    int n;
};

// The lateral faces of a tile's columns: east, west, north, south.
struct TurbCols {
    double w[64 / kSegP][4];  // weights
    int face[64 / kSegP][4];  // first level at which the face is wet (nz: none)
};

// Level tables of a block: dd[k] = the diffusivity's factor in delta at level k
// (0 on the top level), rz[k], rl[k] = 1 / dzw (1 / (0.5 dzw) on the top level) and its
// rounding's rest, with which the rows round as with the reference's divisions.
struct TurbLevels {
    double dd[kMaxNz], rz[kMaxNz], rl[kMaxNz], zw[kMaxNz];
};

__device__ __forceinline__ int first_wet_of(int kb, int nz) { return kb >= 1 && kb <= nz ? kb - 1 : nz; }

// The wave's tile: columns [col0, col0 + 64 / P) of the X * Y, in order.
template <int P>
__device__ __forceinline__ int64_t turb_col0(int wave) {
    return (xcd_contiguous_block() * (kTurbBlock / 64) + wave) * (64 / P);
}
template <int S, int P>
__device__ __forceinline__ Tile<S, P> turb_tile(const TurbGrid& g, int64_t col0) {
    const int64_t left = (int64_t)g.X * g.Y - col0;
    const int n = left >= 64 / P ? 64 / P : (left > 0 ? (int)left : 0);
    return make_tile<S, P>(n > 0 ? col0 * g.nz : 0, n, g.nz, (uint32_t)g.nz, depth_reciprocal(g.nz));
}

// The lane's group column (segments): what the masks need, known before the
// first load is issued.
struct TurbLane {
    int i, j;
    bool interior;
    int kw, k0;  // first wet and first solved level (nz: none)
};
template <int S, int P>
__device__ __forceinline__ TurbLane turb_lane(const TurbGrid& g, const Tile<S, P>& t, int64_t col0) {
    TurbLane l;
    const bool valid = t.q < t.ncol;
    const int64_t col = valid ? col0 + t.q : 0;
    const int kb = g.kbot[col];
    l.i = (int)(col / g.Y);
    l.j = (int)(col - (int64_t)l.i * g.Y);
    l.interior = valid && l.i >= 2 && l.i < g.X - 2 && l.j >= 2 && l.j < g.Y - 2;
    l.kw = valid ? first_wet_of(kb, g.nz) : g.nz;
    l.k0 = l.interior ? l.kw : g.nz;
    return l;
}

// Fills the block's level tables (scale = dt * coefficient) and the wave's
// columns; every thread of the block calls it, after it has issued its first
// loads (whose latency the divisions here hide). `lateral`: the weights times
// `lw` and the faces are wanted.
template <int S, int P>
__device__ __forceinline__ void turb_setup(const TurbGrid& g, const Tile<S, P>& t, const TurbLane& l, double scale,
                                           double lw, bool lateral, TurbLevels& lv, TurbCols& tc) {
    const int nz = g.nz;
    for (int k = threadIdx.x; k < nz; k += kTurbBlock) {
        const double dzw = g.dzw[k];
        lv.zw[k] = dzw;
        const Recip r = recip(k == nz - 1 ? 0.5 * dzw : dzw);
        lv.rz[k] = r.h;
        lv.rl[k] = r.l;
        lv.dd[k] = k < nz - 1 ? scale / g.dzt[k + 1] * 0.5 : 0.0;
    }
    if (lateral) {
        // div = (fe - fw) / (cost dxt) + (fn - fs) / (cost dyt) with fe = ce (F(i+1) - F(i)) / (cost dxu),
        // fn = cn (F(j+1) - F(j)) / dyu cosu: one factor per face; lane s < 4 of a column forms face s
        // (east, west, north, south)
        const bool on = l.interior && l.kw < nz;
        const int ii = on ? l.i : 1, jj = on ? l.j : 1, f = t.s & 3;
        const double cost = g.cost[jj];
        const int io = f == 1 ? ii - 1 : ii, jo = f == 3 ? jj - 1 : jj;
        // the products' roundings are carried along, so that a weight is rounded once
        const double p0 = cost * (f < 2 ? g.dxt[ii] : g.dyt[jj]), l0 = fma(cost, f < 2 ? g.dxt[ii] : g.dyt[jj], -p0);
        const double m1 = f < 2 ? cost : 1.0, m2 = f < 2 ? g.dxu[io] : g.dyu[jo], p1 = m1 * m2, l1 = fma(m1, m2, -p1);
        const double den = p0 * p1, denl = fma(p0, p1, -den) + (p0 * l1 + l0 * p1);
        const double cu = f < 2 ? 1.0 : g.cosu[jo], num = lw * cu, numl = fma(lw, cu, -num);
        const double wq = num / den;
        const int64_t cc = (int64_t)ii * g.Y + jj;
        const int kn = first_wet_of(g.kbot[cc + (f == 0 ? g.Y : (f == 1 ? -g.Y : (f == 2 ? 1 : -1)))], nz);
        if (t.s < 4) {
            tc.w[t.q][f] = wq + (fma(-wq, den, num) + (numl - wq * denl)) / den;
            tc.face[t.q][f] = on ? (kn > l.kw ? kn : l.kw) : nz;
        }
    }
    __syncthreads();
}

// Adds the lateral diffusion of the tau level (veros/core/tke.py:250-276;
// eke.py:168-200; idemix.py:186-218) to v on the cells with a wet face:
// sum over the faces of weight * coefficient * (F(neighbour) - F(cell)).
// F and the coefficient come from the arrays A and B (one or two of them):
// COMB(face values of the neighbour's A and B, the cell's a and b) returns
// coefficient * difference. Two directions at a time, so that the loads of a
// pair are in flight together and hold few registers. The kernels store their
// diagnostics after it: a load waits for the stores issued before it (the three
// models on 1440x720x80: 4.13 -> 4.10 ms).
template <int S, bool TWO, int P, class COMB>
__device__ __forceinline__ void add_lateral(const TurbGrid& g, const Tile<S, P>& t, const TurbCols& tc, const double* A,
                                            uint32_t csA, const double* B, const double (&a)[S],
                                            const double (&b)[TWO ? S : 1], COMB comb, double (&v)[S]) {
    const int64_t nz = g.nz, row = (int64_t)g.Y * nz;
    const int64_t d[4] = {row, -row, nz, -nz};
    // the faces' terms are summed first and rounded into v once (one after the other
    // they made TKE's mean error 1.2 times that of float64 in the reference's order,
    // summed first 1.1); in pairs where the sum's registers would spill
    constexpr bool PAIRS = TWO && S == 6;
    double sum[S];
#pragma unroll
    for (int h = 0; h < 4; h += 2) {
        double nA[2][S], nB[2][TWO ? S : 1];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const BufRsrc ra = tile_buf(t, A, d[h + f], (int)csA);
            const BufRsrc rb = tile_buf(t, TWO ? B : A, d[h + f]);
#pragma unroll
            for (int r = 0; r < S; ++r) {
                const uint32_t o = t.k[r] >= tc.face[t.c[r]][h + f] ? t.off[r] : kNoAccess;
                nA[f][r] = buf_load(ra, o * csA);
                if constexpr (TWO) nB[f][r] = buf_load(rb, o);
            }
        }
#pragma unroll
        for (int f = 0; f < 2; ++f) {
#pragma unroll
            for (int r = 0; r < S; ++r) {
                const double x = tc.w[t.c[r]][h + f] * comb(nA[f][r], TWO ? nB[f][TWO ? r : 0] : 0.0, a[r], TWO ? b[TWO ? r : 0] : 0.0);
                const double y = t.k[r] >= tc.face[t.c[r]][h + f] ? x : 0.0;
                sum[r] = f == 0 && (PAIRS || h == 0) ? y : sum[r] + y;
            }
        }
        if (PAIRS || h == 2) {
#pragma unroll
            for (int r = 0; r < S; ++r) v[r] += sum[r];
        }
    }
}

#ifndef VX_TERMS_GROUP
#define VX_TERMS_GROUP 3
#endif
// f plus the signed forcing terms on the cells of `off`, summed left to right;
// with `first` the sum replaces f. VX_TERMS_GROUP terms are loaded at a time,
// before the group's first use.
template <int S, int P>
__device__ __forceinline__ void add_terms(const Terms& T, const Tile<S, P>& t, const uint32_t (&off)[S], bool first,
                                          double (&f)[S]) {
    constexpr int G = VX_TERMS_GROUP;
    for (int q0 = 0; q0 < T.n; q0 += G) {
        double v[G][S];
#pragma unroll
        for (int r = 0; r < G; ++r) {
            if (q0 + r < T.n) tile_load(tile_buf(t, T.p[q0 + r]), off, 1, v[r]);
        }
#pragma unroll
        for (int r = 0; r < G; ++r) {
            if (q0 + r < T.n) {
                const double sg = T.sgn[q0 + r];
                const bool set = first && q0 + r == 0;
#pragma unroll
                for (int x = 0; x < S; ++x) f[x] = set ? sg * v[r][x] : f[x] + sg * v[r][x];
            }
        }
    }
}

// Forms and solves the group columns' systems: kap, diss (the diagonal's
// dissipation) and rhs images in, the solution into the rhs image. MUL (IDEMIX):
// the rows are scaled by kap at their own column's level,
// a = -delta[k-1] kap[k-1], b = 1 + (delta[k] + delta[k-1]) kap[k], c = -delta[k] kap[k+1].
template <int S, bool MUL, int P>
__device__ __forceinline__ void turb_solve(const Tile<S, P>& t, const TurbLevels& lv, int nz, int k0, const double* kap,
                                           const double* diss, double* rhs) {
    double km[S], va[S], vb[S], vc[S], z[1][S];
    seg_get(t, kap, km);
    seg_get(t, diss, vb);
    seg_get(t, rhs, z[0]);
    const double below = seg_below(t, kap), above = seg_above(t, kap);
    const int kp = t.lo - 1;
    double dm = kp >= k0 && kp < nz - 1 ? lv.dd[kp] * (below + km[0]) : 0.0;
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const int k = t.lo + r;
        const bool wet = k >= k0 && k < nz;
        const int kc = k < nz ? k : nz - 1;
        const double kn = r < S - 1 ? km[r < S - 1 ? r + 1 : r] : above;
        const double kb = r > 0 ? km[r > 0 ? r - 1 : 0] : below;
        const double dk = wet && k < nz - 1 ? lv.dd[kc] * (km[r] + kn) : 0.0;
        const bool edge = k == k0;
        double A, B, C;
        if constexpr (MUL) {
            // entries of 1e7 around a row sum of about 1: formed in the
            // reference's order (veros/core/idemix.py:134-153), since every
            // other rounding of them moves the solution as much as another
            // elimination order would
            const double zw = lv.zw[kc];
            if (k < nz - 1) {
                A = -dm * kb / zw;
                B = edge ? 1 + dk / zw * km[r] + vb[r] : 1 + dk * km[r] / zw + dm * km[r] / zw + vb[r];
            } else {
                A = -dm / (0.5 * zw) * kb;
                B = edge ? 1 + vb[r] : 1 + dm / (0.5 * zw) * km[r] + vb[r];
            }
            C = -dk / zw * kn;
        } else {
            const double rz = lv.rz[kc], rl = lv.rl[kc];
            A = -scaled(dm, rz, rl);
            B = 1 + scaled(dk + (edge ? 0.0 : dm), rz, rl) + vb[r];
            C = -scaled(dk, rz, rl);
        }
        va[r] = wet && !edge ? A : 0.0;
        vb[r] = wet ? B : 1.0;
        vc[r] = wet && k < nz - 1 ? C : 0.0;
        z[0][r] = wet ? z[0][r] : 0.0;
        dm = dk;
    }
    col_solve<S, 1, !MUL>(t, va, vb, vc, z);
    seg_put(t, rhs, z[0]);
}

// LDS of a block: three images per wave, the columns, the level tables.
template <int S, int P>
struct TurbShared {
    double img[kTurbBlock / 64][3][Tile<S, P>::IMG];
    TurbCols cols[kTurbBlock / 64];
    TurbLevels lv;
};

// Waves per SIMD: as many as the registers allow without spilling (5 levels
// per lane at four waves: 24 to 44 bytes of scratch per lane, 4.61 ms for the
// three on 1440x720x80 against 4.08 at three and 4.29 at two).
#define VX_TURB_WAVES(S) ((S) < 5 ? 4 : ((S) <= 6 ? 3 : 2))

// ---------------------------------------------------------------------------
// TKE (veros/core/tke.py:123-321)
// ---------------------------------------------------------------------------
struct TkeArgs {
    TurbGrid g;
    double* tke;  // time levels
    int tau, taup1;
    const double *kappaM, *sqrttke, *mxl, *forc_surf;
    Terms forc;
    double *surf_corr, *diss;
    double dt, alpha, c_eps, K_h;
    int hor;
};

template <int S, int P>
__global__ __launch_bounds__(kTurbBlock) __attribute__((amdgpu_waves_per_eu(VX_TURB_WAVES(S)))) void tke_kernel(TkeArgs a) {
    const TurbGrid& g = a.g;
    __shared__ TurbShared<S, P> sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int64_t col0 = turb_col0<P>(wave);
    const Tile<S, P> t = turb_tile<S, P>(g, col0);
    const double dt = a.dt;
    TurbCols& tc = sh.cols[wave];
    const TurbLane l = turb_lane(g, t, col0);
    const int nz = g.nz;
    const uint32_t cs = (uint32_t)g.cs;
    const double* E0 = a.tke + a.tau * g.ls;
    double* E1 = a.tke + a.taup1 * g.ls;
    uint32_t wet[S], dry[S];  // solved cells; the others of the run
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const bool w = t.k[r] >= __shfl(l.k0, t.c[r] * P);
        wet[r] = w ? t.off[r] : kNoAccess;
        dry[r] = w ? kNoAccess : t.off[r];
    }
    const double fsurf = a.forc_surf[t.q < t.ncol ? col0 + t.q : 0];
    double e0[S], e1[S], rate[S], f[S];
    {
        double km[S], sq[S], ml[S];
        tile_load(tile_buf(t, a.kappaM), wet, 1, km);
        tile_load(tile_buf(t, a.sqrttke), t.off, 1, sq);
        tile_load(tile_buf(t, a.mxl), t.off, 1, ml);
        tile_load(tile_buf(t, E0, 0, (int)cs), wet, cs, e0);
        // taup1 off the solved cells (kept there and read by the diagnostic)
        tile_load(tile_buf(t, E1, 0, (int)cs), dry, cs, e1);
        turb_setup(g, t, l, dt * a.alpha, dt * a.K_h, a.hor != 0, sh.lv, tc);
        add_terms(a.forc, t, wet, true, f);
        tile_put(t, sh.img[wave][0], km);
        // on the diagonal dt c_eps sqrttke / mxl, rounded as often as when divided once:
        // dt times the diagnostic's rate, corrected by its remainder
        const double dtc = dt * a.c_eps, rc = a.c_eps != 0.0 ? 1.0 / a.c_eps : 0.0;
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const double q = a.c_eps / ml[r];
            rate[r] = q * sq[r];
            const double x = dt * rate[r];
            const double y = fma(fma(-x, ml[r], dtc * sq[r]), q * rc, x);
            sq[r] = y == y ? y : x;  // an infinite mxl dissipates nothing, but leaves 0 * inf in the remainder
        }
        tile_put(t, sh.img[wave][1], sq);
    }
    {
        double x[S];
        const double ftop = scaled(dt * fsurf, sh.lv.rz[nz - 1], sh.lv.rl[nz - 1]);
#pragma unroll
        for (int r = 0; r < S; ++r) {
            x[r] = e0[r] + dt * f[r];
            const double fs = __shfl(ftop, t.c[r] * P);
            if (t.k[r] == nz - 1) x[r] += fs;
        }
        tile_put(t, sh.img[wave][2], x);
    }
    turb_solve<S, false>(t, sh.lv, nz, l.k0, sh.img[wave][0], sh.img[wave][1], sh.img[wave][2]);
    double v[S], dg[S];
    uint32_t st[S];
    tile_get(t, sh.img[wave][2], v);
#pragma unroll
    for (int r = 0; r < S; ++r) {
        v[r] = wet[r] != kNoAccess ? v[r] : e1[r];
        dg[r] = rate[r] * v[r];  // tke_diss over the whole array (:230)
        st[r] = wet[r];
    }
    // surface correction and clamp of every interior column (:235-244)
    double corr[S];
    bool top[S];
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const int in = __shfl((int)l.interior, t.c[r] * P);
        top[r] = in != 0 && t.k[r] == nz - 1 && t.off[r] != kNoAccess;
        corr[r] = v[r];
        v[r] = top[r] ? fmax(0.0, v[r]) : v[r];
        st[r] = top[r] ? t.off[r] : st[r];
    }
    if (a.hor) {
        const double none[1] = {0.0};
        add_lateral<S, false>(g, t, tc, E0, cs, nullptr, e0, none,
                              [](double nA, double, double ea, double) { return nA - ea; }, v);
    }
    tile_store(tile_buf(t, a.diss), t.off, 1, dg);
#pragma unroll
    for (int r = 0; r < S; ++r) {
        if (top[r]) a.surf_corr[col0 + t.c[r]] = corr[r] < 0.0 ? -corr[r] * 0.5 * sh.lv.zw[nz - 1] / dt : 0.0;
    }
    tile_store(tile_buf(t, E1, 0, (int)cs), st, cs, v);
}

// ---------------------------------------------------------------------------
// EKE (veros/core/eke.py:93-255)
// ---------------------------------------------------------------------------
struct EkeArgs {
    TurbGrid g;
    double* eke;
    int tau, taup1;
    const double *kappaM, *sqrteke, *eke_len, *K_gm;
    Terms forc;
    double *diss_iw, *diss_tke;
    double dt, alpha, c_eps;
};

template <int S, int P>
__global__ __launch_bounds__(kTurbBlock) __attribute__((amdgpu_waves_per_eu(VX_TURB_WAVES(S)))) void eke_kernel(EkeArgs a) {
    const TurbGrid& g = a.g;
    __shared__ TurbShared<S, P> sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int64_t col0 = turb_col0<P>(wave);
    const Tile<S, P> t = turb_tile<S, P>(g, col0);
    const double dt = a.dt;
    TurbCols& tc = sh.cols[wave];
    const TurbLane l = turb_lane(g, t, col0);
    const int nz = g.nz;
    const uint32_t cs = (uint32_t)g.cs;
    const double* E0 = a.eke + a.tau * g.ls;
    double* E1 = a.eke + a.taup1 * g.ls;
    // solved cells; wet cells (c_int is 0 elsewhere, :121); wet cells that are not solved (halo columns)
    uint32_t wet[S], sea[S], halo[S];
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const bool w = t.k[r] >= __shfl(l.k0, t.c[r] * P), m = t.k[r] >= __shfl(l.kw, t.c[r] * P);
        wet[r] = w ? t.off[r] : kNoAccess;
        sea[r] = m ? t.off[r] : kNoAccess;
        halo[r] = m && !w ? t.off[r] : kNoAccess;
    }
    double e0[S], e1[S], cint[S], f[S], kg[S];
    {
        double km[S], sq[S], el[S];
        tile_load(tile_buf(t, a.kappaM), wet, 1, km);
        tile_load(tile_buf(t, a.sqrteke), sea, 1, sq);
        tile_load(tile_buf(t, a.eke_len), sea, 1, el);
        tile_load(tile_buf(t, E0, 0, (int)cs), wet, cs, e0);
        tile_load(tile_buf(t, E1, 0, (int)cs), halo, cs, e1);
        turb_setup(g, t, l, dt * a.alpha, dt, true, sh.lv, tc);
        add_terms(a.forc, t, wet, true, f);
        tile_load(tile_buf(t, a.K_gm), wet, 1, kg);
        tile_put(t, sh.img[wave][0], km);
#pragma unroll
        for (int r = 0; r < S; ++r) cint[r] = sea[r] != kNoAccess ? a.c_eps * sq[r] / el[r] : 0.0;
    }
    {
        double x[S];
#pragma unroll
        for (int r = 0; r < S; ++r) x[r] = dt * cint[r];
        tile_put(t, sh.img[wave][1], x);
#pragma unroll
        for (int r = 0; r < S; ++r) x[r] = e0[r] + dt * f[r];
        tile_put(t, sh.img[wave][2], x);
    }
    turb_solve<S, false>(t, sh.lv, nz, l.k0, sh.img[wave][0], sh.img[wave][1], sh.img[wave][2]);
    double v[S], dg[S];
    tile_get(t, sh.img[wave][2], v);
#pragma unroll
    for (int r = 0; r < S; ++r) {
        v[r] = wet[r] != kNoAccess ? v[r] : e1[r];
        dg[r] = cint[r] * v[r];  // (:151)
    }
    add_lateral<S, true>(g, t, tc, E0, cs, a.K_gm, e0, kg, [](double nE, double nK, double ea, double ka) {
        return 0.5 * fmax(500.0, nK + ka) * (nE - ea);
    }, v);
    tile_store(tile_buf(t, a.diss_iw), t.off, 1, dg);
#pragma unroll
    for (int r = 0; r < S; ++r) dg[r] = 0.0;  // (:152)
    tile_store(tile_buf(t, a.diss_tke), t.off, 1, dg);
    tile_store(tile_buf(t, E1, 0, (int)cs), wet, cs, v);
}

// ---------------------------------------------------------------------------
// IDEMIX (veros/core/idemix.py:47-265)
// ---------------------------------------------------------------------------
struct IdemixArgs {
    TurbGrid g;
    double* E;
    int tau, taup1;
    const double *c0, *v0, *alpha_c, *forc_bot, *forc_surf;
    Terms forc;       // before the optional move to the bottom / surface cells
    Terms forc_post;  // added afterwards (bottom friction)
    double* iw_diss;
    double dt, tau_v, tau_h, frac;
    int hor;
    int diss_mode;  // 0: as is; 1: column integral at the bottom cell; 2: split bottom / surface
};

template <int S, int P>
__global__ __launch_bounds__(kTurbBlock) __attribute__((amdgpu_waves_per_eu(VX_TURB_WAVES(S)))) void idemix_kernel(IdemixArgs a) {
    const TurbGrid& g = a.g;
    __shared__ TurbShared<S, P> sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int64_t col0 = turb_col0<P>(wave);
    const Tile<S, P> t = turb_tile<S, P>(g, col0);
    const double dt = a.dt;
    TurbCols& tc = sh.cols[wave];
    const TurbLane l = turb_lane(g, t, col0);
    const int nz = g.nz;
    const uint32_t cs = (uint32_t)g.cs;
    const double* E0 = a.E + a.tau * g.ls;
    double* E1 = a.E + a.taup1 * g.ls;
    uint32_t wet[S], dry[S];
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const bool w = t.k[r] >= __shfl(l.k0, t.c[r] * P);
        wet[r] = w ? t.off[r] : kNoAccess;
        dry[r] = w ? kNoAccess : t.off[r];
    }
    const int64_t gcol = t.q < t.ncol ? col0 + t.q : 0;
    const double fbot = a.forc_bot[gcol], fsurf = a.forc_surf[gcol];
    double e0[S], e1[S], rate[S], f[S];
    {
        double c0[S], al[S];
        tile_load(tile_buf(t, a.c0), wet, 1, c0);
        tile_load(tile_buf(t, a.alpha_c), t.off, 1, al);
        // E_iw at tau on every cell, at taup1 off the solved ones (kept there and read by the diagnostic)
        tile_load(tile_buf(t, E0, 0, (int)cs), t.off, cs, e0);
        tile_load(tile_buf(t, E1, 0, (int)cs), dry, cs, e1);
        turb_setup(g, t, l, dt * a.tau_v, dt * a.tau_h * 0.5, a.hor != 0, sh.lv, tc);
        add_terms(a.forc, t, wet, true, f);
        tile_put(t, sh.img[wave][0], c0);
#pragma unroll
        for (int r = 0; r < S; ++r) rate[r] = al[r] * fmax(0.0, e0[r]);  // alpha_c max(0, E_iw[tau]) (:118)
    }
    if (a.diss_mode != 0) {  // (:70-103): the forcing's column integral moved to the bottom (and surface) cell
        double* const img = sh.img[wave][1];
        tile_put(t, img, f);
        const int k0 = l.k0;
        double part = 0.0;
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const int k = t.lo + r;
            const double fk = img[t.seg + r];
            if (k >= k0 && k < nz) part += (k < nz - 1 ? sh.lv.zw[k] : 0.5 * sh.lv.zw[k]) * fk;
        }
        part += __shfl_xor(part, 1, P);
        part += __shfl_xor(part, 2, P);
        part += __shfl_xor(part, 4, P);
        if constexpr (P == 16) part += __shfl_xor(part, 8, P);
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const double a_loc = __shfl(part, t.c[r] * P);
            const int k = t.k[r];
            double x = 0.0;
            if (k == __shfl(l.k0, t.c[r] * P)) x = (a.diss_mode == 1 ? 1.0 : a.frac) * a_loc / sh.lv.zw[k];
            if (a.diss_mode == 2 && k == nz - 1) x = (1.0 - a.frac) * a_loc / (0.5 * sh.lv.zw[k]);
            f[r] = x;
        }
    }
    add_terms(a.forc_post, t, wet, false, f);
    {
        double x[S];
#pragma unroll
        for (int r = 0; r < S; ++r) x[r] = dt * rate[r];
        tile_put(t, sh.img[wave][1], x);
        const double ftop = scaled(dt * fsurf, sh.lv.rz[nz - 1], sh.lv.rl[nz - 1]);
#pragma unroll
        for (int r = 0; r < S; ++r) {
            x[r] = e0[r] + dt * f[r];
            const bool edge = t.k[r] == __shfl(l.k0, t.c[r] * P);
            const double fb = __shfl(fbot, t.c[r] * P), fs = __shfl(ftop, t.c[r] * P);
            if (edge) x[r] += dt * fb / sh.lv.zw[t.k[r]];  // d_edge (:157-159)
            else if (t.k[r] == nz - 1) x[r] += fs;
        }
        tile_put(t, sh.img[wave][2], x);
    }
    turb_solve<S, true>(t, sh.lv, nz, l.k0, sh.img[wave][0], sh.img[wave][1], sh.img[wave][2]);
    double v[S], dg[S];
    tile_get(t, sh.img[wave][2], v);
#pragma unroll
    for (int r = 0; r < S; ++r) {
        v[r] = wet[r] != kNoAccess ? v[r] : e1[r];
        dg[r] = rate[r] * v[r];  // (:174)
    }
    if (a.hor) {  // (:186-218): the fluxes of v0 E with the coefficient 0.5 tau_h (v0 + v0')
        double v0[S];
        tile_load(tile_buf(t, a.v0), wet, 1, v0);
        add_lateral<S, true>(g, t, tc, E0, cs, a.v0, e0, v0, [](double nE, double nV, double ea, double va) {
            return (nV + va) * (nV * nE - va * ea);
        }, v);
    }
    tile_store(tile_buf(t, a.iw_diss), t.off, 1, dg);
    tile_store(tile_buf(t, E1, 0, (int)cs), wet, cs, v);
}

namespace {

int make_turb_grid(const vx_grid* in, TurbGrid& g, const char* who) {
    if (!in) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid", who);
    if (in->nx < 1 || in->ny < 1 || in->nz < 2)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: need nx, ny >= 1 and nz >= 2", who);
    if (in->nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d exceeds %d", who, in->nz, kMaxNz);
    if (!in->kbot || !in->dxt || !in->dxu || !in->dyt || !in->dyu || !in->cost || !in->cosu || !in->dzt || !in->dzw)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid array", who);
    if (in->time_layout != VX_LEVELS_INNER && in->time_layout != VX_LEVELS_OUTER)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: time_layout must be VX_LEVELS_INNER or VX_LEVELS_OUTER", who);
    g.kbot = in->kbot;
    g.dxt = in->dxt, g.dxu = in->dxu, g.dyt = in->dyt, g.dyu = in->dyu;
    g.cost = in->cost, g.cosu = in->cosu, g.dzt = in->dzt, g.dzw = in->dzw;
    g.X = (int32_t)(in->nx + 4);
    g.Y = (int32_t)(in->ny + 4);
    g.nz = in->nz;
    const bool outer = in->time_layout == VX_LEVELS_OUTER;
    g.cs = outer ? 1 : 3;
    g.ls = outer ? (int64_t)g.X * g.Y * g.nz : 1;
    return VX_OK;
}

int make_terms(const vx_terms* in, Terms& t, bool allow_empty, const char* who) {
    t.n = 0;
    if (!in) {
        if (allow_empty) return VX_OK;
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null forcing terms", who);
    }
    if (in->n < (allow_empty ? 0 : 1) || in->n > kMaxTerms)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: forcing needs 1..%d terms (got %d)", who, kMaxTerms, in->n);
    for (int q = 0; q < in->n; ++q) {
        if (!in->arr[q]) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null forcing term %d", who, q);
        t.p[q] = in->arr[q];
        t.sgn[q] = in->sign[q];
    }
    t.n = in->n;
    return VX_OK;
}

template <class Args, template <int, int> class K>
int launch_turb(const Args& a, const TurbGrid& g, hipStream_t s, const char* who) {
    const int lanes = col_lanes(g.nz), cols = 64 / lanes;
    const int64_t threads = ((int64_t)g.X * g.Y + cols - 1) / cols * 64;
    const dim3 grid(blocks_mult8(threads, kTurbBlock)), block(kTurbBlock);
    switch (col_levels(g.nz)) {
        case 2: hipLaunchKernelGGL((K<2, kSegP>::fn), grid, block, 0, s, a); break;
        case 3:
            if (lanes == kSegP) hipLaunchKernelGGL((K<3, kSegP>::fn), grid, block, 0, s, a);
            else hipLaunchKernelGGL((K<3, kTileP>::fn), grid, block, 0, s, a);
            break;
        case 4:
            if (lanes == kSegP) hipLaunchKernelGGL((K<4, kSegP>::fn), grid, block, 0, s, a);
            else hipLaunchKernelGGL((K<4, kTileP>::fn), grid, block, 0, s, a);
            break;
        case 5: hipLaunchKernelGGL((K<5, kTileP>::fn), grid, block, 0, s, a); break;
        case 6: hipLaunchKernelGGL((K<6, kTileP>::fn), grid, block, 0, s, a); break;
        case 7: hipLaunchKernelGGL((K<7, kTileP>::fn), grid, block, 0, s, a); break;
        case 8: hipLaunchKernelGGL((K<8, kTileP>::fn), grid, block, 0, s, a); break;
        default: return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, g.nz);
    }
    return check_launch(who);
}

template <int N, int P>
struct TkeK {
    static constexpr auto fn = tke_kernel<N, P>;
};
template <int N, int P>
struct EkeK {
    static constexpr auto fn = eke_kernel<N, P>;
};
template <int N, int P>
struct IdemixK {
    static constexpr auto fn = idemix_kernel<N, P>;
};

bool levels_ok(int tau, int taup1) { return tau >= 0 && tau <= 2 && taup1 >= 0 && taup1 <= 2 && tau != taup1; }

}  // namespace
}  // namespace vx

extern "C" int vx_integrate_tke_f64(void* stream, const vx_grid* grid, const vx_tke_params* prm, double* tke,
                                    int32_t tau, int32_t taup1, const double* kappaM, const double* sqrttke,
                                    const double* mxl, const double* forc_tke_surface, const vx_terms* forc,
                                    double* tke_surf_corr, double* tke_diss) {
    using namespace vx;
    const char* who = "vx_integrate_tke_f64";
    TkeArgs a{};
    int rc = make_turb_grid(grid, a.g, who);
    if (rc) return rc;
    if (!prm) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null parameters", who);
    if (!levels_ok(tau, taup1)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: tau, taup1 must be distinct in 0..2", who);
    if (!tke || !kappaM || !sqrttke || !mxl || !forc_tke_surface || !tke_surf_corr || !tke_diss)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((rc = make_terms(forc, a.forc, false, who))) return rc;
    if (!(prm->dt_mom > 0.0)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: dt_mom must be positive", who);
    a.tke = tke, a.tau = tau, a.taup1 = taup1;
    a.kappaM = kappaM, a.sqrttke = sqrttke, a.mxl = mxl, a.forc_surf = forc_tke_surface;
    a.surf_corr = tke_surf_corr, a.diss = tke_diss;
    a.dt = prm->dt_mom, a.alpha = prm->alpha_tke, a.c_eps = prm->c_eps, a.K_h = prm->K_h_tke;
    a.hor = prm->hor_diffusion != 0;
    return launch_turb<TkeArgs, TkeK>(a, a.g, (hipStream_t)stream, who);
}

extern "C" int vx_integrate_eke_f64(void* stream, const vx_grid* grid, const vx_eke_params* prm, double* eke,
                                    int32_t tau, int32_t taup1, const double* kappaM, const double* sqrteke,
                                    const double* eke_len, const double* K_gm, const vx_terms* forc,
                                    double* eke_diss_iw, double* eke_diss_tke) {
    using namespace vx;
    const char* who = "vx_integrate_eke_f64";
    EkeArgs a{};
    int rc = make_turb_grid(grid, a.g, who);
    if (rc) return rc;
    if (!prm) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null parameters", who);
    if (!levels_ok(tau, taup1)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: tau, taup1 must be distinct in 0..2", who);
    if (!eke || !kappaM || !sqrteke || !eke_len || !K_gm || !eke_diss_iw || !eke_diss_tke)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((rc = make_terms(forc, a.forc, false, who))) return rc;
    if (!(prm->dt_tracer > 0.0)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: dt_tracer must be positive", who);
    a.eke = eke, a.tau = tau, a.taup1 = taup1;
    a.kappaM = kappaM, a.sqrteke = sqrteke, a.eke_len = eke_len, a.K_gm = K_gm;
    a.diss_iw = eke_diss_iw, a.diss_tke = eke_diss_tke;
    a.dt = prm->dt_tracer, a.alpha = prm->alpha_eke, a.c_eps = prm->eke_c_eps;
    return launch_turb<EkeArgs, EkeK>(a, a.g, (hipStream_t)stream, who);
}

extern "C" int vx_integrate_idemix_f64(void* stream, const vx_grid* grid, const vx_idemix_params* prm, double* E_iw,
                                       int32_t tau, int32_t taup1, const double* c0, const double* v0,
                                       const double* alpha_c, const double* forc_iw_bottom,
                                       const double* forc_iw_surface, const vx_terms* forc,
                                       const vx_terms* forc_post, double* iw_diss) {
    using namespace vx;
    const char* who = "vx_integrate_idemix_f64";
    IdemixArgs a{};
    int rc = make_turb_grid(grid, a.g, who);
    if (rc) return rc;
    if (!prm) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null parameters", who);
    if (!levels_ok(tau, taup1)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: tau, taup1 must be distinct in 0..2", who);
    if (!E_iw || !c0 || !v0 || !alpha_c || !forc_iw_bottom || !forc_iw_surface || !iw_diss)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((rc = make_terms(forc, a.forc, false, who))) return rc;
    if ((rc = make_terms(forc_post, a.forc_post, true, who))) return rc;
    if (prm->eke_diss_mode < 0 || prm->eke_diss_mode > 2)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: eke_diss_mode must be 0, 1 or 2", who);
    if (!(prm->dt_tracer > 0.0)) return fail(VX_ERR_INVALID_ARGUMENT, "%s: dt_tracer must be positive", who);
    a.E = E_iw, a.tau = tau, a.taup1 = taup1;
    a.c0 = c0, a.v0 = v0, a.alpha_c = alpha_c, a.forc_bot = forc_iw_bottom, a.forc_surf = forc_iw_surface;
    a.iw_diss = iw_diss;
    a.dt = prm->dt_tracer, a.tau_v = prm->tau_v, a.tau_h = prm->tau_h, a.frac = prm->eke_diss_surfbot_frac;
    a.hor = prm->hor_diffusion != 0;
    a.diss_mode = prm->eke_diss_mode;
    return launch_turb<IdemixArgs, IdemixK>(a, a.g, (hipStream_t)stream, who);
}
