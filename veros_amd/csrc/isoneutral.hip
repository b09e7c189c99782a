// Isoneutral triad-tensor stencils for gfx950 (float64).
//
//   iso_pre_kernel       isoneutral_diffusion_pre  veros/core/isoneutral/isoneutral.py:18-229
//   iso_flux_kernel      _calc_tracer_fluxes       veros/core/isoneutral/diffusion.py:9-113
//   iso_step_wet_kernel  _calc_explicit_part, _calc_implicit_part, the tracer and
//                        dtr_iso updates and the energy branch, over the wet cells
//                                                  veros/core/isoneutral/diffusion.py:116-283,
//                                                  veros/core/diffusion.py:9-62
//   iso_adj_*_kernel     the adjoint of one isoneutral tracer step
//
// Layout: veros state arrays with 2-cell halos, z contiguous, k = 0 deepest.
// Cell-parallel kernels put consecutive lanes on consecutive levels of one
// column, so every stencil read of a neighbouring column is itself a
// contiguous run. Masks are derived from kbot exactly as calc_topo_kernel
// builds them (veros/core/numerics.py:195-221): maskT = kbot>0 & k>=kbot-1,
// maskU/V = min of the two adjacent maskT, maskW = min(maskT[k], maskT[k+1]).
#include <algorithm>
#include <map>
#include <mutex>

#include "col_tile.hpp"

// Tuning knob (compile-time): minimum waves per SIMD requested for the pre
// kernel (caps its VGPRs).
#ifndef VX_PRE_MIN_WAVES
#define VX_PRE_MIN_WAVES 2
#endif

namespace vx {

constexpr double kEpsln = 1e-20;  // veros/core/isoneutral/isoneutral.py:28

struct Grid {
    const int32_t* kbot;
    const double *dxt, *dxu, *dyt, *dyu, *cost, *cosu, *dzt, *dzw;
    int32_t X, Y, nz;
    // time-level arrays (temp, salt, tracer, int_drhodX): level l of cell c at
    // l * ls + c * cs; cs = 3, ls = 1 for the reference's (X, Y, nz, 3)
    // layout, cs = 1, ls = X*Y*nz for levels stored one after another
    uint32_t cs, ls;
};

struct Prm {
    double drhodT, drhodS, K_iso_steep, iso_slopec, iso_dslope, dt_tracer, grav, rho_0;
};

// Level k of a column with bottom index kb is a wet T cell (maskT = 1).
__device__ __forceinline__ bool wet(int kb, int k) { return kb > 0 && kb - 1 <= k; }

// temp and salt and the time level that the stencil reads.
struct Fields {
    const double* __restrict__ T;
    const double* __restrict__ S;
    int tau;
};

// Blocks are dispatched round-robin over the 8 XCDs; remap so that each XCD
// walks a contiguous range of the domain and neighbouring rows share its L2.
// `nb` must be a multiple of 8.
__device__ __forceinline__ int64_t xcd_block(int64_t nb) {
    const int64_t b = blockIdx.x;
    return (b & 7) * (nb >> 3) + (b >> 3);
}

// 1/x from v_rcp_f64 refined by two Newton steps (about 1 ulp; finite
// non-zero x only).
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

// Masked face gradients of the two tracers (veros/core/isoneutral/isoneutral.py:46-95).
struct Grad {
    double T, S;
};

// exp(x) for |x| <= 64 by Cody-Waite reduction: x = n ln2 + r with ln2 split
// into a 32-bit-exact high part and a low part, |r| <= ln2/2, e^r from its
// Taylor series to degree 13 (truncation < 5e-18 relative), then 2^n.
// The coefficients are read once per kernel into an ExpCoef (uniform, so
// they stay in scalar registers and feed v_fma_f64 directly).
__constant__ double kExpTable[16] = {
    1.4426950408889634,                       // log2(e)
    6.93147180369123816490e-01,               // ln2, high part
    1.90821492927058770002e-10,               // ln2, low part
    1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0, 1.0 / 3628800.0, 1.0 / 362880.0,
    1.0 / 40320.0, 1.0 / 5040.0, 1.0 / 720.0, 1.0 / 120.0, 1.0 / 24.0, 1.0 / 6.0, 0.5, 1.0};

struct ExpCoef {
    double c[16];
};

__device__ __forceinline__ ExpCoef load_exp_coef() {
    ExpCoef e;
#pragma unroll
    for (int q = 0; q < 16; ++q) e.c[q] = kExpTable[q];
    return e;
}

__device__ __forceinline__ double exp_reduced(const ExpCoef& e, double x) {
    const double n = rint(x * e.c[0]);
    double r = fma(-n, e.c[1], x);
    r = fma(-n, e.c[2], r);
    double q = e.c[3];
#pragma unroll
    for (int t = 4; t < 16; ++t) q = fma(q, r, e.c[t]);
    q = fma(q, r, 1.0);
    return ldexp(q, (int)n);
}

// dm_taper (veros/core/isoneutral/isoneutral.py:10-15):
//   0.5*(1 + tanh(u)) == 1/(1 + exp(-2u)),  u = (slopec - |s|)/dslope.
// In float64 tanh(u) rounds to exactly -1 / +1 for |u| > 55*ln(2)/2 (~19.06),
// which makes the reference taper exactly 0 / 1 there; those branches are
// taken without evaluating the exponential. `two_over_dslope` = 2/dslope.
__device__ __forceinline__ double taper(const Prm& p, const ExpCoef& ec, double two_over_dslope, double s) {
    const double x = (fabs(s) - p.iso_slopec) * two_over_dslope;  // -2u
    // branch-free: the exponential of the clamped argument, then the exact
    // end values by selection (a NaN slope stays NaN)
    const double t = rcp_nr(1.0 + exp_reduced(ec, fmin(fmax(x, -38.12), 38.12)));
    return x > 38.12 ? 0.0 : (x < -38.12 ? 1.0 : (x == x ? t : x));
}

// Horizontal and vertical density gradients of one triad, weighted by the
// drho/dX of one T point (the 0/1 mask is folded into the weights).
struct Dens {
    double drdT, drdS;
};
__device__ __forceinline__ Dens dens(const Prm& p, double mt) { return {mt * p.drhodT, mt * p.drhodS}; }
__device__ __forceinline__ double dot(const Dens& w, const Grad& gr) { return w.drdT * gr.T + w.drdS * gr.S; }
// 1 / (min(0, drho/dz) - epsln): the slope denominator
__device__ __forceinline__ double rden(double drodz) { return rcp_nr(fmin(0.0, drodz) - kEpsln); }

// ---------------------------------------------------------------------------
// Cell-parallel launch geometry: block = (nz levels) x (cpb columns along j);
// consecutive lanes are consecutive levels of one column, so every read of a
// neighbouring column is a contiguous run. Blocks are ordered in strips of
// kStripBlocks blocks along j, walked row by row along i, and the 1-D grid is
// remapped XCD-contiguously: the i-1 / i / i+1 rows of a strip are then in
// flight on the same XCD together and their shared reads hit its L2.
// ---------------------------------------------------------------------------
#ifndef VX_STRIP_BLOCKS
#define VX_STRIP_BLOCKS 16
#endif
constexpr int kStripBlocks = VX_STRIP_BLOCKS;
// the pre and flux kernels' strips: at most so many columns along j (strip_blocks; the
// fused call on 1440x720x80, on 300x200x128 and the calls on 360x160x60, the last two
// with the levels innermost: 64 columns 6.04 ms, 773 and 958 us, 96 5.97, 752 and 966,
// 192 5.87, 737 and 956, 256 5.98, 735 and 955)
#ifndef VX_PRE_STRIP_COLS
#define VX_PRE_STRIP_COLS 192
#endif
constexpr int kPreStripCols = VX_PRE_STRIP_COLS;

struct CellIdx {
    int i, j, k;
    bool valid;
};

// The block's row i and first column jb when blocks own cpb columns each.
struct BlockCols {
    int i, j;
    bool valid;  // false for a padding block
};
__device__ __forceinline__ BlockCols block_cols(int i0, int ni, int j0, int nj, int cpb, int sb = kStripBlocks) {
    const int sw = sb * cpb;                          // strip width in columns
    const int nstrips = (nj + sw - 1) / sw;
    const int per_strip = ni * sb;
    const int L = (int)xcd_block(gridDim.x);
    const int sidx = L / per_strip;
    const int rem = L - sidx * per_strip;
    const int ii = rem / sb;
    const int b = rem - ii * sb;
    BlockCols r;
    r.i = i0 + ii;
    r.j = j0 + sidx * sw + b * cpb;
    r.valid = sidx < nstrips && r.j < j0 + nj;
    return r;
}
__device__ __forceinline__ CellIdx cell_of(int i0, int ni, int j0, int nj) {
    const BlockCols bc = block_cols(i0, ni, j0, nj, (int)blockDim.y);
    CellIdx r;
    r.i = bc.i;
    r.j = bc.j + (int)threadIdx.y;
    r.k = (int)threadIdx.x;
    r.valid = bc.valid && r.j < j0 + nj;
    return r;
}

__device__ __forceinline__ double m01(int kb, int k) { return (kb > 0 && kb - 1 <= k) ? 1.0 : 0.0; }

// ---------------------------------------------------------------------------
// isoneutral_diffusion_pre: thread per cell (i, j, k), i in [1, X-2), j in [1, Y-2).
// The 13 tracer points of the stencil are loaded once per field; all face
// gradients are formed from them in registers. Offsets are 32-bit element
// offsets (the host checks the arrays fit).
// ---------------------------------------------------------------------------
// Metric factors of a block's columns and of the levels, in LDS: the cells read
// them as factors instead of dividing (a float64 division is about 14
// instructions; pre with its fluxes had 35 divisions and reciprocals per cell).
// Each is one division, made once per block.
struct ColMetrics {
    double rx, rxw;    // 1 / (dxu cost), the same at i-1
    double ry, rys;    // 1 / dyu, the same at j-1
    double rcost;      // 1 / cost
    double cosu, cosus;
    double fyc, fys;   // cosu dyu, the same at j-1
    double ryt;        // 1 / (4 dyt cost)
};
struct LevelMetrics {
    double rzw[kMaxNz];   // 1 / dzw
    double dzw[kMaxNz];
    double r4zt[kMaxNz];   // 1 / (4 dzt)
    double r4ztl[kMaxNz];  // what its rounding cuts off: K_11 and K_22 round as when divided
};
constexpr int kCellBlock = 64;  // threads of a pre or flux block: one wave
constexpr int kBlockCols = 32;  // most columns of one
struct BlockMetrics {
    ColMetrics col[kBlockCols];
    LevelMetrics lev;
    int kb[kBlockCols + 2], kbe[kBlockCols], kbw[kBlockCols];  // kbot at j-1 .. j+1 of row i; at rows i+1, i-1
    int run[kBlockCols + 1];                                   // prefix sums of the columns' run lengths
};
// Every thread of the block calls it; visible after the next barrier.
__device__ __forceinline__ void fill_metrics(const Grid& g, int i, int jb, int ncb, BlockMetrics& m) {
    const int tid = (int)threadIdx.x, nthr = (int)blockDim.x;
    for (int q = tid; q < ncb; q += nthr) {
        const int j = jb + q <= g.Y - 3 ? jb + q : g.Y - 3;
        const double cost = g.cost[j], cosu = g.cosu[j], cosus = g.cosu[j - 1], dyu = g.dyu[j], dyus = g.dyu[j - 1];
        ColMetrics& c = m.col[q];
        c.rx = 1.0 / (cost * g.dxu[i]);
        c.rxw = 1.0 / (cost * g.dxu[i - 1]);
        c.ry = 1.0 / dyu;
        c.rys = 1.0 / dyus;
        c.rcost = 1.0 / cost;
        c.cosu = cosu;
        c.cosus = cosus;
        c.fyc = cosu * dyu;
        c.fys = cosus * dyus;
        c.ryt = 1.0 / (4 * g.dyt[j] * cost);
        m.kbe[q] = g.kbot[(i + 1) * g.Y + j];
        m.kbw[q] = g.kbot[(i - 1) * g.Y + j];
    }
    for (int q = tid; q < ncb + 2; q += nthr) {
        const int j = jb - 1 + q <= g.Y - 2 ? jb - 1 + q : g.Y - 2;
        m.kb[q] = g.kbot[i * g.Y + j];
    }
    for (int k = tid; k < g.nz; k += nthr) {
        const double dzw = g.dzw[k];
        m.lev.dzw[k] = dzw;
        m.lev.rzw[k] = 1.0 / dzw;
        const Recip r4zt = recip(4.0 * g.dzt[k]);
        m.lev.r4zt[k] = r4zt.h;
        m.lev.r4ztl[k] = r4zt.l;
    }
}
// Turns r[1 .. ncb] (lengths) into prefix sums with r[0] = 0; between barriers.
__device__ __forceinline__ void scan_runs(int* r, int ncb) {
    if (threadIdx.x < 64) {
        const int lane = (int)threadIdx.x;
        int v = lane < ncb ? r[lane + 1] : 0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(v, d);
            v += lane >= d ? u : 0;
        }
        if (lane < ncb) r[lane + 1] = v;
        if (lane == 0) r[0] = 0;
    }
}
// the column q with run[q] <= t < run[q + 1]
__device__ __forceinline__ int run_column(const int* run, int ncb, int t) {
    int lo = 0, hi = ncb - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (run[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Face-flux arithmetic (veros/core/isoneutral/diffusion.py:22-111), shared by
// the flux kernel and the fused pre + flux kernel; the fused multiply-adds are
// written out so that both produce the same values, whatever the compiler
// would contract in either. A01/A23 are the (ip=0, kr=0..1) / (ip=1, kr=0..1) entries of Ai_ez or
// Ai_nz; t0* the tracer at the cell (u = k+1, d = k-1, clamped at the ends),
// t1* at the east or north neighbour.
__device__ __forceinline__ double east_flux_core(double diffloc, double2 A01, double2 A23, double t0, double t0u,
                                                 double t0d, double t1, double t1u, double t1d, double r4zt,
                                                 double rx, double K11) {
    double sumz = diffloc * A01.x * (t0 - t0d);     // kr=0, ip=0
    sumz = fma(diffloc * A23.x, t1 - t1d, sumz);  // kr=0, ip=1
    sumz = fma(diffloc * A01.y, t0u - t0, sumz);  // kr=1, ip=0
    sumz = fma(diffloc * A23.y, t1u - t1, sumz);  // kr=1, ip=1
    return fma(sumz, r4zt, (t1 - t0) * rx * K11);
}
__device__ __forceinline__ double north_flux_core(double diffloc, double2 A01, double2 A23, double t0, double t0u,
                                                  double t0d, double t1, double t1u, double t1d, double r4zt,
                                                  double cosu, double ry, double K22) {
    double sumz = diffloc * A01.x * (t0 - t0d);
    sumz = fma(diffloc * A23.x, t1 - t1d, sumz);
    sumz = fma(diffloc * A01.y, t0u - t0, sumz);
    sumz = fma(diffloc * A23.y, t1u - t1, sumz);
    return cosu * fma(sumz, r4zt, (t1 - t0) * ry * K22);
}
// tc/tw/te/ts/tn = the tracer at the cell and its west/east/south/north
// neighbours, levels k (0) and k+1 (1); r4xt = 1 / (4 dxt)
__device__ __forceinline__ double top_flux_core(double diffloc, double2 B01, double2 B23, double2 C01, double2 C23,
                                                double tc0, double tc1, double tw0, double tw1, double te0,
                                                double te1, double ts0, double ts1, double tn0, double tn1,
                                                const ColMetrics& m, double r4xt) {
    const double dx = diffloc * m.rcost;
    double sumx = dx * B01.x * (tc0 - tw0);    // ip=0, kr=0
    sumx = fma(dx * B01.y, tc1 - tw1, sumx);  // ip=0, kr=1
    sumx = fma(dx * B23.x, te0 - tc0, sumx);  // ip=1, kr=0
    sumx = fma(dx * B23.y, te1 - tc1, sumx);  // ip=1, kr=1
    const double ds = diffloc * m.cosus, dn = diffloc * m.cosu;
    double sumy = ds * C01.x * (tc0 - ts0);
    sumy = fma(ds * C01.y, tc1 - ts1, sumy);
    sumy = fma(dn * C23.x, tn0 - tc0, sumy);
    sumy = fma(dn * C23.y, tn1 - tc1, sumy);
    return fma(sumx, r4xt, sumy * m.ryt);
}

// Face-flux outputs of the fused pre + flux kernel (temperature, salinity).
struct PreFlux {
    double *fe, *fn, *ft;
};
// Two tracers' flux at one cell; the caller's workspace may be aligned to 8 bytes only.
typedef double vx_d2a8 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void store_pair(double* p, double t, double s) {
    *reinterpret_cast<vx_d2a8*>(p) = (vx_d2a8){t, s};
}

// The dry cells of isoneutral_diffusion_pre: every output exactly zero (its own
// maskT factor is in maskU (Ai_ez, K_11), maskV (Ai_nz, K_22) and maskW (Ai_bx,
// Ai_by, K_33), which multiply each entry and each summed term), over the index
// ranges the reference writes: levels 0 .. nd-1 of column (i, j), one run per
// array, stored by the wave's lanes in order. Nothing in the call reads them, so
// they are stored nontemporal and leave the L2 to the wet cells.
typedef double vx_d2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void zero_run(double* __restrict__ p, int n, int lane) {
    for (int m = lane; m < n; m += 64) __builtin_nontemporal_store(0.0, p + m);
}
// Ai entries 4 c + 2 ip + kr of the cells 0 .. nd-1 of a column; at level 0
// only the kr = 1 entries are written (the kr = 0 ones keep their values).
__device__ __forceinline__ void zero_ai_run(double* __restrict__ p, int nd, int lane, bool keep_level0_kr0) {
    const int n2 = 2 * nd;  // double2 pieces
    for (int m = lane; m < n2; m += 64) {
        if (keep_level0_kr0 && m < 2) __builtin_nontemporal_store(0.0, p + 2 * m + 1);
        else __builtin_nontemporal_store((vx_d2){0.0, 0.0}, reinterpret_cast<vx_d2*>(p + 2 * m));
    }
}
__device__ __forceinline__ void zero_column(const Grid& g, int i, int j, int nd, int lane, double* __restrict__ Aez,
                                            double* __restrict__ Anz, double* __restrict__ Abx,
                                            double* __restrict__ Aby, double* __restrict__ K11,
                                            double* __restrict__ K22, double* __restrict__ K33) {
    const uint32_t c0 = ((uint32_t)i * (uint32_t)g.Y + (uint32_t)j) * (uint32_t)g.nz;
    if (j >= 2) {
        zero_ai_run(Aez + 4u * c0, nd, lane, true);
        zero_run(K11 + c0, nd, lane);
    }
    if (i >= 2) {
        zero_ai_run(Anz + 4u * c0, nd, lane, true);
        zero_run(K22 + c0, nd, lane);
    }
    if (i >= 2 && j >= 2) {
        const int nt = nd < g.nz - 1 ? nd : g.nz - 1;  // top faces: levels below nz-1
        zero_ai_run(Abx + 4u * c0, nt, lane, false);
        zero_ai_run(Aby + 4u * c0, nt, lane, false);
        zero_run(K33 + c0, nd, lane);  // a dry column's top level too
    }
}

// The values of one cell's stencil, in flight: the tracers at the cell c, its
// east (e), west (w), north (n) and south (s) neighbours, levels k, k+1 (p) and
// k-1 (m), and the diffusivity.
struct PreIn {
    double Tc, Tcp, Tcm, Te, Tep, Tem, Tw, Twp, Tn, Tnp, Tnm, Ts, Tsp;
    double Sc, Scp, Scm, Se, Sep, Sem, Sw, Swp, Sn, Snp, Snm, Ss, Ssp;
    double Kc, Kcl, Ke, Kel, Kn, Knl;
};
// Loaded whether or not they are used (k+1 at the top and k-1 at the bottom
// are cells of the next and previous columns, in bounds for every cell pre
// visits, i in [1, X-3], j in [1, Y-3]): a load under a per-lane condition is
// waited for at once. Offsets are 32-bit element offsets (the host checks the
// arrays fit).
__device__ __forceinline__ void pre_load(const Grid& g, const Fields& f, const double* __restrict__ K, int i, int j,
                                         int k, PreIn& v) {
    const uint32_t sj = (uint32_t)g.nz, si = (uint32_t)g.Y * (uint32_t)g.nz;
    const uint32_t c = (uint32_t)i * si + (uint32_t)j * sj + (uint32_t)k;
    const uint32_t ce = c + si, cw = c - si, cn = c + sj, cs = c - sj;
    const double* __restrict__ T = f.T + (uint32_t)f.tau * g.ls;
    const double* __restrict__ S = f.S + (uint32_t)f.tau * g.ls;
    auto L2 = [&](uint32_t o, double& t, double& sv) {
        t = T[g.cs * o];
        sv = S[g.cs * o];
    };
    L2(c, v.Tc, v.Sc);
    L2(c + 1, v.Tcp, v.Scp);
    L2(c - 1, v.Tcm, v.Scm);
    L2(ce, v.Te, v.Se);
    L2(ce + 1, v.Tep, v.Sep);
    L2(ce - 1, v.Tem, v.Sem);
    L2(cw, v.Tw, v.Sw);
    L2(cw + 1, v.Twp, v.Swp);
    L2(cn, v.Tn, v.Sn);
    L2(cn + 1, v.Tnp, v.Snp);
    L2(cn - 1, v.Tnm, v.Snm);
    L2(cs, v.Ts, v.Ss);
    L2(cs + 1, v.Tsp, v.Ssp);
    v.Kc = K[c], v.Kcl = K[c - 1], v.Ke = K[ce], v.Kel = K[ce - 1], v.Kn = K[cn], v.Knl = K[cn - 1];
}

// One wet cell (i, j, k) of isoneutral_diffusion_pre. FUSED: also the face
// fluxes of temperature and salinity at level tau from the tensor just formed
// (the flux kernel's work for the step that follows pre), into `fo`.
template <bool FUSED>
__device__ __forceinline__ void pre_wet_cell(const Grid& g, const Prm& p, const PreIn& v, double* __restrict__ Aez,
                                             double* __restrict__ Anz, double* __restrict__ Abx,
                                             double* __restrict__ Aby, double* __restrict__ K11,
                                             double* __restrict__ K22, double* __restrict__ K33, const PreFlux& fo,
                                             const BlockMetrics& bm, const double dxu_i, const double dxu_w,
                                             const double r4xt, const int i, const int j, const int q, const int k) {
    const int nz = g.nz;
    const ColMetrics& cm = bm.col[q];
    const uint32_t c = ((uint32_t)i * (uint32_t)g.Y + (uint32_t)j) * (uint32_t)nz + (uint32_t)k;
    const bool hp = k < nz - 1, hm = k >= 1;
    const int kb_c = bm.kb[q + 1], kb_e = bm.kbe[q], kb_w = bm.kbw[q];
    const int kb_n = bm.kb[q + 2], kb_s = bm.kb[q];
    auto sel = [](bool ok, double x) { return ok ? x : 0.0; };
    const double Tc = v.Tc, Tcp = sel(hp, v.Tcp), Tcm = sel(hm, v.Tcm), Te = v.Te, Tep = sel(hp, v.Tep);
    const double Tem = sel(hm, v.Tem), Tw = v.Tw, Twp = sel(hp, v.Twp), Tn = v.Tn, Tnp = sel(hp, v.Tnp);
    const double Tnm = sel(hm, v.Tnm), Ts = v.Ts, Tsp = sel(hp, v.Tsp);
    const double Sc = v.Sc, Scp = sel(hp, v.Scp), Scm = sel(hm, v.Scm), Se = v.Se, Sep = sel(hp, v.Sep);
    const double Sem = sel(hm, v.Sem), Sw = v.Sw, Swp = sel(hp, v.Swp), Sn = v.Sn, Snp = sel(hp, v.Snp);
    const double Snm = sel(hm, v.Snm), Ss = v.Ss, Ssp = sel(hp, v.Ssp);
    const double Kc = v.Kc, Kcm = sel(hm, v.Kcl), Ke = v.Ke, Kem = sel(hm, v.Kel), Kn = v.Kn, Knm = sel(hm, v.Knl);
    const double dzw_k = bm.lev.dzw[k], dzw_m = hm ? bm.lev.dzw[hm ? k - 1 : k] : 0.0;
    const double r4zt = bm.lev.r4zt[k], r4ztl = bm.lev.r4ztl[k];

    // reciprocal metric factors
    const double rz_c = hp ? bm.lev.rzw[k] : 0.0;
    const double rz_m = hm ? bm.lev.rzw[hm ? k - 1 : k] : 0.0;
    const double rx_c = cm.rx, ry_c = cm.ry;

    // masked face gradients (veros/core/isoneutral/isoneutral.py:46-95)
    auto G = [](double m, double a1, double a0, double b1, double b0, double rd) -> Grad {
        return {m * (a1 - a0) * rd, m * (b1 - b0) * rd};
    };
    const double mc = m01(kb_c, k), mcp = m01(kb_c, k + 1), mcm = m01(kb_c, k - 1);
    const double me = m01(kb_e, k), mep = m01(kb_e, k + 1), mem = m01(kb_e, k - 1);
    const double mn = m01(kb_n, k), mnp = m01(kb_n, k + 1), mnm = m01(kb_n, k - 1);
    const Grad gz_c = hp ? G(mc * mcp, Tcp, Tc, Scp, Sc, rz_c) : Grad{0.0, 0.0};
    const Grad gz_m = hm ? G(mcm * mc, Tc, Tcm, Sc, Scm, rz_m) : Grad{0.0, 0.0};

    const double tds = 2.0 / p.iso_dslope;
    const ExpCoef ec = load_exp_coef();

    // Two triads belong to two faces of this cell: east (ip=0, kr=1) is the
    // top-face x triad (ip=1, kr=0) and north (jp=0, kr=1) the top-face y triad
    // (jp=1, kr=0); same density point, same gradients, so the same slope
    // and taper, formed once here.
    const Dens w_c = dens(p, mc);
    const double rd_c = rden(dot(w_c, gz_c));
    double sl_x = 0.0, tp_x = 0.0, sl_y = 0.0, tp_y = 0.0;
    if (j >= 2) {
        sl_x = -dot(w_c, G(mc * me, Te, Tc, Se, Sc, rx_c)) * rd_c;
        tp_x = taper(p, ec, tds, sl_x);
    }
    if (i >= 2) {
        sl_y = -dot(w_c, G(mc * mn, Tn, Tc, Sn, Sc, ry_c)) * rd_c;
        tp_y = taper(p, ec, tds, sl_y);
    }

    // --- east face (i+1/2, j, k), j in [2, Y-2)   (:97-132)
    if (j >= 2) {
        const double mU = mc * me;
        const Grad gx = G(mU, Te, Tc, Se, Sc, rx_c);
        const Grad gz_e = hp ? G(me * mep, Tep, Te, Sep, Se, rz_c) : Grad{0.0, 0.0};
        const Grad gz_em = hm ? G(mem * me, Te, Tem, Se, Sem, rz_m) : Grad{0.0, 0.0};
        const double diffloc = hm ? 0.25 * (Kc + Kcm + Ke + Kem) : 0.5 * (Kc + Ke);
        double sumz = 0.0;
        double out[4];
#pragma unroll
        for (int kr = 0; kr < 2; ++kr) {
#pragma unroll
            for (int ip = 0; ip < 2; ++ip) {
                out[ip * 2 + kr] = 0.0;
                if (kr == 0 && !hm) continue;  // levels k >= 1 - kr
                double sl = sl_x, tp = tp_x;
                if (ip != 0 || kr != 1) {
                    const Dens w = dens(p, ip ? me : mc);
                    const Grad& gz = ip ? (kr ? gz_e : gz_em) : (kr ? gz_c : gz_m);
                    sl = -dot(w, gx) * rden(dot(w, gz));
                    tp = taper(p, ec, tds, sl);
                }
                sumz += (kr ? dzw_k : dzw_m) * mU * fmax(p.K_iso_steep, diffloc * tp);
                out[ip * 2 + kr] = tp * sl * mU;
            }
        }
        if (hm) {
            *reinterpret_cast<double2*>(Aez + 4u * c) = make_double2(out[0], out[1]);
        } else {
            Aez[4u * c + 1] = out[1];  // (ip=0, kr=0) keeps its value at k = 0
        }
        if (hm) {
            *reinterpret_cast<double2*>(Aez + 4u * c + 2) = make_double2(out[2], out[3]);
        } else {
            Aez[4u * c + 3] = out[3];
        }
        const double k11v = scaled(sumz, r4zt, r4ztl);
        K11[c] = k11v;
        if constexpr (FUSED) {
            // at level 0 the kr = 0 entries keep their values (their tracer
            // differences vanish there)
            const double a0 = hm ? out[0] : Aez[4u * c], a2 = hm ? out[2] : Aez[4u * c + 2];
            const double2 A01 = make_double2(a0, out[1]), A23 = make_double2(a2, out[3]);
            const double feT = east_flux_core(diffloc, A01, A23, Tc, hp ? Tcp : Tc, hm ? Tcm : Tc, Te, hp ? Tep : Te,
                hm ? Tem : Te, r4zt, rx_c, k11v);
            const double feS = east_flux_core(diffloc, A01, A23, Sc, hp ? Scp : Sc, hm ? Scm : Sc, Se, hp ? Sep : Se,
                hm ? Sem : Se, r4zt, rx_c, k11v);
            store_pair(fo.fe + 2u * c, feT, feS);
        }
    }

    // --- north face (i, j+1/2, k), i in [2, X-2)   (:134-168)
    if (i >= 2) {
        const double mV = mc * mn;
        const Grad gy = G(mV, Tn, Tc, Sn, Sc, ry_c);
        const Grad gz_n = hp ? G(mn * mnp, Tnp, Tn, Snp, Sn, rz_c) : Grad{0.0, 0.0};
        const Grad gz_nm = hm ? G(mnm * mn, Tn, Tnm, Sn, Snm, rz_m) : Grad{0.0, 0.0};
        const double diffloc = hm ? 0.25 * (Kc + Kcm + Kn + Knm) : 0.5 * (Kc + Kn);
        double sumz = 0.0;
        double out[4];
#pragma unroll
        for (int kr = 0; kr < 2; ++kr) {
#pragma unroll
            for (int jp = 0; jp < 2; ++jp) {
                out[jp * 2 + kr] = 0.0;
                if (kr == 0 && !hm) continue;
                double sl = sl_y, tp = tp_y;
                if (jp != 0 || kr != 1) {
                    const Dens w = dens(p, jp ? mn : mc);
                    const Grad& gz = jp ? (kr ? gz_n : gz_nm) : (kr ? gz_c : gz_m);
                    sl = -dot(w, gy) * rden(dot(w, gz));
                    tp = taper(p, ec, tds, sl);
                }
                sumz += (kr ? dzw_k : dzw_m) * mV * fmax(p.K_iso_steep, diffloc * tp);
                out[jp * 2 + kr] = tp * sl * mV;
            }
        }
        if (hm) {
            *reinterpret_cast<double2*>(Anz + 4u * c) = make_double2(out[0], out[1]);
            *reinterpret_cast<double2*>(Anz + 4u * c + 2) = make_double2(out[2], out[3]);
        } else {
            Anz[4u * c + 1] = out[1];
            Anz[4u * c + 3] = out[3];
        }
        const double k22v = scaled(sumz, r4zt, r4ztl);
        K22[c] = k22v;
        if constexpr (FUSED) {
            const double a0 = hm ? out[0] : Anz[4u * c], a2 = hm ? out[2] : Anz[4u * c + 2];
            const double2 A01 = make_double2(a0, out[1]), A23 = make_double2(a2, out[3]);
            const double fnT = north_flux_core(diffloc, A01, A23, Tc, hp ? Tcp : Tc, hm ? Tcm : Tc, Tn, hp ? Tnp : Tn,
                hm ? Tnm : Tn, r4zt, cm.cosu, ry_c, k22v);
            const double fnS = north_flux_core(diffloc, A01, A23, Sc, hp ? Scp : Sc, hm ? Scm : Sc, Sn, hp ? Snp : Sn,
                hm ? Snm : Sn, r4zt, cm.cosu, ry_c, k22v);
            store_pair(fo.fn + 2u * c, fnT, fnS);
        }
    }

    // --- top face (i, j, k+1/2), i, j in [2, X/Y-2), k < nz-1   (:170-225)
    if (i >= 2 && j >= 2 && hp) {
        const int kb_w2 = kb_w, kb_s2 = kb_s;
        const double mW = mc * mcp;
        const double rx_w = cm.rxw, ry_s = cm.rys;
        const double mw = m01(kb_w2, k), mwp = m01(kb_w2, k + 1);
        const double ms = m01(kb_s2, k), msp = m01(kb_s2, k + 1);
        // horizontal gradients at (i-1+ip, k+kr) and (j-1+jp, k+kr)
        const Grad gx_w = G(mw * mc, Tc, Tw, Sc, Sw, rx_w);
        const Grad gx_wp = G(mwp * mcp, Tcp, Twp, Scp, Swp, rx_w);
        const Grad gx_c = G(mc * me, Te, Tc, Se, Sc, rx_c);
        const Grad gx_cp = G(mcp * mep, Tep, Tcp, Sep, Scp, rx_c);
        const Grad gy_s = G(ms * mc, Tc, Ts, Sc, Ss, ry_s);
        const Grad gy_sp = G(msp * mcp, Tcp, Tsp, Scp, Ssp, ry_s);
        const Grad gy_c = G(mc * mn, Tn, Tc, Sn, Sc, ry_c);
        const Grad gy_cp = G(mcp * mnp, Tnp, Tcp, Snp, Scp, ry_c);
        double sumx = 0.0, sumy = 0.0;
        double ox[4], oy[4];
#pragma unroll
        for (int kr = 0; kr < 2; ++kr) {
            const Dens w = dens(p, kr ? mcp : mc);
            const double rd = kr ? rden(dot(w, gz_c)) : rd_c;
#pragma unroll
            for (int ip = 0; ip < 2; ++ip) {
                double sl = sl_x, tp = tp_x;
                if (ip != 1 || kr != 0) {
                    const Grad& gx = ip ? (kr ? gx_cp : gx_c) : (kr ? gx_wp : gx_w);
                    sl = -dot(w, gx) * rd;
                    tp = taper(p, ec, tds, sl);
                }
                sumx += (ip ? dxu_i : dxu_w) * Kc * tp * (sl * sl) * mW;
                ox[ip * 2 + kr] = tp * sl * mW;
            }
#pragma unroll
            for (int jp = 0; jp < 2; ++jp) {
                double sl = sl_y, tp = tp_y;
                if (jp != 1 || kr != 0) {
                    const Grad& gy = jp ? (kr ? gy_cp : gy_c) : (kr ? gy_sp : gy_s);
                    sl = -dot(w, gy) * rd;
                    tp = taper(p, ec, tds, sl);
                }
                const double facty = jp ? cm.fyc : cm.fys;
                sumy += facty * Kc * tp * (sl * sl) * mW;
                oy[jp * 2 + kr] = tp * sl * mW;
            }
        }
        *reinterpret_cast<double2*>(Abx + 4u * c) = make_double2(ox[0], ox[1]);
        *reinterpret_cast<double2*>(Abx + 4u * c + 2) = make_double2(ox[2], ox[3]);
        *reinterpret_cast<double2*>(Aby + 4u * c) = make_double2(oy[0], oy[1]);
        *reinterpret_cast<double2*>(Aby + 4u * c + 2) = make_double2(oy[2], oy[3]);
        K33[c] = sumx * r4xt + sumy * cm.ryt;
        if constexpr (FUSED) {
            const double2 B01 = make_double2(ox[0], ox[1]), B23 = make_double2(ox[2], ox[3]);
            const double2 C01 = make_double2(oy[0], oy[1]), C23 = make_double2(oy[2], oy[3]);
            const double ftT = top_flux_core(Kc, B01, B23, C01, C23, Tc, Tcp, Tw, Twp, Te, Tep, Ts, Tsp, Tn, Tnp, cm,
                r4xt);
            const double ftS = top_flux_core(Kc, B01, B23, C01, C23, Sc, Scp, Sw, Swp, Se, Sep, Ss, Ssp, Sn, Snp, cm,
                r4xt);
            store_pair(fo.ft + 2u * c, ftT, ftS);
        }
    }
    if (i >= 2 && j >= 2 && !hp) {
        K33[c] = 0.0;  // (:225)
        if constexpr (FUSED) {  // no flux through the top level
            store_pair(fo.ft + 2u * c, 0.0, 0.0);
        }
    }
}

// isoneutral_diffusion_pre. Block-local compaction: a block (one wave) owns the
// columns (i, jb .. jb+ncb-1); their wet cells (the wet suffixes) are numbered
// in column order and taken 64 at a time, so the slope work fills the wave
// whatever the land fraction; the dry cells of its columns are zeroed last.
//
// A wave waits for its memory operations in order, so a load issued after
// stores waits until those are acknowledged, which takes several microseconds
// where writes are the bound: the next round's stencil is therefore loaded
// before the current round is computed and stored, and the zeros go out when
// no load is left to wait for. The two stencils in flight take the registers
// of two waves per SIMD (three spill them and lose more than they hide).
// Bound by writes: on 1440x720x80 (35% land) the fused call takes 4.58 ms
// without the 8.7 GB of zeros and 6.04 ms with them; the zeros alone, by a
// kernel of their own beside this one on a helper stream, and 183 registers of
// divisions in this one: 6.10 ms. The same on 360x160x60 (levels innermost, all
// isoneutral calls of a step): 1355 -> 1160 us; 90x40x15, pre + T + S: 77 -> 54 us
// (no second stream to fork and join).
template <bool FUSED>
__global__ __launch_bounds__(kCellBlock) __attribute__((amdgpu_waves_per_eu(VX_PRE_MIN_WAVES))) void iso_pre_kernel(
    Grid g, Prm p, Fields f, const double* __restrict__ K, double* __restrict__ Aez, double* __restrict__ Anz,
    double* __restrict__ Abx, double* __restrict__ Aby, double* __restrict__ K11, double* __restrict__ K22,
    double* __restrict__ K33, PreFlux fo, int ncb) {
    __shared__ BlockMetrics bm;
    const int tid = (int)threadIdx.x, nz = g.nz;
    // K_33[..., nz-1] = 0 (veros/core/isoneutral/isoneutral.py:225) of the halo
    // columns: rows 0, 1, X-2, X-1, then columns 0, 1, Y-2, Y-1
    for (int64_t c = (int64_t)blockIdx.x * kCellBlock + tid; c < 4 * ((int64_t)g.X + g.Y);
         c += (int64_t)gridDim.x * kCellBlock) {
        const bool row = c < 4 * (int64_t)g.Y;
        const int64_t r = row ? c : c - 4 * (int64_t)g.Y;
        const int64_t n = row ? g.Y : g.X;
        const int64_t h = r / n, m = r - h * n;  // which of the four, where along it
        const int64_t e = h < 2 ? h : (row ? g.X : g.Y) - 4 + h;
        K33[((row ? e * g.Y + m : m * g.Y + e) + 1) * nz - 1] = 0.0;
    }
    const BlockCols bc = block_cols(1, g.X - 3, 1, g.Y - 3, ncb, strip_blocks(kPreStripCols, ncb, g.Y - 3));
    if (!bc.valid) return;  // padding block (uniform)
    const int i = bc.i, jb = bc.j;
    fill_metrics(g, i, jb, ncb, bm);
    __syncthreads();
    if (tid < ncb) {
        const bool have = jb + tid <= g.Y - 3;
        const int kbq = bm.kb[tid + 1];
        const int n = (have && kbq >= 1 && kbq <= nz) ? nz - kbq + 1 : 0;
        bm.run[tid + 1] = n;
    }
    __syncthreads();
    scan_runs(bm.run, ncb);
    __syncthreads();
    const int nwet = bm.run[ncb];
    const double dxu_i = g.dxu[i], dxu_w = g.dxu[i - 1], r4xt = 1.0 / (4 * g.dxt[i]);
    if (nwet > 0) {
        // this lane's cell of a round (a lane past the last cell: that cell, not stored)
        auto locate = [&](int t, int& q, int& k) {
            const int tt = t < nwet ? t : nwet - 1;
            q = run_column(bm.run, ncb, tt);
            k = nz - (bm.run[q + 1] - bm.run[q]) + (tt - bm.run[q]);  // wet suffix of column q
        };
        int q, k;
        PreIn v;
        locate(tid, q, k);
        pre_load(g, f, K, i, jb + q, k, v);
        for (int t0 = 0;;) {
            const bool more = t0 + kCellBlock < nwet;
            int qn = q, kn = k;
            PreIn vn;
            if (more) {
                locate(t0 + kCellBlock + tid, qn, kn);
                pre_load(g, f, K, i, jb + qn, kn, vn);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (t0 + tid < nwet)
                pre_wet_cell<FUSED>(g, p, v, Aez, Anz, Abx, Aby, K11, K22, K33, fo, bm, dxu_i, dxu_w, r4xt, i, jb + q,
                                    q, k);
            if (!more) break;
            t0 += kCellBlock;
            q = qn;
            k = kn;
            v = vn;
        }
    }
    for (int q = 0; q < ncb && jb + q <= g.Y - 3; ++q) {
        const int nd = nz - (bm.run[q + 1] - bm.run[q]);
        if (nd > 0) zero_column(g, i, jb + q, nd, tid, Aez, Anz, Abx, Aby, K11, K22, K33);
    }
}

// ---------------------------------------------------------------------------
// Tracer step (veros/core/isoneutral/diffusion.py:9-283 with
// veros/core/diffusion.py:9-62), NTR tracers sharing one pass over the
// isoneutral tensor, covering (i, j) in [1, X-1) x [1, Y-1):
//   iso_flux_kernel (thread per cell): the face fluxes -> workspace (in the
//     fused pre + temperature/salinity call, iso_pre_kernel<true> instead)
//   iso_step_wet_kernel phase 1 (thread per wet cell): lateral dissipation on
//     T points, the flux divergence, rhs = tr[taup1] + dt*dtr, and the K33
//     rows -> LDS
//   phase 2 (8 lanes per interior column and tracer): segmented elimination in LDS
//   phase 3 (thread per wet cell): tracer, dtr_iso and P_diss updates
// ---------------------------------------------------------------------------
struct TracerArgs {
    double* tr;           // (X, Y, nz, 3)
    double* dtr;          // (X, Y, nz)
    const double* I;      // int_drhodX (X, Y, nz, 3), nullable
};

struct StepArgs {
    TracerArgs t[2];
    // workspace: flux_east, flux_north, flux_top, (X, Y, nz) cells with the
    // tracers' values side by side
    double *fe, *fn, *ft;
    int tau, taup1;
    // K1 = K_iso - K_skew (east/north faces), K2 = K_iso + K_skew (top faces);
    // a null pointer is a zero term (veros/core/isoneutral/diffusion.py:15-16,180-188)
    const double* Kiso;
    const double* Kskew;
    const double *Aez, *Anz, *Abx, *Aby, *K11, *K22, *K33;
    double* P;            // P_diss_iso / P_diss_skew, nullable (energy branch off)
};

// K1 = K_iso - K_skew (east/north faces) and K2 = K_iso + K_skew (top faces)
// (veros/core/isoneutral/diffusion.py:15-16,180-188); one of the two is zero.
template <bool ISO>
__device__ __forceinline__ double k1_of(double K) { return ISO ? K : 0.0 - K; }
template <bool ISO>
__device__ __forceinline__ double k2_of(double K) { return ISO ? K : 0.0 + K; }

// Face fluxes of NTR tracers (veros/core/isoneutral/diffusion.py:9-113):
// flux_east for (i, j) in [1, X-3] x [2, Y-3], flux_north for [2, X-3] x
// [1, Y-3], flux_top for [2, X-3] x [2, Y-3] (0 at the top level); the tracers
// share every read of the isoneutral tensor. Every use of a face flux is
// multiplied by the maskT of a cell next to the face (the divergence, the
// lateral dissipation and the vertical mixing term of that cell), so only the
// faces touching a wet cell are formed and written; the step kernel reads no
// other. The cells that need one are compacted like the wet-cell pre kernel's:
// a column (i, j) needs levels from the lowest of its own wet
// cells, the top face of the dry cell below them, and the wet cells of its east
// and north neighbours, up to nz-1 (one contiguous run); a block owns ncb
// columns of row i and deals their runs round-robin to its threads. The
// tracer stencil is read straight from global memory (every read issued
// before the first flux), so no lane of a dry region is launched.
__device__ __forceinline__ int first_wet(int kb, int nz) { return (kb >= 1 && kb <= nz) ? kb - 1 : nz; }
// first level of the run of block column q (row i, column j)
__device__ __forceinline__ int flux_run_start(const BlockMetrics& m, int nz, int i, int j, int q) {
    const int fc = first_wet(m.kb[q + 1], nz);
    int s0 = fc < nz ? (fc >= 1 ? fc - 1 : 0) : nz;             // top face of the dry cell below
    const int fe = j >= 2 ? first_wet(m.kbe[q], nz) : nz;
    const int fn = i >= 2 ? first_wet(m.kb[q + 2], nz) : nz;
    s0 = fe < s0 ? fe : s0;
    return fn < s0 ? fn : s0;
}

typedef unsigned int vx_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ double2 buf_load2(BufRsrc b, uint32_t off) {
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
}
__device__ __forceinline__ void buf_store2(BufRsrc b, uint32_t off, double2 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vx_u4, v), b, off, 0, 0);
}

// Every read is a buffer load at an offset that is past the buffer's end where
// the cell does not need it (no traffic, no branch around the load, all of a
// cell's loads in flight together). A block's cells lie in the columns
// jb-1 .. jb+ncb of the rows i-1, i, i+1: one buffer per row and array, from
// column jb-1 on. On 360x160x60, levels innermost, one tracer: 142 us with the
// loads under the conditions of their faces, 121 now.
template <int NTR, bool ISO>
__global__ __launch_bounds__(kCellBlock) void iso_flux_kernel(Grid g, StepArgs a, int ncb) {
    __shared__ BlockMetrics bm;
    const BlockCols bc = block_cols(1, g.X - 3, 1, g.Y - 3, ncb, strip_blocks(kPreStripCols, ncb, g.Y - 3));
    if (!bc.valid) return;  // padding block (uniform)
    const int nz = g.nz, i = bc.i, jb = bc.j;
    const int tid = (int)threadIdx.x, nthr = (int)blockDim.x;
    fill_metrics(g, i, jb, ncb, bm);
    __syncthreads();
    for (int q = tid; q < ncb; q += nthr)
        bm.run[q + 1] = jb + q <= g.Y - 3 ? nz - flux_run_start(bm, nz, i, jb + q, q) : 0;
    __syncthreads();
    scan_runs(bm.run, ncb);
    __syncthreads();
    const int ncell = bm.run[ncb];
    const uint32_t sj = (uint32_t)nz;
    const double r4xt = 1.0 / (4 * g.dxt[i]);
    // the rows' cells from column jb-1 on, up to column jb+ncb or the row's end
    const int64_t row = (int64_t)g.Y * nz, o0 = (int64_t)i * row + (int64_t)(jb - 1) * nz;
    const uint32_t ncells = (uint32_t)(jb + ncb < g.Y ? ncb + 2 : g.Y - jb + 1) * (uint32_t)nz;
    const double* Kf = ISO ? a.Kiso : a.Kskew;
    const BufRsrc bK = make_buf(Kf + o0, ncells * 8u), bKe = make_buf(Kf + o0 + row, ncells * 8u);
    const BufRsrc bez = make_buf(a.Aez + 4 * o0, ncells * 32u), bnz = make_buf(a.Anz + 4 * o0, ncells * 32u);
    const BufRsrc bbx = make_buf(a.Abx + 4 * o0, ncells * 32u), bby = make_buf(a.Aby + 4 * o0, ncells * 32u);
    const BufRsrc b11 = make_buf(a.K11 + o0, ncells * 8u), b22 = make_buf(a.K22 + o0, ncells * 8u);
    const uint32_t cb = 8u * g.cs;  // bytes from a level to the next in the time-level arrays
    for (int t = tid; t < ncell; t += nthr) {
        const int q = run_column(bm.run, ncb, t);
        const int j = jb + q;
        const int k = nz - (bm.run[q + 1] - bm.run[q]) + (t - bm.run[q]);
        const int kb = bm.kb[q + 1], kb_e = bm.kbe[q], kb_n = bm.kb[q + 2];
        const bool wc = wet(kb, k);
        const bool need_e = j >= 2 && (wc || wet(kb_e, k));
        const bool need_n = i >= 2 && (wc || wet(kb_n, k));
        const bool need_t = i >= 2 && j >= 2 && (wc || (k + 1 < nz && wet(kb, k + 1)));
        const bool hm = k >= 1, hp = k + 1 < nz;
        const bool top = need_t && hp, any = need_e || need_n || need_t;
        const uint32_t e = (uint32_t)(q + 1) * sj + (uint32_t)k;  // cell in the buffers
        const uint32_t up = hp ? 1u : 0u, dn = hm ? 1u : 0u;      // pad_z_edges clamping
        auto at = [](bool on, uint32_t off) { return on ? off : kNoAccess; };
        const double K_c = buf_load(bK, at(any, 8u * e)), K_cm = buf_load(bK, at(any && hm, 8u * (e - 1u)));
        const double K_e = buf_load(bKe, at(need_e, 8u * e)), K_em = buf_load(bKe, at(need_e && hm, 8u * (e - 1u)));
        const double K_n = buf_load(bK, at(need_n, 8u * (e + sj)));
        const double K_nm = buf_load(bK, at(need_n && hm, 8u * (e + sj - 1u)));
        const uint32_t oe = at(need_e, 32u * e), on = at(need_n, 32u * e), ot = at(top, 32u * e);
        const double2 ez01 = buf_load2(bez, oe), ez23 = buf_load2(bez, oe + 16u);
        const double2 nz01 = buf_load2(bnz, on), nz23 = buf_load2(bnz, on + 16u);
        const double2 bx01 = buf_load2(bbx, ot), bx23 = buf_load2(bbx, ot + 16u);
        const double2 by01 = buf_load2(bby, ot), by23 = buf_load2(bby, ot + 16u);
        const double K11 = buf_load(b11, at(need_e, 8u * e)), K22 = buf_load(b22, at(need_n, 8u * e));
        // tracer at level tau: centre and east/north columns at k, k+up, k-dn;
        // west/south at k, k+1 (top faces only)
        double Tc[NTR], Tcu[NTR], Tcd[NTR], Te[NTR], Teu[NTR], Ted[NTR], Tn[NTR], Tnu[NTR], Tnd[NTR];
        double Tw[NTR], Twu[NTR], Ts[NTR], Tsu[NTR];
        const bool ue = need_e || top, un = need_n || top;
#pragma unroll
        for (int r = 0; r < NTR; ++r) {
            const double* T = a.t[r].tr + (int64_t)a.tau * g.ls + o0 * g.cs;
            const BufRsrc bT = make_buf(T, ncells * cb), bTe = make_buf(T + row * g.cs, ncells * cb);
            const BufRsrc bTw = make_buf(T - row * g.cs, ncells * cb);
            Tc[r] = buf_load(bT, at(any, cb * e));
            Tcu[r] = buf_load(bT, at(any, cb * (e + up)));
            Tcd[r] = buf_load(bT, at(any, cb * (e - dn)));
            Te[r] = buf_load(bTe, at(ue, cb * e));
            Teu[r] = buf_load(bTe, at(ue, cb * (e + up)));
            Ted[r] = buf_load(bTe, at(need_e, cb * (e - dn)));
            Tn[r] = buf_load(bT, at(un, cb * (e + sj)));
            Tnu[r] = buf_load(bT, at(un, cb * (e + sj + up)));
            Tnd[r] = buf_load(bT, at(need_n, cb * (e + sj - dn)));
            Tw[r] = buf_load(bTw, at(top, cb * e));
            Twu[r] = buf_load(bTw, at(top, cb * (e + 1u)));
            Ts[r] = buf_load(bT, at(top, cb * (e - sj)));
            Tsu[r] = buf_load(bT, at(top, cb * (e - sj + 1u)));
        }
        // flux_east (:22-47), flux_north (:49-77), flux_top (:79-111)
        const ColMetrics& cm = bm.col[q];
        const double r4zt = bm.lev.r4zt[k];
        const double dl_e = hm ? 0.25 * (k1_of<ISO>(K_c) + k1_of<ISO>(K_cm) + k1_of<ISO>(K_e) + k1_of<ISO>(K_em))
                               : 0.5 * (k1_of<ISO>(K_c) + k1_of<ISO>(K_e));
        const double dl_n = hm ? 0.25 * (k1_of<ISO>(K_c) + k1_of<ISO>(K_cm) + k1_of<ISO>(K_n) + k1_of<ISO>(K_nm))
                               : 0.5 * (k1_of<ISO>(K_c) + k1_of<ISO>(K_n));
        double fe[NTR], fn[NTR], ft[NTR];
#pragma unroll
        for (int r = 0; r < NTR; ++r) {
            fe[r] = east_flux_core(dl_e, ez01, ez23, Tc[r], Tcu[r], Tcd[r], Te[r], Teu[r], Ted[r], r4zt, cm.rx, K11);
            fn[r] = north_flux_core(dl_n, nz01, nz23, Tc[r], Tcu[r], Tcd[r], Tn[r], Tnu[r], Tnd[r], r4zt, cm.cosu,
                                    cm.ry, K22);
            const double ftv = top_flux_core(k2_of<ISO>(K_c), bx01, bx23, by01, by23, Tc[r], Tcu[r], Tw[r], Twu[r],
                                             Te[r], Teu[r], Ts[r], Tsu[r], Tn[r], Tnu[r], cm, r4xt);
            ft[r] = top ? ftv : 0.0;
        }
        constexpr uint32_t fb = 8u * NTR;  // bytes of a cell's fluxes
        auto put = [&](double* f, bool on, const double (&v)[NTR]) {
            const BufRsrc bf = make_buf(f + o0 * NTR, ncells * fb);
            if constexpr (NTR == 2) buf_store2(bf, at(on, fb * e), make_double2(v[0], v[1]));
            else buf_store(bf, at(on, fb * e), v[0]);
        };
        put(a.fe, need_e, fe);
        put(a.fn, need_n, fn);
        put(a.ft, need_t, ft);
    }
}

constexpr int kStepThreads = 256;  // threads of a tracer-step block, and the most cells of a group
constexpr int kStepCols = 64;      // most columns of a block

// One column's K33 system (rows a, b, c of n levels in LDS, right-hand side
// in r) solved in place into r by the kSegP lanes of a group, lane sg owning
// the rows [sg * S, sg * S + S) with S = max(2, ceil(n / kSegP)); rows from n
// on are identity rows. Each lane eliminates its interior rows with the spike
// from the row below (q: c', then gamma; w: the spike, then beta; r: dp, then
// alpha), the interface rows are solved across the group (iface_solve), and
// each lane writes its rows of x = alpha + beta L_{s-1} + gamma L_s. Every
// lane of the group must call it.
__device__ __forceinline__ void seg_lds_column(const double* a, const double* b, const double* c, double* r,
                                               double* q, double* w, int n, int sg) {
    const int S = max(2, (n + kSegP - 1) / kSegP);
    const int m0 = sg * S;
    auto A = [&](int m) { return m < n ? a[m] : 0.0; };
    auto B = [&](int m) { return m < n ? b[m] : 1.0; };
    auto C = [&](int m) { return m < n ? c[m] : 0.0; };
    auto D = [&](int m) { return m < n ? r[m] : 0.0; };
    // forward sweep over the interior rows t = 0 .. S-2 (c', spike, dp to LDS)
    double cp = 0.0, wp = 0.0, dp = 0.0;
    for (int t = 0; t < S - 1; ++t) {
        const int m = m0 + t;
        const double at = A(m);
        const double rr = seg_rcp(t == 0 ? B(m) : B(m) - at * cp);
        cp = C(m) * rr;
        wp = (t == 0 ? at : -at * wp) * rr;
        dp = (t == 0 ? D(m) : D(m) - at * dp) * rr;
        if (m < n) {
            q[m] = cp;
            w[m] = wp;
            r[m] = dp;
        }
    }
    // back substitution: alpha, beta, gamma of the interior rows (rows past
    // the run have c' = spike = dp = 0)
    const double alS = dp, beS = -wp, gaS = -cp;  // row S-2
    if (m0 + S - 2 < n) {
        r[m0 + S - 2] = alS;
        w[m0 + S - 2] = beS;
        q[m0 + S - 2] = gaS;
    }
    double al = alS, be = beS, ga = gaS;
    for (int t = S - 3; t >= 0; --t) {
        const int m = m0 + t;
        const bool real = m < n;
        const double cpt = real ? q[m] : 0.0, dpt = real ? r[m] : 0.0, wpt = real ? w[m] : 0.0;
        al = dpt - cpt * al;
        be = -wpt - cpt * be;
        ga = -cpt * ga;
        if (real) {
            r[m] = al;
            w[m] = be;
            q[m] = ga;
        }
    }
    // the interface row (row S-1) with the next segment's row 0 by DPP
    const int mL = m0 + S - 1;
    const double aL = A(mL), bL = B(mL), cL = C(mL), dL = D(mL);
    const double n_al = grp_next(sg, al), n_be = grp_next(sg, be), n_ga = grp_next(sg, ga);
    const double RA = aL * beS;
    const double RB = bL + aL * gaS + cL * n_be;
    const double RC = cL * n_ga;
    const double RD[1] = {dL - aL * alS - cL * n_al};
    double Ls[1], Lm[1];
    iface_solve<1>(sg, RA, RB, RC, RD, Ls, Lm);
    for (int t = 0; t < S - 1; ++t) {
        const int m = m0 + t;
        if (m < n) r[m] = r[m] + w[m] * Lm[0] + q[m] * Ls[0];
    }
    if (mL < n) r[mL] = Ls[0];
}

// Per-block tables of the tracer step, in LDS.
struct StepTables {
    double rxc[kStepCols], ryc[kStepCols];             // 1 / (dxt cost), 1 / (dyt cost)
    double rzt[kMaxNz], rzw[kMaxNz], dzw[kMaxNz];      // 1 / dzt, 1 / dzw, dzw
    int kb[kStepCols + 1], kbw[kStepCols];             // kbot at j-1 .. of row i; at row i-1
    int off[kStepCols + 1];                            // prefix sums of the columns' wet cells
    double rdt, g05, gr;                               // 1 / dt, grav / (2 rho_0), -grav / rho_0
};

// One lane's cell of a group of columns.
struct StepCell {
    int q, k, kb;
    uint32_t e;  // cells from the block's first column's level 0
    bool have, interior;
};
// The global reads of one cell. Every lane loads (a lane past the group's last
// cell that cell's values), at an offset inside the arrays; what a cell does
// not have reads a value it has and is set to zero afterwards.
template <int NTR>
struct StepIn {
    double fe_c[NTR], fe_w[NTR], fn_c[NTR], fn_s[NTR], ft_c[NTR], ft_b[NTR];
    double Ic[NTR], Ie[NTR], Iw[NTR], In[NTR], Is[NTR], Iu[NTR], trp[NTR], dtr0[NTR];
    double K33k, K33m, P0;
};
// Loads at a byte offset from a pointer that is the same for the whole wave:
// held in scalar registers, they need one vector register of address.
template <class V>
__device__ __forceinline__ V load_at(const double* base, uint32_t off) {
    typedef const __attribute__((address_space(1))) char* gptr;
    gptr p = (gptr)base;
    asm("" : "+s"(p));
    return *(const __attribute__((address_space(1))) V*)(p + off);
}
template <int NTR>
__device__ __forceinline__ void load_fluxes(const double* base, uint32_t e, double (&v)[NTR]) {
    if constexpr (NTR == 2) {
        const vx_d2a8 w = load_at<vx_d2a8>(base, 16u * e);
        v[0] = w.x;
        v[1] = w.y;
    } else {
        v[0] = load_at<double>(base, 8u * e);
    }
}
// o0: the cell of the block's first column's level 0; offsets start one column
// before it, so that they stay positive for the south column and level k-1
template <int NTR, bool IMPLICIT, bool WETFLUX>
__device__ __forceinline__ void step_load(const Grid& g, const StepArgs& a, const StepTables& tb, int64_t o0,
                                          const StepCell& s, StepIn<NTR>& v) {
    const uint32_t sj = (uint32_t)g.nz;
    const int64_t b = o0 - g.nz, row = (int64_t)g.Y * g.nz;
    const uint32_t e = s.e + sj;
    const int k = s.k;
    const bool south = !WETFLUX || wet(tb.kb[s.q], k);
    load_fluxes<NTR>(a.fe + NTR * b, e, v.fe_c);
    load_fluxes<NTR>(a.fe + NTR * (b - row), e, v.fe_w);
    load_fluxes<NTR>(a.fn + NTR * b, e, v.fn_c);
    load_fluxes<NTR>(a.fn + NTR * b, south ? e - sj : e, v.fn_s);
    load_fluxes<NTR>(a.ft + NTR * b, e, v.ft_c);
    // the top face of the dry cell below the lowest wet cell
    const bool below = !WETFLUX && k == s.kb - 1 && k >= 1;
    if constexpr (!WETFLUX) load_fluxes<NTR>(a.ft + NTR * b, below ? e - 1u : e, v.ft_b);
    const uint32_t cb = 8u * g.cs;  // bytes from a level to the next in the time-level arrays
#pragma unroll
    for (int t = 0; t < NTR; ++t) {
        v.trp[t] = load_at<double>(a.t[t].tr + (b * g.cs + (int64_t)a.taup1 * g.ls), cb * e);
        v.dtr0[t] = load_at<double>(a.t[t].dtr + b, 8u * e);
    }
    if constexpr (IMPLICIT) {
        v.K33k = load_at<double>(a.K33 + b, 8u * e);
        v.K33m = load_at<double>(a.K33 + b, 8u * (e - 1u));
    }
    v.P0 = 0.0;
    if (a.P) {
        v.P0 = load_at<double>(a.P + b, 8u * e);
#pragma unroll
        for (int t = 0; t < NTR; ++t) {
            const double* I = a.t[t].I + (b * g.cs + (int64_t)a.tau * g.ls);
            v.Ic[t] = load_at<double>(I, cb * e);
            v.Ie[t] = load_at<double>(I + row * g.cs, cb * e);
            v.Iw[t] = load_at<double>(I - row * g.cs, cb * e);
            v.In[t] = load_at<double>(I, cb * (e + sj));
            v.Is[t] = load_at<double>(I, cb * (e - sj));
            v.Iu[t] = load_at<double>(I, cb * (e + 1u));
        }
    }
}
// Fluxes outside the range the flux kernels write (veros/core/isoneutral/
// diffusion.py:22-111), and those of faces touching a dry cell (WETFLUX), are zero.
template <int NTR, bool WETFLUX>
__device__ __forceinline__ void step_mask(const Grid& g, const StepTables& tb, int i, int j, const StepCell& s,
                                          StepIn<NTR>& v) {
    const bool jin = j >= 2 && j <= g.Y - 3, iin = i >= 2 && i <= g.X - 3;
    const bool west = !WETFLUX || wet(tb.kbw[s.q], s.k), south = !WETFLUX || wet(tb.kb[s.q], s.k);
    const bool ec = jin && i <= g.X - 3, ew = jin && i >= 2 && west;
    const bool nc = iin && j <= g.Y - 3, ns = iin && j >= 2 && south;
    const bool below = !WETFLUX && s.k == s.kb - 1 && s.k >= 1;
#pragma unroll
    for (int t = 0; t < NTR; ++t) {
        v.fe_c[t] = ec ? v.fe_c[t] : 0.0;
        v.fe_w[t] = ew ? v.fe_w[t] : 0.0;
        v.fn_c[t] = nc ? v.fn_c[t] : 0.0;
        v.fn_s[t] = ns ? v.fn_s[t] : 0.0;
        if constexpr (!WETFLUX) v.ft_b[t] = below ? v.ft_b[t] : 0.0;
    }
}

// A block owns ncb consecutive columns of row i (strips as in block_cols) and
// steps their wet cells in groups of whole columns, as many as fit its threads:
// thread per cell, except in phase 2. IMPLICIT: the K33 part (isoneutral step);
// else the explicit step only (skew). WETFLUX: the face fluxes exist for wet
// cells only (the fused pre formed them from the tensor it wrote, in which every
// face touching a dry cell carries a zero flux), so a face whose other cell is
// dry counts as zero; else they come from iso_flux_kernel, which writes every
// face of a wet cell, including the top face of the dry cell below the lowest
// wet one. The multiply-adds are written out so that all variants round alike.
//
// Bound by the wait for its loads: a group's 20 loads are issued together, then
// the block computes behind barriers while the CU's other blocks load. Blocks
// over fixed columns replace a plan of all wet cells (three scan kernels a
// call) with groups taken from a counter (four dependent reads before the first
// load), the tracers' fluxes side by side halve the flux loads, and the metric
// factors come from LDS. Four waves per SIMD hold all loads in registers (at
// five they spill: 1440x720x80 5.90 ms against 5.43). pre + T + S on 1440x720x80
// 6.05 -> 5.43 ms, on 90x40x15 54 -> 32 us; all isoneutral calls of a step on
// 360x160x60, levels innermost, 1120 -> 910 us.
#ifndef VX_STEP_WAVES
#define VX_STEP_WAVES 4
#endif
// columns along j of a strip: 64 and 192 are within 0.2% on 1440x720x80
#ifndef VX_STEP_STRIP_COLS
#define VX_STEP_STRIP_COLS 192
#endif
constexpr int kStepStripCols = VX_STEP_STRIP_COLS;
template <int NTR, bool IMPLICIT, bool WETFLUX>
__global__ __launch_bounds__(kStepThreads) __attribute__((amdgpu_waves_per_eu(VX_STEP_WAVES))) void iso_step_wet_kernel(
    Grid g, Prm p, StepArgs a, int ncb, int sb) {
#pragma clang fp contract(off)
    constexpr int T = kStepThreads;
    // rows A, B, C, shared by the tracers; per tracer flux_top, then the solve's c' -> gamma; lateral
    // dissipation; rhs -> alpha -> new; spike -> beta
    __shared__ double sA[T], sB[T], sC[T], sF[NTR][T], sD[NTR][T], sR[NTR][T], sW[NTR][T];
    __shared__ StepTables tb;
    const BlockCols bc = block_cols(1, g.X - 2, 1, g.Y - 2, ncb, sb);
    if (!bc.valid) return;  // padding block (uniform)
    const int tid = (int)threadIdx.x, nz = g.nz;
    const int i = __builtin_amdgcn_readfirstlane(bc.i), jb = __builtin_amdgcn_readfirstlane(bc.j);
    const int64_t first = ((int64_t)i * g.Y + jb) * nz;
    const double dt = p.dt_tracer;
    for (int q = tid; q < ncb; q += T) {
        const bool real = jb + q <= g.Y - 2;
        const int j = real ? jb + q : g.Y - 2;
        const int kb = g.kbot[i * g.Y + j];
        tb.kb[q + 1] = kb;
        tb.kbw[q] = g.kbot[(i - 1) * g.Y + j];
        tb.off[q + 1] = real && kb >= 1 && kb <= nz ? nz - kb + 1 : 0;
        tb.rxc[q] = 1.0 / (g.dxt[i] * g.cost[j]);
        tb.ryc[q] = 1.0 / (g.dyt[j] * g.cost[j]);
    }
    if (tid == T - 1) {
        tb.kb[0] = g.kbot[i * g.Y + jb - 1];
        tb.rdt = 1.0 / dt;
        tb.g05 = 0.5 * p.grav / p.rho_0;
        tb.gr = -p.grav / p.rho_0;
    }
    for (int k = tid; k < nz; k += T) {
        const double dzw = g.dzw[k];
        tb.dzw[k] = dzw;
        tb.rzw[k] = 1.0 / dzw;
        tb.rzt[k] = 1.0 / g.dzt[k];
    }
    __syncthreads();
    scan_runs(tb.off, ncb);
    __syncthreads();
    const int nwet = tb.off[ncb];
    const bool iin = i >= 2 && i <= g.X - 3;
    const bool energy = a.P != nullptr;

    // the group that starts at column q0: its end (as many whole columns as fit) and this thread's cell
    auto locate = [&](int q0, StepCell& s) {
        const int p0 = tb.off[q0], lane = tid & 63;
        const int q = q0 + 1 + lane;
        const int q1 = q0 + (int)__popcll(__ballot(q <= ncb && tb.off[q <= ncb ? q : ncb] - p0 <= T));
        const int n = tb.off[q1] - p0;
        s.have = tid < n;
        const int t = p0 + (s.have ? tid : n - 1);
        s.q = run_column(tb.off, ncb, t);
        s.kb = tb.kb[s.q + 1];
        s.k = s.kb - 1 + (t - tb.off[s.q]);
        const int j = jb + s.q;
        s.interior = s.have && iin && j >= 2 && j <= g.Y - 3;
        s.e = (uint32_t)(s.q * nz + s.k);
        return q1;
    };
    if (nwet == 0) return;  // uniform
    for (int q0 = 0;;) {
        StepCell s;
        StepIn<NTR> v;
        const int q1 = locate(q0, s);
        // what follows from the thread and the block alone (addresses, the
        // solve's lane numbers) is formed anew for each group: kept over the
        // loop it takes some 40 registers
        int64_t o0 = first;
        int lo = tid;
        asm volatile("" : "+s"(o0), "+v"(lo));
        step_load<NTR, IMPLICIT, WETFLUX>(g, a, tb, o0, s, v);
        __builtin_amdgcn_sched_barrier(0);
        const int k = s.k;
        const int j = jb + s.q;
        step_mask<NTR, WETFLUX>(g, tb, i, j, s, v);
        const double rzt = tb.rzt[k];

        // ---- phase 1a: flux_top and lateral dissipation -> LDS, K33 rows -> LDS
        if (s.have) {
#pragma unroll
            for (int t = 0; t < NTR; ++t) {
                sF[t][lo] = v.ft_c[t];
                if (energy) {
                    // compute_dissipation (veros/core/diffusion.py:13-33)
                    const double de = fma(v.Ie[t] - v.Ic[t], v.fe_c[t], (v.Ic[t] - v.Iw[t]) * v.fe_w[t]);
                    const double dn = fma(v.In[t] - v.Ic[t], v.fn_c[t], (v.Ic[t] - v.Is[t]) * v.fn_s[t]);
                    sD[t][lo] = tb.g05 * fma(de, tb.rxc[s.q], dn * tb.ryc[s.q]);
                }
            }
        }
        if (IMPLICIT && s.interior) {
            // rows of the K33 system (veros/core/isoneutral/diffusion.py:154-164); the
            // edge row k = kbot-1 takes b_edge and a = 0 (veros/core/operators.py:72)
            const bool edge = k == s.kb - 1;
            const double up = (k < nz - 1) ? dt * tb.rzw[k] * v.K33k * rzt : 0.0;
            const double dn = edge ? 0.0 : dt * tb.rzw[k >= 1 ? k - 1 : 0] * v.K33m * rzt;
            sA[lo] = -dn;
            sB[lo] = 1 + (up + dn);
            sC[lo] = -up;
        }
        __syncthreads();

        // ---- phase 1b: divergence and rhs (veros/core/isoneutral/diffusion.py:116-139,196-197)
        double dtr1[NTR], rhs[NTR], dI[NTR];  // dtr plus the explicit tendency
#pragma unroll
        for (int t = 0; t < NTR; ++t) {
            // below the lowest wet cell: with the fused pre's fluxes the top
            // face there is zero (its maskW), else it was read above
            const double ftm = (k >= s.kb) ? sF[t][lo > 0 ? lo - 1 : 0] : (WETFLUX ? 0.0 : v.ft_b[t]);
            const double hor = fma(v.fe_c[t] - v.fe_w[t], tb.rxc[s.q], (v.fn_c[t] - v.fn_s[t]) * tb.ryc[s.q]);
            const double vert = (k == 0 ? v.ft_c[t] : v.ft_c[t] - ftm) * rzt;
            const double dtrk = hor + vert;
            dtr1[t] = v.dtr0[t] + dtrk;
            dI[t] = energy ? v.Ic[t] - v.Iu[t] : 0.0;
            rhs[t] = fma(dt, dtrk, v.trp[t]);
            sR[t][lo] = rhs[t];
        }
        __syncthreads();

        // ---- phase 2: a group of kSegP lanes per (interior column, tracer)
        // solves the column's run in LDS by the segmented elimination
        // (tdma_seg.hpp), segments of S = max(2, ceil(n / kSegP)) rows, rows
        // past the run identity rows
        if (IMPLICIT && iin) {
            const int sg = lo & (kSegP - 1), ncol = q1 - q0, p0 = tb.off[q0];
            for (int task = lo / kSegP; task < ncol * NTR; task += T / kSegP) {
                const int t = NTR == 2 && task >= ncol ? 1 : 0, cq = q0 + task - t * ncol;
                const int cj = jb + cq, b0 = tb.off[cq] - p0, n = tb.off[cq + 1] - tb.off[cq];
                if (cj < 2 || cj > g.Y - 3 || n == 0) continue;  // uniform in the group
                seg_lds_column(sA + b0, sB + b0, sC + b0, &sR[t][b0], &sF[t][b0], &sW[t][b0], n, sg);
            }
        }
        __syncthreads();

        // ---- phase 3
        if (s.have) {
            double Pk = v.P0;
            asm volatile("" : "+s"(o0));
            const double rzw = tb.rzw[k], dzw_lo = tb.dzw[k >= 1 ? k - 1 : 0];  // pad_z_edges(dzw)[k]
#pragma unroll
            for (int t = 0; t < NTR; ++t) {
                const double newk = sR[t][lo], newu = sR[t][lo + 1 < T ? lo + 1 : lo];
                if (s.interior) {
                    (a.t[t].tr + (o0 * g.cs + (int64_t)a.taup1 * g.ls))[g.cs * s.e] = newk;
                    (a.t[t].dtr + o0)[s.e] = fma(newk - rhs[t], tb.rdt, dtr1[t]);
                }
                if (energy) {
                    // dissipation_on_wgrid (veros/core/diffusion.py:39-62)
                    const double d0 = sD[t][lo];
                    const double avg = 0.5 * (d0 + sD[t][lo + 1 < T ? lo + 1 : lo]);
                    const double low = k == s.kb - 1 ? 0.5 * (d0 * dzw_lo * rzw) : 0.0;
                    Pk = Pk + (k == nz - 1 ? d0 : avg + low);
                    // vertical mixing term (veros/core/isoneutral/diffusion.py:254-279)
                    if (s.interior && k < nz - 1) {
                        const double fxa = dI[t] * rzw;
                        const double flux = IMPLICIT ? fma(v.K33k * rzw, newu - newk, v.ft_c[t]) : v.ft_c[t];
                        Pk = fma(tb.gr * fxa, flux, Pk);
                    }
                }
            }
            if (energy) (a.P + o0)[s.e] = Pk;
        }
        if (tb.off[q1] == nwet) break;  // uniform: only dry columns are left
        __syncthreads();  // the group's LDS is no longer read
        q0 = q1;
    }
}

// ---------------------------------------------------------------------------
// Adjoint of one isoneutral tracer step (iso=True, energy branch off) with the
// isoneutral tensor (Ai_*, K_11, K_22, K_33) held fixed:
//   T_new = M^-1 (T[taup1] + dt * D(T[tau], K_iso))   on interior wet cells,
//   T_new = T[taup1] + dt * D                          on interior dry cells,
//   T_new = T[taup1]                                   elsewhere,
// with D the flux divergence (linear in T[tau], and in K_iso through K1 = K2 =
// K_iso). Given mu = dL/dT_new:
//   adj_column : lam = M^-T mu (transposed K33 system, rows re-derived from
//                K_33), g_taup1 = lam, nu = dt * lam on the interior wet cells and
//                0 elsewhere, g_tau = g_K = 0
//   adj_scatter: the adjoints of flux_east / flux_north / flux_top from nu, and
//                each face's contributions to dL/dT[tau] and dL/dK_iso, summed
//                over the levels they reach and added to the columns (atomics)
// ---------------------------------------------------------------------------
struct AdjArgs {
    const double* tr;       // forward input tracer (X, Y, nz, 3), level tau read
    int tau;
    const double* Kiso;
    const double *Aez, *Anz, *Abx, *Aby, *K11, *K22, *K33;
    const double* mu;       // dL/dT_new (X, Y, nz)
    double *g_tau, *g_taup1, *g_K;
    double* nu;             // workspace (X, Y, nz); the caller's holds four such arrays
};

// A wave per tile of 8 columns of the whole grid (col_tile.hpp): one flat pass
// over K_33 and mu. A lane per column with the factors in registers, and an
// initialisation pass before it, took 50 + 8 us on 180x90x40, this 11 us.
constexpr int kAdjP = 8;
constexpr int kAdjBlock = 128;
template <int S>
__global__ __launch_bounds__(kAdjBlock) __attribute__((amdgpu_waves_per_eu(2))) void iso_adj_column_kernel(Grid g, Prm p, AdjArgs a) {
    using T = Tile<S, kAdjP>;
    __shared__ double lds[kAdjBlock / 64][T::IMG];
    __shared__ double rdt[kMaxNz], dtw[kMaxNz];  // 1 / dzt, dt / dzw
    const int nz = g.nz;
    for (int k = threadIdx.x; k < nz; k += kAdjBlock) {
        rdt[k] = 1.0 / g.dzt[k];
        dtw[k] = p.dt_tracer / g.dzw[k];
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    double* const img = lds[wave];
    const int64_t col0 = ((int64_t)blockIdx.x * (kAdjBlock / 64) + wave) * T::C;
    const int64_t left = (int64_t)g.X * g.Y - col0;
    const int n = left >= T::C ? T::C : (left > 0 ? (int)left : 0);
    const T t = make_tile<S, kAdjP>(n > 0 ? col0 * nz : 0, n, nz, (uint32_t)nz, depth_reciprocal(nz));
    SegLane L;
    L.s = t.s;
    L.lo = t.lo;
    L.valid = t.q < n;
    const int64_t col = L.valid ? col0 + t.q : 0;
    const int i = (int)(col / g.Y), j = (int)(col - (int64_t)i * g.Y);
    const bool interior = L.valid && i >= 2 && i <= g.X - 3 && j >= 2 && j <= g.Y - 3;
    const int kb = g.kbot[col];
    L.k0 = interior && kb >= 1 && kb <= nz ? kb - 1 : nz;
    L.base = 0;
    double mu[S], z[S], va[S], vb[S], vc[S];
    {
        double kv[S];
        uint32_t wet[S];
#pragma unroll
        for (int r = 0; r < S; ++r) wet[r] = t.k[r] >= __shfl(L.k0, t.c[r] * kAdjP) ? t.off[r] : kNoAccess;
        tile_load(tile_buf(t, a.K33), wet, 1, kv);
        tile_load(tile_buf(t, a.mu), t.off, 1, mu);
        tile_put(t, img, kv);
    }
    double km[S];
    seg_get(t, img, km);
    const double below = seg_below(t, img);
    tile_put(t, img, mu);
    seg_get(t, img, z);
    // sub'[k] = c[k-1] = -delta[k-1] / dzt[k-1], sup'[k] = a[k+1] = -delta[k] / dzt[k+1]
    double dm = L.lo > L.k0 && L.lo < nz ? dtw[L.lo - 1] * below : 0.0;
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const int k = L.lo + r;
        const bool w = k >= L.k0 && k < nz;
        const int kc = k < nz ? k : nz - 1;
        const double dl = w && k < nz - 1 ? dtw[kc] * km[r] : 0.0;
        va[r] = w && k > L.k0 ? -dm * rdt[kc > 0 ? kc - 1 : 0] : 0.0;
        vb[r] = w ? 1 + (dl + dm) * rdt[kc] : 1.0;
        vc[r] = w && k < nz - 1 ? -dl * rdt[kc < nz - 1 ? kc + 1 : kc] : 0.0;
        z[r] = w ? z[r] : 0.0;
        dm = dl;
    }
    seg_solve_f64<S, 2>(L, va, vb, vc, z);
    seg_put(t, img, z);
    double lam[S], nu[S];
    tile_get(t, img, lam);
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const bool w = t.k[r] >= __shfl(L.k0, t.c[r] * kAdjP);
        nu[r] = w ? p.dt_tracer * lam[r] : 0.0;
        lam[r] = w ? lam[r] : mu[r];
        z[r] = 0.0;
    }
    tile_store(tile_buf(t, a.g_taup1), t.off, 1, lam);
    tile_store(tile_buf(t, a.nu), t.off, 1, nu);
    tile_store(tile_buf(t, a.g_tau), t.off, 1, z);
    tile_store(tile_buf(t, a.g_K), t.off, 1, z);
}

__device__ __forceinline__ void adj_add(double* p, double v) {
    if (v != 0.0) unsafeAtomicAdd(p, v);
}

// Thread per cell (i, j, k), i in [1, X-2), j in [1, Y-2): the three faces whose
// lower cell it is. A face's contributions go to the levels k-1, k and k+1 of the
// cell's own, east, north, west and south columns (and of the first three for
// K_iso); those of the levels next to it pass through LDS to the thread of
// that level, so each thread adds 8 sums instead of up to 35 single terms
// (180x90x40: 43 us and 11 us for a kernel that stored the face adjoints first;
// now 26 us).
__global__ __launch_bounds__(256) void iso_adj_scatter_kernel(Grid g, AdjArgs a) {
    const CellIdx ci = cell_of(1, g.X - 3, 1, g.Y - 3);
    const int nz = g.nz;
    const uint32_t si = (uint32_t)g.Y * (uint32_t)nz, sj = (uint32_t)nz;
    const int i = ci.valid ? ci.i : 1, j = ci.valid ? ci.j : 1, k = ci.k;
    const uint32_t c = (uint32_t)i * si + (uint32_t)j * sj + (uint32_t)k;
    const uint32_t ce = c + si, cn = c + sj;
    const double* __restrict__ tr = a.tr + (uint32_t)a.tau * g.ls;
    const bool hm = k >= 1, hp = k + 1 < nz;
    const uint32_t up = hp ? 1u : 0u, dn = hm ? 1u : 0u;
    const double* K = a.Kiso;
    // columns: 0 own, 1 east, 2 north, 3 west, 4 south; at level k, and passed up and down
    double c0[5] = {}, cu[5] = {}, cd[3] = {}, k0[3] = {}, kd[3] = {};
    if (ci.valid) {
        const double nc = a.nu[c], ne = a.nu[ce], nn = a.nu[cn], nt = hp ? a.nu[c + 1] : 0.0;
        const double cost = g.cost[j];
        const double mue = j >= 2 ? nc / (cost * g.dxt[i]) - ne / (cost * g.dxt[i + 1]) : 0.0;
        const double mun =
            i >= 2 ? (nc / (cost * g.dyt[j]) - nn / (g.cost[j + 1] * g.dyt[j + 1])) * g.cosu[j] : 0.0;
        const double mut = i >= 2 && j >= 2 && hp ? nc / g.dzt[k] - nt / g.dzt[k + 1] : 0.0;
        const double q4 = 1.0 / (4.0 * g.dzt[k]);
        // flux_east and flux_north (veros/core/isoneutral/diffusion.py:22-77)
        auto lateral = [&](int q, double mu, uint32_t cx, const double* A, double k_over_d) {
            if (mu == 0.0) return;
            const double diffloc = hm ? 0.25 * (K[c] + K[c - 1] + K[cx] + K[cx - 1]) : 0.5 * (K[c] + K[cx]);
            const double t0 = tr[g.cs * c], t0u = tr[g.cs * (c + up)], t0d = tr[g.cs * (c - dn)];
            const double t1 = tr[g.cs * cx], t1u = tr[g.cs * (cx + up)], t1d = tr[g.cs * (cx - dn)];
            const double2 A01 = *reinterpret_cast<const double2*>(A + 4u * c);
            const double2 A23 = *reinterpret_cast<const double2*>(A + 4u * c + 2);
            const double m = mu * diffloc * q4, wk = mu * k_over_d;
            const double w00 = m * A01.x, w01 = m * A01.y, w10 = m * A23.x, w11 = m * A23.y;
            c0[0] += w00 - w01 - wk;
            c0[q] += w10 - w11 + wk;
            // the clamped ends keep their terms
            c0[0] += (hp ? 0.0 : w01) - (hm ? 0.0 : w00);
            c0[q] += (hp ? 0.0 : w11) - (hm ? 0.0 : w10);
            cu[0] += hp ? w01 : 0.0;
            cu[q] += hp ? w11 : 0.0;
            cd[0] -= hm ? w00 : 0.0;
            cd[q] -= hm ? w10 : 0.0;
            const double S = (A01.x * (t0 - t0d) + A23.x * (t1 - t1d) + A01.y * (t0u - t0) + A23.y * (t1u - t1)) * q4;
            const double wK = mu * S * (hm ? 0.25 : 0.5);
            k0[0] += wK;
            k0[q] += wK;
            kd[0] += hm ? wK : 0.0;
            kd[q] += hm ? wK : 0.0;
        };
        lateral(1, mue, ce, a.Aez, a.K11[c] / (cost * g.dxu[i]));
        lateral(2, mun, cn, a.Anz, a.K22[c] / g.dyu[j]);
        if (mut != 0.0) {  // flux_top (:79-111)
            const double m = mut * K[c];
            const double* B = a.Abx + 4u * c;
            const double* C = a.Aby + 4u * c;
            const uint32_t cw = c - si, cs = c - sj;
            const double fx = 1.0 / (4 * g.dxt[i]) / cost;
            const double fy = 1.0 / (4 * g.dyt[j] * cost);
            double S = 0.0;
#pragma unroll
            for (int kr = 0; kr < 2; ++kr) {
                // x: (ip=0) tr[i] - tr[i-1], (ip=1) tr[i+1] - tr[i], at level k + kr
                const double bx0 = B[kr] * fx, bx1 = B[2 + kr] * fx;
                const double cy0 = C[kr] * g.cosu[j - 1] * fy, cy1 = C[2 + kr] * g.cosu[j] * fy;
                const double t = tr[g.cs * (c + kr)];
                S += bx0 * (t - tr[g.cs * (cw + kr)]) + bx1 * (tr[g.cs * (ce + kr)] - t) +
                     cy0 * (t - tr[g.cs * (cs + kr)]) + cy1 * (tr[g.cs * (cn + kr)] - t);
                double(&o)[5] = kr ? cu : c0;
                o[0] += m * (bx0 - bx1 + cy0 - cy1);
                o[1] += m * bx1;
                o[2] += m * cy1;
                o[3] -= m * bx0;
                o[4] -= m * cy0;
            }
            k0[0] += mut * S;
        }
    }
    // sums over the levels: from the thread below (its k + 1) and above (its k - 1)
    __shared__ double lu[5][256], ld[6][256];
    const int tid = (int)(threadIdx.y * blockDim.x + threadIdx.x);
#pragma unroll
    for (int q = 0; q < 5; ++q) lu[q][tid] = cu[q];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        ld[q][tid] = cd[q];
        ld[3 + q][tid] = kd[q];
    }
    __syncthreads();
    if (!ci.valid) return;
    if (hm) {
#pragma unroll
        for (int q = 0; q < 5; ++q) c0[q] += lu[q][tid - 1];
    }
    if (hp) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            c0[q] += ld[q][tid + 1];
            k0[q] += ld[3 + q][tid + 1];
        }
    }
    adj_add(a.g_tau + c, c0[0]);
    adj_add(a.g_tau + ce, c0[1]);
    adj_add(a.g_tau + cn, c0[2]);
    adj_add(a.g_tau + (c - si), c0[3]);
    adj_add(a.g_tau + (c - sj), c0[4]);
    adj_add(a.g_K + c, k0[0]);
    adj_add(a.g_K + ce, k0[1]);
    adj_add(a.g_K + cn, k0[2]);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

int make_grid(const vx_grid* in, Grid& g, const char* who) {
    if (!in) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid", who);
    if (in->nx < 1 || in->ny < 1 || in->nz < 2)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: need nx, ny >= 1 and nz >= 2 (got %lld, %lld, %d)", who,
                    (long long)in->nx, (long long)in->ny, in->nz);
    if (in->nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d exceeds %d", who, in->nz, kMaxNz);
    if (in->nx + 4 > INT32_MAX / 8 || in->ny + 4 > INT32_MAX / 8)
        return fail(VX_ERR_UNSUPPORTED, "%s: horizontal size too large", who);
    if (!in->kbot || !in->dxt || !in->dxu || !in->dyt || !in->dyu || !in->cost || !in->cosu || !in->dzt || !in->dzw)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null grid array", who);
    g.kbot = in->kbot;
    g.dxt = in->dxt;
    g.dxu = in->dxu;
    g.dyt = in->dyt;
    g.dyu = in->dyu;
    g.cost = in->cost;
    g.cosu = in->cosu;
    g.dzt = in->dzt;
    g.dzw = in->dzw;
    g.X = (int32_t)(in->nx + 4);
    g.Y = (int32_t)(in->ny + 4);
    if (in->time_layout != VX_LEVELS_INNER && in->time_layout != VX_LEVELS_OUTER)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: time_layout must be VX_LEVELS_INNER or VX_LEVELS_OUTER (got %d)",
                    who, in->time_layout);
    if ((in->nx + 4) * (in->ny + 4) * (int64_t)in->nz * 3 >= ((int64_t)1 << 32))
        return fail(VX_ERR_UNSUPPORTED, "%s: grid too large for 32-bit offsets", who);
    const bool outer = in->time_layout == VX_LEVELS_OUTER;
    g.cs = outer ? 1u : 3u;
    g.ls = outer ? (uint32_t)((in->nx + 4) * (in->ny + 4) * (int64_t)in->nz) : 1u;
    g.nz = in->nz;
    return VX_OK;
}

Prm make_prm(const vx_iso_params* q) {
    Prm p;
    p.drhodT = q->drhodT;
    p.drhodS = q->drhodS;
    p.K_iso_steep = q->K_iso_steep;
    p.iso_slopec = q->iso_slopec;
    p.iso_dslope = q->iso_dslope;
    p.dt_tracer = q->dt_tracer;
    p.grav = q->grav;
    p.rho_0 = q->rho_0;
    return p;
}

#ifndef VX_PRE_CELLS
#define VX_PRE_CELLS 640
#endif
// Columns per block (one wave) of the pre and flux kernels: about VX_PRE_CELLS
// cells (8 columns at nz = 80), so that a wave deals several rounds of cells
// and the partly filled last one wastes few lanes, but at least eight waves per CU
// on small grids, as many as pre's registers allow at once (pre + T + S on
// 180x90x40, levels innermost: 90 us with four, 77 with eight, 80 with 16). The
// fused call on 1440x720x80 and the calls on 360x160x60 (levels innermost): 640
// cells 6.04 ms and 1162 us, 1280 5.98 and 1204, 2400 6.38 and 1262.
int cell_columns(const Grid& g) {
    const int64_t spread = ((int64_t)(g.X - 3) * (g.Y - 3) + 8 * cu_count() - 1) / (8 * cu_count());
    const int n = (int)std::min<int64_t>((VX_PRE_CELLS + g.nz - 1) / g.nz, spread);
    return n < 4 ? 4 : (n > kBlockCols ? kBlockCols : n);
}
// blocks of ncb columns over the cells' range, for block_cols
dim3 cell_column_grid(const Grid& g, int ncb) {
    const int sb = strip_blocks(kPreStripCols, ncb, g.Y - 3);
    const int64_t nstrips = (g.Y - 3 + (int64_t)sb * ncb - 1) / (sb * ncb);
    return dim3((unsigned)((nstrips * (g.X - 3) * sb + 7) / 8 * 8));
}

unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// block of nz levels x cpb columns (about 256 threads); 1-D grid of ni row
// groups, rounded up to a multiple of 8 for the XCD remap
dim3 cell_block(int nz) { return dim3(nz, nz >= 256 ? 1 : 256 / nz); }
dim3 cell_grid(int ni, int nj, dim3 blk) {
    const int sb = kStripBlocks;
    const int64_t sw = (int64_t)sb * blk.y;
    const int64_t nstrips = (nj + sw - 1) / sw;
    return dim3((unsigned)((nstrips * ni * sb + 7) / 8 * 8));
}

#ifndef VX_STEP_COLS
#define VX_STEP_COLS 32
#endif
// Columns per block: a group is about six wet columns at nz = 80, and the last
// group of a block is partly empty, so the more columns the fewer idle lanes; but
// at least eight blocks per CU on small grids, the four that run at once and
// four to follow (pre + T + S on 180x90x40, levels innermost: 77 us with four, 73 with
// eight, 75 with 12). 1440x720x80 pre + T + S and the
// calls on 360x160x60: 16 columns 5.00 ms and 958 us, 32 4.89 and 963, 64 4.85
// and 1006 (one placement of the arrays; 48 0.8% faster and 1.7% slower than 32).
template <int NTR, bool IMPLICIT, bool WETFLUX>
int launch_wet_step(const Grid& g, const Prm& p, const StepArgs& a, hipStream_t s, const char* who) {
    const int64_t spread = ((int64_t)(g.X - 2) * (g.Y - 2) + 8 * cu_count() - 1) / (8 * cu_count());
    int ncb = (int)std::min<int64_t>(VX_STEP_COLS, spread);
    ncb = ncb < 4 ? 4 : ncb;
    const int sb = strip_blocks(kStepStripCols + ncb - 1, ncb, g.Y - 2);
    const int64_t nstrips = (g.Y - 2 + (int64_t)sb * ncb - 1) / (sb * ncb);
    const unsigned nblk = (unsigned)((nstrips * (g.X - 2) * sb + 7) / 8 * 8);
    hipLaunchKernelGGL((iso_step_wet_kernel<NTR, IMPLICIT, WETFLUX>), dim3(nblk), dim3(kStepThreads), 0, s, g, p, a,
                       ncb, sb);
    return check_launch(who);
}

template <int NTR, bool IMPLICIT>
int launch_step(const Grid& g, const Prm& p, const StepArgs& a, hipStream_t s, const char* who) {
    if ((int64_t)g.X * g.Y * g.nz * 4 >= ((int64_t)1 << 32))
        return fail(VX_ERR_UNSUPPORTED, "%s: grid too large for 32-bit offsets", who);
    if (g.nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d too deep", who, g.nz);
    const int ncb = cell_columns(g);
    hipLaunchKernelGGL((iso_flux_kernel<NTR, IMPLICIT>), cell_column_grid(g, ncb), dim3(kCellBlock), 0, s, g, a,
                       ncb);
    const int rc = check_launch(who);
    return rc ? rc : launch_wet_step<NTR, IMPLICIT, false>(g, p, a, s, who);
}

int check_common(const vx_grid* grid, const vx_iso_params* prm, int32_t tau, int32_t taup1, Grid& g,
                 const char* who) {
    int rc = make_grid(grid, g, who);
    if (rc) return rc;
    if (!prm) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null params", who);
    if (tau < 0 || tau > 2 || taup1 < 0 || taup1 > 2)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: time levels must be 0..2", who);
    return VX_OK;
}

bool tensor_ok(const double* Ai_ez, const double* Ai_nz, const double* Ai_bx, const double* Ai_by,
               const double* K_11, const double* K_22) {
    return Ai_ez && Ai_nz && Ai_bx && Ai_by && K_11 && K_22;
}

// isoneutral_diffusion_pre; FUSED also writes the step's face fluxes into `fo`.
template <bool FUSED>
int launch_pre(const Grid& g, const Prm& p, const Fields& f, const double* K_iso, double* Ai_ez, double* Ai_nz,
               double* Ai_bx, double* Ai_by, double* K_11, double* K_22, double* K_33, PreFlux fo, hipStream_t s,
               const char* who) {
    const int ncb = cell_columns(g);
    hipLaunchKernelGGL(iso_pre_kernel<FUSED>, cell_column_grid(g, ncb), dim3(kCellBlock), 0, s, g, p, f, K_iso, Ai_ez,
                       Ai_nz, Ai_bx, Ai_by, K_11, K_22, K_33, fo, ncb);
    return check_launch(who);
}

void wire_workspace(const Grid& g, StepArgs& a, int ntr, void* ws) {
    const int64_t n3 = (int64_t)g.X * g.Y * g.nz;
    double* w = static_cast<double*>(ws);
    a.fe = w;
    a.fn = w + ntr * n3;
    a.ft = w + 2 * ntr * n3;
}
}  // namespace
}  // namespace vx

extern "C" int vx_iso_diffusion_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm, double* tracer,
                                    int32_t tau, int32_t taup1, const double* K_iso, const double* Ai_ez,
                                    const double* Ai_nz, const double* Ai_bx, const double* Ai_by,
                                    const double* K_11, const double* K_22, const double* K_33, double* dtr_iso,
                                    const double* int_drhodX, double* P_diss, void* workspace) {
    using namespace vx;
    const char* who = "vx_iso_diffusion_f64";
    Grid g;
    int rc = check_common(grid, prm, tau, taup1, g, who);
    if (rc) return rc;
    if (!tracer || !K_iso || !tensor_ok(Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22) || !K_33 || !dtr_iso)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((P_diss == nullptr) != (int_drhodX == nullptr))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: P_diss and int_drhodX must both be given or both be NULL", who);
    StepArgs a{};
    if (!workspace) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null workspace", who);
    a.t[0] = {tracer, dtr_iso, int_drhodX};
    wire_workspace(g, a, 1, workspace);
    a.tau = tau;
    a.taup1 = taup1;
    a.Kiso = K_iso;
    a.Kskew = nullptr;
    a.Aez = Ai_ez, a.Anz = Ai_nz, a.Abx = Ai_bx, a.Aby = Ai_by, a.K11 = K_11, a.K22 = K_22, a.K33 = K_33;
    a.P = P_diss;
    return launch_step<1, true>(g, make_prm(prm), a, (hipStream_t)stream, who);
}

extern "C" int vx_iso_diffusion_ts_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm, double* temp,
                                       double* salt, int32_t tau, int32_t taup1, const double* K_iso,
                                       const double* Ai_ez, const double* Ai_nz, const double* Ai_bx,
                                       const double* Ai_by, const double* K_11, const double* K_22,
                                       const double* K_33, double* dtemp_iso, double* dsalt_iso,
                                       const double* int_drhodT, const double* int_drhodS, double* P_diss,
                                       void* workspace) {
    using namespace vx;
    const char* who = "vx_iso_diffusion_ts_f64";
    Grid g;
    int rc = check_common(grid, prm, tau, taup1, g, who);
    if (rc) return rc;
    if (!temp || !salt || !K_iso || !tensor_ok(Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22) || !K_33 || !dtemp_iso ||
        !dsalt_iso)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if (temp == salt) return fail(VX_ERR_INVALID_ARGUMENT, "%s: temp and salt must be distinct arrays", who);
    const bool e = P_diss != nullptr;
    if (e != (int_drhodT != nullptr) || e != (int_drhodS != nullptr))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: P_diss, int_drhodT and int_drhodS must all be given or all be NULL",
                    who);
    StepArgs a{};
    if (!workspace) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null workspace", who);
    a.t[0] = {temp, dtemp_iso, int_drhodT};
    a.t[1] = {salt, dsalt_iso, int_drhodS};
    wire_workspace(g, a, 2, workspace);
    a.tau = tau;
    a.taup1 = taup1;
    a.Kiso = K_iso;
    a.Kskew = nullptr;
    a.Aez = Ai_ez, a.Anz = Ai_nz, a.Abx = Ai_bx, a.Aby = Ai_by, a.K11 = K_11, a.K22 = K_22, a.K33 = K_33;
    a.P = P_diss;
    return launch_step<2, true>(g, make_prm(prm), a, (hipStream_t)stream, who);
}

extern "C" int vx_iso_skew_diffusion_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm,
                                         double* tracer, int32_t tau, int32_t taup1, const double* K_gm,
                                         const double* Ai_ez, const double* Ai_nz, const double* Ai_bx,
                                         const double* Ai_by, const double* K_11, const double* K_22,
                                         double* dtr_iso, const double* int_drhodX, double* P_diss_skew,
                                         void* workspace) {
    using namespace vx;
    const char* who = "vx_iso_skew_diffusion_f64";
    Grid g;
    int rc = check_common(grid, prm, tau, taup1, g, who);
    if (rc) return rc;
    if (!tracer || !K_gm || !tensor_ok(Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22) || !dtr_iso)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((P_diss_skew == nullptr) != (int_drhodX == nullptr))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: P_diss_skew and int_drhodX must both be given or both be NULL", who);
    StepArgs a{};
    if (!workspace) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null workspace", who);
    a.t[0] = {tracer, dtr_iso, int_drhodX};
    wire_workspace(g, a, 1, workspace);
    a.tau = tau;
    a.taup1 = taup1;
    a.Kiso = nullptr;
    a.Kskew = K_gm;
    a.Aez = Ai_ez, a.Anz = Ai_nz, a.Abx = Ai_bx, a.Aby = Ai_by, a.K11 = K_11, a.K22 = K_22, a.K33 = nullptr;
    a.P = P_diss_skew;
    return launch_step<1, false>(g, make_prm(prm), a, (hipStream_t)stream, who);
}

extern "C" int64_t vx_iso_workspace_bytes(const vx_grid* grid, int32_t ntracers) {
    if (!grid || ntracers < 1 || ntracers > 2 || grid->nx < 1 || grid->ny < 1 || grid->nz < 1) return -1;
    // the face fluxes, and per column and 2048 columns the room of the index
    // tables that callers' buffers have always held
    const int64_t X = grid->nx + 4, Y = grid->ny + 4, cols = (Y - 2 + 63) / 64 * (X - 2) * 64;
    const int64_t ints = 3 * cols + 2 + 12;
    return 3 * (int64_t)ntracers * X * Y * (int64_t)grid->nz * (int64_t)sizeof(double) +
           (ints * (int64_t)sizeof(int) + 7) / 8 * 8 + (cols + 2047) / 2048 * 8;
}

extern "C" int64_t vx_iso_pre_diffusion_ts_workspace_bytes(const vx_grid* grid) {
    return vx_iso_workspace_bytes(grid, 2);
}

extern "C" int64_t vx_iso_adjoint_workspace_bytes(const vx_grid* grid) {
    if (!grid) return -1;
    return 4 * (grid->nx + 4) * (grid->ny + 4) * (int64_t)grid->nz * (int64_t)sizeof(double);
}

extern "C" int vx_iso_diffusion_adjoint_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm,
                                            const double* tracer, int32_t tau, const double* K_iso,
                                            const double* Ai_ez, const double* Ai_nz, const double* Ai_bx,
                                            const double* Ai_by, const double* K_11, const double* K_22,
                                            const double* K_33, const double* g_new, double* g_tau,
                                            double* g_taup1, double* g_K_iso, void* workspace) {
    using namespace vx;
    const char* who = "vx_iso_diffusion_adjoint_f64";
    Grid g;
    int rc = check_common(grid, prm, tau, 0, g, who);
    if (rc) return rc;
    if (!tracer || !K_iso || !tensor_ok(Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22) || !K_33 || !g_new || !g_tau ||
        !g_taup1 || !g_K_iso || !workspace)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if ((int64_t)g.X * g.Y * g.nz * 4 >= ((int64_t)1 << 32))
        return fail(VX_ERR_UNSUPPORTED, "%s: grid too large for 32-bit offsets", who);
    AdjArgs a{tracer, tau, K_iso, Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22, K_33, g_new, g_tau, g_taup1, g_K_iso,
              static_cast<double*>(workspace)};
    hipStream_t s = (hipStream_t)stream;
    const Prm p = make_prm(prm);
    const int64_t ntiles = ((int64_t)g.X * g.Y + 64 / kAdjP - 1) / (64 / kAdjP);
    const dim3 cgrid(blocks_for(ntiles * 64, kAdjBlock)), cblk(kAdjBlock);
#define VX_ADJ_CASE(N) \
    case N: hipLaunchKernelGGL(iso_adj_column_kernel<N>, cgrid, cblk, 0, s, g, p, a); break;
    switch (seg_levels(g.nz)) {
        VX_ADJ_CASE(2)
        VX_ADJ_CASE(4)
        VX_ADJ_CASE(6)
        VX_ADJ_CASE(8)
        VX_ADJ_CASE(10)
        VX_ADJ_CASE(12)
        VX_ADJ_CASE(14)
        VX_ADJ_CASE(16)
        default: return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d", who, g.nz);
    }
#undef VX_ADJ_CASE
    if ((rc = check_launch(who))) return rc;
    const dim3 blk = cell_block(g.nz);
    hipLaunchKernelGGL(iso_adj_scatter_kernel, cell_grid(g.X - 3, g.Y - 3, blk), blk, 0, s, g, a);
    return check_launch(who);
}

namespace vx {
namespace {

// The one call (pre, then the temperature and salinity steps) with the given
// workspace.
int pre_diffusion_ts(hipStream_t s, const vx_grid* grid, const vx_iso_params* prm, double* temp, double* salt,
                     int32_t tau, int32_t taup1, const double* K_iso, double* Ai_ez, double* Ai_nz, double* Ai_bx,
                     double* Ai_by, double* K_11, double* K_22, double* K_33, double* dtemp_iso, double* dsalt_iso,
                     const double* int_drhodT, const double* int_drhodS, double* P_diss, void* workspace,
                     const char* who) {
    Grid g;
    int rc = check_common(grid, prm, tau, taup1, g, who);
    if (rc) return rc;
    if (!temp || !salt || !K_iso || !tensor_ok(Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22) || !K_33 || !dtemp_iso ||
        !dsalt_iso)
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: null array pointer", who);
    if (temp == salt) return fail(VX_ERR_INVALID_ARGUMENT, "%s: temp and salt must be distinct arrays", who);
    const bool e = P_diss != nullptr;
    if (e != (int_drhodT != nullptr) || e != (int_drhodS != nullptr))
        return fail(VX_ERR_INVALID_ARGUMENT, "%s: P_diss, int_drhodT and int_drhodS must all be given or all be NULL",
                    who);
    if (!workspace) return fail(VX_ERR_INVALID_ARGUMENT, "%s: null workspace", who);
    if ((int64_t)g.X * g.Y * g.nz * 4 >= ((int64_t)1 << 32))
        return fail(VX_ERR_UNSUPPORTED, "%s: grid too large for 32-bit offsets", who);
    if (g.nz > kMaxNz) return fail(VX_ERR_UNSUPPORTED, "%s: nz=%d too deep", who, g.nz);
    StepArgs a{};
    a.t[0] = {temp, dtemp_iso, int_drhodT};
    a.t[1] = {salt, dsalt_iso, int_drhodS};
    wire_workspace(g, a, 2, workspace);
    a.tau = tau;
    a.taup1 = taup1;
    a.Kiso = K_iso;
    a.Kskew = nullptr;
    a.Aez = Ai_ez, a.Anz = Ai_nz, a.Abx = Ai_bx, a.Aby = Ai_by, a.K11 = K_11, a.K22 = K_22, a.K33 = K_33;
    a.P = P_diss;
    const Prm p = make_prm(prm);
    const PreFlux fo{a.fe, a.fn, a.ft};
    rc = launch_pre<true>(g, p, Fields{temp, salt, tau}, K_iso, Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22, K_33, fo, s,
                          who);
    return rc ? rc : launch_wet_step<2, true, true>(g, p, a, s, who);
}

}  // namespace
}  // namespace vx

extern "C" int vx_iso_pre_diffusion_ts_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm, double* temp,
                                           double* salt, int32_t tau, int32_t taup1, const double* K_iso,
                                           double* Ai_ez, double* Ai_nz, double* Ai_bx, double* Ai_by, double* K_11,
                                           double* K_22, double* K_33, double* dtemp_iso, double* dsalt_iso,
                                           const double* int_drhodT, const double* int_drhodS, double* P_diss,
                                           void* workspace) {
    return vx::pre_diffusion_ts((hipStream_t)stream, grid, prm, temp, salt, tau, taup1, K_iso, Ai_ez, Ai_nz, Ai_bx,
                                Ai_by, K_11, K_22, K_33, dtemp_iso, dsalt_iso, int_drhodT, int_drhodS, P_diss,
                                workspace, "vx_iso_pre_diffusion_ts_f64");
}

// ---------------------------------------------------------------------------
// The one call without a caller workspace: the face fluxes live in `scratch`,
// a device array of the library (one per GPU, held until the process ends). Its device address is taken once per device with
// hipGetSymbolAddress; host code never passes the array's own name to a
// kernel. The entry point allocates nothing: no hipMalloc, no helper stream.
// ---------------------------------------------------------------------------
namespace {
constexpr int64_t kNoAllocScratchBytes = int64_t(192) << 20;  // 192 MiB
}
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace vx {
namespace {
// Device address of `scratch` on the current device, looked up on the first
// call on that device (null and an error message if the lookup fails).
void* scratch_on_current_device(const char* who) {
    static std::mutex m;
    static std::map<int, void*> per_device;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        fail(VX_ERR_LAUNCH, "%s: hipGetDevice failed", who);
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(m);
    auto it = per_device.find(dev);
    if (it != per_device.end()) return it->second;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
        fail(VX_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) failed: %s", who, hipGetErrorString(e));
        return nullptr;
    }
    per_device[dev] = ptr;
    return ptr;
}
}  // namespace
}  // namespace vx

extern "C" int vx_iso_pre_diffusion_ts_f64_noalloc(void* stream, const vx_grid* grid, const vx_iso_params* prm,
                                                   double* temp, double* salt, int32_t tau, int32_t taup1,
                                                   const double* K_iso, double* Ai_ez, double* Ai_nz, double* Ai_bx,
                                                   double* Ai_by, double* K_11, double* K_22, double* K_33,
                                                   double* dtemp_iso, double* dsalt_iso, const double* int_drhodT,
                                                   const double* int_drhodS, double* P_diss) {
    using namespace vx;
    const char* who = "vx_iso_pre_diffusion_ts_f64_noalloc";
    const int64_t need = vx_iso_pre_diffusion_ts_workspace_bytes(grid);
    if (need < 0) return fail(VX_ERR_INVALID_ARGUMENT, "%s: invalid grid", who);
    if (need > kNoAllocScratchBytes)
        return fail(VX_ERR_UNSUPPORTED,
                    "%s: the grid needs %lld bytes of scratch, above the library's fixed %lld (use "
                    "vx_iso_pre_diffusion_ts_f64 with a workspace)",
                    who, (long long)need, (long long)kNoAllocScratchBytes);
    void* ws = scratch_on_current_device(who);
    if (!ws) return VX_ERR_LAUNCH;
    return pre_diffusion_ts((hipStream_t)stream, grid, prm, temp, salt, tau, taup1, K_iso, Ai_ez, Ai_nz, Ai_bx,
                            Ai_by, K_11, K_22, K_33, dtemp_iso, dsalt_iso, int_drhodT, int_drhodS, P_diss, ws, who);
}

extern "C" int vx_iso_pre_f64(void* stream, const vx_grid* grid, const vx_iso_params* prm, const double* temp,
                              const double* salt, int32_t tau, const double* K_iso, double* Ai_ez, double* Ai_nz,
                              double* Ai_bx, double* Ai_by, double* K_11, double* K_22, double* K_33) {
    using namespace vx;
    Grid g;
    int rc = make_grid(grid, g, "vx_iso_pre_f64");
    if (rc) return rc;
    if (!prm) return fail(VX_ERR_INVALID_ARGUMENT, "vx_iso_pre_f64: null params");
    if (tau < 0 || tau > 2) return fail(VX_ERR_INVALID_ARGUMENT, "vx_iso_pre_f64: tau must be 0..2");
    if (!temp || !salt || !K_iso || !Ai_ez || !Ai_nz || !Ai_bx || !Ai_by || !K_11 || !K_22 || !K_33)
        return fail(VX_ERR_INVALID_ARGUMENT, "vx_iso_pre_f64: null array pointer");
    hipStream_t s = (hipStream_t)stream;
    Fields f{temp, salt, tau};
    const Prm p = make_prm(prm);
    if ((int64_t)g.X * g.Y * g.nz * 4 >= ((int64_t)1 << 32))
        return fail(VX_ERR_UNSUPPORTED, "vx_iso_pre_f64: grid too large for 32-bit offsets");
    return launch_pre<false>(g, p, f, K_iso, Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22, K_33, PreFlux{}, s,
                             "vx_iso_pre_f64");
}
