// Column tiles: a wave owns C = 64 / P consecutive (i, j) columns of an
// (X, Y, nz) grid (with sy = nz one contiguous run of C * nz cells) and sees
// them in two layouts.
//
//   flat:     element t of lane l is cell 64 t + l of the run. Every global
//             access is made here: consecutive lanes touch consecutive cells
//             whatever nz's parity, the arrays' alignment or the storage of the
//             time levels (levels innermost: every third double). Loads and
//             stores are raw buffer accesses whose descriptor spans the run; a
//             lane that must not take part gets an offset past its end, which
//             the hardware turns into 0 (a dropped store) without traffic and
//             without a branch, so all loads of a phase are in flight together.
//   segments: lane s of a column's P lanes holds levels [s S, s S + S),
//             the layout of the segmented tridiagonal solve.
//
// Values pass between the layouts through an LDS image of the run (odd
// segment stride, so that the segments' starts spread over the banks).
// Everything elementwise (forcing sums, right-hand sides, diagnostics, lateral
// fluxes) is done flat, only the rows' neighbours and the solve need
// segments. P = 16 where many arrays are in flight (a lane holds nz/16 values of
// each, which leaves registers for more waves), P = 8 where the solve itself is
// most of the work (half the interface rows per column).
#pragma once
#include "tdma_seg.hpp"

namespace vx {

constexpr int kTileP = 16;  // lanes per column, unless a kernel says otherwise: one DPP row

// levels per lane for a depth nz (>= 2)
__host__ __device__ constexpr int tile_levels(int nz) {
    const int s = (nz + kTileP - 1) / kTileP;
    return s < 2 ? 2 : s;
}

// An offset past the end of every buffer, also when scaled by 3.
constexpr uint32_t kNoAccess = 0x20000000u;

typedef __amdgpu_buffer_rsrc_t BufRsrc;
// A buffer of `bytes` bytes at the wave-uniform address p; accesses past its
// end read 0 or are dropped.
__device__ __forceinline__ BufRsrc make_buf(const double* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, bytes, 0x00027000);
}
typedef unsigned int vx_u2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double buf_load(BufRsrc b, uint32_t off) {
    const vx_u2 v = __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0);
    return __builtin_bit_cast(double, v);
}
__device__ __forceinline__ void buf_store(BufRsrc b, uint32_t off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(vx_u2, v), b, off, 0, 0);
}

template <int S, int P = kTileP>
struct Tile {
    static constexpr int C = 64 / P;              // columns
    static constexpr int SP = S | 1;              // segment stride in an image
    static constexpr int CS = P * SP;             // column stride
    static constexpr int DUMMY = C * CS;          // slot of the lanes past the run
    static constexpr int IMG = C * CS + 2;        // doubles of an image
    int lane, s, q;       // lane of the wave; segment and column (segments)
    int lo;               // first level of the segment
    int seg;              // the segment's position in an image
    int k[S], c[S];       // level and column of the flat elements
    int pos[S];           // their positions in an image
    uint32_t off[S];      // their byte offsets in an (X, Y, nz) array's run
    uint32_t bytes;       // bytes of that run
    int64_t cell0;        // first cell of the run
    int ncol;             // columns of the run (< C in a row's or the grid's last tile)
};

// The tile of `ncol` columns of nz levels, `sy` cells apart, from cell0 on
// (ncol = 0: no columns; the addresses formed are those of cell0). All
// arguments wave-uniform; C * sy * 8 < kNoAccess. m: depth_reciprocal(nz), with
// which e / nz is (e * m) >> 20, exactly for e <= 1024, nz <= 128.
__host__ __device__ __forceinline__ uint32_t depth_reciprocal(int nz) {
    return ((1u << 20) + (uint32_t)nz - 1u) / (uint32_t)nz;
}
// Flat element e of such a tile.
struct FlatCell {
    int k, c, pos;
    uint32_t off;  // kNoAccess past the run; c is 0 there
};
template <int S, int P>
__host__ __device__ __forceinline__ FlatCell flat_cell(uint32_t e, int ncol, int nz, uint32_t sy, uint32_t m) {
    using T = Tile<S, P>;
    const uint32_t c = (e * m) >> 20, k = e - c * (uint32_t)nz;
    const bool in = (int)c < ncol;
    FlatCell f;
    f.k = (int)k;
    f.c = in ? (int)c : 0;
    f.pos = (int)c < T::C ? (int)(c * T::CS + k + k / S * (T::SP - S)) : T::DUMMY;
    f.off = in ? (c * sy + k) * 8u : kNoAccess;
    return f;
}
template <int S, int P = kTileP>
__device__ __forceinline__ Tile<S, P> make_tile(int64_t cell0, int ncol, int nz, uint32_t sy, uint32_t m) {
    using T = Tile<S, P>;
    T t;
    t.lane = (int)(threadIdx.x & 63);
    t.s = t.lane % P;
    t.q = t.lane / P;
    t.lo = t.s * S;
    t.seg = t.q * T::CS + t.s * T::SP;
    t.cell0 = cell0;
    t.ncol = ncol;
    t.bytes = ncol > 0 ? ((uint32_t)(ncol - 1) * sy + (uint32_t)nz) * 8u : 0u;
#pragma unroll
    for (int r = 0; r < S; ++r) {
        const FlatCell f = flat_cell<S, P>(64u * r + (uint32_t)t.lane, ncol, nz, sy, m);
        t.k[r] = f.k;
        t.c[r] = f.c;
        t.pos[r] = f.pos;
        t.off[r] = f.off;
    }
    return t;
}
// Image positions of the levels below and above a flat element in its column;
// the element's own where the column has no level from k0 on there, and for an
// element past the run, whose slot may be the image's last.
template <int S, int P>
__host__ __device__ __forceinline__ void flat_neighbours(const FlatCell& f, int k0, int nz, int& below, int& above) {
    constexpr int step = Tile<S, P>::SP - S;  // more between two segments
    const bool on = f.off != kNoAccess && f.k >= k0;
    below = on && f.k > k0 ? f.pos - 1 - (f.k % S == 0 ? step : 0) : f.pos;
    above = on && f.k < nz - 1 ? f.pos + 1 + (f.k % S == S - 1 ? step : 0) : f.pos;
}

// The run of a (X, Y, nz) array, `d` cells further on, cs doubles per cell.
template <int S, int P>
__device__ __forceinline__ BufRsrc tile_buf(const Tile<S, P>& t, const double* a, int64_t d = 0, int cs = 1) {
    return make_buf(a + (t.cell0 + d) * cs, t.bytes * (uint32_t)cs);
}

// flat elements where on[r] (0 elsewhere)
template <int S>
__device__ __forceinline__ void tile_load(BufRsrc b, const uint32_t (&off)[S], uint32_t cs, double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) v[r] = buf_load(b, off[r] * cs);
}
template <int S>
__device__ __forceinline__ void tile_store(BufRsrc b, const uint32_t (&off)[S], uint32_t cs, const double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) buf_store(b, off[r] * cs, v[r]);
}
// flat <-> image
template <int S, int P>
__device__ __forceinline__ void tile_put(const Tile<S, P>& t, double* img, const double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) img[t.pos[r]] = v[r];
}
template <int S, int P>
__device__ __forceinline__ void tile_get(const Tile<S, P>& t, const double* img, double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) v[r] = img[t.pos[r]];
}
// segments <-> image
template <int S, int P>
__device__ __forceinline__ void seg_get(const Tile<S, P>& t, const double* img, double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) v[r] = img[t.seg + r];
}
template <int S, int P>
__device__ __forceinline__ void seg_put(const Tile<S, P>& t, double* img, const double (&v)[S]) {
#pragma unroll
    for (int r = 0; r < S; ++r) img[t.seg + r] = v[r];
}
// the value of the level below lo (lane s = 0: unspecified) and above lo + S - 1
// (lane s = P - 1: unspecified) in an image
template <int S, int P>
__device__ __forceinline__ double seg_below(const Tile<S, P>& t, const double* img) {
    return img[t.s > 0 ? t.seg - 1 - (Tile<S, P>::SP - S) : t.seg];
}
template <int S, int P>
__device__ __forceinline__ double seg_above(const Tile<S, P>& t, const double* img) {
    return img[t.s < P - 1 ? t.seg + Tile<S, P>::SP : t.seg];
}

// ---------------------------------------------------------------------------
// The segmented solve of tdma_seg.hpp with kTileP lanes per column: the
// interface system has kTileP rows and its cyclic reduction one more stride.
// A DPP row holds exactly one column, so a move past the column's end reads 0.
// ---------------------------------------------------------------------------
template <int D, int NR>
__device__ __forceinline__ void tile_pcr_step(int s, double& A, double& B, double& C, double (&R)[NR], double& al,
                                              double& ga) {
    double Bm = dpp_move<kDppShr + D>(B), Bp = dpp_move<kDppShl + D>(B);  // every lane moves
    Bm = s < D ? 1.0 : Bm;
    Bp = s + D >= kTileP ? 1.0 : Bp;
    const double Am = dpp_move<kDppShr + D>(A), Cm = dpp_move<kDppShr + D>(C);
    const double Ap = dpp_move<kDppShl + D>(A), Cp = dpp_move<kDppShl + D>(C);
    al = -A * seg_rcp(Bm);
    ga = -C * seg_rcp(Bp);
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        const double Rm = dpp_move<kDppShr + D>(R[q]), Rp = dpp_move<kDppShl + D>(R[q]);
        R[q] = R[q] + al * Rm + ga * Rp;
    }
    A = al * Am;
    C = ga * Cp;
    B = B + al * Cm + ga * Ap;
}
template <int D>
__device__ __forceinline__ double tile_rhs_step(double R, double al, double ga) {
    return R + al * dpp_move<kDppShr + D>(R) + ga * dpp_move<kDppShl + D>(R);
}

// The interface system with NR right-hand sides: cyclic reduction, then one step
// of iterative refinement (the rows' float64 residual, solved with the same
// factors). With eight lanes (iface_solve) only columns with a weakly dominant row
// need the step; the fourth stride's roundings make up for it on every column.
// The residual starts with R - B x, whose terms cancel, and REST: takes in what the
// forming of B and R cut off (Bl, Rl), so that a strongly dominant row's level is
// rounded about once; it is one level in nz / 16. Mean error of columns of 34 to 113
// levels against extended precision, in units of that of a sequential sweep, with the
// residual summed first and without Bl, Rl / now: temperature 1.02 to 1.07 / 0.86 to
// 1.00, velocity 1.05 to 1.12 / 0.93 to 1.07, energies 1.04 to 1.07 / 0.91 to 1.04. The
// same from the interface level's own row after the solve keeps ten registers more:
// vertical mixing and friction on 1440x720x80 2.26 -> 2.72 ms, now 2.27.
template <int NR, bool REST>
__device__ __forceinline__ void tile_iface(int s, double A, double B, double Bl, double C, const double (&R)[NR],
                                           const double (&Rl)[NR], double (&Ls)[NR], double (&Lm)[NR]) {
    double a = A, b = B, c = C, al[4], ga[4];
#pragma unroll
    for (int q = 0; q < NR; ++q) Ls[q] = R[q];
    tile_pcr_step<1, NR>(s, a, b, c, Ls, al[0], ga[0]);
    tile_pcr_step<2, NR>(s, a, b, c, Ls, al[1], ga[1]);
    tile_pcr_step<4, NR>(s, a, b, c, Ls, al[2], ga[2]);
    tile_pcr_step<8, NR>(s, a, b, c, Ls, al[3], ga[3]);
    const double rb = seg_rcp(b);
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        Ls[q] *= rb;
        double r = fma(-B, Ls[q], R[q]);
        if constexpr (REST) r += fma(-Bl, Ls[q], Rl[q]);
        r = fma(-A, dpp_move<kDppShr + 1>(Ls[q]), r);
        r = fma(-C, dpp_move<kDppShl + 1>(Ls[q]), r);
        r = tile_rhs_step<1>(r, al[0], ga[0]);
        r = tile_rhs_step<2>(r, al[1], ga[1]);
        r = tile_rhs_step<4>(r, al[2], ga[2]);
        r = tile_rhs_step<8>(r, al[3], ga[3]);
        Ls[q] = Ls[q] + r * rb;
        Lm[q] = dpp_move<kDppShr + 1>(Ls[q]);
    }
}

// NR right-hand sides of one matrix; z in, their solutions out. va and vc are
// overwritten by the sweep's factors (see seg_solve_f64). REST: see tile_iface (off for
// IDEMIX, whose rows' conditioning sets the error: 0.2% of it, and its four registers
// cost a wave at three levels per lane, 600x400x40 597 -> 610 us for the three models).
template <int S, int NR, bool REST>
__device__ __forceinline__ void tile_solve(const Tile<S>& t, double (&va)[S], const double (&vb)[S], double (&vc)[S],
                                           double (&z)[NR][S]) {
    const double aL = va[S - 1], bL = vb[S - 1], cL = vc[S - 1];
    {
        const double r = seg_rcp(vb[0]);
        vc[0] *= r;
        va[0] *= r;
#pragma unroll
        for (int q = 0; q < NR; ++q) z[q][0] *= r;
    }
#pragma unroll
    for (int i = 1; i < S - 1; ++i) {
        const double at = va[i];
        const double r = seg_rcp(vb[i] - at * vc[i - 1]);
        vc[i] *= r;
        va[i] = -at * va[i - 1] * r;
#pragma unroll
        for (int q = 0; q < NR; ++q) z[q][i] = (z[q][i] - at * z[q][i - 1]) * r;
    }
    va[S - 2] = -va[S - 2];
    vc[S - 2] = -vc[S - 2];
#pragma unroll
    for (int i = S - 3; i >= 0; --i) {
        const double cp = vc[i];
#pragma unroll
        for (int q = 0; q < NR; ++q) z[q][i] = z[q][i] - cp * z[q][i + 1];
        va[i] = -va[i] - cp * va[i + 1];
        vc[i] = -cp * vc[i + 1];
    }
    const double RA = aL * va[S - 2], nb = dpp_move<kDppShl + 1>(va[0]);
    const double RB = fma(cL, nb, fma(aL, vc[S - 2], bL));
    const double RBl = fma(cL, nb, fma(aL, vc[S - 2], bL - RB));
    const double RC = cL * dpp_move<kDppShl + 1>(vc[0]);
    double RD[NR], RDl[NR], Ls[NR], Lm[NR];
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        const double na = dpp_move<kDppShl + 1>(z[q][0]);
        RD[q] = fma(-cL, na, fma(-aL, z[q][S - 2], z[q][S - 1]));
        RDl[q] = fma(-cL, na, fma(-aL, z[q][S - 2], z[q][S - 1] - RD[q]));
    }
    tile_iface<NR, REST>(t.s, RA, RB, RBl, RC, RD, RDl, Ls, Lm);
#pragma unroll
    for (int q = 0; q < NR; ++q) {
#pragma unroll
        for (int i = 0; i < S - 1; ++i) z[q][i] = z[q][i] + fma(va[i], Lm[q], vc[i] * Ls[q]);  // the small terms first
        z[q][S - 1] = Ls[q];
    }
}

// The same with P lanes per column: kTileP as above, or kSegP by the
// elimination of tdma_seg.hpp.
template <int S, int NR, bool REST = true, int P>
__device__ __forceinline__ void col_solve(const Tile<S, P>& t, double (&va)[S], const double (&vb)[S], double (&vc)[S],
                                          double (&z)[NR][S]) {
    if constexpr (P == kTileP) {
        tile_solve<S, NR, REST>(t, va, vb, vc, z);
    } else {
        SegLane L;
        L.s = t.s;
        L.lo = t.lo;
        L.valid = true;
        L.base = 0;
        L.k0 = 0;
        if constexpr (NR == 1) seg_solve_f64<S, 1>(L, va, vb, vc, z[0]);
        else seg_solve2_f64<S, 1>(L, va, vb, vc, z[0], z[1]);
    }
}
// the next lane's value of the column (last lane: unspecified)
template <int P>
__device__ __forceinline__ double col_next(int s, double x) {
    if constexpr (P == kTileP) return dpp_move<kDppShl + 1>(x);
    else return grp_next(s, x);
}

// h = 1 / y and what its rounding cuts off: x (h + l) is x / y rounded once (but for
// ties to 2^-50), in two instructions where a division takes about 14.
struct Recip {
    double h, l;
};
__device__ __forceinline__ Recip recip(double y) {
    const double h = 1.0 / y;
    return {h, h * fma(-h, y, 1.0)};
}
__device__ __forceinline__ double scaled(double x, double h, double l) { return fma(x, h, x * l); }

// Lanes per column and levels per lane of the kernels that choose between the two:
// 8 lanes up to 32 levels, so that a wave takes 8 columns, else 16, which halve a
// lane's registers. us on 1435x896 (friction, vertical mixing) and 1000x600 (TKE +
// EKE + IDEMIX), 16 lanes / 8 lanes: nz 9 853 / 416, 287 / 177, 885 / 535; 17 936 /
// 606, 322 / 261, 977 / 774; 24 983 / 637, 341 / 322, 1043 / 845; 32 1031 / 853, 405 /
// 391, 1080 / 1017. Eight lanes from 33 levels on need five or more levels a lane,
// whose registers cost a wave per SIMD.
constexpr int col_lanes(int nz) { return nz <= 32 ? kSegP : kTileP; }
constexpr int col_levels(int nz) {
    const int s = (nz + col_lanes(nz) - 1) / col_lanes(nz);
    return s < 2 ? 2 : s;
}

}  // namespace vx
