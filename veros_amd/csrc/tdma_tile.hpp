// The kbot-masked solves on column tiles (col_tile.hpp): a wave owns a tile of
// up to 8 columns of one row (8 lanes per column), loads the wet cells of a, b,
// c and d flat, passes them through one LDS image to the segments, solves
// (seg_solve_f64, or the mixed form), and stores x flat over every cell. Any
// strides and alignments, any depth.
//
// Bound by HBM, whose rate the sparse reads lower: streaming five whole arrays
// with these accesses runs at 5.4 TB/s, the wet suffixes only (1.67 GB on
// 1440x720x80) at 4.2-4.4 TB/s, with or without the solve between the loads and
// the stores. A persistent grid with the next tile's loads issued before the
// solve was no faster (0.41 against 0.38 ms).
#pragma once
#include "col_tile.hpp"

namespace vx {

constexpr int kTdmaP = 8;               // lanes per column
constexpr int kTdmaCols = 64 / kTdmaP;  // columns per tile

// How the columns (i, j) are cut into tiles: `tpr` tiles of `cpt` columns per
// row i of `ny` columns. When the columns follow each other at one stride all
// through, arrays and kbot alike, they are taken as one row. cpt is 8, or 1 when
// 8 columns would not fit a buffer's 32-bit offsets.
struct TdmaTiling {
    int64_t ny, tpr, ntiles;
    int32_t cpt;
};
inline TdmaTiling tdma_tiling(const TdmaArgs& p) {
    TdmaTiling g;
    const int64_t nx = p.ncol / p.ny;
    const bool one_row = nx == 1 || (p.sx == p.ny * p.sy && p.kx == p.ny * p.ky);
    g.ny = one_row ? p.ncol : p.ny;
    g.cpt = (int64_t)kTdmaCols * p.sy * 8 < (int64_t)kNoAccess ? kTdmaCols : 1;
    g.tpr = (g.ny + g.cpt - 1) / g.cpt;
    g.ntiles = g.tpr * (p.ncol / g.ny);
    return g;
}

// Tile w of the columns (no columns from ntiles on), and the lane's group
// column: its first wet level (nz: none) and offset.
template <int S>
__device__ __forceinline__ Tile<S, kTdmaP> tdma_tile_of(const TdmaArgs& p, const TdmaTiling& g, int64_t w, SegLane& L) {
    const bool in = w < g.ntiles;
    const int64_t i = in ? w / g.tpr : 0;
    const int64_t j0 = in ? (w - i * g.tpr) * g.cpt : 0;
    const int64_t left = g.ny - j0;
    const int n = in ? (int)(left < g.cpt ? left : g.cpt) : 0;
    const int64_t base = i * p.sx + j0 * p.sy;
    const Tile<S, kTdmaP> t = make_tile<S, kTdmaP>(base, n, p.nz, g.cpt > 1 ? (uint32_t)p.sy : 0u);
    L.s = t.s;
    L.lo = t.lo;
    L.valid = t.q < n;
    const int kb = p.kbot[L.valid ? i * p.kx + (j0 + t.q) * p.ky : 0];
    L.k0 = L.valid && kb >= 1 && kb <= p.nz ? kb - 1 : p.nz;
    L.base = base + (L.valid ? t.q * p.sy : 0);
    return t;
}

// Whether 16-byte copies straight into LDS fit the operands.
inline bool tdma_vec_ok(const TdmaArgs& p) {
    if ((p.nz & 1) || (p.sx & 1) || (p.sy & 1)) return false;
    return aligned16(p.a) && aligned16(p.b) && aligned16(p.c) && aligned16(p.d) && aligned16(p.x);
}

// The LDS-staged solve (those copies, tdma_seg.hpp) against the tiles, on 38.4 M
// cells (us, float64 / mixed with one step): nz 40 189 / 188 against 192 / 196,
// 60 196 / 195 against 179 / 187, 80 168 / 170 against 173 / 173, 96 188 / 189
// against 171 / 207, 112 236 / 240 against 194 / 211, 128 246 / 251 against
// 204 / 233. It wins where the segment stride in its images spreads over the
// LDS banks (S / 2 odd: 2, 6, 10 levels per lane) and four blocks fit a CU
// (S <= 10); and for the mixed form at S = 12, where the tiles' flat loads cost
// a wave per SIMD.
__host__ __device__ constexpr bool tdma_lds_wins(int S, bool mixed) {
    return (S <= 10 && (S / 2) % 2 == 1) || (mixed && S == 12);
}

// LDS doubles of a wave
template <int S>
__host__ __device__ constexpr int tdma_tile_lds() {
    return Tile<S, kTdmaP>::IMG;
}

// Solves one tile; `img` is the wave's LDS image. MODE: -1 float64, else the
// mixed form with MODE refinement steps. The segments are those of the other
// segmented kernels (seg_levels), so the results are theirs bit for bit.
template <int S, int MODE>
__device__ __forceinline__ void tdma_tile(const TdmaArgs& p, const Tile<S, kTdmaP>& t, const SegLane& L, double* img) {
    double x[S];
    if (__any(L.k0 < p.nz)) {
        double va[S], vb[S], vc[S], vd[S];
        {
            uint32_t wet[S];
#pragma unroll
            for (int r = 0; r < S; ++r)
                wet[r] = t.k[r] >= __shfl(L.k0, t.c[r] * kTdmaP) ? t.off[r] : kNoAccess;
            tile_load(tile_buf(t, p.a), wet, 1, va);
            tile_load(tile_buf(t, p.b), wet, 1, vb);
            tile_load(tile_buf(t, p.c), wet, 1, vc);
            tile_load(tile_buf(t, p.d), wet, 1, vd);
        }
        double be, de;
        seg_edge_values(p, L, S, be, de);
        tile_put(t, img, va);
        seg_get(t, img, va);
        tile_put(t, img, vb);
        seg_get(t, img, vb);
        tile_put(t, img, vc);
        seg_get(t, img, vc);
        tile_put(t, img, vd);
        seg_get(t, img, vd);
        seg_mask_rows<S>(p, L, be, de, va, vb, vc, vd);
        if constexpr (MODE < 0) {
            seg_solve_f64<S>(L, va, vb, vc, vd);
            seg_put(t, img, vd);
        } else {
            seg_mixed_core<S, MODE>(L, va, vb, vc, vd, x);
            seg_put(t, img, x);
        }
        tile_get(t, img, x);
    } else {
#pragma unroll
        for (int r = 0; r < S; ++r) x[r] = 0.0;
    }
    tile_store(tile_buf(t, (const double*)p.x), t.off, 1, x);
}

}  // namespace vx
