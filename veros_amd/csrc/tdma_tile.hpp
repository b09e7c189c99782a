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
    const int64_t i = in && w >= g.tpr ? w / g.tpr : 0;  // columns in one row: no division in the chain to the loads
    const int64_t j0 = in ? (w - i * g.tpr) * g.cpt : 0;
    const int64_t left = g.ny - j0;
    const int n = in ? (int)(left < g.cpt ? left : g.cpt) : 0;
    const int64_t base = i * p.sx + j0 * p.sy;
    const Tile<S, kTdmaP> t = make_tile<S, kTdmaP>(base, n, p.nz, g.cpt > 1 ? (uint32_t)p.sy : 0u, depth_reciprocal(p.nz));
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

// The LDS-staged solve (those copies, tdma_seg.hpp) against the tiles, us,
// float64 / mixed with one step:
//   38.4 M cells   nz 40 189 / 188 against 192 / 196, 60 196 / 195 against
//                  179 / 187, 80 168 / 170 against 173 / 173, 96 188 / 189 against
//                  171 / 207, 112 236 / 240 against 194 / 211, 128 246 / 251
//                  against 204 / 233
//   640x640        nz 24 51 / 50 against 54 / 56, 60 128 / 127 against 119 / 124
//   128x128        nz 24 4.2 / 4.0 against 4.7 / 4.7, 60 6.5 / 6.3 against 7.3 /
//                  7.4, 96 10.9 / 11.0 against 10.0 / 11.0
//   96x96          nz 60 5.4 / 5.2 against 6.1 / 5.9, 96 6.6 / 6.6 against 8.3 /
//                  6.6, 112 10.1 / 10.3 against 9.3 / 9.2
// At any size it wins up to S = 6 and at S = 10, and for the mixed form at
// S = 12, where the tiles' flat loads cost a wave per SIMD. Elsewhere its LDS
// (one block of two waves holds 8 KB per level of a lane) leaves too few waves on a
// large grid, and it wins while all of them are resident at once
// (tdma_lds_resident): nothing waits for a free slot then, and its chain from
// kbot to the rows is the shorter one. In the batched kernel the tiles' registers
// cost a wave per SIMD at S = 12, and spill at S = 14 in the mixed form: 640x640x96
// 198 against 244, x112 mixed 309 against 338 (float64 301 against 281).
__host__ __device__ constexpr bool tdma_lds_wins(int S, bool mixed, bool batch) {
    return S <= 6 || S == 10 || (S == 12 && (mixed || batch)) || (S == 14 && mixed && batch);
}
// Two levels per lane (nz <= 16) with operands those copies don't fit: each lane
// loads its own levels; the 8 lanes of a column then read it whole, so the flat
// loads gain nothing. 320x320x13 10.4 against 10.7 us (tiles), 1200x1200x13 124
// against 126, 128x128x15 3.5 against 3.8; at four levels (nz 25) 1200x1200 265
// against 211.
__host__ __device__ constexpr bool tdma_own_levels(int S) { return S == 2; }
inline bool tdma_lds_resident(int S, int64_t ntiles) {
    const int blocks = (160 << 10) / (seg_lds_wave_bytes(S) * (kSegLdsBlock / 64));
    return ntiles <= (int64_t)blocks * (kSegLdsBlock / 64) * cu_count();
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
