// Halo'd tile store of the deposit and its fold into the real-space grid.
//
// Tile t = (tx*nty + ty)*ntz + tz covers cells [tx*TX, tx*TX+wx) x ... with
// wx = min(TX, d - tx*TX); its accumulator has (TX+1)(TY+1)(TZ+1) cells
// (local index 0..TX along x, and so on).  Local index wx (the halo layer)
// holds the CIC weight that belongs to the first cell of the next tile along
// that axis (periodically), so the value of grid cell (x, y, z) is the sum
// over the one or two (tile, local) sources per axis.
//
// Store layout: rows of TZ values for local z < TZ, HX*HY rows per tile,
// tile after tile (each row is 32 floats = 128 bytes, aligned), followed by
// the z-halo plane (local z = TZ) of every tile, HX*HY values per tile.  The
// halos stay where the deposit put them; the readers (the z pass, the export)
// add them while they load: rows of a tile's first x or y layer, 1 in TX and
// 1 in TY, read up to three more rows.  (Folding y and x halos in place after
// the deposit wrote those faces and zeroed the halos in two launches: 0.43
// ms at 1024^3 FP32.)
#pragma once
#include "common.h"

namespace genpk {

struct FoldGeom {
  int d;
  int TX, TY, TZ, sx, sy, sz;
  int ntx, nty, ntz;
  int HY, HZ;
  int64_t cm;     // row-store values per tile: HX*HY*TZ
  int64_t cz;     // z-halo values per tile: HX*HY
  int64_t zoff;   // start of the z-halo planes: K*cm
};

// Store offset of (tile t, local lx, ly, lz), lz <= TZ.
__device__ __forceinline__ int64_t tile_at(const FoldGeom &P, int64_t t, int lx, int ly, int lz) {
  const int64_t r = (int64_t)lx * P.HY + ly;
  return lz < P.TZ ? t * P.cm + r * P.TZ + lz : P.zoff + t * P.cz + r;
}

// Store offset of grid cell (x, y, z) in the tile that contains it (its own
// accumulator cell; halo contributions of the previous tiles are separate).
__device__ __forceinline__ int64_t cell_at(const FoldGeom &P, int x, int y, int z) {
  const int64_t t = (((int64_t)(x >> P.sx) * P.nty + (y >> P.sy)) * P.ntz) + (z >> P.sz);
  return tile_at(P, t, x & (P.TX - 1), y & (P.TY - 1), z & (P.TZ - 1));
}

// The stored rows (tile row txy = tx*nty + ty, local row lx*HY + ly) whose
// sum is the grid's row (x, y): its own, the y halo of the previous tile along
// y (ly = 0 only), the x halo of the previous tile along x (lx = 0 only), and
// that halo's own y halo (both).
struct RowFold {
  int64_t t, r;            // own
  bool fx, fy;
  int64_t ty, ry, tx, rx, txy, rxy;
};
__device__ __forceinline__ RowFold row_fold(const FoldGeom &P, int x, int y) {
  RowFold f;
  const int tx = x >> P.sx, ty = y >> P.sy, lx = x & (P.TX - 1), ly = y & (P.TY - 1);
  f.t = (int64_t)tx * P.nty + ty;
  f.r = (int64_t)lx * P.HY + ly;
  f.fx = lx == 0;
  f.fy = ly == 0;
  if (f.fx || f.fy) {
    const int txp = tx == 0 ? P.ntx - 1 : tx - 1, typ = ty == 0 ? P.nty - 1 : ty - 1;
    const int hx = min(P.TX, P.d - txp * P.TX), hy = min(P.TY, P.d - typ * P.TY);
    f.ty = (int64_t)tx * P.nty + typ;
    f.ry = (int64_t)lx * P.HY + hy;
    f.tx = (int64_t)txp * P.nty + ty;
    f.rx = (int64_t)hx * P.HY + ly;
    f.txy = (int64_t)txp * P.nty + typ;
    f.rxy = (int64_t)hx * P.HY + hy;
  }
  return f;
}

// Place along z of grid cell z within any stored row: its own cell, and for
// the first cell of a tile along z the z-halo cell of the previous tile along
// z (at local z = that tile's width: the z-halo plane for full tiles, the row
// store for a partial last tile).
struct ZPlace {
  int64_t at;       // own cell: txy * ntz * cm + r * TZ + at
  bool halo, hrow;  // halo cell: txy * ntz * cm + r * TZ + h (hrow), else txy * ntz * cz + r + h
  int64_t h;
};
__device__ __forceinline__ ZPlace z_place(const FoldGeom &P, int z) {
  ZPlace p;
  const int tz = z >> P.sz, lz = z & (P.TZ - 1);
  p.at = (int64_t)tz * P.cm + lz;
  p.halo = lz == 0;
  const int tzp = tz == 0 ? P.ntz - 1 : tz - 1;
  const int w = min(P.TZ, P.d - tzp * P.TZ);
  p.hrow = w < P.TZ;
  p.h = p.hrow ? (int64_t)tzp * P.cm + w : P.zoff + (int64_t)tzp * P.cz;
  return p;
}
__device__ __forceinline__ int64_t row_at(const FoldGeom &P, int64_t txy, int64_t r, const ZPlace &z) {
  return txy * P.ntz * P.cm + r * P.TZ + z.at;
}
__device__ __forceinline__ int64_t row_halo_at(const FoldGeom &P, int64_t txy, int64_t r, const ZPlace &z) {
  return z.hrow ? txy * P.ntz * P.cm + r * P.TZ + z.h : txy * P.ntz * P.cz + r + z.h;
}

// The x and y halos of N cell pairs (z_i, z_i + 1) of row f added to v[i] (the
// own cells) and zh[i] (the z-halo cells, 0 where there is none): own + y
// halo, then + (x halo + its y halo), each sum rounded once in T.  Few rows
// take this, so it works on GRP pairs at a time (the memory clobber keeps the
// others' loads behind them): all eight at once would triple the z pass's
// registers and halve its occupancy (2.71 ms at 1024^3 FP32, 2.06 in fours,
// 2.12 in twos).
template <typename T, int N, int GRP, typename C, typename ZOf>
__device__ __forceinline__ void add_halo_rows(const T *__restrict__ tiles, const FoldGeom &P, const RowFold &f, ZOf z_of,
                                              C (&v)[N], T (&zh)[N]) {
  static_assert(N % GRP == 0, "whole groups");
#pragma unroll
  for (int g = 0; g < N; g += GRP) {
    ZPlace z[GRP];
#pragma unroll
    for (int i = 0; i < GRP; i++) z[i] = z_place(P, z_of(g + i));
    auto read = [&](int64_t txy, int64_t r, C (&w)[GRP], T (&wh)[GRP]) {
#pragma unroll
      for (int i = 0; i < GRP; i++) {
        const int64_t at = row_at(P, txy, r, z[i]);
        w[i] = C{tiles[at], tiles[at + 1]};
        wh[i] = z[i].halo ? tiles[row_halo_at(P, txy, r, z[i])] : (T)0;
      }
    };
    C a[GRP], b[GRP];
    T ah[GRP], bh[GRP];
#pragma unroll
    for (int i = 0; i < GRP; i++) {
      a[i] = b[i] = C{0, 0};
      ah[i] = bh[i] = (T)0;
    }
    if (f.fy) {
      read(f.ty, f.ry, a, ah);
#pragma unroll
      for (int i = 0; i < GRP; i++) {
        v[g + i] = C{v[g + i].x + a[i].x, v[g + i].y + a[i].y};
        zh[g + i] = zh[g + i] + ah[i];
      }
    }
    if (f.fx) {
      read(f.tx, f.rx, a, ah);
      if (f.fy) {
        read(f.txy, f.rxy, b, bh);
#pragma unroll
        for (int i = 0; i < GRP; i++) {
          a[i] = C{a[i].x + b[i].x, a[i].y + b[i].y};
          ah[i] = ah[i] + bh[i];
        }
      }
#pragma unroll
      for (int i = 0; i < GRP; i++) {
        v[g + i] = C{v[g + i].x + a[i].x, v[g + i].y + a[i].y};
        zh[g + i] = zh[g + i] + ah[i];
      }
    }
    asm volatile("" ::: "memory");
  }
}

}  // namespace genpk
