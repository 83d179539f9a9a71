// Partition of particles by deposit tile (sort.hip) and the per-particle
// cell arithmetic shared by the deposit and the adjoint gather.
#pragma once
#include "plan.h"

namespace genpk {

struct KeyGeom {
  double units;
  int d;
  int TX, TY, TZ;      // tile edge, powers of two
  int sx, sy, sz;      // log2 of the tile edges
  int ntx, nty, ntz;
};

KeyGeom key_geom(const Plan &p, double boxsize);

// Floor cell of one coordinate, wrapped into [0, d), and the fractional part
// (fieldize.cpp:66-75).  The floor is converted to a 32-bit integer as the
// reference does; positions more than one box outside [0, box) take the
// general modulo.  A floor outside the int range converts with the GPU's
// saturation (NaN to 0), so every record still gets a valid tile; the
// deposit skips a record whose fractional part is not finite, and k_poison
// finds its cells with cell_of_x86.
__device__ __forceinline__ int cell_of(float p, double units, int d, double &frac) {
  const double u = (double)p * units;
  const double f = floor(u);
  frac = u - f;
  int c = (int)f;
  if ((unsigned)c >= (unsigned)d) {
    c %= d;
    if (c < 0) c += d;
  }
  return c;
}

// cell_of with the conversion x86-64 makes (cvttsd2si): a floor outside the
// int range, NaN or an infinity converts to INT_MIN (the "integer
// indefinite"), so a non-finite position maps to the cells the reference
// gives it.
__device__ __forceinline__ int cell_of_x86(float p, double units, int d, double &frac) {
  const double u = (double)p * units;
  const double f = floor(u);
  frac = u - f;
  int c = (f >= -2147483648.0 && f < 2147483648.0) ? (int)f : (int)0x80000000u;
  if ((unsigned)c >= (unsigned)d) {
    c %= d;
    if (c < 0) c += d;
  }
  return c;
}

// Work item -> tile k and its list entries [lb, le).  Items below nsplit are
// those of split tiles, which divide a tile's blocks evenly; the others are
// one per tile.  One 16-byte record per item: with an item -> tile table and
// the tile's list start to read after it, that chain came into every item
// (deposit 2.29 -> 1.96 ms for 2^22 records in 2^18 tiles of 4^3 cells, 2.44 ->
// 2.14 for 2^26 in 2^18 of 8^3, 0.267 -> 0.245 for 2^22 in 16 000 of 16 x 32 x 32).
struct ItemRange {
  int64_t k;
  uint32_t lb, le;
};
// The table comes as a restrict kernel argument (not inside a struct), so that
// this uniform read is a scalar load also after the kernel has stored.
__device__ __forceinline__ void item_range(const uint4 *__restrict__ items, uint32_t nsplit, uint32_t max_parts,
                                           uint32_t item, ItemRange &r) {
  const uint4 t = items[item < nsplit ? item : item - nsplit + max_parts];
  r.k = t.x;
  r.lb = t.y;
  r.le = t.z;
}

// Records per work item at most for n particles over `tiles` tiles:
// DEPOSIT_ITEM_MAX, halved (down to DEPOSIT_ITEM_MIN) while the items would
// number fewer than four per CU or one full item would hold more than half of
// a CU's share of the particles (a quarter, where that leaves tiles of twice
// the mean in one item), so that heavy tiles spread evenly over the CUs (their
// items' partial tiles are summed afterwards).  Without that limit a quarter
// cut half the tiles of a 256^3 lattice (forward 0.385 -> 0.479 ms); with half
// as many items clumped particles fill the CUs less evenly (2e7 at 384^3: the
// fullest 1.13 times the mean, 1.06 with a quarter).
uint32_t deposit_item_max(int64_t n, int64_t tiles);

// Workgroups of the deposit over records of rw floats: those that stay
// resident, at most DEPOSIT_WGS_MAX and one per item.
constexpr int64_t DEPOSIT_WGS_MAX = 1024;
int64_t deposit_wgs(const Plan &p, int rw, int64_t max_items);

// Partition the n particles of one call (n <= 2^31) by tile into plan
// scratch and build the work items (at most deposit_item_max records each).
// Records are x, y, z, then the mass when masses != nullptr.  with_perm: also
// record where every particle went (perm1: input -> pass-1 slot; perm2, two
// passes only: pass-1 slot -> slot in rec), for taking results back to the
// input order without scattered writes.  every_tile: every tile gets at
// least one item (the deposit then writes untouched tiles as zeros);
// otherwise empty tiles get none.
TileOrder sort_by_tile(Plan &p, const KeyGeom &kg, int64_t n, const float *pos, const float *masses, bool with_perm,
                       bool every_tile);

}  // namespace genpk
