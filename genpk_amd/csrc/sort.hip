// Partition of particles by deposit tile on gfx950: a radix partition of one
// or two passes over the tile key.  The last pass is always paged: every
// workgroup ranks the records of its chunk with LDS atomics, stages them in
// LDS by digit and appends each digit's run to blocks of record slots that
// it takes from a range of its own, so there is no histogram pass and no
// shared cursor; a small directory (k_dir, k_list) then lists every tile's
// blocks and its work items, and the tile kernels read the records through
// that list.  A first pass is paged the same way where each workgroup holds
// many records of each digit; elsewhere it counts first (k_upsweep, an
// offset scan) and writes contiguous runs.  Global atomics are avoided but
// for one per workgroup and digit: on this chip they run at ~27 Gop/s.  The
// order of the records within one tile is not specified (the tile kernels
// do not depend on it).
#include "tilesort.h"

#include <algorithm>

namespace genpk {

namespace {

// 16 waves per workgroup, one workgroup per CU in the downsweep: a
// sub-chunk of 1024 * PL records is staged in LDS at a time and written out
// as one run per digit, and longer runs write faster (at 2^30 records and
// 256 digits, 8192-record sub-chunks take 6.9 ms per downsweep against 7.2
// ms for two 512-thread workgroups per CU staging 4096 records each).
constexpr int SORT_THREADS = 1024;
constexpr int SORT_WAVES = SORT_THREADS / 64;
// Records per workgroup of the counted first pass: from SORT_CHUNK_MIN (one
// sub-chunk) up to SORT_CHUNK_MAX, the smallest that keeps at most four
// chunks per CU (small sets then still spread over every CU).
constexpr int64_t SORT_CHUNK_MIN = 8192, SORT_CHUNK_MAX = 32768;

// Source of records: either the caller's arrays (positions [n][3], optional
// masses [n]) or a packed record buffer of RW floats per record.
template <int NM>
struct Src {
  static constexpr int RW = 3 + NM;
  const float *pos;     // raw positions (stride 3) or packed records (stride RW)
  const float *masses;  // raw masses when reading the caller's arrays
  bool raw;
  __device__ __forceinline__ void load_pos(int64_t i, float *r) const {
    const int64_t st = raw ? 3 : RW;
    r[0] = pos[st * i + 0];
    r[1] = pos[st * i + 1];
    r[2] = pos[st * i + 2];
  }
  __device__ __forceinline__ void load(int64_t i, float *r) const {
    if (raw) {
      r[0] = pos[3 * i + 0];
      r[1] = pos[3 * i + 1];
      r[2] = pos[3 * i + 2];
      if (NM) r[3] = masses[i];
    } else {
#pragma unroll
      for (int k = 0; k < RW; k++) r[k] = pos[RW * i + k];
    }
  }
};

// Input of a pass: workgroup g takes slots [g * chunk, (g + 1) * chunk).
//   IN_RAW: slots are the caller's n records.
//   IN_SEG / IN_LIST: slots are the records, or the record slots of the
//   block-list entries (2^lg each), of a first pass's buckets, bucket s from
//   record or entry start[s] on; first_seg[g] is the bucket of g's first slot.
//   A workgroup handles the part of each bucket in its range as a piece of
//   its own (a bucket's digits are not another's); piece w + s is workgroup
//   w's of bucket s, and lacks[w + s] (IN_LIST; null: not counted) the slots
//   of its blocks that hold no record.
enum { IN_RAW = 0, IN_SEG = 1, IN_LIST = 2 };
struct InMap {
  int64_t n = 0, chunk = 0;
  int nseg = 0;
  int lg = 0;
};

// Output of a paged pass: a pool of blocks of 2^lg record slots, in which
// every piece has a range large enough for its full blocks and one partly
// filled block per digit: it starts at block (records before the piece, or
// slots where lacks are not counted, >> lg) + (w + s) (nb + 1).
struct PgOut {
  uint16_t *hdr = nullptr;    // digit of each taken block, written with the block's first record
  uint32_t *cnt = nullptr;    // [pieces * nb] records per digit of each piece (written where not 0)
  uint32_t *last = nullptr;   // [pieces * nb] the digit's last block (the one that may be partly filled)
  uint32_t *base = nullptr;   // [pieces * nb] number of the piece's first block among its bucket's
  uint4 *piece = nullptr;     // first block, blocks taken, bucket (blocks taken: 0 where there is no piece)
  unsigned long long *tot = nullptr;  // per output bucket: blocks << 32 | records, summed over the pieces
  int lg = 0;
};

// A block-list entry: the block in the low 32 - lg bits, its fill (1 to 2^lg
// records) less one above, so that one load gives both.
__device__ __forceinline__ uint32_t pg_entry(uint32_t blk, uint32_t fill, int lg) {
  return blk | (fill - 1) << (32 - lg);
}

// Tile key of a position with the cells along the axes not in `axes` (bit a:
// axis a of x, y, z) taken as 0 and not computed: cell_of's cells, with one
// branch for the rare wrap of any of them into [0, d).
__device__ __forceinline__ uint32_t key_on_axes(const float *r, const KeyGeom &g, int axes) {
  int c[3];
#pragma unroll
  for (int a = 0; a < 3; a++) c[a] = (axes >> a) & 1 ? (int)floor((double)r[a] * g.units) : 0;
  const unsigned ud = (unsigned)g.d;
  if (((unsigned)c[0] >= ud) | ((unsigned)c[1] >= ud) | ((unsigned)c[2] >= ud)) {
#pragma unroll
    for (int a = 0; a < 3; a++)
      if ((unsigned)c[a] >= ud) {
        c[a] %= g.d;
        if (c[a] < 0) c[a] += g.d;
      }
  }
  return (uint32_t)((((c[0] >> g.sx) * g.nty + (c[1] >> g.sy)) * g.ntz) + (c[2] >> g.sz));
}

struct DigitSel {
  int shift;
  uint32_t mask;
  int axes;  // bit a set: the digit depends on the tile index along axis a (x, y, z)
  __device__ __forceinline__ uint32_t of_key(uint32_t key) const { return (key >> shift) & mask; }
  // digit of a record; cells along axes the digit does not depend on are not computed
  __device__ __forceinline__ uint32_t of(const float *r, const KeyGeom &g) const {
    return of_key(key_on_axes(r, g, axes));
  }
};

int log2_floor(int v) {
  int l = 0;
  while ((1 << (l + 1)) <= v) l++;
  return l;
}

// Digit of key bits [shift, shift + width).  The key is (tx * nty + ty) * ntz
// + tz; when nty and ntz are powers of two its bits are tz, then ty, then tx,
// and a digit needs only the axes whose bits it covers.
DigitSel digit_sel(const KeyGeom &g, int shift, int width) {
  DigitSel s{shift, (uint32_t)((1u << width) - 1), 7};
  if ((g.nty & (g.nty - 1)) != 0 || (g.ntz & (g.ntz - 1)) != 0) return s;
  const int bz = log2_floor(g.ntz), by = log2_floor(g.nty);
  const int lo[3] = {bz + by, bz, 0}, hi[3] = {32, bz + by, bz};
  s.axes = 0;
  for (int a = 0; a < 3; a++)
    if (lo[a] < hi[a] && lo[a] < shift + width && shift < hi[a]) s.axes |= 1 << a;
  return s;
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// counts[dg * G + g] = number of records of chunk g with digit dg
template <int NM>
__global__ void __launch_bounds__(SORT_THREADS) k_upsweep(Src<NM> src, InMap im, KeyGeom kg, DigitSel ds, int nb,
                                                          uint32_t *__restrict__ counts) {
  constexpr int UNR = 8;
  extern __shared__ uint32_t hist[];
  const int64_t b = blockIdx.x * im.chunk, e = min(im.n, b + im.chunk);
  for (int i = threadIdx.x; i < nb; i += SORT_THREADS) hist[i] = 0;
  __syncthreads();
  for (int64_t base = b; base < e; base += SORT_THREADS * UNR) {
    float r[UNR][3];
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const int64_t i = base + u * SORT_THREADS + threadIdx.x;
      if (i < e) src.load_pos(i, r[u]);
    }
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const int64_t i = base + u * SORT_THREADS + threadIdx.x;
      const bool valid = i < e;
      const uint32_t dg = valid ? ds.of(r[u], kg) : 0u;
      // a wavefront whose records share one digit adds them with one atomic
      const uint64_t vmask = __ballot(valid);
      const uint32_t d0 = __builtin_amdgcn_readlane(dg, (int)__builtin_ctzll(vmask | (1ull << 63)));
      if (__ballot(valid && dg == d0) == vmask) {
        if (valid && (vmask & lanemask_lt()) == 0) atomicAdd(&hist[d0], (uint32_t)__popcll(vmask));
      } else if (valid) {
        atomicAdd(&hist[dg], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += SORT_THREADS) counts[(int64_t)i * gridDim.x + blockIdx.x] = hist[i];
}

// Rank of each of a lane's PL record slots among the wave's slots of its
// digit in this sub-chunk, from LDS atomic adds that return the old count on
// the wave's count row (a wave whose 64 slots share one digit adds them with
// one atomic, from lane 0).  Slots not in vm hold no record: they take the
// digit `trash` (one past the last), so that they rank and stage like
// records, after every real one.  Equal digits are ordered by the LDS unit's
// processing order of one instruction's lanes and, where waves share a count
// row, by the order in which they run: the order of the records within a
// tile is not specified (the tile kernels do not depend on it).  pk
// receives each slot's rank (bits 0-12, below the sub-chunk's 8192 slots)
// and its digit from bit 13: one register per slot.  Called by whole waves.
template <int NM, int PL>
__device__ __forceinline__ void rank_records(const float (&rec)[PL][Src<NM>::RW], uint32_t vm, const KeyGeom &kg,
                                             const DigitSel &ds, uint32_t trash, uint32_t *wrow, uint32_t (&pk)[PL]) {
  const uint32_t lane = threadIdx.x & 63;
  uint32_t rnk[PL];
  uint32_t uni = 0;  // bit it: the wave's slots `it` share one digit
#pragma unroll
  for (int it = 0; it < PL; it++) {
    const uint32_t dg = (vm >> it) & 1u ? ds.of(rec[it], kg) : trash;
    const uint32_t d0 = __builtin_amdgcn_readfirstlane(dg);
    uint32_t r = 0;
    if (__ballot(dg == d0) == ~0ull) {
      if (lane == 0) r = atomicAdd(&wrow[d0], 64u);
      uni |= 1u << it;
    } else {
      r = atomicAdd(&wrow[dg], 1u);
    }
    pk[it] = dg << 13;
    rnk[it] = r;
  }
  // a one-digit wave's slots follow lane 0's old count
#pragma unroll
  for (int it = 0; it < PL; it++)
    pk[it] |= (uni >> it) & 1u ? __builtin_amdgcn_readlane(rnk[it], 0) + lane : rnk[it];
}

// Per-row counts of digit dg -> per-row exclusive offsets in place; returns the total.
__device__ __forceinline__ uint32_t wave_offsets(uint32_t *whist, int nbt, int hw, int dg) {
  uint32_t tot = 0;
  for (int w = 0; w < hw; w++) {
    const uint32_t t = whist[w * nbt + dg];
    whist[w * nbt + dg] = tot;
    tot += t;
  }
  return tot;
}

// Inclusive scan of a whole wave by DPP moves, with no LDS round trip: within
// the rows of 16 lanes, then row 0's and 2's sums into the rows after them and
// the first half's into the second.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return v;
}

// Of the waves' totals in LDS: the sum of those before this wave's, and of
// all (one read per lane and a scan, not a read and an add per wave).
__device__ __forceinline__ uint32_t waves_before(const uint32_t *wtot, uint32_t &all) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t t = wtot[lane & (SORT_WAVES - 1)], incl = wave_incl_scan(lane < SORT_WAVES ? t : 0u);
  all = __builtin_amdgcn_readlane(incl, SORT_WAVES - 1);
  return __builtin_amdgcn_readlane(incl, wave) - __builtin_amdgcn_readlane(t, wave);
}

// One round of a block-wide exclusive scan (one value per thread), added to
// and advancing the running total 'carry'.  Contains a barrier; wtot rows
// alternate between rounds.
__device__ __forceinline__ uint32_t block_scan_round(uint32_t v, uint32_t (*wtot)[SORT_WAVES], int rd,
                                                     uint32_t &carry) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t incl = wave_incl_scan(v);
  if (lane == 63) wtot[rd & 1][wave] = incl;
  __syncthreads();
  uint32_t all;
  const uint32_t run = carry + incl - v + waves_before(wtot[rd & 1], all);
  carry += all;
  return run;
}

// Partition of each piece by digit.  PERM: perm[i] = output
// position of input record i (IN_LIST: of pool slot i).
// Per sub-chunk of SORT_THREADS * PL record slots (each wave owns 64 * PL
// consecutive ones): ranks (rank_records; the slots without a record take
// the digit nb, one past the last), then one thread per digit turns the
// per-wave counts into offsets and a block scan gives the digit's start in a
// digit-sorted staging copy, records go to the staging copy, and the staging
// copy's records (every slot before digit nb's start) are written out as
// contiguous runs while the next sub-chunk's records load.  With DB the
// per-wave counts are double-buffered: this sub-chunk's buffer is cleared
// during the write-out and the next sub-chunk ranks into the other one, so
// no barrier separates them.  hw count rows (a divisor of the wave count)
// serve the waves, wave w on row w % hw.
//   PAGED: each digit's records are appended to its current block of 2^lg
//     slots until that is full, then to new blocks of the piece's own range of
//     the pool: staging position p of digit dg goes to dinfo[dg].z + p below
//     dinfo[dg].y, else to dinfo[dg].w + p (dinfo[dg].x is the digit's staging
//     start).  At a piece's end its blocks and records of each digit are added
//     to the bucket's totals with one atomic, whose old value numbers the
//     piece's blocks among the bucket's.
//   else: record p goes to dinfo[its digit].z + p, from the chunk's scanned
//     offsets[dg * gridDim.x + g].
// blist (IN_LIST): block and fill of each list entry (pg_entry).
template <int NM, int PL, bool DB, int IN, bool PAGED, bool PERM>
__global__ void __launch_bounds__(SORT_THREADS, 4) k_partition(const float *__restrict__ pos,
                                                               const float *__restrict__ masses,
                                                               const uint32_t *__restrict__ blist,
                                                               const uint32_t *__restrict__ start,
                                                               const uint32_t *__restrict__ first_seg,
                                                               const uint32_t *__restrict__ lacks,
                                                               float *__restrict__ dst, InMap im, KeyGeom kg,
                                                               DigitSel ds, int nb, int hw,
                                                               const uint32_t *__restrict__ offsets,
                                                               uint32_t *__restrict__ perm,
                                                               uint32_t *__restrict__ mrange_w, PgOut pg) {
  constexpr int RW = Src<NM>::RW;
  const Src<NM> src{pos, masses, IN == IN_RAW};
  constexpr int SUBN = SORT_THREADS * PL;
  constexpr int NBUF = DB ? 2 : 1;
  static_assert(SUBN <= 8192, "ranks take 13 bits (rank_records)");
  extern __shared__ uint4 sm4[];
  const int nbt = nb + 1;                                    // digits and the empty slots' digit nb
  uint4 *dinfo = sm4;                                        // [nbt]
  uint32_t *whist_all = reinterpret_cast<uint32_t *>(dinfo + nbt);  // [NBUF][hw][nbt]
  uint32_t *dcnt = whist_all + NBUF * hw * nbt;              // PAGED [nb]: records of the digit so far
  uint32_t *dblk = dcnt + (PAGED ? nb : 0);                  // PAGED [nb]: the digit's last block
  uint16_t *sdig = reinterpret_cast<uint16_t *>(dblk + (PAGED ? nb : 0));  // [SUBN]
  float *stage = reinterpret_cast<float *>(sdig + SUBN);      // [SUBN][RW]
  __shared__ uint32_t wtot[2][SORT_WAVES];
  __shared__ uint32_t smr[2];  // masses: largest, smallest nonzero |mass| bits of this chunk

  // this workgroup's slots, and the piece [., pe) of them in bucket seg
  const int sh = IN == IN_LIST ? im.lg : 0;
  const int64_t cb = blockIdx.x * im.chunk;
  const int64_t ce = min(IN == IN_RAW ? im.n : (int64_t)start[im.nseg] << sh, cb + im.chunk);
  if (cb >= ce) return;
  uint32_t seg = IN == IN_RAW ? 0u : first_seg[blockIdx.x];
  int64_t pe = IN == IN_RAW ? ce : min(ce, (int64_t)start[seg + 1] << sh);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t pb = 1u << pg.lg;
  // slots before the piece that hold no record
  uint32_t lack = 0;
  if (IN == IN_LIST && lacks) {
    uint32_t t = 0;
    for (uint32_t p = threadIdx.x; p < blockIdx.x + seg; p += SORT_THREADS) t += lacks[p];
    block_scan_round(t, wtot, 0, lack);
    __syncthreads();  // wtot is written again
  }
  // the piece's blocks
  uint32_t blk0 = PAGED ? (uint32_t)((cb - lack) >> pg.lg) + (blockIdx.x + seg) * (uint32_t)(nb + 1) : 0u;
  uint32_t taken = 0;                                                                      // blocks taken so far
  for (int i = threadIdx.x; i < nb; i += SORT_THREADS) {
    if constexpr (PAGED) dcnt[i] = 0;
    else dinfo[i].y = offsets[(int64_t)i * gridDim.x + blockIdx.x];
  }
  for (int i = threadIdx.x; i < NBUF * hw * nbt; i += SORT_THREADS) whist_all[i] = 0;
  const int row = (wave % hw) * nbt;
  if (threadIdx.x == 0) {
    smr[0] = 0u;
    smr[1] = 0xffffffffu;
  }
  uint32_t mx = 0u, mn = 0xffffffffu;

  float rec[PL][RW] = {};
  uint32_t vm = 0;  // bit it: this lane's slot `it` of the sub-chunk holds a record
  const int wbase = wave * (PL * 64) + lane;
  // IN_LIST: blocks hold at least 64 slots and sub-chunks start at multiples
  // of 64, so 64 consecutive slots lie in one block: the block is looked up
  // once per wave and `it`, with scalar loads
  uint32_t wslot[IN == IN_LIST ? PL : 1];  // pool slot of the wave's first slot `it`
  // records of the sub-chunk at s0 of a piece that ends at `end`
  auto load_sub = [&](int64_t s0, int64_t end) {
    if constexpr (IN == IN_LIST) {
      const int64_t w0 = s0 + __builtin_amdgcn_readfirstlane(wave) * (PL * 64);
      const uint32_t ibm = (1u << im.lg) - 1;
      uint32_t ent[PL];
#pragma unroll
      for (int it = 0; it < PL; it++) ent[it] = w0 + it * 64 < end ? blist[(w0 + it * 64) >> im.lg] : 0u;
      vm = 0;
#pragma unroll
      for (int it = 0; it < PL; it++) {
        const uint32_t in = (uint32_t)(w0 + it * 64) & ibm;  // slot within the block
        const uint32_t fill = w0 + it * 64 < end ? (ent[it] >> (32 - im.lg)) + 1 : 0u;
        wslot[it] = (ent[it] << im.lg) + in;
        if (in + lane < fill) {
          vm |= 1u << it;
          src.load((int64_t)(wslot[it] + lane), rec[it]);
        }
      }
    } else {
      const int64_t i0 = s0 + wbase;
      const int64_t lim = end - i0;  // slot i0 + 64 it holds a record iff 64 it < lim
      const uint32_t nv = lim <= 0 ? 0u : (uint32_t)min((int64_t)PL, (lim + 63) >> 6);
      vm = (1u << nv) - 1;
#pragma unroll
      for (int it = 0; it < PL; it++)
        if ((uint32_t)it < nv) src.load(i0 + it * 64, rec[it]);
    }
  };
  load_sub(cb, pe);
  // nothing in flight on entry to the loop, so that the wait for a
  // sub-chunk's records there is not a wait for the write-out's stores
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  int sub = 0;
  for (int64_t s0 = cb; s0 < ce; sub++) {
    // the next sub-chunk: of this piece, or the next piece's first
    const bool last = s0 + SUBN >= pe;  // of the piece
    const int64_t s1 = last ? pe : s0 + SUBN;
    uint32_t nseg = seg;
    int64_t npe = pe;
    if (IN != IN_RAW && last && s1 < ce) {
      do npe = (int64_t)start[++nseg + 1] << sh;
      while (npe == s1);  // empty buckets
      npe = min(npe, ce);
    }
    uint32_t *whist = whist_all + (DB ? (sub & 1) * hw * nbt : 0);
    uint32_t pk[PL];
    rank_records<NM, PL>(rec, vm, kg, ds, (uint32_t)nb, whist + row, pk);
    __syncthreads();
    uint32_t total = 0;  // records of this sub-chunk (PAGED: and blocks taken << 16)
    if (threadIdx.x == SORT_THREADS - 1) wave_offsets(whist, nbt, hw, nb);
    for (int r0 = 0, rd = 0; r0 < nb; r0 += SORT_THREADS, rd++) {
      const int dg = r0 + threadIdx.x;
      const uint32_t tot = dg < nb ? wave_offsets(whist, nbt, hw, dg) : 0u;
      if constexpr (PAGED) {
        // the run fills the open block (a records), then `need` new blocks;
        // counts and block numbers scan together (at most SUBN slots and
        // SUBN / 8 + nb blocks)
        const uint32_t c0 = dg < nb ? dcnt[dg] : 0u;
        const uint32_t f = c0 & (pb - 1);
        const uint32_t a = f ? min(tot, pb - f) : 0u;
        const uint32_t need = (tot - a + pb - 1) >> pg.lg;
        const uint32_t run = block_scan_round(tot | need << 16, wtot, rd, total);
        if (dg < nb) {
          const uint32_t lr = run & 0xffffu, first = blk0 + taken + (run >> 16);
          // the first part is used only when a > 0, i.e. the block is open
          dinfo[dg] = make_uint4(lr, lr + a, ((f ? dblk[dg] : 0u) << pg.lg) + f - lr, (first << pg.lg) - (lr + a));
          if (need) dblk[dg] = first + need - 1;
          dcnt[dg] = c0 + tot;
        }
      } else {
        const uint32_t run = block_scan_round(tot, wtot, rd, total);
        if (dg < nb) {
          const uint32_t g = dinfo[dg].y;
          dinfo[dg].x = run;
          dinfo[dg].y = g + tot;
          dinfo[dg].z = g - run;
        }
      }
    }
    const uint32_t nrec = PAGED ? total & 0xffffu : total;  // staging positions [0, nrec) hold records
    if constexpr (PAGED) taken += total >> 16;
    if (threadIdx.x == SORT_THREADS - 1) dinfo[nb].x = nrec;
    __syncthreads();
    // output position of the record at staging position p of digit d
    auto dest_of = [&](uint32_t p, uint32_t d) -> uint32_t {
      if constexpr (PAGED) {
        const uint4 di = dinfo[d];
        return p < di.y ? di.z + p : di.w + p;
      } else {
        return dinfo[d].z + p;
      }
    };
#pragma unroll
    for (int it = 0; it < PL; it++) {
      const int loc = wbase + it * 64;
      const uint32_t dg = pk[it] >> 13;
      const uint32_t p = dinfo[dg].x + whist[row + dg] + (pk[it] & 0x1fffu);
#pragma unroll
      for (int k = 0; k < RW; k++) stage[p * RW + k] = rec[it][k];
      sdig[p] = (uint16_t)dg;
      if ((vm >> it) & 1u) {
        if constexpr (NM == 1) {
          // |mass| as bits orders like the value (a NaN above every finite one)
          const uint32_t mb = __float_as_uint(rec[it][3]) & 0x7fffffffu;
          mx = max(mx, mb);
          if (mb) mn = min(mn, mb);
        }
        // where this record goes (coalesced writes, by input position or pool slot)
        if constexpr (PERM)
          perm[IN == IN_LIST ? (int64_t)(wslot[IN == IN_LIST ? it : 0] + lane) : s0 + loc] = dest_of(p, dg);
      }
    }
    // the next sub-chunk loads during the barrier and the write-out
    load_sub(s1, npe);
    __syncthreads();
    auto put = [&](int p) {
      const uint32_t sd = sdig[p], dest = dest_of((uint32_t)p, sd);
      // a block's first record names its digit (one thread per digit naming
      // all its new blocks was a serial loop of up to 512 stores where a
      // sub-chunk's records share few digits: 57 -> 32 us for 1.2e6 clumped
      // records in 637 tiles)
      if (PAGED && (dest & (pb - 1)) == 0) pg.hdr[dest >> pg.lg] = (uint16_t)sd;
      float v[RW];
#pragma unroll
      for (int k = 0; k < RW; k++) v[k] = stage[p * RW + k];
#pragma unroll
      for (int k = 0; k < RW; k++) dst[(int64_t)dest * RW + k] = v[k];
    };
    // four stores in flight per lane (all eight cost pass 2 6.5 -> 7.0 ms at
    // 2^30 records: registers); the last sub-chunk may be partial
    if (nrec == SUBN) {
#pragma unroll PAGED ? 4 : PL
      for (int it = 0; it < PL; it++) put(threadIdx.x + it * SORT_THREADS);
    } else {
      for (int p = threadIdx.x; p < (int)nrec; p += SORT_THREADS) put(p);
    }
    for (int i = threadIdx.x; i < hw * nbt; i += SORT_THREADS) whist[i] = 0;
    if (PAGED && last) {
      // the piece's totals (each digit's state is its own thread's)
      const uint32_t p = blockIdx.x + seg;
      for (int dg = threadIdx.x; dg < nb; dg += SORT_THREADS) {
        const uint32_t c = dcnt[dg];
        if (c == 0) continue;
        dcnt[dg] = 0;
        const unsigned long long add = (unsigned long long)((c + pb - 1) >> pg.lg) << 32 | c;
        const int64_t at = (int64_t)p * nb + dg;
        pg.cnt[at] = c;
        pg.last[at] = dblk[dg];
        pg.base[at] = (uint32_t)(atomicAdd(&pg.tot[(int64_t)seg * nb + dg], add) >> 32);
      }
      if (threadIdx.x == 0) pg.piece[p] = make_uint4(blk0, taken, seg, 0u);
      if (IN == IN_LIST && lacks) lack += lacks[p];
      blk0 = (uint32_t)((s1 - lack) >> pg.lg) + (blockIdx.x + nseg) * (uint32_t)(nb + 1);
      taken = 0;
    }
    s0 = s1;
    seg = nseg;
    pe = npe;
    if (!DB) __syncthreads();
  }
  if constexpr (NM == 1) {
    if (mrange_w) {
      atomicMax(&smr[0], mx);
      atomicMin(&smr[1], mn);
      __syncthreads();
      if (threadIdx.x < 2) mrange_w[2 * (int64_t)blockIdx.x + threadIdx.x] = smr[threadIdx.x];
    }
  }
}

// Bucket totals of a counted first pass, from its scanned table: records in
// both halves (one record per list entry).
__global__ void k_seg_tot(const uint32_t *__restrict__ t1scan, int64_t g1, int nseg, int64_t n,
                          unsigned long long *__restrict__ tot) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const uint32_t st = t1scan[(int64_t)s * g1];
  const uint32_t en = (s + 1 < nseg) ? t1scan[(int64_t)(s + 1) * g1] : (uint32_t)n;
  tot[s] = (unsigned long long)(en - st) << 32 | (en - st);
}

// Directory of the buckets of a pass, from their totals (list entries << 32
// | records): every bucket's first list entry; of the segments of a second
// pass, the bucket of each workgroup's first slot; of tiles, the work items,
// the table of the items and the deposit's schedule.  The totals are cleared
// for the next sort.
//
// Up to DIR_ONE buckets one workgroup does it all (k_dir; the scans, tables and
// flags that it replaces were a dozen launches of 2 to 5 us each).  It takes
// 6.5 us per round of 4096 buckets, so more of them are cut into sections, a
// workgroup each: k_dir_sums (a section's sums), k_dir (each section from the
// sums of those before it) and k_dir_end (split items, shares).  With the
// lists 105 -> 23 us at 65 536 tiles, 359 -> 27 at 2^18, 2990 -> 47 at 2^21
// (2^20 particles or fewer); 16384 buckets 30 -> 21.
//
// Schedule: the deposit's workgroup w takes the items w, w + wgs, ... of split
// tiles, then a run of the items of one tile, whose bounds share every
// workgroup the same cost in all (an item costs its record slots and icost).
// Without split tiles no tile is heavy and the items are strided over the
// workgroups (shared by cost they took 5 us more here and gained nothing:
// 13.8e6 lattice particles at 360^3).  With
// all items strided over the workgroups the one with the most heavy tiles held
// 1.5 to 2 times the mean of clumped particles: deposit 0.221 -> 0.173 ms for
// 2e7 at 384^3, 0.83 -> 0.55 for 1e8 at 512^3, 5.70 -> 5.12 for 2^30 at 1024^3.
// Heavy items first also end the adjoint gather, whose items the hardware
// hands out in order, more evenly: 0.826 -> 0.78 ms at 512^3.
struct DirArgs {
  unsigned long long *tot;
  int64_t nb, kreal;      // buckets; those below kreal are real tiles
  uint32_t *start;        // [nb + 1]
  uint32_t *first_seg;    // segments: the bucket of each workgroup's first slot
  uint4 *items;           // tiles: TileList::items
  uint32_t unit;          // segments: list entries per workgroup (0: tiles)
  FastDiv funit;
  uint4 *piece;           // segments: the second pass's pieces and their lacks, cleared
  uint32_t *lacks;
  int64_t npiece;
  // tiles: items of at most 2^limax records and 2^17 record slots; store: every
  // real tile gets at least one item (so untouched tiles are written as zeros)
  int store, lg, limax;
  // [nb + 1]; split tiles; TileList (counts[3]: cost of the items of one tile)
  uint32_t *pstart, *heavy, *counts, *cost, *share;
  uint32_t max_parts, wgs, icost;
  FastDiv fwgs;
  int cshift;  // costs are in units of 2^cshift records, so that their sum stays below 2^31
  uint32_t *nonfinite;
  uint32_t *mrange;       // with masses: reduced from mrange_w[2 * nw]
  const uint32_t *mrange_w;
  int64_t nw;
  int64_t sec;            // buckets of a workgroup's section (whole rounds)
  uint4 *secsum;          // [sections] (one section: none)
};
constexpr int DIR_PER = 4;  // buckets per thread and round
constexpr int64_t DIR_ROUND = (int64_t)SORT_THREADS * DIR_PER;
constexpr int64_t DIR_ONE = 2 * DIR_ROUND;
constexpr uint32_t DIR_HEAVY = 1024;  // split tiles that one workgroup keeps in LDS
constexpr int DIR_NV = 4;  // prefix sums: list entries, items of one tile, items of split tiles, cost of the former

// Entries and items of bucket k with totals t: v as in DIR_NV, but for v[3],
// the cost of an item (also of a split tile).
__device__ __forceinline__ void dir_values(const DirArgs &D, int64_t k, unsigned long long t, uint32_t (&v)[DIR_NV]) {
  const uint32_t eslots = 1u << (LG_ITEM_MAX - D.lg);  // list entries of 2^17 record slots
  const uint32_t ents = (uint32_t)(t >> 32), recs = (uint32_t)t;
  uint32_t m = 0;
  if (D.unit == 0 && k < D.kreal) {
    if (recs == 0) m = D.store ? 1u : 0u;
    else m = max((recs + (1u << D.limax) - 1) >> D.limax, (ents + (eslots - 1)) >> (LG_ITEM_MAX - D.lg));
  }
  v[0] = ents;
  v[1] = m == 1 ? 1u : 0u;
  v[2] = m > 1 ? m : 0u;
  const uint32_t slots = (ents << D.lg) >> D.cshift;
  v[3] = m == 0 ? 0u : (m > 1 ? slots / m : slots) + D.icost;
}

__global__ void __launch_bounds__(SORT_THREADS) k_dir_sums(DirArgs D) {
  __shared__ uint32_t wt[DIR_NV][SORT_WAVES];
  const int64_t b0 = blockIdx.x * D.sec, b1 = min(D.nb, b0 + D.sec);
  uint32_t sum[DIR_NV] = {};
  for (int64_t k = b0 + threadIdx.x; k < b1; k += SORT_THREADS) {
    uint32_t v[DIR_NV];
    dir_values(D, k, D.tot[k], v);
#pragma unroll
    for (int j = 0; j < DIR_NV; j++) sum[j] += j == 3 && v[2] ? 0u : v[j];
  }
#pragma unroll
  for (int j = 0; j < DIR_NV; j++) {
    const uint32_t incl = wave_incl_scan(sum[j]);
    if ((threadIdx.x & 63) == 63) wt[j][threadIdx.x >> 6] = incl;
  }
  __syncthreads();
  uint32_t all[DIR_NV];
#pragma unroll
  for (int j = 0; j < DIR_NV; j++) waves_before(wt[j], all[j]);
  if (threadIdx.x == 0) {
    D.secsum[blockIdx.x] = make_uint4(all[0], all[1], all[2], all[3]);
    if (blockIdx.x == 0) D.counts[0] = 0;
  }
}

// The split tiles' items, numbered from pstart on, the deposit's shares and the
// masses' range, by one workgroup, once every bucket's start and the nheavy
// split tiles are written; the first nknown of them also stand in known (tile,
// first item, items, cost of one) and known_at (list entries), which saves two
// round trips to memory.
// carry: the sums of all buckets.
__device__ __forceinline__ void dir_end(const DirArgs &D, uint32_t nheavy, const uint4 *known, const uint2 *known_at,
                                        uint32_t nknown, const uint32_t (&carry)[DIR_NV]) {
  __shared__ uint32_t wtot[2][SORT_WAVES];
  __shared__ uint32_t load_of[DEPOSIT_WGS_MAX];  // cost of each workgroup's items of split tiles
  __shared__ uint32_t smr[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  load_of[threadIdx.x] = 0;
  static_assert(DEPOSIT_WGS_MAX == SORT_THREADS, "one thread per workgroup of the deposit");
  if (threadIdx.x == 0) {
    smr[0] = 0u;
    smr[1] = 0xffffffffu;
  }
  __syncthreads();
  // every wave reads up to 64 split tiles at once (each wave's SORT_WAVES
  // apart, so that few tiles spread over the waves), then writes the items of
  // one after another (one thread per tile was a chain of up to hundreds of stores)
  for (uint32_t h0 = wave; h0 < nheavy; h0 += SORT_THREADS) {
    const uint32_t h = h0 + lane * SORT_WAVES;
    uint4 t = make_uint4(0u, 0u, 0u, 0u);
    uint2 at = make_uint2(0u, 0u);
    if (h < nknown) {
      t = known[h];
      at = known_at[h];
    } else if (h < nheavy) {
      t.x = D.heavy[h];
      t.y = D.pstart[t.x];
      t.z = D.pstart[t.x + 1] - t.y;
      at = make_uint2(D.start[t.x], D.start[t.x + 1]);
      t.w = (((at.y - at.x) << D.lg) >> D.cshift) / t.z + D.icost;
    }
    const uint32_t entries = t.z ? (at.y - at.x + t.z - 1) / t.z : 0u;  // of an item
    for (int i = 0; i < 64 && h0 + i * SORT_WAVES < nheavy; i++) {
      const uint32_t k = __builtin_amdgcn_readlane(t.x, i), p0 = __builtin_amdgcn_readlane(t.y, i);
      const uint32_t m = __builtin_amdgcn_readlane(t.z, i), c = __builtin_amdgcn_readlane(t.w, i);
      const uint32_t lb = __builtin_amdgcn_readlane(at.x, i), le = __builtin_amdgcn_readlane(at.y, i);
      const uint32_t per = __builtin_amdgcn_readlane(entries, i);
      for (uint32_t j = lane; j < m; j += 64) {
        const uint32_t q = p0 + j, b = min(le, lb + j * per);
        D.items[q] = make_uint4(k, b, min(le, b + per), 0u);
        atomicAdd(&load_of[q - D.fwgs.div(q) * D.wgs], c);
      }
    }
  }
  if (carry[2] && carry[1] + carry[2] > D.wgs) {
    // what each workgroup has left to the mean of all, in proportion of the
    // cost of the items of one tile (fewer items: one each, k_deposit)
    __syncthreads();
    const uint32_t own = threadIdx.x < D.wgs ? load_of[threadIdx.x] : 0u;
    uint32_t all = 0, rest = 0;
    block_scan_round(own, wtot, 0, all);
    const uint32_t mean = (uint32_t)(((unsigned long long)all + carry[3] + D.wgs - 1) / D.wgs);
    const uint32_t before = block_scan_round(threadIdx.x < D.wgs && mean > own ? mean - own : 0u, wtot, 1, rest);
    if (threadIdx.x < D.wgs) D.share[threadIdx.x] = (uint32_t)((double)carry[3] * before / max(rest, 1u));
  }
  if (D.mrange) {
    uint32_t mx = 0u, mn = 0xffffffffu;
    for (int64_t i = threadIdx.x; i < D.nw; i += SORT_THREADS) {
      mx = max(mx, D.mrange_w[2 * i]);
      mn = min(mn, D.mrange_w[2 * i + 1]);
    }
    atomicMax(&smr[0], mx);
    atomicMin(&smr[1], mn);
    __syncthreads();
    if (threadIdx.x < 2) D.mrange[threadIdx.x] = smr[threadIdx.x];
  }
}

__global__ void __launch_bounds__(SORT_THREADS) k_dir_end(DirArgs D) {
  const uint32_t carry[DIR_NV] = {0u, D.counts[2], D.counts[1], D.counts[3]};
  dir_end(D, D.counts[0], nullptr, nullptr, 0u, carry);
}

template <bool ONE>
__global__ void __launch_bounds__(SORT_THREADS) k_dir(DirArgs D) {
  constexpr int NV = DIR_NV;
  __shared__ uint32_t wt[2][NV][SORT_WAVES];
  __shared__ uint4 split_tiles[ONE ? DIR_HEAVY : 1];  // as dir_end's known and known_at
  __shared__ uint2 split_at[ONE ? DIR_HEAVY : 1];
  __shared__ uint32_t hcount;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t b0 = ONE ? 0 : blockIdx.x * D.sec, b1 = ONE ? D.nb : min(D.nb, b0 + D.sec);
  if (threadIdx.x == 0) {
    hcount = 0;
    if (D.nonfinite && blockIdx.x == 0) *D.nonfinite = 0u;
  }
  unsigned long long t[DIR_PER];
  auto load = [&](int64_t r0) {
#pragma unroll
    for (int i = 0; i < DIR_PER; i++) {
      const int64_t k = r0 + threadIdx.x * DIR_PER + i;
      t[i] = k < b1 ? D.tot[k] : 0ull;
    }
  };
  load(b0);
  uint32_t carry[NV] = {};
  if constexpr (!ONE) {
    uint32_t sum[NV] = {};
    for (uint32_t w = threadIdx.x; w < blockIdx.x; w += SORT_THREADS) {
      const uint4 s = D.secsum[w];
      sum[0] += s.x;
      sum[1] += s.y;
      sum[2] += s.z;
      sum[3] += s.w;
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const uint32_t incl = wave_incl_scan(sum[j]);
      if (lane == 63) wt[1][j][wave] = incl;  // (the first round writes wt[0])
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; j++) waves_before(wt[1][j], carry[j]);
  }
  auto div_up = [&](uint32_t x) { return x == 0 ? 0u : D.funit.div(x - 1) + 1; };  // entries < 2^31
  int rd = 0;
  for (int64_t r0 = b0; r0 < b1; r0 += DIR_ROUND, rd ^= 1) {
    const int64_t k0 = r0 + threadIdx.x * DIR_PER;
    uint32_t v[DIR_PER][NV], sum[NV] = {};
#pragma unroll
    for (int i = 0; i < DIR_PER; i++) {
      dir_values(D, k0 + i, t[i], v[i]);
      if (k0 + i < b1) D.tot[k0 + i] = 0ull;
#pragma unroll
      for (int j = 0; j < NV; j++) sum[j] += j == 3 && v[i][2] ? 0u : v[i][j];
    }
    load(r0 + DIR_ROUND);
    uint32_t run[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const uint32_t incl = wave_incl_scan(sum[j]);
      run[j] = carry[j] + incl - sum[j];
      if (lane == 63) wt[rd][j][wave] = incl;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; j++) {
      uint32_t all;
      run[j] += waves_before(wt[rd][j], all);
      carry[j] += all;
    }
#pragma unroll
    for (int i = 0; i < DIR_PER; i++) {
      const int64_t k = k0 + i;
      if (k < b1) {
        D.start[k] = run[0];
        if (D.unit) {
          // the workgroups whose first entry lies in this bucket
          const uint32_t w1 = div_up(run[0] + v[i][0]);
          for (uint32_t w = div_up(run[0]); w < w1; w++) D.first_seg[w] = (uint32_t)k;
        } else {
          D.pstart[k] = run[2];
          if (v[i][1]) {
            D.items[D.max_parts + run[1]] = make_uint4((uint32_t)k, run[0], run[0] + v[i][0], 0u);
            D.cost[run[1]] = run[3] + v[i][3] / 2;
          } else if (v[i][2]) {
            const uint32_t h = atomicAdd(ONE ? &hcount : &D.counts[0], 1u);
            D.heavy[h] = (uint32_t)k;
            if (ONE && h < DIR_HEAVY) {
              split_tiles[h] = make_uint4((uint32_t)k, run[2], v[i][2], v[i][3]);
              split_at[h] = make_uint2(run[0], run[0] + v[i][0]);
            }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < NV; j++) run[j] += j == 3 && v[i][2] ? 0u : v[i][j];
    }
  }
  for (int64_t i = threadIdx.x; i < D.npiece; i += SORT_THREADS) {
    D.piece[i] = make_uint4(0u, 0u, 0u, 0u);
    D.lacks[i] = 0u;
  }
  if (b1 == D.nb && threadIdx.x == 0) {
    D.start[D.nb] = carry[0];
    if (!D.unit) {
      D.pstart[D.nb] = carry[2];
      D.counts[1] = carry[2];
      D.counts[2] = carry[1];
      D.counts[3] = carry[3];
    }
  }
  if (ONE && !D.unit) {
    if (carry[2] || D.mrange) {
      // beyond split_tiles, dir_end reads what other waves of this workgroup
      // have written (a fence among workgroups would write the L2 back: 4 us)
      __threadfence_block();
      __syncthreads();
      dir_end(D, hcount, split_tiles, split_at, min(hcount, (uint32_t)DIR_HEAVY), carry);
    }
    if (threadIdx.x == 0) D.counts[0] = carry[2] ? hcount : 0u;
  }
}

// The block list: bucket k's blocks from list entry start[k] on, each piece's
// of a digit side by side in any order.  One workgroup per piece.
__global__ void __launch_bounds__(SORT_THREADS) k_list(PgOut pg, int nb, const uint32_t *__restrict__ start,
                                                       uint32_t *__restrict__ blist) {
  extern __shared__ uint32_t lcnt[];  // [nb]
  const int64_t p = blockIdx.x;
  const uint4 pc = pg.piece[p];
  if (pc.y == 0) return;
  for (int i = threadIdx.x; i < nb; i += SORT_THREADS) lcnt[i] = 0;
  __syncthreads();
  const int64_t bucket0 = (int64_t)pc.z * nb;
  for (uint32_t k = threadIdx.x; k < pc.y; k += SORT_THREADS) {
    const uint32_t blk = pc.x + k, d = pg.hdr[blk];
    const int64_t at = p * nb + d;
    const uint32_t part = pg.cnt[at] & ((1u << pg.lg) - 1);
    const uint32_t fill = part && blk == pg.last[at] ? part : 1u << pg.lg;
    blist[start[bucket0 + d] + pg.base[at] + atomicAdd(&lcnt[d], 1u)] = pg_entry(blk, fill, pg.lg);
  }
}

// lacks[w + s]: the empty slots of the listed blocks of piece w + s of a second
// pass, whose workgroup w takes entries [w * unit, (w + 1) * unit).  One
// workgroup each.  (Added up with global atomics where the list is written it
// took 13 us at 2^27 records instead of 2.5.)
constexpr int LACK_THREADS = 256;
__global__ void __launch_bounds__(LACK_THREADS) k_lacks(const uint32_t *__restrict__ blist,
                                                        const uint32_t *__restrict__ start,
                                                        const uint32_t *__restrict__ first_seg, int nseg, int lg,
                                                        uint32_t unit, uint32_t *__restrict__ lacks) {
  __shared__ uint32_t part[2][LACK_THREADS / 64];
  const uint32_t e0 = blockIdx.x * unit, e1 = min(start[nseg], e0 + unit);
  if (e0 >= e1) return;
  uint32_t s = first_seg[blockIdx.x];
  for (uint32_t lo = e0, rd = 0; lo < e1; rd ^= 1) {
    const uint32_t hi = min(e1, start[s + 1]);
    uint32_t t = 0;
    for (uint32_t e = lo + threadIdx.x; e < hi; e += LACK_THREADS) t += (1u << lg) - ((blist[e] >> (32 - lg)) + 1);
    t = wave_incl_scan(t);
    if ((threadIdx.x & 63) == 63) part[rd][threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0 && lo < hi) lacks[blockIdx.x + s] = part[rd][0] + part[rd][1] + part[rd][2] + part[rd][3];
    lo = hi;
    s++;
  }
}

struct PtShape {
  int pl;
  bool db;
  int hw;
};

// LDS of a partition shape (nb digits and the empty slots' digit); a paged
// pass keeps two more arrays per digit.
size_t partition_lds(int nb, int rw, const PtShape &h, bool paged) {
  const size_t sub = (size_t)SORT_THREADS * h.pl, nbt = (size_t)nb + 1;
  return ((4 + (h.db ? 2 : 1) * h.hw) * nbt + (paged ? 2 * (size_t)nb : 0)) * 4 + sub * 2 + sub * rw * 4;
}

// The first shape whose LDS fits one workgroup per CU: four count rows (each
// shared by four waves: 16 rows measured 0.1 ms slower per pass at 2^30
// records, the per-digit offsets running over more rows), then the most
// records per lane (at most plmax), then double-buffered counts.
PtShape partition_shape(int nb, int rw, bool paged, int plmax) {
  const size_t cap = 160 * 1024 - 512;
  for (int hw : {SORT_WAVES / 4, 1})
    for (int pl : {8, 4, 2})
      for (bool db : {true, false}) {
        const PtShape h{pl, db, hw};
        if (pl <= plmax && !(pl == 2 && db) && partition_lds(nb, rw, h, paged) <= cap) return h;
      }
  return PtShape{2, false, 1};
}

// Records per lane and sub-chunk of a pass over n records: fewer for small
// sets, so that they spread over the CUs.
int partition_plmax(int64_t n) {
  const int64_t per = n / (2 * (int64_t)num_cus());
  return per <= 2 * SORT_THREADS ? 2 : per <= 4 * SORT_THREADS ? 4 : 8;
}

// Arguments of a partition pass: what it reads (the caller's arrays, or a first
// pass's records with their bucket starts and, paged, their block list), what
// it writes, and of a counted pass the scanned offsets, of a paged one the pool.
struct PtArgs {
  const float *pos = nullptr, *masses = nullptr;
  const uint32_t *blist = nullptr, *start = nullptr, *first_seg = nullptr, *lacks = nullptr;
  InMap im;
  int64_t grid = 0;
  DigitSel ds;
  int nb = 0;
  PtShape h;
  float *dst = nullptr;
  uint32_t *perm = nullptr, *mrange_w = nullptr;
  const uint32_t *offsets = nullptr;
  PgOut pg;
};

template <int NM, int IN, bool PAGED, bool PERM>
void launch_partition_perm(const PtArgs &A, const KeyGeom &kg, hipStream_t s) {
  GENPK_REQUIRE(A.nb <= 2048, "sort digit too wide");
  const size_t lds = partition_lds(A.nb, Src<NM>::RW, A.h, PAGED);
  GENPK_REQUIRE(lds <= 160 * 1024 - 512, "sort pass does not fit in LDS");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)A.grid), dim3(SORT_THREADS), lds, s, A.pos, A.masses, A.blist, A.start,
                       A.first_seg, A.lacks, A.dst, A.im, kg, A.ds, A.nb, A.h.hw, A.offsets, A.perm, A.mrange_w, A.pg);
  };
  if (A.h.pl == 8 && A.h.db) go(k_partition<NM, 8, true, IN, PAGED, PERM>);
  else if (A.h.pl == 8) go(k_partition<NM, 8, false, IN, PAGED, PERM>);
  else if (A.h.pl == 4 && A.h.db) go(k_partition<NM, 4, true, IN, PAGED, PERM>);
  else if (A.h.pl == 4) go(k_partition<NM, 4, false, IN, PAGED, PERM>);
  else go(k_partition<NM, 2, false, IN, PAGED, PERM>);
  GENPK_LAUNCH_CHECK();
}

template <int NM, int IN, bool PAGED>
void launch_partition(const PtArgs &A, const KeyGeom &kg, hipStream_t s) {
  if (A.perm) launch_partition_perm<NM, IN, PAGED, true>(A, kg, s);
  else launch_partition_perm<NM, IN, PAGED, false>(A, kg, s);
}

// log2 of a paged pass's block: a quarter to a half of the records that a
// piece holds of a digit on average.  Longer blocks write faster (2^30
// records: pass 2 7.1, 6.8, 6.5 ms with an eighth to a sixteenth, a quarter
// to an eighth, and this), shorter ones leave fewer slots empty.
int pick_lg(int64_t recs, int64_t nb, int lo, int hi) {
  int lg = 0;
  while (((int64_t)2 << (lg + 1)) * nb <= recs) lg++;
  return std::min(std::max(lg, lo), hi);
}

// Shape of a paged pass: G workgroups of `chunk` input slots each, and the
// pool of its pieces' blocks of 2^lg record slots.
struct PgLayout {
  PtShape h;
  int64_t G = 0, chunk = 0, pieces = 0, blocks = 0;
  int lg = 0;
  int64_t slots() const { return blocks << lg; }
};

// A paged pass of n records (or, for the pool, as many as the input's slots) in
// at most `slots` input slots (in blocks of 2^inlg) of nseg buckets.  Every workgroup takes the same number of slots: one round of one
// workgroup per CU, or more rounds as long as each workgroup keeps minsub
// sub-chunks and the partly filled blocks (one per piece and digit at most)
// stay below a sixth of the records (or 2^26: about 1 GB).  Shorter ranges run
// beside each other in time on neighbouring parts of the pools, and finish
// evenly: with two rounds instead of eight the first pass takes 0.80 instead
// of 0.74 ms (2^27 records, 64 digits), with two instead of 16 the second 7.2
// instead of 6.5 ms (2^30 records).  Few slots in many buckets are cut below a
// sub-chunk, down to a workgroup per bucket: a piece takes 2.5 us whatever it
// holds, and one workgroup that walked all of them 624 us (1000
// records in 256 buckets; 13 spread out).
PgLayout paged_layout(int64_t n, int64_t slots, int64_t nseg, int nb, int rw, int lo, int hi, int minsub,
                      int inlg = 0) {
  PgLayout L;
  L.h = partition_shape(nb, rw, true, partition_plmax(slots));
  const int64_t subn = (int64_t)SORT_THREADS * L.h.pl, cus = num_cus();
  for (int64_t rounds = 1; rounds <= 16; rounds *= 2) {
    PgLayout M = L;
    M.chunk = std::max(subn, ceil_div(ceil_div(slots, rounds * cus), subn) * subn);
    if (nseg > 1 && M.chunk == subn)
      M.chunk = std::min(subn, std::max((int64_t)1, ceil_div(slots >> inlg, std::min(nseg, cus))) << inlg);
    M.G = ceil_div(slots, M.chunk);
    M.pieces = nseg > 1 ? M.G + nseg : M.G;
    M.lg = pick_lg(slots / M.pieces, nb, lo, hi);
    const int64_t partial = M.pieces * (nb + 1), most = std::max(n / 6, (int64_t)1 << 26);
    while (rounds == 1 && M.lg > lo && (partial << M.lg) > most) M.lg--;  // (2^22 tiles, 2^31 records)
    M.blocks = (n >> M.lg) + partial + 1;
    if (rounds > 1 && (M.chunk < minsub * subn || (partial << M.lg) > most)) break;
    L = M;
  }
  return L;
}

// Whether the first of two passes is paged (of 2^hi_bits digits): each
// workgroup has to hold many records of a digit.  With 256 digits (32769 to
// 65536 tiles) the counted pass keeps sorts below 2^29 records, against which
// the tests check the paged one.  That costs up to 15% of the sort: at 1024^3
// FP32 both take 0.20 ms at 2^23 records, paged and counted 0.32 and 0.33 (uniform
// and clumped 0.32 and 0.34) at 2^24, 0.58 and 0.61 at 2^25, 1.00 and 1.13 at 2^26,
// 3.58 and 4.19 at 2^28.
bool first_paged(const Plan &p, int64_t n) {
  const int64_t nhi = (int64_t)1 << p.tg.hi_bits, cus = num_cus();
  if (nhi > 256) return false;
  if (nhi == 256) return 2 * cus * nhi * 1024 <= n / 4;
  return n >= cus * nhi * 128;
}

// Workspace of a paged pass in one buffer: pieces, per-piece counts, last
// blocks and bases, the block list, the blocks' digits and the
// pieces' lacks.
uint32_t *pg_buffers(DevBuf &buf, const PgLayout &L, int nb, PgOut &pg, unsigned long long *tot, uint32_t **lacks) {
  const size_t blocks = (size_t)L.blocks, wd = (size_t)L.pieces * nb;
  GENPK_REQUIRE((uint64_t)L.slots() <= ((uint64_t)1 << 32), "sort pool too large");
  uint32_t *b = static_cast<uint32_t *>(buf.ensure((5 * (size_t)L.pieces + 3 * wd + blocks + (blocks + 1) / 2) * 4));
  pg.piece = reinterpret_cast<uint4 *>(b);
  *lacks = b + 4 * L.pieces;
  pg.cnt = b + 5 * L.pieces;
  pg.last = pg.cnt + wd;
  pg.base = pg.last + wd;
  uint32_t *blist = pg.base + wd;
  pg.hdr = reinterpret_cast<uint16_t *>(blist + blocks);
  pg.tot = tot;
  pg.lg = L.lg;
  return blist;
}

// Sections of a directory of nb buckets (k_dir): a workgroup each, at most 1024.
int64_t dir_section(int64_t nb) {
  if (nb <= DIR_ONE) return ceil_div(nb, DIR_ROUND) * DIR_ROUND;
  return ceil_div(ceil_div(nb, DIR_ROUND), SORT_THREADS) * DIR_ROUND;
}

void launch_dir(DirArgs &D, hipStream_t s) {
  D.sec = dir_section(D.nb);
  const dim3 grid((unsigned)ceil_div(D.nb, D.sec)), block(SORT_THREADS);
  GENPK_REQUIRE(grid.x == 1 || (!D.unit && D.secsum), "directory of segments in sections");
  if (grid.x == 1) {
    hipLaunchKernelGGL(k_dir<true>, grid, block, 0, s, D);
    GENPK_LAUNCH_CHECK();
    return;
  }
  hipLaunchKernelGGL(k_dir_sums, grid, block, 0, s, D);
  GENPK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_dir<false>, grid, block, 0, s, D);
  GENPK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_dir_end, dim3(1), block, 0, s, D);
  GENPK_LAUNCH_CHECK();
}

// Counted first pass: chunk size and count.
int64_t counted_chunk(int64_t n) {
  int64_t chunk = SORT_CHUNK_MIN;
  while (chunk < SORT_CHUNK_MAX && chunk * 4 * num_cus() < n) chunk *= 2;
  return chunk;
}

struct SortLayout {
  bool two = false, paged1 = false;
  PgLayout L1, L2;  // paged first pass (of two), last pass
  int64_t slots1 = 0;  // slots that a first pass of two writes
  bool lacks = false;  // the last pass's pool is sized from the records (k_lacks), not from those slots
  uint32_t imax = 0;   // records of a work item at most
  int64_t max_parts = 0;  // items of split tiles at most
};

// Items of split tiles at most: a tile of r records in r + w slots has m =
// max(ceil(r / imax), ceil((r + w) / 2^17)) items, and where m > 1 the first is at
// most 2 r / imax, the second at most 2 r / 2^17 + 2 w / 2^17 (imax <= 2^17), so m
// is at most 2 r / imax + 2 w / 2^17.
void set_max_parts(SortLayout &S, const Plan &p, int64_t n) {
  S.imax = deposit_item_max(n, p.tg.K);
  S.max_parts = 2 * (ceil_div(n, (int64_t)S.imax) + ceil_div(S.L2.slots() - n, (int64_t)DEPOSIT_ITEM_MAX));
}

SortLayout sort_layout(const Plan &p, int64_t n, int rw) {
  SortLayout S;
  const TileGeom &tg = p.tg;
  const int nhi = 1 << tg.hi_bits, nlo = 1 << tg.lo_bits;
  S.two = tg.passes == 2;
  if (!S.two) {
    S.L2 = paged_layout(n, n, 1, nhi, rw, 3, 8, 8);
    set_max_parts(S, p, n);
    return S;
  }
  S.paged1 = first_paged(p, n);
  if (S.paged1) {
    S.L1 = paged_layout(n, n, 1, nhi, rw, 6, 8, 8);
    S.slots1 = S.L1.slots();
    S.paged1 = S.slots1 <= ((int64_t)1 << 32);
  }
  if (!S.paged1) S.slots1 = n;
  // a paged first pass's slots hold empty ones, which the last pass's pool need
  // not repeat: they are counted where the pool would grow by more than one
  // pass's allowance (16.3 -> 14.7 GB at 2^30 records), which costs the second pass
  // 5 us (0.6% of a forward at 360^3)
  const int inlg = S.paged1 ? S.L1.lg : 0;
  S.L2 = paged_layout(S.slots1, S.slots1, nhi, nlo, rw, 3, 8, 2, inlg);
  S.lacks = S.L2.slots() > n + std::max(n / 6, (int64_t)1 << 26);
  if (S.lacks) S.L2 = paged_layout(n, S.slots1, nhi, nlo, rw, 3, 8, 2, inlg);
  set_max_parts(S, p, n);
  return S;
}

template <int NM>
TileOrder sort_impl(Plan &p, const KeyGeom &kg, int64_t n, const float *pos, const float *masses, bool with_perm,
                    bool every_tile, const SortLayout &S) {
  constexpr int RW = Src<NM>::RW;
  hipStream_t s = p.stream;
  const TileGeom &tg = p.tg;
  const int nhi = 1 << tg.hi_bits, nlo = 1 << tg.lo_bits;
  const int64_t ks = (int64_t)nhi * nlo;
  float *A = p.recA.as<float>();
  float *B = p.recB.as<float>();
  Src<NM> raw{pos, masses, true};
  uint32_t *perm1 = with_perm ? p.permA.as<uint32_t>() : nullptr;
  uint32_t *perm2 = (with_perm && S.two) ? p.permB.as<uint32_t>() : nullptr;

  // bucket totals, of the tiles and of a first pass's segments: zero between
  // sorts (k_dir clears what it read)
  const int64_t ntot = ks + (S.two ? nhi : 0);
  unsigned long long *tot = static_cast<unsigned long long *>(p.sort_tot.ensure((size_t)ntot * 8));
  if (p.sort_tot_zero != ntot) fill_zero(tot, (size_t)ntot * 8, s);
  p.sort_tot_zero = 0;

  // with masses, pass 1 (which reads every mass) records their range for the deposit
  const int64_t chunk1 = S.two && !S.paged1 ? counted_chunk(n) : 0;
  const int64_t g1 = !S.two ? S.L2.G : S.paged1 ? S.L1.G : ceil_div(n, chunk1);
  uint32_t *mrange = nullptr, *mrange_w = nullptr;
  if (NM == 1) {
    mrange = static_cast<uint32_t *>(p.mrange.ensure((size_t)(2 + 2 * g1) * 4));
    mrange_w = mrange + 2;
  }

  // the last pass, and before it the first of two
  PtArgs P2;
  uint32_t *lacks;
  uint32_t *blist = pg_buffers(p.pages, S.L2, S.two ? nlo : nhi, P2.pg, tot, &lacks);
  const PgOut &pg2 = P2.pg;
  P2.grid = S.L2.G;
  P2.im.n = n;
  P2.im.chunk = S.L2.chunk;
  P2.ds = digit_sel(kg, 0, S.two ? tg.lo_bits : tg.hi_bits);
  P2.nb = S.two ? nlo : nhi;
  P2.h = S.L2.h;
  P2.dst = S.two ? B : A;
  if (!S.two) {
    P2.pos = pos;
    P2.masses = masses;
    P2.perm = perm1;
    P2.mrange_w = mrange_w;
    Stage st(p, "sort_downsweep1");
    launch_partition<NM, IN_RAW, true>(P2, kg, s);
  } else {
    PtArgs P1;
    P1.pos = pos;
    P1.masses = masses;
    P1.im.n = n;
    P1.im.chunk = S.paged1 ? S.L1.chunk : chunk1;
    P1.grid = g1;
    P1.ds = digit_sel(kg, tg.lo_bits, tg.hi_bits);
    P1.nb = nhi;
    P1.dst = A;
    P1.perm = perm1;
    P1.mrange_w = mrange_w;
    // segments of pass 2: first list entry (or record), and the segment of
    // each workgroup's first
    const int64_t ss = nhi + 4;
    uint32_t *sb = static_cast<uint32_t *>(p.seginfo.ensure((size_t)(ss + S.L2.G) * 4));
    DirArgs D{};
    D.tot = tot + ks;
    D.nb = D.kreal = nhi;
    D.start = sb;
    D.first_seg = sb + ss;
    D.piece = pg2.piece;
    D.lacks = lacks;
    D.npiece = S.L2.pieces;
    P2.pos = A;
    P2.start = sb;
    P2.first_seg = sb + ss;
    P2.lacks = S.lacks ? lacks : nullptr;
    P2.im.nseg = nhi;
    P2.perm = perm2;
    if (S.paged1) {
      // pass 1, paged: the positions are read once
      uint32_t *lacks1;
      uint32_t *blist1 = pg_buffers(p.pages1, S.L1, nhi, P1.pg, tot + ks, &lacks1);
      P1.h = S.L1.h;
      {
        Stage st(p, "sort_downsweep1");
        launch_partition<NM, IN_RAW, true>(P1, kg, s);
      }
      Stage st(p, "sort_pages");
      D.unit = (uint32_t)(S.L2.chunk >> S.L1.lg);
      D.funit = FastDiv(D.unit);
      launch_dir(D, s);
      hipLaunchKernelGGL(k_list, dim3((unsigned)S.L1.pieces), dim3(SORT_THREADS), nhi * 4, s, P1.pg, nhi, D.start,
                         blist1);
      GENPK_LAUNCH_CHECK();
      if (S.lacks) {
        hipLaunchKernelGGL(k_lacks, dim3((unsigned)S.L2.G), dim3(LACK_THREADS), 0, s, blist1, sb, sb + ss, nhi, S.L1.lg,
                           D.unit, lacks);
        GENPK_LAUNCH_CHECK();
      }
      P2.blist = blist1;
      P2.im.lg = S.L1.lg;
    } else {
      // pass 1, counted
      uint32_t *t1 = static_cast<uint32_t *>(p.table1.ensure((size_t)nhi * g1 * 4));
      P1.h = partition_shape(nhi, RW, false, 8);
      P1.offsets = t1;
      {
        Stage st(p, "sort_upsweep1");
        hipLaunchKernelGGL((k_upsweep<NM>), dim3((unsigned)g1), dim3(SORT_THREADS), nhi * 4, s, raw, P1.im, kg, P1.ds,
                           nhi, t1);
        GENPK_LAUNCH_CHECK();
      }
      exclusive_scan_u32(t1, t1, (int64_t)nhi * g1, p.scan_tmp, s);
      {
        Stage st(p, "sort_downsweep1");
        launch_partition<NM, IN_RAW, false>(P1, kg, s);
      }
      hipLaunchKernelGGL(k_seg_tot, dim3((unsigned)ceil_div(nhi, 256)), dim3(256), 0, s, t1, g1, nhi, n, tot + ks);
      GENPK_LAUNCH_CHECK();
      D.unit = (uint32_t)S.L2.chunk;
      D.funit = FastDiv(D.unit);
      launch_dir(D, s);
    }
    Stage st(p, "sort_downsweep2");
    if (S.paged1)
      launch_partition<NM, IN_LIST, true>(P2, kg, s);
    else
      launch_partition<NM, IN_SEG, true>(P2, kg, s);
  }

  // the tiles' block lists and work items
  TileOrder o;
  const int64_t slots = S.L2.slots();
  const int64_t max_items = tg.K + S.max_parts;
  const int64_t ts = (ks + 4) / 4 * 4;
  const int64_t nsec = ceil_div(ks, dir_section(ks));
  uint32_t *ib = static_cast<uint32_t *>(p.item_start.ensure((size_t)(ts + nsec) * 4 * 4 + 64));
  DirArgs D{};
  D.tot = tot;
  D.nb = ks;
  D.kreal = tg.K;
  D.start = ib;
  D.cost = ib + ts;
  D.items = static_cast<uint4 *>(p.items.ensure((size_t)max_items * 16));
  D.store = every_tile ? 1 : 0;
  D.lg = S.L2.lg;
  D.limax = ilog2(S.imax);
  D.pstart = ib + 2 * ts;
  D.heavy = ib + 3 * ts;
  D.secsum = reinterpret_cast<uint4 *>(ib + 4 * ts);
  D.counts = static_cast<uint32_t *>(p.heavy.ensure(64 + DEPOSIT_WGS_MAX * 4));
  D.share = D.counts + 16;
  D.max_parts = (uint32_t)S.max_parts;
  D.wgs = (uint32_t)deposit_wgs(p, RW, max_items);
  D.fwgs = FastDiv(D.wgs);
  // the flush of a tile and the waits around it take about as long as the
  // records of an eighth of its cells (a quarter and a half measured the same
  // within 3%)
  const int64_t icost = tg.cells / 8;
  while (((slots + max_items * icost) >> D.cshift) >= (int64_t)1 << 31) D.cshift++;
  D.icost = (uint32_t)(icost >> D.cshift);
  D.nonfinite = static_cast<uint32_t *>(p.nonfinite.ensure(64));
  D.mrange = mrange;
  D.mrange_w = mrange_w;
  D.nw = g1;
  {
    Stage st(p, "sort_tiles");
    launch_dir(D, s);
    hipLaunchKernelGGL(k_list, dim3((unsigned)S.L2.pieces), dim3(SORT_THREADS), P2.nb * 4, s, pg2, P2.nb, D.start,
                       blist);
    GENPK_LAUNCH_CHECK();
  }
  p.sort_tot_zero = ntot;

  o.rec = P2.dst;
  o.rw = RW;
  o.has_mass = NM != 0;
  o.has_perm = with_perm;
  o.perm1 = perm1;
  o.perm2 = perm2;
  o.list = {D.start, D.pstart, D.items, D.counts, D.cost,      D.share,
            blist,   S.L2.lg,  ks,      max_items, D.max_parts, D.wgs};
  o.heavy = D.heavy;
  o.partials = (S.two ? p.recA : p.partials).as<double>();
  o.mrange = mrange;
  o.n = n;
  return o;
}
}  // namespace

uint32_t deposit_item_max(int64_t n, int64_t tiles) {
  const int64_t cus = num_cus();
  uint32_t m = DEPOSIT_ITEM_MAX;
  while (m > DEPOSIT_ITEM_MIN && (tiles + n / m < 4 * cus || (int64_t)m * 2 * cus > n ||
                                  ((int64_t)m * 4 * cus > n && (int64_t)m * tiles >= 4 * n)))
    m /= 2;
  return m;
}

KeyGeom key_geom(const Plan &p, double boxsize) {
  KeyGeom g;
  g.units = (double)p.d / boxsize;
  g.d = (int)p.d;
  g.TX = p.tg.TX; g.TY = p.tg.TY; g.TZ = p.tg.TZ;
  g.sx = p.tg.sx; g.sy = p.tg.sy; g.sz = p.tg.sz;
  g.ntx = p.tg.ntx; g.nty = p.tg.nty; g.ntz = p.tg.ntz;
  return g;
}

TileOrder sort_by_tile(Plan &p, const KeyGeom &kg, int64_t n, const float *pos, const float *masses, bool with_perm,
                       bool every_tile) {
  GENPK_REQUIRE(n > 0 && n <= ((int64_t)1 << 31), "sort_by_tile: particle count out of range");
  const int rw = 3 + (masses ? 1 : 0);
  const SortLayout S = sort_layout(p, n, rw);
  // the first pass of two writes recA and the last pass recB (a single pass:
  // recA); with the permutations the other one also takes the adjoint
  // gather's output records (up to 4 floats per slot of the sorted pool).
  // perm2 is indexed by pass-1 slots.
  // The partial tiles too lie in the pool that the last pass has read (2.8 GB
  // of their own at 2^30 records).
  const size_t last = (size_t)S.L2.slots(), gather = with_perm ? last * 16 : 0;
  const size_t parts = (size_t)S.max_parts * p.tg.cells * 8 + 64;
  if (S.two) {
    p.recA.ensure(std::max({(size_t)S.slots1 * rw * 4, gather, parts}));
    p.recB.ensure(last * rw * 4);
  } else {
    p.recA.ensure(last * rw * 4);
    if (with_perm) p.recB.ensure(gather);
    p.partials.ensure(parts);
  }
  if (with_perm) {
    p.permA.ensure((size_t)n * 4);
    if (S.two) p.permB.ensure((size_t)S.slots1 * 4);
  }
  if (masses) return sort_impl<1>(p, kg, n, pos, masses, with_perm, every_tile, S);
  return sort_impl<0>(p, kg, n, pos, nullptr, with_perm, every_tile, S);
}

}  // namespace genpk
