// 3-D real-to-complex FFT on the padded in-place layout the reference hands
// to FFTW (gen-pk.cpp:176-193: real [d][d][2(d/2+1)] in, complex
// [d][d][d/2+1] out, unnormalised, forward sign -1), and its unnormalised
// inverse.  Three passes over HBM:
//   z: r2c of each contiguous row; d reals are packed as d/2 complex, one
//      d/2-point Stockham FFT in LDS, then the even/odd split to d/2+1 bins;
//   y, x: length-d c2c FFTs over column blocks of B consecutive kz, loaded
//      as B-wide rows (coalesced) into LDS, transformed in place.
#include "fft_core.h"
#include "plan.h"
#include "tiles.h"

#include <cmath>
#include <vector>

namespace genpk {

namespace {

// Workgroup shapes (measured at 1024^3): the z passes run 512 threads and
// the column passes 1024 threads over the same LDS footprint (ELEMS complex
// values per workgroup, two workgroups per CU), i.e. MAXE staged values per
// thread; more waves per CU hide the global-memory latency of the staged
// loads (z pass 3.7 -> 3.0 ms, y pass 2.9 -> 2.0 ms against 256 threads).
constexpr int FFT_THREADS = 512;   // z passes
constexpr int COL_THREADS = 1024;  // y and x passes
template <typename T> struct FftCfg;
template <> struct FftCfg<float> { static constexpr int ELEMS = 8192; static constexpr int MAXE = 16; static constexpr int COLE = 8; };
template <> struct FftCfg<double> { static constexpr int ELEMS = 4096; static constexpr int MAXE = 8; static constexpr int COLE = 4; };

// z pass, forward: rows of d reals -> d/2+1 complex, L rows per workgroup.
// FROM_TILES: the rows are assembled from the deposit's tile store while
// loading, halo cells folded in (the fold), so the real-space grid is never
// written.
// Two workgroups share a CU (up to 80 KB of LDS each, and registers for four
// waves per SIMD: waves_per_eu).  The rows sit in LDS
// with one element of padding per 32 (lds_ix), which spreads the strided
// writes of the FFT stages over the banks.
// BFLY (from the tile store; the first stage's radix, 0: element by element):
// each thread loads the inputs of whole butterflies of the first stage
// straight from the tile store, one row's place for all of a butterfly's, and
// runs that stage from registers.  The pass fills the SIMDs where each
// element looks up its own place: 0.173 -> 0.138 ms at 360^3 FP32 (first radix
// 4), 0.037 -> 0.029 at 200^3, 0.106 -> 0.088 at 300^3 (first radix 2); FP64
// 0.243 -> 0.206 at 360^3, 1.00 -> 0.84 at 600^3.
// CT = 512: the plan is M = 512 = 8 * 8 * 8 (d = 1024), run with
// compile-time stages (fft_stage_ct); 0: any plan.  STD (with CT = 512):
// the default 16 x 32 x 32 tiles, whose store offsets (below 2^31 at d =
// 1024) are computed in 32 bits from compile-time strides, in the butterfly
// loader (FP32) or the element-wise one (FP64).
// Rows of a tile's first x or y layer add the halos of the previous tiles
// while they load (add_halo_rows), within the registers of two workgroups per
// CU (waves_per_eu: four waves per SIMD): fold and z pass together 2.28 ->
// 2.06 ms at 1024^3 FP32 and 0.069 -> 0.061 at 256^3 against two in-place
// fold launches before the pass.
template <typename T, bool FROM_TILES, int BFLY = 0, int CT = 0, bool STD = false>
__global__ void __launch_bounds__(FFT_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_r2c_z(T *__restrict__ field, const T *__restrict__ tiles, FoldGeom fg, FastDiv fdd, int64_t rowlen, int64_t nrows,
        int L, FastDiv fdM, FastDiv fdK, RadixPlan rp, const typename Cx<T>::C *__restrict__ twM,
        const typename Cx<T>::C *__restrict__ twd) {
  using C = typename Cx<T>::C;
  constexpr int MAXE = FftCfg<T>::MAXE;
  extern __shared__ unsigned char lds_raw[];
  C *buf = reinterpret_cast<C *>(lds_raw);
  const int M = CT ? CT : rp.n;
  const int64_t row0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * L;
  const int nl = (int)min((int64_t)L, nrows - row0);
  const int tot = L * M;
  // twiddles of the M-point FFT and of the even/odd split, staged in LDS
  C *stw = buf + lds_len<true>((int64_t)L * M);  // [M]
  C *sxw = stw + M;               // [NK]
  if constexpr (BFLY != 0) {
    constexpr int R0 = BFLY, NB = R0 == 8 ? 2 : (MAXE + R0 - 1) / R0;
    constexpr int HG = R0 % 4 ? R0 : sizeof(T) == 4 ? 4 : 2;  // pairs that add halos at a time
    // butterfly u = threadIdx.x + FFT_THREADS * i: row u / NQ, inputs
    // u % NQ + NQ * r (NQ = M / R0)
    const int NQ = M / R0;
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int u = threadIdx.x + FFT_THREADS * i;
      const int b = CT ? u / (CT / 8) : (int)fdM.div((uint32_t)(R0 * u)), j = u - b * NQ;
      if (b < L) {
        C w[R0];
        if (STD && b < nl) {
          static_assert(!STD || CT == 512, "standard tiles with the d = 1024 loaders");
          // d = 1024, tiles 16 x 32 x 32 (17 x 33 halo'd rows of 32 per tile):
          // z = 2 (j + 64 r) lies in tile column tz = 4 r + j / 16 at lz = 2 (j % 16)
          constexpr uint32_t CM = 17 * 33 * 32, CZ = 17 * 33;
          const uint32_t row = (uint32_t)(row0 + b);
          const uint32_t x = row >> 10, y = row & 1023u;
          const uint32_t txy = (x >> 4) * 32u + (y >> 5), rr = (x & 15u) * 33u + (y & 31u);
          const uint32_t jz = (uint32_t)j >> 4, lz = 2u * ((uint32_t)j & 15u);
          const uint32_t base = (txy * 32u + jz) * CM + rr * 32u + lz;
          const T *tb = tiles + base;
          T zh8[R0];
#pragma unroll
          for (int r = 0; r < R0; r++) {
            w[r] = C{tb[r * 4 * CM], tb[r * 4 * CM + 1]};
            // the previous tile along z's z-halo cell: tile column 4 r + jz - 1
            // (for r = jz = 0 the last column, 31, periodically)
            const uint32_t tzp = (4u * r + jz + 31u) & 31u;
            zh8[r] = lz == 0 ? tiles[(uint32_t)fg.zoff + (txy * 32u + tzp) * CZ + rr] : (T)0;
          }
          if ((x & 15u) == 0 || (y & 31u) == 0)
            add_halo_rows<T, R0, HG>(
                tiles, fg, row_fold(fg, (int)x, (int)y), [&](int r) { return 2 * (j + 64 * r); }, w, zh8);
          if (lz == 0) {
#pragma unroll
            for (int r = 0; r < R0; r++) w[r].x = w[r].x + zh8[r];  // one rounding, as below
          }
        } else if (b < nl) {
          const int64_t row = row0 + b;
          const int x = (int)fdd.div((uint32_t)row), y = (int)(row - (int64_t)x * fg.d);
          const RowFold rf = row_fold(fg, x, y);
          const int64_t txy = rf.t, rr = rf.r;
          T zh8[R0];
#pragma unroll
          for (int r = 0; r < R0; r++) {
            const int z = 2 * (j + NQ * r);
            const int tz = z >> fg.sz, lz = z & (fg.TZ - 1);
            const int64_t at = txy * fg.ntz * fg.cm + (int64_t)tz * fg.cm + rr * fg.TZ + lz;
            w[r] = C{tiles[at], tiles[at + 1]};
            zh8[r] = (T)0;
            if (lz == 0) {
              // the previous tile along z's z-halo cell (in its row store when partial)
              const int tzp = tz == 0 ? fg.ntz - 1 : tz - 1;
              const int hw = min(fg.TZ, fg.d - tzp * fg.TZ);
              const int64_t h = hw < fg.TZ ? (int64_t)tzp * fg.cm + hw + txy * fg.ntz * fg.cm + rr * fg.TZ
                                           : fg.zoff + (int64_t)tzp * fg.cz + txy * fg.ntz * fg.cz + rr;
              zh8[r] = tiles[h];
            }
          }
          if (rf.fx || rf.fy)
            add_halo_rows<T, R0, HG>(tiles, fg, rf, [&](int r) { return 2 * (j + NQ * r); }, w, zh8);
#pragma unroll
          for (int r = 0; r < R0; r++) w[r].x = w[r].x + zh8[r];  // as the element-wise load: one rounding
        } else {
#pragma unroll
          for (int r = 0; r < R0; r++) w[r] = C{0, 0};
        }
        Dft<R0, -1, C>::run(w);
#pragma unroll
        for (int r = 0; r < R0; r++) buf[lds_ix<true>(b * M + R0 * j + r)] = w[r];
      }
    }
    for (int i = threadIdx.x; i < M; i += FFT_THREADS) stw[i] = twM[i];
    for (int i = threadIdx.x; i < (M + 1) / 2; i += FFT_THREADS) sxw[i] = twd[i];
    __syncthreads();
    if constexpr (CT == 512)
      lds_fft_ct<512, 8, -1, false, MAXE, false, C, true, 8, 8>(buf, buf, L, 0, stw);
    else
      for (int st = 1; st < rp.nst; st++)
        fft_stage_r<-1, false, MAXE, false, C, true>(rp.st[st].R, buf, buf, L, 0, 1, M, rp.st[st], stw);
  } else {
  C v[MAXE];
  T zh[FROM_TILES ? MAXE : 1];
  // the x and y halos of element q (a row of a tile's first x or y layer)
  auto fold_q = [&](int q, int x, int y, int z) {
    if ((x & (fg.TX - 1)) == 0 || (y & (fg.TY - 1)) == 0) {
      C w[1] = {v[q]};
      T wh[1] = {zh[FROM_TILES ? q : 0]};
      add_halo_rows<T, 1, 1>(tiles, fg, row_fold(fg, x, y), [&](int) { return z; }, w, wh);
      v[q] = w[0];
      zh[FROM_TILES ? q : 0] = wh[0];
    }
  };
  if (FROM_TILES && M == FFT_THREADS && STD) {
    // d = 1024 with the default tiles (the FP64 plan): as below, with 32-bit
    // store offsets from compile-time strides (the store holds fewer than
    // 2^31 values; every tile is full, so a z halo sits in the z-halo plane)
    constexpr uint32_t CM = 17 * 33 * 32, CZ = 17 * 33;
    const uint32_t z = 2u * threadIdx.x, tz = z >> 5, lz = z & 31u, tzp = (tz + 31u) & 31u;
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      v[q] = C{0, 0};
      zh[FROM_TILES ? q : 0] = (T)0;
      if (q < L && q < nl) {
        const uint32_t row = (uint32_t)(row0 + q);
        const uint32_t x = row >> 10, y = row & 1023u;
        const uint32_t txy = (x >> 4) * 32u + (y >> 5), rr = (x & 15u) * 33u + (y & 31u);
        const uint32_t at = (txy * 32u + tz) * CM + rr * 32u + lz;
        v[q] = C{tiles[at], tiles[at + 1]};
        if (lz == 0) zh[FROM_TILES ? q : 0] = tiles[(uint32_t)fg.zoff + (txy * 32u + tzp) * CZ + rr];
        fold_q(q, (int)x, (int)y, (int)z);
      }
    }
  } else if (FROM_TILES && M == FFT_THREADS) {
    // element q of this thread is row row0 + q, reals 2m and 2m + 1 with m =
    // threadIdx.x: the row's part of the store offset is the same for the
    // whole workgroup (scalar), the z part is the lane's own
    const int z = 2 * (int)threadIdx.x;
    const int tz = z >> fg.sz, lz = z & (fg.TZ - 1);
    const int64_t lane_off = (int64_t)tz * fg.cm + lz;
    // z-halo cell added to the first cell of a tile along z: local z = width
    // of the previous tile, in its row store when that tile is partial
    const int tzp = tz == 0 ? fg.ntz - 1 : tz - 1;
    const int hw = min(fg.TZ, fg.d - tzp * fg.TZ);
    const bool hrow = hw < fg.TZ;
    const int64_t h_off = hrow ? (int64_t)tzp * fg.cm + hw : fg.zoff + (int64_t)tzp * fg.cz;
    const int64_t h_tmul = hrow ? (int64_t)fg.ntz * fg.cm : (int64_t)fg.ntz * fg.cz;
    const int64_t h_rmul = hrow ? fg.TZ : 1;
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      v[q] = C{0, 0};
      zh[FROM_TILES ? q : 0] = (T)0;
      if (q < L && q < nl) {
        const int64_t row = row0 + q;
        const int x = (int)fdd.div((uint32_t)row), y = (int)(row - (int64_t)x * fg.d);
        const int64_t txy = (int64_t)(x >> fg.sx) * fg.nty + (y >> fg.sy);
        const int64_t r = (int64_t)(x & (fg.TX - 1)) * fg.HY + (y & (fg.TY - 1));
        const int64_t at = txy * fg.ntz * fg.cm + r * fg.TZ + lane_off;
        v[q] = C{tiles[at], tiles[at + 1]};
        if (lz == 0) zh[FROM_TILES ? q : 0] = tiles[h_off + txy * h_tmul + r * h_rmul];
        fold_q(q, x, y, z);
      }
    }
  } else {
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * FFT_THREADS;
    v[q] = C{0, 0};
    if (FROM_TILES) zh[FROM_TILES ? q : 0] = (T)0;
    if (i < tot) {
      const int l = (int)fdM.div((uint32_t)i), m = i - l * M;
      if (l < nl) {
        const int64_t row = row0 + l;
        if (FROM_TILES) {
          // both reals sit in one aligned tile row (TZ even); the first cell
          // of a tile along z adds the previous tile's z-halo cell
          const int x = (int)fdd.div((uint32_t)row), y = (int)(row - (int64_t)x * fg.d);
          const RowFold rf = row_fold(fg, x, y);
          const ZPlace zp = z_place(fg, 2 * m);
          const int64_t at = row_at(fg, rf.t, rf.r, zp);
          v[q] = C{tiles[at], tiles[at + 1]};
          if (zp.halo) zh[FROM_TILES ? q : 0] = tiles[row_halo_at(fg, rf.t, rf.r, zp)];
          fold_q(q, x, y, 2 * m);
        } else {
          const T *r = field + row * rowlen;
          v[q] = C{r[2 * m], r[2 * m + 1]};
        }
      }
    }
  }
  }
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * FFT_THREADS;
    // z-halo added after all loads are in flight (a + b rounds once, as in k_fold)
    if (FROM_TILES) v[q].x = v[q].x + zh[FROM_TILES ? q : 0];
    if (i < tot) buf[lds_ix<true>(i)] = v[q];
  }
  for (int i = threadIdx.x; i < M; i += FFT_THREADS) stw[i] = twM[i];
  for (int i = threadIdx.x; i < (M + 1) / 2; i += FFT_THREADS) sxw[i] = twd[i];
  __syncthreads();
  if constexpr (CT == 512)
    lds_fft_ct<512, 1, -1, false, MAXE, false, C, true, 8, 8, 8>(buf, buf, L, 0, stw);
  else
    lds_fft<-1, false, MAXE, C, true>(buf, rp, L, 0, 1, M, stw);
  }
  // X_k = E + w^k O and X_{M-k} = conj(E - w^k O) with E = (Z_k + conj Z_{M-k}) / 2,
  // O = (Z_k - conj Z_{M-k}) / 2i, w = exp(-2 pi i / d) and Z_M = Z_0: one thread
  // forms both (each by its own thread took twice the LDS reads and index
  // arithmetic, in a pass that fills the SIMDs (0.9 to 1.0 VALU instructions a
  // cycle in FP32): 0.258 -> 0.244 ms at 360^3 FP64, 0.570 -> 0.550 at 512^3,
  // 0.99 -> 0.91 at 720^3 FP32; even at 1024^3, 2.00 to 2.19 ms either way from
  // one process to the next)
  auto split = [&](int l, int k, C w) {
    const C zk = buf[lds_ix<true>(l * M + k)], zc = buf[lds_ix<true>(l * M + (k == 0 ? 0 : M - k))];
    const C e = C{(zk.x + zc.x) * (T)0.5, (zk.y - zc.y) * (T)0.5};
    const C o = cmul(C{(zk.y + zc.y) * (T)0.5, (zc.x - zk.x) * (T)0.5}, w);
    C *row = reinterpret_cast<C *>(field + (row0 + l) * rowlen);
    row[k] = cadd(e, o);
    row[M - k] = C{e.x - o.x, o.y - e.y};
    // k = M / 2 is its own partner, with w^(M/2) = -i
    if (k == 0 && M % 2 == 0) row[M / 2] = cconj(buf[lds_ix<true>(l * M + M / 2)]);
  };
  const int NK = (M + 1) / 2;
  if ((NK & (NK - 1)) == 0 && NK <= FFT_THREADS) {
    // a power of two: a thread keeps its k
    const int k = threadIdx.x & (NK - 1), rpi = FFT_THREADS / NK;
    const C w = sxw[k];
#pragma unroll 4
    for (int l = threadIdx.x / NK; l < nl; l += rpi) split(l, k, w);
    return;
  }
  for (int i = threadIdx.x; i < nl * NK; i += FFT_THREADS) {
    const int l = (int)fdK.div((uint32_t)i), k = i - l * NK;
    split(l, k, sxw[k]);
  }
}

// z pass, inverse: d/2+1 complex -> d reals (unnormalised c2r); the
// imaginary parts of kz = 0 and kz = d/2 do not contribute.
//   Z_k = (X_k + conj X_{M-k}) + i w^-k (X_k - conj X_{M-k}),  w = exp(-2 pi i / d)
// Each thread reads the pairs X_k, X_{M-k} (k <= M/2) of a row and forms Z_k and
// Z_{M-k} from them in registers, so that the half spectrum takes no round
// trip through LDS of its own (0.49 ms at 512^3 FP32 with it and with
// element-wise 4-byte accesses, 0.28 now).
template <typename T>
__global__ void __launch_bounds__(FFT_THREADS) k_c2r_z(T *__restrict__ field, int64_t rowlen, int64_t nrows, int L,
                                                      FastDiv fdM, FastDiv fdP, RadixPlan rp,
                                                      const typename Cx<T>::C *__restrict__ twM,
                                                      const typename Cx<T>::C *__restrict__ twd) {
  using C = typename Cx<T>::C;
  constexpr int U = FftCfg<T>::MAXE / 2;  // pairs in flight per thread
  extern __shared__ unsigned char lds_raw[];
  C *buf = reinterpret_cast<C *>(lds_raw);  // L padded rows of M (lds_ix)
  const int M = rp.n, NP = M / 2 + 1;       // pairs per row (k = 0 with M, M/2 with itself)
  C *stw = buf + lds_len<true>((int64_t)L * M);
  const int64_t row0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * L;
  const int nl = (int)min((int64_t)L, nrows - row0), np = nl * NP;
  for (int i = threadIdx.x; i < M; i += FFT_THREADS) stw[i] = twM[i];
  for (int i0 = threadIdx.x; i0 < np; i0 += FFT_THREADS * U) {
    C xa[U], xb[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * FFT_THREADS;
      xa[u] = xb[u] = C{0, 0};
      if (i < np) {
        const int l = (int)fdP.div((uint32_t)i), k = i - l * NP;
        const C *row = reinterpret_cast<const C *>(field + (row0 + l) * rowlen);
        xa[u] = row[k];
        xb[u] = row[M - k];
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * FFT_THREADS;
      if (i >= np) continue;
      const int l = (int)fdP.div((uint32_t)i), k = i - l * NP;
      if (k == 0) xa[u].y = xb[u].y = (T)0;
      const C t = twd[k];
      auto zof = [&](C x, C y, C w) {  // x = X_k, y = X_{M-k}, w = w^-k
        const C yc = cconj(y);
        const C s = cadd(x, yc), dd = cmul(csub(x, yc), w);
        return C{s.x - dd.y, s.y + dd.x};
      };
      buf[lds_ix<true>(l * M + k)] = zof(xa[u], xb[u], C{t.x, -t.y});
      // w^-(M-k) = -conj(w^-k)
      if (k != 0 && 2 * k != M) buf[lds_ix<true>(l * M + M - k)] = zof(xb[u], xa[u], C{-t.x, -t.y});
    }
  }
  __syncthreads();
  lds_fft<+1, false, FftCfg<T>::MAXE, C, true>(buf, rp, nl, 0, 1, M, stw);
  for (int i = threadIdx.x; i < nl * M; i += FFT_THREADS) {
    const int l = (int)fdM.div((uint32_t)i), m = i - l * M;
    C *row = reinterpret_cast<C *>(field + (row0 + l) * rowlen);
    row[m] = buf[lds_ix<true>(i)];
    if (m == 0) row[M] = C{0, 0};
  }
}

// c2c along y (axis = 1) or x (axis = 0) over column blocks (ColMap).  CT =
// 1024: the plan is n = 1024 = 8 * 8 * 8 * 2, run with compile-time stages; 0:
// any plan.  R0 (a first radix below COLE): each thread loads the inputs of
// COLE / R0 whole butterflies of the first stage and runs it from registers
// (y pass FP32 0.060 -> 0.052 ms at 300^3, 0.261 -> 0.214 at 486^3, 1.54 -> 1.35
// at 900^3; cols_impl says where not).
template <typename T, int SIGN, int CT = 0, int R0 = 0>
__global__ void __launch_bounds__(COL_THREADS) k_cols(typename Cx<T>::C *__restrict__ f, ColMap cm, int axis,
                                                     RadixPlan rp, const typename Cx<T>::C *__restrict__ tw) {
  using C = typename Cx<T>::C;
  constexpr int MAXE = FftCfg<T>::COLE;
  extern __shared__ unsigned char lds_raw[];
  C *buf = reinterpret_cast<C *>(lds_raw);  // [n][B]
  const int n = CT ? CT : rp.n;
  const int lgb = cm.lgb, B = 1 << lgb;
  const int64_t d = cm.d, hz = cm.hz;
  const ColMap::Block c = cm.at(xcd_block(blockIdx.x, gridDim.x));
  const int64_t estride = axis == 1 ? hz : d * hz;
  C *base = f + (int64_t)c.outer * (axis == 1 ? d * hz : hz) + c.kz0;
  const int b = threadIdx.x & (B - 1);  // a thread's elements lie in one column
  const int tot = n * B;
  if constexpr (R0 != 0) {
    constexpr int NB = MAXE / R0;
    const int nq = n / R0, j0 = (int)threadIdx.x >> lgb, jstep = COL_THREADS >> lgb;
    C v[NB][R0];
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
      for (int r = 0; r < R0; r++) {
        const int j = j0 + i * jstep;
        v[i][r] = j < nq && b < c.nb ? base[(int64_t)(j + r * nq) * estride + b] : C{0, 0};
      }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int j = j0 + i * jstep;
      Dft<R0, SIGN, C>::run(v[i]);
      if (j < nq) {
#pragma unroll
        for (int r = 0; r < R0; r++) buf[((j * R0 + r) << lgb) + b] = v[i][r];
      }
    }
  } else {
    C v[MAXE];
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      const int i = threadIdx.x + q * COL_THREADS;
      v[q] = (i < tot && b < c.nb) ? base[(i >> lgb) * estride + b] : C{0, 0};
    }
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      const int i = threadIdx.x + q * COL_THREADS;
      if (i < tot) buf[i] = v[q];
    }
  }
  C *stw = buf + tot;  // twiddles staged in LDS
  for (int i = threadIdx.x; i < n; i += COL_THREADS) stw[i] = tw[i];
  __syncthreads();
  if constexpr (CT == 1024)
    lds_fft_ct<1024, 1, SIGN, true, MAXE, false, C, false, 8, 8, 8, 2>(buf, buf, B, lgb, stw);
  else
    for (int st = R0 ? 1 : 0; st < rp.nst; st++)
      fft_stage_r<SIGN, true, MAXE, false, C, false>(rp.st[st].R, buf, buf, B, lgb, B, 1, rp.st[st], stw);
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * COL_THREADS;
    if (i < tot && b < c.nb) base[(i >> lgb) * estride + b] = buf[i];
  }
}

// k_cols for a first radix of COLE: every thread (below n * B / COLE) loads
// exactly the inputs of one first-stage butterfly (elements j + q * n/R of
// column b, j = tid >> lgb, b = tid & (B-1)), so the first stage runs from
// registers and the load's LDS round trip and two barriers are saved.
// L2 (last radix 2): the last stage's butterflies (rows k and k + n/2 of a
// column, twiddle w^k) write their outputs straight to global memory.
// FULL: n * B / COLE is the thread count (else smaller, and guarded).  CT =
// 1024 (with FULL): compile-time stages for n = 1024 as 8, 8, 8, 2 (FP32, with
// L2) or 4, 8, 8, 4 (FP64 without L2).
template <typename T, int SIGN, bool L2, bool FULL, int CT = 0>
__global__ void __launch_bounds__(COL_THREADS) k_cols_r1(typename Cx<T>::C *__restrict__ f, ColMap cm, int axis,
                                                        RadixPlan rp, const typename Cx<T>::C *__restrict__ tw) {
  using C = typename Cx<T>::C;
  constexpr int R = FftCfg<T>::COLE;
  extern __shared__ unsigned char lds_raw[];
  C *buf = reinterpret_cast<C *>(lds_raw);  // [n][B]
  const int n = CT ? CT : rp.n;
  const int lgb = cm.lgb, B = 1 << lgb;
  const int64_t d = cm.d, hz = cm.hz;
  const int b = threadIdx.x & (B - 1), j = threadIdx.x >> lgb, nq = n / R;
  const ColMap::Block c = cm.at(xcd_block(blockIdx.x, gridDim.x));
  const int64_t estride = axis == 1 ? hz : d * hz;
  C *base = f + (int64_t)c.outer * (axis == 1 ? d * hz : hz) + c.kz0;
  const bool mine = FULL || j < nq;
  C v[R];
#pragma unroll
  for (int q = 0; q < R; q++) v[q] = mine && b < c.nb ? base[(int64_t)(j + q * nq) * estride + b] : C{0, 0};
  C *stw = buf + (int64_t)n * B;  // twiddles staged in LDS
  for (int i = threadIdx.x; i < n; i += COL_THREADS) stw[i] = tw[i];
  if (mine) fft_first_regs<R, SIGN>(v, buf, B, lgb, B, 1);
  __syncthreads();
  if constexpr (CT == 1024 && L2 && R == 8)
    lds_fft_ct<1024, 8, SIGN, true, R, false, C, false, 8, 8>(buf, buf, B, lgb, stw);
  else if constexpr (CT == 1024 && !L2 && R == 4)
    lds_fft_ct<1024, 4, SIGN, true, R, false, C, false, 8, 8, 4>(buf, buf, B, lgb, stw);
  else
    for (int s = 1; s < rp.nst - (L2 ? 1 : 0); s++)
      fft_stage_r<SIGN, true, R, false, C, false>(rp.st[s].R, buf, buf, B, lgb, B, 1, rp.st[s], stw);
  if constexpr (L2) {
    const int h = n / 2;
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
      const int k = j + i * (COL_THREADS >> lgb);  // butterfly b + k * B of B * n/2
      if (!FULL && k >= h) continue;
      C t = stw[k];
      if (SIGN > 0) t.y = -t.y;
      C w[2] = {buf[k * B + b], cmul(buf[(k + h) * B + b], t)};
      Dft<2, SIGN, C>::run(w);
      if (b < c.nb) {
        base[(int64_t)k * estride + b] = w[0];
        base[(int64_t)(k + h) * estride + b] = w[1];
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int i = threadIdx.x + q * COL_THREADS, e = i >> lgb;
      if ((FULL || e < n) && b < c.nb) base[(int64_t)e * estride + b] = buf[i];
    }
  }
}

// Rows per workgroup of the z passes: as many as the registers take (ELEMS
// complex values, in LDS that lets two workgroups share a CU; one less of the
// longest rows: 2.28 -> 2.05 ms at 1024^3 FP32 with 15 rows), no more than
// spread the rows over every CU.  At 256^3 FP32 64 rows make two whole rounds
// of workgroups (63 left a third round of 17: 61 -> 50 us).
template <typename T>
int rows_per_block(int64_t M, int64_t nrows) {
  const int64_t m = std::max<int64_t>(M, 1);
  int64_t L = std::max<int64_t>(1, FftCfg<T>::ELEMS / (m + (m >= 512 ? 1 : 0)));
  while (L > 1 && (lds_len<true>(L * m) + 2 * m + 1) * 2 * (int64_t)sizeof(T) > 80 * 1024) L--;
  return (int)std::min(L, std::max<int64_t>(1, ceil_div(nrows, num_cus())));
}

}  // namespace

// Columns per block of the y and x passes: as many as the registers take,
// fewer where the blocks would not cover the CUs, down to one 64- or 128-byte
// piece of a row.  (Sharing blocks between the outer indices for the last kz,
// alone in its block where B divides d/2, measured slower: 33 -> 46 us at
// 256^3 FP32, its single-element reads in a few late blocks.)
int col_block(int prec, int64_t d, int64_t hz) {
  const int elems = prec == 4 ? FftCfg<float>::ELEMS : FftCfg<double>::ELEMS;
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(64, hz - 1));  // most blocks are full
  int B = 1;
  while (B * 2 * d <= elems && B * 2 <= most) B *= 2;
  while (B > 8 && d * ceil_div(hz - 1, B) < num_cus()) B /= 2;
  return B;
}

void fft_tables_init(Plan &p) {
  const int64_t d = p.d, M = d / 2;
  std::vector<double> td(2 * d), tm(2 * std::max<int64_t>(M, 1));
  std::vector<float> fd(2 * d), fm(2 * std::max<int64_t>(M, 1));
  const long double two_pi = 6.283185307179586476925286766559005768L;
  for (int64_t m = 0; m < d; m++) {
    const long double a = two_pi * (long double)m / (long double)d;
    td[2 * m] = (double)cosl(a);
    td[2 * m + 1] = (double)(-sinl(a));
    fd[2 * m] = (float)cosl(a);
    fd[2 * m + 1] = (float)(-sinl(a));
  }
  for (int64_t m = 0; m < M; m++) {
    const long double a = two_pi * (long double)m / (long double)M;
    tm[2 * m] = (double)cosl(a);
    tm[2 * m + 1] = (double)(-sinl(a));
    fm[2 * m] = (float)cosl(a);
    fm[2 * m + 1] = (float)(-sinl(a));
  }
  auto up = [&](DevBuf &b, const void *src, size_t bytes) {
    b.ensure(bytes);
    GENPK_HIP(hipMemcpy(b.ptr, src, bytes, hipMemcpyHostToDevice));
  };
  up(p.fft.tw_d_f64, td.data(), td.size() * 8);
  up(p.fft.tw_d_f32, fd.data(), fd.size() * 4);
  up(p.fft.tw_h_f64, tm.data(), tm.size() * 8);
  up(p.fft.tw_h_f32, fm.data(), fm.size() * 4);
}

template <typename T>
static void r2c_z_impl(Plan &p, bool from_tiles) {
  using C = typename Cx<T>::C;
  const int64_t M = p.d / 2;
  const int64_t nrows = p.d * p.d;
  const int L = rows_per_block<T>(M, nrows);
  const RadixPlan &rp = p.rp_h;
  const C *twM = (p.prec == 4) ? (const C *)p.fft.tw_h_f32.ptr : (const C *)p.fft.tw_h_f64.ptr;
  const C *twd = (p.prec == 4) ? (const C *)p.fft.tw_d_f32.ptr : (const C *)p.fft.tw_d_f64.ptr;
  const FoldGeom fg = fold_geom(p);
  const dim3 grid((unsigned)ceil_div(nrows, L));
  const size_t lds = ((size_t)lds_len<true>((int64_t)L * M) + M + (M + 1) / 2) * sizeof(C);
  // the d = 1024 plan of radices 8, 8, 8 runs compile-time stages
  const bool ct512 = M == 512 && rp.nst == 3 && rp.st[0].R == 8 && rp.st[1].R == 8 && rp.st[2].R == 8;
  // FP64 at d = 1024 (seven rows a workgroup) reads the rows element-wise:
  // the butterfly loader measured 3.50 -> 3.73 ms there (0.52 -> 0.47 ms at 512)
  // the first stage from registers, for every radix it can have (one stage alone,
  // d <= 16, runs element by element)
  const int r0 = rp.nst >= 2 ? rp.st[0].R : 0;
  const bool bfly = r0 == 8 && (int64_t)L * (M / 8) <= 2 * FFT_THREADS && (sizeof(T) == 4 || !ct512);
  const bool std_tiles = p.d == 1024 && fg.TX == 16 && fg.TY == 32 && fg.TZ == 32;
  if (from_tiles && bfly && ct512 && std_tiles) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true, 8, 512, true>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else if (from_tiles && bfly && ct512) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true, 8, 512>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else if (from_tiles && bfly) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true, 8>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else if (from_tiles && ct512 && std_tiles) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true, 0, 512, true>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else if (from_tiles && ct512) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true, 0, 512>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else if (from_tiles && r0 >= 2 && r0 <= 5) {
    Stage st(p, "fold_fft_z");
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(), p.tiles.as<const T>(), fg,
                         FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M), FastDiv((uint32_t)((M + 1) / 2)),
                         rp, twM, twd);
    };
    if (r0 == 2) go(k_r2c_z<T, true, 2>);
    else if (r0 == 3) go(k_r2c_z<T, true, 3>);
    else if (r0 == 4) go(k_r2c_z<T, true, 4>);
    else go(k_r2c_z<T, true, 5>);
  } else if (from_tiles) {
    Stage st(p, "fold_fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, true>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       p.tiles.as<const T>(), fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  } else {
    Stage st(p, "fft_z");
    hipLaunchKernelGGL((k_r2c_z<T, false>), grid, dim3(FFT_THREADS), lds, p.stream, p.field.as<T>(),
                       (const T *)nullptr, fg, FastDiv((uint32_t)p.d), p.rowlen, nrows, L, FastDiv((uint32_t)M),
                       FastDiv((uint32_t)((M + 1) / 2)), rp, twM, twd);
  }
  GENPK_LAUNCH_CHECK();
}

template <typename T>
static void c2r_z_impl(Plan &p) {
  using C = typename Cx<T>::C;
  const int64_t M = p.d / 2;
  const int64_t nrows = p.d * p.d;
  const int L = rows_per_block<T>(M, nrows);
  const RadixPlan &rp = p.rp_h;
  const C *twM = (p.prec == 4) ? (const C *)p.fft.tw_h_f32.ptr : (const C *)p.fft.tw_h_f64.ptr;
  const C *twd = (p.prec == 4) ? (const C *)p.fft.tw_d_f32.ptr : (const C *)p.fft.tw_d_f64.ptr;
  Stage st(p, "ifft_z");
  hipLaunchKernelGGL(k_c2r_z<T>, dim3((unsigned)ceil_div(nrows, L)), dim3(FFT_THREADS),
                     ((size_t)lds_len<true>((int64_t)L * M) + M) * sizeof(C), p.stream, p.field.as<T>(), p.rowlen,
                     nrows, L, FastDiv((uint32_t)M), FastDiv((uint32_t)(M / 2 + 1)), rp, twM, twd);
  GENPK_LAUNCH_CHECK();
}

template <typename T, int SIGN>
static void cols_impl(Plan &p, int axis) {
  using C = typename Cx<T>::C;
  const int B = col_block(p.prec, p.d, p.hz);
  const ColMap cm = col_map(p.d, p.hz, B);
  const RadixPlan &rp = p.rp_d;
  const C *tw = (p.prec == 4) ? (const C *)p.fft.tw_d_f32.ptr : (const C *)p.fft.tw_d_f64.ptr;
  const size_t lds = (size_t)p.d * (B + 1) * sizeof(C);
  const dim3 grid(cm.nblk), block(COL_THREADS);
  Stage st(p, axis == 1 ? (SIGN < 0 ? "fft_y" : "ifft_y") : (SIGN < 0 ? "fft_x" : "ifft_x"));
  // the compile-time instances fill every thread (n * B = COL_THREADS * COLE)
  const bool full = p.d * B == (int64_t)COL_THREADS * FftCfg<T>::COLE;
  const bool ct1024 = is_plan_8882(rp) && full;
  // FP32 blocks of less than a line (8 columns of 8 bytes from d = 514 on): the
  // x pass is faster element by element than with a partly filled workgroup's
  // first stage, or one of a smaller radix, from registers, by 2 to 16% (1.62
  // against 1.84 ms at 900^3, 1.90 against 2.10 at 960^3; even from 1200 on), and the y
  // pass by up to 8% with a first radix of 8 (0.416 against 0.451 ms at 600^3,
  // 5.02 against 5.18 at 1280^3; 2% slower at 720^3).  With whole lines, in FP64
  // and along y with a smaller radix the register stage is the faster one, or even
  constexpr int COLE = FftCfg<T>::COLE;
  const bool by_elements = sizeof(T) == 4 && p.d > 512 && (rp.st[0].R == COLE ? !full : axis == 0);
  if (by_elements) {
    hipLaunchKernelGGL((k_cols<T, SIGN>), grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
  } else if (rp.st[0].R == FftCfg<T>::COLE && p.d * B <= (int64_t)COL_THREADS * FftCfg<T>::COLE) {
    const bool l2 = rp.nst > 1 && rp.st[rp.nst - 1].R == 2;
    constexpr int CT4 = FftCfg<T>::COLE == 4 ? 1024 : 0;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
    };
    if (l2 && ct1024) go(k_cols_r1<T, SIGN, true, true, 1024>);
    else if (l2 && full) go(k_cols_r1<T, SIGN, true, true>);
    else if (l2) go(k_cols_r1<T, SIGN, true, false>);
    else if (CT4 && full && is_plan_4884(rp)) go(k_cols_r1<T, SIGN, false, true, CT4>);
    else if (full) go(k_cols_r1<T, SIGN, false, true>);
    else go(k_cols_r1<T, SIGN, false, false>);
  } else if (ct1024) {
    hipLaunchKernelGGL((k_cols<T, SIGN, 1024>), grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
  } else if (FftCfg<T>::COLE > 4 && rp.st[0].R == 4) {
    hipLaunchKernelGGL((k_cols<T, SIGN, 0, 4>), grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
  } else if (rp.st[0].R == 2) {
    hipLaunchKernelGGL((k_cols<T, SIGN, 0, 2>), grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
  } else {
    hipLaunchKernelGGL((k_cols<T, SIGN>), grid, block, lds, p.stream, p.field.as<C>(), cm, axis, rp, tw);
  }
  GENPK_LAUNCH_CHECK();
}

void r2c_zpass(Plan &p) {
  // a fresh deposit (no imported density) is folded while the z pass loads it
  const bool from_tiles = p.tiles_live && p.fstate != FieldState::Real;
  if (!from_tiles) tiles_to_field(p);
  GENPK_REQUIRE(from_tiles || p.fstate == FieldState::Real, "r2c needs a real-space density");
  if (p.prec == 4) r2c_z_impl<float>(p, from_tiles); else r2c_z_impl<double>(p, from_tiles);
  p.tiles_live = false;
  p.fstate = FieldState::Real;
}
void c2r_zpass(Plan &p) {
  if (p.prec == 4) c2r_z_impl<float>(p); else c2r_z_impl<double>(p);
}
void c2c_ypass(Plan &p, int sign) {
  if (p.prec == 4) {
    if (sign < 0) cols_impl<float, -1>(p, 1); else cols_impl<float, 1>(p, 1);
  } else {
    if (sign < 0) cols_impl<double, -1>(p, 1); else cols_impl<double, 1>(p, 1);
  }
}
void c2c_xpass(Plan &p, int sign) {
  if (p.prec == 4) {
    if (sign < 0) cols_impl<float, -1>(p, 0); else cols_impl<float, 1>(p, 0);
  } else {
    if (sign < 0) cols_impl<double, -1>(p, 0); else cols_impl<double, 1>(p, 0);
  }
}

void r2c(Plan &p) {
  r2c_zpass(p);
  c2c_ypass(p, -1);
  c2c_xpass(p, -1);
  p.fstate = FieldState::Spectrum;
}

void c2r(Plan &p) {
  GENPK_REQUIRE(p.fstate == FieldState::Spectrum, "c2r needs a spectrum");
  c2c_xpass(p, +1);
  c2c_ypass(p, +1);
  c2r_zpass(p);
  p.fstate = FieldState::Real;
}

}  // namespace genpk
