// Hand-written adjoint of the auto power spectrum (no counterpart in the
// reference, which has no gradients).
//
// Forward: P_b = sum_{k in H, bin(k) = b} h_k g_k |F_k|^2 / (M^2 C_b), with
// F = r2c(rho), H the half spectrum, h_k the Hermitian weight, g_k the CIC
// deconvolution factor and C_b the mode count.  For lambda_b = dL/dP_b:
//   A_k      = 2 lambda_{b(k)} g_k F_k / (M^2 C_{b(k)}),  A_0 = 0
//   dL/drho  = c2r(A)   (unnormalised inverse; interior kz implicitly doubled)
//   dL/dm_j  = sum_c w_jc G(c)
//   dL/dx_ja = m_j (d/box) sum_c (dw_jc/du_a) G(c)
// where w_jc are the CIC weights of fieldize.cpp:77-84 and G = dL/drho.
//
// dL/drho is formed from whichever forward state the plan holds: a kept
// spectrum (weight, then the three inverse passes), the field after the
// forward z and y passes (left there by the fused power), or a deposit or
// density (z and y passes first).  In the last two cases the x pass runs
// forward FFT -> weight -> inverse FFT on each column block in LDS, so the
// spectrum is never written.  The gather visits the particles in tile order
// (the deposit's partition), reads dL/drho from a halo'd tile staged in LDS
// and writes the gradients in tile order; the sort's permutations then take
// them back to the particles' order.
#include "binlookup.h"
#include "fft_core.h"
#include "tilesort.h"

#include <algorithm>
#include <cmath>

namespace genpk {

int col_block(int prec, int64_t d, int64_t hz);

namespace {

constexpr int ADJ_THREADS = 1024;  // as the transform's column passes
constexpr int GATHER_THREADS = 512;
constexpr int GATHER_RUN = 32;
template <typename T> struct AdjCfg;
template <> struct AdjCfg<float> { static constexpr int MAXE = 8; };
template <> struct AdjCfg<double> { static constexpr int MAXE = 4; };

__device__ __forceinline__ int64_t kv(int64_t n, int64_t d) { return n <= d / 2 ? n : n - d; }

struct AdjWeight {
  const int *q2bin;
  const int *count;
  const double *lambda;
  const float *wtab;
  double inv_m2;
  const int64_t *thr;  // bin thresholds [nrbins + 1] (smallest q whose bin is >= b)
  int nrbins;
  float lq;            // bin(q) ~ lq * log2(q)
  // 2 lambda_b g_k / (M^2 C_b) of the mode at array indices (x, y, kz); 0 at k = 0
  __device__ __forceinline__ double at(int64_t x, int64_t y, int64_t kz, int64_t d) const {
    const int64_t kx = kv(x, d), ky = kv(y, d);
    const int64_t q = kx * kx + ky * ky + kz * kz;
    if (q == 0) return 0.0;
    const int b = q2bin[q];
    const int c = count[b];
    const float gw = (wtab[x] * wtab[y]) * wtab[kz];
    double g = (double)gw * (double)gw;
    g *= g;
    return c ? 2.0 * lambda[b] * g * inv_m2 / (double)c : 0.0;
  }
};

// The adjoint weight from LDS: the per-bin factors 2 lambda_b / (M^2 C_b), the
// window factors and the bin thresholds, so that a mode's weight costs no
// global read and no division.  Only the thresholds that bin_lds reads: at
// 1024^3 in FP64 the tables of 1024 bins then fit to the byte (adjoint x pass
// 8.83 -> 6.97 ms).
struct LdsWeight {
  double *sfb;  // [nrbins]
  float *swt;   // [d]
  int *sthr;    // [bin_lds_slots(nrbins)]
  int nrbins;
  float lq;
  static size_t bytes(int64_t d, int nrbins) {
    return (size_t)nrbins * 8 + (size_t)d * 4 + (size_t)bin_lds_slots(nrbins) * 4;
  }
  // fill the tables (16-byte aligned at) with the whole workgroup; no barrier
  __device__ __forceinline__ void init(void *at, const AdjWeight &w, int64_t d) {
    sfb = static_cast<double *>(at);
    swt = reinterpret_cast<float *>(sfb + w.nrbins);
    sthr = reinterpret_cast<int *>(swt + d);
    nrbins = w.nrbins;
    lq = w.lq;
    for (int i = threadIdx.x; i < w.nrbins; i += blockDim.x) {
      const int c = w.count[i];
      sfb[i] = c ? 2.0 * w.lambda[i] * w.inv_m2 / (double)c : 0.0;
    }
    for (int i = threadIdx.x; i < d; i += blockDim.x) swt[i] = w.wtab[i];
    for (int i = threadIdx.x; i < bin_lds_slots(w.nrbins); i += blockDim.x) sthr[i] = (int)w.thr[i];
  }
  // weight of array index xi along x of a column with a = ky^2 + kz^2 and
  // window factors wy, wz
  __device__ __forceinline__ double at(int xi, int n, int a, float wy, float wz) const {
    const int kx = xi <= n / 2 ? xi : xi - n;
    const int qk = a + kx * kx;
    const float gw = (swt[xi] * wy) * wz;  // the forward's ((wx*wy)*wz) in float
    double g = (double)gw * (double)gw;
    g *= g;
    const double s = g * sfb[bin_lds(max(qk, 1), sthr, nrbins, lq)];
    return qk ? s : 0.0;
  }
};

template <typename T>
__global__ void k_weight(typename Cx<T>::C *__restrict__ f, int64_t d, int64_t hz, AdjWeight w) {
  using C = typename Cx<T>::C;
  const int64_t total = d * d * hz;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t kz = i % hz;
    const int64_t row = i / hz;
    const double s = w.at(row / d, row % d, kz, d);
    const C v = f[i];
    f[i] = C{(T)((double)v.x * s), (T)((double)v.y * s)};
  }
}

// x pass of the adjoint on the field after the forward z and y passes:
// per column block (fixed y, B consecutive kz), forward length-d FFT along
// x, multiply by the adjoint weight, inverse FFT, store back.  One block
// per workgroup, the stages in place in one LDS buffer (k_adjoint_x_pp
// covers the usual shapes).  LW: the weight from LDS tables (where they fit
// beside the columns; with six global reads and a division per mode the pass
// took 0.27 ms at 360^3 FP32, with the tables 0.24, and
// 0.15 with all loads in flight together and no 64-bit division).
template <typename T, bool LW>
__global__ void __launch_bounds__(ADJ_THREADS) k_adjoint_x(typename Cx<T>::C *__restrict__ f, ColMap cm, RadixPlan rp,
                                                          const typename Cx<T>::C *__restrict__ tw, AdjWeight w) {
  using C = typename Cx<T>::C;
  constexpr int MAXE = AdjCfg<T>::MAXE;
  extern __shared__ unsigned char lds_raw[];
  C *buf = reinterpret_cast<C *>(lds_raw);  // [n][B]
  const int n = rp.n;
  const int lgb = cm.lgb, B = 1 << lgb;
  const int64_t d = cm.d, hz = cm.hz;
  const ColMap::Block c = cm.at(xcd_block(blockIdx.x, gridDim.x));
  const int64_t estride = d * hz;
  C *base = f + (int64_t)c.outer * hz + c.kz0;
  // ADJ_THREADS is a multiple of B: a thread's elements lie in one column
  const int b = threadIdx.x & (B - 1);
  const int tot = n * B;
  C v[MAXE];
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * ADJ_THREADS;
    v[q] = i < tot && b < c.nb ? base[(i >> lgb) * estride + b] : C{0, 0};
  }
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * ADJ_THREADS;
    if (i < tot) buf[i] = v[q];
  }
  C *stw = buf + tot;
  for (int i = threadIdx.x; i < n; i += ADJ_THREADS) stw[i] = tw[i];
  LdsWeight lw;
  if constexpr (LW) lw.init(stw + n, w, d);
  __syncthreads();
  lds_fft<-1, true, MAXE>(buf, rp, B, lgb, B, 1, stw);
  __syncthreads();
  if (b < c.nb) {
    const int ky = (int)kv(c.outer, d), kz = (int)c.kz0 + b;
    for (int i = threadIdx.x; i < tot; i += ADJ_THREADS) {
      const int e = i >> lgb;
      const double s = LW ? lw.at(e, n, ky * ky + kz * kz, lw.swt[c.outer], lw.swt[kz]) : w.at(e, c.outer, kz, d);
      const C a = buf[i];
      buf[i] = C{(T)((double)a.x * s), (T)((double)a.y * s)};
    }
  }
  __syncthreads();
  lds_fft<+1, true, MAXE>(buf, rp, B, lgb, B, 1, stw);
#pragma unroll
  for (int q = 0; q < MAXE; q++) {
    const int i = threadIdx.x + q * ADJ_THREADS;
    if (i < tot && b < c.nb) base[(i >> lgb) * estride + b] = buf[i];
  }
}

// k_adjoint_x for n * B = ADJ_THREADS * MAXE and a first radix of MAXE,
// persistent over the column blocks (v, v + gridDim.x, ...): the first
// stage runs from the loaded registers, the stages alternate between two
// LDS buffers (one barrier each), and the next block's loads are in flight
// during this block's inverse transform and stores.
// LW: the weight from LDS tables (LdsWeight).  LT (with LW, a last radix 2):
// the last forward stage runs in registers, each mode weighted before it is
// written.  (Compile-time stages for n = 1024 spill registers here: 5.2 -> 7.3
// ms at 1024^3, against 4.3 ms without.)
template <typename T, bool LT, bool LW>
__global__ void __launch_bounds__(ADJ_THREADS) k_adjoint_x_pp(typename Cx<T>::C *__restrict__ f, ColMap cm,
                                                             RadixPlan rp, const typename Cx<T>::C *__restrict__ tw,
                                                             AdjWeight w) {
  using C = typename Cx<T>::C;
  constexpr int MAXE = AdjCfg<T>::MAXE;
  extern __shared__ unsigned char lds_raw[];
  const int n = rp.n;
  const int lgb = cm.lgb, B = 1 << lgb;
  const int64_t d = cm.d, hz = cm.hz;
  const int tot = n * B;
  C *buf = reinterpret_cast<C *>(lds_raw);  // [n][B]
  C *buf2 = buf + tot;
  C *stw = buf2 + tot;
  for (int i = threadIdx.x; i < n; i += ADJ_THREADS) stw[i] = tw[i];
  LdsWeight lw;
  if constexpr (LW) lw.init(stw + n, w, d);
  const int64_t estride = d * hz;
  const int64_t nblk = cm.nblk;
  const int b = threadIdx.x & (B - 1);
  C v[MAXE];
  // column block vb's loads: the inputs of this thread's first-stage butterfly
  // (a grid that is a multiple of the XCD count keeps vb on this workgroup's XCD)
  auto load = [&](int64_t vb) {
    const ColMap::Block c = cm.at(xcd_block((uint32_t)vb, (uint32_t)nblk));
    const C *src = f + (int64_t)c.outer * hz + c.kz0;
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      const int i = threadIdx.x + q * ADJ_THREADS;
      v[q] = b < c.nb ? src[(i >> lgb) * estride + b] : C{0, 0};
    }
  };
  if ((int64_t)blockIdx.x < nblk) load(blockIdx.x);
  for (int64_t vb = blockIdx.x; vb < nblk; vb += gridDim.x) {
    const ColMap::Block c = cm.at(xcd_block((uint32_t)vb, (uint32_t)nblk));
    const int64_t y = c.outer;
    C *base = f + y * hz + c.kz0;
    // the previous block's stores have read their buffer before this barrier
    fft_first_regs<MAXE, -1>(v, buf2, B, lgb, B, 1);
    __syncthreads();
    C *res;
    if (LT) {
      // the last forward stage (radix 2) and the adjoint weight in registers:
      // butterfly jj pairs stage inputs jj and jj + n/2 (the latter times
      // w^jj) into modes jj and jj + n/2, written weighted to the other buffer
      C *x = lds_fft_pp<-1, true, MAXE>(buf2, buf, rp, B, lgb, B, 1, stw, 1, rp.nst - 1);
      res = x == buf ? buf2 : buf;
      constexpr int HB = MAXE / 2;
      const int half = n / 2;
      const int jb = (threadIdx.x >> lgb) * HB;
      const int kz = (int)c.kz0 + b, ky = (int)kv(y, d);
      const int a = ky * ky + kz * kz;
      const float wy = lw.swt[y], wz = lw.swt[min(kz, (int)d - 1)];
#pragma unroll
      for (int q = 0; q < HB; q++) {
        const int jj = jb + q;
        const C a0 = x[jj * B + b];
        const C v1 = cmul(x[(jj + half) * B + b], stw[jj]);
        C o0 = cadd(a0, v1), o1 = csub(a0, v1);
        if (b < c.nb) {
          const double s0 = lw.at(jj, n, a, wy, wz);
          const double s1 = lw.at(jj + half, n, a, wy, wz);
          o0 = C{(T)((double)o0.x * s0), (T)((double)o0.y * s0)};
          o1 = C{(T)((double)o1.x * s1), (T)((double)o1.y * s1)};
        }
        res[jj * B + b] = o0;
        res[(jj + half) * B + b] = o1;
      }
    } else {
      res = lds_fft_pp<-1, true, MAXE>(buf2, buf, rp, B, lgb, B, 1, stw, 1);
      const int kz = (int)c.kz0 + b, ky = (int)kv(y, d);
      for (int i = threadIdx.x; i < tot; i += ADJ_THREADS) {
        const int e = i >> lgb;
        if (b < c.nb) {
          const double s = LW ? lw.at(e, n, ky * ky + kz * kz, lw.swt[y], lw.swt[kz]) : w.at(e, y, kz, d);
          const C a = res[i];
          res[i] = C{(T)((double)a.x * s), (T)((double)a.y * s)};
        }
      }
    }
    __syncthreads();
    // the next block's loads (v is free since the first stage)
    if (vb + gridDim.x < nblk) load(vb + gridDim.x);
    res = lds_fft_pp<+1, true, MAXE>(res, res == buf ? buf2 : buf, rp, B, lgb, B, 1, stw);
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      const int i = threadIdx.x + q * ADJ_THREADS;
      const int e = i >> lgb;
      if (b < c.nb) base[e * estride + b] = res[i];
    }
  }
}

struct GatherParams {
  KeyGeom kg;
  int HY, HZ;
  int64_t cells;
  TileList list;
  int64_t rowlen;
  double mass;
  FastDiv fhz, fhy;
  FastDiv fntz, fnty;  // tile index -> (tx, ty, tz)
};

// One workgroup per work item of the tile order: stage the halo'd tile of
// G = dL/drho in LDS, then the gradients of the item's records, written at
// the records' own pool slots as (dL/dx, dL/dy, dL/dz[, dL/dm]):
// coalesced.
template <typename T, int NM, int GM>
__global__ void __launch_bounds__(GATHER_THREADS) k_gather_tiles(const T *__restrict__ G, const float *__restrict__ rec,
                                                                 const uint4 *__restrict__ items,
                                                                 const uint32_t *__restrict__ blist,
                                                                 const uint32_t *__restrict__ counts,
                                                                 GatherParams P, float *__restrict__ out) {
  constexpr int RW = 3 + NM;
  constexpr int RWO = 3 + GM;
  extern __shared__ unsigned char lds_raw[];
  T *g = reinterpret_cast<T *>(lds_raw);
  // items in runs of GATHER_RUN per XCD (workgroup id mod 8), the XCDs' runs
  // side by side: consecutive tiles along z share the lines at their z edges
  // in G, which one L2 then serves to both (the grid is a multiple of
  // 8 * GATHER_RUN; ids past the last item return)
  const uint32_t xcd = blockIdx.x % NUM_XCD, slot = blockIdx.x / NUM_XCD;
  const uint32_t item = ((slot / GATHER_RUN) * NUM_XCD + xcd) * GATHER_RUN + slot % GATHER_RUN;
  const uint32_t nsplit = counts[1];
  if (item >= nsplit + counts[2]) return;
  ItemRange ir;
  item_range(items, nsplit, P.list.max_parts, item, ir);
  if (ir.lb >= ir.le) return;
  const int64_t k = ir.k;
  const int ntz = P.kg.ntz, nty = P.kg.nty, d = P.kg.d;
  const uint32_t kxy = P.fntz.div((uint32_t)k), kx = P.fnty.div(kxy);
  const int tz = (int)((uint32_t)k - kxy * (uint32_t)ntz);
  const int ty = (int)(kxy - kx * (uint32_t)nty);
  const int tx = (int)kx;
  const int ox = tx << P.kg.sx, oy = ty << P.kg.sy, oz = tz << P.kg.sz;
  // four loads in flight per thread while staging, and four records while
  // gathering: the next batch's records, through the list entries loaded one
  // batch earlier, load while this batch is worked on (the first ones during
  // the staging)
  constexpr int UNR = 4;
  const int lg = P.list.lg;
  // a thread's place in the blocks is the same in every batch (blocks of at
  // most 256 slots divide the 512 threads)
  const uint32_t in = threadIdx.x & ((1u << lg) - 1), te = threadIdx.x >> lg, eu = (uint32_t)GATHER_THREADS >> lg;
  const uint32_t ents = ir.le - ir.lb;
  float rr[UNR][RW], nx[UNR][RW];
  uint32_t ent[UNR], at_slot[UNR], nslot[UNR];
  uint32_t em = 0, vm = 0, nvm = 0;
  auto load_entries = [&](uint32_t rel) {
    em = 0;
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const uint32_t e = rel + u * eu + te;
      if (e < ents) {
        ent[u] = blist[ir.lb + e];
        em |= 1u << u;
      }
    }
  };
  auto load_records = [&]() {
    nvm = 0;
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      if (((em >> u) & 1u) && in < P.list.fill(ent[u])) {
        nvm |= 1u << u;
        nslot[u] = P.list.slot0(ent[u]) + in;
#pragma unroll
        for (int q = 0; q < RW; q++) nx[u][q] = rec[(int64_t)nslot[u] * RW + q];
      }
    }
  };
  load_entries(0);
  load_records();
  load_entries(UNR * eu);
  for (int c0 = threadIdx.x; c0 < (int)P.cells; c0 += GATHER_THREADS * UNR) {
    T t[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const int c = c0 + u * GATHER_THREADS;
      if (c < (int)P.cells) {
        const int row = (int)P.fhz.div((uint32_t)c);
        const int lz = c - row * P.HZ;
        const int lx = (int)P.fhy.div((uint32_t)row);
        const int ly = row - lx * P.HY;
        int x = ox + lx, y = oy + ly, z = oz + lz;
        if (x >= d) x -= d;
        if (y >= d) y -= d;
        if (z >= d) z -= d;
        t[u] = G[((int64_t)x * d + y) * P.rowlen + z];
      }
    }
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const int c = c0 + u * GATHER_THREADS;
      if (c < (int)P.cells) g[c] = t[u];
    }
  }
  __syncthreads();
  const int sy = P.HZ, sx = P.HY * P.HZ;
  const double units = P.kg.units;
  for (uint32_t e0 = 0; e0 < ents; e0 += UNR * eu) {
    vm = nvm;
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      at_slot[u] = nslot[u];
#pragma unroll
      for (int q = 0; q < RW; q++) rr[u][q] = nx[u][q];
    }
    load_records();
    load_entries(e0 + 2 * UNR * eu);
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      if (!((vm >> u) & 1u)) continue;
      const float *r = rr[u];
      double fx, fy, fz;
      const int lx = cell_of(r[0], units, d, fx) - ox;
      const int ly = cell_of(r[1], units, d, fy) - oy;
      const int lz = cell_of(r[2], units, d, fz) - oz;
      if ((unsigned)lx >= (unsigned)P.kg.TX || (unsigned)ly >= (unsigned)P.kg.TY || (unsigned)lz >= (unsigned)P.kg.TZ)
        continue;  // cannot happen for records of this tile; guards the LDS bounds
      const int at = lx * sx + ly * sy + lz;
      const double g000 = (double)g[at], g001 = (double)g[at + 1];
      const double g100 = (double)g[at + sx], g101 = (double)g[at + sx + 1];
      const double g010 = (double)g[at + sy], g011 = (double)g[at + sy + 1];
      const double g110 = (double)g[at + sx + sy], g111 = (double)g[at + sx + sy + 1];
      // corners (bx, by, bz); weights (1-f or f) per axis
      const double ex = 1.0 - fx, ey = 1.0 - fy, ez = 1.0 - fz;
      // interpolate along z first
      const double a00 = ez * g000 + fz * g001, a10 = ez * g100 + fz * g101;
      const double a01 = ez * g010 + fz * g011, a11 = ez * g110 + fz * g111;
      const double dgx = ey * (a10 - a00) + fy * (a11 - a01);
      const double dgy = ex * (a01 - a00) + fx * (a11 - a10);
      const double b00 = ex * ey, b10 = fx * ey, b01 = ex * fy, b11 = fx * fy;
      const double dgz = b00 * (g001 - g000) + b10 * (g101 - g100) + b01 * (g011 - g010) + b11 * (g111 - g110);
      const double gm = b00 * a00 + b10 * a10 + b01 * a01 + b11 * a11;
      const double m = NM ? (double)r[3] : P.mass;
      const double s = m * units;
      float *o = out + (int64_t)at_slot[u] * RWO;
      o[0] = (float)(dgx * s);
      o[1] = (float)(dgy * s);
      o[2] = (float)(dgz * s);
      if (GM) o[3] = (float)gm;
    }
  }
}

// Gradients back to the particles' input order: particle j sits at sorted
// position perm2[perm1[j]] (perm1 alone after a one-pass sort).  Reads of
// perm1 and writes are coalesced; the two lookups are random reads, which
// cost far less than scattered partial-line writes.  Each XCD (workgroup id
// mod 8) takes runs of UNP_RUN consecutive blocks, the eight XCDs' runs side
// by side: a workgroup of the first pass writes to a range of slots of its own,
// so a run's particles of one bucket sit together in perm2 and its lines are
// fetched by one L2, while all XCDs stay within one window of the particles.
// The grid is a multiple of 8 * UNP_RUN.
constexpr int UNP_RUN = 256;
template <int RWO, int TWO>
__global__ void k_unpermute(const float *__restrict__ rec, const uint32_t *__restrict__ perm1,
                            const uint32_t *__restrict__ perm2, int64_t n, float *__restrict__ gpos,
                            float *__restrict__ gmass) {
  const uint32_t x = blockIdx.x % NUM_XCD, slot = blockIdx.x / NUM_XCD;
  const int64_t lb = ((int64_t)(slot / UNP_RUN) * NUM_XCD + x) * UNP_RUN + slot % UNP_RUN;
  for (int64_t j = lb * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    int64_t at = perm1[j];
    if (TWO) at = perm2[at];
    const float *r = rec + at * RWO;
    gpos[3 * j + 0] = r[0];
    gpos[3 * j + 1] = r[1];
    gpos[3 * j + 2] = r[2];
    if (RWO == 4) gmass[j] = r[3];
  }
}

AdjWeight adj_weight(Plan &p, int nrbins, const double *lambda, double m) {
  const BinTables &bt = bin_tables(p, nrbins);
  AdjWeight w;
  w.q2bin = bt.q2bin.as<int>();
  w.count = bt.count.as<int>();
  w.lambda = lambda;
  w.wtab = p.wtab.as<float>();
  w.inv_m2 = 1.0 / (m * m);
  w.thr = bt.thr.as<int64_t>();
  w.nrbins = bt.nrbins;
  w.lq = bt.lq;
  return w;
}

template <typename T>
void adjoint_x_impl(Plan &p, const AdjWeight &w) {
  using C = typename Cx<T>::C;
  const int B = col_block(p.prec, p.d, p.hz);
  const ColMap cm = col_map(p.d, p.hz, B);
  const C *tw = (p.prec == 4) ? (const C *)p.fft.tw_d_f32.ptr : (const C *)p.fft.tw_d_f64.ptr;
  const int64_t tot = p.d * B;
  GENPK_REQUIRE(tot <= (int64_t)AdjCfg<T>::MAXE * ADJ_THREADS, "adjoint x pass: column block too large");
  Stage st(p, "adjoint_x");
  const size_t lds_w = LdsWeight::bytes(p.d, w.nrbins), lds_pp = (size_t)(2 * tot + p.d) * sizeof(C), cap = 160 * 1024;
  // the register first stage takes a plan of its length with a first radix of
  // MAXE; FP32: one that also ends in a radix 2, where the plan's own (the
  // column passes') does not (512 = 8 8 8 -> 8 8 4 2: 0.56 -> 0.48 ms at 512^3)
  RadixPlan rp = p.rp_d;
  auto last2 = [](const RadixPlan &r) { return r.st[r.nst - 1].R == 2; };
  if (sizeof(T) == 4 && !(rp.st[0].R == 8 && last2(rp))) {
    const RadixPlan xp = radix_plan_8_to_2((int)p.d);
    if (xp.nst > 0) rp = xp;
  }
  const bool pp = rp.st[0].R == AdjCfg<T>::MAXE && tot == (int64_t)ADJ_THREADS * AdjCfg<T>::MAXE && lds_pp <= cap;
  const bool lw = lds_pp + lds_w <= cap, lt = lw && last2(rp);
  if (pp) {
    // persistent: as many workgroups as stay resident, at most one per column block
    // (4.3 ms at 1024^3 against 5.2 ms for one workgroup per block)
    const void *fn = lt   ? reinterpret_cast<const void *>(&k_adjoint_x_pp<T, true, true>)
                     : lw ? reinterpret_cast<const void *>(&k_adjoint_x_pp<T, false, true>)
                          : reinterpret_cast<const void *>(&k_adjoint_x_pp<T, false, false>);
    const size_t lds = lw ? lds_pp + lds_w : lds_pp;
    int per_cu = 0;
    GENPK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, ADJ_THREADS, lds));
    const int64_t most = std::min<int64_t>((int64_t)std::max(per_cu, 1) * num_cus(), (int64_t)cm.nblk);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)std::max<int64_t>(1, most)), dim3(ADJ_THREADS), lds, p.stream,
                         p.field.as<C>(), cm, rp, tw, w);
    };
    if (lt) go(k_adjoint_x_pp<T, true, true>);
    else if (lw) go(k_adjoint_x_pp<T, false, true>);
    else go(k_adjoint_x_pp<T, false, false>);
  } else {
    const size_t lds = (size_t)(tot + p.d) * sizeof(C);
    auto go = [&](auto kernel, size_t bytes) {
      hipLaunchKernelGGL(kernel, dim3(cm.nblk), dim3(ADJ_THREADS), bytes, p.stream, p.field.as<C>(), cm, p.rp_d, tw, w);
    };
    if (lds + lds_w <= cap) go(k_adjoint_x<T, true>, lds + lds_w);
    else go(k_adjoint_x<T, false>, lds);
  }
  GENPK_LAUNCH_CHECK();
}

template <typename T, int NM, int GM>
void gather_impl(Plan &p, const KeyGeom &kg, const TileOrder &o, double mass, float *out) {
  const TileGeom &tg = p.tg;
  GatherParams P;
  P.kg = kg;
  P.HY = tg.HY;
  P.HZ = tg.HZ;
  P.cells = tg.cells;
  P.list = o.list;
  P.rowlen = p.rowlen;
  P.mass = mass;
  P.fhz = FastDiv((uint32_t)tg.HZ);
  P.fhy = FastDiv((uint32_t)tg.HY);
  P.fntz = FastDiv((uint32_t)tg.ntz);
  P.fnty = FastDiv((uint32_t)tg.nty);
  const int64_t grid = ceil_div(o.list.max_items, 8 * GATHER_RUN) * 8 * GATHER_RUN;
  hipLaunchKernelGGL((k_gather_tiles<T, NM, GM>), dim3((unsigned)grid), dim3(GATHER_THREADS),
                     (size_t)tg.cells * sizeof(T), p.stream, p.field.as<const T>(), o.rec, o.list.items, o.list.blist,
                     o.list.counts, P, out);
  GENPK_LAUNCH_CHECK();
}

}  // namespace

void adjoint_density(Plan &p, int nrbins, const double *lambda, double m) {
  GENPK_REQUIRE(m != 0, "total mass must be nonzero");
  GENPK_REQUIRE(lambda != nullptr, "null lambda");
  const AdjWeight w = adj_weight(p, nrbins, lambda, m);
  if (!p.tiles_live && p.fstate == FieldState::Spectrum) {
    // kept spectrum: weight every mode, then the inverse passes
    const int64_t total = p.d * p.d * p.hz;
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(total, 256), 65536);
    {
      Stage st(p, "adjoint_weight");
      if (p.prec == 4)
        hipLaunchKernelGGL(k_weight<float>, dim3(grid), dim3(256), 0, p.stream, p.field.as<float2>(), p.d, p.hz, w);
      else
        hipLaunchKernelGGL(k_weight<double>, dim3(grid), dim3(256), 0, p.stream, p.field.as<double2>(), p.d, p.hz, w);
      GENPK_LAUNCH_CHECK();
    }
    c2r(p);
    return;
  }
  if (p.tiles_live || p.fstate == FieldState::Real) {
    // forward density (deposit or imported): forward z and y passes first
    r2c_zpass(p);
    c2c_ypass(p, -1);
    p.fstate = FieldState::YDone;
  }
  GENPK_REQUIRE(p.fstate == FieldState::YDone,
                "adjoint needs the forward spectrum, the forward density or the state left by the fused power");
  if (p.prec == 4) adjoint_x_impl<float>(p, w); else adjoint_x_impl<double>(p, w);
  c2c_ypass(p, +1);
  c2r_zpass(p);
  p.fstate = FieldState::Real;
}

void adjoint_gather(Plan &p, double boxsize, int64_t n, const float *pos, const float *masses, double mass,
                    float *grad_pos, float *grad_mass) {
  GENPK_REQUIRE(p.fstate == FieldState::Real && !p.tiles_live,
                "gather needs dL/drho in the plan (run the adjoint first)");
  GENPK_REQUIRE(boxsize > 0 && std::isfinite(boxsize), "boxsize must be positive and finite");
  GENPK_REQUIRE(n >= 0, "negative particle count");
  if (n == 0) return;
  GENPK_REQUIRE(pos && grad_pos, "null positions or gradient output");
  const int64_t cap = (int64_t)1 << 31;
  const RetainedOrder &r = p.order;
  const bool reuse = r.valid && r.pos == pos && r.masses == masses && r.n == n && r.boxsize == boxsize &&
                     r.to.has_perm;
  const KeyGeom kg = key_geom(p, boxsize);
  int64_t done = 0;
  do {
    const int64_t m = std::min(n - done, cap);
    const float *mp = masses ? masses + done : nullptr;
    TileOrder o;
    if (reuse) {
      o = r.to;
    } else {
      o = sort_by_tile(p, kg, m, pos + 3 * done, mp, true, false);
      p.order.valid = n <= cap;
      p.order.pos = pos;
      p.order.masses = masses;
      p.order.n = n;
      p.order.boxsize = boxsize;
      p.order.mass = mass;
      p.order.every_tile = false;
      p.order.to = o;
    }
    float *gp = grad_pos + 3 * done;
    float *gmp = grad_mass ? grad_mass + done : nullptr;
    // output records go to the record buffer that does not hold the sorted records
    float *out = (o.rec == p.recA.as<float>()) ? p.recB.as<float>() : p.recA.as<float>();
    const int gm = grad_mass ? 1 : 0;
    {
      Stage st(p, "adjoint_gather");
      if (p.prec == 4) {
        if (masses)
          gm ? gather_impl<float, 1, 1>(p, kg, o, mass, out) : gather_impl<float, 1, 0>(p, kg, o, mass, out);
        else
          gm ? gather_impl<float, 0, 1>(p, kg, o, mass, out) : gather_impl<float, 0, 0>(p, kg, o, mass, out);
      } else {
        if (masses)
          gm ? gather_impl<double, 1, 1>(p, kg, o, mass, out) : gather_impl<double, 1, 0>(p, kg, o, mass, out);
        else
          gm ? gather_impl<double, 0, 1>(p, kg, o, mass, out) : gather_impl<double, 0, 0>(p, kg, o, mass, out);
      }
    }
    {
      Stage st(p, "adjoint_unpermute");
      const unsigned grid = (unsigned)(ceil_div(std::min<int64_t>(ceil_div(m, 256), 1 << 22), 8 * UNP_RUN) * 8 * UNP_RUN);
      const bool two = o.perm2 != nullptr;
      if (gm && two)
        hipLaunchKernelGGL((k_unpermute<4, 1>), dim3(grid), dim3(256), 0, p.stream, out, o.perm1, o.perm2, m, gp, gmp);
      else if (gm)
        hipLaunchKernelGGL((k_unpermute<4, 0>), dim3(grid), dim3(256), 0, p.stream, out, o.perm1, o.perm2, m, gp, gmp);
      else if (two)
        hipLaunchKernelGGL((k_unpermute<3, 1>), dim3(grid), dim3(256), 0, p.stream, out, o.perm1, o.perm2, m, gp, gmp);
      else
        hipLaunchKernelGGL((k_unpermute<3, 0>), dim3(grid), dim3(256), 0, p.stream, out, o.perm1, o.perm2, m, gp, gmp);
      GENPK_LAUNCH_CHECK();
    }
    done += m;
  } while (done < n);
}

}  // namespace genpk
