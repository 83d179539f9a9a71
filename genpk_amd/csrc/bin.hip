// CIC-deconvolved, log-binned power (the reference's powerspectrum(),
// powerspectrum.c:35-110) on gfx950.
//
// * Bin index: the reference computes floor(binsperunit * log(|k|)) per mode
//   (powerspectrum.c:38,66,75,84).  It depends only on the integer
//   q = |k|^2, so the host evaluates that exact FP64 formula once per q and
//   the kernels look the bin up (no device log, identical rounding).
// * Deconvolution: invwindow() squared (fieldize.cpp:125-133,
//   powerspectrum.c:68,77,86) = ((float)(wx*wy)*wz)^4 with per-axis float
//   factors; the factor tables are built on the host with the reference's
//   double formula and rounded to float as it does.
// * Weights: 1 on the planes kz = 0 (DC skipped) and kz = d/2, 2 elsewhere
//   (powerspectrum.c:61-89).
// * Counts and effective k depend only on (d, nrbins): computed once per plan.
// * Power: FP64 accumulation.  Each thread sums a run of modes that share a
//   bin in registers and adds to per-workgroup LDS bins only at bin changes;
//   per-workgroup partials are summed in a fixed order and normalised as in
//   powerspectrum.c:102-108.
// The fused kernel performs the last (x) FFT pass and bins the modes while
// they are still in LDS, so the spectrum is never written back.
#include "binlookup.h"
#include "fft_core.h"
#include "plan.h"

#include <cmath>
#include <vector>

namespace genpk {

int col_block(int prec, int64_t d, int64_t hz);

namespace {

// 16 waves per workgroup with 8 staged values per thread (MAXE): few enough
// registers (~80) for 16 resident waves per CU, twice the waves of 256 threads
// x 32 values (x pass + bin 4.0 -> 3.4 ms at 1024^3).
constexpr int BIN_THREADS = 1024;
constexpr int LDS_LIMIT = 160 * 1024;
constexpr int LGC_MAX = 3;
template <typename T> struct BinCfg;
template <> struct BinCfg<float> { static constexpr int ELEMS = 8192; static constexpr int MAXE = 8; };
template <> struct BinCfg<double> { static constexpr int ELEMS = 4096; static constexpr int MAXE = 4; };

__device__ __forceinline__ int64_t kval(int64_t n, int64_t d) { return n <= d / 2 ? n : n - d; }

// Mode count per |k|^2 = q over the half spectrum, weighted by the Hermitian
// weight h (1 on the planes kz = 0 and kz = d/2, else 2): with r2[a] the
// number of (x, y) array indices whose kx^2 + ky^2 = a,
//   qcnt[q] = sum_kz h(kz) r2[q - kz^2].
// Integer sums: the result is independent of scheduling.
__global__ void k_qcount(int64_t d, int64_t qmax, const uint32_t *__restrict__ r2, int64_t amax,
                         uint32_t *__restrict__ qcnt) {
  const int64_t hz = d / 2 + 1;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q <= qmax; q += (int64_t)gridDim.x * blockDim.x) {
    uint32_t s = 0;
    for (int64_t kz = 0; kz < hz && kz * kz <= q; kz++) {
      const int64_t a = q - kz * kz;
      if (a > amax) continue;
      s += ((kz == 0 || kz == d / 2) ? 1u : 2u) * r2[a];
    }
    qcnt[q] = s;
  }
}

// Accumulates one spectrum contribution run-by-run in registers.
struct RunAcc {
  int cur = -1;
  double v[3] = {0, 0, 0};
};

// bins: this lane's copy of the LDS bins, 1 << lgc copies side by side.  Lanes
// beside each other mostly end runs of one bin together, and their adds to
// one address are taken one after another: with up to eight copies, as the
// LDS has room, the x pass + bin takes 2.41 -> 2.23 ms at 1024^3 FP32, 0.74 ->
// 0.68 with two fields at 512^3, and leaving the adds out saves no more.
template <int NS>
__device__ __forceinline__ void run_flush(RunAcc &r, double *bins, int nrbins, int lgc) {
  if (r.cur >= 0) {
#pragma unroll
    for (int s = 0; s < NS; s++) atomicAdd(&bins[(s * nrbins + r.cur) << lgc], r.v[s]);
  }
}

template <int NS>
__device__ __forceinline__ void run_add(RunAcc &r, int b, const double *c, double *bins, int nrbins, int lgc) {
  if (b != r.cur) {
    run_flush<NS>(r, bins, nrbins, lgc);
    r.cur = b;
#pragma unroll
    for (int s = 0; s < NS; s++) r.v[s] = 0;
  }
#pragma unroll
  for (int s = 0; s < NS; s++) r.v[s] += c[s];
}

// Terms of a pair of modes of one weight, kx and -kx: their products add before
// the weight (the second pair of values 0 for a mode alone).
template <typename C, int NF>
__device__ __forceinline__ void pair_terms(const C &fa, const C &ga, const C &fb, const C &gb, double h, double dc,
                                           double *c) {
  auto dot = [](const C &u, const C &v) { return (double)u.x * (double)v.x + (double)u.y * (double)v.y; };
  c[0] = h * (dot(fa, fa) + dot(ga, ga)) * dc;
  if (NF == 2) {
    c[1] = h * (dot(fb, fb) + dot(gb, gb)) * dc;
    c[2] = h * (dot(fa, fb) + dot(ga, gb)) * dc;
  }
}

template <typename C, int NF>
__device__ __forceinline__ void mode_terms(const C &fa, const C &fb, double h, double dc, double *c) {
  const double ax = (double)fa.x, ay = (double)fa.y;
  if (NF == 1) {
    c[0] = h * (ax * ax + ay * ay) * dc;
  } else {
    const double bx = (double)fb.x, by = (double)fb.y;
    c[0] = h * (ax * ax + ay * ay) * dc;
    c[1] = h * (bx * bx + by * by) * dc;
    c[2] = h * (ax * bx + ay * by) * dc;
  }
}

struct BinGeom {
  int64_t d, hz;
  int nrbins;
  const int *q2bin;
  const int64_t *thr;
  const float *wtab;
  float lq;  // bin(q) ~ lq * log2(q): binsperunit * ln(2) / 2
};

// Fused final FFT pass along x + deconvolved binning.  NF fields (1: auto,
// 2: auto a, auto b and cross a.b*).  Persistent over column blocks.
//
// REG1 (a first stage of radix MAXE; one field: ping-pong buffers): the MAXE
// loaded elements of each thread below n * B / MAXE are the inputs of its butterfly
// in the first stage, which then runs from registers into buf2 (the threads
// above it load nothing).  Where the binning reads buf2 (an odd number of
// stages, or the last one left to the binning) the buffers swap roles
// between blocks, so no barrier comes before that stage.  FP32 360^3: 0.15 ->
// 0.11 ms; FP64 200^3 0.044 -> 0.036, 64^3 (three stages) 0.012 -> 0.010.  With
// two fields the first stage runs from registers in place: 0.58 -> 0.53 ms
// at 512^3 FP32.
//
// R2L (with REG1, a last stage of radix 2): the last stage runs in the
// binning, each thread pairing stage inputs j and j + n/2 into modes j and
// j + n/2 in registers.
//
// Binning: a thread takes the modes kx and -kx of a column together, which
// share |k|^2, so that a pair takes one bin lookup, one weight and one step of
// the run: x pass + bin 1.87 -> 1.61 ms at 1024^3 FP32, 0.113 -> 0.098 at
// 360^3; FP64 3.82 -> 3.60 at 1024^3, 0.036 -> 0.033 at 200^3.
//
// The registers hold the next block's loads while a block is binned: a
// spilled value read back there waits for all of them (one spilled register
// made the binning of a block 4.9 us instead of 2.7 at 1024^3 FP32), so each
// element's address is one column address plus a scalar multiple.
template <typename T, int NF, bool REG1, bool R2L = false, int CT = 0>
__global__ void __launch_bounds__(BIN_THREADS) k_xpass_bin(typename Cx<T>::C *__restrict__ fa,
                                                            typename Cx<T>::C *__restrict__ fb, BinGeom g, ColMap cm,
                                                            RadixPlan rp,
                                                            const typename Cx<T>::C *__restrict__ tw, int pp,
                                                            int lgc, double *__restrict__ part) {
  using C = typename Cx<T>::C;
  constexpr int NS = NF == 1 ? 1 : 3;
  static_assert(!R2L || REG1, "the radix-2 last stage in the binning needs the register first stage");
  extern __shared__ unsigned char lds_raw[];
  double *bins = reinterpret_cast<double *>(lds_raw);
  C *buf = reinterpret_cast<C *>(bins + (((NS * g.nrbins << lgc) + 1) & ~1));  // [NF][n][B], 16-byte aligned
  const int n = CT ? CT : rp.n;
  const int lgb = cm.lgb, B = 1 << lgb;
  // pp (one field): a second buffer lets the FFT stages alternate (one barrier each)
  C *buf2 = buf + (size_t)NF * n * B;
  C *stw = buf2 + (pp ? (size_t)n * B : 0);  // twiddles staged in LDS
  float *wt = reinterpret_cast<float *>(stw + n);  // deconvolution weights [d]
  int *thr32 = reinterpret_cast<int *>(wt + g.d);  // bin thresholds
  for (int i = threadIdx.x; i < n; i += BIN_THREADS) stw[i] = tw[i];
  for (int i = threadIdx.x; i < NS * g.nrbins << lgc; i += BIN_THREADS) bins[i] = 0;
  double *my_bins = bins + (threadIdx.x & ((1 << lgc) - 1));
  for (int i = threadIdx.x; i < g.d; i += BIN_THREADS) wt[i] = g.wtab[i];
  for (int i = threadIdx.x; i < bin_lds_slots(g.nrbins); i += BIN_THREADS) thr32[i] = (int)g.thr[i];
  const int64_t d = g.d, hz = g.hz;
  const int64_t estride = d * hz;
  const int64_t nblk = cm.nblk;
  // bin-phase mapping: thread -> column b, contiguous run of kx >= 0
  const int tpc = BIN_THREADS >> lgb;            // threads per column (B divides BIN_THREADS)
  const int my_b = threadIdx.x & (B - 1);
  const int half = n / 2, per = (half + tpc - 1) / tpc;
  const int e0 = (int)(threadIdx.x >> lgb) * per;
  // register-staged loads of column block v: all its global reads in flight
  // together; with REG1 at a stride of the first stage's butterfly count
  constexpr int MAXE = BinCfg<T>::MAXE;
  const int tot = n * B;
  const int lst = REG1 ? tot / MAXE : BIN_THREADS;
  const bool loader = !REG1 || (int)threadIdx.x < lst;
  C va[MAXE], vb[NF == 2 ? MAXE : 1];
  const int64_t my_off = (threadIdx.x >> lgb) * estride + my_b, qstep = (int64_t)(lst >> lgb) * estride;
  auto load = [&](int64_t v) {
    // a grid that is a multiple of the XCD count keeps v on this workgroup's XCD
    const ColMap::Block c = cm.at(xcd_block((uint32_t)v, (uint32_t)nblk));
    const int64_t off = (int64_t)c.outer * hz + c.kz0;
    const C *pa = fa + off + my_off, *pb = fb + off + my_off;
    const bool ok = loader && my_b < c.nb;
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
      const bool okq = ok && (REG1 || (int)threadIdx.x + q * lst < tot);
      va[q] = okq ? pa[q * qstep] : C{0, 0};
      if (NF == 2) vb[NF == 2 ? q : 0] = okq ? pb[q * qstep] : C{0, 0};
    }
  };
  // block v + gridDim.x loads into the registers while block v is binned
  // (their live range misses the FFT stages, where the registers peak)
  if ((int64_t)blockIdx.x < nblk) load(blockIdx.x);
  for (int64_t v = blockIdx.x; v < nblk; v += gridDim.x) {
    const ColMap::Block c = cm.at(xcd_block((uint32_t)v, (uint32_t)nblk));
    const int64_t y = c.outer;
    C *res = buf;
    if constexpr (REG1 && NF == 2) {
      __syncthreads();  // the previous block's binning is done with buf
      if (loader) {
        fft_first_regs<MAXE, -1>(va, buf, B, lgb, B, 1);
        fft_first_regs<MAXE, -1>(vb, buf + tot, B, lgb, B, 1);
      }
      __syncthreads();
      for (int s = 1; s < rp.nst; s++)
        for (int f = 0; f < 2; f++)
          fft_stage_r<-1, true, MAXE, false, C>(rp.st[s].R, buf + f * tot, buf + f * tot, B, lgb, B, 1, rp.st[s], stw);
    } else if constexpr (REG1) {
      if (loader) fft_first_regs<MAXE, -1>(va, buf2, B, lgb, B, 1);
      __syncthreads();
      if constexpr (CT == 1024 && R2L && MAXE == 8)
        res = lds_fft_ct<1024, 8, -1, true, MAXE, true, C, false, 8, 8>(buf2, buf, B, lgb, stw);
      else
        res = lds_fft_pp<-1, true, MAXE>(buf2, buf, rp, B, lgb, B, 1, stw, 1, R2L ? rp.nst - 1 : -1);
    } else {
      __syncthreads();  // the previous block's binning is done with buf
#pragma unroll
      for (int q = 0; q < MAXE; q++) {
        const int i = threadIdx.x + q * BIN_THREADS;
        if (i < tot) {
          buf[i] = va[q];
          if (NF == 2) buf[tot + i] = vb[NF == 2 ? q : 0];
        }
      }
      __syncthreads();
      if (NF == 1 && pp) {
        res = lds_fft_pp<-1, true, MAXE>(buf, buf2, rp, B, lgb, B, 1, stw);
      } else {
        lds_fft<-1, true, MAXE>(buf, rp, B, lgb, B, 1, stw);
        if (NF == 2) lds_fft<-1, true, MAXE>(buf + n * B, rp, B, lgb, B, 1, stw);
      }
    }
    if (v + gridDim.x < nblk) load(v + gridDim.x);
    if (my_b < c.nb) {
      const int kz = (int)c.kz0 + my_b;
      const int ky = (int)kval(y, d);
      const double h = (kz == 0 || kz == d / 2) ? 1.0 : 2.0;
      const int a = ky * ky + kz * kz;
      const float wy = wt[y], wz = wt[kz];
      RunAcc r;
      // the modes kx and -kx of a column share |k|^2, so bin and weight: they
      // are binned as one (see the kernel's comment)
      auto weight = [&](int kx) {
        const float gw = (wt[kx] * wy) * wz;  // the reference's ((wx*wy)*wz) in float
        double dc = (double)gw * (double)gw;
        return dc * dc;
      };
      auto bin_of = [&](int kx) { return bin_lds(max(a + kx * kx, 1), thr32, g.nrbins, g.lq); };
      const C zero = C{0, 0};
      if constexpr (R2L) {
        // the last stage: butterfly jj pairs stage inputs jj and jj + n/2
        // (the latter times w^jj) into modes jj and jj + n/2; with butterfly
        // n/2 - jj, whose modes are -jj - n/2 and -jj, a thread holds two
        // pairs.  Butterfly 0 (modes 0 and n/2, alone) goes with butterfly
        // n/4 (modes n/4 and -n/4).
        constexpr int HB = MAXE / 4;
        const int jb = (int)(threadIdx.x >> lgb) * HB;  // below n/4 exactly for the loaders
        C lo[HB], hi[HB], lo2[HB], hi2[HB];
        if (loader) {
          auto last_stage = [&](int jj, C &l, C &u) {
            const C a0 = res[(jj << lgb) + my_b];
            const C v1 = cmul(res[((jj + half) << lgb) + my_b], stw[jj]);
            l = cadd(a0, v1);
            u = csub(a0, v1);
          };
#pragma unroll
          for (int q = 0; q < HB; q++) {
            const int jj = jb + q;
            last_stage(jj, lo[q], hi[q]);
            last_stage(jj == 0 ? half / 2 : half - jj, lo2[q], hi2[q]);
          }
          int bq[2 * HB];
#pragma unroll
          for (int q = 0; q < HB; q++) {
            bq[q] = bin_of(jb + q);
            bq[q + HB] = bin_of(half - jb - q);
          }
          double t[3];
#pragma unroll
          for (int q = 0; q < HB; q++) {
            const int kx = jb + q;
            if (a != 0 || kx != 0) {
              pair_terms<C, NF>(lo[q], kx == 0 ? zero : hi2[q], zero, zero, h, weight(kx), t);
              run_add<NS>(r, bq[q], t, my_bins, g.nrbins, lgc);
            }
          }
#pragma unroll
          for (int q = 0; q < HB; q++) {
            const int kx = half - jb - q;
            pair_terms<C, NF>(hi[q], kx == half ? zero : lo2[q], zero, zero, h, weight(kx), t);
            run_add<NS>(r, bq[q + HB], t, my_bins, g.nrbins, lgc);
          }
          if (jb == 0) {
            pair_terms<C, NF>(lo2[0], hi2[0], zero, zero, h, weight(half / 2), t);
            run_add<NS>(r, bin_of(half / 2), t, my_bins, g.nrbins, lgc);
          }
        }
      } else {
        // this thread's run of at most MAXP pairs kx, -kx along x (per <= MAXP as
        // n * B <= BIN_THREADS * MAXE); kx = 0 goes with kx = n/2, both alone.
        // With one field all its LDS reads are issued first (two fields would
        // not fit the registers)
        constexpr int MAXP = MAXE / 2;
        constexpr bool BATCH = NF == 1;
        C ma[BATCH ? MAXP : 1], mb[BATCH ? MAXP : 1];
        auto at = [&](int e) { return (e << lgb) + my_b; };
        auto partner = [&](int e) { return e == 0 ? half : n - e; };
        if (BATCH) {
#pragma unroll
          for (int j = 0; j < MAXP; j++) {
            const int e = e0 + j;
            if (j < per && e < half) {
              ma[BATCH ? j : 0] = res[at(e)];
              mb[BATCH ? j : 0] = res[at(partner(e))];
            }
          }
        }
#pragma unroll
        for (int j = 0; j < MAXP; j++) {
          const int e = e0 + j;
          if (j < per && e < half) {
            const C f = BATCH ? ma[BATCH ? j : 0] : res[at(e)];
            const C fm = BATCH ? mb[BATCH ? j : 0] : res[at(partner(e))];
            const C u = NF == 2 ? res[tot + at(e)] : zero, um = NF == 2 ? res[tot + at(partner(e))] : zero;
            double t[3];
            if (a + e != 0) {
              pair_terms<C, NF>(f, e == 0 ? zero : fm, u, e == 0 ? zero : um, h, weight(e), t);
              run_add<NS>(r, bin_of(e), t, my_bins, g.nrbins, lgc);
            }
            if (e == 0) {
              pair_terms<C, NF>(fm, zero, um, zero, h, weight(half), t);
              run_add<NS>(r, bin_of(half), t, my_bins, g.nrbins, lgc);
            }
          }
        }
      }
      run_flush<NS>(r, my_bins, g.nrbins, lgc);
    }
    if constexpr (REG1 && NF == 1) {
      // the next first stage writes the buffer the binning did not read
      if (res == buf2) {
        C *t = buf;
        buf = buf2;
        buf2 = t;
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < NS * g.nrbins; i += BIN_THREADS) {
    double t = 0;
    for (int k = 0; k < 1 << lgc; k++) t += bins[(i << lgc) + k];
    part[(int64_t)blockIdx.x * NS * g.nrbins + i] = t;
  }
}

// Binning of stored spectra [d][d][hz] (no FFT).  A thread takes one (kx, kz)
// at STORED_RUN consecutive y: along y |k|^2 changes slowly, so the modes
// share few bins, and the lanes of a wave, kz fastest over the (kx, kz) pairs,
// read whole lines.  The next block's reads are in flight while one is
// binned.  Bound by HBM: 360^3 FP64 0.157 -> 0.076 ms (4.9 TB/s), 512^3 FP32
// 0.354 -> 0.150 (one wave per row with a contiguous run of kz per lane read
// every line several times, and looked bins up in global memory).  LT: window
// factors and bin thresholds from LDS, where they fit beside the bins.
constexpr int STORED_RUN = 8;
template <typename T, int NF, bool LT>
__global__ void __launch_bounds__(BIN_THREADS) k_bin_stored(const typename Cx<T>::C *__restrict__ fa,
                                                             const typename Cx<T>::C *__restrict__ fb, BinGeom g,
                                                             FastDiv fhz, FastDiv fny, int lgc,
                                                             double *__restrict__ part) {
  using C = typename Cx<T>::C;
  constexpr int NS = NF == 1 ? 1 : 3, RUN = STORED_RUN;
  extern __shared__ unsigned char lds_raw[];
  double *bins = reinterpret_cast<double *>(lds_raw);
  float *wt = reinterpret_cast<float *>(bins + ((size_t)NS * g.nrbins << lgc));
  int *thr32 = reinterpret_cast<int *>(wt + g.d);
  for (int i = threadIdx.x; i < NS * g.nrbins << lgc; i += BIN_THREADS) bins[i] = 0;
  if (LT) {
    for (int i = threadIdx.x; i < g.d; i += BIN_THREADS) wt[i] = g.wtab[i];
    for (int i = threadIdx.x; i < bin_lds_slots(g.nrbins); i += BIN_THREADS) thr32[i] = (int)g.thr[i];
  }
  __syncthreads();
  double *my_bins = bins + (threadIdx.x & ((1 << lgc) - 1));
  const int d = (int)g.d, hz = (int)g.hz;
  const int64_t estride = (int64_t)d * hz;
  // unit u: the runs of y from (u % ny) * RUN of pairs (u / ny) * BIN_THREADS on
  const uint32_t ny = fny.d, npair = (uint32_t)(d * hz);
  const uint32_t nunit = (npair + BIN_THREADS - 1) / BIN_THREADS * ny;
  C va[RUN], vb[NF == 2 ? RUN : 1];
  int kx, kz, y0, x;
  bool ok;
  auto load = [&](uint32_t u) {
    const uint32_t blk = fny.div(u), pair = blk * BIN_THREADS + threadIdx.x;
    y0 = (int)(u - blk * ny) * RUN;
    ok = pair < npair;
    x = (int)fhz.div(ok ? pair : 0u);
    kz = (int)((ok ? pair : 0u) - (uint32_t)x * hz);
    const int64_t at = x * estride + (int64_t)y0 * hz + kz;
#pragma unroll
    for (int q = 0; q < RUN; q++)
      if (ok && y0 + q < d) {
        va[q] = fa[at + (int64_t)q * hz];
        if (NF == 2) vb[NF == 2 ? q : 0] = fb[at + (int64_t)q * hz];
      }
  };
  uint32_t u = blockIdx.x;
  if (u < nunit) load(u);
  for (; u < nunit; u += gridDim.x) {
    C ma[RUN], mb[NF == 2 ? RUN : 1];
#pragma unroll
    for (int q = 0; q < RUN; q++) {
      ma[q] = va[q];
      if (NF == 2) mb[NF == 2 ? q : 0] = vb[NF == 2 ? q : 0];
    }
    const bool okc = ok;
    const int xc = x, kzc = kz, yc = y0;
    if (u + gridDim.x < nunit) load(u + gridDim.x);
    if (!okc) continue;
    kx = xc <= d / 2 ? xc : xc - d;
    const int a = kx * kx + kzc * kzc;
    const double h = (kzc == 0 || kzc == d / 2) ? 1.0 : 2.0;
    const float wx = LT ? wt[xc] : g.wtab[xc], wz = LT ? wt[kzc] : g.wtab[kzc];
    RunAcc r;
#pragma unroll
    for (int q = 0; q < RUN; q++) {
      const int y = yc + q, ky = y <= d / 2 ? y : y - d;
      const int qk = a + ky * ky;
      if (y < d && qk != 0) {
        const int b = LT ? bin_lds(qk, thr32, g.nrbins, g.lq) : g.q2bin[qk];
        const float gw = (wx * (LT ? wt[y] : g.wtab[y])) * wz;  // the reference's ((wx*wy)*wz) in float
        double dc = (double)gw * (double)gw;
        dc *= dc;
        double c[3];
        mode_terms<C, NF>(ma[q], NF == 2 ? mb[NF == 2 ? q : 0] : ma[q], h, dc, c);
        run_add<NS>(r, b, c, my_bins, g.nrbins, lgc);
      }
    }
    run_flush<NS>(r, my_bins, g.nrbins, lgc);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < NS * g.nrbins; i += BIN_THREADS) {
    double t = 0;
    for (int k = 0; k < 1 << lgc; k++) t += bins[(i << lgc) + k];
    part[(int64_t)blockIdx.x * NS * g.nrbins + i] = t;
  }
}

// Sum per-workgroup partials (fixed order) and normalise (powerspectrum.c:102-108).
// One workgroup per FIN_BINS bins and spectrum: FIN_SLICES threads per bin sum
// a contiguous range of the partials each, eight loads in flight, and the
// slices add in order.  (One thread per bin summing all G partials was a
// chain of G / 8 memory round trips in one to four workgroups: 14 us for 256
// partials, 26 for 512; this 4.)
constexpr int FIN_BINS = 16, FIN_SLICES = 16;
__global__ void __launch_bounds__(FIN_BINS * FIN_SLICES)
    k_bin_finish(int nrbins, int ns, int G, const double *__restrict__ part,
                             const int *__restrict__ count, const double *__restrict__ keffsum, double m_aa,
                             double m_bb, double m_ab, double *__restrict__ p_aa, double *__restrict__ p_bb,
                             double *__restrict__ p_ab, int *__restrict__ count_out, double *__restrict__ keffs_out) {
  __shared__ double sums[FIN_SLICES][FIN_BINS];
  const int lb = threadIdx.x % FIN_BINS, sl = threadIdx.x / FIN_BINS;
  const int b = blockIdx.x * FIN_BINS + lb, k = blockIdx.y;
  const int64_t gs = (int64_t)ns * nrbins;
  double acc = 0;
  if (b < nrbins) {
    const double *pk = part + (int64_t)k * nrbins + b;
    const int per = (G + FIN_SLICES - 1) / FIN_SLICES;
    const int g1 = min(G, (sl + 1) * per);
    int gi = sl * per;
    for (; gi + 8 <= g1; gi += 8) {
      double t[8];
#pragma unroll
      for (int q = 0; q < 8; q++) t[q] = pk[(int64_t)(gi + q) * gs];
#pragma unroll
      for (int q = 0; q < 8; q++) acc += t[q];
    }
    for (; gi < g1; gi++) acc += pk[(int64_t)gi * gs];
  }
  sums[sl][lb] = acc;
  __syncthreads();
  if (sl != 0 || b >= nrbins) return;
  double s = 0;
  for (int i = 0; i < FIN_SLICES; i++) s += sums[i][lb];
  const int c = count[b];
  double *out = k == 0 ? p_aa : k == 1 ? p_bb : p_ab;
  const double m = k == 0 ? m_aa : k == 1 ? m_bb : m_ab;
  if (out) {
    double v = 0;
    if (c) {
      v = s / m;
      v /= c;
    }
    out[b] = v;
  }
  if (k == 0) {
    if (count_out) count_out[b] = c;
    if (keffs_out) keffs_out[b] = c ? keffsum[b] / c : 0.0;
  }
}

}  // namespace

int num_cus() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    GENPK_HIP(hipGetDevice(&dev));
    GENPK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  }
  return cus;
}

// float(onedinvwindow(KVAL(k), d)) for k < d, the factor of fieldize.cpp:117-121
static double onedinvwindow_host(int64_t kx, int64_t n) {
  return kx ? M_PI * kx / (n * sin(M_PI * kx / (float)n)) : 1.0;
}

BinTables &bin_tables(Plan &p, int nrbins) {
  GENPK_REQUIRE(nrbins >= 1 && nrbins <= 8192, "nrbins must be in [1, 8192]");
  auto it = p.bins.find(nrbins);
  if (it != p.bins.end() && it->second->counts_ready) return *it->second;
  auto bt = std::make_unique<BinTables>();
  bt->nrbins = nrbins;
  const int64_t d = p.d, h = d / 2;
  const int64_t qmax = 3 * h * h;
  std::vector<int> tab((size_t)qmax + 1);
  // binsperunit and the per-mode index exactly as powerspectrum.c:38,66
  const double binsperunit = (nrbins - 1) / log(sqrt(3) * d / 2.0);
  bt->lq = (float)(binsperunit * log(2.0) / 2);
  tab[0] = -1;
  for (int64_t q = 1; q <= qmax; q++) {
    const double kk = sqrt((double)q);
    const int64_t b = (int64_t)floor(binsperunit * log(kk));
    GENPK_REQUIRE(b >= 0 && b < nrbins, "a mode falls outside [0, nrbins): nrbins too small for dims");
    tab[q] = (int)b;
  }
  bt->q2bin.ensure(tab.size() * 4);
  GENPK_HIP(hipMemcpy(bt->q2bin.ptr, tab.data(), tab.size() * 4, hipMemcpyHostToDevice));
  // thr[b] = smallest q >= 1 with bin(q) >= b (bins are non-decreasing in q)
  std::vector<int64_t> thr((size_t)nrbins + 1, qmax + 1);
  {
    int64_t q = 1;
    for (int b = 0; b <= nrbins; b++) {
      while (q <= qmax && tab[q] < b) q++;
      thr[b] = q;
    }
    for (int64_t q2 = 2; q2 <= qmax; q2++)
      GENPK_REQUIRE(tab[q2] >= tab[q2 - 1], "bin index not monotonic in |k|^2");
  }
  bt->thr.ensure(thr.size() * 8);
  GENPK_HIP(hipMemcpy(bt->thr.ptr, thr.data(), thr.size() * 8, hipMemcpyHostToDevice));
  if (!p.wtab.ptr) {
    std::vector<float> w(d);
    for (int64_t k = 0; k < d; k++) {
      const int64_t kv = k <= d / 2 ? k : k - d;
      w[k] = (float)onedinvwindow_host(kv, d);
    }
    p.wtab.ensure(d * 4);
    GENPK_HIP(hipMemcpy(p.wtab.ptr, w.data(), d * 4, hipMemcpyHostToDevice));
  }
  // counts and keffs, once: per-q mode counts on the device, then per-bin
  // sums on the host in ascending q (deterministic)
  {
    const int64_t amax = 2 * h * h;
    std::vector<uint32_t> r2((size_t)amax + 1, 0);
    for (int64_t x = 0; x < d; x++) {
      const int64_t kx = x <= h ? x : x - d;
      for (int64_t y = 0; y < d; y++) {
        const int64_t ky = y <= h ? y : y - d;
        r2[(size_t)(kx * kx + ky * ky)]++;
      }
    }
    DevBuf dr2, dq;
    dr2.ensure(r2.size() * 4);
    dq.ensure(((size_t)qmax + 1) * 4);
    GENPK_HIP(hipMemcpy(dr2.ptr, r2.data(), r2.size() * 4, hipMemcpyHostToDevice));
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(qmax + 1, 256), 65536);
    hipLaunchKernelGGL(k_qcount, dim3(grid), dim3(256), 0, p.stream, d, qmax, dr2.as<uint32_t>(), amax,
                       dq.as<uint32_t>());
    GENPK_LAUNCH_CHECK();
    std::vector<uint32_t> qcnt((size_t)qmax + 1);
    GENPK_HIP(hipMemcpyAsync(qcnt.data(), dq.ptr, qcnt.size() * 4, hipMemcpyDeviceToHost, p.stream));
    GENPK_HIP(hipStreamSynchronize(p.stream));
    std::vector<int64_t> cnt(nrbins, 0);
    std::vector<double> ke(nrbins, 0.0);
    for (int64_t q = 1; q <= qmax; q++) {
      if (!qcnt[q]) continue;
      cnt[tab[q]] += qcnt[q];
      ke[tab[q]] += (double)qcnt[q] * sqrt((double)q);
    }
    std::vector<int> cnt32(nrbins);
    for (int b = 0; b < nrbins; b++) {
      GENPK_REQUIRE(cnt[b] <= 2147483647, "a bin holds more than 2^31-1 modes");
      cnt32[b] = (int)cnt[b];
    }
    bt->count.ensure((size_t)nrbins * 4);
    bt->keffsum.ensure((size_t)nrbins * 8);
    GENPK_HIP(hipMemcpy(bt->count.ptr, cnt32.data(), (size_t)nrbins * 4, hipMemcpyHostToDevice));
    GENPK_HIP(hipMemcpy(bt->keffsum.ptr, ke.data(), (size_t)nrbins * 8, hipMemcpyHostToDevice));
  }
  bt->counts_ready = true;
  BinTables &ref = *bt;
  p.bins[nrbins] = std::move(bt);
  return ref;
}

const BinTables &built_bin_tables(const Plan &p, int nrbins) {
  GENPK_REQUIRE(nrbins >= 1 && nrbins <= 8192, "nrbins must be in [1, 8192]");
  auto it = p.bins.find(nrbins);
  GENPK_REQUIRE(it != p.bins.end() && it->second->counts_ready && p.wtab.ptr,
                "the bin tables of this nrbins are not built on the plan: call genpk_power or genpk_bin with it once "
                "first");
  return *it->second;
}

// Largest column block for the fused x-pass + bin kernel, 0 if none fits.
static int fused_block(int prec, int64_t d, int64_t hz, int nf, int ns, int nrbins) {
  const int csize = 2 * prec;
  const int elems = prec == 4 ? BinCfg<float>::ELEMS : BinCfg<double>::ELEMS;
  int B = col_block(prec, d, hz);
  while (B >= 1) {
    const int64_t lds = ((int64_t)nf * B + 1) * d * csize + (int64_t)((ns * nrbins + 1) & ~1) * 8 + d * 4 +
                        bin_lds_slots(nrbins) * 4;
    if (lds <= LDS_LIMIT && d * B <= elems && BIN_THREADS % B == 0) return B;
    B /= 2;
  }
  return 0;
}

template <typename T, int NF>
static size_t fused_lds(const Plan &a, int B, int nrbins, bool pp, int lgc = 0) {
  using C = typename Cx<T>::C;
  constexpr int NS = NF == 1 ? 1 : 3;
  return ((size_t)NF * B + (pp ? B : 0) + 1) * a.d * sizeof(C) + (size_t)(((NS * nrbins << lgc) + 1) & ~1) * 8 +
         (size_t)a.d * 4 + (size_t)bin_lds_slots(nrbins) * 4;
}

// Whether every thread holds at most one butterfly of plan rp's first stage
// (exactly: one each), as the REG1 instances need.
template <typename T>
static bool fused_reg1(const Plan &a, int B, const RadixPlan &rp, bool exactly) {
  const int64_t tot = a.d * B, cap = (int64_t)BIN_THREADS * BinCfg<T>::MAXE;
  return rp.st[0].R == BinCfg<T>::MAXE && (exactly ? tot == cap : tot <= cap);
}

// Persistent grid of the fused kernel: as many workgroups as stay resident
// (occupancy of this instance x CUs), at most one per column block.
template <typename T, int NF, bool REG1, bool R2L = false, int CT = 0>
static int fused_grid(const Plan &a, int B, int nrbins, bool pp, int lgc) {
  int per_cu = 0;
  GENPK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu,
                                                          reinterpret_cast<const void *>(&k_xpass_bin<T, NF, REG1, R2L, CT>),
                                                          BIN_THREADS, fused_lds<T, NF>(a, B, nrbins, pp, lgc)));
  const int64_t nblk = col_map(a.d, a.hz, B).nblk;
  return (int)std::max<int64_t>(1, std::min<int64_t>((int64_t)std::max(per_cu, 1) * num_cus(), nblk));
}

template <typename T, int NF, bool REG1, bool R2L = false, int CT = 0>
static void launch_fused(Plan &a, Plan *b, const BinTables &bt, const RadixPlan &rp, int B, bool pp,
                         int lgc, double *part, int G) {
  using C = typename Cx<T>::C;
  const C *tw = (a.prec == 4) ? (const C *)a.fft.tw_d_f32.ptr : (const C *)a.fft.tw_d_f64.ptr;
  BinGeom g{a.d, a.hz, bt.nrbins, bt.q2bin.as<int>(), bt.thr.as<int64_t>(), a.wtab.as<float>(), bt.lq};
  const size_t lds = fused_lds<T, NF>(a, B, bt.nrbins, pp, lgc);
  Stage st(a, "xpass_bin");
  hipLaunchKernelGGL((k_xpass_bin<T, NF, REG1, R2L, CT>), dim3(G), dim3(BIN_THREADS), lds, a.stream, a.field.as<C>(),
                     b ? b->field.as<C>() : (C *)nullptr, g, col_map(a.d, a.hz, B), rp, tw, pp ? 1 : 0, lgc, part);
  GENPK_LAUNCH_CHECK();
}

template <typename T, int NF>
static void launch_stored(Plan &a, Plan *b, const BinTables &bt, double *part, int G) {
  using C = typename Cx<T>::C;
  constexpr int NS = NF == 1 ? 1 : 3;
  BinGeom g{a.d, a.hz, bt.nrbins, bt.q2bin.as<int>(), bt.thr.as<int64_t>(), a.wtab.as<float>(), bt.lq};
  // tables and copies of the bins in half the LDS (two workgroups per CU),
  // the tables in all of it, or the bins alone
  const size_t tables = (size_t)a.d * 4 + (size_t)bin_lds_slots(bt.nrbins) * 4, one = (size_t)NS * bt.nrbins * 8;
  const bool lt = one + tables <= (size_t)LDS_LIMIT;
  int lgc = 0;
  while (lt && lgc < LGC_MAX && (one << (lgc + 1)) + tables <= (size_t)LDS_LIMIT / 2) lgc++;
  const FastDiv fhz((uint32_t)a.hz), fny((uint32_t)ceil_div(a.d, STORED_RUN));
  const size_t lds = (one << lgc) + (lt ? tables : 0);
  Stage st(a, "bin_stored");
  if (lt)
    hipLaunchKernelGGL((k_bin_stored<T, NF, true>), dim3(G), dim3(BIN_THREADS), lds, a.stream, a.field.as<C>(),
                       b ? b->field.as<C>() : (const C *)nullptr, g, fhz, fny, lgc, part);
  else
    hipLaunchKernelGGL((k_bin_stored<T, NF, false>), dim3(G), dim3(BIN_THREADS), lds, a.stream, a.field.as<C>(),
                       b ? b->field.as<C>() : (const C *)nullptr, g, fhz, fny, lgc, part);
  GENPK_LAUNCH_CHECK();
}

// Launch shape of the fused x pass + bin: the radix plan of its transforms
// (rp), column block B, ping-pong buffers (pp), the register first stage
// (reg1), the radix-2 last stage in the binning (r2l), compile-time stages
// for the n = 1024 plan 8, 8, 8, 2 (ct, with r2l), and the persistent grid G.
struct FusedShape {
  RadixPlan rp;
  int B = 0;
  bool pp = false, reg1 = false, r2l = false, ct = false;
  int lgc = 0;
  int G = 0;
};

template <typename T>
static int fused_grid_of(const Plan &a, bool cross, const FusedShape &s, int nrbins) {
  if (cross && s.reg1) return fused_grid<T, 2, true>(a, s.B, nrbins, false, s.lgc);
  if (cross) return fused_grid<T, 2, false>(a, s.B, nrbins, false, s.lgc);
  if (s.r2l && s.ct) return fused_grid<T, 1, true, true, 1024>(a, s.B, nrbins, s.pp, s.lgc);
  if (s.r2l) return fused_grid<T, 1, true, true>(a, s.B, nrbins, s.pp, s.lgc);
  if (s.reg1) return fused_grid<T, 1, true>(a, s.B, nrbins, s.pp, s.lgc);
  return fused_grid<T, 1, false>(a, s.B, nrbins, s.pp, s.lgc);
}

template <typename T>
static void launch_fused_of(Plan &a, Plan *b, const BinTables &bt, const FusedShape &s, double *part) {
  if (b && s.reg1) launch_fused<T, 2, true>(a, b, bt, s.rp, s.B, false, s.lgc, part, s.G);
  else if (b) launch_fused<T, 2, false>(a, b, bt, s.rp, s.B, false, s.lgc, part, s.G);
  else if (s.r2l && s.ct) launch_fused<T, 1, true, true, 1024>(a, b, bt, s.rp, s.B, s.pp, s.lgc, part, s.G);
  else if (s.r2l) launch_fused<T, 1, true, true>(a, b, bt, s.rp, s.B, s.pp, s.lgc, part, s.G);
  else if (s.reg1) launch_fused<T, 1, true>(a, b, bt, s.rp, s.B, s.pp, s.lgc, part, s.G);
  else launch_fused<T, 1, false>(a, b, bt, s.rp, s.B, s.pp, s.lgc, part, s.G);
}

static FusedShape fused_shape(const Plan &a, const Plan *b, int nrbins) {
  const int nf = b ? 2 : 1, ns = b ? 3 : 1;
  FusedShape s;
  s.B = fused_block(a.prec, a.d, a.hz, nf, ns, nrbins);
  GENPK_REQUIRE(s.B > 0, "fused x-pass does not fit in LDS for this size");
  const int B = s.B;
  // one field: ping-pong FFT buffers where the LDS has room for them
  s.pp = !b && (a.prec == 4 ? fused_lds<float, 1>(a, B, nrbins, true)
                            : fused_lds<double, 1>(a, B, nrbins, true)) <= (size_t)LDS_LIMIT;
  s.rp = a.rp_d;
  auto reg1 = [&](const RadixPlan &rp, bool exactly) {
    return (b || s.pp) && (a.prec == 4 ? fused_reg1<float>(a, B, rp, exactly) : fused_reg1<double>(a, B, rp, exactly));
  };
  s.reg1 = reg1(s.rp, false);
  if (!b && a.prec == 4) {
    // FP32 with a last stage of radix 2: that stage runs in the binning
    s.r2l = s.rp.nst % 2 == 0 && s.rp.st[s.rp.nst - 1].R == 2 && reg1(s.rp, true);
    // the plan's own ordering (the column passes') does not start with a
    // radix 8 and end with a radix 2 in an even number of stages, or its
    // columns leave threads idle: the x pass takes a plan of its length that
    // does, where the register first stage applies (512 = 8 8 8 -> 8 8 4 2:
    // 0.40 -> 0.30 ms at 512^3)
    const RadixPlan xp = s.r2l ? RadixPlan{} : radix_plan_8_to_2((int)a.d);
    if (!s.r2l && xp.nst > 0 && reg1(xp, false)) {
      s.rp = xp;
      s.reg1 = s.r2l = true;
    }
  }
  // compile-time stages where they pay: the FP32 register-first instance at
  // n = 1024 (the others would spill registers)
  s.ct = s.r2l && is_plan_8882(s.rp);
  const bool cross = b != nullptr;
  auto lds_of = [&](int lgc) {
    if (a.prec == 4)
      return cross ? fused_lds<float, 2>(a, B, nrbins, false, lgc) : fused_lds<float, 1>(a, B, nrbins, s.pp, lgc);
    return cross ? fused_lds<double, 2>(a, B, nrbins, false, lgc) : fused_lds<double, 1>(a, B, nrbins, s.pp, lgc);
  };
  while (s.lgc < LGC_MAX && lds_of(s.lgc + 1) <= (size_t)LDS_LIMIT) s.lgc++;
  s.G = a.prec == 4 ? fused_grid_of<float>(a, cross, s, nrbins) : fused_grid_of<double>(a, cross, s, nrbins);
  return s;
}

int64_t fused_partial_doubles(const Plan &a, const Plan *b, int nrbins) {
  return (int64_t)fused_shape(a, b, nrbins).G * (b ? 3 : 1) * nrbins;
}

void bin_spectra(Plan &a, Plan *b, int nrbins, bool fused_xpass, double *pow_aa, double *pow_bb, double *pow_ab,
                 int *count, double *keffs, double ma, double mb, double *scratch, size_t scratch_doubles) {
  if (b) {
    GENPK_REQUIRE(b->d == a.d && b->prec == a.prec, "cross spectrum needs plans of equal dims and precision");
    GENPK_REQUIRE(b->stream == a.stream, "cross spectrum needs plans on the same stream");
  }
  const BinTables &bt = scratch ? built_bin_tables(a, nrbins) : bin_tables(a, nrbins);
  const int nf = b ? 2 : 1, ns = b ? 3 : 1;
  int G = std::max(1, std::min<int>(2 * num_cus(), (int)std::min<int64_t>(a.d * a.d, 1 << 20)));
  double *part = nullptr;
  // per-workgroup partial bins: the caller's scratch, or the plan's buffer
  auto partials = [&](int64_t doubles) -> double * {
    if (!scratch) return static_cast<double *>(a.bin_part.ensure((size_t)doubles * 8));
    GENPK_REQUIRE((size_t)doubles <= scratch_doubles,
                  "the partial bins (" + std::to_string(doubles) + " doubles: workgroups x spectra x nrbins) exceed "
                  "the scratch of " + std::to_string(scratch_doubles) + " doubles: use fewer bins");
    return scratch;
  };
  if (fused_xpass) {
    GENPK_REQUIRE(a.fstate == FieldState::YDone && (!b || b->fstate == FieldState::YDone),
                  "fused binning needs fields after the z and y passes");
    const FusedShape fs = fused_shape(a, b, nrbins);
    G = fs.G;
    part = partials((int64_t)G * ns * nrbins);
    if (a.prec == 4)
      launch_fused_of<float>(a, b, bt, fs, part);
    else
      launch_fused_of<double>(a, b, bt, fs, part);
    // the field keeps the forward state after the z and y passes (an adjoint can start from it)
    a.fstate = FieldState::YDone;
    if (b) b->fstate = FieldState::YDone;
  } else {
    GENPK_REQUIRE(a.fstate == FieldState::Spectrum && (!b || b->fstate == FieldState::Spectrum),
                  "binning needs transformed fields");
    part = partials((int64_t)G * ns * nrbins);
    if (a.prec == 4) {
      if (b) launch_stored<float, 2>(a, b, bt, part, G); else launch_stored<float, 1>(a, b, bt, part, G);
    } else {
      if (b) launch_stored<double, 2>(a, b, bt, part, G); else launch_stored<double, 1>(a, b, bt, part, G);
    }
  }
  hipLaunchKernelGGL(k_bin_finish, dim3((unsigned)ceil_div(nrbins, FIN_BINS), (unsigned)ns),
                     dim3(FIN_BINS * FIN_SLICES), 0, a.stream, nrbins, ns, G, part,
                     bt.count.as<int>(), bt.keffsum.as<double>(), b ? ma * ma : ma * mb, mb * mb, ma * mb, pow_aa,
                     b ? pow_bb : (double *)nullptr, b ? pow_ab : (double *)nullptr, count, keffs);
  GENPK_LAUNCH_CHECK();
}

}  // namespace genpk
