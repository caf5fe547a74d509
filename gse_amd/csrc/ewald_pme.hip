// Comparators beside the GSE path, on the same device infrastructure:
//
// SPME reciprocal space (the reference's cuda/CudaPMERecip.cu, order 4/6/8):
//   k_pme_bin       particles into bins of 8^3 cells, max |q| and the
//                   rejected-particle count of one call
//   k_pme_spread    B-spline spread of one bin into an int64 fixed-point
//                   brick in LDS (one lane per (x, y) spline offset, a loop
//                   over z; the same exponent rule as the GSE spread, so the
//                   grid is bit-identical for any particle order); the GSE
//                   path's k_brick_reduce sums and converts the bricks
//   k_pme_scalar_sum  the spectrum times the SPME kernel with FP64 energy and
//                   virial partial sums per workgroup (fixed order)
//   k_pme_finalize  energy and the 3x3 virial from the partial sums
//   k_pme_gather    energy gradient per particle: one lane group per particle
//                   (16 lanes for order 4, a wave for 6 and 8), lanes on the
//                   (x, y) offsets, a loop over z, a fixed-order butterfly
// The spline position, weights and moduli follow CudaPMERecip.cu:266-327,
// :436-588, :946-1256 and :1612-1890 term for term.
//
// Ewald direct space (CpuEwaldDirect.cpp:45-131):
//   k_ew_cell_count / k_ew_scan / k_ew_scatter / k_ew_sort
//                   particles into cells, each cell's list in ascending
//                   particle index (deterministic order); partial sums of q^2
//   k_ew_force      one wave per particle: candidates of the cells
//                   within reach pass a 32-bit distance filter into a queue,
//                   full queues are evaluated in FP64 with the reference's
//                   operand order and minimum-image loops
//   k_ew_finalize   energy of the particles and the self term
#include <algorithm>
#include <cmath>
#include <vector>

#include <math.h>

#include "erfcx_table.h"
#include "gse_device.h"
#include "gse_internal.h"

namespace gse {

template <typename T>
struct alignas(4 * sizeof(T)) P4 {
  T x, y, z, w;
};

__global__ void k_zero_i32(int* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

// ---------------------------------------------------------------------------
// SPME
// ---------------------------------------------------------------------------
// fractional grid position (CudaPMERecip.cu:471-476, in FP64)
__device__ __forceinline__ void pme_pos(double x, double recip, int nfft, int& i0,
                                        double& frac) {
  const double w = x * recip + 2.0;
  const double fr = (double)nfft * (w - (floor(w + 0.5) - 0.5));
  const int fi = (int)fr;
  frac = fr - (double)fi;
  i0 = fi;
}

// B-spline weights and derivatives (CudaPMERecip.cu:266-327)
template <int ORDER>
__device__ __forceinline__ void pme_theta(double w, double* th, double* dth) {
  th[ORDER - 1] = 0.0;
  th[1] = w;
  th[0] = 1.0 - w;
#pragma unroll
  for (int k = 3; k <= ORDER - 1; k++) {
    const double div = 1.0 / (double)(k - 1);
    th[k - 1] = div * w * th[k - 2];
#pragma unroll
    for (int j = 1; j <= k - 2; j++)
      th[k - j - 1] = div * ((w + j) * th[k - j - 2] + (k - j - w) * th[k - j - 1]);
    th[0] = div * (1.0 - w) * th[0];
  }
  dth[0] = -th[0];
#pragma unroll
  for (int j = 2; j <= ORDER; j++) dth[j - 1] = th[j - 2] - th[j - 1];
  const double div = 1.0 / (double)(ORDER - 1);
  th[ORDER - 1] = div * w * th[ORDER - 2];
#pragma unroll
  for (int j = 1; j <= ORDER - 2; j++)
    th[ORDER - j - 1] = div * ((w + j) * th[ORDER - j - 2] + (ORDER - j - w) * th[ORDER - j - 1]);
  th[0] = div * (1.0 - w) * th[0];
}

// A particle takes part when its record is finite and its scaled coordinates
// are small enough for the integer grid position.
template <typename CT>
__device__ __forceinline__ bool pme_valid(const P4<CT>& r, double rx, double ry, double rz) {
  const double x = r.x, y = r.y, z = r.z, q = r.w;
  return isfinite(x) && isfinite(y) && isfinite(z) && isfinite(q) && fabs(x * rx) < 1e9 &&
         fabs(y * ry) < 1e9 && fabs(z * rz) < 1e9;
}

// lanes per particle: order^2 (x, y) offsets rounded up to 16 or 64
template <int ORDER>
struct PmeLanes {
  static constexpr int G = ORDER * ORDER <= 16 ? 16 : 64;
};

// Particles into bins of kPmeEdge^3 grid cells by the first cell of their
// support, with max |q| and the rejected count of the call.  Slots are
// claimed as the GSE binning claims them: one global atomic per workgroup
// and touched bin, ranks within it from LDS (above kPmeAggBins bins, one per
// particle: a workgroup's particles then touch most bins once).  Without
// counts, the statistics only.
constexpr int kPmeEdge = 8, kPmeAggBins = 16384;
template <typename CT>
__global__ __launch_bounds__(1024) void k_pme_bin(const P4<CT>* __restrict__ xyzq, int n,
                                                  PmeGrid a, int cap, int agg,
                                                  int* __restrict__ counts,
                                                  BinStats* __restrict__ st,
                                                  int* __restrict__ ovf,
                                                  P4<CT>* __restrict__ sorted) {
  extern __shared__ int pme_hist[];
  __shared__ double wmax[16];
  __shared__ int wbad[16];
  const int i = blockIdx.x * 1024 + threadIdx.x;
  if (agg)
    for (int j = threadIdx.x; j < a.b.nbins; j += 1024) pme_hist[j] = 0;
  __syncthreads();
  int bin = -1, rank = 0, bad = 0;
  double qm = 0.0;
  P4<CT> r{};
  if (i < n) {
    r = xyzq[i];
    if (pme_valid(r, a.rx, a.ry, a.rz)) {
      int ix, iy, iz;
      double f;
      pme_pos((double)r.x, a.rx, a.X, ix, f);
      pme_pos((double)r.y, a.ry, a.Y, iy, f);
      pme_pos((double)r.z, a.rz, a.Z, iz, f);
      // a fraction rounded up to one counts as the first cell
      ix = ix >= a.X ? ix - a.X : ix;
      iy = iy >= a.Y ? iy - a.Y : iy;
      iz = iz >= a.Z ? iz - a.Z : iz;
      bin = ix / kPmeEdge + a.b.nbx * (iy / kPmeEdge + a.b.nby * (iz / kPmeEdge));
      if (agg) rank = atomicAdd(&pme_hist[bin], 1);
      qm = fabs((double)r.w);
    } else {
      bad = 1;
    }
  }
  __syncthreads();
  if (agg)
    for (int j = threadIdx.x; j < a.b.nbins; j += 1024) {
      const int c = pme_hist[j];
      if (c > 0) pme_hist[j] = atomicAdd(&counts[j], c);
    }
  __syncthreads();
  if (bin >= 0 && counts) {
    const int slot = agg ? pme_hist[bin] + rank : atomicAdd(&counts[bin], 1);
    if (slot < cap)
      sorted[(size_t)bin * cap + slot] = r;
    else
      ovf[atomicAdd(&st->overflow, 1)] = i;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    qm = fmax(qm, __shfl_xor(qm, m, kWave));
    bad += __shfl_xor(bad, m, kWave);
  }
  if ((threadIdx.x & 63) == 0) {
    wmax[threadIdx.x >> 6] = qm;
    wbad[threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) {
      qm = fmax(qm, wmax[w]);
      bad += wbad[w];
    }
    if (qm > 0.0) atomicMax(&st->qmax_bits, (unsigned long long)__double_as_longlong(qm));
    if (bad) atomicAdd(&st->invalid, bad);
  }
}

// Spline of one axis per thread for a chunk of particles, in LDS: the lanes
// of a particle share it.  (With every lane computing all three axes for
// itself the order-6 spread and gather took 127 and 161 us for 200,001
// charges on 125 x 126 x 128, 42 and 82 us with this.)
constexpr int kPmeChunk = 64;
template <int ORDER, bool DERIV>
struct PmeSplines {
  double th[kPmeChunk][3][ORDER];
  double dth[DERIV ? kPmeChunk : 1][3][ORDER];
  double q[kPmeChunk];  // charge; NaN marks a rejected particle
  int cell[kPmeChunk][3];
};

// particle k of the chunk is load(k); 3 kPmeChunk threads; needs a barrier
template <int ORDER, bool DERIV, typename CT, typename F>
__device__ __forceinline__ void pme_splines(PmeSplines<ORDER, DERIV>& s, const PmeGrid& a, int cnt,
                                            F load) {
  const int k = threadIdx.x / 3, ax = threadIdx.x - 3 * k;
  if (k >= cnt) return;
  const P4<CT> r = load(k);
  const bool ok = pme_valid(r, a.rx, a.ry, a.rz);
  if (ax == 0) s.q[k] = ok ? (double)r.w : __builtin_nan("");
  if (!ok) return;
  const int M = ax == 0 ? a.X : ax == 1 ? a.Y : a.Z;
  int c;
  double f, th[ORDER], d[ORDER];
  pme_pos((double)(ax == 0 ? r.x : ax == 1 ? r.y : r.z), ax == 0 ? a.rx : ax == 1 ? a.ry : a.rz, M,
          c, f);
  s.cell[k][ax] = c >= M ? c - M : c;  // a fraction rounded up to one: the first cell
  pme_theta<ORDER>(f, th, d);
#pragma unroll
  for (int j = 0; j < ORDER; j++) {
    s.th[k][ax][j] = th[j];
    if (DERIV) s.dth[k][ax][j] = d[j];
  }
}

// one lane's contributions of chunk particle k: offset (ax, ay) of its
// support and every z offset; put(x, y, z, value) receives unwrapped cells
template <int ORDER, typename F>
__device__ __forceinline__ void pme_contrib(const PmeSplines<ORDER, false>& s, int k, double scale,
                                            int ax, int ay, F put) {
  // ((q tx) ty) tz as the reference orders it; the exact power-of-two
  // scale changes no rounding
  const double qxy = s.q[k] * scale * s.th[k][0][ax] * s.th[k][1][ay];
  const int x = s.cell[k][0] + ax, y = s.cell[k][1] + ay, z = s.cell[k][2];
#pragma unroll
  for (int c = 0; c < ORDER; c++) put(x, y, z + c, fixed_round_prod(qxy, s.th[k][2][c]));
}

// B-spline spread of one bin per workgroup into an int64 brick in LDS
// (kPmeEdge + ORDER - 1 cells a side), stored whole; k_brick_reduce adds the
// bricks.  The workgroups after the bins' add the particles that found their
// bin full to the int64 grid with global atomics, `per` at a time (without an
// overflow list and bins, all the particles).  Spreading
// every particle that way, 64 atomics of 8 bytes each to memory, took 49 us
// of the 48,000-charge step at order 4, after 11 us for max |q|; binning,
// spread and reduce take 5.7 + 10.3 + 8.4 (order 6, 200,001 charges on
// 125 x 126 x 128: the whole step 870 -> 301 us).  The counts are cleared here
// by their only reader; st_kept receives the statistics for k_brick_reduce,
// which clears st.  A call so leaves counts and st zero, with no host state
// that a replay of its captured launches would not change.
template <int ORDER, typename CT>
__global__ __launch_bounds__(256) void k_pme_spread(
    const P4<CT>* __restrict__ xyzq, int n, PmeGrid a, int cap, int* __restrict__ counts,
    const BinStats* __restrict__ st, BinStats* __restrict__ st_kept,
    const int* __restrict__ ovf, const P4<CT>* __restrict__ sorted, long long* __restrict__ bricks,
    int* __restrict__ bshift, unsigned long long* __restrict__ g64, int per) {
  constexpr int G = PmeLanes<ORDER>::G, PER = 256 / G;
  constexpr int L = kPmeEdge + ORDER - 1, VOL = L * L * L;
  __shared__ unsigned long long brick[VOL];
  __shared__ PmeSplines<ORDER, false> sp;
  const int lane = threadIdx.x & (G - 1), ax = lane % ORDER, ay = lane / ORDER;
  const bool live = lane < ORDER * ORDER;
  const BinStats s = *st;
  const double scale = ldexp(1.0, fixed_exponent(s.qmax_bits, n - s.invalid, 1, 1.0));
  const int bin = blockIdx.x;
  if (bin >= a.b.nbins) {
    const int w = bin - a.b.nbins, nw = (int)gridDim.x - a.b.nbins;
    if (w == 0 && threadIdx.x == 0) *st_kept = s;
    const int novf = ovf ? s.overflow : n;
    for (int k0 = w * per; k0 < novf; k0 += nw * per) {
      const int m = min(per, novf - k0);
      pme_splines<ORDER, false, CT>(sp, a, m,
                                    [&](int k) { return xyzq[ovf ? ovf[k0 + k] : k0 + k]; });
      __syncthreads();
      for (int k = threadIdx.x / G; k < m; k += PER)
        if (live && sp.q[k] == sp.q[k])
          pme_contrib<ORDER>(sp, k, scale, ax, ay, [&](int x, int y, int z, long long v) {
            x = x >= a.X ? x - a.X : x;
            y = y >= a.Y ? y - a.Y : y;
            z = z >= a.Z ? z - a.Z : z;
            atomicAdd(&g64[x + (size_t)a.X * (y + (size_t)a.Y * z)], (unsigned long long)v);
          });
      __syncthreads();
    }
    return;
  }
  const int cnt = min(counts[bin], cap);
  for (int j = threadIdx.x; j < VOL; j += 256) brick[j] = 0ull;
  __syncthreads();
  if (threadIdx.x == 0) {
    counts[bin] = 0;
    bshift[bin] = cnt > 0 ? 0 : -1;
  }
  if (cnt == 0) return;
  const int x0 = bin % a.b.nbx * kPmeEdge, y0 = bin / a.b.nbx % a.b.nby * kPmeEdge,
            z0 = bin / (a.b.nbx * a.b.nby) * kPmeEdge;
  for (int k0 = 0; k0 < cnt; k0 += kPmeChunk) {
    const int m = min(kPmeChunk, cnt - k0);
    pme_splines<ORDER, false, CT>(sp, a, m,
                                  [&](int k) { return sorted[(size_t)bin * cap + k0 + k]; });
    __syncthreads();
    for (int k = threadIdx.x / G; k < m; k += PER)
      if (live)
        pme_contrib<ORDER>(sp, k, scale, ax, ay, [&](int x, int y, int z, long long v) {
          atomicAdd(&brick[x - x0 + L * (y - y0 + L * (z - z0))], (unsigned long long)v);
        });
    __syncthreads();
  }
  for (int j = threadIdx.x; j < VOL; j += 256)
    bricks[(size_t)bin * VOL + j] = (long long)brick[j];
}

struct PmeSum {
  int X, Y, Z;
  double rx, ry, rz, fac, piv_inv;
};

__device__ __forceinline__ double pme_eterm(const PmeSum& a, int k1, int k2, int k3,
                                            const double* p1, const double* p2,
                                            const double* p3, double* mh) {
  const int nf1 = a.X / 2 + a.X % 2, nf2 = a.Y / 2 + a.Y % 2, nf3 = a.Z / 2 + a.Z % 2;
  const int m1 = k1 >= nf1 ? k1 - a.X : k1, m2 = k2 >= nf2 ? k2 - a.Y : k2,
            m3 = k3 >= nf3 ? k3 - a.Z : k3;
  mh[0] = a.rx * m1;
  mh[1] = a.ry * m2;
  mh[2] = a.rz * m3;
  const double msq = mh[0] * mh[0] + mh[1] * mh[1] + mh[2] * mh[2];
  return exp(-a.fac * msq) * a.piv_inv * p1[k1] * p2[k2] * p3[k3] / msq;
}

// CudaPMERecip.cu:946-1256: the element and, for x index >= 1, its
// conjugate partner enter the energy and virial (the x Nyquist plane of an
// even grid twice, as in the reference).  Partial sums per workgroup in
// partials[blockIdx][7] (energy, then the six upper-triangle moments).
template <typename CT>
__global__ __launch_bounds__(256) void k_pme_scalar_sum(PmeSum a, const double* __restrict__ p1,
                                                        const double* __restrict__ p2,
                                                        const double* __restrict__ p3,
                                                        CT* __restrict__ spec, int want,
                                                        double* __restrict__ partials) {
  const int size1 = a.X / 2 + 1;
  const long long K = (long long)size1 * a.Y * a.Z;
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < K;
       e += (long long)gridDim.x * blockDim.x) {
    CT* q = spec + 2 * e;
    if (e == 0) {
      q[0] = (CT)0;
      q[1] = (CT)0;
      continue;
    }
    const int k1 = (int)(e % size1);
    const long long r = e / size1;
    const int k2 = (int)(r % a.Y), k3 = (int)(r / a.Y);
    double mh[3];
    const double et = pme_eterm(a, k1, k2, k3, p1, p2, p3, mh);
    if (want) {
      const double q2 = (double)q[0] * (double)q[0] + (double)q[1] * (double)q[1];
      for (int part = 0; part < (k1 >= 1 ? 2 : 1); part++) {
        double ee = et, m[3] = {mh[0], mh[1], mh[2]};
        if (part == 1)
          ee = pme_eterm(a, a.X - k1, (a.Y - k2) % a.Y, (a.Z - k3) % a.Z, p1, p2, p3, m);
        const double msq = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
        const double t1 = ee * q2, vt = 2.0 * (a.fac + 1.0 / msq), t2 = t1 * vt;
        acc[0] += t1;
        acc[1] += t1 * (vt * m[0] * m[0] - 1.0);
        acc[2] += t2 * m[0] * m[1];
        acc[3] += t2 * m[0] * m[2];
        acc[4] += t1 * (vt * m[1] * m[1] - 1.0);
        acc[5] += t2 * m[1] * m[2];
        acc[6] += t1 * (vt * m[2] * m[2] - 1.0);
      }
    }
    q[0] = (CT)((double)q[0] * et);
    q[1] = (CT)((double)q[1] * et);
  }
  if (!want) return;
  __shared__ double sh[4][7];
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 7; c++) {
    const double t = wave_sum(acc[c]);
    if ((threadIdx.x & 63) == 0) sh[w][c] = t;
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    const int c = threadIdx.x;
    partials[blockIdx.x * 7 + c] = (sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c]);
  }
}

// E = ccelec/2 sum, virial_ab = -ccelec/2 sum (CudaPMERecip.cu:1222-1239)
// the workgroup's threads sum strided partials, then the waves' sums are
// added in wave order (fixed order, deterministic)
__global__ void __launch_bounds__(256)
    k_pme_finalize(const double* __restrict__ partials, int nblocks, double ccelec,
                   double* energy, double* virial) {
  double sh[7];
  reduce_partials_block<7>(partials, nblocks, 7, sh);
  if (threadIdx.x == 0) {
    const double h = 0.5 * ccelec;
    if (energy) energy[0] = h * sh[0];
    if (virial) {
      virial[0] = -h * sh[1];
      virial[1] = -h * sh[2];
      virial[2] = -h * sh[3];
      virial[3] = -h * sh[2];
      virial[4] = -h * sh[4];
      virial[5] = -h * sh[5];
      virial[6] = -h * sh[3];
      virial[7] = -h * sh[5];
      virial[8] = -h * sh[6];
    }
  }
}

// CudaPMERecip.cu:1612-1890: dE/dr_a = q ccelec (M_a/L_a) sum dtheta_a theta
// theta Qc; written times `sign` into out{x,y,z}[i].
// Workgroups of `per` (at most kPmeChunk) consecutive particles.
template <int ORDER, typename CT, typename AT>
__global__ __launch_bounds__(256) void k_pme_gather(const P4<CT>* __restrict__ xyzq, int n,
                                                    PmeGrid g, int per, double ccelec, double sign,
                                                    const CT* __restrict__ Qc, AT* __restrict__ ox,
                                                    AT* __restrict__ oy, AT* __restrict__ oz) {
  constexpr int G = PmeLanes<ORDER>::G;
  constexpr int PER = 256 / G;
  __shared__ PmeSplines<ORDER, true> sp;
  const int lane = threadIdx.x & (G - 1);
  const int a = lane % ORDER, b = lane / ORDER;
  const bool live = lane < ORDER * ORDER;
  const int p0 = blockIdx.x * per, m = min(per, n - p0);
  pme_splines<ORDER, true, CT>(sp, g, m, [&](int k) { return xyzq[p0 + k]; });
  __syncthreads();
  // uniform trip count over the group so the butterfly sees every lane
  for (int k0 = 0; k0 < m; k0 += PER) {
    const int k = k0 + (int)(threadIdx.x / G);
    CT f1 = 0, f2 = 0, f3 = 0;
    const double q = k < m ? sp.q[k] : 0.0;
    const bool ok = k < m && q == q;
    if (ok && live) {
      int xi = sp.cell[k][0] + a, yi = sp.cell[k][1] + b;
      if (xi >= g.X) xi -= g.X;
      if (yi >= g.Y) yi -= g.Y;
      const CT* row = Qc + (size_t)xi + (size_t)yi * g.X;
      const double tx = sp.th[k][0][a], ty = sp.th[k][1][b];
      const CT w1 = (CT)(sp.dth[k][0][a] * ty), w2 = (CT)(tx * sp.dth[k][1][b]), w3 = (CT)(tx * ty);
#pragma unroll
      for (int c = 0; c < ORDER; c++) {
        int zi = sp.cell[k][2] + c;
        if (zi >= g.Z) zi -= g.Z;
        const CT v = row[(size_t)zi * g.X * g.Y];
        const CT zc = (CT)sp.th[k][2][c], zd = (CT)sp.dth[k][2][c];
        f1 += w1 * zc * v;
        f2 += w2 * zc * v;
        f3 += w3 * zd * v;
      }
    }
#pragma unroll
    for (int i = G / 2; i >= 1; i >>= 1) {
      f1 += __shfl_xor(f1, i, kWave);
      f2 += __shfl_xor(f2, i, kWave);
      f3 += __shfl_xor(f3, i, kWave);
    }
    if (lane == 0 && k < m) {
      const double s = ok ? q * ccelec * sign : 0.0;
      ox[p0 + k] = (AT)(s * g.rx * (double)f1 * g.X);
      oy[p0 + k] = (AT)(s * g.ry * (double)f2 * g.Y);
      oz[p0 + k] = (AT)(s * g.rz * (double)f3 * g.Z);
    }
  }
}

static unsigned blocks_for(long long count, unsigned threads, unsigned cap) {
  long long b = (count + threads - 1) / threads;
  if (b < 1) b = 1;
  return (unsigned)(b < cap ? b : cap);
}

PmeGrid pme_grid_make(int X, int Y, int Z, int order, const double* r) {
  PmeGrid a;
  a.X = X;
  a.Y = Y;
  a.Z = Z;
  a.rx = r[0];
  a.ry = r[1];
  a.rz = r[2];
  BinShape& b = a.b;
  b.Bx = b.By = b.Bz = kPmeEdge;
  b.nbx = (X + kPmeEdge - 1) / kPmeEdge;
  b.nby = (Y + kPmeEdge - 1) / kPmeEdge;
  b.nbz = (Z + kPmeEdge - 1) / kPmeEdge;
  b.nbins = b.nbx * b.nby * b.nbz;
  b.Lx = b.Ly = b.Lz = kPmeEdge + order - 1;
  b.direct = 0;
  return a;
}

hipError_t launch_pme_bin(bool dbl, const void* xyzq, int n, const PmeGrid& a, int cap,
                          int* counts, BinStats* st, int* ovf, void* sorted, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int agg = counts && a.b.nbins <= kPmeAggBins ? 1 : 0;
  const unsigned g = (unsigned)((n + 1023) / 1024);
  const size_t lds = agg ? sizeof(int) * (size_t)a.b.nbins : 0;
  if (dbl)
    k_pme_bin<double><<<g, 1024, lds, s>>>((const P4<double>*)xyzq, n, a, cap, agg, counts, st,
                                           ovf, (P4<double>*)sorted);
  else
    k_pme_bin<float><<<g, 1024, lds, s>>>((const P4<float>*)xyzq, n, a, cap, agg, counts, st, ovf,
                                          (P4<float>*)sorted);
  return hipGetLastError();
}

// particles per workgroup: whole chunks once they still make four workgroups
// per CU
template <int ORDER>
static int pme_per_wg(int n) {
  constexpr int PER = 256 / PmeLanes<ORDER>::G;
  return std::min(kPmeChunk, std::max(1, n / (1024 * PER)) * PER);
}

template <int ORDER, typename CT>
static void pme_spread_t(const void* xyzq, int n, const PmeGrid& a, int cap, int* counts,
                         const BinStats* st, BinStats* st_kept, const int* ovf,
                         const void* sorted, void* bricks, int* bshift, unsigned long long* g64,
                         hipStream_t s) {
  // Overflow workgroups for all the particles (up to eight per CU): a box
  // filled in a tenth of its volume has most of them on the overflow list.
  // The call then took 205 us at order 4 (48,000 charges, 80^3) and 699 at
  // order 8 with eight such workgroups, 57 and
  // 208 now; without overflow it takes 22 and 42.
  const int per = pme_per_wg<ORDER>(n);
  const int ovf_wg = std::max(1, std::min(2048, (n + per - 1) / per));
  k_pme_spread<ORDER, CT><<<a.b.nbins + ovf_wg, 256, 0, s>>>(
      (const P4<CT>*)xyzq, n, a, cap, counts, st, st_kept, ovf, (const P4<CT>*)sorted,
      (long long*)bricks, bshift, g64, per);
}

hipError_t launch_pme_spread(bool dbl, int order, const void* xyzq, int n, const PmeGrid& a,
                             int cap, int* counts, const BinStats* st, BinStats* st_kept,
                             const int* ovf, const void* sorted, void* bricks, int* bshift,
                             unsigned long long* g64, hipStream_t s) {
#define GSE_PME_SPREAD(O)                                                                      \
  if (dbl)                                                                                     \
    pme_spread_t<O, double>(xyzq, n, a, cap, counts, st, st_kept, ovf, sorted, bricks, bshift, \
                            g64, s);                                                           \
  else                                                                                         \
    pme_spread_t<O, float>(xyzq, n, a, cap, counts, st, st_kept, ovf, sorted, bricks, bshift,  \
                           g64, s);
  switch (order) {
    case 4: GSE_PME_SPREAD(4) break;
    case 6: GSE_PME_SPREAD(6) break;
    case 8: GSE_PME_SPREAD(8) break;
    default: return hipErrorInvalidValue;
  }
#undef GSE_PME_SPREAD
  return hipGetLastError();
}

hipError_t launch_pme_scalar_sum(bool dbl, int X, int Y, int Z, const double* recip3,
                                 double kappa, const double* prefac, void* spec, bool want,
                                 double* partials, hipStream_t s) {
  PmeSum a;
  a.X = X;
  a.Y = Y;
  a.Z = Z;
  a.rx = recip3[0];
  a.ry = recip3[1];
  a.rz = recip3[2];
  a.fac = M_PI * M_PI / (kappa * kappa);
  a.piv_inv = recip3[0] * recip3[1] * recip3[2] / M_PI;
  const double* p1 = prefac;
  const double* p2 = prefac + X;
  const double* p3 = prefac + X + Y;
  if (dbl)
    k_pme_scalar_sum<double><<<kPmeSumBlocks, 256, 0, s>>>(a, p1, p2, p3, (double*)spec,
                                                           want ? 1 : 0, partials);
  else
    k_pme_scalar_sum<float><<<kPmeSumBlocks, 256, 0, s>>>(a, p1, p2, p3, (float*)spec,
                                                          want ? 1 : 0, partials);
  return hipGetLastError();
}

hipError_t launch_pme_finalize(const double* partials, double ccelec, double* energy,
                               double* virial, hipStream_t s) {
  k_pme_finalize<<<1, 256, 0, s>>>(partials, kPmeSumBlocks, ccelec, energy, virial);
  return hipGetLastError();
}

template <int ORDER, typename CT>
static void pme_gather_o(bool at_dbl, const void* xyzq, int n, int X, int Y, int Z,
                         const double* r, double ccelec, double sign, const void* Qc, void* ox,
                         void* oy, void* oz, hipStream_t s) {
  const int per = pme_per_wg<ORDER>(n);
  const unsigned grid = (unsigned)((n + per - 1) / per);
  const PmeGrid g = pme_grid_make(X, Y, Z, ORDER, r);
  if (at_dbl)
    k_pme_gather<ORDER, CT, double><<<grid, 256, 0, s>>>((const P4<CT>*)xyzq, n, g, per, ccelec,
                                                         sign, (const CT*)Qc, (double*)ox,
                                                         (double*)oy, (double*)oz);
  else
    k_pme_gather<ORDER, CT, float><<<grid, 256, 0, s>>>((const P4<CT>*)xyzq, n, g, per, ccelec,
                                                        sign, (const CT*)Qc, (float*)ox,
                                                        (float*)oy, (float*)oz);
}

hipError_t launch_pme_gather(bool ct_dbl, bool at_dbl, int order, const void* xyzq, int n, int X,
                             int Y, int Z, const double* recip3, double ccelec, double sign,
                             const void* Qc, void* ox, void* oy, void* oz, hipStream_t s) {
  if (n <= 0) return hipGetLastError();
#define GSE_PME_GATHER(O)                                                                     \
  if (ct_dbl)                                                                                 \
    pme_gather_o<O, double>(at_dbl, xyzq, n, X, Y, Z, recip3, ccelec, sign, Qc, ox, oy, oz, s); \
  else                                                                                        \
    pme_gather_o<O, float>(at_dbl, xyzq, n, X, Y, Z, recip3, ccelec, sign, Qc, ox, oy, oz, s);
  switch (order) {
    case 4: GSE_PME_GATHER(4) break;
    case 6: GSE_PME_GATHER(6) break;
    case 8: GSE_PME_GATHER(8) break;
    default: return hipErrorInvalidValue;
  }
#undef GSE_PME_GATHER
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ewald direct space
// ---------------------------------------------------------------------------
// one coordinate wrapped into [0, L) (NaN for a non-finite one) and its cell
// of edge L/nc
__device__ __forceinline__ double ew_wrap(double x, double L) {
  const double w = x - L * floor(x / L);
  return w >= L || w < 0.0 ? 0.0 : w;
}
__device__ __forceinline__ int ew_cell1(double w, double L, int nc) {
  if (!(w >= 0.0)) return 0;
  const int c = (int)(w * ((double)nc / L));
  return c < nc ? c : nc - 1;
}

// Cell and arrival rank of every particle, and the partial sums of q^2 for
// the self term (one per workgroup, fixed order).  The cells hold about six
// particles, so few atomics meet on one counter (a cell of edge rcut holds
// ninety, and 48,000 atomics on 512 counters took 26 us).
__global__ __launch_bounds__(256) void k_ew_cell_count(const P4<double>* __restrict__ xyzq, int n,
                                                       EwCells c, int* __restrict__ cell_of,
                                                       int* __restrict__ rank,
                                                       int* __restrict__ counts,
                                                       double* __restrict__ q2) {
  __shared__ double sh[4];
  double acc = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const P4<double> r = xyzq[i];
    const int cx = ew_cell1(ew_wrap(r.x, c.box[0]), c.box[0], c.nc[0]),
              cy = ew_cell1(ew_wrap(r.y, c.box[1]), c.box[1], c.nc[1]),
              cz = ew_cell1(ew_wrap(r.z, c.box[2]), c.box[2], c.nc[2]);
    const int cell = cx + (cy + cz * c.nc[1]) * c.nc[0];
    cell_of[i] = cell;
    rank[i] = atomicAdd(&counts[cell], 1);
    acc += r.w * r.w;
  }
  const double w = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) q2[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// exclusive scan of the cell counts by one workgroup, consecutive cells per
// thread; starts[ncell] = all particles
__global__ __launch_bounds__(1024) void k_ew_scan(const int* __restrict__ counts, int ncell,
                                                  int* __restrict__ starts) {
  __shared__ int sh[16];
  const int per = (ncell + 1023) / 1024;
  const int i0 = min((int)threadIdx.x * per, ncell), i1 = min(i0 + per, ncell);
  int sum = 0;
  for (int i = i0; i < i1; i++) sum += counts[i];
  int v = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(v, d, kWave);
    if ((int)(threadIdx.x & 63) >= d) v += t;
  }
  if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  int run = v - sum;
  for (int w = 0; w < (int)(threadIdx.x >> 6); w++) run += sh[w];
  for (int i = i0; i < i1; i++) {
    starts[i] = run;
    run += counts[i];
  }
  if (threadIdx.x == 1023) starts[ncell] = run;
}

__global__ void k_ew_scatter(int n, const int* __restrict__ cell_of, const int* __restrict__ rank,
                             const int* __restrict__ starts, int* __restrict__ tmp) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    tmp[starts[cell_of[i]] + rank[i]] = i;
}

// Each cell's particles in ascending index (deterministic): the rank of a
// slot is the number of the cell's particles with a smaller index.  sf holds
// the wrapped position in units of rcut, rounded to 32 bits, and the cell,
// for the distance filter of k_ew_force.
__global__ void k_ew_sort(int n, EwCells c, double inv_rcut, const int* __restrict__ cell_of,
                          const int* __restrict__ starts, const int* __restrict__ tmp,
                          const P4<double>* __restrict__ xyzq, int* __restrict__ sidx,
                          P4<double>* __restrict__ sx, P4<float>* __restrict__ sf) {
  for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += gridDim.x * blockDim.x) {
    const int i = tmp[s];
    const int cell = cell_of[i];
    const int st = starts[cell], en = starts[cell + 1];
    int k = st;
    for (int t = st; t < en; t++) k += tmp[t] < i;
    const P4<double> r = xyzq[i];
    sidx[k] = i;
    sx[k] = r;
    sf[k] = P4<float>{(float)(ew_wrap(r.x, c.box[0]) * inv_rcut),
                      (float)(ew_wrap(r.y, c.box[1]) * inv_rcut),
                      (float)(ew_wrap(r.z, c.box[2]) * inv_rcut), __int_as_float(cell)};
  }
}

// the reference's minimum-image loops (CpuEwaldDirect.cpp:93-98), bounded:
// after four steps a coordinate still outside is folded in one go (only
// coordinates many boxes away, or non-finite ones, get there)
__device__ __forceinline__ double ew_image(double d, double L, double h) {
  for (int it = 0; it < 4 && d < -h; it++) d += L;
  for (int it = 0; it < 4 && d > h; it++) d -= L;
  if (d < -h || d > h) d -= L * rint(d / L);
  return d;
}

// the same value for the common case, at most one step either way, without
// loops; `far` collects coordinates that need them
__device__ __forceinline__ double ew_image1(double d, double L, double h, bool& far) {
  double v = d < -h ? d + L : d;
  v = v > h ? v - L : v;
  far = far || !(v >= -h && v <= h);
  return v;
}

const double* ew_erfcx_table() {
  static const std::vector<double> table = make_erfcx_table();
  return table.data();
}
size_t ew_erfcx_bytes() { return sizeof(double) * kErfcxRows * kErfcxPitch; }

// Force and energy of one particle per wave, in the order of the cells.
//
// The pair term costs about 150 FP64 instructions and one candidate in three
// is within rcut, so testing and evaluating in one loop runs the pair term
// with a third of the lanes.  Here the wave takes 64 candidates at a time,
// tests them in 32 bits (rcut widened by the rounding of the positions, so no
// pair is lost), and appends the survivors to a queue in LDS; 64 of them are
// evaluated with all lanes in FP64 (the reference's operand order and strict
// r2 < rcut2 test on the exact positions).  Two and four particles per wave,
// sharing the candidate loads, were no faster (293 against 288 us) for want
// of waves.
// Candidates are the cells within reach: rows of cells along x are one
// contiguous range of the sorted particles (two where the row wraps), found
// by one lane per range and cut to the sphere around the particle.  Cells of
// rcut/4 x rcut/2 x rcut/2 make a row range at most about 50 particles of
// liquid water, one batch of 64; cells of edge rcut take 2,500 candidates.
// On the 48,000-charge box at rcut 9 (14.6 M pair terms): 240 us, 110 M VALU
// instructions (180 us of issue), against 1475 us with one loop over the 27
// cells of edge rcut around each; 3,000 charges 31 us.
// Each lane adds its terms in the order of the cells, then the lanes are
// added in a fixed order: no atomics, the same bits on every run.
constexpr int kEwWaves = 4;
template <bool FOLD>
__global__ __launch_bounds__(64 * kEwWaves) void k_ew_force(
    int n, EwCells c, EwPair pr, const int* __restrict__ starts, const int* __restrict__ sidx,
    const P4<double>* __restrict__ sx, const P4<float>* __restrict__ sf,
    const int* __restrict__ xofs, const int* __restrict__ xlist,
    const double* __restrict__ erfcx, double* __restrict__ gx, double* __restrict__ gy,
    double* __restrict__ gz, double* __restrict__ partials) {
  __shared__ int queue[kEwWaves][128];
  __shared__ alignas(16) double ertab[kErfcxRows * kErfcxPitch];
  for (int k = threadIdx.x; k < kErfcxRows * kErfcxPitch; k += 64 * kEwWaves) ertab[k] = erfcx[k];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int islot = blockIdx.x * kEwWaves + wave;
  if (islot >= n) return;  // no barrier follows
  int* q = queue[wave];

  const P4<float> pf = sf[islot];
  const int cell = __builtin_amdgcn_readfirstlane(__float_as_int(pf.w));
  const int a = sidx[islot];
  const P4<double> pa = sx[islot];
  // the first exclusions stay in registers (a water atom has two)
  const int ex0 = xofs ? xofs[a] : 0, ex1 = xofs ? xofs[a + 1] : 0;
  int ex[4];
#pragma unroll
  for (int x = 0; x < 4; x++) ex[x] = ex0 + x < ex1 ? xlist[ex0 + x] : -1;

  // candidate ranges: lane 2r + part holds part 0 or 1 of row r's range.  An
  // axis whose cells all lie within reach is visited once and its distances
  // folded to the nearest image; the others carry the image's shift.
  const bool ally = FOLD && c.nc[1] <= 2 * c.reach[1] + 1,
             allz = FOLD && c.nc[2] <= 2 * c.reach[2] + 1;
  const int nyr = ally ? c.nc[1] : 2 * c.reach[1] + 1;
  const int nzr = allz ? c.nc[2] : 2 * c.reach[2] + 1;
  int s = 0, t = 0;
  float hx = 0.f, hy = 0.f, hz = 0.f;  // added to the candidate's position
  bool whole = false;
  {
    const int r = lane >> 1, part = lane & 1;
    if (r < nyr * nzr) {
      const int row = cell / c.nc[0];
      int y = r % nyr, z = r / nyr;
      float d2 = 0.f;  // squared distance of the particle to the row
      if (!ally) {
        y += row % c.nc[1] - c.reach[1];
        const float e = c.len[1] / (float)c.nc[1], lo = e * (float)y;
        const float d = fmaxf(fmaxf(lo - pf.y, pf.y - (lo + e)) - pr.slack, 0.f);
        d2 += d * d;
        if (y < 0) {
          y += c.nc[1];
          hy = -c.len[1];
        } else if (y >= c.nc[1]) {
          y -= c.nc[1];
          hy = c.len[1];
        }
      }
      if (!allz) {
        z += row / c.nc[1] - c.reach[2];
        const float e = c.len[2] / (float)c.nc[2], lo = e * (float)z;
        const float d = fmaxf(fmaxf(lo - pf.z, pf.z - (lo + e)) - pr.slack, 0.f);
        d2 += d * d;
        if (z < 0) {
          z += c.nc[2];
          hz = -c.len[2];
        } else if (z >= c.nc[2]) {
          z -= c.nc[2];
          hz = c.len[2];
        }
      }
      int x0 = 0, x1 = -1;
      if (d2 <= pr.filter2) {  // false for a particle at a position that is not finite
        const float w = sqrtf(pr.filter2 - d2) + pr.slack, ie = (float)c.nc[0] / c.len[0];
        const int lo = (int)floorf((pf.x - w) * ie), hi = (int)floorf((pf.x + w) * ie);
        whole = FOLD && hi - lo + 1 >= c.nc[0];
        if (whole) {
          if (part == 0) x1 = c.nc[0] - 1;
        } else if (lo < 0) {
          x0 = part ? 0 : lo + c.nc[0];
          x1 = part ? hi : c.nc[0] - 1;
          hx = part ? 0.f : -c.len[0];
        } else if (hi >= c.nc[0]) {
          x0 = part ? 0 : lo;
          x1 = part ? hi - c.nc[0] : c.nc[0] - 1;
          hx = part ? c.len[0] : 0.f;
        } else if (part == 0) {
          x0 = lo;
          x1 = hi;
        }
      }
      if (x1 >= x0) {
        const int rc = (y + z * c.nc[1]) * c.nc[0];
        s = starts[rc + x0];
        t = starts[rc + x1 + 1];
      }
    }
  }
  unsigned long long pieces = __ballot(t > s);
  const float fy = ally ? 1.f / c.len[1] : 0.f, fz = allz ? 1.f / c.len[2] : 0.f;
  const float fx = FOLD ? (whole ? 1.f / c.len[0] : 0.f) : 0.f;

  int k = 0, kend = 0, held = 0;
  float px = 0.f, py = 0.f, pz = 0.f, pfx = 0.f;
  P4<float> cand{0.f, 0.f, 0.f, 0.f};
  bool have = false;
  auto fetch = [&]() {
    k += 64;
    have = true;
    if (k >= kend) {
      have = pieces != 0ull;
      if (have) {
        const int p = __builtin_ctzll(pieces);
        pieces &= pieces - 1ull;
        k = __builtin_amdgcn_readlane(s, p);
        kend = __builtin_amdgcn_readlane(t, p);
        px = readlane(hx, p);
        py = readlane(hy, p);
        pz = readlane(hz, p);
        if (FOLD) pfx = readlane(fx, p);
      }
    }
    if (have) cand = sf[min(k + lane, kend - 1)];
  };
  double g0 = 0.0, g1 = 0.0, g2 = 0.0, e = 0.0;
  fetch();
  for (;;) {
    const bool more = have;
    if (more) {
      const int slot = k + lane;
      const bool in = slot < kend;
      float dx = pf.x - (cand.x + px), dy = pf.y - (cand.y + py), dz = pf.z - (cand.z + pz);
      if (FOLD) {
        dx -= c.len[0] * rintf(dx * pfx);
        dy -= c.len[1] * rintf(dy * fy);
        dz -= c.len[2] * rintf(dz * fz);
      }
      fetch();  // the next candidates load while these are tested
      const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
      const bool hit = in & (r2 < pr.filter2);
      const unsigned long long m = __ballot(hit);
      const unsigned at = __builtin_amdgcn_mbcnt_hi(
          (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)held));
      if (hit) q[at] = slot;
      held += __popcll(m);
    }
    // 64 fill the wave; after the last candidates, all that is left
    if (held < 64 && (more || held == 0)) {
      if (!more) break;
      continue;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < held) {
      const int sl = q[lane];
      const P4<double> pb = sx[sl];
      const int b = sidx[sl];
      bool far = false;
      double ddx = ew_image1(pa.x - pb.x, c.box[0], 0.5 * c.box[0], far);
      double ddy = ew_image1(pa.y - pb.y, c.box[1], 0.5 * c.box[1], far);
      double ddz = ew_image1(pa.z - pb.z, c.box[2], 0.5 * c.box[2], far);
      if (__builtin_expect(far, 0)) {
        ddx = ew_image(pa.x - pb.x, c.box[0], 0.5 * c.box[0]);
        ddy = ew_image(pa.y - pb.y, c.box[1], 0.5 * c.box[1]);
        ddz = ew_image(pa.z - pb.z, c.box[2], 0.5 * c.box[2]);
      }
      const double r2 = ddx * ddx + ddy * ddy + ddz * ddz;
      bool ok = r2 < pr.rcut2 && sl != islot;
#pragma unroll
      for (int x = 0; x < 4; x++) ok = ok && ex[x] != b;
      for (int x = ex0 + 4; x < ex1; x++) ok = ok && xlist[x] != b;
      if (ok) {
        // qq = (q_j ccelec) q_i with j the smaller index (:69, :101)
        const double qq = a < b ? (pa.w * pr.ccelec) * pb.w : (pb.w * pr.ccelec) * pa.w;
        const double r = sqrt(r2);
        const double expval = exp(-r2 * pr.inv_2sigmasq);
        const double er = expval * ew_erfcx(ertab, r * pr.inv_sqrt2sigma) / r;
        const double f = -qq * (pr.two_sqrtpi * pr.inv_sqrt2sigma * expval + er) / r2;
        g0 += f * ddx;
        g1 += f * ddy;
        g2 += f * ddz;
        e += qq * er;
      }
    }
    // the queue's tail moves to its front
    held = max(held - 64, 0);
    const int tail = lane < held ? q[64 + lane] : 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < held) q[lane] = tail;
  }
  g0 = wave_total(g0);
  g1 = wave_total(g1);
  g2 = wave_total(g2);
  e = wave_total(e);
  if (lane == 0) {
    gx[a] = g0;
    gy[a] = g1;
    gz[a] = g2;
    // every pair is met from both ends
    partials[islot] = 0.5 * e;
  }
}

// energy = sum of the particles' partials (sorted order) + the self term
// -ccelec sum q^2 / sqrt(2 pi sigma^2) (CpuEwaldDirect.cpp:124-128)
__global__ __launch_bounds__(1024) void k_ew_finalize(const double* __restrict__ partials,
                                                      int n, const double* __restrict__ q2,
                                                      int nq2, double self, double* energy) {
  __shared__ double she[16], shq[16];
  double s = 0.0, w = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) s += partials[i];
  for (int i = threadIdx.x; i < nq2; i += 1024) w += q2[i];
  s = wave_sum(s);
  w = wave_sum(w);
  if ((threadIdx.x & 63) == 0) {
    she[threadIdx.x >> 6] = s;
    shq[threadIdx.x >> 6] = w;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double te = 0.0, tq = 0.0;
    for (int k = 0; k < 16; k++) {
      te += she[k];
      tq += shq[k];
    }
    energy[0] = te + self * tq;
  }
}

void ew_cells_make(const double* box, double rcut, int n, EwCells* c) {
  // about eight cells per particle at most (16 for one), so that a sparse box
  // does not spend its time on empty cells
  const int cap = std::max(2, std::min(64, (int)std::cbrt(4.0 * n)));
  c->ncell = 1;
  for (int a = 0; a < 3; a++) {
    const int split = a == 0 ? 4 : 2, top = a == 0 ? 2 * cap : cap;
    c->box[a] = box[a];
    c->len[a] = (float)(box[a] / rcut);
    // the margin keeps rounding from letting a pair within rcut lie one cell
    // beyond the reach
    const double fit = box[a] / rcut * split * (1.0 - 1e-9);
    c->nc[a] = fit >= top ? top : std::max(1, (int)fit);
    const double need = rcut / box[a] * c->nc[a] * (1.0 + 1e-12);
    c->reach[a] = need >= c->nc[a] ? c->nc[a] : (int)std::ceil(need);
    c->ncell *= c->nc[a];
  }
}

void ew_filter_make(const EwCells& c, EwPair* p) {
  // Positions in units of rcut are rounded to 24 bits, shifted and
  // subtracted, cell edges multiplied out: each is off by less than 8 * 2^-24
  // of the longest edge, the squares by a few units in the last place.
  const double len = std::max(1.0, (double)std::max(c.len[0], std::max(c.len[1], c.len[2])));
  const double slack = 16.0 * len / 16777216.0;
  p->slack = (float)slack;
  p->filter2 = (float)((1.0 + slack) * (1.0 + slack) * (1.0 + 1e-6));
}

hipError_t launch_ew_cells(const void* xyzq, int n, const EwCells& c, double rcut, int* cell_of,
                           int* rank, int* counts, int* starts, int* tmp, int* sidx, void* sx,
                           void* sf, double* q2, hipStream_t s) {
  k_zero_i32<<<blocks_for(c.ncell, 256, 1024), 256, 0, s>>>(counts, c.ncell);
  const unsigned g = blocks_for(n > 0 ? n : 1, 256, 4096);
  k_ew_cell_count<<<kEwCountBlocks, 256, 0, s>>>((const P4<double>*)xyzq, n, c, cell_of, rank,
                                                 counts, q2);
  k_ew_scan<<<1, 1024, 0, s>>>(counts, c.ncell, starts);
  if (n > 0) {
    k_ew_scatter<<<g, 256, 0, s>>>(n, cell_of, rank, starts, tmp);
    k_ew_sort<<<g, 256, 0, s>>>(n, c, 1.0 / rcut, cell_of, starts, tmp, (const P4<double>*)xyzq,
                                sidx, (P4<double>*)sx, (P4<float>*)sf);
  }
  return hipGetLastError();
}

hipError_t launch_ew_force(int n, const EwCells& c, const EwPair& p, const int* starts,
                           const int* sidx, const void* sx, const void* sf, const int* xofs,
                           const int* xlist, const double* erfcx, double* gx, double* gy, double* gz,
                           double* partials, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const unsigned g = (unsigned)((n + kEwWaves - 1) / kEwWaves);
  const P4<double>* x = (const P4<double>*)sx;
  const P4<float>* f = (const P4<float>*)sf;
  // no axis is short enough to visit all its cells: every image is a shift
  const bool fold = c.nc[0] <= 2 * c.reach[0] + 2 || c.nc[1] <= 2 * c.reach[1] + 1 ||
                    c.nc[2] <= 2 * c.reach[2] + 1;
  if (fold)
    k_ew_force<true><<<g, 64 * kEwWaves, 0, s>>>(n, c, p, starts, sidx, x, f, xofs, xlist, erfcx,
                                                 gx, gy, gz, partials);
  else
    k_ew_force<false><<<g, 64 * kEwWaves, 0, s>>>(n, c, p, starts, sidx, x, f, xofs, xlist,
                                                  erfcx, gx, gy, gz, partials);
  return hipGetLastError();
}

hipError_t launch_ew_finalize(const double* partials, int n, const double* q2, double self,
                              double* energy, hipStream_t s) {
  k_ew_finalize<<<1, 1024, 0, s>>>(partials, n, q2, kEwCountBlocks, self, energy);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ewald reciprocal sum (CpuEwaldRecip.cpp:87-147), FP64
// ---------------------------------------------------------------------------
// k-vectors of the cube |kx|,|ky|,|kz| <= kcut, x fastest as the reference
// loops, kept when 0 < kx^2+ky^2+kz^2 <= kcut^2.  One thread per k: its
// structure factor S(k) = sum q (cos, sin)(k.r) over all particles (staged
// through LDS, particle order), pek = pref exp(-k^2 sigma^2/2)/k^2, and the
// energy term pek |S|^2 (partial sums per workgroup).
constexpr int kErBlock = 256;

__device__ __forceinline__ bool er_kvec(const ErArgs& a, int idx, double* kv) {
  const int n1 = 2 * a.kcut + 1;
  const int kx = idx % n1 - a.kcut, ky = (idx / n1) % n1 - a.kcut, kz = idx / (n1 * n1) - a.kcut;
  const int k2 = kx * kx + ky * ky + kz * kz;
  if ((kx == 0 && ky == 0 && kz == 0) || k2 > a.kcut * a.kcut) return false;
  kv[0] = 2.0 * M_PI * ((double)kx) * a.ib[0];
  kv[1] = 2.0 * M_PI * ((double)ky) * a.ib[1];
  kv[2] = 2.0 * M_PI * ((double)kz) * a.ib[2];
  return true;
}

__global__ __launch_bounds__(kErBlock) void k_er_sfac(ErArgs a, const P4<double>* __restrict__ xyzq,
                                                      int n, double* __restrict__ sk,
                                                      double* __restrict__ partials) {
  __shared__ P4<double> sh[kErBlock];
  __shared__ double she[kErBlock / 64];
  const int idx = blockIdx.x * kErBlock + threadIdx.x;
  double kv[3] = {0, 0, 0};
  const bool live = idx < a.ncube && er_kvec(a, idx, kv);
  double re = 0.0, im = 0.0;
  for (int base = 0; base < n; base += kErBlock) {
    __syncthreads();
    if (base + (int)threadIdx.x < n) sh[threadIdx.x] = xyzq[base + threadIdx.x];
    __syncthreads();
    const int m = min(kErBlock, n - base);
    if (live)
      for (int i = 0; i < m; i++) {
        const P4<double> p = sh[i];
        const double kr = kv[0] * p.x + kv[1] * p.y + kv[2] * p.z;
        double sn, cs;
        sincos(kr, &sn, &cs);
        re += p.w * cs;
        im += p.w * sn;
      }
  }
  double e = 0.0;
  if (live) {
    const double ksq = kv[0] * kv[0] + kv[1] * kv[1] + kv[2] * kv[2];
    const double pek = a.pref * exp(-ksq * a.half_sigmasq) / ksq;
    e = pek * (re * re + im * im);
    sk[3 * (size_t)idx + 0] = re;
    sk[3 * (size_t)idx + 1] = im;
    sk[3 * (size_t)idx + 2] = pek;
  } else if (idx < a.ncube) {
    sk[3 * (size_t)idx + 2] = 0.0;  // outside the sphere: no term
  }
  const double w = wave_sum(e);
  if ((threadIdx.x & 63) == 0) she[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = (she[0] + she[1]) + (she[2] + she[3]);
}

// forces -dE/dr_i (CpuEwaldRecip.cpp:125-139): one thread per particle, the
// k-vectors in the reference's order, staged through LDS
__global__ __launch_bounds__(kErBlock) void k_er_force(ErArgs a, const P4<double>* __restrict__ xyzq,
                                                       int n, const double* __restrict__ sk,
                                                       double* __restrict__ fx,
                                                       double* __restrict__ fy,
                                                       double* __restrict__ fz) {
  __shared__ double shk[kErBlock][6];
  const int i = blockIdx.x * kErBlock + threadIdx.x;
  P4<double> p{0, 0, 0, 0};
  if (i < n) p = xyzq[i];
  double f0 = 0.0, f1 = 0.0, f2 = 0.0;
  for (int base = 0; base < a.ncube; base += kErBlock) {
    __syncthreads();
    const int k = base + threadIdx.x;
    if (k < a.ncube) {
      double kv[3];
      const bool ok = er_kvec(a, k, kv);
      shk[threadIdx.x][0] = kv[0];
      shk[threadIdx.x][1] = kv[1];
      shk[threadIdx.x][2] = kv[2];
      shk[threadIdx.x][3] = ok ? sk[3 * (size_t)k + 0] : 0.0;
      shk[threadIdx.x][4] = ok ? sk[3 * (size_t)k + 1] : 0.0;
      shk[threadIdx.x][5] = ok ? sk[3 * (size_t)k + 2] : 0.0;
    }
    __syncthreads();
    const int m = min(kErBlock, a.ncube - base);
    if (i < n)
      for (int j = 0; j < m; j++) {
        const double pek = shk[j][5];
        if (pek == 0.0) continue;
        const double kx = shk[j][0], ky = shk[j][1], kz = shk[j][2];
        const double re = shk[j][3], im = shk[j][4];
        const double kr = kx * p.x + ky * p.y + kz * p.z;
        double sn, cs;
        sincos(kr, &sn, &cs);
        const double fac = -pek * p.w * 2.0;
        f0 += fac * (re * (-kx * sn) + im * kx * cs);
        f1 += fac * (re * (-ky * sn) + im * ky * cs);
        f2 += fac * (re * (-kz * sn) + im * kz * cs);
      }
  }
  if (i < n) {
    fx[i] = f0;
    fy[i] = f1;
    fz[i] = f2;
  }
}

__global__ void k_er_finalize(const double* __restrict__ partials, int nb, double* energy) {
  __shared__ double sh[256];
  double s = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) s += partials[b];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) energy[0] = sh[0];
}

int ewald_recip_blocks(const ErArgs& a) { return (a.ncube + kErBlock - 1) / kErBlock; }

hipError_t launch_ewald_recip(const ErArgs& a, const void* xyzq, int n, double* sk,
                              double* partials, double* fx, double* fy, double* fz,
                              double* energy, hipStream_t s) {
  const int nb = ewald_recip_blocks(a);
  k_er_sfac<<<nb, kErBlock, 0, s>>>(a, (const P4<double>*)xyzq, n, sk, partials);
  k_er_finalize<<<1, 256, 0, s>>>(partials, nb, energy);
  if (n > 0 && fx)
    k_er_force<<<(n + kErBlock - 1) / kErBlock, kErBlock, 0, s>>>(a, (const P4<double>*)xyzq, n,
                                                                  sk, fx, fy, fz);
  return hipGetLastError();
}

}  // namespace gse
