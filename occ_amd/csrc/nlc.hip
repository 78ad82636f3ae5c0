// nlc.hip -- VV10 non-local correlation on the GPU:
// NonLocalCorrelationFunctional::vv10 (src/dft/nonlocal_correlation.cpp:
// 246-306) with vv10_kernel (nonlocal_correlation.cpp:37-103).
//
// The reference sums, for each grid point i with rho_i >= 1e-8, over the
// points j < i in its input order (each pair counted twice, the self term
// once):
//   F_i = -1.5 [rho_i w_i / (2 k_i^3) + sum_j 2 rho_j w_j / (g_i g_j (g_i + g_j))]
//   U_i = [self] + sum_j t_ij (1/g_i + 1/(g_i + g_j)),  W_i = sum_j t_ij (...) r_ij^2
// with g = r^2 omega0 + kappa.  The energy is the symmetric double sum; the
// per-point potential depends on the point order, so the pair kernel works
// in input order (the context records each padded point's input index).
//
// Layout: the context's points are in leaf order; k_vv10_prep scatters each
// real point's (x, y, z, rho w, omega0, kappa, rho) into input-order planes
// of npts; k_vv10_pairs gives partial sums of F, U, W per input point and
// segment of j (nlc_segments.hpp); k_vv10_coef adds them up per leaf point and forms the weighted
// exc / vrho / vsigma and the GGA Vxc coefficients, which the restricted Vxc
// kernel contracts (Vxc = ktmp + ktmp^T, nonlocal_correlation.cpp:295-303).
#include <hip/hip_runtime.h>

#include <cmath>
#include <stdexcept>
#include <string>

#include "kernels.hpp"
#include "nlc_segments.hpp"

namespace occxc {
namespace {

constexpr double kVvPi = 3.14159265358979323846;
constexpr double kVvRhoMin = 1e-8;  // nonlocal_correlation.cpp:68,77

enum : int { kX = 0, kY, kZ, kRW, kOM, kKA, kRHO, kNlcPlanes };

void check(const char *what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

__device__ inline double block_sum(double v, double *s_red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) s_red[wave] = v;
  __syncthreads();
  const double r = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
  __syncthreads();
  return r;
}

struct Vv10Consts {
  double C, kappa_factor, beta;
};

Vv10Consts vv10_consts(double b, double C) {
  Vv10Consts k;
  k.C = C;
  k.kappa_factor = b * 1.5 * kVvPi * std::pow(9.0 * kVvPi, -1.0 / 6.0);
  k.beta = std::pow(3.0 / (b * b), 0.75) / 32.0;
  return k;
}

// omega0 and kappa of one point (nonlocal_correlation.cpp:53-61)
__device__ inline void vv10_point(double rho, double sigma, const Vv10Consts &k, double &tmp,
                                  double &omega0, double &kappa) {
  const double pi4_3 = 4.0 * kVvPi / 3.0;
  tmp = sigma / (rho * rho);
  tmp = k.C * tmp * tmp;
  omega0 = sqrt(tmp + pi4_3 * rho);
  kappa = k.kappa_factor * pow(rho, 1.0 / 6.0);
}

// leaf order -> input order (one block per leaf, one thread per point)
__global__ __launch_bounds__(256) void k_vv10_prep(BuildArgs a, const double *__restrict__ rho4,
                                                   const int *__restrict__ porig, Vv10Consts k,
                                                   double *__restrict__ nlc, long long npts) {
  const LeafDev L = a.leaves[blockIdx.x];
  const int p = threadIdx.x;
  if (p >= L.n) return;
  const long long q = L.pt_off + p, P = a.ptot;
  const long long o = porig[q];
  if (o < 0 || o >= npts) return;
  const double rho = rho4[q];
  const double gx = rho4[P + q], gy = rho4[2 * P + q], gz = rho4[3 * P + q];
  double tmp, om, ka;
  vv10_point(rho, gx * gx + gy * gy + gz * gz, k, tmp, om, ka);
  nlc[kX * npts + o] = a.px[q];
  nlc[kY * npts + o] = a.py[q];
  nlc[kZ * npts + o] = a.pz[q];
  nlc[kRW * npts + o] = rho * a.pw[q];
  nlc[kOM * npts + o] = om;
  nlc[kKA * npts + o] = ka;
  nlc[kRHO * npts + o] = rho;
}

// 1/x for the pair denominators: the hardware reciprocal refined by two
// Newton-Raphson steps, r <- r + r (1 - x r) (within about an ulp; x lies in
// [1e-3, 1e30] in ordinary use: g >= kappa(1e-8) ~ 0.7, so no scaling is needed)
__device__ inline double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  r = fma(r, fma(-x, r, 1.0), r);
  return r;
}

// The same for four numbers with one hardware reciprocal: the product's,
// refined by one third-order step r <- r + r (e + e^2), e = 1 - x r, times the
// other three.  The product stays in range for the x of vv10_narrow points (at
// most 1e56, at least 1e-30 each).
__device__ inline void recip4(double x0, double x1, double x2, double x3, double (&r)[4]) {
  const double a = x0 * x1, b = x2 * x3, x = a * b;
  double q = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, q, 1.0);
  q = fma(q, fma(e, e, e), q);
  const double qa = q * b, qb = q * a;
  r[0] = qa * x1;
  r[1] = qa * x0;
  r[2] = qb * x3;
  r[3] = qb * x2;
}

// Points whose pair denominators (below) recip4 may take: coordinates within
// 1e3 Bohr and omega0, kappa at most 1e4 give g <= 1.3e11, and kappa >= 1e-6
// bounds it below.  Others (far larger systems, a tiny b) take one reciprocal
// a pair.
__device__ inline bool vv10_narrow(double x, double y, double z, double om, double ka) {
  return fabs(x) <= 1e3 && fabs(y) <= 1e3 && fabs(z) <= 1e3 && om <= 1e4 && ka <= 1e4 && ka >= 1e-6;
}

struct VvPoint {
  double x, y, z, om, ka, f, u, w;
};

// One pair's terms up to its reciprocal: R = 1 / ((g_i s)^2 g_j), s = g_i + g_j,
// gives t = 2 rho_j w_j / (g_i g_j s) = q (g_i s) R and t (1/g_i + 1/s) =
// q (s + g_i) R.
struct VvPair {
  double r2, gis, h, den;
};
__device__ inline VvPair vv_pair(const VvPoint &p, const double2 &xy, const double2 &zq,
                                 const double2 &ok) {
  const double dx = p.x - xy.x, dy = p.y - xy.y, dz = p.z - zq.x;
  VvPair v;
  v.r2 = dx * dx + dy * dy + dz * dz;
  const double gi = v.r2 * p.om + p.ka, gj = v.r2 * ok.x + ok.y, s = gi + gj;
  v.gis = gi * s;
  v.h = s + gi;
  v.den = v.gis * v.gis * gj;
  return v;
}
__device__ inline void vv_add(VvPoint &p, const VvPair &v, double q, double R) {
  const double qr = q * R;
  p.f += qr * v.gis;
  const double tu = qr * v.h;
  p.u += tu;
  p.w += tu * v.r2;
}

// Partial F, U, W of every input point i over the points j < i of one segment.
// Block (b, seg), b heaviest first, owns points [512 b, 512 b + 512), two a
// thread, and walks the segment's j tiles up to its own; a j's data is read
// from LDS once for two pairs, and two j's four pairs share one reciprocal.
// Dead j (rho_j < 1e-8, or beyond npts) enter with weight 0, which adds exactly
// 0; the block's own two tiles run pair by pair and stop at i.  FP64
// VALU-bound: 23 instruction slots a pair (26 with a reciprocal each, 24.5 with
// one for two).  (H2O)16 / def2-SVP, 50 x 110 grid, 3.5e10 pairs: 32.4 ms with
// one workgroup per 256 points and a reciprocal each, 22.0 ms now.
__global__ __launch_bounds__(256) void k_vv10_pairs(const double *__restrict__ nlc, long long npts,
                                                    int seg_tiles, double *__restrict__ part) {
  __shared__ double2 s_xy[kVvTile], s_zq[kVvTile], s_ok[kVvTile];
  const long long b = (long long)gridDim.x - 1 - blockIdx.x;
  const int seg = blockIdx.y;
  if (seg >= vv_block_segs(b, npts, seg_tiles)) return;
  const long long jt0 = (long long)seg * seg_tiles;
  const long long jt1 = min(jt0 + seg_tiles, vv_last_tile(b, npts) + 1);
  VvPoint p[2];
  long long i[2];
  bool live[2], wide = false;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    i[k] = b * kVvRows + k * kVvTile + threadIdx.x;
    live[k] = i[k] < npts && nlc[kRHO * npts + i[k]] >= kVvRhoMin;
    p[k] = VvPoint{0, 0, 0, 0, 1, 0, 0, 0};
    if (live[k]) {
      p[k].x = nlc[kX * npts + i[k]];
      p[k].y = nlc[kY * npts + i[k]];
      p[k].z = nlc[kZ * npts + i[k]];
      p[k].om = nlc[kOM * npts + i[k]];
      p[k].ka = nlc[kKA * npts + i[k]];
      wide = wide || !vv10_narrow(p[k].x, p[k].y, p[k].z, p[k].om, p[k].ka);
      if (seg == 0) {
        p[k].f = nlc[kRW * npts + i[k]] / (2 * p[k].ka * p[k].ka * p[k].ka);
        p[k].u = p[k].f * (1.0 / p[k].ka + 1.0 / (2 * p[k].ka));
      }
    }
  }
  const bool any = __syncthreads_or(live[0] || live[1]);
  const bool wide_i = __syncthreads_or(wide);
  for (long long jt = jt0; any && jt < jt1; ++jt) {
    __syncthreads();
    const long long j = jt * kVvTile + threadIdx.x;
    const bool lj = j < npts && nlc[kRHO * npts + j] >= kVvRhoMin;
    double2 xy{0, 0}, zq{0, 0}, ok{0, 1};
    if (lj) {
      xy = double2{nlc[kX * npts + j], nlc[kY * npts + j]};
      zq = double2{nlc[kZ * npts + j], 2.0 * nlc[kRW * npts + j]};
      ok = double2{nlc[kOM * npts + j], nlc[kKA * npts + j]};
    }
    s_xy[threadIdx.x] = xy;
    s_zq[threadIdx.x] = zq;
    s_ok[threadIdx.x] = ok;
    const bool wide_j = __syncthreads_or(lj && !vv10_narrow(xy.x, xy.y, zq.x, ok.x, ok.y));
    if (!wide_i && !wide_j && jt < 2 * b) {
#pragma unroll 2
      for (int jj = 0; jj < kVvTile; jj += 2) {
        VvPair v[4];
        double q[2], r[4];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const double2 a = s_xy[jj + m], c = s_zq[jj + m], d = s_ok[jj + m];
          q[m] = c.y;
#pragma unroll
          for (int k = 0; k < 2; ++k) v[2 * m + k] = vv_pair(p[k], a, c, d);
        }
        recip4(v[0].den, v[1].den, v[2].den, v[3].den, r);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int k = 0; k < 2; ++k) vv_add(p[k], v[2 * m + k], q[m], r[2 * m + k]);
      }
      continue;
    }
    for (int jj = 0; jj < kVvTile; ++jj) {
      const double2 a = s_xy[jj], c = s_zq[jj], d = s_ok[jj];
      const long long jg = jt * kVvTile + jj;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (jg >= i[k]) continue;
        const VvPair v = vv_pair(p[k], a, c, d);
        vv_add(p[k], v, c.y, recip(v.den));
      }
    }
  }
  double *out = part + 3 * (long long)seg * npts;
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (i[k] < npts) {
      out[i[k]] = live[k] ? p[k].f * -1.5 : 0.0;
      out[npts + i[k]] = live[k] ? p[k].u : 0.0;
      out[2 * npts + i[k]] = live[k] ? p[k].w : 0.0;
    }
}

// input order -> leaf order: weighted exc, vrho, vsigma (nonlocal_correlation.
// cpp:94-101), the energy and N_elec partials of the leaf, and the Vxc
// coefficients c0 = vrho / 2, c_k = 2 vsigma d_k rho (nonlocal_correlation.cpp:
// 295-303).  A point with rho < 1e-8 keeps exc = vrho = beta w, vsigma = 0.
__global__ __launch_bounds__(256) void k_vv10_coef(BuildArgs a, const double *__restrict__ rho4,
                                                   const int *__restrict__ porig, Vv10Consts k,
                                                   const double *__restrict__ part, long long npts,
                                                   int seg_tiles) {
  __shared__ double s_red[4];
  const int leaf = blockIdx.x;
  const LeafDev L = a.leaves[leaf];
  const int p = threadIdx.x;
  const bool live = p < L.np, real = p < L.n;
  const long long q = L.pt_off + p, P = a.ptot;
  double e_part = 0.0, n_part = 0.0, c[4] = {0, 0, 0, 0};
  if (real) {
    const long long o = porig[q];
    const double rho = rho4[q];
    const double g[3] = {rho4[P + q], rho4[2 * P + q], rho4[3 * P + q]};
    const double sigma = g[0] * g[0] + g[1] * g[1] + g[2] * g[2];
    const double w = a.pw[q];
    double vr = k.beta * w, vs = 0.0, ex = k.beta * w;
    if (rho >= kVvRhoMin && o >= 0 && o < npts) {
      const double pi4_3 = 4.0 * kVvPi / 3.0;
      double tmp, om, ka;
      vv10_point(rho, sigma, k, tmp, om, ka);
      const double dom_dr = (0.5 * pi4_3 * rho - 2.0 * tmp) / om;
      const double dom_dg = sigma > 0.0 ? tmp * rho / (sigma * om) : 0.0;
      const double dka_dr = (1.0 / 6.0) * ka;
      // the segments that the point's block has, in order
      double F = 0.0, U = 0.0, W = 0.0;
      const int nseg = vv_block_segs(o / kVvRows, npts, seg_tiles);
      for (int g = 0; g < nseg; ++g) {
        const double *f = part + 3 * (long long)g * npts + o;
        F += f[0];
        U += f[npts];
        W += f[2 * npts];
      }
      ex = (k.beta + 0.5 * F) * w;
      vr = (k.beta + F + 1.5 * (U * dka_dr + W * dom_dr)) * w;
      vs = (1.5 * W * dom_dg) * w;
    }
    e_part = ex * rho;
    n_part = rho * w;
    c[0] = 0.5 * vr;
    for (int d = 0; d < 3; ++d) c[d + 1] = 2.0 * vs * g[d];
  }
  const double e = block_sum(e_part, s_red);
  const double n = block_sum(n_part, s_red);
  if (live)
    for (int d = 0; d < 4; ++d) a.coef[d * P + q] = c[d];
  if (threadIdx.x == 0) {
    a.leaf_part[2 * leaf] = e;
    a.leaf_part[2 * leaf + 1] = n;
    a.leaf_active[leaf] = 1;
  }
}

} // namespace

size_t nlc_buffer_elems(long long npts) {
  return (size_t)(kNlcPlanes + 3 * vv_segs(npts).n) * (size_t)npts;
}

void launch_vv10(const BuildArgs &a, const double *rho4, const int *porig, double b, double C,
                 double *nlc, long long npts, hipStream_t s) {
  if (a.nleaves == 0 || npts == 0) return;
  const Vv10Consts k = vv10_consts(b, C);
  const VvSegs g = vv_segs(npts);
  double *part = nlc + (size_t)kNlcPlanes * npts;
  // points outside every leaf keep rho = 0 and so stay out of the sums
  launch_zero(nlc + kRHO * npts, npts, s);
  k_vv10_prep<<<a.nleaves, 256, 0, s>>>(a, rho4, porig, k, nlc, npts);
  check("k_vv10_prep");
  k_vv10_pairs<<<dim3((unsigned)vv_blocks(npts), g.n), 256, 0, s>>>(nlc, npts, g.tiles, part);
  check("k_vv10_pairs");
  k_vv10_coef<<<a.nleaves, 256, 0, s>>>(a, rho4, porig, k, part, npts, g.tiles);
  check("k_vv10_coef");
}

} // namespace occxc
