// grad.hip -- XC contribution to the nuclear gradient on gfx950.
//
// Replaces DFT::compute_xc_gradient_impl<d, Restricted> (include/occ/dft/
// dft.h:598-749) and kernels::process_grid_block_gradient<d, Restricted>
// (src/dft/dft_gradient_kernels.cpp:473-552).  The reference forms, per leaf,
// three m x m matrices V_k (accumulate_gradient_contribution_R, :26-90) and
// contracts them with 2 P (P = 2 D):
//   G(k, A) -= sum_{mu on A} sum_nu 2 P(mu,nu) V_k(mu,nu),
//   V_k(mu,nu) = sum_p [d_k phi_mu aow_nu + aow_k,mu phi_nu]          (GGA)
//   aow   = c0 phi + sum_j c_j d_j phi,  aow_k = c0 d_k phi + sum_j c_j d_kj phi
// with the build's coefficients c0 = w vrho / 2 and c_j = 2 w vsigma d_j rho
// (for LDA c_j = 0 and V_k = d_k phi^T (w vrho phi)).  Summing over nu first
// gives the same number with two leaf GEMMs instead of three m x m ones:
//   G(k, A) = -2 sum_{mu on A} sum_p [d_k phi_mu U_mu + aow_k,mu T_mu],
//   T = Phi P (the density's own product), U = Aow P.
// One workgroup per (leaf, column block of AOs): it walks the leaf's points 64
// at a time, forms the products on the FP64 matrix cores from operands staged
// by direct-to-LDS loads, and adds the integrand into per-lane sums of its
// AOs.  The meta-GGA's tau terms (accumulate_gradient_contribution_R<2>,
// dft_gradient_kernels.cpp:152-172),
//   V_k += sum_j d_kj phi^T ((vtau / 2) d_j phi),
// contract to sum_p sum_j d_kj phi_mu (vtau / 2) T_j,mu with T_j = (d_j Phi) P;
// there U = c0 T + sum_j c_j T_j needs no product of its own.
// The per-AO sums go to gpart; two more kernels reduce them per atom in a
// fixed order (no atomics: the gradient repeats bit for bit).
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>
#include <type_traits>

#include "kernels.hpp"
#include "tile_dma.hpp"
#include "tile_shapes.hpp"

namespace occxc {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ d4 mma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <typename S> __device__ __forceinline__ d2 load2d(const S *p);
template <> __device__ __forceinline__ d2 load2d<double>(const double *p) {
  return *reinterpret_cast<const d2 *>(p);
}
template <> __device__ __forceinline__ d2 load2d<float>(const float *p) {
  const f2 v = *reinterpret_cast<const f2 *>(p);
  return d2{(double)v[0], (double)v[1]};
}

template <typename T> __device__ __forceinline__ const T *at(const T *base, unsigned bytes) {
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
}

// Staging of the gradient items.  A chunk is kGk AOs: their rows of the NQ
// planes at the item's 64 points ([plane][AO][point], as stored) and of P,
// gathered through the AO map ([AO][column], each double as two 4-byte pieces
// from two lanes).  NT products: 1 (LDA: T), 2 (GGA: T and U) or 4 (meta-GGA:
// T and the three T_j), 16 accumulator tiles a wavefront in all, so the
// meta-GGA's column blocks are half as wide.  Three chunk buffers, two chunks
// in flight; every wavefront issues the same number of loads for a chunk.
// Bound by HBM: the nine derivative planes of the integrand are read once
// (1.9e10 bytes on (H2O)32 / def2-SVP, FP64), the four of the products once per
// column block: 3.6e10 bytes past L2 in all.  PBE there 11.76 -> 6.48 ms (5.6
// TB/s) against the per-leaf form, which read the products' planes once per 32
// AOs through each lane's own loads (5.7e10 bytes); the TPSS terms of C11H24,
// 5.98 -> 2.40 ms for both spins (five products of two kernels then, four of one
// now; 2.59 ms while a half with one tile ran two).
constexpr int kGk = 8, kGp = kGradPoints;
template <typename S, int NT> struct GradDma {
  static constexpr int NS = 3;
  static constexpr int NQ = NT == 1 ? 1 : 4;
  static constexpr int CW = NT == 4 ? 64 : 128;              // widest column block
  static constexpr int PLANE = kGk * kGp * (int)sizeof(S);   // bytes of a plane's rows
  static constexpr int STAGE = NQ * PLANE + kGk * CW * 8;
  static constexpr int PI = PLANE / 1024;                    // loads of a plane
  static constexpr int PL = NQ == 4 ? PI : PI / 4 + (PI < 4);  // a wavefront's (LDA: shared out)
  static constexpr int LOADS = PL + 2 * (CW / 32);
  static constexpr int NC = NT == 1 ? 1 : NT == 2 ? 4 : 5;   // coefficient planes
};

// MFMA layout (v_mfma_f64_16x16x4f64): lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; accumulator register r of lane l holds row l/16 + 4r,
// column l%16.  Point row i of a 16-point tile is fed as point
// 4(i%4) + i/4, so lane group g's accumulator rows are the 4 consecutive
// points 4g..4g+3 (vector loads in the integrand).
template <typename S, int NT>
__device__ __forceinline__ void grad_item(const BuildArgs &a, const S *__restrict__ ao,
                                          const double *__restrict__ ao2,
                                          const int *__restrict__ ao_map, const DenItem &it,
                                          double *__restrict__ gpart, char *s_stage) {
  using P = GradDma<S, NT>;
  constexpr int CT = NT == 4 ? 2 : 4;  // column tiles of a wavefront
  const LeafDev L = a.leaves[it.leaf];
  double *gp = gpart + 3LL * (L.map_off + it.c0);
  const int t = threadIdx.x, lane = t & 63;
  if (!a.leaf_active[it.leaf]) {
    // skipped by the max-rho rule (dft_gradient_kernels.cpp:488-491)
    for (int i = t; i < 3 * it.wc; i += 256) gp[i] = 0.0;
    return;
  }
  const MolDev MD = a.mols[L.mol];
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int wp = wave & 1, wc = wave >> 1;
  const int hc = it.wc >> 1;
  const int pa = 4 * (l16 & 3) + (l16 >> 2);
  const long long cs = (long long)L.mp * L.np;
  const S *phi = ao + L.ao_off;
  // gradient of phi: cache components 1..3 (GGA) or the extra block (LDA);
  // Hessian xx,xy,xz,yy,yz,zz: the extra block (GGA)
  const double *x2 = ao2 + L.ao_off / a.ncomp * (NT == 1 ? 3 : 6);
  const double *Dm = a.D2 + MD.moff;
  const int *map = ao_map + L.map_off;
  // addresses are a wavefront-uniform base plus a 32-bit lane offset in bytes
  // (at most a leaf's plane, 16 MB): 64-bit ones per load fill the registers
  unsigned colbase[P::CW / 32];
#pragma unroll
  for (int cb = 0; cb < P::CW / 32; ++cb)
    colbase[cb] = 8u * map[it.c0 + min(32 * cb + (lane >> 1), it.wc - 1)] + 4u * (lane & 1);
  // plane rows: LPR lanes a row of 64 points, RPI rows a load
  constexpr int LPR = kGp * (int)sizeof(S) / 16, RPI = 64 / LPR;
  const int q0 = P::NQ == 4 ? wave : 0;
  const S *src = phi + q0 * cs;
  const unsigned loff = (unsigned)((lane / LPR) * L.np) * (unsigned)sizeof(S) + 16u * (lane % LPR);
  auto dma = [&](int p0, int k0, char *st) __attribute__((always_inline)) {
    long long kmap[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) kmap[r] = (long long)map[k0 + 2 * wave + r] * MD.nbf;
#pragma unroll
    for (int i = 0; i < P::PL; ++i) {
      // LDA: the plane's loads shared out over the wavefronts (with FP32
      // storage wavefronts w and w + 2 load the same rows)
      const int ii = P::NQ == 4 ? i : (wave + 4 * i) % P::PI;
      __builtin_amdgcn_global_load_lds(at(src + (long long)(k0 + ii * RPI) * L.np + p0, loff),
                                       st + q0 * P::PLANE + ii * 1024, 16, 0, 0);
    }
    char *sd = st + P::NQ * P::PLANE;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int cb = 0; cb < P::CW / 32; ++cb)
        __builtin_amdgcn_global_load_lds(at(Dm + kmap[r], colbase[cb]),
                                         sd + ((2 * wave + r) * P::CW + 32 * cb) * 8, 4, 0, 0);
  };
  double(*s_c)[kGp] = reinterpret_cast<double(*)[kGp]>(s_stage + P::NS * P::STAGE);
  const int nch = (L.m + kGk - 1) / kGk;
  // exactly the tiles that hold real AOs: the integrand reads its columns' rows
  // from memory, and in a block of 32 a half has one tile
  const int CTl = half_tiles(L.m - (it.c0 + wc * hc), hc);
  double gs[CT][3];
#pragma unroll
  for (int j = 0; j < CT; ++j) gs[j][0] = gs[j][1] = gs[j][2] = 0.0;
  auto body = [&](auto Cn) __attribute__((always_inline)) {
    constexpr int NCt = decltype(Cn)::value;
    for (int p0 = 0; p0 < L.n; p0 += kGp) {
      __syncthreads();  // the previous points' buffers and coefficients are consumed
      for (int c = 0; c < P::NS - 1 && c < nch; ++c) dma(p0, c * kGk, s_stage + c * P::STAGE);
      for (int i = t; i < P::NC * kGp; i += 256) {
        const int q = i / kGp, p = i % kGp;
        s_c[q][p] = q == 4 ? 2.0 * a.coef_tau[L.pt_off + p0 + p] : a.coef[q * a.ptot + L.pt_off + p0 + p];
      }
      d4 acc[NT][2][CT];
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < CT; ++j) acc[n][i][j] = d4{0.0, 0.0, 0.0, 0.0};
      const bool any = L.n > p0 + 32 * wp;  // the wavefront's points hold real ones
      double ca[2][4];
      int cur = 0;
      for (int c = 0; c < nch; ++c) {
        if (c + 1 < nch && c > 0) vmcnt_barrier<P::LOADS>();
        else vmcnt_barrier<0>();  // the first also waits for the coefficients
        if (NT == 2 && c == 0) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) ca[i][q] = s_c[q][32 * wp + 16 * i + pa];
        }
        const int nxt = cur == 0 ? P::NS - 1 : cur - 1;
        if (c + P::NS - 1 < nch) dma(p0, (c + P::NS - 1) * kGk, s_stage + nxt * P::STAGE);
        const S *sp = reinterpret_cast<const S *>(s_stage + cur * P::STAGE);
        const double *sd = reinterpret_cast<const double *>(s_stage + cur * P::STAGE + P::NQ * P::PLANE);
        if (NCt > 0 && any) {
#pragma unroll
          for (int ks = 0; ks < kGk / 4; ++ks) {
            const int kk = 4 * ks + g;
            double yv[NCt ? NCt : 1], xv[P::NQ][2];
#pragma unroll
            for (int j = 0; j < NCt; ++j) yv[j] = sd[kk * P::CW + wc * hc + 16 * j + l16];
#pragma unroll
            for (int q = 0; q < P::NQ; ++q)
#pragma unroll
              for (int i = 0; i < 2; ++i)
                xv[q][i] = (double)sp[(q * kGk + kk) * kGp + 32 * wp + 16 * i + pa];
            if constexpr (NT == 2) {
#pragma unroll
              for (int i = 0; i < 2; ++i)
                xv[1][i] = ca[i][0] * xv[0][i] + ca[i][1] * xv[1][i] + ca[i][2] * xv[2][i] +
                           ca[i][3] * xv[3][i];
            }
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
              for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NCt; ++j) acc[n][i][j] = mma(xv[n][i], yv[j], acc[n][i][j]);
          }
        }
        cur = cur + 1 == P::NS ? 0 : cur + 1;
      }
      // the integrand at the lane's 4 points of each tile for its AO column
      if (!any) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < NCt; ++j) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            // two points of a tile at a time; an opaque 0 (no instruction) and
            // a scheduling barrier keep each round's addresses, loads and
            // coefficients in the round: shared between rounds they spill
            int zero = 0;
            asm volatile("" : "+s"(zero));
            __builtin_amdgcn_sched_barrier(0);
            const int pl = 32 * wp + 16 * i + 4 * g + 2 * h + zero;
            const unsigned off = (unsigned)((it.c0 + wc * hc + 16 * j + l16) * L.np + p0 + pl);
            auto hess = [&](int k) __attribute__((always_inline)) {
              return load2d<double>(at(x2 + k * cs, 8u * off));
            };
            auto grad = [&](int k) __attribute__((always_inline)) {
              return load2d<S>(at(phi + k * cs, (unsigned)sizeof(S) * off));
            };
            if constexpr (NT == 1) {
              const d2 gx = hess(0), gy = hess(1), gz = hess(2);  // the gradient planes
#pragma unroll
              for (int r = 0; r < 2; ++r) {
                const double v = 2.0 * s_c[0][pl + r] * acc[0][i][j][2 * h + r];
                gs[j][0] += gx[r] * v;
                gs[j][1] += gy[r] * v;
                gs[j][2] += gz[r] * v;
              }
            } else {
              const d2 gx = grad(1), gy = grad(2), gz = grad(3);
              const d2 hxx = hess(0), hxy = hess(1), hxz = hess(2), hyy = hess(3), hyz = hess(4),
                       hzz = hess(5);
#pragma unroll
              for (int r = 0; r < 2; ++r) {
                const double c0 = s_c[0][pl + r], c1 = s_c[1][pl + r], c2 = s_c[2][pl + r],
                             c3 = s_c[3][pl + r];
                const double v = acc[0][i][j][2 * h + r];
                double u, b1 = c1 * v, b2 = c2 * v, b3 = c3 * v;
                if constexpr (NT == 2) {
                  u = acc[1][i][j][2 * h + r] + c0 * v;
                } else {
                  const double ct = s_c[P::NC - 1][pl + r];
                  const double tx = acc[1][i][j][2 * h + r], ty = acc[2][i][j][2 * h + r],
                               tz = acc[3][i][j][2 * h + r];
                  u = 2.0 * c0 * v + c1 * tx + c2 * ty + c3 * tz;
                  b1 += ct * tx;
                  b2 += ct * ty;
                  b3 += ct * tz;
                }
                gs[j][0] += gx[r] * u + (b1 * hxx[r] + b2 * hxy[r] + b3 * hxz[r]);
                gs[j][1] += gy[r] * u + (b1 * hxy[r] + b2 * hyy[r] + b3 * hyz[r]);
                gs[j][2] += gz[r] * u + (b1 * hxz[r] + b2 * hyz[r] + b3 * hzz[r]);
              }
            }
          }
        }
      }
    }
  };
  switch (CTl) {
  case 0: body(std::integral_constant<int, 0>{}); break;
  case 1: body(std::integral_constant<int, 1>{}); break;
  case 2: body(std::integral_constant<int, 2>{}); break;
  case 3: body(std::integral_constant<int, CT < 3 ? CT : 3>{}); break;
  default: body(std::integral_constant<int, CT>{}); break;
  }
  // sums over the four lane groups, then over the two wavefronts of a column half
  double *s_g = reinterpret_cast<double *>(s_stage);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double v = gs[j][k];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      gs[j][k] = v;
      if (wp == 1 && g == 0) s_g[3 * (64 * wc + 16 * j + l16) + k] = v;
    }
  __syncthreads();
  if (wp == 0 && g == 0)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      if (16 * j >= hc) break;
#pragma unroll
      for (int k = 0; k < 3; ++k)
        gp[3 * (wc * hc + 16 * j + l16) + k] = gs[j][k] + s_g[3 * (64 * wc + 16 * j + l16) + k];
    }
}

template <typename S, int NT>
__global__ __launch_bounds__(256, 2) void k_xc_grad(BuildArgs a, const S *__restrict__ ao,
                                                   const double *__restrict__ ao2,
                                                   const int *__restrict__ ao_map,
                                                   const DenItem *__restrict__ items,
                                                   double *__restrict__ gpart) {
  using P = GradDma<S, NT>;
  __shared__ __align__(16) char s_stage[P::NS * P::STAGE + P::NC * kGp * 8];
  static_assert(P::STAGE >= 3 * 128 * 8, "the column sums fit");
  const DenItem it = items[blockIdx.x];
  if (it.leaf < 0) return;
  grad_item<S, NT>(a, ao, ao2, ao_map, it, gpart, s_stage);
}

// Per-atom sums in a fixed order: block (A, y) sums every kGradSplit-th run of
// 256 entries of atom A (per-thread strided sums, then a fixed tree), then
// grad[3 A + k] = -2 times the sum of the atom's blocks.  gpart2: the beta spin
// of an unrestricted gradient (null otherwise).  With one block per atom a
// 96-atom cluster's 2e6 entries kept 96 of the 256 CUs busy for 134 us.
__global__ __launch_bounds__(256) void k_grad_reduce(const double *__restrict__ gpart,
                                                     const double *__restrict__ gpart2,
                                                     const int *__restrict__ atom_off,
                                                     const int *__restrict__ atom_ent,
                                                     double *__restrict__ red) {
  __shared__ double s_r[3][256];
  const int A = blockIdx.x;
  const int e0 = atom_off[A], e1 = atom_off[A + 1];
  double v[3] = {0.0, 0.0, 0.0};
  for (int i = e0 + blockIdx.y * 256 + threadIdx.x; i < e1; i += 256 * kGradSplit) {
    const long long e = 3LL * atom_ent[i];
    v[0] += gpart[e];
    v[1] += gpart[e + 1];
    v[2] += gpart[e + 2];
    if (gpart2) {
      v[0] += gpart2[e];
      v[1] += gpart2[e + 1];
      v[2] += gpart2[e + 2];
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) s_r[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int k = 0; k < 3; ++k) s_r[k][threadIdx.x] += s_r[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 3) red[(A * kGradSplit + blockIdx.y) * 3 + threadIdx.x] = s_r[threadIdx.x][0];
}

__global__ void k_grad_final(const double *__restrict__ red, int n3, double *__restrict__ grad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n3) return;
  double v = 0.0;
  for (int y = 0; y < kGradSplit; ++y) v += red[(i / 3 * kGradSplit + y) * 3 + i % 3];
  grad[i] = -2.0 * v;
}

void check(const char *what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

} // namespace

void launch_xc_gradient_partials(const BuildArgs &a, const void *ao, bool ao_fp32,
                                 const double *ao2, const DenItem *items, int nitems,
                                 double *gpart, hipStream_t s) {
  if (a.nleaves == 0 || nitems == 0) return;
  auto launch = [&](auto s_tag) {
    using S = decltype(s_tag);
    (a.deriv == 0 ? k_xc_grad<S, 1> : a.coef_tau ? k_xc_grad<S, 4> : k_xc_grad<S, 2>)
        <<<nitems, 256, 0, s>>>(a, static_cast<const S *>(ao), ao2, a.ao_map, items, gpart);
  };
  if (ao_fp32) launch(float{});
  else launch(double{});
  check("k_xc_grad");
}

void launch_grad_reduce(const double *gpart, const double *gpart2, int natoms,
                        const int *atom_off, const int *atom_ent, double *red, double *grad,
                        hipStream_t s) {
  k_grad_reduce<<<dim3(natoms, kGradSplit), 256, 0, s>>>(gpart, gpart2, atom_off, atom_ent, red);
  check("k_grad_reduce");
  k_grad_final<<<(3 * natoms + 255) / 256, 256, 0, s>>>(red, 3 * natoms, grad);
  check("k_grad_final");
}

} // namespace occxc
