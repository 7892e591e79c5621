// dwf_force.hip -- DWF fermion force kernels (FP64).
//
// Tensor products of the even-odd DWF force (the reference's lexical
// force_udiv1_D / _Ddag followed by tensorProd_5din,
// aforce_F_Domainwall_5din-tmpl.h:338-933, afield_Spinor-inc.h:322-370):
//   F_mu(x) (+)= scale * sum_{s,d} { [(1 - gamma_mu) Y(x + mu)]_{a,d,s} conj(B(x)_{b,d,s})
//                                  + [(1 + gamma_mu) B(x + mu)]_{a,d,s} conj(Y(x)_{b,d,s}) }
// (times bc when x + mu wraps), the first term for the D part, the second for the
// Ddag part.  One thread per (site, s); the sum over s runs through LDS inside the
// block.
// mult_generator (lib_alt_QXS/Force/Fermion/aforce_F.cpp:97-110):
//   F <- -2 at(U F).
#include <type_traits>

#include "dwf_device.h"
#include "dwf_kernels.h"

namespace dwf {

// acc += sum over the spins of [(1 -+ gamma_mu) v]_a conj(z_b), DIR = 2 mu (minus) or
// 2 mu + 1: (1 -+ gamma_mu) has rank two, so with the half spinors h of v and g of z
// the four spin terms are h1 conj(g1) + h2 conj(g2).
template <int DIR>
__device__ __forceinline__ void tensor_term(double (&acc)[18], const double (&v)[24],
                                            const double (&z)[24]) {
  double h1[6], h2[6], g1[6], g2[6];
  project<DIR>(v, h1, h2);
  project<DIR>(z, g1, g2);
  const double f = DIR >= 6 ? 0.5 : 1.0;   // the t projection doubles both
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    g1[c] *= f;
    g2[c] *= f;
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      double &re = acc[2 * (3 * a + b)], &im = acc[2 * (3 * a + b) + 1];
      re += h1[2 * a] * g1[2 * b] + h1[2 * a + 1] * g1[2 * b + 1];
      im += h1[2 * a + 1] * g1[2 * b] - h1[2 * a] * g1[2 * b + 1];
      re += h2[2 * a] * g2[2 * b] + h2[2 * a + 1] * g2[2 * b + 1];
      im += h2[2 * a + 1] * g2[2 * b] - h2[2 * a] * g2[2 * b + 1];
    }
}

// TERMS: 1 the D term, 2 the Ddag term, 3 both; b and y of the two parities;
// blockIdx.y = the parity of x.  Both terms and parities in one launch write F once
// (force_udiv read it back three times with a launch per term and parity).
// 32x16x16x24, Ls = 12: 4 x 187 -> 598 us; the L2 gather of the neighbour spinors is
// 290 us of it (4.2 GB), the rest latency at two waves per SIMD.
template <int TERMS>
__global__ void __launch_bounds__(256, 2)
k_force_tensor(double* __restrict__ F, const double* __restrict__ b0,
               const double* __restrict__ b1, const double* __restrict__ y0,
               const double* __restrict__ y1, const int* __restrict__ nbr, int Nx, int Ny, int Nz,
               int Nt, int bcx, int bcy, int bcz, int bct, int Ls, int spb, double scale,
               int accumulate) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* sh = reinterpret_cast<double*>(smem_raw);   // [spb][Ls][18]
  const int Vh = Nx / 2 * Ny * Nz * Nt;
  const size_t V = 2 * (size_t)Vh;
  const int parity = blockIdx.y;
  const double* bx = parity ? b1 : b0;    // at x
  const double* yx = parity ? y1 : y0;
  const double* bn = parity ? b0 : b1;    // at x + mu
  const double* yn = parity ? y0 : y1;
  const int tid = threadIdx.x;
  const int lsite = tid / Ls, ls = tid - lsite * Ls;
  const int site = xcd_block(blockIdx.x, gridDim.x) * spb + lsite;
  const bool valid = lsite < spb && site < Vh;
  const size_t own = (size_t)(valid ? site : 0) * 24 * Ls + ls;
  // coordinates of the output site
  int x = 0, y = 0, z = 0, t = 0;
  size_t lex = 0;
  if (valid) {
    const int Nx2 = Nx / 2;
    int r = site / Nx2;
    const int x2 = site - r * Nx2;
    y = r % Ny;
    r /= Ny;
    z = r % Nz;
    t = r / Nz;
    x = 2 * x2 + ((y + z + t + parity) & 1);
    lex = x + (size_t)Nx * (y + (size_t)Ny * (z + (size_t)Nz * t));
  }
  double zb[24], zy[24];
  if (valid) {
#pragma unroll
    for (int k = 0; k < 24; ++k) {
      if (TERMS & 1) zb[k] = bx[own + k * Ls];
      if (TERMS & 2) zy[k] = yx[own + k * Ls];
    }
  }
  auto direction = [&](auto dir, bool wraps, int bc) {
    constexpr int MU = decltype(dir)::value;
    double acc[18];
#pragma unroll
    for (int e = 0; e < 18; ++e) acc[e] = 0;
    if (valid) {
      const size_t nb =
          (size_t)nbr[((size_t)parity * 8 + 2 * MU) * Vh + site] * 24 * Ls + ls;
      double v[24];
      if (TERMS & 1) {
#pragma unroll
        for (int k = 0; k < 24; ++k) v[k] = yn[nb + k * Ls];
        tensor_term<2 * MU>(acc, v, zb);
      }
      if (TERMS & 2) {
#pragma unroll
        for (int k = 0; k < 24; ++k) v[k] = bn[nb + k * Ls];
        tensor_term<2 * MU + 1>(acc, v, zy);
      }
    }
    __syncthreads();
    if (valid) {
#pragma unroll
      for (int e = 0; e < 18; ++e) sh[(lsite * Ls + ls) * 18 + e] = acc[e];
    }
    __syncthreads();
    // the Ls threads of a site sum over s and write the 18 reals of F_mu(x)
    if (valid) {
      const double f = scale * (wraps ? (double)bc : 1.0);
      for (int e = ls; e < 18; e += Ls) {
        double sum = 0;
        for (int s = 0; s < Ls; ++s) sum += sh[(lsite * Ls + s) * 18 + e];
        double* dst = F + 18 * (lex + V * MU) + e;
        *dst = accumulate ? *dst + f * sum : f * sum;
      }
    }
  };
  direction(std::integral_constant<int, 0>{}, x == Nx - 1, bcx);
  direction(std::integral_constant<int, 1>{}, y == Ny - 1, bcy);
  direction(std::integral_constant<int, 2>{}, z == Nz - 1, bcz);
  direction(std::integral_constant<int, 3>{}, t == Nt - 1, bct);
}

hipError_t launch_force_tensor(double* F, int terms, const double* const* b,
                               const double* const* y, const int* nbr, const int* N,
                               const int* bc, int Ls, double scale, bool accumulate,
                               hipStream_t st) {
  const int Vh = N[0] / 2 * N[1] * N[2] * N[3];
  int spb = 256 / Ls;
  if (spb < 1) return hipErrorInvalidValue;
  while (spb > 1 && (size_t)spb * Ls * 18 * 8 > 64 * 1024) --spb;
  const size_t lds = (size_t)spb * Ls * 18 * 8;
  const dim3 grid((Vh + spb - 1) / spb, 2), block(spb * Ls);
#define FT(T)                                                                                    \
  hipLaunchKernelGGL(k_force_tensor<T>, grid, block, lds, st, F, b[0], b[1], y[0], y[1], nbr, N[0], \
                     N[1], N[2], N[3], bc[0], bc[1], bc[2], bc[3], Ls, spb, scale, accumulate ? 1 : 0)
  switch (terms) {
    case 1: FT(1); break;
    case 2: FT(2); break;
    case 3: FT(3); break;
    default: return hipErrorInvalidValue;
  }
#undef FT
  return hipGetLastError();
}

// F_mu(x) <- -2 at(U_mu(x) F_mu(x)); the links are taken from the packed
// forward entries (which carry the boundary factor bc) times bc, i.e. U_mu(x)
// for bc = +-1.
__global__ void __launch_bounds__(256)
k_mult_generator(double* __restrict__ F, const double* __restrict__ links, int Nx, int Ny,
                 int Nz, int Nt, int bcx, int bcy, int bcz, int bct) {
  const int Vh = Nx / 2 * Ny * Nz * Nt;
  const size_t V = 2 * (size_t)Vh;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= 2 * Vh) return;
  const int p = idx / Vh, s2 = idx - p * Vh;
  const int Nx2 = Nx / 2;
  int r = s2 / Nx2;
  const int x2 = s2 - r * Nx2;
  const int y = r % Ny;
  r /= Ny;
  const int z = r % Nz;
  const int t = r / Nz;
  const int x = 2 * x2 + ((y + z + t + p) & 1);
  const int xc[4] = {x, y, z, t};
  const int N[4] = {Nx, Ny, Nz, Nt};
  const int bc[4] = {bcx, bcy, bcz, bct};
  const size_t lex = x + (size_t)Nx * (y + (size_t)Ny * (z + (size_t)Nz * t));
  for (int mu = 0; mu < 4; ++mu) {
    const double f = (xc[mu] == N[mu] - 1) ? (double)bc[mu] : 1.0;
    const double* L = links + ((size_t)(p * 8 + 2 * mu) * 18) * Vh + s2;
    double u[18], fm[18], m[18];
    for (int e = 0; e < 18; ++e) u[e] = f * L[(size_t)e * Vh];
    double* Fp = F + 18 * (lex + V * mu);
    for (int e = 0; e < 18; ++e) fm[e] = Fp[e];
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) {
        double re = 0, im = 0;
        for (int c = 0; c < 3; ++c) {
          const double ur = u[2 * (3 * a + c)], ui = u[2 * (3 * a + c) + 1];
          const double vr = fm[2 * (3 * c + b)], vi = fm[2 * (3 * c + b) + 1];
          re += ur * vr - ui * vi;
          im += ur * vi + ui * vr;
        }
        m[2 * (3 * a + b)] = re;
        m[2 * (3 * a + b) + 1] = im;
      }
    // at(m) = (m - m^+)/2 - tr(m - m^+)/6, times -2
    double o[18];
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) {
        o[2 * (3 * a + b)] = 0.5 * (m[2 * (3 * a + b)] - m[2 * (3 * b + a)]);
        o[2 * (3 * a + b) + 1] = 0.5 * (m[2 * (3 * a + b) + 1] + m[2 * (3 * b + a) + 1]);
      }
    const double tr = (o[1] + o[9] + o[17]) / 3.0;
    o[1] -= tr;
    o[9] -= tr;
    o[17] -= tr;
    for (int e = 0; e < 18; ++e) Fp[e] = -2.0 * o[e];
  }
}

hipError_t launch_mult_generator(double* F, const double* links, int Nx, int Ny, int Nz, int Nt,
                                 const int* bc, hipStream_t st) {
  const int Vh = Nx / 2 * Ny * Nz * Nt;
  hipLaunchKernelGGL(k_mult_generator, dim3((2 * Vh + 255) / 256), dim3(256), 0, st, F, links, Nx,
                     Ny, Nz, Nt, bc[0], bc[1], bc[2], bc[3]);
  return hipGetLastError();
}

}  // namespace dwf
