// dwf_smear.hip -- stout smearing and plaquette kernels (FP64).
//
// One smearing level (APE staples with stout projection):
//   C_mu(x) = rho sum_{nu != mu} [ U_nu(x) U_mu(x+nu) U_nu(x+mu)^+
//                                 + U_nu(x-nu)^+ U_mu(x-nu) U_nu(x-nu+mu) ]
//   iQ = at(C_mu U_mu^+)   (anti-hermitian traceless part)
//   U'_mu(x) = exp(iQ) U_mu(x),  exp by the Cayley-Hamilton form of
//   Morningstar and Peardon, Phys. Rev. D 69 (2004) 054501.
// Same steps as src/lib_alt_QXS/Smear/asmear_APE-tmpl.h:183-223 and
// aprojection_Stout_SU3-tmpl.h:477-553, 897-977; one thread per (site, mu).
#include "dwf_device.h"
#include "dwf_kernels.h"
#include "dwf_su3.h"

namespace dwf {

__device__ M3 exp_iQ(const M3& iQ) {
  double n2 = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) n2 += iQ.a[i][j].r * iQ.a[i][j].r + iQ.a[i][j].i * iQ.a[i][j].i;
  M3 r;
  if (!(n2 > 1.0e-10)) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) r.a[i][j] = {i == j ? 1.0 : 0.0, 0.0};
    return r;
  }
  const M3 iQ2 = mul_nn(iQ, iQ);
  const M3 iQ3 = mul_nn(iQ, iQ2);
  // Q = -i iQ: c0 = det Q = -Im tr(iQ^3)/3, c1 = tr(Q^2)/2 = -Re tr(iQ^2)/2
  const double c0 = -(iQ3.a[0][0].i + iQ3.a[1][1].i + iQ3.a[2][2].i) / 3.0;
  const double c1 = -0.5 * (iQ2.a[0][0].r + iQ2.a[1][1].r + iQ2.a[2][2].r);
  const double c13r = sqrt(c1 / 3.0);
  const double c0max = 2.0 * c13r * c13r * c13r;
  double ratio = c0 / c0max;
  ratio = fmin(1.0, fmax(-1.0, ratio));
  const double theta = acos(ratio);
  const double u = c13r * cos(theta / 3.0);
  const double w = sqrt(c1) * sin(theta / 3.0);
  const double xi0 = (w == 0.0) ? 1.0 : sin(w) / w;
  const double u2 = u * u, w2 = w * w, cw = cos(w);
  const cplx emiu = {cos(u), -sin(u)};
  const cplx e2iu = {cos(2.0 * u), sin(2.0 * u)};
  const cplx h0 = cadd(cscal(u2 - w2, e2iu),
                       cmul(emiu, cplx{8.0 * u2 * cw, 2.0 * u * (3.0 * u2 + w2) * xi0}));
  const cplx t1 = cmul(emiu, cplx{2.0 * u * cw, -(3.0 * u2 - w2) * xi0});
  const cplx h1 = {2.0 * u * e2iu.r - t1.r, 2.0 * u * e2iu.i - t1.i};
  const cplx t2 = cmul(emiu, cplx{cw, 3.0 * u * xi0});
  const cplx h2 = {e2iu.r - t2.r, e2iu.i - t2.i};
  const double fden = 1.0 / (9.0 * u2 - w2);
  const cplx f0 = cscal(fden, h0), f1 = cscal(fden, h1), f2 = cscal(fden, h2);
  // exp(iQ) = f0 + f1 Q + f2 Q^2 with Q = -i iQ, Q^2 = -iQ^2
  const cplx f1mi = {f1.i, -f1.r};  // f1 * (-i)
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx v = cmul(f1mi, iQ.a[i][j]);
      const cplx q2 = cmul(f2, iQ2.a[i][j]);
      v.r -= q2.r;
      v.i -= q2.i;
      if (i == j) v = cadd(v, f0);
      r.a[i][j] = v;
    }
  return r;
}

// One wave per (mu, 64 consecutive sites), the four directions of a chunk next to
// each other: their staples share links in L2.  From the chunked form these kernels
// run at the 14.5 TB/s that gathers reach in L2 (19, 20 and 37 matrices per link at
// 32x16x16x24: smearing 279 -> 159 us, force link part 358 -> 264, staple part 428 ->
// 284); from the Field_G rows the L1's line lookups bound them, and gathering the
// rows through LDS took 183, 330 and 320 us.
struct GaugeWave {
  int mu, first, lane;
  dbl2v_t* sh;
  __device__ __forceinline__ GaugeWave(dbl2v_t* slots) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = xcd_block(blockIdx.x, gridDim.x) * 2 + wave;
    mu = w & 3;
    first = (w >> 2) * 64;
    lane = threadIdx.x & 63;
    sh = slots + wave * kRowsLds;
  }
};

// Field_G -> chunked form (see dwf_su3.h); 41 us at 32x16x16x24, a copy's time.
template <bool WIDE>
__global__ void __launch_bounds__(128)
k_gauge_chunk(double* __restrict__ Uc, const double* __restrict__ U, GaugeLat L) {
  __shared__ dbl2v_t slots[2 * kRowsLds];
  const GaugeWave g(slots);
  const M3 m = rows_load<WIDE>(U + (size_t)18 * L.V * g.mu, g.first, L.V, g.sh);
  store3c(reinterpret_cast<dbl2v_t*>(Uc) + chunked_mu(L) * g.mu, g.first + g.lane, m);
}

// C_mu(x) = rho sum_{nu != mu} (upper + lower staple), U in chunked form
__device__ __forceinline__ M3 staple_sum(const double* __restrict__ Uc, const GaugeLat& L,
                                         const GaugeSite& x, int mu, double rho) {
  const size_t vol = chunked_mu(L);
  const dbl2v_t* u0 = reinterpret_cast<const dbl2v_t*>(Uc);
  const dbl2v_t* um = u0 + vol * mu;
  const int pm = x.off(L, mu, 1);
  M3 C = m3_zero();
  for (int i = 0; i < 3; ++i) {
    const int nu = i + (i >= mu ? 1 : 0);
    const dbl2v_t* un = u0 + vol * nu;
    const int pn = x.off(L, nu, 1), mn = x.off(L, nu, -1);
    // upper: U_nu(x) [U_mu(x+nu) U_nu(x+mu)^+]
    M3 t = mul_nd(load3c(um, x.s + pn), load3c(un, x.s + pm));
    m3_axpy(C, rho, mul_nn(load3c(un, x.s), t));
    // lower: U_nu(x-nu)^+ [U_mu(x-nu) U_nu(x-nu+mu)]
    t = mul_nn(load3c(um, x.s + mn), load3c(un, x.s + mn + pm));
    m3_axpy(C, rho, mul_dn(load3c(un, x.s + mn), t));
  }
  return C;
}

// One smearing level from the chunked links; Unext: the same level in chunked form
// for the one after it (nullptr: not wanted).
template <bool WIDE>
__global__ void __launch_bounds__(128, 2)
k_stout(double* __restrict__ Uout, double* __restrict__ Unext, const double* __restrict__ Uc,
        GaugeLat L, double rho) {
  __shared__ dbl2v_t slots[2 * kRowsLds];
  const GaugeWave g(slots);
  const GaugeSite x(L, g.first + g.lane);
  const M3 C = staple_sum(Uc, L, x, g.mu, rho);
  const M3 U = load3c(reinterpret_cast<const dbl2v_t*>(Uc) + chunked_mu(L) * g.mu, x.s);
  const M3 iQ = at3(mul_nd(C, U));
  const M3 V = mul_nn(exp_iQ(iQ), U);
  if (Unext) store3c(reinterpret_cast<dbl2v_t*>(Unext) + chunked_mu(L) * g.mu, g.first + g.lane, V);
  rows_store<WIDE>(Uout + (size_t)18 * L.V * g.mu, g.first, L.V, g.sh, V);
}

size_t gauge_chunked_bytes(size_t V) { return chunked_doubles(V) * sizeof(double); }

hipError_t launch_gauge_chunk(double* Uc, const double* U, const int* dims, hipStream_t st) {
  const GaugeLat L = gauge_lat(dims);
  const dim3 grid(2 * L.chunks), block(128);
  if (m3_wide(U)) hipLaunchKernelGGL(k_gauge_chunk<true>, grid, block, 0, st, Uc, U, L);
  else hipLaunchKernelGGL(k_gauge_chunk<false>, grid, block, 0, st, Uc, U, L);
  return hipGetLastError();
}

hipError_t launch_stout(double* Uout, double* Unext, const double* Uc, const int* dims, double rho,
                        hipStream_t st) {
  const GaugeLat L = gauge_lat(dims);
  const dim3 grid(2 * L.chunks), block(128);
  if (m3_wide(Uout))
    hipLaunchKernelGGL(k_stout<true>, grid, block, 0, st, Uout, Unext, Uc, L, rho);
  else
    hipLaunchKernelGGL(k_stout<false>, grid, block, 0, st, Uout, Unext, Uc, L, rho);
  return hipGetLastError();
}

// ---- stout force recursion --------------------------------------------------
// One level of AForceSmear_APE::force_udiv (lib_alt_QXS/Smear/aforceSmear_APE-tmpl.h:
// 157-206): Sigma = dS/dU from Sigma' = dS/dU' of U' = exp(iQ) U.  Per link, the
// Morningstar-Peardon chain rule (AProjection_Stout_SU3::force_recursive,
// aprojection_Stout_SU3-tmpl.h:691-895):
//   Gamma = tr(U S' B1) Q + tr(U S' B2) Q^2 + f1 U S' + f2 (Q U S' + U S' Q),
//   iLambda = at(i Gamma),  iTheta = iLambda U,  Xi = S' exp(iQ) + C^+ iLambda,
// then Sigma_mu(x) = Xi + rho sum_nu (six staple products of U and iTheta).

__device__ __forceinline__ M3 m3_poly(cplx c0, cplx c1, cplx c2, const M3& Q, const M3& Q2) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx v = cadd(cmul(c1, Q.a[i][j]), cmul(c2, Q2.a[i][j]));
      if (i == j) v = cadd(v, c0);
      r.a[i][j] = v;
    }
  return r;
}
__device__ __forceinline__ cplx m3_tr(const M3& x) {
  return cadd(cadd(x.a[0][0], x.a[1][1]), x.a[2][2]);
}
// tr(x y)
__device__ __forceinline__ cplx m3_trm(const M3& x, const M3& y) {
  cplx s = {0.0, 0.0};
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) s = cadd(s, cmul(x.a[i][j], y.a[j][i]));
  return s;
}
__device__ __forceinline__ cplx cexp_i(double phi) { return {cos(phi), sin(phi)}; }

__device__ double stout_xi1(double w) {
  if (w < 0.25) {
    const double w2 = w * w;
    return -1.0 / 3.0 +
           w2 * (1.0 / 30.0 + w2 * (-1.0 / 840.0 + w2 * (1.0 / 45360.0 - w2 / 3991680.0)));
  }
  return (w * cos(w) - sin(w)) / (w * w * w);
}

template <bool WIDE>
__global__ void __launch_bounds__(128, 2)
k_stout_force_link(double* Sigma, double* __restrict__ iTheta, const double* Sigmap,
                   const double* __restrict__ Uc, GaugeLat L, double rho) {
  __shared__ dbl2v_t slots[2 * kRowsLds];
  const GaugeWave gw(slots);
  const GaugeSite x(L, gw.first + gw.lane);
  const size_t off = (size_t)18 * L.V * gw.mu, offc = chunked_mu(L) * gw.mu;
  const M3 C = staple_sum(Uc, L, x, gw.mu, rho);
  const dbl2v_t* ul = reinterpret_cast<const dbl2v_t*>(Uc) + offc;
  M3 iQ, US;
  {
    const M3 U = load3c(ul, x.s);
    iQ = at3(mul_nd(C, U));
    US = mul_nn(U, rows_load<WIDE>(Sigmap + off, gw.first, L.V, gw.sh));
  }
  double n2 = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) n2 += iQ.a[i][j].r * iQ.a[i][j].r + iQ.a[i][j].i * iQ.a[i][j].i;
  M3 eiQ = m3_zero(), iGam = m3_zero();
#pragma unroll
  for (int i = 0; i < 3; ++i) eiQ.a[i][i].r = 1.0;
  if (n2 > 1.0e-10) {
    const M3 iQ2 = mul_nn(iQ, iQ);
    M3 Q, Q2;   // Q = -i iQ, Q^2 = -iQ^2
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        Q.a[i][j] = {iQ.a[i][j].i, -iQ.a[i][j].r};
        Q2.a[i][j] = {-iQ2.a[i][j].r, -iQ2.a[i][j].i};
      }
    const double q3 = m3_trm(iQ, iQ2).i;
    const double c0 = -(q3) / 3.0;
    const double c1 = -0.5 * (iQ2.a[0][0].r + iQ2.a[1][1].r + iQ2.a[2][2].r);
    const double c13r = sqrt(c1 / 3.0);
    const double ratio = fmin(1.0, fmax(-1.0, c0 / (2.0 * c13r * c13r * c13r)));
    const double theta = acos(ratio);
    const double u = c13r * cos(theta / 3.0), w = sqrt(c1) * sin(theta / 3.0);
    const double u2 = u * u, w2 = w * w, cw = cos(w);
    const double xi0 = (w == 0.0) ? 1.0 : sin(w) / w;
    const double xi1 = stout_xi1(w);
    const cplx emiu = cexp_i(-u), e2iu = cexp_i(2.0 * u);
    // f_j
    const double fd = 1.0 / (9.0 * u2 - w2);
    const cplx f0 = cscal(fd, cadd(cscal(u2 - w2, e2iu),
                                   cmul(emiu, cplx{8.0 * u2 * cw, 2.0 * u * (3.0 * u2 + w2) * xi0})));
    const cplx f1 = cscal(fd, cadd(cscal(2.0 * u, e2iu),
                                   cmul(emiu, cplx{-2.0 * u * cw, (3.0 * u2 - w2) * xi0})));
    const cplx f2 = cscal(fd, cadd(e2iu, cmul(emiu, cplx{-cw, -3.0 * u * xi0})));
    // r_j^(1), r_j^(2)
    const cplx r01 = cadd(cmul(cplx{2.0 * u, 2.0 * (u2 - w2)}, e2iu),
                          cmul(emiu, cplx{16.0 * u * cw + 2.0 * u * (3.0 * u2 + w2) * xi0,
                                          -8.0 * u2 * cw + 2.0 * (9.0 * u2 + w2) * xi0}));
    const cplx r11 = cadd(cmul(cplx{2.0, 4.0 * u}, e2iu),
                          cmul(emiu, cplx{-2.0 * cw + (3.0 * u2 - w2) * xi0,
                                          2.0 * u * cw + 6.0 * u * xi0}));
    const cplx r21 = cadd(cmul(cplx{0.0, 2.0}, e2iu),
                          cmul(emiu, cplx{-3.0 * u * xi0, cw - 3.0 * xi0}));
    const cplx r02 = cadd(cscal(-2.0, e2iu),
                          cmul(emiu, cplx{-8.0 * u2 * xi0, 2.0 * u * (cw + xi0 + 3.0 * u2 * xi1)}));
    const cplx r12 = cmul(emiu, cplx{2.0 * u * xi0, -cw - xi0 + 3.0 * u2 * xi1});
    const cplx r22 = cmul(emiu, cplx{xi0, -3.0 * u * xi1});
    // b_ij
    const double bd = 1.0 / (2.0 * (9.0 * u2 - w2) * (9.0 * u2 - w2));
    const double g1 = 3.0 * u2 - w2, g2 = 30.0 * u2 + 2.0 * w2;
    auto bj1 = [&](cplx ra, cplx rb, cplx f) {
      return cscal(bd, cadd(cadd(cscal(2.0 * u, ra), cscal(g1, rb)), cscal(-g2, f)));
    };
    auto bj2 = [&](cplx ra, cplx rb, cplx f) {
      return cscal(bd, cadd(cadd(ra, cscal(-3.0 * u, rb)), cscal(-24.0 * u, f)));
    };
    // tr(U S' B_j), B_j = b_j0 + b_j1 Q + b_j2 Q^2
    const M3 USQ = mul_nn(US, Q);
    const cplx s0 = m3_tr(US), s1 = m3_tr(USQ), s2 = m3_trm(US, Q2);
    const cplx t1 = cadd(cadd(cmul(bj1(r01, r02, f0), s0), cmul(bj1(r11, r12, f1), s1)),
                         cmul(bj1(r21, r22, f2), s2));
    const cplx t2 = cadd(cadd(cmul(bj2(r01, r02, f0), s0), cmul(bj2(r11, r12, f1), s1)),
                         cmul(bj2(r21, r22, f2), s2));
    const M3 QUS = mul_nn(Q, US);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        cplx g = cadd(cmul(t1, Q.a[i][j]), cmul(t2, Q2.a[i][j]));
        g = cadd(g, cmul(f1, US.a[i][j]));
        g = cadd(g, cmul(f2, cadd(QUS.a[i][j], USQ.a[i][j])));
        iGam.a[i][j] = {-g.i, g.r};   // i Gamma
      }
    eiQ = m3_poly(f0, f1, f2, Q, Q2);
  }
  const M3 iLam = at3(iGam);
  // U and S' are read again (from L2) rather than kept: holding them spills
  asm volatile("" : "+s"(ul));
  const M3 U = load3c(ul, x.s);
  const M3 Sp = rows_load<WIDE>(Sigmap + off, gw.first, L.V, gw.sh);
  store3c(reinterpret_cast<dbl2v_t*>(iTheta) + offc, gw.first + gw.lane, mul_nn(iLam, U));
  M3 Xi = mul_nn(Sp, eiQ);
  m3_add(Xi, mul_dn(C, iLam));
  rows_store<WIDE>(Sigma + off, gw.first, L.V, gw.sh, Xi);
}

// Sigma_mu(x) += rho sum_{nu != mu} of the six staple products (force_each,
// aforceSmear_APE-tmpl.h:280-360), V the links and T = iTheta, two of the three
// products of each side sharing a factor:
//   [T_nu(x+mu) V_mu(x+nu)^+ + V_nu(x+mu) T_mu(x+nu)^+] V_nu(x)^+
//     + V_nu(x+mu) V_mu(x+nu)^+ T_nu(x)^+
//   [V_nu(b)^+ T_mu(m)^+ + T_nu(b)^+ V_mu(m)^+] V_nu(m) + V_nu(b)^+ V_mu(m)^+ T_nu(m),
// m = x-nu, b = x-nu+mu.
template <bool WIDE>
__global__ void __launch_bounds__(128, 2)
k_stout_force_staple(double* __restrict__ Sigma, const double* __restrict__ Uc,
                     const double* __restrict__ iTheta, GaugeLat L, double rho) {
  __shared__ dbl2v_t slots[2 * kRowsLds];
  const GaugeWave g(slots);
  const int mu = g.mu;
  const GaugeSite x(L, g.first + g.lane);
  const size_t vol = chunked_mu(L);
  const dbl2v_t* u0 = reinterpret_cast<const dbl2v_t*>(Uc);
  const dbl2v_t* t0 = reinterpret_cast<const dbl2v_t*>(iTheta);
  const dbl2v_t *vm = u0 + vol * mu, *tm = t0 + vol * mu;
  const int pm = x.off(L, mu, 1);
  M3 acc = m3_zero();
  for (int i = 0; i < 3; ++i) {
    const int nu = i + (i >= mu ? 1 : 0);
    const dbl2v_t *vn = u0 + vol * nu, *tn = t0 + vol * nu;
    const int pn = x.off(L, nu, 1), m = x.s + x.off(L, nu, -1), b = m + pm;
    {
      const M3 Vn = load3c(vn, x.s + pm), Vm = load3c(vm, x.s + pn);
      m3_axpy(acc, rho, mul_nd(mul_nd(Vn, Vm), load3c(tn, x.s)));
      M3 t = mul_nd(load3c(tn, x.s + pm), Vm);
      m3_add(t, mul_nd(Vn, load3c(tm, x.s + pn)));
      m3_axpy(acc, rho, mul_nd(t, load3c(vn, x.s)));
    }
    const M3 Vb = load3c(vn, b), Vm = load3c(vm, m);
    m3_axpy(acc, rho, mul_nn(mul_dd(Vb, Vm), load3c(tn, m)));
    M3 t = mul_dd(Vb, load3c(tm, m));
    m3_add(t, mul_dd(load3c(tn, b), Vm));
    m3_axpy(acc, rho, mul_nn(t, load3c(vn, m)));
  }
  double* out = Sigma + (size_t)18 * L.V * mu;
  m3_add(acc, rows_load<WIDE>(out, g.first, L.V, g.sh));
  rows_store<WIDE>(out, g.first, L.V, g.sh, acc);
}

hipError_t launch_stout_force(double* Sigma, double* iTheta, const double* Sigmap,
                              const double* Uc, const int* dims, double rho, hipStream_t st) {
  const GaugeLat L = gauge_lat(dims);
  const dim3 grid(2 * L.chunks), block(128);
  if (m3_wide(Sigma, Sigmap)) {
    hipLaunchKernelGGL(k_stout_force_link<true>, grid, block, 0, st, Sigma, iTheta, Sigmap, Uc, L,
                       rho);
    hipLaunchKernelGGL(k_stout_force_staple<true>, grid, block, 0, st, Sigma, Uc,
                       (const double*)iTheta, L, rho);
  } else {
    hipLaunchKernelGGL(k_stout_force_link<false>, grid, block, 0, st, Sigma, iTheta, Sigmap, Uc, L,
                       rho);
    hipLaunchKernelGGL(k_stout_force_staple<false>, grid, block, 0, st, Sigma, Uc,
                       (const double*)iTheta, L, rho);
  }
  return hipGetLastError();
}

// F <- -2 at(U F) with a lexical gauge field U (the thin links of a smeared force)
__global__ void __launch_bounds__(128)
k_mult_generator_gauge(double* __restrict__ F, const double* __restrict__ U, size_t n) {
  const size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const M3 A = at3(mul_nn(load3(U + 18 * idx), load3(F + 18 * idx)));
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) r.a[i][j] = cscal(-2.0, A.a[i][j]);
  store3(F + 18 * idx, r);
}

hipError_t launch_mult_generator_gauge(double* F, const double* U, size_t nlinks,
                                       hipStream_t st) {
  hipLaunchKernelGGL(k_mult_generator_gauge, dim3((unsigned)((nlinks + 127) / 128)), dim3(128), 0,
                     st, F, U, nlinks);
  return hipGetLastError();
}

__device__ __forceinline__ double wave_sum_g(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

__global__ void __launch_bounds__(256)
k_plaquette(const double* __restrict__ U, int Nx, int Ny, int Nz, int Nt, double* partial,
            unsigned* counter, double* result) {
  const size_t V = (size_t)Nx * Ny * Nz * Nt;
  double acc = 0;
  for (size_t site = blockIdx.x * (size_t)blockDim.x + threadIdx.x; site < V;
       site += (size_t)gridDim.x * blockDim.x) {
    for (int mu = 0; mu < 4; ++mu)
      for (int nu = mu + 1; nu < 4; ++nu) {
        const size_t xpmu = shift_site(site, mu, +1, Nx, Ny, Nz, Nt);
        const size_t xpnu = shift_site(site, nu, +1, Nx, Ny, Nz, Nt);
        const M3 a = mul_nn(load3(U + 18 * (site + V * mu)), load3(U + 18 * (xpmu + V * nu)));
        const M3 b = mul_nn(load3(U + 18 * (site + V * nu)), load3(U + 18 * (xpnu + V * mu)));
        // Re tr(a b^+)
        for (int i = 0; i < 3; ++i)
          for (int k = 0; k < 3; ++k) acc += a.a[i][k].r * b.a[i][k].r + a.a[i][k].i * b.a[i][k].i;
      }
  }
  // block and grid reduction (same scheme as the field reductions)
  __shared__ double sh[4];
  __shared__ bool amlast;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double t = wave_sum_g(acc);
  if (lane == 0) sh[wid] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    __threadfence();
    unsigned prev = atomicAdd(counter, 1u);
    amlast = (prev == gridDim.x - 1);
  }
  __syncthreads();
  if (!amlast) return;
  __threadfence();
  double w = 0;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += blockDim.x)
    w += __hip_atomic_load(partial + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  t = wave_sum_g(w);
  if (lane == 0) sh[wid] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    *result = sh[0] + sh[1] + sh[2] + sh[3];
    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

hipError_t launch_plaquette(const double* U, int Nx, int Ny, int Nz, int Nt,
                            const RedScratch& red, int slot, hipStream_t st) {
  const size_t V = (size_t)Nx * Ny * Nz * Nt;
  size_t g = (V + 255) / 256;
  if (g > (size_t)kRedBlocks) g = kRedBlocks;
  hipLaunchKernelGGL(k_plaquette, dim3((unsigned)g), dim3(256), 0, st, U, Nx, Ny, Nz, Nt,
                     red.partial, red.counter, red.result + slot);
  return hipGetLastError();
}

}  // namespace dwf
