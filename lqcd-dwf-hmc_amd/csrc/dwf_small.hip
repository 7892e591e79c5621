// dwf_small.hip -- the fused operator launch (see dwf_kernels.hip) for lattices that
// do not fill the GPU.
//
// There k_dwf is a chain of memory latencies: the staging of the block's links, eight
// gathers one after the other, the Ls-mixing matrix by one thread per (site, s), in
// 8 blocks on a 4^3 x 8 lattice (17 us per hop, 0.4 MB of data).  Here a block is eight
// waves over the same 64 (site, s) points, one wave per direction:
//   1. every wave gathers its direction's spinor and link (all loads in flight at
//      once), projects, multiplies, and leaves a1 = U h1, a2 = U h2 in LDS;
//   2. six waves (one per colour and re / im) add the directions up and write the
//      chiral components of the core;
//   3. the twelve chiral rows are spread over the waves: out = E core + ..., out2 = F out.
// Same sums as k_dwf, the directions and the s in the same order; the 16-bit storage
// types keep the core and the matrices in FP32.  Epilogue features as in struct Epi.
#include "dwf_device.h"
#include "dwf_kernels.h"

namespace dwf {

constexpr int kSmallThreads = 512;

template <typename T> struct SmallArgs {
  using C = typename St<T>::C;
  T* out; const T* in; const T* links; const int* nbr;
  const C *E, *F, *G;
  const T* X; T* out2; const T* X2; T* upd;
  double* nrm;
  const double *xnum, *xden, *unum, *uden;
  const double* fin_partial; double* fin_result;
  size_t rstride;
  C scale, xcoef;
  int parity, Vh, Ls, nrs;
  unsigned fin_n;
};

// P[(12 DIR + k) * 64 + lane] = a1 (k < 6), a2 of one direction
template <int DIR, bool DAG, typename T, typename C>
__device__ __forceinline__ void small_gather(C* P, const T* in, const T* __restrict__ links,
                                             const int* __restrict__ nbr, int parity, int Vh,
                                             int Ls, int site, int s, int lane) {
  using S = St<T>;
  const int nb = nbr[((size_t)parity * 8 + DIR) * Vh + site];
  const T* wp = in + (size_t)nb * 24 * Ls + s;
  const T* L = links + ((size_t)parity * 8 + DIR) * 18 * Vh + site;
  C w[24], u[18];
#pragma unroll
  for (int k = 0; k < 24; ++k) w[k] = S::ld(wp + (DAG ? (k + 12) % 24 : k) * Ls);
#pragma unroll
  for (int e = 0; e < 18; ++e) u[e] = S::ld(L + (size_t)e * Vh);
  C h1[6], h2[6], a1[6], a2[6];
  project<DIR>(w, h1, h2);
  su3_mul(u, h1, a1);
  su3_mul(u, h2, a2);
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    P[(12 * DIR + k) * 64 + lane] = a1[k];
    P[(12 * DIR + 6 + k) * 64 + lane] = a2[k];
  }
}

template <typename T, int OP>
__global__ void __launch_bounds__(kSmallThreads, 4)
k_dwf_small(const SmallArgs<T> a) {
  using S = St<T>;
  using C = typename S::C;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  C* P = reinterpret_cast<C*>(smem_raw);           // 96 x 64, then the chiral rows:
  C* U = P;                                        // core, [chi][12][64]
  C* XU = P + 24 * 64;                             // X, the same
  C* mats = P + (OP == K_SITE ? 48 : 96) * 64;
  const int Ls = a.Ls, LL = Ls * Ls;
  C *sE = mats, *sF = sE + 2 * LL, *sG = sF + (a.out2 ? 2 * LL : 0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NS = 64 / Ls, ls = lane / Ls, s = lane - ls * Ls;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int v = blk * NS + ls;                     // virtual site (site * nr + rhs)
  const bool valid = ls < NS && v < (a.Vh << a.nrs);
  const int site = valid ? v >> a.nrs : 0;
  const size_t rhs = valid ? (size_t)(v & ((1 << a.nrs) - 1)) * a.rstride : 0;
  const size_t base = rhs + (size_t)site * 24 * Ls + s;
  if (a.fin_partial && blk == (int)gridDim.x - 1) {   // an earlier launch's deferred norm
    __shared__ double fsh[8];
    const double t = block_sum(a.fin_partial, a.fin_n, fsh);
    if (tid == 0) a.fin_result[0] = t;
  }
  const C xc = a.xnum ? (C)(a.xnum[0] / a.xden[0]) : a.xcoef;
  const C ua = a.upd ? (C)(a.unum[0] / a.uden[0]) : C(0);
  // loads that nothing below has to wait for: the matrices, transposed to
  // [chi][s][s_out] in LDS, and the rows of X of this thread's output rows
  // k = wave (and wave + 8 in the first four waves)
  constexpr int NM = 2;   // 2 Ls^2 values per matrix, Ls <= 22
  C ev[NM], fv[NM], gv[NM];
#pragma unroll
  for (int j = 0; j < NM; ++j) {
    const int i = tid + j * kSmallThreads;
    ev[j] = a.E && i < 2 * LL ? a.E[i] : C(0);
    fv[j] = a.F && i < 2 * LL ? a.F[i] : C(0);
    gv[j] = a.G && i < 2 * LL ? a.G[i] : C(0);
  }
  C x1[2] = {C(0), C(0)}, x2[2] = {C(0), C(0)};
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (a.X && valid && (r == 0 || wave < 4)) {
      x1[r] = S::ld(a.X + base + (wave + 8 * r) * Ls);
      x2[r] = S::ld(a.X + base + (wave + 8 * r + 12) * Ls);
    }
  C c1[2] = {C(0), C(0)}, c2[2] = {C(0), C(0)};
  if (OP == K_SITE) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (valid && (r == 0 || wave < 4)) {
        c1[r] = S::ld(a.in + base + (wave + 8 * r) * Ls);
        c2[r] = S::ld(a.in + base + (wave + 8 * r + 12) * Ls);
      }
  } else if (valid) {
    const T* in = a.in + rhs;
#define GATHER(d)                                                                               \
  case d:                                                                                       \
    small_gather<d, OP == K_HOPDAG, T>(P, in, a.links, a.nbr, a.parity, a.Vh, Ls, site, s, lane); \
    break;
    switch (wave) {
      GATHER(0) GATHER(1) GATHER(2) GATHER(3) GATHER(4) GATHER(5) GATHER(6) GATHER(7)
    }
#undef GATHER
  }
#pragma unroll
  for (int j = 0; j < NM; ++j) {
    const int i = tid + j * kSmallThreads;
    if (i < 2 * LL) {
      const int chi = i / LL, q = i - chi * LL, so = q / Ls, si = q - so * Ls;
      const int to = chi * LL + si * Ls + so;
      if (a.E) sE[to] = ev[j];
      if (a.out2) sF[to] = fv[j];
      if (a.G) sG[to] = gv[j];
    }
  }
  if (OP != K_SITE) {
    // core(k) for k = wave < 6: the four spins of colour k / 2, part k % 2
    __syncthreads();
    C o0 = 0, o1 = 0, o2 = 0, o3 = 0;
    if (wave < 6) {
      const C sg = (wave & 1) ? C(-1) : C(1);
      auto A1 = [&](int d) { return P[(12 * d + wave) * 64 + lane]; };
      auto A2 = [&](int d) { return P[(12 * d + 6 + wave) * 64 + lane]; };
      auto B1 = [&](int d) { return sg * P[(12 * d + (wave ^ 1)) * 64 + lane]; };
      auto B2 = [&](int d) { return sg * P[(12 * d + 6 + (wave ^ 1)) * 64 + lane]; };
      const C p0 = A1(0), p1 = A1(1), p2 = A1(2), p3 = A1(3), p4 = A1(4), p5 = A1(5);
      const C q0 = A2(0), q1 = A2(1), q2 = A2(2), q3 = A2(3), q4 = A2(4), q5 = A2(5);
      o0 = ((((p0 + p1) + p2) + p3) + p4) + p5 + A1(7);
      o1 = ((((q0 + q1) + q2) + q3) + q4) + q5 + A2(7);
      o2 = ((((B2(0) - B2(1)) - q2) + q3) + B1(4)) - B1(5) + A1(6);
      o3 = ((((B1(0) - B1(1)) + p2) - p3) - B2(4)) + B2(5) + A2(6);
      if (OP == K_HOPDAG) {   // gamma_5 exchanges the upper and lower pairs
        const C t0 = o0, t1 = o1;
        o0 = o2; o1 = o3;
        o2 = t0; o3 = t1;
      }
    }
    if (!a.E) {
      if (valid && wave < 6) {
        S::st(a.out + base + wave * Ls, a.scale * o0);
        S::st(a.out + base + (wave + 6) * Ls, a.scale * o1);
        S::st(a.out + base + (wave + 12) * Ls, a.scale * o2);
        S::st(a.out + base + (wave + 18) * Ls, a.scale * o3);
      }
      return;
    }
    __syncthreads();   // P is read; its place takes the chiral rows
    if (wave < 6) {
      U[wave * 64 + lane] = o0 + o2;
      U[(wave + 6) * 64 + lane] = o1 + o3;
      U[(wave + 12) * 64 + lane] = o0 - o2;
      U[(wave + 18) * 64 + lane] = o1 - o3;
    }
  } else {
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (r == 0 || wave < 4) {
        U[(wave + 8 * r) * 64 + lane] = c1[r] + c2[r];
        U[(wave + 8 * r + 12) * 64 + lane] = c1[r] - c2[r];
      }
  }
  if (a.G) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (r == 0 || wave < 4) {
        XU[(wave + 8 * r) * 64 + lane] = x1[r] + x2[r];
        XU[(wave + 8 * r + 12) * 64 + lane] = x1[r] - x2[r];
      }
  }
  __syncthreads();
  // (up, down) += M+ u(k), M- u(k + 12) for row s of this site
  const int col0 = ls * Ls;
  auto apply = [&](const C* M, const C* V, int k, C& up, C& dn) {
    const C *u = V + k * 64 + col0, *l = u + 12 * 64, *m = M + s;
    for (int t = 0; t < Ls; ++t) {
      up += m[t * Ls] * u[t];
      dn += m[LL + t * Ls] * l[t];
    }
  };
  C o1[2] = {C(0), C(0)}, o2[2] = {C(0), C(0)};
  double nacc = 0;
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (valid && (r == 0 || wave < 4)) {
      const int k = wave + 8 * r;
      C up = 0, dn = 0;
      apply(sE, U, k, up, dn);
      if (a.G) apply(sG, XU, k, up, dn);
      o1[r] = up + dn;
      o2[r] = up - dn;
      const size_t p1 = base + k * Ls, p2 = p1 + 12 * Ls;
      if (a.X && !a.G) {
        o1[r] += xc * x1[r];
        o2[r] += xc * x2[r];
        if (OP == K_SITE && a.upd) {
          S::st(a.upd + p1, S::ld(a.upd + p1) + ua * x1[r]);
          S::st(a.upd + p2, S::ld(a.upd + p2) + ua * x2[r]);
        }
      }
      C n1 = o1[r], n2 = o2[r];
      if (OP != K_SITE && a.upd) {
        T t1, t2;   // the norm is that of the stored (rounded) values
        S::st(&t1, S::ld(a.upd + p1) - ua * o1[r]);
        S::st(&t2, S::ld(a.upd + p2) - ua * o2[r]);
        a.upd[p1] = t1;
        a.upd[p2] = t2;
        n1 = S::ld(&t1);
        n2 = S::ld(&t2);
      } else if (a.out) {
        S::st(a.out + p1, o1[r]);
        S::st(a.out + p2, o2[r]);
      }
      nacc += (double)n1 * (double)n1 + (double)n2 * (double)n2;
    }
  if (a.nrm) {
    __shared__ double wsum[8];
    const double t = wave_sum(nacc);
    if (lane == 0) wsum[wave] = t;
    __syncthreads();
    if (tid == 0) {
      double n = 0;
      for (int w = 0; w < kSmallThreads / 64; ++w) n += wsum[w];
      a.nrm[blk] = n;
    }
  }
  if (!a.out2) return;
  __syncthreads();   // U is read
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (r == 0 || wave < 4) {
      U[(wave + 8 * r) * 64 + lane] = o1[r] + o2[r];
      U[(wave + 8 * r + 12) * 64 + lane] = o1[r] - o2[r];
    }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (valid && (r == 0 || wave < 4)) {
      const int k = wave + 8 * r;
      C up = 0, dn = 0;
      apply(sF, U, k, up, dn);
      const size_t p1 = base + k * Ls, p2 = p1 + 12 * Ls;
      C y1 = up + dn, y2 = up - dn;
      if (a.X2) {
        y1 += S::ld(a.X2 + p1);
        y2 += S::ld(a.X2 + p2);
      }
      S::st(a.out2 + p1, y1);
      S::st(a.out2 + p2, y2);
    }
}

static size_t small_lds(int prec, int op, int Ls, const Epi& e) {
  const size_t mats = 2 * (size_t)Ls * Ls *
                      ((e.E ? 1 : 0) + (e.out2 ? 1 : 0) + (e.G ? 1 : 0));
  return ((op == K_SITE ? 48 : 96) * 64 + mats) * (prec == P64 ? 8 : 4);
}

// The line between this kernel and k_dwf, in blocks of this one (64 / Ls sites): up to it
// this kernel was the faster or within a few per cent of it (but for single sizes: site FP16
// Ls = 9 2963 11.2 / 13.0, where it is ahead below and above).  Measured over volumes of 256
// to 663,000 sites for every Ls below, per launch (us, k_dwf against this kernel, blocks):
// * Ls = 12, 16, where k_dwf has the matrix cores: hop FP64 Ls = 16 512 14.4 / 10.8,
//   1024 15.1 / 19.4; BF16, whose k_dwf hop is not packed, 1024 14.5 / 9.9, 1800 14.8 / 16.9.
// * Ls = 8 (compiled, no matrix cores): hop FP64 900 19.5 / 17.9, 1728
//   26.9 / 28.6; FP16 8192 72 / 52; site FP16 900 5.7 / 5.2, 8192 16.6 / 26.1.
// * Ls up to 11 otherwise, where k_dwf has a runtime Ls (one element per access), ahead at
//   most sizes: hop FP32 Ls = 10 36864 356 / 332, site FP16 Ls = 6 33178 180 / 105; not
//   so FP64 hops that fill the GPU (Ls = 6 9831 155 / 171), nor FP16 sites at Ls = 10
//   (5462 14.2 / 21.1).
// * larger Ls: the transposed matrices take LDS, and from Ls = 17 on lanes idle: FP16 site
//   Ls = 14 1024 7.3 / 6.5, 3456 10.9 / 16.1; hop FP16 Ls = 22 2048 28 / 20, 6912 47 / 58.
// 16-bit storage at Ls = 12 and 16 keeps the hops' line for its sites, too: k_dwf rounds the
// operands of its matrix-core epilogue to the storage type, this kernel does not (FP16 D_ee^-1
// errors 4.0e-4 and 2.9e-4), and that is worth more than the microsecond or two it takes longer
// between (site BF16 Ls = 16 1024 5.0 / 6.7).
// A hop without E lacks the epilogue that this kernel spreads over its waves, and a site
// launch the gathers: both leave it earlier than a hop does.
static long small_max_blocks(int prec, int op, bool mat, int Ls) {
  constexpr long all = 1L << 40;
  const bool f64 = prec == P64, f32 = prec == P32, b16 = !f64 && !f32;
  if (op == K_SITE) {
    if (Ls == 4) return f64 ? 600 : f32 ? 1000 : all;
    if (Ls == 8) return f64 ? 600 : f32 ? 900 : 1200;
    if (Ls == 10) return b16 ? 2000 : all;
    if ((Ls == 12 || Ls == 16) && b16) return prec == PBF16 ? 1500 : 640;
    if (Ls == 12) return 400;
    if (Ls == 16) return f64 ? 250 : 400;
    return Ls <= 11 ? all : f64 ? 1500 : 1100;
  }
  if (Ls == 12 || Ls == 16) return prec == PBF16 ? 1500 : 640;
  if (Ls == 8) return b16 ? 8192 : mat ? 1300 : f64 ? 700 : 1000;
  if (Ls <= 5 || (Ls <= 7 && !f64)) return all;
  if (Ls <= 10) {
    if (f64) return !mat ? 1500 : Ls == 9 ? 2000 : 7000;
    if (f32) return !mat || Ls == 9 ? 20000 : all;
    return mat ? all : 40000;
  }
  if (b16) return Ls < 20 || (mat && Ls < 22) ? 8192 : 2400;
  return mat ? (f64 ? 1200 : 1500) : f64 ? 700 : 1000;
}
bool small_dwf_applies(int prec, int op, int Vh, int Ls, const Epi& e) {
  if (Ls > 22 || small_lds(prec, op, Ls, e) > 64 * 1024 - 256) return false;
  if (e.kernel) return e.kernel == EPI_SMALL;
  const int NS = 64 / Ls;
  const long blocks = (((long)Vh << e.nrs) + NS - 1) / NS;
  return blocks <= small_max_blocks(prec, op, e.E != nullptr, Ls);
}

template <typename T>
static hipError_t launch_small_t(int op, void* out, const void* in, const void* links,
                                 const int* nbr, int parity, int Vh, int Ls, const Epi& e,
                                 size_t lds, hipStream_t st, unsigned* nblocks) {
  using C = typename St<T>::C;
  SmallArgs<T> a;
  a.out = (T*)out; a.in = (const T*)in; a.links = (const T*)links; a.nbr = nbr;
  a.E = (const C*)e.E; a.F = e.out2 ? (const C*)e.F : nullptr; a.G = (const C*)e.G;
  a.X = (const T*)e.X; a.out2 = (T*)e.out2; a.X2 = (const T*)e.X2; a.upd = (T*)e.upd;
  a.nrm = e.nrm_partial;
  a.xnum = e.xnum; a.xden = e.xden; a.unum = e.unum; a.uden = e.uden;
  a.fin_partial = e.fin_partial; a.fin_result = e.fin_result; a.fin_n = e.fin_n;
  a.rstride = e.rstride;
  a.scale = (C)e.scale; a.xcoef = (C)e.xcoef;
  a.parity = parity; a.Vh = Vh; a.Ls = Ls; a.nrs = e.nrs;
  const int NS = 64 / Ls;
  const dim3 grid(((Vh << e.nrs) + NS - 1) / NS), block(kSmallThreads);
  *nblocks = grid.x;
  switch (op) {
    case K_SITE: hipLaunchKernelGGL((k_dwf_small<T, K_SITE>), grid, block, lds, st, a); break;
    case K_HOP: hipLaunchKernelGGL((k_dwf_small<T, K_HOP>), grid, block, lds, st, a); break;
    default: hipLaunchKernelGGL((k_dwf_small<T, K_HOPDAG>), grid, block, lds, st, a); break;
  }
  return hipGetLastError();
}

hipError_t launch_dwf_small(int prec, int op, void* out, const void* in, const void* links,
                            const int* nbr, int parity, int Vh, int Ls, const Epi& e,
                            hipStream_t st, unsigned* nblocks) {
  const size_t lds = small_lds(prec, op, Ls, e);
  switch (prec) {
    case P64: return launch_small_t<double>(op, out, in, links, nbr, parity, Vh, Ls, e, lds, st, nblocks);
    case P32: return launch_small_t<float>(op, out, in, links, nbr, parity, Vh, Ls, e, lds, st, nblocks);
    case P16: return launch_small_t<__half>(op, out, in, links, nbr, parity, Vh, Ls, e, lds, st, nblocks);
    case PBF16:
      return launch_small_t<__hip_bfloat16>(op, out, in, links, nbr, parity, Vh, Ls, e, lds, st, nblocks);
  }
  return hipErrorInvalidValue;
}

}  // namespace dwf
