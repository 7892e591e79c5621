// dwf_ptc.hip -- gauge-covariant parallel-transport convolution (PTC) network
// kernels: the learned preconditioner of the flexible CG.
//
// A layer maps C_in channels to C_out channels of 5D spinor fields on the full
// lattice (both parities):
//   out[a](x, s) = sum_{q < 11} sum_b W[q][a][b] T_q(in[b])(x, s)
// with W[q][a][b] a complex 4x4 matrix on spin (identity on colour) and the
// transports
//   q = 0          identity
//   q = 1 + dir    U(x, dir) in(x + dir), dir = 2 mu + fb the 8 hops of the
//                  operator (the packed links of the even-odd operator, boundary
//                  phases included: forward U_mu(x), backward U_mu(x - mu)^+)
//   q = 9, 10      in(x, s + 1), in(x, s - 1)   (zero beyond the walls)
// Every T_q commutes with gauge transformations of in and out, so the layer
// is gauge covariant.  The adjoint layer (the backward pass for the input
// gradient) is the same kernel with the reversed transport (dir -> dir ^ 1,
// 9 <-> 10) and W^+.  Weights are stored in bfloat16 and applied in FP32.
//
// Activation layout: channel-major, then parity, then the device spinor
// layout of the operator, element ((site * 24 + k) * Ls + s), k = ri + 2 (c + 3 d).
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "dwf_device.h"
#include "dwf_kernels.h"

namespace dwf {

constexpr int kPtcPaths = 11;
constexpr int kPtcLinkDir = 20, kPtcLinkSite = 8 * kPtcLinkDir;   // links of a site in LDS, floats

// (re, im) += (ar + i ai)(br + i bi), two fused multiply-adds per part
__device__ __forceinline__ void cmac(float& re, float& im, float ar, float ai, float br,
                                     float bi) {
  re = fmaf(-ai, bi, fmaf(ar, br, re));
  im = fmaf(ai, br, fmaf(ar, bi, im));
}

__device__ __forceinline__ int ptc_rev(int q) {
  if (q == 0) return 0;
  if (q <= 8) return 1 + ((q - 1) ^ 1);
  return q == 9 ? 10 : 9;
}

// t = T_q(in)(p, site, s) for one channel field `in` (both parities, Vh each);
// returns false if the path leaves the fifth dimension (t = 0)
__device__ __forceinline__ bool ptc_transport(float (&t)[24], const float* __restrict__ in,
                                              const float* __restrict__ links,
                                              const int* __restrict__ nbr, int q, int p,
                                              int site, int s, int Vh, int Ls) {
  const size_t fsz = (size_t)Vh * 24 * Ls;
  if (q == 0 || q >= 9) {
    const int ss = q == 0 ? s : (q == 9 ? s + 1 : s - 1);
    if (ss < 0 || ss >= Ls) return false;
    const float* src = in + (size_t)p * fsz + (size_t)site * 24 * Ls + ss;
#pragma unroll
    for (int k = 0; k < 24; ++k) t[k] = src[k * Ls];
    return true;
  }
  const int dir = q - 1;
  const int nb = nbr[((size_t)p * 8 + dir) * Vh + site];
  const float* src = in + (size_t)(1 - p) * fsz + (size_t)nb * 24 * Ls + s;
  float w[24];
#pragma unroll
  for (int k = 0; k < 24; ++k) w[k] = src[k * Ls];
  const float* L = links + ((size_t)p * 8 + dir) * 18 * Vh + site;
  float u[18];
#pragma unroll
  for (int e = 0; e < 18; ++e) u[e] = L[(size_t)e * Vh];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      float re = 0, im = 0;
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        cmac(re, im, u[2 * (b + 3 * a)], u[2 * (b + 3 * a) + 1], w[2 * (b + 3 * d)],
             w[2 * (b + 3 * d) + 1]);
      }
      t[2 * (a + 3 * d)] = re;
      t[2 * (a + 3 * d) + 1] = im;
    }
  return true;
}

// One layer (ADJ = false) or its adjoint (ADJ = true).  Thread per (parity,
// site, s), s fastest; block row blockIdx.y owns the AG output channels
// a0 .. a0 + AG - 1, so each transport T_q(in[b]) is formed once per thread and
// applied to AG output channels, and the weight addresses are uniform over the
// block (scalar loads).  W: bf16 [q][a][b][alpha][beta][ri] of the forward layer
// (C_out x C_in channels), read as one 32-bit word per complex entry (re low,
// im high); for ADJ the kernel's input channels are the forward outputs and
// out[b] = sum W^+ T_rev(q)(in[a]).  Each output channel's sum runs over q, then
// b, as in the per-channel form.
template <bool ADJ, int AG>
__global__ void __launch_bounds__(256)
k_ptc_layer(float* __restrict__ out, const float* __restrict__ in, int cin,
            const unsigned* __restrict__ W, int wcin, int wcout,
            const float* __restrict__ links, const int* __restrict__ nbr, int Vh, int Ls) {
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const size_t total = (size_t)2 * Vh * Ls;
  const int a0 = blockIdx.y * AG;
  for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total;
       idx += (size_t)gridDim.x * blockDim.x) {
    const int s = (int)(idx % Ls);
    const size_t r = idx / Ls;
    const int site = (int)(r % Vh);
    const int p = (int)(r / Vh);
    float acc[AG][24];
#pragma unroll
    for (int j = 0; j < AG; ++j)
#pragma unroll
      for (int k = 0; k < 24; ++k) acc[j][k] = 0;
    for (int q = 0; q < kPtcPaths; ++q) {
      const int qw = ADJ ? ptc_rev(q) : q;   // weight path
      for (int b = 0; b < cin; ++b) {
        float t[24];
        if (!ptc_transport(t, in + (size_t)b * 2 * fsz, links, nbr, q, p, site, s, Vh, Ls))
          continue;
#pragma unroll
        for (int j = 0; j < AG; ++j) {
          // forward: W[qw][a][b];  adjoint: (W[qw][b][a])^+
          const int a = a0 + j;
          const int wa = ADJ ? b : a, wb = ADJ ? a : b;
          const unsigned* w = W + (((size_t)qw * wcout + wa) * wcin + wb) * 16;
#pragma unroll
          for (int al = 0; al < 4; ++al)
#pragma unroll
            for (int be = 0; be < 4; ++be) {
              // element (al, be) of the applied spin matrix
              const unsigned e = w[ADJ ? (be * 4 + al) : (al * 4 + be)];
              const float wr = __uint_as_float(e << 16);
              const float wi = ADJ ? -__uint_as_float(e & 0xffff0000u)
                                   : __uint_as_float(e & 0xffff0000u);
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                cmac(acc[j][2 * (c + 3 * al)], acc[j][2 * (c + 3 * al) + 1], wr, wi,
                     t[2 * (c + 3 * be)], t[2 * (c + 3 * be) + 1]);
              }
            }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < AG; ++j) {
      float* o = out + (size_t)(a0 + j) * 2 * fsz + (size_t)p * fsz + (size_t)site * 24 * Ls + s;
#pragma unroll
      for (int k = 0; k < 24; ++k) o[k * Ls] = acc[j][k];
    }
  }
}

// Raw buffer resource over nbytes at base (gfx9 descriptor word 3): loads at
// byte offsets >= nbytes return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ptc_rsrc(const void* base, unsigned nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)nbytes, 0x00020000);
}
// the b32 load returns the 32 loaded bits as an integer: reinterpret, never convert
__device__ __forceinline__ unsigned ptc_ldu(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                            unsigned soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0);
  static_assert(sizeof(v) == 4, "32-bit buffer load");
  return __builtin_bit_cast(unsigned, v);
}
__device__ __forceinline__ float ptc_ld(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __uint_as_float(ptc_ldu(r, voff, soff));
}

typedef unsigned ptc_w2_t __attribute__((ext_vector_type(2)));
typedef short ptc_s4_t __attribute__((ext_vector_type(4)));

// The splits below are exact where every part is a bfloat16, denormals (multiples of 2^-133)
// included: for finite numbers from about 2^-109 up.  Smaller ones lose their last bits, and
// an infinity leaves inf - inf (with rounded parts a number beyond the largest bfloat16, too).
// So a tile whose sums hold a NaN, or in a lane nothing but numbers so small that they can
// stem from such transports, is formed again in FP32; what is lost in the others is below
// 2^-133 beside sums of at least 2^-88.
constexpr float kPtcTiny = 0x1p-88f;
__device__ __forceinline__ float ptc_absmax(float m, float x, float y) {   // NaN stays
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, fabsf(x)), fabsf(y));
}
__device__ __forceinline__ bool ptc_in_range(float m) { return m == 0.f || m >= kPtcTiny; }

// t = hi + mid + lo, each part with at most 8 significant bits, i.e. a bfloat16 (the first
// sixteen bits of its float): truncate, subtract, truncate.  The parts of (re, im) are
// returned as one word each, re low; the subtraction takes its part from the word
// (v_dot2_f32_bf16 with (-1, 0) and (0, -1), exact here).
__device__ __forceinline__ void ptc_split(float re, float im, unsigned& hi, unsigned& mid,
                                          unsigned& lo) {
  typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
  constexpr unsigned kHigh = 0x07060302u;   // the upper halves of both
  // kept in registers: as an inline constant the instruction reads -1.0 differently
  unsigned kre = 0x0000bf80u, kim = 0xbf800000u;
  asm("" : "+s"(kre), "+s"(kim));
  const b2_t mre = __builtin_bit_cast(b2_t, kre), mim = __builtin_bit_cast(b2_t, kim);
  auto top = [&](float x, float y) {
    return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), kHigh);
  };
  auto minus = [&](float x, unsigned w, b2_t m) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2_t, w), m, x, false);
  };
  hi = top(re, im);
  const float re1 = minus(re, hi, mre), im1 = minus(im, hi, mim);
  mid = top(re1, im1);
  lo = top(minus(re1, mid, mre), minus(im1, mid, mim));
}

// The same split with rounded parts (their signs are then as good as random, so that a
// dropped product of parts leaves no bias).
__device__ __forceinline__ void ptc_split_round(float x, float y, unsigned& hi, unsigned& mid,
                                                unsigned& lo) {
  typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
  typedef float f2_t __attribute__((ext_vector_type(2)));
  unsigned kx = 0x0000bf80u, ky = 0xbf800000u;
  asm("" : "+s"(kx), "+s"(ky));
  auto pack = [](float p, float q) { return __builtin_convertvector(f2_t{p, q}, b2_t); };
  auto minus = [](float p, b2_t w, unsigned m) {
    return __builtin_amdgcn_fdot2_f32_bf16(w, __builtin_bit_cast(b2_t, m), p, false);
  };
  const b2_t h = pack(x, y);
  const float x1 = minus(x, h, kx), y1 = minus(y, h, ky);
  const b2_t m = pack(x1, y1);
  const b2_t l = pack(minus(x1, m, kx), minus(y1, m, ky));
  hi = __builtin_bit_cast(unsigned, h);
  mid = __builtin_bit_cast(unsigned, m);
  lo = __builtin_bit_cast(unsigned, l);
}

// a tile's sums to the output: register r of lane (n, g) is row 4 g + r = channel
// 2 mt + (g >> 1), spin 2 (g & 1) + (r >> 1), re / im r & 1, of point n
template <int NMT>
__device__ __forceinline__ void ptc_tile_store(float* out, const flt4_t (&acc)[NMT][3], int cout,
                                               size_t fsz, int p, int site, int s, int g, int Ls) {
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt) {
    if (2 * mt + (g >> 1) >= cout) continue;
    float* o = out + (size_t)(2 * mt + (g >> 1)) * 2 * fsz + (size_t)p * fsz +
               (size_t)site * 24 * Ls + s;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int alo = 2 * (g & 1) + (r >> 1);
        o[(size_t)((r & 1) + 2 * (c + 3 * alo)) * Ls] = acc[mt][c][r];
      }
  }
}

// One tile of k_ptc_layer_mfma again on the FP32 matrix cores, for transports outside the range
// of the split: D(16x16) += A(16x4) B(4x16), K the 4 spins, t_re and t_im in turn.  A function
// of its own: inlined, its registers cost the layers where it never runs (8.9 ms an application
// at 16^3 x 32, Ls = 16, against 8.65; 8.55 without the check).
template <bool ADJ, int NMT>
__device__ __attribute__((noinline)) void ptc_tile_f32(
    float* out, const float* in, int cin, int cout, const unsigned* W, int wcin, int wcout,
    const float* su, const int* nbr, int Vh, int Ls, int tile) {
  constexpr unsigned kOut = 0x80000000u;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int am = n >> 3, al = (n >> 1) & 3, ro = n & 1;   // as in k_ptc_layer_mfma
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const int npts = Vh * Ls, tpp = (npts + 15) / 16, p = tile / tpp;
  const int P0 = (tile - p * tpp) * 16;
  const bool valid = P0 + n < npts;
  const int P = valid ? P0 + n : npts - 1, site = P / Ls, s = P - site * Ls;
  const float* ul = su + (site - P0 / Ls) * kPtcLinkSite;
  const __amdgpu_buffer_rsrc_t rw = ptc_rsrc(W, 4u * (unsigned)(kPtcPaths * wcin * wcout * 16));
  flt4_t acc[NMT][3];
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[mt][c] = flt4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int q = 0; q < kPtcPaths; ++q) {
    const int qw = ADJ ? ptc_rev(q) : q;
    const bool hop = q >= 1 && q <= 8;
    const int ss = s + (q == 9) - (q == 10);
    const int x = hop ? nbr[((size_t)p * 8 + q - 1) * Vh + site] : site;
    const unsigned off =
        valid && ss >= 0 && ss < Ls
            ? 4u * (unsigned)((hop ? 1 - p : p) * fsz + ((size_t)x * 24 + 6 * g) * Ls + ss)
            : kOut;
#pragma unroll 1
    for (int b = 0; b < cin; ++b) {
      const __amdgpu_buffer_rsrc_t r = ptc_rsrc(in + (size_t)b * 2 * fsz, 8u * (unsigned)fsz);
      float w[6], t[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) w[k] = t[k] = ptc_ld(r, off, 4u * (unsigned)(k * Ls));
      if (hop) {
        const float* u = ul + (q - 1) * kPtcLinkDir;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          float re = 0.f, im = 0.f;
#pragma unroll
          for (int cb = 0; cb < 3; ++cb)
            cmac(re, im, u[2 * (cb + 3 * c)], u[2 * (cb + 3 * c) + 1], w[2 * cb], w[2 * cb + 1]);
          t[2 * c] = re;
          t[2 * c + 1] = im;
        }
      }
#pragma unroll
      for (int mt = 0; mt < NMT; ++mt) {
        const unsigned wblk = ADJ ? (unsigned)(((qw * wcout + b) * wcin + 2 * mt) * 16)
                                  : (unsigned)(((qw * wcout + 2 * mt) * wcin + b) * 16);
        const unsigned wl = ADJ ? (unsigned)(am * 16 + g * 4 + al)
                                : (unsigned)(am * wcin * 16 + al * 4 + g);
        const unsigned e = ptc_ldu(rw, 2 * mt + am < cout ? 4u * wl : kOut, 4u * wblk);
        const float wr = __uint_as_float(e << 16);
        const float wi = ADJ ? -__uint_as_float(e & 0xffff0000u) : __uint_as_float(e & 0xffff0000u);
        const float ar = ro ? wi : wr, ai = ro ? wr : -wi;   // multiply t_re, t_im
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          acc[mt][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar, t[2 * c], acc[mt][c], 0, 0, 0);
          acc[mt][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai, t[2 * c + 1], acc[mt][c], 0, 0, 0);
        }
      }
    }
  }
  if (valid) ptc_tile_store<NMT>(out, acc, cout, fsz, p, site, s, g, Ls);
}

// Matrix-core form of the same layer (any number of output channels up to 16;
// an odd count leaves the second channel of the last tile with zero weights and
// does not store it).  Per path q and input channel b the contraction is the
// real product
//   [out_re; out_im](a, alpha) += [Wr -Wi; Wi Wr](a, alpha; beta) [t_re; t_im](beta)
// for every colour.  The weights are bfloat16, and the FP32 transports are the exact sum
// of three bfloat16 parts (ptc_split), so the products run on the BF16 matrix cores without loss
// (v_mfma_f32_16x16x16_bf16, FP32 accumulation): 3 x 16 cycles per tile, colour and two
// input channels where the FP32 cores take 4 x 32.  Tiles D(16x16) += A(16x16) B(16x16) with
//   D rows  m = 8 a' + 2 alpha + re/im  (NMT tiles of two output channels),
//   K       (spin beta, input channel b or b + 1, re/im), one product per part,
//   columns 16 points (site, s) of one parity, consecutive in site * Ls + s.
// Lane l holds A[l % 16][4 (l / 16) + i] and B[4 (l / 16) + i][l % 16], so lane l computes
// the transport of spin beta = l / 16 at point l % 16 itself (3 colours, 36
// multiply-adds for a hop path) and holds the weights of row l % 16, column
// beta, which are the weight's own word for t: (Wr, -Wi) in a re row, (Wi, Wr) in an im
// row; register r of its result holds D[4 (l / 16) + r][l % 16].  One wave
// per 16 points, all output channels; each output element is a sum over
// (q, b pairs, parts) of 8-term matrix-core products in FP32.
// 1 -> 8 -> 8 -> 8 -> 1 channels at 16^3 x 32, Ls = 16: 13.5 -> 8.7 ms (error against
// 64 bits 9.5e-7 -> 6e-7).  Bound by the gathers: every channel is read nine times through
// L1 (14.5 GB per 8 -> 8 layer, 9.9 GB of it past the L2s); the vector unit has 1.4 ms
// of work per such layer (36 operations of transport and 21 of splitting per hop path
// and channel), the matrix cores 1.35 ms.  Two s per lane with eight-byte loads (9.9 ms),
// all channels per path (9.9) and no per-XCD order (9.6, before the shifts by lane, against
// 9.6) were no faster.
// The paths are the inner loop and the channel pairs the outer one: the points in flight
// on an XCD then gather from two channels at a time, which its L2 holds between the nine
// uses better than all of them.  The links of the wave's sites sit in LDS (they are read
// once per pair), and so do the layer's weights where they fit (LW).  S16: Ls = 16, where
// a tile is one site and the shifts in s are row shifts (DPP) of the split words.  NB: the
// channels of a pair that are loaded, 1 for cin = 1 (half the transports of the pair: 84 -> 76
// us for the same network).
__host__ __device__ constexpr int ptc_wave_sites(int Ls) { return 15 / Ls + 2; }
template <bool ADJ, int NMT, bool LW, bool S16, int NB>
__global__ void __launch_bounds__(256, NMT <= 2 ? 4 : NMT <= 5 ? 3 : 2)
k_ptc_layer_mfma(float* __restrict__ out, const float* __restrict__ in, int cin, int cout,
                 const unsigned* __restrict__ W, int wcin, int wcout,
                 const float* __restrict__ links, const int* __restrict__ nbr, int Vh, int Ls) {
  // loads go through buffer resources with 32-bit byte offsets: per lane the
  // point / spin part, per wave (SGPR) the channel and element part; a lane
  // whose source is outside the lattice or the fifth dimension reads at
  // kOut and gets 0.  The launcher checks that every offset fits.
  constexpr unsigned kOut = 0x80000000u;
  extern __shared__ __align__(16) unsigned ptc_sw[];
  const int lane = threadIdx.x & 63;
  const int n = lane & 15, g = lane >> 4;
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const int npts = Vh * Ls;            // points of one parity
  const int tpp = (npts + 15) / 16;    // tiles of one parity
  const unsigned lsb = 4u * (unsigned)Ls;
  const int nwords = kPtcPaths * wcin * wcout * 16;
  const __amdgpu_buffer_rsrc_t rw = ptc_rsrc(W, 4u * (unsigned)nwords);
  const int wsites = ptc_wave_sites(Ls);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* su = reinterpret_cast<float*>(ptc_sw) + (size_t)wave * wsites * kPtcLinkSite;
  unsigned* sw = ptc_sw + (size_t)4 * wsites * kPtcLinkSite;
  // the A row of this lane: channel 2 mt + am, spin row al, re (0) / im (1);
  // its weight word within the (q, b, mt) block
  const int am = n >> 3, al = (n >> 1) & 3, ro = n & 1;
  // its word (Wr, Wi) as the coefficients of (t_re, t_im): halves exchanged in an im row,
  // one sign (conjugated for the adjoint)
  const unsigned wsel = ro ? 0x01000302u : 0x03020100u;
  const unsigned wmask = ADJ ? (ro ? 0x8000u : 0u) : (ro ? 0u : 0x80000000u);
  const unsigned wlane =
      ADJ ? (unsigned)(am * 16 + g * 4 + al) : (unsigned)(am * wcin * 16 + al * 4 + g);
  // every XCD walks a contiguous range of sites: the neighbours of a tile share its L2
  const int tile0 = xcd_block(blockIdx.x, gridDim.x) * 4 + wave;
  const int tile = min(tile0, 2 * tpp - 1);
  const int p = tile / tpp;
  const int P0 = (tile - p * tpp) * 16, P = P0 + n;
  const bool valid = P < npts;
  const int Pc = valid ? P : npts - 1;
  const int site = Pc / Ls, s = Pc - (Pc / Ls) * Ls;
  // What every wave needs first, each in loads that are in flight together (one after the
  // other they took most of a small lattice's time: 1 -> 3 -> 1 channels at 8^3 x 16, Ls = 12,
  // 90 -> 84 us): the neighbours, the weights, the links of sites site0 .. site0 +
  // wsites - 1 (those below Vh) as [site][dir][20].
  int nb[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) nb[d] = nbr[((size_t)p * 8 + d) * Vh + site];
  if (LW) {
    for (int i0 = threadIdx.x; i0 < nwords / 4; i0 += 4 * 256) {
      u32x4_t v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = reinterpret_cast<const u32x4_t*>(W)[min(i0 + 256 * k, nwords / 4 - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        reinterpret_cast<u32x4_t*>(sw)[min(i0 + 256 * k, nwords / 4 - 1)] = v[k];
    }
  }
  const int site0 = P0 / Ls;
  for (int i0 = lane; i0 < 144 * wsites; i0 += 5 * 64) {
    float v[5];
    int to[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const int i = min(i0 + 64 * k, 144 * wsites - 1);
      const int r = i / wsites, j = i - r * wsites, d = r / 18;   // row = dir * 18 + e
      const int x = site0 + j < Vh ? site0 + j : Vh - 1;
      v[k] = links[((size_t)p * 144 + r) * Vh + x];
      to[k] = j * kPtcLinkSite + d * kPtcLinkDir + (r - 18 * d);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) su[to[k]] = v[k];
  }
  if (LW) __syncthreads();
  if (tile0 >= 2 * tpp) return;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const float* ul = su + (site - site0) * kPtcLinkSite;
  // byte offsets of spin g of the source points in a channel
  const unsigned own = 4u * (unsigned)(p * fsz + ((size_t)site * 24 + 6 * g) * Ls + s);
  unsigned off[kPtcPaths];
  off[0] = valid ? own : kOut;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    off[1 + d] = 4u * (unsigned)((1 - p) * fsz + ((size_t)nb[d] * 24 + 6 * g) * Ls + s);
    if (!valid) off[1 + d] = kOut;
  }
  off[9] = valid && s + 1 < Ls ? own + 4u : kOut;
  off[10] = valid && s > 0 ? own - 4u : kOut;
  flt4_t acc[NMT][3];
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[mt][c] = flt4_t{0.f, 0.f, 0.f, 0.f};
  for (int b = 0; b < cin; b += 2) {
    // the spinors of input channels b and b + 1 at the source points of path q, loaded one
    // path ahead of the matrix-core products; a channel beyond cin reads zeros
    const bool two = b + 1 < cin;
    const __amdgpu_buffer_rsrc_t r0 = ptc_rsrc(in + (size_t)b * 2 * fsz, 8u * (unsigned)fsz);
    const __amdgpu_buffer_rsrc_t r1 =
        ptc_rsrc(in + (size_t)(two ? b + 1 : b) * 2 * fsz, two ? 8u * (unsigned)fsz : 0u);
    auto load = [&](int q, float (&w)[NB][6]) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int k = 0; k < 6; ++k) w[j][k] = ptc_ld(j ? r1 : r0, off[q], (unsigned)k * lsb);
    };
    // element (al, beta = g) of the applied spin matrix of channel a = 2 mt + am:
    // forward W[qw][a][b], adjoint (W[qw][b][a])^+, as the coefficients of (re, im);
    // an odd cout pads the last tile, an odd cin the last pair with zeros
    auto weights = [&](int q, ptc_w2_t (&A)[NMT]) {
      const int qw = ADJ ? ptc_rev(q) : q;   // weight path
#pragma unroll
      for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (j >= NB) {
            A[mt][j] = 0u;
            continue;
          }
          const unsigned wblk = ADJ ? (unsigned)(((qw * wcout + b + j) * wcin + 2 * mt) * 16)
                                    : (unsigned)(((qw * wcout + 2 * mt) * wcin + b + j) * 16);
          const bool on = (j == 0 || two) && 2 * mt + am < cout;
          unsigned e;
          if constexpr (LW) {
            e = sw[on ? wblk + wlane : 0u];
            e = on ? e : 0u;
          } else {
            e = ptc_ldu(rw, on ? 4u * wlane : kOut, 4u * wblk);
          }
          A[mt][j] = __builtin_amdgcn_perm(e, e, wsel) ^ wmask;
        }
    };
    // the products of colour c, the parts in order of size
    auto products = [&](const ptc_w2_t (&A)[NMT], const ptc_w2_t (&B)[3], int c) {
#pragma unroll
      for (int part = 0; part < 3; ++part)
#pragma unroll
        for (int mt = 0; mt < NMT; ++mt)
          acc[mt][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
              __builtin_bit_cast(ptc_s4_t, A[mt]), __builtin_bit_cast(ptc_s4_t, B[part]),
              acc[mt][c], 0, 0, 0);
    };
    auto split = [&](float re, float im, ptc_w2_t (&B)[3], int j) {
      unsigned hi, mid, lo;
      ptc_split(re, im, hi, mid, lo);
      B[0][j] = lo;
      B[1][j] = mid;
      B[2][j] = hi;
    };
    // paths without a link
    auto plain = [&](int q, const float (&w)[NB][6]) {
      ptc_w2_t A[NMT];
      weights(q, A);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        ptc_w2_t B[3] = {};
#pragma unroll
        for (int j = 0; j < NB; ++j) split(w[j][2 * c], w[j][2 * c + 1], B, j);
        products(A, B, c);
        if constexpr (S16) {   // s + 1 and s - 1: the neighbouring lanes, 0 beyond the walls
          ptc_w2_t U[3] = {}, D[3] = {}, Au[NMT], Ad[NMT];
          weights(9, Au);
          weights(10, Ad);
#pragma unroll
          for (int part = 0; part < 3; ++part)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
              U[part][j] = __builtin_amdgcn_update_dpp(0, (int)B[part][j], 0x101, 0xf, 0xf, true);
              D[part][j] = __builtin_amdgcn_update_dpp(0, (int)B[part][j], 0x111, 0xf, 0xf, true);
            }
          products(Au, U, c);
          products(Ad, D, c);
        }
      }
    };
    // a hop: colour by colour the transported component of spin g at this point, both
    // channels, split, then its products
    auto hop = [&](int q, const float (&w)[NB][6]) {
      ptc_w2_t A[NMT];
      weights(q, A);
      float u[18];
#pragma unroll
      for (int e = 0; e < 18; ++e) u[e] = ul[(q - 1) * kPtcLinkDir + e];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        ptc_w2_t B[3] = {};
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          float re = 0.f, im = 0.f;
#pragma unroll
          for (int cb = 0; cb < 3; ++cb)
            cmac(re, im, u[2 * (cb + 3 * c)], u[2 * (cb + 3 * c) + 1], w[j][2 * cb],
                 w[j][2 * cb + 1]);
          split(re, im, B, j);
        }
        products(A, B, c);
      }
    };
    float wa[NB][6], wb[NB][6];
    load(0, wa);
    if constexpr (S16) {
      load(1, wb); plain(0, wa);
      load(2, wa);
    } else {
      load(9, wb);  plain(0, wa);
      load(10, wa); plain(9, wb);
      load(1, wb);  plain(10, wa);
      load(2, wa);
    }
    hop(1, wb); load(3, wb);
    hop(2, wa); load(4, wa);
    hop(3, wb); load(5, wb);
    hop(4, wa); load(6, wa);
    hop(5, wb); load(7, wb);
    hop(6, wa); load(8, wa);
    hop(7, wb);
    hop(8, wa);
  }
  float m = 0.f;
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      m = ptc_absmax(m, acc[mt][c][0], acc[mt][c][1]);
      m = ptc_absmax(m, acc[mt][c][2], acc[mt][c][3]);
    }
  if (__builtin_expect(__ballot(!ptc_in_range(m)) != 0, 0)) {
    ptc_tile_f32<ADJ, NMT>(out, in, cin, cout, W, wcin, wcout, su, nbr, Vh, Ls, tile);
    return;
  }
  if (valid) ptc_tile_store<NMT>(out, acc, cout, fsz, p, site, s, g, Ls);
}

// Weight gradient of one layer: block (x, y = q * cin + b, z) adds, over its
// share of the lattice, G[q][a][b][al][be] = sum_{x, s, c}
// g[a](al, c) conj(T_q(in[b])(be, c)) for the AG output channels
// a = z AG .. z AG + AG - 1 (the transport formed once for all of them);
// block partials [y][a][block][32].
template <int AG>
__global__ void __launch_bounds__(256)
k_ptc_wgrad(double* __restrict__ partial, const float* __restrict__ g,
            const float* __restrict__ in, int cin, int cout, const float* __restrict__ links,
            const int* __restrict__ nbr, int Vh, int Ls) {
  const int q = blockIdx.y / cin, b = blockIdx.y - (blockIdx.y / cin) * cin;
  const int a0 = blockIdx.z * AG;
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const size_t total = (size_t)2 * Vh * Ls;
  float acc[AG][32];
#pragma unroll
  for (int j = 0; j < AG; ++j)
#pragma unroll
    for (int k = 0; k < 32; ++k) acc[j][k] = 0;
  for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total;
       idx += (size_t)gridDim.x * blockDim.x) {
    const int s = (int)(idx % Ls);
    const size_t r = idx / Ls;
    const int site = (int)(r % Vh);
    const int p = (int)(r / Vh);
    float t[24];
    if (!ptc_transport(t, in + (size_t)b * 2 * fsz, links, nbr, q, p, site, s, Vh, Ls)) continue;
#pragma unroll
    for (int j = 0; j < AG; ++j) {
      const float* gp =
          g + (size_t)(a0 + j) * 2 * fsz + (size_t)p * fsz + (size_t)site * 24 * Ls + s;
      float gv[24];
#pragma unroll
      for (int k = 0; k < 24; ++k) gv[k] = gp[k * Ls];
#pragma unroll
      for (int al = 0; al < 4; ++al)
#pragma unroll
        for (int be = 0; be < 4; ++be)
#pragma unroll
          for (int c = 0; c < 3; ++c)
            // g conj(t)
            cmac(acc[j][2 * (al * 4 + be)], acc[j][2 * (al * 4 + be) + 1], gv[2 * (c + 3 * al)],
                 gv[2 * (c + 3 * al) + 1], t[2 * (c + 3 * be)], -t[2 * (c + 3 * be) + 1]);
    }
  }
  __shared__ double sh[4][AG * 32];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < AG; ++j)
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      double v = acc[j][k];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
      if (lane == 0) sh[wv][j * 32 + k] = v;
    }
  __syncthreads();
  if (threadIdx.x < AG * 32) {
    const int j = threadIdx.x >> 5, k = threadIdx.x & 31;
    const double v = sh[0][threadIdx.x] + sh[1][threadIdx.x] + sh[2][threadIdx.x] +
                     sh[3][threadIdx.x];
    partial[(((size_t)blockIdx.y * cout + a0 + j) * gridDim.x + blockIdx.x) * 32 + k] = v;
  }
}

// One block's part of the weight gradient of output channel a and input channel b again, in
// FP32, for k_ptc_wgrad_mfma: the points of its groups first .. last - 1; sh 128 doubles.
__device__ __forceinline__ void ptc_wgrad_f32(double* dst, const float* __restrict__ g,
                              const float* __restrict__ in, int a, int b,
                              const float* __restrict__ links, const int* __restrict__ nbr, int q,
                              int first, int last, int Vh, int Ls, double* sh) {
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const int npts = Vh * Ls, gpp = (npts + 15) / 16;
  float acc[32];
#pragma unroll
  for (int k = 0; k < 32; ++k) acc[k] = 0;
  for (int i = 16 * first + (int)threadIdx.x; i < 16 * last; i += 256) {
    const int p = i >= 16 * gpp ? 1 : 0, P = i - p * 16 * gpp;
    if (P >= npts) continue;
    const int site = P / Ls, s = P - site * Ls;
    float t[24];
    if (!ptc_transport(t, in + (size_t)b * 2 * fsz, links, nbr, q, p, site, s, Vh, Ls)) continue;
    const float* gp = g + ((size_t)a * 2 + p) * fsz + (size_t)site * 24 * Ls + s;
#pragma unroll
    for (int al = 0; al < 4; ++al)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float gr = gp[(6 * al + 2 * c) * Ls], gi = gp[(6 * al + 2 * c + 1) * Ls];
#pragma unroll
        for (int be = 0; be < 4; ++be)   // g conj(t)
          cmac(acc[2 * (al * 4 + be)], acc[2 * (al * 4 + be) + 1], gr, gi, t[2 * (c + 3 * be)],
               -t[2 * (c + 3 * be) + 1]);
      }
  }
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    double v = acc[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[(threadIdx.x >> 6) * 32 + k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 32)
    dst[threadIdx.x] = sh[threadIdx.x] + sh[32 + threadIdx.x] + sh[64 + threadIdx.x] +
                       sh[96 + threadIdx.x];
  __syncthreads();
}

// The same for Ls a multiple of 4 on the matrix cores: per path one real product
//   P(64 x 64) = sum over points, colours of  g(a, alpha, re/im) t(b, beta, re/im)
// with both operands split into three bfloat16 parts (rounded, so that what is left out has
// no bias).  Six of the nine part products are taken, two at a time, as one
// v_mfma_f32_16x16x32_bf16 per pair (K = 16 points x 2 parts): (hi lo)(lo hi),
// (mid hi)(hi mid), (mid hi)(mid hi); the others are 2^-25 of a product and below, and with
// (mid lo)(lo mid) the error against 64 bits is the same.  A block of four waves takes 16
// points at a time (a lane four consecutive s of one component: 16-byte loads): wave w
// loads, transports and splits the operands of row tile w and column tile w (a tile: two
// channels) into LDS, then multiplies a quadrant of the 4 x 4 tiles; the sums over 16
// points are added up in FP64.  The matrix cores round towards minus infinity, an error of
// one sign that the sum over the lattice adds up (8 -> 8, 4096 sites a parity, Ls = 16, random signs:
// 4.7e-7 of the sum, the other kernel 1.3e-7): every other group is multiplied with its rows
// negated, which leaves 8.4e-8 and costs no time.  Grid: blocks of points, paths, groups of 4 x 4 tiles.
// Bound by the serial chain of a group (gather, transport, split, LDS, products, two
// barriers: 3.4 us with three blocks per CU), neither by issue (fewer moves or address
// instructions change nothing) nor by memory (nor does an order in which the paths share
// an L2).  8 -> 8 channels at 8^3 x 16, Ls = 16: 1290 -> 507 us.
__global__ void __launch_bounds__(256, 3)
k_ptc_wgrad_mfma(double* __restrict__ partial, const float* __restrict__ gr,
                 const float* __restrict__ in, int cin, int cout,
                 const float* __restrict__ links, const int* __restrict__ nbr, int Vh, int Ls) {
  typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
  // [tile][colour][part hi, mid, lo][lane]: any two parts are one conflict-free ds_read2_b64
  __shared__ u32x2_t shA[4 * 3 * 3 * 64], shB[4 * 3 * 3 * 64];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = blockIdx.y;
  const int RT = (cout + 1) / 2, CT = (cin + 1) / 2, RB = (RT + 3) / 4;
  const int rt0 = (blockIdx.z % RB) * 4, ct0 = (blockIdx.z / RB) * 4;
  const bool hop = q >= 1 && q <= 8;
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const int npts = Vh * Ls, gpp = (npts + 15) / 16;
  // this block's 16-point groups
  const int per = (2 * gpp + gridDim.x - 1) / gridDim.x;
  const int first = blockIdx.x * per, last = min(first + per, 2 * gpp);
  // row / column of this lane: channel, spin, part
  const int ch = n >> 3, sp = (n >> 1) & 3, ri = n & 1;
  const int a = 2 * (rt0 + wave) + ch, b = 2 * (ct0 + wave) + ch;
  const bool rowt = rt0 + wave < RT, colt = ct0 + wave < CT;   // (wave-uniform)
  const float sgn = ri ? 1.f : -1.f;   // re: u_r t_r - u_i t_i; im: u_r t_i + u_i t_r
  flt4_t va[3], vb[3];
  float edge[3], u[18];
  const flt4_t zero = {0.f, 0.f, 0.f, 0.f};
  const bool tail = (npts & 15) != 0;
  // site and s of this lane's four points of a group; the lanes beyond the last point take
  // the last ones, and their row operand is set to zero below.  (The division is that of
  // the group's first point, in scalar registers.)
  auto locate = [&](int grp, int& p, int& site, int& s) -> bool {
    p = grp >= gpp ? 1 : 0;
    const int P0 = (grp - p * gpp) * 16, base = P0 / Ls;
    int r = P0 - base * Ls + 4 * g;
    const bool ok = P0 + 4 * g < npts;
    const int k = (r >= Ls) + (r >= 2 * Ls) + (r >= 3 * Ls);
    site = ok ? base + k : Vh - 1;
    s = ok ? r - k * Ls : Ls - 4;
    return ok;
  };
  // rows and columns beyond the channels repeat the last one (their results are dropped)
  const int ac = min(a, cout - 1), bc = min(b, cin - 1);
  // the neighbour of group grp's site, fetched a group before the spinors it addresses
  auto neighbour = [&](int grp) -> int {
    int p, site, s;
    locate(grp, p, site, s);
    return (nbr + ((size_t)p * 8 + q - 1) * Vh)[(unsigned)site];
  };
  auto fetch = [&](int grp, int nb) {
    int p, site, s;
    const bool ok = locate(grp, p, site, s);
    const unsigned comp = (unsigned)(ri + 6 * sp) * Ls + s, step = 2u * Ls;
    if (rowt) {
      const float* x = gr + ((size_t)ac * 2 + p) * fsz + (size_t)site * 24 * Ls + comp;
#pragma unroll
      for (int c = 0; c < 3; ++c) va[c] = *reinterpret_cast<const flt4_t*>(x + c * step);
      if (tail && !ok)
#pragma unroll
        for (int c = 0; c < 3; ++c) va[c] = zero;
    }
    if (!colt) return;
    const float* x = in + ((size_t)bc * 2 + (hop ? 1 - p : p)) * fsz +
                     (size_t)(hop ? nb : site) * 24 * Ls + comp;
#pragma unroll
    for (int c = 0; c < 3; ++c) vb[c] = *reinterpret_cast<const flt4_t*>(x + c * step);
    if (hop) {
#pragma unroll
      for (int e = 0; e < 18; ++e) {
        // scalar base and 32-bit offset (left alone, the compiler adds up 64-bit addresses)
        typedef const __attribute__((address_space(1))) char* gptr_t;
        gptr_t ub = (gptr_t)(links + (((size_t)p * 8 + q - 1) * 18 + e) * Vh);
        asm("" : "+s"(ub));
        u[e] = *(const __attribute__((address_space(1))) float*)(ub + 4u * (unsigned)site);
      }
    } else if (q == 9) {
#pragma unroll
      for (int c = 0; c < 3; ++c) edge[c] = s + 4 < Ls ? x[c * step + 4] : 0.f;
    } else if (q == 10) {
#pragma unroll
      for (int c = 0; c < 3; ++c) edge[c] = s > 0 ? (x + c * step)[-1] : 0.f;
    }
  };
  // largest operands of this lane, one colour's for all (every sum runs over the colours)
  float max_a = 0.f, max_b = 0.f;
  auto parts = [&](flt4_t v, unsigned (&hi)[2], unsigned (&mid)[2], unsigned (&lo)[2]) {
    ptc_split_round(v[0], v[1], hi[0], mid[0], lo[0]);
    ptc_split_round(v[2], v[3], hi[1], mid[1], lo[1]);
  };
  auto put = [](u32x2_t* d, const unsigned (&hi)[2], const unsigned (&mid)[2],
                const unsigned (&lo)[2]) {
    d[0] = u32x2_t{hi[0], hi[1]};
    d[64] = u32x2_t{mid[0], mid[1]};
    d[128] = u32x2_t{lo[0], lo[1]};
  };
  auto stage = [&](unsigned flip) {
    unsigned hi[2], mid[2], lo[2];
    if (rowt) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          va[c][i] = __uint_as_float(__float_as_uint(va[c][i]) ^ flip);
        parts(va[c], hi, mid, lo);
        put(shA + (wave * 3 + c) * 192 + lane, hi, mid, lo);
      }
      max_a = ptc_absmax(ptc_absmax(max_a, va[0][0], va[0][1]), va[0][2], va[0][3]);
    }
    if (colt) {
      flt4_t x[3];
      if (hop) {
        // the other part of each component sits in the neighbouring lane
        flt4_t o[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[c][i] = __uint_as_float(__builtin_amdgcn_update_dpp(
                0, (int)__float_as_uint(vb[c][i]), 0xb1, 0xf, 0xf, true));   // quad_perm 1 0 3 2
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          x[c] = zero;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const float ur = u[2 * (k + 3 * c)], ui = sgn * u[2 * (k + 3 * c) + 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[c][i] = fmaf(ui, o[k][i], fmaf(ur, vb[k][i], x[c][i]));
          }
        }
      } else if (q == 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] = vb[c];
      } else if (q == 9) {
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] = flt4_t{vb[c][1], vb[c][2], vb[c][3], edge[c]};
      } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] = flt4_t{edge[c], vb[c][0], vb[c][1], vb[c][2]};
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        parts(x[c], hi, mid, lo);
        put(shB + (wave * 3 + c) * 192 + lane, hi, mid, lo);
      }
      max_b = ptc_absmax(ptc_absmax(max_b, x[0][0], x[0][1]), x[0][2], x[0][3]);
    }
  };
  const int tr = 2 * (wave >> 1), tc = 2 * (wave & 1);   // this wave's quadrant
  double acc[2][2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0;
  int nb = 0;
  if (first < last) {
    if (hop) nb = neighbour(first);
    fetch(first, nb);
    if (hop && first + 1 < last) nb = neighbour(first + 1);
  }
  for (int grp = first; grp < last; ++grp) {
    stage((unsigned)(grp & 1) << 31);
    __syncthreads();
    if (grp + 1 < last) {
      fetch(grp + 1, nb);
      if (hop && grp + 2 < last) nb = neighbour(grp + 2);
    }
    if (rt0 + tr < RT && ct0 + tc < CT) {
      const double sign = grp & 1 ? -1.0 : 1.0;
      flt4_t d[2][2] = {{zero, zero}, {zero, zero}};
      // parts (a0 a1) of the row tiles times (b0 b1) of the column tiles; 0 hi, 1 mid, 2 lo
      auto mma = [&](int c, int a0, int a1, int b0, int b1) {
        b8_t A[2], B[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const u32x2_t* x = shA + ((tr + i) * 3 + c) * 192 + lane;
          const u32x2_t* y = shB + ((tc + i) * 3 + c) * 192 + lane;
          const u32x2_t x0 = x[64 * a0], x1 = x[64 * a1], y0 = y[64 * b0], y1 = y[64 * b1];
          A[i] = __builtin_bit_cast(b8_t, u32x4_t{x0[0], x0[1], x1[0], x1[1]});
          B[i] = __builtin_bit_cast(b8_t, u32x4_t{y0[0], y0[1], y1[0], y1[1]});
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            d[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[i], B[j], d[i][j], 0, 0, 0);
      };
      // the small products of all three colours first: only the three large ones round at
      // the size of the result
#pragma unroll
      for (int c = 0; c < 3; ++c) mma(c, 0, 2, 2, 0);
      // (parts read anew for each pass come as whole operands; kept, they cost moves)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int c = 0; c < 3; ++c) mma(c, 1, 0, 0, 1);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int c = 0; c < 3; ++c) mma(c, 1, 0, 1, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] = fma(sign, (double)d[i][j][r], acc[i][j][r]);
    }
    __syncthreads();
  }
  if (__syncthreads_or(!ptc_in_range(max_a) || !ptc_in_range(max_b))) {
    // outside the range of the split: this block's points in FP32, pair by pair
    double* sh = reinterpret_cast<double*>(shA);
    const int a1 = min(2 * rt0 + 8, cout), b1 = min(2 * ct0 + 8, cin);
#pragma unroll 1
    for (int gb = 2 * ct0; gb < b1; ++gb)
#pragma unroll 1
      for (int ga = 2 * rt0; ga < a1; ++ga)
        ptc_wgrad_f32(partial + (((size_t)(q * cin + gb) * cout + ga) * gridDim.x + blockIdx.x) * 32,
                      gr, in, ga, gb, links, nbr, q, first, last, Vh, Ls, sh);
    return;
  }
  // P -> g conj(t): the lane of t_re holds (g_re, g_im) t_re in registers 2 k, 2 k + 1, its
  // neighbour those of t_im;  re = g_re t_re + g_im t_im,  im = g_im t_re - g_re t_im
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int ga = 2 * (rt0 + tr + i) + (g >> 1), gb = 2 * (ct0 + tc + j) + ch;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double x = acc[i][j][2 * k], py = __shfl_xor(acc[i][j][2 * k + 1], 1, 64);
        const double v = ri ? py - x : x + py;
        const int al = 2 * (g & 1) + k;
        if (ga < cout && gb < cin)
          partial[(((size_t)(q * cin + gb) * cout + ga) * gridDim.x + blockIdx.x) * 32 +
                  2 * (al * 4 + sp) + ri] = v;
      }
    }
}

// out[(y z) 32 + k] = sum over the nblk block partials, fixed order
__global__ void __launch_bounds__(64)
k_ptc_wgrad_finish(double* __restrict__ out, const double* __restrict__ partial, int nblk,
                   int nyz) {
  const int yz = blockIdx.x;
  const int k = threadIdx.x;
  if (yz >= nyz || k >= 32) return;
  double v = 0;
  for (int i = 0; i < nblk; ++i) v += partial[((size_t)yz * nblk + i) * 32 + k];
  out[(size_t)yz * 32 + k] = v;
}

// even part of channel 0 <- x (FP32 eo field), odd part <- 0
__global__ void __launch_bounds__(256)
k_ptc_embed(float* __restrict__ act, const float* __restrict__ x, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    act[i] = x[i];
    act[n + i] = 0.f;
  }
}

// g = 2 (y - t) on the even part of channel 0 (y = act), 0 on the odd part;
// block partials of |y - t|^2
__global__ void __launch_bounds__(256)
k_ptc_residual(float* __restrict__ g, const float* __restrict__ act, const float* __restrict__ t,
               size_t n, double* __restrict__ partial) {
  double acc = 0;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const float d = act[i] - t[i];
    acc += (double)d * (double)d;
    g[i] = 2.f * d;
    g[n + i] = 0.f;
  }
  __shared__ double sh[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if (lane == 0) sh[wv] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

static unsigned ptc_grid(size_t n) {
  size_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  return (unsigned)(g < 1 ? 1 : g);
}

template <bool ADJ, int AG>
static void ptc_layer_launch(float* out, const float* in, int cin, int cout, const unsigned* W,
                             int wcin, int wcout, const float* links, const int* nbr, int Vh,
                             int Ls, hipStream_t st) {
  const dim3 grid(ptc_grid((size_t)2 * Vh * Ls), cout / AG);
  hipLaunchKernelGGL((k_ptc_layer<ADJ, AG>), grid, dim3(256), 0, st, out, in, cin, W, wcin, wcout,
                     links, nbr, Vh, Ls);
}

// weights in LDS where they and the links of the four waves fit in 64 KB
template <bool ADJ, int NMT>
static void ptc_layer_mfma_launch(float* out, const float* in, int cin, int cout,
                                  const unsigned* W, int wcin, int wcout, const float* links,
                                  const int* nbr, int Vh, int Ls, hipStream_t st) {
  const size_t tiles = 2 * (((size_t)Vh * Ls + 15) / 16);
  const size_t wbytes = (size_t)kPtcPaths * wcin * wcout * 64;
  const size_t lbytes = (size_t)4 * ptc_wave_sites(Ls) * kPtcLinkSite * sizeof(float);
  const dim3 grid((unsigned)((tiles + 3) / 4)), block(256);
  const bool lw = lbytes + wbytes <= 64 * 1024 && reinterpret_cast<uintptr_t>(W) % 16 == 0;
#define PTC_GO(L, S, NB)                                                                      \
  hipLaunchKernelGGL((k_ptc_layer_mfma<ADJ, NMT, L, S, NB>), grid, block,                     \
                     lbytes + (L ? wbytes : 0), st, out, in, cin, cout, W, wcin, wcout, links, nbr, \
                     Vh, Ls)
  if (lw && cin == 1 && Ls == 16) PTC_GO(true, true, 1);
  else if (lw && cin == 1) PTC_GO(true, false, 1);
  else if (lw && Ls == 16) PTC_GO(true, true, 2);
  else if (lw) PTC_GO(true, false, 2);
  else if (Ls == 16) PTC_GO(false, true, 2);
  else PTC_GO(false, false, 2);
#undef PTC_GO
}

// DWF_PTC_KERNEL: "valu" selects the VALU kernels everywhere, "valu-wgrad" only for the weight
// gradients (the tests run them, and compare both gradients of the same layers)
static bool ptc_valu(bool wgrad) {
  const char* k = std::getenv("DWF_PTC_KERNEL");
  return k && (std::strcmp(k, "valu") == 0 || (wgrad && std::strcmp(k, "valu-wgrad") == 0));
}

template <bool ADJ>
static void ptc_layer_dispatch(float* out, const float* in, int cin, int cout, const unsigned* W,
                               int wcin, int wcout, const float* links, const int* nbr, int Vh,
                               int Ls, hipStream_t st) {
  // the matrix-core form (all output channels of 16 points per wave, an odd
  // count padded with a zero channel) wherever its 32-bit buffer offsets fit:
  // one channel's two parities, the links and the weights each below 2^31 bytes
  const size_t fsz = (size_t)Vh * 24 * Ls;
  const bool fits = 8 * fsz < (1ull << 31) && (size_t)2 * 8 * 18 * 4 * Vh < (1ull << 31);
  if (fits && !ptc_valu(false)) {
    switch ((cout + 1) / 2) {
#define PTC_MFMA(n)                                                                          \
  case n:                                                                                    \
    return ptc_layer_mfma_launch<ADJ, n>(out, in, cin, cout, W, wcin, wcout, links, nbr, Vh, \
                                         Ls, st);
      PTC_MFMA(1) PTC_MFMA(2) PTC_MFMA(3) PTC_MFMA(4)
      PTC_MFMA(5) PTC_MFMA(6) PTC_MFMA(7) PTC_MFMA(8)
#undef PTC_MFMA
      default: break;
    }
  }
  // otherwise the VALU form: four output channels per thread (227 registers, two
  // waves per SIMD); eight need 324 registers, one wave per SIMD, and are slower;
  // a thread per point and group, with 64-bit addressing
  if (cout % 4 == 0)
    ptc_layer_launch<ADJ, 4>(out, in, cin, cout, W, wcin, wcout, links, nbr, Vh, Ls, st);
  else if (cout % 2 == 0)
    ptc_layer_launch<ADJ, 2>(out, in, cin, cout, W, wcin, wcout, links, nbr, Vh, Ls, st);
  else
    ptc_layer_launch<ADJ, 1>(out, in, cin, cout, W, wcin, wcout, links, nbr, Vh, Ls, st);
}

hipError_t launch_ptc_layer(bool adj, float* out, const float* in, int cin, int cout,
                            const unsigned short* W, int wcin, int wcout, const float* links,
                            const int* nbr, int Vh, int Ls, hipStream_t st) {
  // each complex weight is one aligned 32-bit word (re, im)
  if (reinterpret_cast<uintptr_t>(W) % 4 != 0 || cout < 1) return hipErrorInvalidValue;
  const unsigned* w = reinterpret_cast<const unsigned*>(W);
  if (adj)
    ptc_layer_dispatch<true>(out, in, cin, cout, w, wcin, wcout, links, nbr, Vh, Ls, st);
  else
    ptc_layer_dispatch<false>(out, in, cin, cout, w, wcin, wcout, links, nbr, Vh, Ls, st);
  return hipGetLastError();
}

hipError_t launch_ptc_wgrad(double* G, double* partial, int maxblk, const float* g, const float* in,
                            int cin, int cout, const float* links, const int* nbr, int Vh, int Ls,
                            hipStream_t st) {
  if (cout < 1) return hipErrorInvalidValue;
  const int nyz = kPtcPaths * cin * cout;
  const size_t pts = (size_t)2 * Vh * Ls;
  // The matrix-core form needs four consecutive s per lane.  Its time hardly depends on how
  // far its 8 x 8 channel tiles are filled (8^3 x 16, Ls = 16: 8 -> 8 507 us, 1 -> 8 377),
  // the other one's is that of cin cout (1290 and 181): they would be equal near 25 products
  // a tile group, and the line lies a little above.
  const int tb = ((cout + 1) / 2 + 3) / 4 * (((cin + 1) / 2 + 3) / 4);
  if (Ls % 4 == 0 && cin * cout > 32 * tb && !ptc_valu(true)) {
    // four 16-point groups a block until all maxblk blocks are there (with the 64 groups
    // that the other form takes, 8 -> 8 at 4^3 x 8, Ls = 8, had 44 blocks on 256 CUs)
    const int nblk = (int)std::max<size_t>(1, std::min<size_t>(maxblk, pts / 64));
    hipLaunchKernelGGL(k_ptc_wgrad_mfma, dim3(nblk, kPtcPaths, tb), dim3(256), 0, st, partial, g,
                       in, cin, cout, links, nbr, Vh, Ls);
    hipLaunchKernelGGL(k_ptc_wgrad_finish, dim3(nyz), dim3(64), 0, st, G, partial, nblk, nyz);
    return hipGetLastError();
  }
  // about 1024 points per block
  const int nblk = (int)std::max<size_t>(1, std::min<size_t>(maxblk, pts / 1024));
  // two output channels per thread: four need 128 accumulators (266 registers,
  // one wave per SIMD), which is slower
  const int ag = cout % 2 == 0 ? 2 : 1;
  const dim3 grid(nblk, kPtcPaths * cin, cout / ag);
  if (ag == 2)
    hipLaunchKernelGGL(k_ptc_wgrad<2>, grid, dim3(256), 0, st, partial, g, in, cin, cout, links,
                       nbr, Vh, Ls);
  else
    hipLaunchKernelGGL(k_ptc_wgrad<1>, grid, dim3(256), 0, st, partial, g, in, cin, cout, links,
                       nbr, Vh, Ls);
  hipLaunchKernelGGL(k_ptc_wgrad_finish, dim3(nyz), dim3(64), 0, st, G, partial, nblk, nyz);
  return hipGetLastError();
}

hipError_t launch_ptc_embed(float* act, const float* x, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_ptc_embed, dim3(ptc_grid(n)), dim3(256), 0, st, act, x, n);
  return hipGetLastError();
}

hipError_t launch_ptc_residual(float* g, const float* act, const float* t, size_t n,
                               double* partial, unsigned* nblk, hipStream_t st) {
  unsigned gr = ptc_grid(n);
  if (gr > (unsigned)kRedBlocks) gr = kRedBlocks;
  *nblk = gr;
  hipLaunchKernelGGL(k_ptc_residual, dim3(gr), dim3(256), 0, st, g, act, t, n, partial);
  return hipGetLastError();
}

}  // namespace dwf
