// dwf_device.h -- device-side types shared by the HIP sources of libdwfhip.
//
// Storage traits: a field is stored as T (double, float, __half, bfloat16) and
// computed in C (double for T = double, float otherwise).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

namespace dwf {

template <typename T> struct St;
// ld/st: ordinary cached access.  ldn/stn: streaming (non-temporal) access for
// data touched once, so that it does not evict reusable lines from L2.
template <> struct St<double> {
  using C = double;
  static __device__ __forceinline__ double ld(const double* p) { return *p; }
  static __device__ __forceinline__ void st(double* p, double v) { *p = v; }
  static __device__ __forceinline__ double ldn(const double* p) { return __builtin_nontemporal_load(p); }
  static __device__ __forceinline__ void stn(double* p, double v) { __builtin_nontemporal_store(v, p); }
};
template <> struct St<float> {
  using C = float;
  static __device__ __forceinline__ float ld(const float* p) { return *p; }
  static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
  static __device__ __forceinline__ float ldn(const float* p) { return __builtin_nontemporal_load(p); }
  static __device__ __forceinline__ void stn(float* p, float v) { __builtin_nontemporal_store(v, p); }
};
template <> struct St<__half> {
  using C = float;
  static __device__ __forceinline__ float ld(const __half* p) { return __half2float(*p); }
  static __device__ __forceinline__ void st(__half* p, float v) { *p = __float2half(v); }
  static __device__ __forceinline__ float ldn(const __half* p) {
    unsigned short b = __builtin_nontemporal_load(reinterpret_cast<const unsigned short*>(p));
    return __half2float(__ushort_as_half(b));
  }
  static __device__ __forceinline__ void stn(__half* p, float v) {
    __builtin_nontemporal_store(__half_as_ushort(__float2half(v)), reinterpret_cast<unsigned short*>(p));
  }
};
template <> struct St<__hip_bfloat16> {
  using C = float;
  static __device__ __forceinline__ float ld(const __hip_bfloat16* p) { return __bfloat162float(*p); }
  static __device__ __forceinline__ void st(__hip_bfloat16* p, float v) { *p = __float2bfloat16(v); }
  static __device__ __forceinline__ float ldn(const __hip_bfloat16* p) {
    unsigned short b = __builtin_nontemporal_load(reinterpret_cast<const unsigned short*>(p));
    return __uint_as_float((unsigned)b << 16);
  }
  static __device__ __forceinline__ void stn(__hip_bfloat16* p, float v) {
    __hip_bfloat16 h = __float2bfloat16(v);
    __builtin_nontemporal_store(*reinterpret_cast<const unsigned short*>(&h),
                                reinterpret_cast<unsigned short*>(p));
  }
};

// Vx<T, V>: V consecutive elements (aligned to V) moved with one vector access.
// R is the raw register form (packed for 16-bit storage); get() unpacks one
// element to the compute type, ld/stn move all V.
typedef double dbl2_t __attribute__((ext_vector_type(2)));
typedef float flt2_t __attribute__((ext_vector_type(2)));
typedef float flt4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

template <typename T, int V> struct Vx;
template <> struct Vx<double, 1> {
  using R = double;
  static __device__ __forceinline__ R ld(const double* p) { return *p; }
  static __device__ __forceinline__ double get(const R& r, int) { return r; }
  static __device__ __forceinline__ void stn(double* p, const double* v) {
    __builtin_nontemporal_store(v[0], p);
  }
};
template <> struct Vx<double, 2> {
  using R = dbl2_t;
  static __device__ __forceinline__ R ld(const double* p) { return *reinterpret_cast<const R*>(p); }
  static __device__ __forceinline__ double get(const R& r, int v) { return r[v]; }
  static __device__ __forceinline__ void stn(double* p, const double* v) {
    R t = {v[0], v[1]};
    __builtin_nontemporal_store(t, reinterpret_cast<R*>(p));
  }
};
template <> struct Vx<float, 1> {
  using R = float;
  static __device__ __forceinline__ R ld(const float* p) { return *p; }
  static __device__ __forceinline__ float get(const R& r, int) { return r; }
  static __device__ __forceinline__ void stn(float* p, const float* v) {
    __builtin_nontemporal_store(v[0], p);
  }
};
template <> struct Vx<float, 2> {
  using R = flt2_t;
  static __device__ __forceinline__ R ld(const float* p) { return *reinterpret_cast<const R*>(p); }
  static __device__ __forceinline__ float get(const R& r, int v) { return r[v]; }
  static __device__ __forceinline__ void stn(float* p, const float* v) {
    R t = {v[0], v[1]};
    __builtin_nontemporal_store(t, reinterpret_cast<R*>(p));
  }
};
template <> struct Vx<float, 4> {
  using R = flt4_t;
  static __device__ __forceinline__ R ld(const float* p) { return *reinterpret_cast<const R*>(p); }
  static __device__ __forceinline__ float get(const R& r, int v) { return r[v]; }
  static __device__ __forceinline__ void stn(float* p, const float* v) {
    R t = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(t, reinterpret_cast<R*>(p));
  }
};
// 16-bit storage: 2 elements per 32-bit word, element 0 in the low half
__device__ __forceinline__ float h_lo(unsigned w) { return __half2float(__ushort_as_half((unsigned short)(w & 0xffffu))); }
__device__ __forceinline__ float h_hi(unsigned w) { return __half2float(__ushort_as_half((unsigned short)(w >> 16))); }
__device__ __forceinline__ unsigned h_pack(float a, float b) {
  return (unsigned)__half_as_ushort(__float2half(a)) | ((unsigned)__half_as_ushort(__float2half(b)) << 16);
}
__device__ __forceinline__ float b_lo(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float b_hi(unsigned w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ unsigned b_pack(float a, float b) {
  const __hip_bfloat16 x = __float2bfloat16(a), y = __float2bfloat16(b);
  return (unsigned)*reinterpret_cast<const unsigned short*>(&x) |
         ((unsigned)*reinterpret_cast<const unsigned short*>(&y) << 16);
}
template <typename T> struct Pk16;
template <> struct Pk16<__half> {
  static __device__ __forceinline__ float lo(unsigned w) { return h_lo(w); }
  static __device__ __forceinline__ float hi(unsigned w) { return h_hi(w); }
  static __device__ __forceinline__ unsigned pack(float a, float b) { return h_pack(a, b); }
};
template <> struct Pk16<__hip_bfloat16> {
  static __device__ __forceinline__ float lo(unsigned w) { return b_lo(w); }
  static __device__ __forceinline__ float hi(unsigned w) { return b_hi(w); }
  static __device__ __forceinline__ unsigned pack(float a, float b) { return b_pack(a, b); }
};
// 16-bit outputs are written as 4- or 8-byte pieces of 32-byte rows: they go
// through L2 as ordinary stores, so that the pieces of a line are merged before
// the line is written back (non-temporal stores wrote 1.33x the bytes).
#ifndef DWF_NT_STORE16
#define DWF_NT_STORE16 0
#endif
template <typename R> __device__ __forceinline__ void st16(R* p, R v) {
#if DWF_NT_STORE16
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
}
template <typename T> struct Vx16_2 {
  using R = unsigned;
  static __device__ __forceinline__ R ld(const T* p) { return *reinterpret_cast<const unsigned*>(p); }
  static __device__ __forceinline__ float get(const R& r, int v) {
    return v == 0 ? Pk16<T>::lo(r) : Pk16<T>::hi(r);
  }
  static __device__ __forceinline__ void stn(T* p, const float* v) {
    st16(reinterpret_cast<unsigned*>(p), Pk16<T>::pack(v[0], v[1]));
  }
};
template <typename T> struct Vx16_4 {
  using R = u32x2_t;
  static __device__ __forceinline__ R ld(const T* p) { return *reinterpret_cast<const R*>(p); }
  static __device__ __forceinline__ float get(const R& r, int v) {
    const unsigned w = r[v >> 1];
    return (v & 1) ? Pk16<T>::hi(w) : Pk16<T>::lo(w);
  }
  static __device__ __forceinline__ void stn(T* p, const float* v) {
    R t = {Pk16<T>::pack(v[0], v[1]), Pk16<T>::pack(v[2], v[3])};
    st16(reinterpret_cast<R*>(p), t);
  }
};
template <> struct Vx<__half, 2> : Vx16_2<__half> {};
template <> struct Vx<__half, 4> : Vx16_4<__half> {};
template <> struct Vx<__hip_bfloat16, 2> : Vx16_2<__hip_bfloat16> {};
template <> struct Vx<__hip_bfloat16, 4> : Vx16_4<__hip_bfloat16> {};
template <> struct Vx<__half, 1> {
  using R = float;
  static __device__ __forceinline__ R ld(const __half* p) { return St<__half>::ld(p); }
  static __device__ __forceinline__ float get(const R& r, int) { return r; }
  static __device__ __forceinline__ void stn(__half* p, const float* v) { St<__half>::stn(p, v[0]); }
};
template <> struct Vx<__hip_bfloat16, 1> {
  using R = float;
  static __device__ __forceinline__ R ld(const __hip_bfloat16* p) { return St<__hip_bfloat16>::ld(p); }
  static __device__ __forceinline__ float get(const R& r, int) { return r; }
  static __device__ __forceinline__ void stn(__hip_bfloat16* p, const float* v) {
    St<__hip_bfloat16>::stn(p, v[0]);
  }
};

// Kernel-side geometry of one even-odd half lattice.
struct Geo {
  int Vh;   // half volume (4D)
  int Ls;   // extent of the 5th dimension
};

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Remap the hardware workgroup id so that every XCD walks a contiguous
// range of sites: neighbouring sites then share an L2.
__device__ __forceinline__ int xcd_block(int w, int G) {
  const int q = G >> 3, r = G & 7;
  const int x = w & 7, i = w >> 3;
  return x * q + (x < r ? x : r) + i;
}

// ---------------------------------------------------------------------------
// spin projection, Dirac basis.  dir = 2*mu + fb,
// fb = 0: (1 - gamma_mu) U_mu(x) psi(x+mu), fb = 1: (1 + gamma_mu) U^+ psi(x-mu).
// w[k], k = ri + 2*(c + 3*d).
// ---------------------------------------------------------------------------
template <int DIR, typename C>
__device__ __forceinline__ void project(const C* w, C* h1, C* h2) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int r = 2 * c, i = 2 * c + 1;
    const C* w0 = w;
    const C* w1 = w + 6;
    const C* w2 = w + 12;
    const C* w3 = w + 18;
    if (DIR == 0) {         // h1 = w0 + i w3, h2 = w1 + i w2
      h1[r] = w0[r] - w3[i]; h1[i] = w0[i] + w3[r];
      h2[r] = w1[r] - w2[i]; h2[i] = w1[i] + w2[r];
    } else if (DIR == 1) {  // h1 = w0 - i w3, h2 = w1 - i w2
      h1[r] = w0[r] + w3[i]; h1[i] = w0[i] - w3[r];
      h2[r] = w1[r] + w2[i]; h2[i] = w1[i] - w2[r];
    } else if (DIR == 2) {  // h1 = w0 + w3, h2 = w1 - w2
      h1[r] = w0[r] + w3[r]; h1[i] = w0[i] + w3[i];
      h2[r] = w1[r] - w2[r]; h2[i] = w1[i] - w2[i];
    } else if (DIR == 3) {  // h1 = w0 - w3, h2 = w1 + w2
      h1[r] = w0[r] - w3[r]; h1[i] = w0[i] - w3[i];
      h2[r] = w1[r] + w2[r]; h2[i] = w1[i] + w2[i];
    } else if (DIR == 4) {  // h1 = w0 + i w2, h2 = w1 - i w3
      h1[r] = w0[r] - w2[i]; h1[i] = w0[i] + w2[r];
      h2[r] = w1[r] + w3[i]; h2[i] = w1[i] - w3[r];
    } else if (DIR == 5) {  // h1 = w0 - i w2, h2 = w1 + i w3
      h1[r] = w0[r] + w2[i]; h1[i] = w0[i] - w2[r];
      h2[r] = w1[r] - w3[i]; h2[i] = w1[i] + w3[r];
    } else if (DIR == 6) {  // h1 = 2 w2, h2 = 2 w3
      h1[r] = w2[r] + w2[r]; h1[i] = w2[i] + w2[i];
      h2[r] = w3[r] + w3[r]; h2[i] = w3[i] + w3[i];
    } else {                // h1 = 2 w0, h2 = 2 w1
      h1[r] = w0[r] + w0[r]; h1[i] = w0[i] + w0[i];
      h2[r] = w1[r] + w1[r]; h2[i] = w1[i] + w1[i];
    }
  }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// Sum of n partials by one block of up to 8 waves, in a fixed order (thread t
// adds t, t + blockDim, ...; then the wave sums in wave order); with 256
// threads it is the order of k_red_finish.  sh holds 8 doubles.
__device__ __forceinline__ double block_sum(const double* __restrict__ p, unsigned n,
                                            double* sh) {
  double w = 0;
  for (unsigned i = threadIdx.x; i < n; i += blockDim.x) w += p[i];
  const double t = wave_sum(w);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = t;
  __syncthreads();
  double r = 0;
  for (unsigned k = 0; k < (blockDim.x >> 6); ++k) r += sh[k];
  __syncthreads();
  return r;
}

// a = U h for a 3x3 row-major complex matrix u[ab], ab = ri + 2*(b + 3*a)
template <typename C>
__device__ __forceinline__ void su3_mul(const C* u, const C* h, C* a) {
#pragma unroll
  for (int ia = 0; ia < 3; ++ia) {
    C re = 0, im = 0;
#pragma unroll
    for (int ib = 0; ib < 3; ++ib) {
      const C ur = u[2 * (ib + 3 * ia)], ui = u[2 * (ib + 3 * ia) + 1];
      re += ur * h[2 * ib] - ui * h[2 * ib + 1];
      im += ur * h[2 * ib + 1] + ui * h[2 * ib];
    }
    a[2 * ia] = re;
    a[2 * ia + 1] = im;
  }
}

}  // namespace dwf
