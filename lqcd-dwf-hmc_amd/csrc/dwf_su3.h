// dwf_su3.h -- 3x3 complex matrix helpers of the FP64 gauge kernels
// (smearing, its force, the HMC gauge action and update).  Matrices are the
// corelib Mat_SU_N layout: 18 doubles, element (a, b) at 2 (3 a + b) (re, im).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dwf {

struct cplx {
  double r, i;
};
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return {a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r};
}
__device__ __forceinline__ cplx cscal(double s, cplx a) { return {s * a.r, s * a.i}; }

struct M3 {
  cplx a[3][3];
};

__device__ __forceinline__ M3 load3(const double* p) {
  M3 m;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) m.a[i][j] = {p[2 * (3 * i + j)], p[2 * (3 * i + j) + 1]};
  return m;
}
__device__ __forceinline__ void store3(double* p, const M3& m) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      p[2 * (3 * i + j)] = m.a[i][j].r;
      p[2 * (3 * i + j) + 1] = m.a[i][j].i;
    }
}
__device__ __forceinline__ M3 mul_nn(const M3& x, const M3& y) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx s = cmul(x.a[i][0], y.a[0][j]);
      s = cadd(s, cmul(x.a[i][1], y.a[1][j]));
      s = cadd(s, cmul(x.a[i][2], y.a[2][j]));
      r.a[i][j] = s;
    }
  return r;
}
// x * y^+
__device__ __forceinline__ M3 mul_nd(const M3& x, const M3& y) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx s = {0, 0};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const cplx a = x.a[i][k], b = y.a[j][k];
        s.r += a.r * b.r + a.i * b.i;
        s.i += a.i * b.r - a.r * b.i;
      }
      r.a[i][j] = s;
    }
  return r;
}
// x^+ * y
__device__ __forceinline__ M3 mul_dn(const M3& x, const M3& y) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx s = {0, 0};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const cplx a = x.a[k][i], b = y.a[k][j];
        s.r += a.r * b.r + a.i * b.i;
        s.i += a.r * b.i - a.i * b.r;
      }
      r.a[i][j] = s;
    }
  return r;
}

// x^+ * y^+ = (y x)^+
__device__ __forceinline__ M3 mul_dd(const M3& x, const M3& y) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cplx s = {0, 0};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const cplx a = x.a[k][i], b = y.a[j][k];
        s.r += a.r * b.r - a.i * b.i;
        s.i -= a.r * b.i + a.i * b.r;
      }
      r.a[i][j] = s;
    }
  return r;
}
// y += a x
__device__ __forceinline__ void m3_axpy(M3& y, double a, const M3& x) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      y.a[i][j].r += a * x.a[i][j].r;
      y.a[i][j].i += a * x.a[i][j].i;
    }
}
__device__ __forceinline__ void m3_add(M3& y, const M3& x) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) y.a[i][j] = cadd(y.a[i][j], x.a[i][j]);
}
__device__ __forceinline__ void m3_scal(M3& y, double a) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) y.a[i][j] = cscal(a, y.a[i][j]);
}
__device__ __forceinline__ M3 m3_zero() {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) r.a[i][j] = {0.0, 0.0};
  return r;
}

__device__ __forceinline__ M3 at3(const M3& m) {
  M3 r;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r.a[i][j] = {0.5 * (m.a[i][j].r - m.a[j][i].r), 0.5 * (m.a[i][j].i + m.a[j][i].i)};
  const double tr = (r.a[0][0].i + r.a[1][1].i + r.a[2][2].i) / 3.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) r.a[i][i].i -= tr;
  return r;
}

// 64 matrices of one wave, gathered through LDS.  A Field_G row is 144 bytes, so a
// lane that loads its own matrix touches 64 cache lines per instruction and the
// kernels that read neighbour links this way are bound by the L1's line lookups
// (75 matrices x 9 loads x 72 lines per wave are the 1.0 ms that the rectangle
// force at 32x16x16x24 took).  Here nine lanes load one row, seven rows (8 lines)
// per instruction, straight to LDS (the asynchronous global-to-LDS load), and
// every lane then reads its own row back (144-byte stride: the 16-byte reads of 8
// lanes cover the 32 banks once).  Two slots per wave: one matrix is in flight
// while another is multiplied.
typedef double dbl2v_t __attribute__((ext_vector_type(2)));
constexpr int kM3Slot = 640;   // 16-byte pieces of one slot: 10 loads of 64 lanes

template <bool WIDE> struct M3Pipe;
template <> struct M3Pipe<true> {
  dbl2v_t* sh;      // this wave's two slots
  int lane;
  int row4;         // 4 (lane / 9): bpermute address of the row this lane helps to load
  unsigned piece;   // 16 (lane % 9): its part of the row
  int mine;         // position of this lane's own row in a slot, in 16-byte pieces

  __device__ __forceinline__ M3Pipe(dbl2v_t* block_slots) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    sh = block_slots + wave * 2 * kM3Slot;
    lane = threadIdx.x & 63;
    row4 = 4 * (lane / 9);
    piece = 16u * (unsigned)(lane % 9);
    mine = (lane / 7) * 64 + (lane % 7) * 9;
  }
  // issue the load of row src (of this lane) of the field at base into a slot:
  // load i brings rows 7 i .. 7 i + 6 (lane 63 an unused piece), the last one row 63
  // (seven times, in place of a branch: across one the compiler sinks products and
  // runs out of registers).  Every lane takes part, src a valid row in all of them; the launchers
  // check that byte offsets fit in 32 bits.
  template <int SLOT> __device__ __forceinline__ void issue(const double* base, int src) const {
    const char* b = reinterpret_cast<const char*>(base);
    const int off = src * 144;
#pragma unroll
    for (int i = 0; i < 10; ++i) {
      const int r = i < 9 ? __builtin_amdgcn_ds_bpermute(row4 + 28 * i, off)
                          : __builtin_amdgcn_readlane(off, 63);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(b + ((unsigned)r + piece)),
          (__attribute__((address_space(3))) void*)(sh + SLOT * kM3Slot + i * 64), 16, 0, 0);
    }
  }
  // the first two matrices
  __device__ __forceinline__ void start(const double* b0, int s0, const double* b1, int s1) {
    issue<0>(b0, s0);
    // take() counts loads: slot 0's must be the older ones, and to the compiler the two
    // slots are unrelated memory
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue<1>(b1, s1);
  }
  // this lane's row of a slot once at most YOUNGER loads are outstanding.  One
  // asm block that waits for its own reads: reads that the compiler schedules
  // itself it would hold back until every load to LDS has landed.
  template <int SLOT, int YOUNGER> __device__ __forceinline__ M3 take() const {
    dbl2v_t q0, q1, q2, q3, q4, q5, q6, q7, q8;
    const unsigned rd = (unsigned)(uintptr_t)(__attribute__((address_space(3))) dbl2v_t*)sh +
                        16u * (unsigned)mine;
    asm volatile(
        "s_waitcnt vmcnt(%c10)\n\t"
        "ds_read_b128 %0, %9 offset:%c11\n\t"
        "ds_read_b128 %1, %9 offset:%c11+16\n\t"
        "ds_read_b128 %2, %9 offset:%c11+32\n\t"
        "ds_read_b128 %3, %9 offset:%c11+48\n\t"
        "ds_read_b128 %4, %9 offset:%c11+64\n\t"
        "ds_read_b128 %5, %9 offset:%c11+80\n\t"
        "ds_read_b128 %6, %9 offset:%c11+96\n\t"
        "ds_read_b128 %7, %9 offset:%c11+112\n\t"
        "ds_read_b128 %8, %9 offset:%c11+128\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(q3), "=&v"(q4), "=&v"(q5), "=&v"(q6), "=&v"(q7),
          "=&v"(q8)
        : "v"(rd), "n"(YOUNGER), "n"(SLOT * kM3Slot * 16)
        : "memory");
    M3 m;
    m.a[0][0] = {q0.x, q0.y}; m.a[0][1] = {q1.x, q1.y}; m.a[0][2] = {q2.x, q2.y};
    m.a[1][0] = {q3.x, q3.y}; m.a[1][1] = {q4.x, q4.y}; m.a[1][2] = {q5.x, q5.y};
    m.a[2][0] = {q6.x, q6.y}; m.a[2][1] = {q7.x, q7.y}; m.a[2][2] = {q8.x, q8.y};
    return m;
  }
  // the oldest matrix in flight, which sits in SLOT; the ten loads of the
  // younger one may still be outstanding.  The slot, whose reads have returned,
  // is refilled with row src of base.
  template <int SLOT> __device__ __forceinline__ M3 next(const double* base, int src) {
    const M3 m = take<SLOT, 10>();
    issue<SLOT>(base, src);
    return m;
  }
  // the same without a refill: the last two matrices (SLOT, then 1 - SLOT)
  template <int SLOT> __device__ __forceinline__ M3 drain() { return take<SLOT, 0>(); }
  __device__ __forceinline__ M3 next0(const double* base, int src) { return next<0>(base, src); }
  __device__ __forceinline__ M3 next1(const double* base, int src) { return next<1>(base, src); }
  __device__ __forceinline__ M3 drain0() { return drain<0>(); }
  __device__ __forceinline__ M3 drain1() { return drain<1>(); }
  // lane l's m to row first + l of base for the lanes l < n, n any (nothing in flight)
  __device__ __forceinline__ void store(double* base, int first, int n, const M3& m) const {
    dbl2v_t* p = sh + mine;
#pragma unroll
    for (int e = 0; e < 9; ++e) p[e] = dbl2v_t{m.a[e / 3][e % 3].r, m.a[e / 3][e % 3].i};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    dbl2v_t* g = reinterpret_cast<dbl2v_t*>(base) + (size_t)first * 9;
#pragma unroll
    for (int i = 0; i < 10; ++i) {
      const int c = 63 * i + lane;
      if (lane < 63 && c < 9 * (n < 64 ? n : 64)) g[c] = sh[64 * i + lane];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
};
// Fields that are not 16-byte aligned (a caller's sub-array): every lane loads
// its own matrices, in the same order of calls.
template <> struct M3Pipe<false> {
  const double *b0, *b1;
  int s0, s1;
  __device__ __forceinline__ M3Pipe(dbl2v_t*) {}
  __device__ __forceinline__ void start(const double* p0, int r0, const double* p1, int r1) {
    b0 = p0; s0 = r0;
    b1 = p1; s1 = r1;
  }
  template <int SLOT> __device__ __forceinline__ M3 drain() {
    return SLOT == 0 ? load3(b0 + (size_t)s0 * 18) : load3(b1 + (size_t)s1 * 18);
  }
  template <int SLOT> __device__ __forceinline__ M3 next(const double* base, int src) {
    const M3 m = drain<SLOT>();
    if (SLOT == 0) { b0 = base; s0 = src; }
    else { b1 = base; s1 = src; }
    return m;
  }
  __device__ __forceinline__ M3 next0(const double* base, int src) { return next<0>(base, src); }
  __device__ __forceinline__ M3 next1(const double* base, int src) { return next<1>(base, src); }
  __device__ __forceinline__ M3 drain0() { return drain<0>(); }
  __device__ __forceinline__ M3 drain1() { return drain<1>(); }
  __device__ __forceinline__ void store(double* base, int first, int n, const M3& m) const {
    const int lane = threadIdx.x & 63;
    if (lane < n) store3(base + ((size_t)first + lane) * 18, m);
  }
};

// Periodic lattice of a gauge kernel with one wave per (direction, 64 consecutive
// lexical sites).
struct GaugeLat {
  int N[4], st[4], V;
  int chunks;   // ceil(V / 64)
};
struct GaugeSite {
  int s;                // this lane's site (clamped to the last one in the tail)
  int c0, c1, c2, c3;
  __device__ __forceinline__ GaugeSite(const GaugeLat& L, int site) {
    s = site < L.V ? site : L.V - 1;
    int q = s;
    c0 = q % L.N[0];
    q /= L.N[0];
    c1 = q % L.N[1];
    q /= L.N[1];
    c2 = q % L.N[2];
    c3 = q / L.N[2];
  }
  // site + d mu_hat minus site, |d| <= 2, any extent >= 1 (mu uniform; masks, since
  // a chain of selects becomes an indexed load from memory)
  __device__ __forceinline__ int off(const GaugeLat& L, int mu, int d) const {
    const int x = (c0 & -(mu == 0)) | (c1 & -(mu == 1)) | (c2 & -(mu == 2)) | (c3 & -(mu == 3));
    const int N = L.N[mu], st = L.st[mu];
    int y = x + d;
#pragma unroll
    for (int k = 0; k < 2; ++k) y = y >= N ? y - N : (y < 0 ? y + N : y);
    return (y - x) * st;
  }
};
static inline GaugeLat gauge_lat(const int* dims) {
  GaugeLat L;
  int st = 1;
  for (int i = 0; i < 4; ++i) {
    L.N[i] = dims[i];
    L.st[i] = st;
    st *= dims[i];
  }
  L.V = st;
  L.chunks = (L.V + 63) / 64;
  return L;
}
// Whether 16-byte accesses can be used: device allocations are aligned, a caller's
// sub-arrays may not be.
static inline bool m3_wide(const void* a, const void* b = nullptr) {
  return (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

// Chunked form of a gauge field, [mu][ceil(V / 64)][element 9][site 64] complex:
// the 64 lanes of a wave read one element of 64 consecutive sites as 1 KB, so a
// gathered matrix costs nine L1 instructions of 8 lines instead of nine of 72.
__host__ __device__ __forceinline__ size_t chunked_doubles(size_t V) {
  return (V + 63) / 64 * 64 * 72;
}
__device__ __forceinline__ size_t chunked_mu(const GaugeLat& L) { return (size_t)L.chunks * 576; }
__device__ __forceinline__ M3 load3c(const dbl2v_t* b, int site) {
  const dbl2v_t* p = b + (size_t)(site >> 6) * 576 + (site & 63);
  M3 m;
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    const dbl2v_t v = p[e * 64];
    m.a[e / 3][e % 3] = {v.x, v.y};
  }
  return m;
}
__device__ __forceinline__ void store3c(dbl2v_t* b, int site, const M3& m) {
  dbl2v_t* p = b + (size_t)(site >> 6) * 576 + (site & 63);
#pragma unroll
  for (int e = 0; e < 9; ++e) p[e * 64] = dbl2v_t{m.a[e / 3][e % 3].r, m.a[e / 3][e % 3].i};
}
// Rows first .. first + 63 (those below V) of a Field_G direction to and from one
// matrix per lane of a wave, coalesced through 9 KB of LDS per wave; rows at 16
// bytes when WIDE, else at 8.
constexpr int kRowsLds = 576;   // 16-byte pieces
template <bool WIDE>
__device__ __forceinline__ M3 rows_load(const double* base, int first, int V, dbl2v_t* sh) {
  const int lane = threadIdx.x & 63, n = V - first < 64 ? V - first : 64;
  if constexpr (!WIDE) return load3(base + ((size_t)first + (lane < n ? lane : n - 1)) * 18);
  const dbl2v_t* g = reinterpret_cast<const dbl2v_t*>(base) + (size_t)first * 9;
  dbl2v_t v[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int c = 64 * i + lane;
    v[i] = g[c < 9 * n ? c : 9 * n - 1];
  }
#pragma unroll
  for (int i = 0; i < 9; ++i) sh[64 * i + lane] = v[i];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  M3 m;
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    const dbl2v_t w = sh[lane * 9 + e];
    m.a[e / 3][e % 3] = {w.x, w.y};
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return m;
}
template <bool WIDE>
__device__ __forceinline__ void rows_store(double* base, int first, int V, dbl2v_t* sh,
                                           const M3& m) {
  const int lane = threadIdx.x & 63, n = V - first < 64 ? V - first : 64;
  if constexpr (!WIDE) {
    if (lane < n) store3(base + ((size_t)first + lane) * 18, m);
    return;
  }
#pragma unroll
  for (int e = 0; e < 9; ++e) sh[lane * 9 + e] = dbl2v_t{m.a[e / 3][e % 3].r, m.a[e / 3][e % 3].i};
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  dbl2v_t* g = reinterpret_cast<dbl2v_t*>(base) + (size_t)first * 9;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int c = 64 * i + lane;
    if (c < 9 * n) g[c] = sh[c];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lexical neighbour of site s in direction mu (dir = +1 or -1), periodic
__device__ __forceinline__ size_t shift_site(size_t s, int mu, int dir, int Nx, int Ny, int Nz,
                                             int Nt) {
  int x = (int)(s % Nx);
  size_t q = s / Nx;
  int y = (int)(q % Ny);
  q /= Ny;
  int z = (int)(q % Nz);
  int t = (int)(q / Nz);
  if (mu == 0) x = (x + dir + Nx) % Nx;
  else if (mu == 1) y = (y + dir + Ny) % Ny;
  else if (mu == 2) z = (z + dir + Nz) % Nz;
  else t = (t + dir + Nt) % Nt;
  return x + (size_t)Nx * (y + (size_t)Ny * (z + (size_t)Nz * t));
}

}  // namespace dwf
