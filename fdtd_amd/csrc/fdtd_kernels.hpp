// Device code of libfdtd_hip: fused Yee half-step kernels for MI355X (gfx950).
//
// One E half step is, per cell and in this order (fdtd/grid.py:275-299):
//   curl = backward-difference curl of H                 (grid.py:54-76)
//   E   += (S * inv_eps) * curl                          (grid.py:283)
//   objects in registration order                        (objects.py:118-269)
//   boundaries in registration order: CPML correction    (boundaries.py:409-459)
//     or periodic plane copy                             (boundaries.py:184-219)
//   sources in registration order, then detectors        (sources.py, detectors.py)
// and the H half step mirrors it (grid.py:301-325). Every floating-point
// operation is the one the reference performs, in the same order, with
// contraction disabled (-ffp-contract=off), so float64 results match the
// numpy reference bit for bit.
//
// The kernels are written once over two policies:
//   field storage  PlainField<S, R>  values stored as S, computed in R
//                                    (S = R = cplx<double/float> for the
//                                    complex-field path)
//                  CompField         float plus an 8-bit compensation term
//                                    (the next 8 mantissa bits: a 40-bit
//                                    format), computed in double
//   material       MatArray<S, R>    per-cell (3, N) array
//                  MatPalette<R>     one byte per cell indexing <= 256 float64
//                                    triples
//
// Kernels
//   k_main_E / k_main_H  curl, material update and every CPML face registered
//                        before the first periodic boundary; a workgroup
//                        marches along x over a (y,z) tile (~0.16 flop/B).
//                        k_any_E / k_any_H: the form for any faces, and with
//                        objects; k_object_E: it over the tiles with objects.
//   k_face               one CPML face over its slab, for faces registered
//                        after a periodic boundary (order matters there).
//   k_periodic           plane copy of a periodic boundary.
//   k_tail               sources (in order) then detectors.
//   k_batch_E / k_batch_H  the main kernels' tile bodies over the tiles of
//                        many grids (one launch per half step); k_set_time
//                        sets their device time index.
//   k_adj_H / k_adj_E    transposes of the H and E half steps (reverse mode),
//                        objective and design gradient fused.
//   k_copy               plain streaming copy (bandwidth reference).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fdtd_hip.h"

namespace fdtd_dev {

// ---------------------------------------------------------------- plan data
struct FaceDev {
  int32_t axis, high, t, pad;
  const double* bE;
  const double* cE;
  const double* bH;
  const double* cH;
  void* psiE;  // psi in the arithmetic type R of the plan
  void* psiH;
  int64_t slab;  // cells in the face slab
};

struct ObjDev {
  int32_t kind, x0, x1, y0, y1, z0, z1;
  int32_t real;        // the reference's arrays of this object are real (see absorb_ratio)
  const void* inv;     // in the plan's object type
  const void* absorb;
};

struct SrcDev {
  int32_t kind, n, compE, compH;
  const int64_t* cells;
  const double* profile;
  double amplitude;  // FDTD_SRC_SOFT: the impedance
  // FDTD_SRC_SOFT only
  double spacing;
  int32_t det, pad;  // current detector read
  void* vin;
  void* vout;
  int64_t slot0;     // slot written at E half-step counter c is c - slot0
};

// Current detector: n points (px, py, pz), loop currents after each H half step.
struct CurDev {
  int32_t n, pad;
  const int32_t* pts;  // px[n], py[n], pz[n]
  double spacing;
  void* buf;           // (capacity, n)
  int64_t slot0;       // slot written at H half-step counter c is c - slot0
};

struct DetDev {
  int32_t n, pad;
  const int64_t* cells;
  void* bufE;
  void* bufH;
  int64_t slot0E, slot0H;  // slot written at half-step counter c is c - slot0
};

// Cell (i, j, k) of a component is at i*px + j*nz + k: z fastest, x planes
// `px` cells apart (px >= ny*nz; the host may round a plane up so that every
// x plane starts on a cache line; the cells past ny*nz are then never read or
// written), components cs = nx*px apart.
struct Dims {
  int32_t nx, ny, nz, pad;
  int64_t cs;  // component stride nx*px
  int64_t px;  // x-plane pitch
};

__host__ __device__ __forceinline__ int64_t cell_of(const Dims& d, int64_t i, int64_t j, int64_t k) {
  return i * d.px + j * d.nz + k;
}

// ------------------------------------------------------- load/store helpers
// Loads and stores of the read-once streams (the updated field and the
// material); NT marks them non-temporal so the L2 keeps the other field,
// whose planes and rows are re-read as halos.
// Every array lives in global memory. Pointers read from tables in device
// memory (the per-grid arguments of the batched kernels, the face, object,
// source and detector tables) carry no address space, and accesses through
// them would be generic (flat) ones; gp() states the global space, which
// gives global loads with a scalar base.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> gp(T* p) {
  return (gptr<T>)p;
}

// Read-only tables: the constant address space, so that uniform reads are
// scalar loads whatever the kernel stores in between.
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ cptr<T> cp(const T* p) {
  return (cptr<T>)p;
}

// Keeps a work-item's offset out of loop-invariant address arithmetic: the
// compiler would otherwise add it to each array's base outside the loop (a
// 64-bit register pair per array and component, and a 64-bit addition per
// access) instead of using the scalar base + 32-bit offset form of an access.
__device__ __forceinline__ void opaque(uint32_t& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(x));
#endif
}
// The same for a table's address: what is read through it is read again each
// time round a loop rather than kept in scalar registers across it.
template <typename P>
__device__ __forceinline__ void opaque_table(P& p) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(p));
#endif
}

// Whether any lane of the wavefront has x (a host build runs its work-items
// one by one: the work-item's own x).
__device__ __forceinline__ bool wave_any(bool x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ballot_w64(x) != 0;
#else
  return x;
#endif
}

// p[0] of an array whose base is the same for the whole wavefront, `off` bytes
// further on.
template <typename T>
__device__ __forceinline__ T* split_ptr(T* p, uint32_t off) {
  return (T*)((gptr<char>)gp(p) + off);
}
template <typename T>
__device__ __forceinline__ const T* split_ptr(const T* p, uint32_t off) {
  return (const T*)((gptr<const char>)gp(p) + off);
}

template <bool NT, typename T>
__device__ __forceinline__ T ld_stream(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(gp(p));
  else return *gp(p);
}
template <bool NT, typename T>
__device__ __forceinline__ void st_stream(T* p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, gp(p));
  else *gp(p) = v;
}

// ------------------------------------------------------------ complex values
// The reference promotes E, H and the CPML state to complex when an object
// with a complex permittivity is registered (grid.py:353-356,
// objects.py:51-52) and then steps with numpy's complex arithmetic. numpy's
// vectorised loop multiplies complex numbers as
//   re = fma(ar, br, -(ai * bi)),  im = fma(ar, bi, ai * br)
// (checked bit for bit against its results), and promotes a real operand x
// to (x, 0), which makes every real-times-complex product exactly the
// componentwise one; sums and differences are componentwise. cplx<S> does
// the same, so the complex path matches the reference bit for bit as well.
// Division is numpy's for complex values (Smith's method, with its
// zero-divisor branch); a real operand of a division is promoted to (x, 0)
// there as well, which is NOT the componentwise quotient. Absorbing objects
// divide (objects.py:215-221).
template <typename S>
struct cplx {
  S re, im;
  __host__ __device__ cplx() : re(0), im(0) {}
  __host__ __device__ cplx(S r) : re(r), im(0) {}
  __host__ __device__ cplx(S r, S i) : re(r), im(i) {}
  friend __host__ __device__ cplx operator+(cplx a, cplx b) { return cplx(a.re + b.re, a.im + b.im); }
  friend __host__ __device__ cplx operator-(cplx a, cplx b) { return cplx(a.re - b.re, a.im - b.im); }
  friend __host__ __device__ cplx operator-(cplx a) { return cplx(-a.re, -a.im); }
  friend __host__ __device__ cplx operator*(cplx a, cplx b) {
    return cplx(fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re));
  }
  friend __host__ __device__ cplx operator/(cplx a, cplx b) {
    if (fabs(b.re) >= fabs(b.im)) {
      if (b.re == S(0) && b.im == S(0)) return cplx(a.re / fabs(b.re), a.im / fabs(b.re));
      const S rat = b.im / b.re, scl = S(1) / (b.re + b.im * rat);
      return cplx((a.re + a.im * rat) * scl, (a.im - a.re * rat) * scl);
    }
    const S rat = b.re / b.im, scl = S(1) / (b.im + b.re * rat);
    return cplx((a.re * rat + a.im) * scl, (a.im * rat - a.re) * scl);
  }
};

template <bool NT, typename S>
__device__ __forceinline__ cplx<S> ld_stream(const cplx<S>* p) {
  const S* q = reinterpret_cast<const S*>(p);
  return cplx<S>(ld_stream<NT>(q), ld_stream<NT>(q + 1));
}
template <bool NT, typename S>
__device__ __forceinline__ void st_stream(cplx<S>* p, cplx<S> v) {
  S* q = reinterpret_cast<S*>(p);
  st_stream<NT>(q, v.re);
  st_stream<NT>(q + 1, v.im);
}

// ------------------------------------------------------------ field storage
// Element i of a field is component i / cs of cell i % cs (component-major).
// get/put/copy/sample take that element index; get_c/get3/put3 take a cell
// and address its components (the main kernels' accesses).
template <typename S, typename R_>
struct PlainField {
  using R = R_;
  using Sample = S;
  using Elem = S;
  static constexpr bool kRecords = false;  // the marching kernels' record path (CompField) is off
  struct Rec {};
  S* p;
  int64_t cs;
  template <int C>
  __device__ __forceinline__ R get_c(int64_t cell) const { return (R)ld_stream<false>(p + C * cs + cell); }
  template <bool NT>
  __device__ __forceinline__ void get3_s(int64_t cell, R v[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = (R)ld_stream<NT>(p + c * cs + cell);
  }
  template <bool NT>
  __device__ __forceinline__ void put3_s(int64_t cell, const R v[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) st_stream<NT>(p + c * cs + cell, (S)v[c]);
  }
  __device__ __forceinline__ R get(int64_t i) const { return (R)ld_stream<false>(p + i); }
  template <bool NT>
  __device__ __forceinline__ R get_s(int64_t i) const { return (R)ld_stream<NT>(p + i); }
  template <bool NT>
  __device__ __forceinline__ void put_s(int64_t i, R v) const { st_stream<NT>(p + i, (S)v); }
  __device__ __forceinline__ void put(int64_t i, R v) const { st_stream<false>(p + i, (S)v); }
  __device__ __forceinline__ void copy(int64_t dst, int64_t src) const { st_stream<false>(p + dst, ld_stream<false>(p + src)); }
  __device__ __forceinline__ Sample sample(int64_t i) const { return ld_stream<false>(p + i); }
  // The same accesses with the cell split into a part that is the same for
  // the whole wavefront and a byte offset of 32 bits per work-item, which is
  // the form a global access takes without any address arithmetic. Own: the
  // three components of a cell, Duo: two of a neighbour's, as loaded.
  static constexpr uint32_t kCell = sizeof(S);
  struct Own {
    S v[3];
  };
  struct Duo {
    S a, b;
  };
  __device__ __forceinline__ S* at(int c, int64_t uni, uint32_t off) const { return split_ptr(p + c * cs + uni, off); }
  template <bool NT>
  __device__ __forceinline__ Own own(int64_t uni, uint32_t off) const {
    return {{ld_stream<NT>(at(0, uni, off)), ld_stream<NT>(at(1, uni, off)), ld_stream<NT>(at(2, uni, off))}};
  }
  template <int C0, int C1>
  __device__ __forceinline__ Duo duo(int64_t uni, uint32_t off) const {
    return {ld_stream<false>(at(C0, uni, off)), ld_stream<false>(at(C1, uni, off))};
  }
  template <int C>
  static __device__ __forceinline__ R value(const Own& o) { return (R)o.v[C]; }
  template <int C0, int C1, int C>
  static __device__ __forceinline__ R value(const Duo& o) { return (R)(C == C0 ? o.a : o.b); }
  template <bool NT>
  __device__ __forceinline__ void put_own(int64_t uni, uint32_t off, const R v[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) st_stream<NT>(at(c, uni, off), (S)v[c]);
  }
  // the value as a store and a load leave it, and as a detector samples it
  static __device__ __forceinline__ R rounded(R v) { return v; }
  static __device__ __forceinline__ Sample sampled(R v) { return (S)v; }
};

// Compensated storage: a value v is kept as the float h holding the top 24
// significant bits of v rounded to 32 significant bits, plus a byte q with
// the next 8 bits -- a 40-bit floating-point format whose byte is the
// compensation term of the float (what rounding v to the float drops).
// Decoding is exact in double: widen h (its mantissa lands in bits 51..29 of
// the double) and insert q at bits 28..21. Encoding rounds |v| to nearest at
// bit 21 by adding 2^20 to the bit pattern (the carry may ripple into the
// exponent, which is the correct rounding of the magnitude), then splits the
// result. Relative error of a store: at most 2^-32. Values below the float
// range (|v| < 2^-126) keep the float's precision only.
__device__ __forceinline__ double comp_decode(float h, uint32_t q) {
  const double w = (double)h;
  const uint32_t lo32 = (uint32_t)__double2loint(w) | (q << 21);
  return __hiloint2double(__double2hiint(w), (int)lo32);
}
__device__ __forceinline__ float comp_hi(double v, uint32_t& q) {
  const uint64_t u = (uint64_t)__double_as_longlong(v) + (1ull << 20);
  q = (uint32_t)((u >> 21) & 0xffu);
  return (float)__longlong_as_double((long long)(u & ~((1ull << 29) - 1)));
}

// A cell is one 16-byte record, (N, 4) floats: its x, y, z floats and a
// 32-bit word holding the three compensation bytes (byte c for component c),
// so a cell's three components and their compensation come in one 16-byte
// access (four 4-byte accesses with the floats (3, N) and the words apart),
// with no padding. Loads are 16-byte vectors; stores are four float stores
// (merged into one 16-byte store by the backend): a store of the vector type
// may alias any table, with the effect described next. The words are accessed
// as float bit patterns (moved, never computed with): stores of
// an integer type could alias the integer fields of the face and object
// tables that the same loops read, and type-based alias analysis would then
// turn those uniform table reads into vector loads that wait for every
// outstanding store, once per face and cell.
// 16-byte vector of four floats (GCC vector extension: element access by [])
typedef float f32x4 __attribute__((vector_size(16)));

struct CompField {
  using R = double;
  using Sample = float;
  using Elem = float;
  // The marching kernels keep the previous plane's record as loaded and
  // decode it where it is used: a decoded carry is computed right after its
  // load, ahead of the branch that guards a cell's store, so the wave would
  // wait for that load before issuing the plane's others (two memory round
  // trips per plane instead of one).
  static constexpr bool kRecords = true;
  using Rec = f32x4;
  float* rec;  // (N, 4): x, y, z rounded to float, then the compensation word
  int64_t cs;
  __device__ __forceinline__ int comp_of(int64_t i) const { return i >= 2 * cs ? 2 : (i >= cs ? 1 : 0); }
  template <bool NT>
  __device__ __forceinline__ f32x4 record(int64_t cell) const {
    return ld_stream<NT>(reinterpret_cast<const f32x4*>(rec) + cell);
  }
  __device__ __forceinline__ uint32_t word(int64_t cell) const { return __float_as_uint(gp(rec)[4 * cell + 3]); }
  __device__ __forceinline__ void set_byte(int64_t cell, int c, uint32_t q) const {
    gp(rec)[4 * cell + 3] = __uint_as_float((word(cell) & ~(0xffu << (8 * c))) | (q << (8 * c)));
  }
  __device__ __forceinline__ double get(int64_t i) const {
    const int c = comp_of(i);
    const int64_t cell = i - c * cs;
    return comp_decode(gp(rec)[4 * cell + c], (word(cell) >> (8 * c)) & 0xffu);
  }
  __device__ __forceinline__ void put(int64_t i, double v) const {
    const int c = comp_of(i);
    const int64_t cell = i - c * cs;
    uint32_t q;
    gp(rec)[4 * cell + c] = comp_hi(v, q);
    set_byte(cell, c, q);
  }
  __device__ __forceinline__ void copy(int64_t dst, int64_t src) const {
    const int cd = comp_of(dst), cs_ = comp_of(src);
    const int64_t celld = dst - cd * cs, cells = src - cs_ * cs;
    gp(rec)[4 * celld + cd] = gp(rec)[4 * cells + cs_];
    set_byte(celld, cd, (word(cells) >> (8 * cs_)) & 0xffu);
  }
  // detectors sample the value rounded to float
  __device__ __forceinline__ float sample(int64_t i) const { return (float)get(i); }
  static constexpr uint32_t kCell = 16;
  using Own = f32x4;
  using Duo = f32x4;
  template <bool NT>
  __device__ __forceinline__ Own own(int64_t uni, uint32_t off) const {
    return ld_stream<NT>(split_ptr(reinterpret_cast<const f32x4*>(rec) + uni, off));
  }
  template <int C0, int C1>
  __device__ __forceinline__ Duo duo(int64_t uni, uint32_t off) const { return own<false>(uni, off); }
  template <int C>
  static __device__ __forceinline__ double value(const f32x4& r) { return decode_c<C>(r); }
  template <int C0, int C1, int C>
  static __device__ __forceinline__ double value(const f32x4& r) { return decode_c<C>(r); }
  template <bool NT>
  __device__ __forceinline__ void put_own(int64_t uni, uint32_t off, const double v[3]) const {
    f32x4 r;
    uint32_t w = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      uint32_t q;
      r[c] = comp_hi(v[c], q);
      w |= q << (8 * c);
    }
    r[3] = __uint_as_float(w);
    float* const at = split_ptr(rec + 4 * uni, off);
#pragma unroll
    for (int c = 0; c < 4; ++c) st_stream<NT>(at + c, (float)r[c]);
  }
  static __device__ __forceinline__ double rounded(double v) {
    uint32_t q;
    const float h = comp_hi(v, q);
    return comp_decode(h, q);
  }
  static __device__ __forceinline__ float sampled(double v) { return (float)rounded(v); }
  __device__ __forceinline__ Rec rec3(int64_t cell) const { return record<false>(cell); }
  template <int C>
  static __device__ __forceinline__ double decode_c(const f32x4& r) {
    return comp_decode(r[C], (__float_as_uint(r[3]) >> (8 * C)) & 0xffu);
  }
  static __device__ __forceinline__ void decode3(const f32x4& r, double v[3]) {
    const uint32_t w = __float_as_uint(r[3]);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = comp_decode(r[c], (w >> (8 * c)) & 0xffu);
  }
  template <int C>
  __device__ __forceinline__ double get_c(int64_t cell) const { return decode_c<C>(record<false>(cell)); }
  template <bool NT>
  __device__ __forceinline__ void get3_s(int64_t cell, double v[3]) const {
    decode3(record<NT>(cell), v);
  }
  template <bool NT>
  __device__ __forceinline__ void put3_s(int64_t cell, const double v[3]) const {
    f32x4 r;
    uint32_t w = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      uint32_t q;
      r[c] = comp_hi(v[c], q);
      w |= q << (8 * c);
    }
    r[3] = __uint_as_float(w);
#pragma unroll
    for (int c = 0; c < 4; ++c) st_stream<NT>(rec + 4 * cell + c, (float)r[c]);
  }
};

// --------------------------------------------------------------- materials
// Materials are read in two parts: key(i) -- what can be loaded a plane
// ahead (the palette index) -- and get3(key, i). The marching kernels load
// the next plane's key with the current plane, so a palette lookup does not
// wait for its index.
struct NoKey {};

template <typename S, typename R>
struct MatArray {
  using Key = NoKey;
  const S* p;  // (3, N)
  int64_t cs;
  template <bool NT>
  __device__ __forceinline__ Key key(int64_t) const { return {}; }
  template <bool NT>
  __device__ __forceinline__ void get3(Key, int64_t i, R m[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c] = (R)ld_stream<NT>(p + c * cs + i);
  }
  // as PlainField's: what is loaded for a cell, and its three values (kAhead:
  // what is loaded leads to them, and the marching kernels load it a plane ahead)
  static constexpr bool kAhead = false;
  static constexpr uint32_t kCell = sizeof(S);
  struct Own {
    S v[3];
  };
  template <bool NT>
  __device__ __forceinline__ Own own(int64_t uni, uint32_t off) const {
    return {{ld_stream<NT>(split_ptr(p + uni, off)), ld_stream<NT>(split_ptr(p + cs + uni, off)),
             ld_stream<NT>(split_ptr(p + 2 * cs + uni, off))}};
  }
  __device__ __forceinline__ void values(const Own& o, R m[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c] = (R)o.v[c];
  }
};

template <typename R>
struct MatPalette {
  using Key = int;
  const uint8_t* id;  // (N)
  const double* tab;  // (256, 3)
  template <bool NT>
  __device__ __forceinline__ Key key(int64_t i) const { return (int)ld_stream<NT>(id + i); }
  template <bool NT>
  __device__ __forceinline__ void get3(Key k, int64_t, R m[3]) const {
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c] = (R)gp(tab)[3 * k + c];
  }
  static constexpr bool kAhead = true;
  static constexpr uint32_t kCell = 1;
  using Own = uint8_t;
  template <bool NT>
  __device__ __forceinline__ Own own(int64_t uni, uint32_t off) const { return ld_stream<NT>(split_ptr(id + uni, off)); }
  __device__ __forceinline__ void values(const Own& o, R m[3]) const {
    const uint32_t at = 3 * sizeof(double) * o;
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c] = (R)ld_stream<false>(split_ptr(tab + c, at));
  }
};

// ------------------------------------------------------------ CPML helpers
// The six one-sided differences of one cell, named after the curl terms:
// zy = difference of component z along y, etc. (grid.py:29-76).
template <typename T>
struct Diffs {
  T zy, yz, xz, zx, yx, xy;
};

// One CPML face at one cell (boundaries.py:409-487). A face normal to axis
// `ax` keeps psi for the two field components other than ax, C0 < C1
// (C0 = ax==0 ? 1 : 0, C1 = ax==2 ? 1 : 2). psi_q <- psi_q*b, plus
// (difference along ax of the other field's component 3-ax-C_q) * c where
// the slab index allows it (E side: l >= 1; H side: l <= t-2). The
// convolution term of C_q is +psi when ax follows C_q cyclically, -psi
// otherwise, so E[C0] gets +-(S inv)*psi_0 and E[C1] +-(S inv)*psi_1 (H with
// the opposite sign). Everything that depends on the axis is chosen with
// selects rather than branches, so no address is formed from values merged
// across control flow. Returns without touching v when the cell is outside
// the face's slab.
template <bool IS_E, typename T>
__device__ __forceinline__ void pml_face(const FaceDev& fd, const Dims& d, int i, int j, int k, T zx, T yx, T zy,
                                         T xy, T yz, T xz, T k0, T k1, T k2, T& v0, T& v1, T& v2) {
  const int ax = fd.axis;
  const int g = ax == 0 ? i : (ax == 1 ? j : k);
  const int n = ax == 0 ? d.nx : (ax == 1 ? d.ny : d.nz);
  const int l = fd.high ? g - (n - fd.t) : g;
  if (l < 0 || l >= fd.t) return;
  // slab: the grid with the normal axis shortened to t
  const int64_t sny = ax == 1 ? fd.t : d.ny;
  const int64_t snz = ax == 2 ? fd.t : d.nz;
  const int64_t li = ax == 0 ? l : i, lj = ax == 1 ? l : j, lk = ax == 2 ? l : k;
  const int64_t off = (li * sny + lj) * snz + lk;
  T* const psi = reinterpret_cast<T*>(IS_E ? fd.psiE : fd.psiH);
  const gptr<const double> bt = gp(IS_E ? fd.bE : fd.bH);
  const gptr<const double> ct = gp(IS_E ? fd.cE : fd.cH);
  const T b = (T)bt[l], c = (T)ct[l];
  const T d0 = ax == 0 ? zx : (ax == 1 ? zy : yz);
  const T d1 = ax == 0 ? yx : (ax == 1 ? xy : xz);
  T p0 = ld_stream<false>(psi + off) * b;
  T p1 = ld_stream<false>(psi + fd.slab + off) * b;
  if (IS_E ? (l >= 1) : (l <= fd.t - 2)) {
    p0 = p0 + d0 * c;
    p1 = p1 + d1 * c;
  }
  st_stream<false>(psi + off, p0);
  st_stream<false>(psi + fd.slab + off, p1);
  const T r0 = (ax == 0 ? k1 : k0) * p0;
  const T r1 = (ax == 2 ? k1 : k2) * p1;
  T n0, n1, n2;
  if (IS_E) {
    // ax 0: E1 -= r0, E2 += r1; ax 1: E0 += r0, E2 -= r1; ax 2: E0 -= r0, E1 += r1
    n0 = ax == 1 ? v0 + r0 : (ax == 2 ? v0 - r0 : v0);
    n1 = ax == 0 ? v1 - r0 : (ax == 2 ? v1 + r1 : v1);
    n2 = ax == 0 ? v2 + r1 : (ax == 1 ? v2 - r1 : v2);
  } else {
    n0 = ax == 1 ? v0 - r0 : (ax == 2 ? v0 + r0 : v0);
    n1 = ax == 0 ? v1 + r0 : (ax == 2 ? v1 - r1 : v1);
    n2 = ax == 0 ? v2 - r1 : (ax == 1 ? v2 + r1 : v2);
  }
  v0 = n0;
  v1 = n1;
  v2 = n2;
}

// All faces in `faces` that contain cell (i,j,k), in registration order.
template <bool IS_E, typename T>
__device__ __forceinline__ void pml_cell(const FaceDev* __restrict__ faces, int nfaces, const Dims& d, int i, int j,
                                         int k, const Diffs<T>& df, const T kc[3], T v[3]) {
  for (int fi = 0; fi < nfaces; ++fi)
    pml_face<IS_E>(faces[fi], d, i, j, k, df.zx, df.yx, df.zy, df.xy, df.yz, df.xz, kc[0], kc[1], kc[2], v[0], v[1],
                   v[2]);
}

// The face of one side of the grid as the main kernels read it: its two psi
// components and its profiles (a table of 6, [axis][low/high]).
struct Side {
  void* psiE[2];
  void* psiH[2];
  const double* bE;
  const double* cE;
  const double* bH;
  const double* cH;
};

// Two psi values of one cell and face, `off` bytes into their arrays.
template <typename T>
struct Psi {
  T p0, p1;
  __device__ __forceinline__ void load(const void* a0, const void* a1, uint32_t off) {
    p0 = ld_stream<false>(split_ptr(reinterpret_cast<const T*>(a0), off));
    p1 = ld_stream<false>(split_ptr(reinterpret_cast<const T*>(a1), off));
  }
  __device__ __forceinline__ void store(void* a0, void* a1, uint32_t off) const {
    st_stream<false>(split_ptr(reinterpret_cast<T*>(a0), off), p0);
    st_stream<false>(split_ptr(reinterpret_cast<T*>(a1), off), p1);
  }
  // psi <- psi b, plus (difference) c where the slab has both of its cells
  __device__ __forceinline__ void advance(T b, T c, bool inner, T d0, T d1) {
    p0 = p0 * b;
    p1 = p1 * b;
    if (inner) {
      p0 = p0 + d0 * c;
      p1 = p1 + d1 * c;
    }
  }
};

// The CPML of one cell column of a tile, for plans with at most one face a side
// whose slabs do not overlap (a cell is then in one slab per axis at most).
// Which slabs of the y and z axes the column is in and its place there do not
// change from plane to plane and are found once; every psi value and
// coefficient of a plane is loaded with the plane's fields, before any of them
// is waited for; and a wavefront that meets no slab does nothing for them.
template <bool IS_E, typename T>
struct TilePml {
  enum : uint32_t { kLoY = 1, kHiY = 2, kLoZ = 4, kHiZ = 8, kInY = 16, kInZ = 32 };
  cptr<Side> sides;
  uint32_t flags = 0;  // the column's slabs; kIn*: the slab has both cells of the difference
  uint32_t qy = 0, qz = 0, ystep = 0, zstep = 0;  // byte offsets in the psi arrays, and a plane further
  uint32_t ly = 0, lz = 0;  // byte offsets in the profiles
  bool any_y, any_z;  // some column of the wavefront is in a y (z) slab
  double by, cy, bz, cz;
  Psi<T> px, py, pz;
  int xs, xl;  // the plane's x slab (side, index), -1: none
  uint32_t qx;

  template <class A>
  __device__ __forceinline__ void init(const A& a, int i, int j, int k) {
    const Dims& d = a.d;
    sides = cp(a.sides);
    const auto inner = [](int l, int t) { return IS_E ? l >= 1 : l <= t - 2; };
    if (j < a.t[2] || j >= d.ny - a.t[3]) {
      const bool lo = j < a.t[2];
      const int t = lo ? a.t[2] : a.t[3], l = lo ? j : j - (d.ny - t);
      ystep = (uint32_t)(t * d.nz) * (uint32_t)sizeof(T);
      qy = (uint32_t)i * ystep + (uint32_t)(l * d.nz + k) * (uint32_t)sizeof(T);
      flags |= (lo ? kLoY : kHiY) | (inner(l, t) ? kInY : 0);
      ly = (uint32_t)l * (uint32_t)sizeof(double);
    }
    if (k < a.t[4] || k >= d.nz - a.t[5]) {
      const bool lo = k < a.t[4];
      const int t = lo ? a.t[4] : a.t[5], l = lo ? k : k - (d.nz - t);
      zstep = (uint32_t)(t * d.ny) * (uint32_t)sizeof(T);
      qz = (uint32_t)i * zstep + (uint32_t)(j * t + l) * (uint32_t)sizeof(T);
      flags |= (lo ? kLoZ : kHiZ) | (inner(l, t) ? kInZ : 0);
      lz = (uint32_t)l * (uint32_t)sizeof(double);
    }
    any_y = wave_any(flags & (kLoY | kHiY));
    any_z = wave_any(flags & (kLoZ | kHiZ));
  }
  __device__ __forceinline__ void fetch(int s, uint32_t& q, Psi<T>& p) const {
    opaque(q);
    const cptr<Side> sd = sides + s;
    if (IS_E) p.load(sd->psiE[0], sd->psiE[1], q);
    else p.load(sd->psiH[0], sd->psiH[1], q);
  }
  __device__ __forceinline__ void fetch(int s, uint32_t& q, uint32_t& l, Psi<T>& p, double& b, double& c) const {
    fetch(s, q, p);
    opaque(l);
    const cptr<Side> sd = sides + s;
    b = ld_stream<false>(split_ptr(IS_E ? sd->bE : sd->bH, l));
    c = ld_stream<false>(split_ptr(IS_E ? sd->cE : sd->cH, l));
  }
  __device__ __forceinline__ void keep(int s, uint32_t& q, const Psi<T>& p) const {
    opaque(q);
    const cptr<Side> sd = sides + s;
    if (IS_E) p.store(sd->psiE[0], sd->psiE[1], q);
    else p.store(sd->psiH[0], sd->psiH[1], q);
  }
  // psi of plane i
  template <class A>
  __device__ __forceinline__ void load(const A& a, int i, uint32_t pc) {
    opaque(flags);
    opaque_table(sides);
    xs = i < a.t[0] ? 0 : (i >= a.d.nx - a.t[1] ? 1 : -1);
    if (xs >= 0) {
      xl = xs ? i - (a.d.nx - a.t[1]) : i;
      qx = ((uint32_t)xl * (uint32_t)(a.d.ny * a.d.nz) + pc) * (uint32_t)sizeof(T);
      fetch(xs, qx, px);
    }
    if (any_y) {
      if (flags & kLoY) fetch(2, qy, ly, py, by, cy);
      if (flags & kHiY) fetch(3, qy, ly, py, by, cy);
    }
    if (any_z) {
      if (flags & kLoZ) fetch(4, qz, lz, pz, bz, cz);
      if (flags & kHiZ) fetch(5, qz, lz, pz, bz, cz);
    }
  }
  // to the next plane of an E (up) or H (down) march
  __device__ __forceinline__ void next_plane() {
    qy = IS_E ? qy + ystep : qy - ystep;
    qz = IS_E ? qz + zstep : qz - zstep;
  }
  // One step of the recursions and their terms in v (pml_face, above), the
  // faces of a cell in the plan's order.
  template <class A>
  __device__ __forceinline__ void apply(const A& a, T zx, T yx, T zy, T xy, T yz, T xz, const T kc[3], T v[3]) {
    if (!any_y && !any_z && xs < 0) return;
#pragma nounroll
    for (int n = 0; n < 3; ++n) {
      const int ax = (a.order >> (2 * n)) & 3;
      if (ax == 0 && xs >= 0) {
        const cptr<Side> sd = sides + xs;
        const T b = (T)cp(IS_E ? sd->bE : sd->bH)[xl], c = (T)cp(IS_E ? sd->cE : sd->cH)[xl];
        px.advance(b, c, IS_E ? xl >= 1 : xl <= a.t[xs] - 2, zx, yx);
        keep(xs, qx, px);
        const T r0 = kc[1] * px.p0, r1 = kc[2] * px.p1;
        v[1] = IS_E ? v[1] - r0 : v[1] + r0;
        v[2] = IS_E ? v[2] + r1 : v[2] - r1;
      } else if (ax == 1 && any_y) {
        if (flags & (kLoY | kHiY)) {
          py.advance((T)by, (T)cy, flags & kInY, zy, xy);
          if (flags & kLoY) keep(2, qy, py);
          if (flags & kHiY) keep(3, qy, py);
          const T r0 = kc[0] * py.p0, r1 = kc[2] * py.p1;
          v[0] = IS_E ? v[0] + r0 : v[0] - r0;
          v[2] = IS_E ? v[2] - r1 : v[2] + r1;
        }
      } else if (ax == 2 && any_z) {
        if (flags & (kLoZ | kHiZ)) {
          pz.advance((T)bz, (T)cz, flags & kInZ, yz, xz);
          if (flags & kLoZ) keep(4, qz, pz);
          if (flags & kHiZ) keep(5, qz, pz);
          const T r0 = kc[0] * pz.p0, r1 = kc[1] * pz.p1;
          v[0] = IS_E ? v[0] - r0 : v[0] + r0;
          v[1] = IS_E ? v[1] + r1 : v[1] - r1;
        }
      }
    }
  }
};

// E factor (1 - f) / (1 + f) of an absorbing object (objects.py:215). With
// complex fields the reference divides in the dtype of f: complex (numpy's
// division) when the object's permittivity is complex, real when it is real
// (its arrays stay real on complex fields), and the real quotient then
// multiplies E as (r, 0).
template <typename T>
__device__ __forceinline__ T absorb_ratio(T f, int) {
  return (T(1) - f) / (T(1) + f);
}
template <typename S>
__device__ __forceinline__ cplx<S> absorb_ratio(cplx<S> f, int real) {
  if (real) return cplx<S>((S(1) - f.re) / (S(1) + f.re), S(0));
  return (cplx<S>(1) - f) / (cplx<S>(1) + f);
}

// Row of the anisotropic 3x3 product inv @ curl (objects.py:262-269, numpy's
// einsum "ijk,ikl->ijl"). Real: the association (m0 c0 + m2 c2) + m1 c1
// numpy's einsum uses for this 3-term contraction. Complex: einsum's complex
// loop, products without fused multiply-adds (re = ar br - ai bi,
// im = ar bi + ai br) summed in order; a real inverse on complex fields is
// promoted to (x, 0) by einsum, which the same loop covers.
template <typename T>
__device__ __forceinline__ T aniso_row(T m0, T m1, T m2, T c0, T c1, T c2) {
  return (m0 * c0 + m2 * c2) + m1 * c1;
}
template <typename S>
__device__ __forceinline__ cplx<S> einsum_product(cplx<S> a, cplx<S> b) {
  return cplx<S>(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
template <typename S>
__device__ __forceinline__ cplx<S> aniso_row(cplx<S> m0, cplx<S> m1, cplx<S> m2, cplx<S> c0, cplx<S> c1,
                                             cplx<S> c2) {
  return (einsum_product(m0, c0) + einsum_product(m1, c1)) + einsum_product(m2, c2);
}

// Object updates of one cell, registration order (objects.py:118-269); the
// object arrays are stored as O and computed in T.
template <typename T, typename O>
__device__ __forceinline__ void objects_update_E(const ObjDev* __restrict__ objs, int nobjs, T sc, int i, int j,
                                                 int k, const T curl[3], T e[3]) {
  for (int o = 0; o < nobjs; ++o) {
    const ObjDev& ob = objs[o];
    if (i < ob.x0 || i >= ob.x1 || j < ob.y0 || j >= ob.y1 || k < ob.z0 || k >= ob.z1) continue;
    const int64_t lo = ((int64_t)(i - ob.x0) * (ob.y1 - ob.y0) + (j - ob.y0)) * (ob.z1 - ob.z0) + (k - ob.z0);
    const O* const inv = reinterpret_cast<const O*>(ob.inv);
    auto at = [](const O* q, int64_t x) { return (T)ld_stream<false>(q + x); };
    if (ob.kind == FDTD_OBJ_PLAIN) {
#pragma unroll
      for (int c = 0; c < 3; ++c) e[c] = e[c] + (sc * at(inv, lo * 3 + c)) * curl[c];
    } else if (ob.kind == FDTD_OBJ_ABSORBING) {
      const O* const fa = reinterpret_cast<const O*>(ob.absorb);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T f = at(fa, lo * 3 + c);
        e[c] = e[c] * absorb_ratio(f, ob.real);
        e[c] = e[c] + ((sc * at(inv, lo * 3 + c)) * curl[c]) / (T(1) + f);
      }
    } else {
      const O* const m = inv + lo * 9;
      T v[3];
#pragma unroll
      for (int r = 0; r < 3; ++r)
        v[r] = aniso_row(at(m, 3 * r), at(m, 3 * r + 1), at(m, 3 * r + 2), curl[0], curl[1], curl[2]);
#pragma unroll
      for (int r = 0; r < 3; ++r) e[r] = e[r] + sc * v[r];
    }
  }
}

// Whether a column (j, k) of the wavefront has, in x plane i, a cell inside an
// object.
__device__ __forceinline__ bool meets_objects(const ObjDev* objs, int nobjs, int i, int j, int k) {
  for (int o = 0; o < nobjs; ++o) {
    const cptr<ObjDev> ob = cp(objs) + o;
    if (i < ob->x0 || i >= ob->x1) continue;
    if (wave_any(j >= ob->y0 && j < ob->y1 && k >= ob->z0 && k < ob->z1)) return true;
  }
  return false;
}

// Division by a number fixed per launch, as a product and a shift (exact for
// numerators below 2^31; Granlund and Montgomery 1994). A division by a
// kernel argument is ~25 instructions, one of 64 bits ~100, in every wavefront's
// first instructions. Two to seven a wavefront replaced: 24 float32 grids of
// 64-160 cells an axis in one batch 771 -> 762 us a step, a 60x52x44 float64
// whole step 14.3 -> 14.1 us, 256^3 within 0.3 %.
struct Divide {
  uint32_t d, mul;
  int32_t shift;
  __host__ __device__ __forceinline__ uint32_t of(uint32_t n) const { return (uint32_t)(((uint64_t)n * mul) >> shift); }
};
inline Divide make_divide(uint32_t d) {
  int l = 0;
  while (((uint64_t)1 << l) < d) ++l;
  return {d, (uint32_t)((((uint64_t)1 << (31 + l)) / d) + 1), 31 + l};
}

// Logical tile of hardware workgroup w: workgroups are dealt round-robin to
// the 8 XCDs (each with its own L2), so consecutive logical tiles -- which
// share halo planes -- are given to the same XCD.
__device__ __forceinline__ unsigned xcd_tile(unsigned w, unsigned nb) {
  const unsigned per = nb / 8, rem = nb % 8, x = w % 8, idx = w / 8;
  return x < rem ? x * (per + 1) + idx : rem * (per + 1) + (x - rem) * per + idx;
}

// Tile of workgroup w in the single-grid kernels of large grids, or -1 for
// an idle workgroup. The x-chunks (`per_chunk` tiles each) are dealt to the
// XCDs cyclically -- chunk c to XCD c mod 8 -- and each XCD walks the tiles of
// its chunks in order, so at any moment the 8 XCDs work on 8 neighbouring
// chunks: the CPML slabs at both x ends, which cost more per cell, are shared
// by all XCDs instead of falling to the first and last (workgroups are
// dispatched in order, so one slow XCD holds back the others). The price is
// the x-halo plane of each chunk, read by another XCD; grids small enough to
// live in the L2s and the memory-side cache keep the contiguous dealing of
// xcd_tile. The grid has 8 * ceil(nchunks / 8) * per_chunk workgroups.
__device__ __forceinline__ int64_t xcd_chunk_tile(unsigned w, const Divide& per_chunk, unsigned nchunks) {
  const unsigned x = w % 8, k = w / 8, round = per_chunk.of(k);
  const unsigned tx = round * 8 + x;
  return tx < nchunks ? (int64_t)tx * per_chunk.d + (k - round * per_chunk.d) : -1;
}

// Half-open box of cells {x0, x1, y0, y1, z0, z1}; its cells are numbered
// z fastest.
struct Box {
  int32_t x0, x1, y0, y1, z0, z1;
};

__host__ __device__ __forceinline__ int64_t box_cells(const Box& b) {
  return (int64_t)(b.x1 - b.x0) * (b.y1 - b.y0) * (b.z1 - b.z0);
}

// index of cell (i,j,k) inside box b, or -1
__device__ __forceinline__ int64_t box_index(const Box& b, int i, int j, int k) {
  if (i < b.x0 || i >= b.x1 || j < b.y0 || j >= b.y1 || k < b.z0 || k >= b.z1) return -1;
  return ((int64_t)(i - b.x0) * (b.y1 - b.y0) + (j - b.y0)) * (b.z1 - b.z0) + (k - b.z0);
}

// grid cell of box index p
__device__ __forceinline__ int64_t box_cell(const Box& b, const Dims& d, int64_t p) {
  const int64_t nz = b.z1 - b.z0, ny = b.y1 - b.y0;
  const int64_t k = b.z0 + p % nz, j = b.y0 + (p / nz) % ny, i = b.x0 + p / (nz * ny);
  return cell_of(d, i, j, k);
}

// ------------------------------------------------------------ main kernels
constexpr int FOLDED_POINTS = 4;

template <class FS, class MS>
struct MainArgs {
  using R = typename FS::R;
  Dims d;
  R sc;
  FS F;  // field updated in this half step (E or H)
  FS G;  // field whose curl drives it (H or E)
  MS M;  // inv_eps or inv_mu
  const FaceDev* faces;
  int32_t nfaces;
  // at most one face a side: the sides, their thicknesses (0: no face), and
  // the order of a cell's faces (axes, two bits each)
  const Side* sides;
  int32_t t[6];
  int32_t order;
  const ObjDev* objs;
  int32_t nobjs;
  int32_t bz_shift;  // block extent along z is 1 << bz_shift
  int32_t cx;        // planes per workgroup along x
  int32_t by;        // block extent along y (threads per block = bz * by)
  int32_t cyclic;    // single-grid launch: x-chunks dealt cyclically to the XCDs
  int32_t flat;      // 0: tiles of bz z-cells by `by` z-rows; else tiles of `flat`
                     // (= threads per block) consecutive cells of the (y, z) plane
  Divide per;        // tiles per x-chunk
  Divide row;        // flat: z-cells of a row; else z tiles of a row of tiles
  uint32_t nchunks;  // x-chunks
  // point sources folded into the E kernel (no periodic stage, no detector):
  // their cells, in registration order, and the waveform table
  int32_t npts;
  int64_t pt_cell[FOLDED_POINTS];
  int32_t pt_plane[FOLDED_POINTS], pt_at[FOLDED_POINTS];  // x plane and place in it
  const double* wave;  // row s = source s
  int64_t wave_cap;
  int64_t q;
  // differentiation record (E kernel, recording variant): the curl of this
  // half step inside box `rb`, (3, cells of rb)
  R* rec;
  Box rb;
  // and the updated field inside box `rbE` (null: left to the tail)
  R* rec_E;
  Box rbE;
  // bytes of the members that follow from others: the CPML by side, the folded
  // points by plane, the divisors
  static constexpr size_t kDerived = 128;
};

// Tiles of one x-chunk: row tiles (bz z-cells by `by` z-rows) or flat tiles
// (`flat` consecutive cells of the (y, z) plane, wrapping from the end of one
// z-row to the start of the next, so that only the plane's last tile has
// idle lanes whatever nz is).
__host__ __device__ __forceinline__ unsigned plane_tiles(const Dims& d, int bz_shift, int by, int flat) {
  if (flat) return (unsigned)(((int64_t)d.ny * d.nz + flat - 1) / flat);
  const int bz = 1 << bz_shift;
  return (unsigned)(((d.nz + bz - 1) / bz) * ((d.ny + by - 1) / by));
}

// This thread's column (j, k) in tile `tile`, the tile's x range [i0, i1),
// and whether the column is inside the grid: threads past the edge take the
// nearest cell (so that their loads stay in bounds) and store nothing.
template <class A>
__device__ __forceinline__ void tile_column(const A& a, unsigned tile, int& j, int& k, int& i0, int& i1, bool& act) {
  const Dims& d = a.d;
  const uint32_t tx = a.per.of(tile), t = tile - tx * a.per.d;
  if (a.flat) {
    const int plane = d.ny * d.nz;  // the host uses flat tiles for planes below 2^31 cells
    const uint32_t p0 = t * (uint32_t)a.flat + threadIdx.x;
    act = p0 < (uint32_t)plane;
    const uint32_t p = min(p0, (uint32_t)plane - 1);
    j = (int)a.row.of(p);
    k = (int)p - j * d.nz;
  } else {
    const int bzs = a.bz_shift, bz = 1 << bzs, by = a.by;
    const uint32_t ty = a.row.of(t), tz = t - ty * a.row.d;
    const int k0 = (int)tz * bz + (int)(threadIdx.x & (bz - 1)), j0 = (int)ty * by + (int)(threadIdx.x >> bzs);
    act = k0 < d.nz && j0 < d.ny;
    k = min(k0, d.nz - 1);
    j = min(j0, d.ny - 1);
  }
  i0 = (int)tx * a.cx;
  i1 = min(i0 + a.cx, d.nx);
}

// Main E kernel, general form: any faces (several a side, overlapping slabs,
// an order that differs between sides: the face table is walked per cell) and
// planes past the 32-bit offsets of the form below. A workgroup owns a (y, z) tile (tile_column) and marches
// along x over a chunk of `cx` planes: the x-neighbours come from registers
// of the previous plane, the y- and z-neighbours from cache (the rows were
// just streamed in by this or the neighbouring wavefront). Every load of a
// plane is issued unconditionally and at once, so a plane costs one memory
// round trip: threads past the grid's edge read the nearest cell and store
// nothing, and at the low edges the neighbour offset is 0 (the difference is
// dropped). ONLY: the wavefronts and planes that meet an object, which the
// main form leaves (below).
template <class FS, class MS, typename O, bool OBJS, bool NT, bool REC = false, bool ONLY = false>
__device__ __forceinline__ void any_E_tile(const MainArgs<FS, MS>& __restrict__ a, unsigned tile, int64_t q) {
  using T = typename FS::R;
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, tile, j, k, i0, i1, act);
  const int64_t sy = d.nz, sx = d.px;
  const int64_t zm = k > 0 ? 1 : 0, ym = j > 0 ? sy : 0;
  const T zero = T(0);
  int64_t cell = (int64_t)i0 * sx + (int64_t)j * sy + k;
  T hz_prev = zero, hy_prev = zero;
  typename FS::Rec hrec{};  // records: H of plane i-1 as loaded
  if (i0 > 0) {
    if constexpr (FS::kRecords) {
      hrec = a.G.rec3(cell - sx);
    } else {
      hz_prev = a.G.template get_c<2>(cell - sx);
      hy_prev = a.G.template get_c<1>(cell - sx);
    }
  }
  typename MS::Key key = a.M.template key<NT>(cell);
  bool skipped = false;
  for (int i = i0; i < i1; ++i, cell += sx) {
    if constexpr (ONLY) {
      if (!meets_objects(a.objs, a.nobjs, i, j, k)) {
        skipped = true;
        continue;
      }
      if (skipped) {  // nothing was carried from the plane before
        skipped = false;
        if constexpr (FS::kRecords) {
          hrec = a.G.rec3(cell - sx);
        } else {
          hz_prev = a.G.template get_c<2>(cell - sx);
          hy_prev = a.G.template get_c<1>(cell - sx);
        }
        key = a.M.template key<NT>(cell);
      }
    }
    T hv[3], m[3], e[3];
    const typename MS::Key kc_ = key;
    if (i + 1 < i1) key = a.M.template key<NT>(cell + sx);  // the next plane's, loaded with this one
    T hy_km, hx_km, hz_jm, hx_jm;
    if constexpr (FS::kRecords) {
      const typename FS::Rec hr = a.G.rec3(cell);
      FS::decode3(hr, hv);
      const f32x4 zr = a.G.rec3(cell - zm), yr = a.G.rec3(cell - ym);
      hx_km = FS::template decode_c<0>(zr), hy_km = FS::template decode_c<1>(zr);
      hx_jm = FS::template decode_c<0>(yr), hz_jm = FS::template decode_c<2>(yr);
      hz_prev = FS::template decode_c<2>(hrec);
      hy_prev = FS::template decode_c<1>(hrec);
      hrec = hr;
    } else {
      a.G.template get3_s<false>(cell, hv);
      hy_km = a.G.template get_c<1>(cell - zm), hx_km = a.G.template get_c<0>(cell - zm);
      hz_jm = a.G.template get_c<2>(cell - ym), hx_jm = a.G.template get_c<0>(cell - ym);
    }
    a.M.template get3<NT>(kc_, cell, m);
    a.F.template get3_s<NT>(cell, e);
    const T hx = hv[0], hy = hv[1], hz = hv[2];
    // backward differences; an absent one contributes nothing (grid.py:67-74)
    Diffs<T> df;
    df.zy = j > 0 ? hz - hz_jm : zero;
    df.yz = k > 0 ? hy - hy_km : zero;
    df.xz = k > 0 ? hx - hx_km : zero;
    df.zx = i > 0 ? hz - hz_prev : zero;
    df.yx = i > 0 ? hy - hy_prev : zero;
    df.xy = j > 0 ? hx - hx_jm : zero;
    T curl[3];
    curl[0] = (zero + df.zy) - df.yz;
    curl[1] = (zero + df.xz) - df.zx;
    curl[2] = (zero + df.yx) - df.xy;
    T kc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      kc[c] = a.sc * m[c];
      e[c] = e[c] + kc[c] * curl[c];
    }
    if (act) {
      if (REC) {
        const int64_t r = box_index(a.rb, i, j, k);
        if (r >= 0) {
          const int64_t nr = box_cells(a.rb);
#pragma unroll
          for (int c = 0; c < 3; ++c) a.rec[c * nr + r] = curl[c];
        }
      }
      if (OBJS) objects_update_E<T, O>(a.objs, a.nobjs, a.sc, i, j, k, curl, e);
      if (a.nfaces) pml_cell<true>(a.faces, a.nfaces, d, i, j, k, df, kc, e);
      for (int s = 0; s < a.npts; ++s)  // sources.py:109, registration order
        if (a.pt_cell[s] == cell) e[2] = e[2] + (T)gp(a.wave)[s * a.wave_cap + q];
      if (REC && a.rec_E) {
        const int64_t r = box_index(a.rbE, i, j, k);
        if (r >= 0) {
          const int64_t nr = box_cells(a.rbE);
#pragma unroll
          for (int c = 0; c < 3; ++c) a.rec_E[c * nr + r] = FS::rounded(e[c]);
        }
      }
      a.F.template put3_s<NT>(cell, e);
    }
    if constexpr (!FS::kRecords) {
      hz_prev = hz;
      hy_prev = hy;
    }
  }
}

// Main E kernel: the form nearly every plan takes. As the general form, with
// CPML per axis (TilePml: psi and coefficients loaded with the plane's fields)
// and every access a scalar base plus a 32-bit offset that steps by a plane,
// where the general form walks the face table cell by cell, each face a chain
// of table, psi and coefficient loads, and forms 64-bit addresses. In float32
// the kernels are bound by issue and by those chains rather than by bandwidth:
// general -> main form 128^3 30.1 -> 24.7 us a launch, 24 grids of 64-160 cells
// edge 0.887 -> 0.775 ms/step, 256^3 0.317 -> 0.293 ms/step; float64 at 256^3 is at
// the fabric's rate either way (0.633 -> 0.626).
// Nothing is guarded against work-items past the plane's edge: a wavefront of
// them ends at once, and the ones beside the plane's last cell do that cell's
// work, in lockstep with its own work-item, and store the same values (a
// guarded block leaves loads unconsumed when it is skipped, and the wait for
// them then stands between a plane's first loads and its others).
// OBJS: wavefronts that meet an object in a plane leave it to k_object_E
// (objects in this kernel would cost every cell the registers of their 3x3
// products: spilling, it took 1.6x the general form's time in float64).
template <class FS, class MS, bool OBJS, bool NT>
__device__ __forceinline__ void main_E_tile(const MainArgs<FS, MS>& __restrict__ a, unsigned tile, int64_t q) {
  using T = typename FS::R;
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, tile, j, k, i0, i1, act);
  if (!wave_any(act)) return;
  const int ib = max(i0 - 1, 0);  // the offsets count from here
  const int64_t base = (int64_t)ib * d.px;
  const uint32_t pc = (uint32_t)(j * d.nz + k), at = (uint32_t)(i0 - ib) * (uint32_t)d.px + pc;
  const uint32_t fstep = (uint32_t)d.px * FS::kCell, mstep = (uint32_t)d.px * MS::kCell;
  uint32_t fo = at * FS::kCell, mo = at * MS::kCell;
  const uint32_t dk = k > 0 ? FS::kCell : 0, dj = j > 0 ? (uint32_t)d.nz * FS::kCell : 0;
  TilePml<true, T> pml;
  pml.init(a, i0, j, k);
  const T zero = T(0);
  typename FS::Own hprev;  // H of plane i-1
  typename MS::Own ahead{};
  constexpr bool kAhead = MS::kAhead && !OBJS;
  if constexpr (kAhead) ahead = a.M.template own<NT>(base, mo);
  bool carried = false;  // hprev is plane i-1's
  for (int i = i0; i < i1; ++i, fo += fstep, mo += mstep, pml.next_plane()) {
    if constexpr (OBJS) {
      if (meets_objects(a.objs, a.nobjs, i, j, k)) {
        carried = false;
        continue;
      }
    }
    opaque(fo);
    if constexpr (MS::kCell == FS::kCell) mo = fo;
    // every load of the plane at once (the first plane's hprev among them:
    // loaded ahead of the loop, it would be waited for before the others)
    if (!carried) hprev = a.G.template own<false>(base, i > 0 ? fo - fstep : fo);
    carried = true;
    const typename FS::Own hown = a.G.template own<false>(base, fo);
    const typename FS::Duo hk = a.G.template duo<0, 1>(base, fo - dk), hj = a.G.template duo<0, 2>(base, fo - dj);
    typename MS::Own mat;
    if constexpr (kAhead) {
      mat = ahead;
      if (i + 1 < i1) ahead = a.M.template own<NT>(base, mo + mstep);
    } else {
      mat = a.M.template own<NT>(base, mo);
    }
    const typename FS::Own eown = a.F.template own<NT>(base, fo);
    pml.load(a, i, pc);
    const T h0 = FS::template value<0>(hown), h1 = FS::template value<1>(hown), h2 = FS::template value<2>(hown);
    // backward differences; an absent one contributes nothing (grid.py:67-74)
    Diffs<T> df;
    df.zy = dj ? h2 - FS::template value<0, 2, 2>(hj) : zero;
    df.yz = dk ? h1 - FS::template value<0, 1, 1>(hk) : zero;
    df.xz = dk ? h0 - FS::template value<0, 1, 0>(hk) : zero;
    df.zx = i > 0 ? h2 - FS::template value<2>(hprev) : zero;
    df.yx = i > 0 ? h1 - FS::template value<1>(hprev) : zero;
    df.xy = dj ? h0 - FS::template value<0, 2, 0>(hj) : zero;
    hprev = hown;
    T e[3] = {FS::template value<0>(eown), FS::template value<1>(eown), FS::template value<2>(eown)};
    T m[3], curl[3], kc[3];
    a.M.values(mat, m);
    curl[0] = (zero + df.zy) - df.yz;
    curl[1] = (zero + df.xz) - df.zx;
    curl[2] = (zero + df.yx) - df.xy;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      kc[c] = a.sc * m[c];
      e[c] = e[c] + kc[c] * curl[c];
    }
    pml.apply(a, df.zx, df.yx, df.zy, df.xy, df.yz, df.xz, kc, e);
    for (int s = 0; s < a.npts; ++s)  // sources.py:109, registration order
      if (a.pt_plane[s] == i && (uint32_t)a.pt_at[s] == pc) e[2] = e[2] + (T)gp(a.wave)[s * a.wave_cap + q];
    opaque(fo);
    a.F.template put_own<NT>(base, fo, e);
  }
}

template <class FS, class MS>
__device__ __forceinline__ int64_t launch_tile(const MainArgs<FS, MS>& a, unsigned& ntiles) {
  ntiles = a.per.d * a.nchunks;
  return a.cyclic ? xcd_chunk_tile(blockIdx.x, a.per, a.nchunks) : (int64_t)xcd_tile(blockIdx.x, gridDim.x);
}

// Occupancy floor of the E kernels: the general form otherwise takes ~118
// VGPRs (4 waves per SIMD) for the anisotropic 3x3 path. Under a floor of 6
// the double-precision ones fit in ~76 VGPRs without spilling, the float32
// ones under a floor of 8 in ~46 (a floor of 8 makes the double ones spill);
// complex128 values need twice the registers and keep a floor of 4. The
// compensated kernels without objects fit 8 waves in 62 VGPRs (66 and 7
// waves unbounded; 0.6 % faster per step at 256^3). The main forms fit under
// the same floors.
template <class FS, bool OBJS = true>
struct EWaves {
  static constexpr int bytes = sizeof(typename FS::R);
  static constexpr int value = FS::kRecords && !OBJS ? 8 : (bytes == 4 ? 8 : (bytes == 8 ? 6 : 4));
};

template <class FS, class MS, bool OBJS, bool NT>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(EWaves<FS>::value)))
k_main_E(MainArgs<FS, MS> a) {
  unsigned n;
  const int64_t t = launch_tile(a, n);
  if (t >= 0) main_E_tile<FS, MS, OBJS, NT>(a, (unsigned)t, a.q);
}

template <class FS, class MS, typename O, bool OBJS, bool REC>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(EWaves<FS, OBJS>::value)))
k_any_E(MainArgs<FS, MS> a) {
  unsigned n;
  const int64_t t = launch_tile(a, n);
  if (t >= 0) any_E_tile<FS, MS, O, OBJS, true, REC>(a, (unsigned)t, a.q);
}

// The tiles that meet an object, one workgroup each.
template <class FS, class MS, typename O>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(EWaves<FS>::value)))
k_object_E(MainArgs<FS, MS> a, const uint32_t* tiles) {
  any_E_tile<FS, MS, O, true, true, false, true>(a, cp(tiles)[blockIdx.x], a.q);
}

// Main H kernel, general form: the mirror image of the E kernel. Its differences are
// forward ones, so workgroups take the tiles in decreasing order (the +y/+z
// neighbour tiles were read just before, by the same XCD) and march along -x,
// keeping E of plane i+1 in registers.
template <class FS, class MS, bool NT>
__device__ __forceinline__ void any_H_tile(const MainArgs<FS, MS>& __restrict__ a, unsigned tile) {
  using T = typename FS::R;
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, tile, j, k, i0, i1, act);
  const int64_t sy = d.nz, sx = d.px;
  const int64_t zp = k < d.nz - 1 ? 1 : 0, yp = j < d.ny - 1 ? sy : 0;
  const T zero = T(0);
  int64_t cell = (int64_t)(i1 - 1) * sx + (int64_t)j * sy + k;
  T ez_next = zero, ey_next = zero;  // E at plane i+1
  typename FS::Rec erec{};          // records: E of plane i+1 as loaded
  if (i1 < d.nx) {
    if constexpr (FS::kRecords) {
      erec = a.G.rec3(cell + sx);
    } else {
      ez_next = a.G.template get_c<2>(cell + sx);
      ey_next = a.G.template get_c<1>(cell + sx);
    }
  }
  typename MS::Key key = a.M.template key<NT>(cell);
  for (int i = i1 - 1; i >= i0; --i, cell -= sx) {
    T ev[3], m[3], h[3];
    const typename MS::Key kc_ = key;
    if (i > i0) key = a.M.template key<NT>(cell - sx);  // the next plane's (marching -x)
    T ey_kp, ex_kp, ez_jp, ex_jp;
    if constexpr (FS::kRecords) {
      const typename FS::Rec er = a.G.rec3(cell);
      FS::decode3(er, ev);
      const f32x4 zr = a.G.rec3(cell + zp), yr = a.G.rec3(cell + yp);
      ex_kp = FS::template decode_c<0>(zr), ey_kp = FS::template decode_c<1>(zr);
      ex_jp = FS::template decode_c<0>(yr), ez_jp = FS::template decode_c<2>(yr);
      ez_next = FS::template decode_c<2>(erec);
      ey_next = FS::template decode_c<1>(erec);
      erec = er;
    } else {
      a.G.template get3_s<false>(cell, ev);
      ey_kp = a.G.template get_c<1>(cell + zp), ex_kp = a.G.template get_c<0>(cell + zp);
      ez_jp = a.G.template get_c<2>(cell + yp), ex_jp = a.G.template get_c<0>(cell + yp);
    }
    a.M.template get3<NT>(kc_, cell, m);
    a.F.template get3_s<NT>(cell, h);
    const T ex = ev[0], ey = ev[1], ez = ev[2];
    // forward differences; an absent one contributes nothing (grid.py:42-49)
    Diffs<T> df;
    df.zy = j < d.ny - 1 ? ez_jp - ez : zero;
    df.yz = k < d.nz - 1 ? ey_kp - ey : zero;
    df.xz = k < d.nz - 1 ? ex_kp - ex : zero;
    df.zx = i < d.nx - 1 ? ez_next - ez : zero;
    df.yx = i < d.nx - 1 ? ey_next - ey : zero;
    df.xy = j < d.ny - 1 ? ex_jp - ex : zero;
    T curl[3];
    curl[0] = (zero + df.zy) - df.yz;
    curl[1] = (zero + df.xz) - df.zx;
    curl[2] = (zero + df.yx) - df.xy;
    T kc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      kc[c] = a.sc * m[c];
      h[c] = h[c] - kc[c] * curl[c];
    }
    if (act) {
      // objects leave H unchanged (objects.py:131-137, 223-229, 271-277)
      if (a.nfaces) pml_cell<false>(a.faces, a.nfaces, d, i, j, k, df, kc, h);
      a.F.template put3_s<NT>(cell, h);
    }
    if constexpr (!FS::kRecords) {
      ez_next = ez;
      ey_next = ey;
    }
  }
}

// Main H kernel: the mirror image of the E kernel, marching along -x.
template <class FS, class MS, bool NT>
__device__ __forceinline__ void main_H_tile(const MainArgs<FS, MS>& __restrict__ a, unsigned tile) {
  using T = typename FS::R;
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, tile, j, k, i0, i1, act);
  if (!wave_any(act)) return;
  const int64_t base = (int64_t)i0 * d.px;  // the offsets count from plane i0
  const uint32_t pc = (uint32_t)(j * d.nz + k), at = (uint32_t)(i1 - 1 - i0) * (uint32_t)d.px + pc;
  const uint32_t fstep = (uint32_t)d.px * FS::kCell, mstep = (uint32_t)d.px * MS::kCell;
  uint32_t fo = at * FS::kCell, mo = at * MS::kCell;
  const uint32_t dk = k < d.nz - 1 ? FS::kCell : 0, dj = j < d.ny - 1 ? (uint32_t)d.nz * FS::kCell : 0;
  TilePml<false, T> pml;
  pml.init(a, i1 - 1, j, k);
  const T zero = T(0);
  typename FS::Own enext;  // E of plane i+1
  typename MS::Own ahead{};
  if constexpr (MS::kAhead) ahead = a.M.template own<NT>(base, mo);
  for (int i = i1 - 1; i >= i0; --i) {
    opaque(fo);
    if constexpr (MS::kCell == FS::kCell) mo = fo;
    if (i == i1 - 1) enext = a.G.template own<false>(base, i1 < d.nx ? fo + fstep : fo);
    const typename FS::Own eown = a.G.template own<false>(base, fo);
    const typename FS::Duo ek = a.G.template duo<0, 1>(base, fo + dk), ej = a.G.template duo<0, 2>(base, fo + dj);
    typename MS::Own mat;
    if constexpr (MS::kAhead) {
      mat = ahead;
      if (i > i0) ahead = a.M.template own<NT>(base, mo - mstep);
    } else {
      mat = a.M.template own<NT>(base, mo);
    }
    const typename FS::Own hown = a.F.template own<NT>(base, fo);
    pml.load(a, i, pc);
    const T e0 = FS::template value<0>(eown), e1 = FS::template value<1>(eown), e2 = FS::template value<2>(eown);
    // forward differences; an absent one contributes nothing (grid.py:42-49)
    Diffs<T> df;
    df.zy = dj ? FS::template value<0, 2, 2>(ej) - e2 : zero;
    df.yz = dk ? FS::template value<0, 1, 1>(ek) - e1 : zero;
    df.xz = dk ? FS::template value<0, 1, 0>(ek) - e0 : zero;
    df.zx = i < d.nx - 1 ? FS::template value<2>(enext) - e2 : zero;
    df.yx = i < d.nx - 1 ? FS::template value<1>(enext) - e1 : zero;
    df.xy = dj ? FS::template value<0, 2, 0>(ej) - e0 : zero;
    enext = eown;
    T h[3] = {FS::template value<0>(hown), FS::template value<1>(hown), FS::template value<2>(hown)};
    T m[3], curl[3], kc[3];
    a.M.values(mat, m);
    curl[0] = (zero + df.zy) - df.yz;
    curl[1] = (zero + df.xz) - df.zx;
    curl[2] = (zero + df.yx) - df.xy;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      kc[c] = a.sc * m[c];
      h[c] = h[c] - kc[c] * curl[c];
    }
    // objects leave H unchanged (objects.py:131-137, 223-229, 271-277)
    pml.apply(a, df.zx, df.yx, df.zy, df.xy, df.yz, df.xz, kc, h);
    opaque(fo);
    a.F.template put_own<NT>(base, fo, h);
    fo -= fstep;
    mo -= mstep;
    pml.next_plane();
  }
}

template <class FS, class MS, bool NT>
__global__ void __launch_bounds__(1024) k_main_H(MainArgs<FS, MS> a) {
  unsigned n;
  const int64_t t = launch_tile(a, n);
  if (t >= 0) main_H_tile<FS, MS, NT>(a, n - 1 - (unsigned)t);
}

template <class FS, class MS>
__global__ void __launch_bounds__(1024) k_any_H(MainArgs<FS, MS> a) {
  unsigned n;
  const int64_t t = launch_tile(a, n);
  if (t >= 0) any_H_tile<FS, MS, true>(a, n - 1 - (unsigned)t);
}

// ------------------------------------------------------------ batched kernels
// Many independent grids stepped by one launch per half step over a work
// list of positions (first[s] = first position of grid s, item_sim[u] = the
// grid of position u). Workgroup w takes positions w', w' + G, w' + 2G, ...
// (G workgroups). With G equal to the number of positions every workgroup has
// one tile, as for a single grid; a smaller G makes the grid of workgroups
// persistent. Two dealings to the 8 XCDs (workgroup w runs on XCD w mod 8):
//  * contiguous (small batches): the positions are every grid's tiles in
//    turn and w' = w dealt so that each XCD gets a contiguous run of them
//    (neighbouring tiles share halo planes in its L2);
//  * cyclic (batches whose fields outgrow the caches): w' = w, and the
//    x-chunks of all grids, taken in turn, are dealt to the XCDs in rotation
//    -- chunk g of that sequence to XCD g mod 8 (grid s starts at XCD rot[s])
//    -- each XCD walking the tiles of its chunks in order. Every XCD then gets
//    an eighth of every grid, so grids of unequal cost per tile (CPML-heavy
//    small grids beside large ones) load the XCDs evenly, and at any moment
//    the 8 XCDs work on neighbouring chunks, as a single grid's cyclic
//    launch does. A grid spans whole rounds of 8 chunks; the positions of a
//    round that fall before its first chunk or after its last are idle.
// The time index lives in device memory so that a captured graph of steps
// can be replayed: the E kernel reads it for the folded point sources, the H
// kernel advances it.
template <class FS, class MS>
struct BatchArgs {
  const MainArgs<FS, MS>* sims;  // per grid, launch shape included
  const int64_t* first;          // nsim + 1 entries
  const int32_t* item_sim;       // grid of each position
  const int32_t* rot;            // cyclic dealing: XCD of each grid's first chunk
  int64_t total;                 // positions (cyclic: a multiple of 8)
  int64_t* q;                    // time index of the next E half step
  int32_t cyclic;
};

// Tile of grid a at position `local` of its span under cyclic dealing
// (the grid's first chunk on XCD rot), or -1 for an idle position.
template <class FS, class MS>
__device__ __forceinline__ int64_t batch_cyclic_tile(const MainArgs<FS, MS>& a, unsigned local, int rot) {
  const unsigned x = local % 8, k = local / 8, round = a.per.of(k);
  const int c = (int)(round * 8 + x) - rot;
  return c >= 0 && c < (int)a.nchunks ? (int64_t)c * a.per.d + (k - round * a.per.d) : -1;
}

// Form of a batched E launch: the main one, or the general one without and
// with objects.
enum { kMainForm, kGeneral, kObjects };

// One position of a batched E launch. The position and its grid are the
// same for the whole workgroup: say so, so that the grid's arguments are read
// with scalar loads (and, through the restrict reference of the tile body,
// not read again after the field stores). The launch arguments come by value:
// taken by reference, the pointers read from them lost their global address
// space, and the face tables were read with vector (flat) loads, each cell's
// face loop waiting on memory (twice the time per launch).
template <class FS, class MS, typename O, bool NT, int FORM>
__device__ __forceinline__ void batch_E_at(BatchArgs<FS, MS> b, int64_t it, int64_t q) {
  const int64_t u = __builtin_amdgcn_readfirstlane((int)it);
  const int s = __builtin_amdgcn_readfirstlane(gp(b.item_sim)[u]);
  int64_t t = u - b.first[s];
  if (b.cyclic) {
    t = batch_cyclic_tile(b.sims[s], (unsigned)t, b.rot[s]);
    if (t < 0) return;
  }
  if constexpr (FORM == kMainForm) main_E_tile<FS, MS, false, NT>(b.sims[s], (unsigned)t, q);
  else any_E_tile<FS, MS, O, FORM == kObjects, NT>(b.sims[s], (unsigned)t, q);
}

// One position of a batched H launch: each grid's tiles in decreasing order
// (the mirror of the E kernel's order, as for one grid; contiguous dealing
// walks the whole list from its end).
template <class FS, class MS, bool NT, bool ANY>
__device__ __forceinline__ void batch_H_at(BatchArgs<FS, MS> b, int64_t it) {
  const int64_t u = __builtin_amdgcn_readfirstlane((int)(b.cyclic ? it : b.total - 1 - it));
  const int s = __builtin_amdgcn_readfirstlane(gp(b.item_sim)[u]);
  int64_t t = u - b.first[s];
  if (b.cyclic) {
    t = batch_cyclic_tile(b.sims[s], (unsigned)t, b.rot[s]);
    if (t < 0) return;
    t = (int64_t)b.sims[s].per.d * b.sims[s].nchunks - 1 - t;
  }
  if constexpr (ANY) any_H_tile<FS, MS, NT>(b.sims[s], (unsigned)t);
  else main_H_tile<FS, MS, NT>(b.sims[s], (unsigned)t);
}

// LOOP: a persistent grid of workgroups walking the list; otherwise one
// position per workgroup, with no loop around the tile body (the loop's
// live values made the compiler spill scalar registers to vector lanes,
// ~50 more vector instructions per wavefront).
template <class FS, class MS, typename O, bool NT, bool LOOP, int FORM>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(EWaves<FS>::value)))
k_batch_E(BatchArgs<FS, MS> b) {
  const int64_t q = *b.q;
  const int64_t it0 = b.cyclic ? (int64_t)blockIdx.x : (int64_t)xcd_tile(blockIdx.x, gridDim.x);
  if constexpr (LOOP) {
    for (int64_t it = it0; it < b.total; it += gridDim.x) batch_E_at<FS, MS, O, NT, FORM>(b, it, q);
  } else if (it0 < b.total) {
    batch_E_at<FS, MS, O, NT, FORM>(b, it0, q);
  }
}

// H half step; one thread advances the time index (nothing else in this
// kernel reads it, and the E kernel of this step has completed).
template <class FS, class MS, bool NT, bool LOOP, bool ANY>
__global__ void __launch_bounds__(1024) k_batch_H(BatchArgs<FS, MS> b) {
  const int64_t it0 = b.cyclic ? (int64_t)blockIdx.x : (int64_t)xcd_tile(blockIdx.x, gridDim.x);
  if constexpr (LOOP) {
    for (int64_t it = it0; it < b.total; it += gridDim.x) batch_H_at<FS, MS, NT, ANY>(b, it);
  } else if (it0 < b.total) {
    batch_H_at<FS, MS, NT, ANY>(b, it0);
  }
  // after the work: a branch at the top would keep the compiler from
  // treating the tile loop's values as uniform
  if (blockIdx.x == 0 && threadIdx.x == 0) b.q[0] = b.q[0] + 1;
}

// Sets the batched time index (a kernel rather than a memory copy, so that
// nothing of the host stays referenced after the call).
__global__ void k_set_time(int64_t* q, int64_t v) {
  if (blockIdx.x == 0 && threadIdx.x == 0) q[0] = v;
}

// One CPML face applied on its own (faces registered after a periodic
// boundary): F is the field being updated, G the other one. AX, the face's
// normal axis, is a template parameter so that no index depends on a runtime
// branch over the axis.
template <class FS, class MS, bool IS_E, int AX>
__global__ void __launch_bounds__(256) k_face(Dims d, typename FS::R sc, FS F, FS G, MS M, FaceDev fd) {
  using T = typename FS::R;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= fd.slab) return;
  // slab-local coordinates, the slab laid out like the grid with axis AX of length t
  const int64_t sny = AX == 1 ? fd.t : d.ny, snz = AX == 2 ? fd.t : d.nz;
  const int64_t li = p / (sny * snz), lj = (p / snz) % sny, lk = p % snz;
  const int l = (int)(AX == 0 ? li : (AX == 1 ? lj : lk));
  const int n = AX == 0 ? d.nx : (AX == 1 ? d.ny : d.nz);
  const int g = fd.high ? n - fd.t + l : l;
  const int i = AX == 0 ? g : (int)li, j = AX == 1 ? g : (int)lj, k = AX == 2 ? g : (int)lk;
  const int64_t cell = cell_of(d, i, j, k);
  const int64_t st = AX == 0 ? d.px : (AX == 1 ? (int64_t)d.nz : 1);
  // the other field's components differenced by this face: 3-AX-C0, 3-AX-C1
  constexpr int S0 = 3 - AX - (AX == 0 ? 1 : 0), S1 = 3 - AX - (AX == 2 ? 1 : 2);
  const int64_t o0 = S0 * d.cs + cell, o1 = S1 * d.cs + cell;
  T d0 = T(0), d1 = T(0);
  if (IS_E && l >= 1) {
    d0 = G.get(o0) - G.get(o0 - st);
    d1 = G.get(o1) - G.get(o1 - st);
  }
  if (!IS_E && l <= fd.t - 2) {
    d0 = G.get(o0 + st) - G.get(o0);
    d1 = G.get(o1 + st) - G.get(o1);
  }
  T m[3], kc[3], v[3];
  M.template get3<false>(M.template key<false>(cell), cell, m);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    kc[c] = sc * m[c];
    v[c] = F.get(c * d.cs + cell);
  }
  // pml_face reads the two normal-axis differences
  pml_face<IS_E>(fd, d, i, j, k, d0, d1, d0, d1, d0, d1, kc[0], kc[1], kc[2], v[0], v[1], v[2]);
#pragma unroll
  for (int c = 0; c < 3; ++c) F.put(c * d.cs + cell, v[c]);
}

// Periodic plane copy: to_low ? plane 0 <- plane n-1 : plane n-1 <- plane 0.
template <class FS>
__global__ void __launch_bounds__(256) k_periodic(Dims d, FS F, int axis, int to_low) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t n_plane, src, dst;
  if (axis == 0) {
    n_plane = (int64_t)d.ny * d.nz;
    if (p >= n_plane) return;
    const int64_t last = (int64_t)(d.nx - 1) * d.px + p;
    src = to_low ? last : p;
    dst = to_low ? p : last;
  } else if (axis == 1) {
    n_plane = (int64_t)d.nx * d.nz;
    if (p >= n_plane) return;
    const int64_t i = p / d.nz, k = p % d.nz;
    const int64_t first = cell_of(d, i, 0, k), last = cell_of(d, i, d.ny - 1, k);
    src = to_low ? last : first;
    dst = to_low ? first : last;
  } else {
    n_plane = (int64_t)d.nx * d.ny;
    if (p >= n_plane) return;
    const int64_t first = cell_of(d, p / d.ny, p % d.ny, 0), last = first + d.nz - 1;
    src = to_low ? last : first;
    dst = to_low ? first : last;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) F.copy(c * d.cs + dst, c * d.cs + src);
}

template <class FS>
struct TailArgs {
  Dims d;
  FS F;  // field of this half step
  int32_t is_H;
  int32_t nsrc, ndet;
  const SrcDev* srcs;
  const DetDev* dets;
  const double* wave;
  int64_t wave_cap;
  int64_t q;
  int64_t counter;  // half steps of this kind already taken by the plan
  int64_t counter_H;  // H half steps taken (the soft sources' current sample)
  int32_t ncur;
  const CurDev* curs;
  // differentiation record (E half step): the field inside box `rb` after
  // the sources, (3, cells of rb), when rec is not null
  typename FS::R* rec;
  Box rb;
};

// Sources in registration order, then detector samples. One workgroup keeps
// the order between sources touching the same cell and the detector reads with
// its barriers; several workgroups are launched over lists of which no two
// share a cell (launch_tail), each list spread over all of them. Bound by the
// chain of loads cell index -> field -> store: in one workgroup a plane source
// and a plane monitor of ~14000 cells took 26 us a half step at 201x150x97,
// spread 5.0 us.
template <class FS>
__global__ void __launch_bounds__(256) k_tail(TailArgs<FS> a) {
  using T = typename FS::R;
  using Sample = typename FS::Sample;
  const int tid = (int)(blockIdx.x * blockDim.x + threadIdx.x), stride = (int)(gridDim.x * blockDim.x);
  for (int s = 0; s < a.nsrc; ++s) {
    const SrcDev& src = a.srcs[s];
    if (a.is_H && src.kind != FDTD_SRC_PLANE) continue;
    const T w = (T)gp(a.wave)[s * a.wave_cap + a.q];
    const int64_t base = (int64_t)(a.is_H ? src.compH : src.compE) * a.d.cs;
    if (src.kind == FDTD_SRC_SOFT) {
      // sources.py:604-631: the voltage v of the waveform, plus R times the
      // current its detector measured after the last H half step
      if (tid == 0) {
        const CurDev& cd = a.curs[src.det];
        const T cur = a.q > 0 ? (T)ld_stream<false>(reinterpret_cast<const Sample*>(cd.buf) +
                                                    (a.counter_H - 1 - cd.slot0) * cd.n)
                              : T(0);
        const T u = src.amplitude > 0 ? w + (T)src.amplitude * cur : w;
        const int64_t cell = base + gp(src.cells)[0];
        a.F.put(cell, a.F.get(cell) + u / (T)src.spacing);
        const int64_t slot = a.counter - src.slot0;
        st_stream<false>(reinterpret_cast<Sample*>(src.vin) + slot, (Sample)w);
        st_stream<false>(reinterpret_cast<Sample*>(src.vout) + slot, (Sample)u);
      }
      __syncthreads();
      continue;
    }
    for (int p = tid; p < src.n; p += stride) {
      const int64_t cell = base + gp(src.cells)[p];
      if (src.kind == FDTD_SRC_POINT)
        a.F.put(cell, a.F.get(cell) + w);
      else if (src.kind == FDTD_SRC_LINE)
        a.F.put(cell, a.F.get(cell) + (T)gp(src.profile)[p] * w);
      else
        a.F.put(cell, (T)src.amplitude * w);
    }
    __syncthreads();
  }
  if (a.is_H) {
    // detectors.py:388-460, X = 0, Y = 1; numpy wraps index -1 to the last
    for (int t = 0; t < a.ncur; ++t) {
      const CurDev& cd = a.curs[t];
      Sample* const buf = reinterpret_cast<Sample*>(cd.buf) + (a.counter - cd.slot0) * cd.n;
      const T dx = (T)cd.spacing;
      for (int p = tid; p < cd.n; p += stride) {
        const int px = gp(cd.pts)[p], py = gp(cd.pts)[cd.n + p], pz = gp(cd.pts)[2 * cd.n + p];
        auto H = [&](int c, int x, int y, int z) {
          x = x < 0 ? x + a.d.nx : x;
          y = y < 0 ? y + a.d.ny : y;
          z = z < 0 ? z + a.d.nz : z;
          return a.F.get(c * a.d.cs + cell_of(a.d, x, y, z));
        };
        T v1 = (H(0, px, py - 1, pz) - H(0, px, py, pz)) * dx;
        T v2 = (H(1, px, py, pz) - H(1, px - 1, py, pz)) * dx;
        const T c1 = v1 + v2;
        v1 = (H(0, px, py - 1, pz - 1) - H(0, px, py, pz - 1)) * dx;
        v2 = v2 + (H(1, px, py, pz - 1) - H(1, px - 1, py, pz - 1)) * dx;
        const T c2 = v1 + v2;
        st_stream<false>(buf + p, (Sample)((c1 + c2) / T(2)));
      }
    }
  }
  if (a.rec) {
    const int64_t nr = box_cells(a.rb);
    for (int64_t p = tid; p < 3 * nr; p += stride) {
      const int c = (int)(p / nr);
      a.rec[p] = a.F.get(c * a.d.cs + box_cell(a.rb, a.d, p - c * nr));
    }
  }
  for (int t = 0; t < a.ndet; ++t) {
    const DetDev& det = a.dets[t];
    const int64_t slot = a.counter - (a.is_H ? det.slot0H : det.slot0E);
    Sample* const buf = reinterpret_cast<Sample*>(a.is_H ? det.bufH : det.bufE) + slot * det.n * 3;
    for (int p = tid; p < det.n * 3; p += stride) {
      const int c = p % 3;
      st_stream<false>(buf + p, a.F.sample(c * a.d.cs + gp(det.cells)[p / 3]));
    }
  }
}

// Non-finite check: flag[0] becomes nonzero when one of the n values of v
// (stride `skip`: with skip = 4 every 4th value is not a field value but a
// compensation word and is ignored) is a NaN or an infinity. The reference
// has no such check (its only guard is the Courant limit, grid.py:123-127);
// it lets a caller find a diverged run without copying the fields back.
template <typename S>
__global__ void __launch_bounds__(256) k_nonfinite(const S* __restrict__ v, int64_t n, int skip, int* flag) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if (skip && i % skip == skip - 1) continue;
    const S x = v[i];
    bad |= !(x - x == S(0));  // NaN - NaN and inf - inf are NaN
  }
  if (bad) atomicOr(flag, 1);
}

// Plain device copy of n 16-byte words: the bandwidth reference for the
// step kernels (a stream that reads and writes every byte once).
__global__ void __launch_bounds__(256) k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}


// ================================================================ adjoint
// The step is linear in (E, H, psi) for fixed materials, so reverse-mode
// differentiation of an objective through T steps applies the transposes of
// the two half steps in reverse order. The kernels below are those exact
// transposes for plain storage with every CPML face folded into the step and
// objects composed into a per-cell affine E update
//   E' = dcoef * E + gcoef * curl_H(H) + CPML + sources
// (sources add constants and drop out). They march like the main kernels:
// the transpose of the H half step gathers backward neighbours (the shape of
// the E kernel), the transpose of the E half step forward ones (the shape of
// the H kernel).

// One CPML face as a transposed kernel sees it at one launch: the adjoint
// psi of its half step that the launch reads and the one it writes (two
// buffers used alternately, (2, slab) values each like the forward psi), the
// half step's b and c profiles (t values) and the slab size; t = 0 when the
// side has no face. A device table holds one per half step, parity, axis and
// side, so a kernel reads each face's entry with one batch of scalar loads
// and no pointer chasing.
template <typename T>
struct AdjSide {
  const T* pin;
  T* pout;
  const double* b;
  const double* c;
  int64_t slab;
  int32_t t, pad;
};

template <typename T>
struct AdjArgs {
  Dims d;
  T sc;
  T* lamE;               // dJ/dE, (3, N)
  T* lamH;               // dJ/dH, (3, N)
  const T* inv_eps;      // grid materials: the CPML terms use S*inv
  const T* inv_mu;
  const T* gcoef;        // (3, N)
  const T* dcoef;        // (3, N) or null (all ones)
  const AdjSide<T>* side;  // [axis][low/high side] of this launch's half step and parity
  Box db;                // design box: grad += S lamE curl
  const T* curl;         // (3, cells of db) recorded for this step
  double* grad;          // (3, cells of db)
  Box pb;                // objective box: lamE += 2 E
  const T* plane;        // (3, cells of pb) recorded for this step
  int32_t bz_shift, cx, by, flat;  // launch shape, as for the main kernels
  Divide per, row;
  uint32_t nchunks;
  // anisotropic objects: the plan's object table and a (3, N) buffer of
  // Y = dJ/d(curl H) of the E half step, written by k_adj_Y
  const ObjDev* objs;
  int32_t nobjs;
  T* ybuf;
};

constexpr int kAdjThreads = 256;

// Slab layout constants of a face normal to AX: the slab is the grid with
// axis AX shortened to t; `st` is the slab offset of one step along AX.
template <int AX>
__device__ __forceinline__ int64_t slab_off(const Dims& d, int t, int i, int j, int k, int l) {
  if constexpr (AX == 0) return ((int64_t)l * d.ny + j) * d.nz + k;
  else if constexpr (AX == 1) return ((int64_t)i * t + l) * d.nz + k;
  else return ((int64_t)i * d.ny + j) * t + l;
}
template <int AX>
__device__ __forceinline__ int64_t slab_step(const Dims& d, int t) {
  if constexpr (AX == 0) return (int64_t)d.ny * d.nz;
  else if constexpr (AX == 1) return d.nz;
  else return 1;
}

// The faces normal to AX at one cell of k_adj_any_H (see there): the face's own
// psi transpose and the difference terms of this cell and of the face cell
// one step back along AX (which holds the Y values yb0, yb1). The face's
// axis is a compile-time constant, so components and signs are too. t_lo and
// t_hi are the slab thicknesses of the two sides (0: no face), read once per
// kernel, so a cell outside every slab reads nothing of the face table.
template <int AX, typename T>
__device__ __forceinline__ void adj_faces_H(const AdjArgs<T>& a, int t_lo, int t_hi, int i, int j, int k, T yc0,
                                           T yc1, T yb0, T yb1, T e[3]) {
  constexpr int C0 = AX == 0 ? 1 : 0, C1 = AX == 2 ? 1 : 2;
  constexpr int S0 = 3 - AX - C0, S1 = 3 - AX - C1;
  // phi_H = psi_{C+1} - psi_{C+2} enters H' with a minus sign
  const T sg0 = AX == (C0 + 1) % 3 ? T(-1) : T(1), sg1 = AX == (C1 + 1) % 3 ? T(-1) : T(1);
  const Dims& d = a.d;
  const int g = AX == 0 ? i : (AX == 1 ? j : k);
  const int n = AX == 0 ? d.nx : (AX == 1 ? d.ny : d.nz);
#pragma nounroll
  for (int side = 0; side < 2; ++side) {
    const int t = side ? t_hi : t_lo;
    const int l = side ? g - (n - t) : g;
    if (t == 0 || l < 0 || l > t) continue;  // neither this cell nor the one back is in the slab
    const AdjSide<T>& fd = a.side[AX * 2 + side];
    const gptr<const T> pin = gp(fd.pin);
    const gptr<T> pout = gp(fd.pout);
    const int64_t off = slab_off<AX>(d, t, i, j, k, l), slab = fd.slab;
    if (l < t) {
      const T w0 = pin[off] + sg0 * yc0;
      const T w1 = pin[slab + off] + sg1 * yc1;
      const T b = (T)gp(fd.b)[l];
      pout[off] = b * w0;
      pout[slab + off] = b * w1;
      if (l <= t - 2) {  // psi'(l) holds c(l) (E(l+1) - E(l))
        const T c = (T)gp(fd.c)[l];
        e[S0] = e[S0] - c * w0;
        e[S1] = e[S1] - c * w1;
      }
    }
    if (l >= 1 && l - 1 <= t - 2) {  // ... and this cell is the E(l+1) of slab cell l-1
      const int64_t ob = off - slab_step<AX>(d, t);
      const T w0 = pin[ob] + sg0 * yb0;
      const T w1 = pin[slab + ob] + sg1 * yb1;
      const T c = (T)gp(fd.c)[l - 1];
      e[S0] = e[S0] + c * w0;
      e[S1] = e[S1] + c * w1;
    }
  }
}

// The faces normal to AX at one cell of k_adj_any_E (see there): the face's own
// psi transpose and the difference terms of this cell and of the face cell
// one step ahead along AX. lc0, lc1 are lamE of the face's components C0, C1
// at this cell, la0, la1 at the cell ahead (already loaded by the caller).
template <int AX, typename T>
__device__ __forceinline__ void adj_faces_E(const AdjArgs<T>& a, int t_lo, int t_hi, int i, int j, int k, int64_t cell,
                                           T lc0, T lc1, T la0, T la1, T h[3]) {
  constexpr int C0 = AX == 0 ? 1 : 0, C1 = AX == 2 ? 1 : 2;
  constexpr int S0 = 3 - AX - C0, S1 = 3 - AX - C1;
  // phi_E = psi_{C+1} - psi_{C+2} enters E' with a plus sign
  const T sg0 = AX == (C0 + 1) % 3 ? T(1) : T(-1), sg1 = AX == (C1 + 1) % 3 ? T(1) : T(-1);
  const Dims& d = a.d;
  const int64_t cs = d.cs;
  const int g = AX == 0 ? i : (AX == 1 ? j : k);
  const int n = AX == 0 ? d.nx : (AX == 1 ? d.ny : d.nz);
  const int64_t st = AX == 0 ? d.px : (AX == 1 ? (int64_t)d.nz : 1);
  const T sc = a.sc;
  auto K = [&](int c, int64_t x) { return sc * a.inv_eps[c * cs + x]; };
#pragma nounroll
  for (int side = 0; side < 2; ++side) {
    const int t = side ? t_hi : t_lo;
    const int l = side ? g - (n - t) : g;
    if (t == 0 || l < -1 || l >= t) continue;  // neither this cell nor the one ahead is in the slab
    const AdjSide<T>& fd = a.side[AX * 2 + side];
    const gptr<const T> pin = gp(fd.pin);
    const gptr<T> pout = gp(fd.pout);
    const int64_t off = slab_off<AX>(d, t, i, j, k, l), slab = fd.slab;
    if (l >= 0) {
      const T w0 = pin[off] + sg0 * (K(C0, cell) * lc0);
      const T w1 = pin[slab + off] + sg1 * (K(C1, cell) * lc1);
      const T b = (T)gp(fd.b)[l];
      pout[off] = b * w0;
      pout[slab + off] = b * w1;
      if (l >= 1) {  // psi'(l) holds c(l) (H(l) - H(l-1))
        const T c = (T)gp(fd.c)[l];
        h[S0] = h[S0] + c * w0;
        h[S1] = h[S1] + c * w1;
      }
    }
    if (l + 1 >= 1 && l + 1 <= t - 1 && g + 1 < n) {  // ... and the H(l-1) of slab cell l+1
      const int64_t ou = off + slab_step<AX>(d, t);
      const T w0 = pin[ou] + sg0 * (K(C0, cell + st) * la0);
      const T w1 = pin[slab + ou] + sg1 * (K(C1, cell + st) * la1);
      const T c = (T)gp(fd.c)[l + 1];
      h[S0] = h[S0] - c * w0;
      h[S1] = h[S1] - c * w1;
    }
  }
}

// Zeroes lam at n cells (one component; lam already offset to it).
template <typename T>
__global__ void __launch_bounds__(256) k_adj_zero(T* lam, const int64_t* cells, int n) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) lam[cells[p]] = T(0);
}

// Transpose of the H half step (grid.py:301-325, boundaries.py:421-431 and
// 461-487). Forward, per face normal to ax and psi component q (H component
// C_q, E component s_q = 3-ax-C_q differenced along ax):
//   psiH'_q = bH psiH_q + cH(l) (E_s(l+1) - E_s(l))     for l <= t-2
//   H'      = H - K_H curl_E(E) + sg_q K_H psiH'_q,       K_H = S inv_mu
// (phi_H = psi_{C+1} - psi_{C+2} enters H' with a minus sign: sg_q = -1 when
// ax = C_q + 1 mod 3, +1 otherwise). With Y = K_H lamH (lamH = dJ/dH' =
// dJ/dH) and w_q = lamPsiH'_q + sg_q Y_{C_q}:
//   lamPsiH_q = bH w_q
//   lamE      = dcoef lamE - curl_E^T(Y) - cH(l) w_q [at E_s(l)]
//                                        + cH(l) w_q [at E_s(l+1)]
// curl_E^T gathers backward neighbours with the masks of curl_E
// (grid.py:39-49): (curl_E^T Y)_x = ([k>=1] Y_y(k-1) - [k<=nz-2] Y_y(k))
// - ([j>=1] Y_z(j-1) - [j<=ny-2] Y_z(j)), and cyclically. The factor dcoef
// comes from the transpose of the following E half step (k_adj_E leaves it);
// after the update the objective's 2 E is added inside the objective box.
//
// General form, for slabs that overlap and planes past 32-bit offsets.
template <typename T>
__global__ void __launch_bounds__(kAdjThreads) k_adj_any_H(AdjArgs<T> a) {
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  // as in the main kernels: every load of a plane at once, threads past the
  // edge on the nearest cell (storing nothing), neighbour offset 0 at an edge
  tile_column(a, xcd_tile(blockIdx.x, gridDim.x), j, k, i0, i1, act);
  const int64_t sy = d.nz, sx = d.px, cs = d.cs;
  const int64_t zm = k > 0 ? 1 : 0, ym = j > 0 ? sy : 0;
  const T zero = T(0), sc = a.sc;
  auto Y = [&](int c, int64_t x) { return (sc * a.inv_mu[c * cs + x]) * a.lamH[c * cs + x]; };
  int ts[6];  // slab thickness of each side's face (0: none), read once
#pragma unroll
  for (int q = 0; q < 6; ++q) ts[q] = a.side[q].t;
  int64_t cell = (int64_t)i0 * sx + (int64_t)j * sy + k;
  // inv_mu and lamH of components 1 and 2 at plane i-1, as loaded: Y is formed
  // where it is used. A carried product is computed right after its loads,
  // ahead of the branch that guards the stores, and the wave then waits for
  // them before it issues the plane's other loads (two round trips a plane).
  T mz_prev = zero, lz_prev = zero, my_prev = zero, ly_prev = zero;
  if (i0 > 0) {
    mz_prev = a.inv_mu[2 * cs + cell - sx];
    lz_prev = a.lamH[2 * cs + cell - sx];
    my_prev = a.inv_mu[cs + cell - sx];
    ly_prev = a.lamH[cs + cell - sx];
  }
  for (int i = i0; i < i1; ++i, cell += sx) {
    const T m1 = a.inv_mu[cs + cell], m2 = a.inv_mu[2 * cs + cell];
    const T lh1 = a.lamH[cs + cell], lh2 = a.lamH[2 * cs + cell];
    const T y0 = Y(0, cell), y1 = (sc * m1) * lh1, y2 = (sc * m2) * lh2;
    const T yz_prev = (sc * mz_prev) * lz_prev, yy_prev = (sc * my_prev) * ly_prev;  // Y at plane i-1
    const T yy_km = Y(1, cell - zm), yx_km = Y(0, cell - zm);
    const T yz_jm = Y(2, cell - ym), yx_jm = Y(0, cell - ym);
    T e0 = a.lamE[cell], e1 = a.lamE[cs + cell], e2 = a.lamE[2 * cs + cell];
    if (a.dcoef) {
      e0 = a.dcoef[cell] * e0;
      e1 = a.dcoef[cs + cell] * e1;
      e2 = a.dcoef[2 * cs + cell] * e2;
    }
    const bool km = k >= 1, kp = k <= d.nz - 2, jm = j >= 1, jp = j <= d.ny - 2, im = i >= 1, ip = i <= d.nx - 2;
    const T t0 = ((km ? yy_km : zero) - (kp ? y1 : zero)) - ((jm ? yz_jm : zero) - (jp ? y2 : zero));
    const T t1 = ((im ? yz_prev : zero) - (ip ? y2 : zero)) - ((km ? yx_km : zero) - (kp ? y0 : zero));
    const T t2 = ((jm ? yx_jm : zero) - (jp ? y0 : zero)) - ((im ? yy_prev : zero) - (ip ? y1 : zero));
    e0 = e0 - t0;
    e1 = e1 - t1;
    e2 = e2 - t2;
    if (act) {
      {
        T e[3] = {e0, e1, e2};
        adj_faces_H<0>(a, ts[0], ts[1], i, j, k, y1, y2, yy_prev, yz_prev, e);
        adj_faces_H<1>(a, ts[2], ts[3], i, j, k, y0, y2, yx_jm, yz_jm, e);
        adj_faces_H<2>(a, ts[4], ts[5], i, j, k, y0, y1, yx_km, yy_km, e);
        e0 = e[0];
        e1 = e[1];
        e2 = e[2];
      }
      const int64_t pp = box_index(a.pb, i, j, k);
      if (pp >= 0) {
        const int64_t np = box_cells(a.pb);
        e0 = e0 + T(2) * a.plane[pp];
        e1 = e1 + T(2) * a.plane[np + pp];
        e2 = e2 + T(2) * a.plane[2 * np + pp];
      }
      a.lamE[cell] = e0;
      a.lamE[cs + cell] = e1;
      a.lamE[2 * cs + cell] = e2;
    }
    mz_prev = m2;
    lz_prev = lh2;
    my_prev = m1;
    ly_prev = lh1;
  }
}

// Transpose of the E half step (grid.py:275-299, objects.py:118-221,
// boundaries.py:409-459). Forward, per face normal to ax and psi component q
// (E component C_q, H component s_q = 3-ax-C_q differenced along ax):
//   psiE'_q = bE psiE_q + cE(l) (H_s(l) - H_s(l-1))      for l >= 1
//   E'      = dcoef E + gcoef curl_H(H) + sg_q K_E psiE'_q,  K_E = S inv_eps
// (phi_E enters E' with a plus sign: sg_q = +1 when ax = C_q + 1 mod 3, -1
// otherwise; K_E is the grid's, zero inside objects). With Y = gcoef lamE
// (lamE = dJ/dE') and w_q = lamPsiE'_q + sg_q K_E lamE_{C_q}:
//   lamPsiE_q = bE w_q
//   lamH     += curl_H^T(Y) + cE(l) w_q [at H_s(l)] - cE(l) w_q [at H_s(l-1)]
//   lamE      = dcoef lamE   (left to the next k_adj_H)
//   grad     += S lamE curl  (dE'/d inv = S curl inside the design box)
// curl_H^T gathers forward neighbours with the masks of curl_H
// (grid.py:65-73): (curl_H^T Y)_x = ([k>=1] Y_y - [k<=nz-2] Y_y(k+1))
// - ([j>=1] Y_z - [j<=ny-2] Y_z(j+1)), and cyclically.
// Y = dJ/d(curl H) of the E half step at every cell when the plan has
// anisotropic objects: gcoef lamE (the diagonal part composed by the host)
// plus, inside each anisotropic object, the transpose of its update
// E += S (inv @ curl) (objects.py:254-269): S inv^T lamE. Overlapping objects
// add their terms in the forward step, so their transposes add here too.
template <typename T>
__global__ void __launch_bounds__(256) k_adj_Y(AdjArgs<T> a) {
  const Dims d = a.d;
  const int64_t cs = d.cs;
  const int64_t cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= cs) return;
  const int64_t r = cell % d.px;  // cell of the x plane; past ny*nz: the plane's padding
  if (r >= (int64_t)d.ny * d.nz) return;
  const T l0 = a.lamE[cell], l1 = a.lamE[cs + cell], l2 = a.lamE[2 * cs + cell];
  T y0 = a.gcoef[cell] * l0, y1 = a.gcoef[cs + cell] * l1, y2 = a.gcoef[2 * cs + cell] * l2;
  const int k = (int)(r % d.nz), j = (int)(r / d.nz), i = (int)(cell / d.px);
  for (int o = 0; o < a.nobjs; ++o) {
    const ObjDev& ob = a.objs[o];
    if (ob.kind != FDTD_OBJ_ANISOTROPIC) continue;
    const Box b{ob.x0, ob.x1, ob.y0, ob.y1, ob.z0, ob.z1};
    const int64_t lo = box_index(b, i, j, k);
    if (lo < 0) continue;
    const gptr<const T> m = gp(reinterpret_cast<const T*>(ob.inv) + lo * 9);
    y0 = y0 + a.sc * ((m[0] * l0 + m[3] * l1) + m[6] * l2);
    y1 = y1 + a.sc * ((m[1] * l0 + m[4] * l1) + m[7] * l2);
    y2 = y2 + a.sc * ((m[2] * l0 + m[5] * l1) + m[8] * l2);
  }
  a.ybuf[cell] = y0;
  a.ybuf[cs + cell] = y1;
  a.ybuf[2 * cs + cell] = y2;
}

// Transpose of a periodic plane copy F[dst] = F[src] along `axis`
// (boundaries.py:184-219; to_low: dst is plane 0, src plane n-1, as for E;
// else the reverse, as for H): lam[src] += lam[dst], lam[dst] = 0.
template <typename T>
__global__ void __launch_bounds__(256) k_adj_periodic(T* lam, Dims d, int axis, int to_low) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t lo_cell, hi_cell;
  if (axis == 0) {
    const int64_t n_plane = (int64_t)d.ny * d.nz;
    if (p >= n_plane) return;
    lo_cell = p;
    hi_cell = (int64_t)(d.nx - 1) * d.px + p;
  } else if (axis == 1) {
    if (p >= (int64_t)d.nx * d.nz) return;
    const int64_t i = p / d.nz, k = p % d.nz;
    lo_cell = cell_of(d, i, 0, k);
    hi_cell = cell_of(d, i, d.ny - 1, k);
  } else {
    if (p >= (int64_t)d.nx * d.ny) return;
    lo_cell = cell_of(d, p / d.ny, p % d.ny, 0);
    hi_cell = lo_cell + d.nz - 1;
  }
  const int64_t dst = to_low ? lo_cell : hi_cell, src = to_low ? hi_cell : lo_cell;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    lam[c * d.cs + src] = lam[c * d.cs + src] + lam[c * d.cs + dst];
    lam[c * d.cs + dst] = T(0);
  }
}

// YB: Y read from ybuf (k_adj_Y ran first) instead of gcoef lamE. General form,
// as for k_adj_any_H.
template <typename T, bool YB>
__global__ void __launch_bounds__(kAdjThreads) k_adj_any_E(AdjArgs<T> a) {
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, gridDim.x - 1 - xcd_tile(blockIdx.x, gridDim.x), j, k, i0, i1, act);
  const int64_t sy = d.nz, sx = d.px, cs = d.cs;
  const int64_t zp = k < d.nz - 1 ? 1 : 0, yp = j < d.ny - 1 ? sy : 0;
  const T zero = T(0), sc = a.sc;
  auto L = [&](int c, int64_t x) { return a.lamE[c * cs + x]; };
  // Y of component c at cell x whose lamE is l
  auto Yc = [&](int c, int64_t x, T l) { return YB ? a.ybuf[c * cs + x] : a.gcoef[c * cs + x] * l; };
  int ts[6];  // slab thickness of each side's face (0: none), read once
#pragma unroll
  for (int q = 0; q < 6; ++q) ts[q] = a.side[q].t;
  int64_t cell = (int64_t)(i1 - 1) * sx + (int64_t)j * sy + k;
  // plane i+1, as loaded: lamE of components 1 and 2 and either their Y
  // (ybuf) or their gcoef (Y = gcoef lamE is formed where it is used, for the
  // reason given in k_adj_any_H)
  T lz_next = zero, ly_next = zero, fz_next = zero, fy_next = zero;
  if (i1 < d.nx) {
    lz_next = L(2, cell + sx);
    ly_next = L(1, cell + sx);
    fz_next = YB ? a.ybuf[2 * cs + cell + sx] : a.gcoef[2 * cs + cell + sx];
    fy_next = YB ? a.ybuf[cs + cell + sx] : a.gcoef[cs + cell + sx];
  }
  for (int i = i1 - 1; i >= i0; --i, cell -= sx) {
    const T le0 = L(0, cell), le1 = L(1, cell), le2 = L(2, cell);
    const T lk0 = L(0, cell + zp), lk1 = L(1, cell + zp);
    const T lj0 = L(0, cell + yp), lj2 = L(2, cell + yp);
    const T f1 = YB ? a.ybuf[cs + cell] : a.gcoef[cs + cell], f2 = YB ? a.ybuf[2 * cs + cell] : a.gcoef[2 * cs + cell];
    const T y0 = Yc(0, cell, le0), y1 = YB ? f1 : f1 * le1, y2 = YB ? f2 : f2 * le2;
    const T yz_next = YB ? fz_next : fz_next * lz_next, yy_next = YB ? fy_next : fy_next * ly_next;  // Y at plane i+1
    const T yy_kp = Yc(1, cell + zp, lk1), yx_kp = Yc(0, cell + zp, lk0);
    const T yz_jp = Yc(2, cell + yp, lj2), yx_jp = Yc(0, cell + yp, lj0);
    const T l0 = a.lamH[cell], l1 = a.lamH[cs + cell], l2 = a.lamH[2 * cs + cell];
    const bool km = k >= 1, kp = k <= d.nz - 2, jm = j >= 1, jp = j <= d.ny - 2, im = i >= 1, ip = i <= d.nx - 2;
    const T t0 = ((km ? y1 : zero) - (kp ? yy_kp : zero)) - ((jm ? y2 : zero) - (jp ? yz_jp : zero));
    const T t1 = ((im ? y2 : zero) - (ip ? yz_next : zero)) - ((km ? y0 : zero) - (kp ? yx_kp : zero));
    const T t2 = ((jm ? y0 : zero) - (jp ? yx_jp : zero)) - ((im ? y1 : zero) - (ip ? yy_next : zero));
    T h0 = l0 + t0, h1 = l1 + t1, h2 = l2 + t2;
    if (act) {
      {
        T h[3] = {h0, h1, h2};
        adj_faces_E<0>(a, ts[0], ts[1], i, j, k, cell, le1, le2, ly_next, lz_next, h);
        adj_faces_E<1>(a, ts[2], ts[3], i, j, k, cell, le0, le2, lj0, lj2, h);
        adj_faces_E<2>(a, ts[4], ts[5], i, j, k, cell, le0, le1, lk0, lk1, h);
        h0 = h[0];
        h1 = h[1];
        h2 = h[2];
      }
      a.lamH[cell] = h0;
      a.lamH[cs + cell] = h1;
      a.lamH[2 * cs + cell] = h2;
      const int64_t pd = box_index(a.db, i, j, k);
      if (pd >= 0) {
        const int64_t nd = box_cells(a.db);
        const T le[3] = {le0, le1, le2};
#pragma unroll
        for (int c = 0; c < 3; ++c)
          a.grad[c * nd + pd] += (double)sc * (double)le[c] * (double)a.curl[c * nd + pd];
      }
    }
    fz_next = f2;
    fy_next = f1;
    lz_next = le2;
    ly_next = le1;
  }
}

// The CPML of a transposed half step at one cell, faces normal to one axis,
// where the slabs of the axis do not overlap: the side whose slab holds the
// cell, its psi and its neighbour's (one step back along the axis for H, ahead
// for E; a cell outside the slab has no term of it) and their coefficients.
template <bool IS_H, typename T>
struct AdjFace {
  bool lo = false, hi = false;          // the side
  bool own = false, near = false;       // the cell's own difference term, its neighbour's
  uint32_t q = 0, step = 0;             // byte offset in the psi arrays, and a plane further
  uint32_t qn = 0, l = 0, ln = 0;       // bytes to the neighbour's psi; byte offsets in the profiles
  double b, c, cn;
  Psi<T> p, n;
  // g: place along the axis of dn cells; at(l, t): the cell's place in a slab
  // of thickness t; st: the slab's cells one step along the axis
  template <class At>
  __device__ __forceinline__ void locate(int g, int dn, int tl, int th, uint32_t st, At&& at) {
    lo = g < tl;
    hi = g >= dn - th;
    if (!lo && !hi) return;
    const int t = lo ? tl : th, at_l = lo ? g : g - (dn - t);
    own = IS_H ? at_l <= t - 2 : at_l >= 1;
    near = IS_H ? at_l >= 1 : at_l <= t - 2;
    q = at(at_l, t) * (uint32_t)sizeof(T);
    qn = near ? (IS_H ? 0u - st : st) * (uint32_t)sizeof(T) : 0;
    l = (uint32_t)at_l * (uint32_t)sizeof(double);
    ln = (uint32_t)(near ? (IS_H ? at_l - 1 : at_l + 1) : at_l) * (uint32_t)sizeof(double);
  }
  __device__ __forceinline__ void fetch(cptr<AdjSide<T>> sd) {
    opaque(q);
    uint32_t r = q + qn;
    opaque(r);
    p.load(sd->pin, sd->pin + sd->slab, q);
    n.load(sd->pin, sd->pin + sd->slab, r);
    opaque(l);
    opaque(ln);
    b = ld_stream<false>(split_ptr(sd->b, l));
    c = ld_stream<false>(split_ptr(sd->c, l));
    cn = ld_stream<false>(split_ptr(sd->c, ln));
  }
  __device__ __forceinline__ void load(cptr<AdjSide<T>> sd) {
    if (lo) fetch(sd);
    if (hi) fetch(sd + 1);
  }
  // v: the updated values of the components 3-AX-C0, 3-AX-C1; y, yn: the
  // weights of the face's components C0, C1 at the cell and at its neighbour
  template <int AX>
  __device__ __forceinline__ void apply(cptr<AdjSide<T>> sd, T y0, T y1, T yn0, T yn1, T v[3]) {
    constexpr int C0 = AX == 0 ? 1 : 0, C1 = AX == 2 ? 1 : 2;
    constexpr int S0 = 3 - AX - C0, S1 = 3 - AX - C1;
    // phi = psi_{C+1} - psi_{C+2} enters H' with a minus sign, E' with a plus sign
    const T sg0 = (AX == (C0 + 1) % 3) == IS_H ? T(-1) : T(1), sg1 = (AX == (C1 + 1) % 3) == IS_H ? T(-1) : T(1);
    if (!lo && !hi) return;
    const T w0 = p.p0 + sg0 * y0, w1 = p.p1 + sg1 * y1;
    const T bt = (T)b, ct = (T)c, cnt = (T)cn;
    const Psi<T> out{bt * w0, bt * w1};
    opaque(q);
    if (lo) out.store(sd->pout, sd->pout + sd->slab, q);
    if (hi) out.store((sd + 1)->pout, (sd + 1)->pout + (sd + 1)->slab, q);
    if (own) {
      v[S0] = IS_H ? v[S0] - ct * w0 : v[S0] + ct * w0;
      v[S1] = IS_H ? v[S1] - ct * w1 : v[S1] + ct * w1;
    }
    if (near) {
      const T u0 = n.p0 + sg0 * yn0, u1 = n.p1 + sg1 * yn1;
      v[S0] = IS_H ? v[S0] + cnt * u0 : v[S0] - cnt * u0;
      v[S1] = IS_H ? v[S1] + cnt * u1 : v[S1] - cnt * u1;
    }
  }
};

// The three axes of a tile's column.
template <bool IS_H, typename T>
struct AdjPml {
  cptr<AdjSide<T>> sides;
  int t0, t1;  // thicknesses of the x slabs
  bool any_x, any_y, any_z;  // the plane is in an x slab; some column of the wavefront in a y (z) slab
  AdjFace<IS_H, T> x, y, z;
  __device__ __forceinline__ void init(const AdjArgs<T>& a, int i, int j, int k) {
    const Dims& d = a.d;
    sides = cp(a.side);
    t0 = sides[0].t;
    t1 = sides[1].t;
    y.locate(j, d.ny, sides[2].t, sides[3].t, (uint32_t)d.nz, [&](int l, int t) {
      y.step = (uint32_t)(t * d.nz) * (uint32_t)sizeof(T);
      return (uint32_t)((i * t + l) * d.nz + k);
    });
    z.locate(k, d.nz, sides[4].t, sides[5].t, 1, [&](int l, int t) {
      z.step = (uint32_t)(t * d.ny) * (uint32_t)sizeof(T);
      return (uint32_t)((i * d.ny + j) * t + l);
    });
    any_y = wave_any(y.lo || y.hi);
    any_z = wave_any(z.lo || z.hi);
  }
  __device__ __forceinline__ void load(const AdjArgs<T>& a, int i, uint32_t pc) {
    const uint32_t plane = (uint32_t)(a.d.ny * a.d.nz);
    any_x = i < t0 || i >= a.d.nx - t1;
    if (any_x) {
      x.locate(i, a.d.nx, t0, t1, plane, [&](int l, int) { return (uint32_t)l * plane + pc; });
      x.load(sides);
    }
    if (any_y) y.load(sides + 2);
    if (any_z) z.load(sides + 4);
  }
  // to the next plane (H marches up, E down)
  __device__ __forceinline__ void next_plane() {
    y.q = IS_H ? y.q + y.step : y.q - y.step;
    z.q = IS_H ? z.q + z.step : z.q - z.step;
  }
};

// The transposed half steps where no slabs overlap: the general forms' sums in
// their order, with a plane's psi and coefficients loaded with its fields and
// 32-bit offsets, as in the main kernels (the general forms walk the six sides
// one after another, each a chain of table, psi and profile loads). Work-items
// past the plane's edge do the last cell's work in lockstep (main_E_tile).
// Bound by the memory latency of a plane's one round trip at 4 waves a SIMD (97
// and 113 registers; held to 5 waves they spill, and take 1.5x the time):
// 128x128x64 float32 with slabs of 12 cells, E 20.8 -> 18.2 us a launch, H
// 19.2 -> 17.8. No fewer registers than that in float64: at most 256 threads.
template <typename T>
__global__ void __launch_bounds__(kAdjThreads) k_adj_H(AdjArgs<T> a) {
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, xcd_tile(blockIdx.x, gridDim.x), j, k, i0, i1, act);
  if (!wave_any(act)) return;
  const int ib = max(i0 - 1, 0);  // the offsets count from here
  const int64_t base = (int64_t)ib * d.px, cs = d.cs;
  const uint32_t pc = (uint32_t)(j * d.nz + k), step = (uint32_t)d.px * (uint32_t)sizeof(T);
  uint32_t fo = ((uint32_t)(i0 - ib) * (uint32_t)d.px + pc) * (uint32_t)sizeof(T);
  const uint32_t dk = k > 0 ? (uint32_t)sizeof(T) : 0, dj = j > 0 ? (uint32_t)d.nz * (uint32_t)sizeof(T) : 0;
  const T zero = T(0), sc = a.sc;
  auto ld = [&](const T* p, int c, uint32_t off) { return ld_stream<false>(split_ptr(p + c * cs + base, off)); };
  AdjPml<true, T> pml;
  pml.init(a, i0, j, k);
  T m1p = zero, m2p = zero, l1p = zero, l2p = zero;  // inv_mu and lamH of plane i-1, as loaded
  for (int i = i0; i < i1; ++i, fo += step, pml.next_plane()) {
    opaque(fo);
    if (i == i0) {
      const uint32_t prev = i > 0 ? fo - step : fo;
      m1p = ld(a.inv_mu, 1, prev), m2p = ld(a.inv_mu, 2, prev);
      l1p = ld(a.lamH, 1, prev), l2p = ld(a.lamH, 2, prev);
    }
    const T m0 = ld(a.inv_mu, 0, fo), m1 = ld(a.inv_mu, 1, fo), m2 = ld(a.inv_mu, 2, fo);
    const T l0 = ld(a.lamH, 0, fo), l1 = ld(a.lamH, 1, fo), l2 = ld(a.lamH, 2, fo);
    const T mk0 = ld(a.inv_mu, 0, fo - dk), mk1 = ld(a.inv_mu, 1, fo - dk);
    const T lk0 = ld(a.lamH, 0, fo - dk), lk1 = ld(a.lamH, 1, fo - dk);
    const T mj0 = ld(a.inv_mu, 0, fo - dj), mj2 = ld(a.inv_mu, 2, fo - dj);
    const T lj0 = ld(a.lamH, 0, fo - dj), lj2 = ld(a.lamH, 2, fo - dj);
    T e[3] = {ld(a.lamE, 0, fo), ld(a.lamE, 1, fo), ld(a.lamE, 2, fo)};
    if (a.dcoef) {
      const T d0 = ld(a.dcoef, 0, fo), d1 = ld(a.dcoef, 1, fo), d2 = ld(a.dcoef, 2, fo);
      pml.load(a, i, pc);
      e[0] = d0 * e[0];
      e[1] = d1 * e[1];
      e[2] = d2 * e[2];
    } else {
      pml.load(a, i, pc);
    }
    const T y0 = (sc * m0) * l0, y1 = (sc * m1) * l1, y2 = (sc * m2) * l2;
    const T yz_prev = (sc * m2p) * l2p, yy_prev = (sc * m1p) * l1p;  // Y at plane i-1
    const T yy_km = (sc * mk1) * lk1, yx_km = (sc * mk0) * lk0, yz_jm = (sc * mj2) * lj2, yx_jm = (sc * mj0) * lj0;
    const bool km = k >= 1, kp = k <= d.nz - 2, jm = j >= 1, jp = j <= d.ny - 2, im = i >= 1, ip = i <= d.nx - 2;
    e[0] = e[0] - (((km ? yy_km : zero) - (kp ? y1 : zero)) - ((jm ? yz_jm : zero) - (jp ? y2 : zero)));
    e[1] = e[1] - (((im ? yz_prev : zero) - (ip ? y2 : zero)) - ((km ? yx_km : zero) - (kp ? y0 : zero)));
    e[2] = e[2] - (((jm ? yx_jm : zero) - (jp ? y0 : zero)) - ((im ? yy_prev : zero) - (ip ? y1 : zero)));
    if (pml.any_x) pml.x.template apply<0>(pml.sides, y1, y2, yy_prev, yz_prev, e);
    if (pml.any_y) pml.y.template apply<1>(pml.sides + 2, y0, y2, yx_jm, yz_jm, e);
    if (pml.any_z) pml.z.template apply<2>(pml.sides + 4, y0, y1, yx_km, yy_km, e);
    const int64_t pp = box_index(a.pb, i, j, k);
    if (wave_any(pp >= 0) && pp >= 0) {
      const int64_t np = box_cells(a.pb);
#pragma unroll
      for (int c = 0; c < 3; ++c) e[c] = e[c] + T(2) * gp(a.plane)[c * np + pp];
    }
    opaque(fo);
#pragma unroll
    for (int c = 0; c < 3; ++c) st_stream<false>(split_ptr(a.lamE + c * cs + base, fo), e[c]);
    m1p = m1, m2p = m2, l1p = l1, l2p = l2;
  }
}

template <typename T, bool YB>
__global__ void __launch_bounds__(kAdjThreads) k_adj_E(AdjArgs<T> a) {
  const Dims d = a.d;
  int j, k, i0, i1;
  bool act;
  tile_column(a, gridDim.x - 1 - xcd_tile(blockIdx.x, gridDim.x), j, k, i0, i1, act);
  if (!wave_any(act)) return;
  const int64_t base = (int64_t)i0 * d.px, cs = d.cs;  // the offsets count from here
  const uint32_t pc = (uint32_t)(j * d.nz + k), step = (uint32_t)d.px * (uint32_t)sizeof(T);
  uint32_t fo = ((uint32_t)(i1 - 1 - i0) * (uint32_t)d.px + pc) * (uint32_t)sizeof(T);
  const uint32_t dk = k < d.nz - 1 ? (uint32_t)sizeof(T) : 0,
                 dj = j < d.ny - 1 ? (uint32_t)d.nz * (uint32_t)sizeof(T) : 0;
  const T zero = T(0), sc = a.sc;
  const T* const fac = YB ? a.ybuf : a.gcoef;  // Y, or gcoef (Y = gcoef lamE)
  auto ld = [&](const T* p, int c, uint32_t off) { return ld_stream<false>(split_ptr(p + c * cs + base, off)); };
  auto Y = [&](T f, T l) { return YB ? f : f * l; };
  AdjPml<false, T> pml;
  pml.init(a, i1 - 1, j, k);
  T l1n = zero, l2n = zero, f1n = zero, f2n = zero;  // plane i+1, as loaded
  for (int i = i1 - 1; i >= i0; --i, fo -= step, pml.next_plane()) {
    opaque(fo);
    const uint32_t next = i < d.nx - 1 ? fo + step : fo;
    if (i == i1 - 1) {
      l1n = ld(a.lamE, 1, next), l2n = ld(a.lamE, 2, next);
      f1n = ld(fac, 1, next), f2n = ld(fac, 2, next);
    }
    const T l0 = ld(a.lamE, 0, fo), l1 = ld(a.lamE, 1, fo), l2 = ld(a.lamE, 2, fo);
    const T lk0 = ld(a.lamE, 0, fo + dk), lk1 = ld(a.lamE, 1, fo + dk);
    const T lj0 = ld(a.lamE, 0, fo + dj), lj2 = ld(a.lamE, 2, fo + dj);
    const T f0 = ld(fac, 0, fo), f1 = ld(fac, 1, fo), f2 = ld(fac, 2, fo);
    const T fk0 = ld(fac, 0, fo + dk), fk1 = ld(fac, 1, fo + dk), fj0 = ld(fac, 0, fo + dj), fj2 = ld(fac, 2, fo + dj);
    T h[3] = {ld(a.lamH, 0, fo), ld(a.lamH, 1, fo), ld(a.lamH, 2, fo)};
    pml.load(a, i, pc);
    // the grid's 1/eps where a face weighs lamE with it
    T g[3] = {zero, zero, zero}, gx1 = zero, gx2 = zero, gy0 = zero, gy2 = zero, gz0 = zero, gz1 = zero;
    if (pml.any_x || pml.any_y || pml.any_z) {
#pragma unroll
      for (int c = 0; c < 3; ++c) g[c] = ld(a.inv_eps, c, fo);
      if (pml.any_x) gx1 = ld(a.inv_eps, 1, next), gx2 = ld(a.inv_eps, 2, next);
      if (pml.any_y) gy0 = ld(a.inv_eps, 0, fo + dj), gy2 = ld(a.inv_eps, 2, fo + dj);
      if (pml.any_z) gz0 = ld(a.inv_eps, 0, fo + dk), gz1 = ld(a.inv_eps, 1, fo + dk);
    }
    const int64_t pd = box_index(a.db, i, j, k), nd = box_cells(a.db);
    const bool design = wave_any(pd >= 0);
    double gr[3] = {0.0, 0.0, 0.0};
    T cu[3] = {zero, zero, zero};
    if (design && pd >= 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        gr[c] = gp(a.grad)[c * nd + pd];
        cu[c] = gp(a.curl)[c * nd + pd];
      }
    }
    const T y0 = Y(f0, l0), y1 = Y(f1, l1), y2 = Y(f2, l2);
    const T yz_next = Y(f2n, l2n), yy_next = Y(f1n, l1n);  // Y at plane i+1
    const T yy_kp = Y(fk1, lk1), yx_kp = Y(fk0, lk0), yz_jp = Y(fj2, lj2), yx_jp = Y(fj0, lj0);
    const bool km = k >= 1, kp = k <= d.nz - 2, jm = j >= 1, jp = j <= d.ny - 2, im = i >= 1, ip = i <= d.nx - 2;
    h[0] = h[0] + (((km ? y1 : zero) - (kp ? yy_kp : zero)) - ((jm ? y2 : zero) - (jp ? yz_jp : zero)));
    h[1] = h[1] + (((im ? y2 : zero) - (ip ? yz_next : zero)) - ((km ? y0 : zero) - (kp ? yx_kp : zero)));
    h[2] = h[2] + (((jm ? y0 : zero) - (jp ? yx_jp : zero)) - ((im ? y1 : zero) - (ip ? yy_next : zero)));
    if (pml.any_x)
      pml.x.template apply<0>(pml.sides, (sc * g[1]) * l1, (sc * g[2]) * l2, (sc * gx1) * l1n, (sc * gx2) * l2n, h);
    if (pml.any_y)
      pml.y.template apply<1>(pml.sides + 2, (sc * g[0]) * l0, (sc * g[2]) * l2, (sc * gy0) * lj0, (sc * gy2) * lj2, h);
    if (pml.any_z)
      pml.z.template apply<2>(pml.sides + 4, (sc * g[0]) * l0, (sc * g[1]) * l1, (sc * gz0) * lk0, (sc * gz1) * lk1, h);
    opaque(fo);
#pragma unroll
    for (int c = 0; c < 3; ++c) st_stream<false>(split_ptr(a.lamH + c * cs + base, fo), h[c]);
    if (design && pd >= 0) {
      const T le[3] = {l0, l1, l2};
#pragma unroll
      for (int c = 0; c < 3; ++c) gp(a.grad)[c * nd + pd] = gr[c] + (double)sc * (double)le[c] * (double)cu[c];
    }
    l1n = l1, l2n = l2, f1n = f1, f2n = f2;
  }
}

}  // namespace fdtd_dev
