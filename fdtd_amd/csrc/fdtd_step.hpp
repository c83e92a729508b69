// Whole-step kernel of libfdtd_hip: the E and the H half step of one time
// step in one sweep over the grid (k_step), for grids without anything
// between the two half steps that needs the finished E field.
#pragma once

#include "fdtd_kernels.hpp"

// Local data share. Where a runtime does not model it (host builds that run a
// workgroup's work-items one after another) a workgroup's array is static.
#if defined(__shared__)
#define FDTD_LDS __shared__
#else
#define FDTD_LDS static
#endif

namespace fdtd_dev {

// Workgroup barrier that orders local memory only. __syncthreads also waits
// for every outstanding global load and store, which would drain a marching
// kernel's memory queue once per plane; the planes exchanged through the LDS
// need the LDS accesses ordered and nothing else.
__device__ __forceinline__ void lds_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#else
  __syncthreads();
#endif
}

// The CPML faces of a whole step by side (2 * axis + high), among the kernel's
// arguments: a work-item selects its side's addresses, where a table in memory
// would be one more load to wait for before the psi loads (60x52x44 float64
// 14.1 -> 12.6 us a step, 200x200x1 5.86 -> 5.73). psiE is read from
// one buffer and written to another (neighbouring workgroups recompute E, and
// so psiE, on their halo cells from the values before the step); psiH belongs
// to one cell and is updated in place. Both are (2, slab) values.
struct StepSides {
  const void* psiE_in[6];
  void* psiE_out[6];
  void* psiH[6];
  const double* coef[6];  // bE, cE, bH, cH, t values each
  int32_t t[6];           // thickness, 0: no face
  int32_t slab[6];        // cells
};

// A source added inside the step: its cells' bounding box, and for a line its
// cells in ascending order with their profile values.
struct StepSrc {
  int32_t kind, compE, compH, n;
  int32_t dense, pad;  // the cells are all of the box
  Box box;
  const int64_t* cells;
  const double* profile;
  double amplitude;
};

// A detector sampled inside the step: its cells in ascending order and the
// position of each in the detector's own order.
struct StepDet {
  int32_t n, dense;
  Box box;
  const int64_t* cells;
  const int32_t* order;
  void* bufE;
  void* bufH;
  int64_t slot0E, slot0H;
};

// Value v of component c of e, chosen with selects.
template <typename T>
__device__ __forceinline__ T pick(const T e[3], int c) {
  return c == 0 ? e[0] : (c == 1 ? e[1] : e[2]);
}
template <typename T>
__device__ __forceinline__ void put(T e[3], int c, T v) {
  e[0] = c == 0 ? v : e[0];
  e[1] = c == 1 ? v : e[1];
  e[2] = c == 2 ? v : e[2];
}

__device__ __forceinline__ bool in_box(cptr<Box> b, int i, int j, int k) {
  return i >= b->x0 && i < b->x1 && j >= b->y0 && j < b->y1 && k >= b->z0 && k < b->z1;
}

__device__ __forceinline__ int dense_index(cptr<Box> b, int i, int j, int k) {
  return ((i - b->x0) * (b->y1 - b->y0) + (j - b->y0)) * (b->z1 - b->z0) + (k - b->z0);
}

// Index of `cell` in the ascending list cells[0..n), or -1.
__device__ __forceinline__ int find_cell(const int64_t* cells, int n, int64_t cell) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (gp(cells)[mid] < cell) lo = mid + 1;
    else hi = mid;
  }
  return lo < n && gp(cells)[lo] == cell ? lo : -1;
}

template <class FS, class MS>
struct StepArgs {
  using R = typename FS::R;
  Dims d;
  R sc;
  FS E, E2, H, H2;  // fields before (E, H) and after (E2, H2) the step
  MS Me, Mu;
  // CPML: at most one face a side, and the order in which a cell's faces are
  // applied: axis 1, 2 and 3 of the order in two bits each
  StepSides sides;
  int32_t order;
  const ObjDev* objs;
  int32_t nobjs;
  int32_t tx, ty, tz, ntx, nty, ntz;  // own cells of a tile, tiles along each axis
  Divide tiles_yz, tiles_z, cells_yz, cells_z, cells_y;  // by nty * ntz, ntz, ty * tz, tz, ty
  int32_t nsrc, ndet;
  int32_t folded;  // point sources join the E update before it is stored
  const StepSrc* srcs;
  const StepDet* dets;
  const double* wave;
  int64_t wave_cap;
  int64_t q;
  int64_t nE, nH;  // half steps already taken (the detectors' clocks)
};

// The CPML face normal to one axis at a cell: the side whose slab holds it
// (-1: none), its place there and what was loaded for it.
template <int AX, typename T>
struct StepAxis {
  int side = -1, l;
  bool e_in, h_in;  // the slab holds both cells of the E and the H difference
  uint32_t at, at1;  // the cell's places in the psi arrays
  T bE, cE, bH, cH;
  Psi<T> e, h;
  // of the axis's two sides, the one the cell is in
  template <typename V>
  __device__ __forceinline__ V mine(const V* by_side) const {
    const V lo = by_side[2 * AX], hi = by_side[2 * AX + 1];
    return side == 2 * AX ? lo : hi;
  }
  // g: the cell's index along the axis of n cells; cells(l, t): its place in a
  // slab of thickness t
  template <class Cells>
  __device__ __forceinline__ void load(const StepSides& s, int g, int n, bool own, Cells&& cells) {
    const int tl = s.t[2 * AX], th = s.t[2 * AX + 1];
    if (g < tl) {
      side = 2 * AX;
      l = g;
    } else if (g >= n - th) {
      side = 2 * AX + 1;
      l = g - (n - th);
    } else {
      return;
    }
    const int t = mine(s.t);
    e_in = l >= 1;
    h_in = l <= t - 2;
    at = (uint32_t)cells(l, t);
    at1 = at + (uint32_t)mine(s.slab);
    const gptr<const T> pe = gp(static_cast<const T*>(mine(s.psiE_in)));
    const gptr<const double> cf = gp(mine(s.coef)) + l;
    e.p0 = pe[at];
    e.p1 = pe[at1];
    bE = (T)cf[0];
    cE = (T)cf[t];
    if (!own) return;
    const gptr<const T> ph = gp(static_cast<const T*>(mine(s.psiH)));
    h.p0 = ph[at];
    h.p1 = ph[at1];
    bH = (T)cf[2 * t];
    cH = (T)cf[3 * t];
  }
  __device__ __forceinline__ void store(const StepSides& s) const {
    if (side < 0) return;
    const gptr<T> pe = gp(static_cast<T*>(mine(s.psiE_out))), ph = gp(static_cast<T*>(mine(s.psiH)));
    pe[at] = e.p0;
    pe[at1] = e.p1;
    ph[at] = h.p0;
    ph[at1] = h.p1;
  }
};

// One whole step of a tile of tx*ty*tz cells, one cell per work-item. The H
// half step of the tile's cells reads the finished E of the cells one further
// along each axis, so a workgroup also computes E on those halo cells (one
// work-item each, nothing of theirs is stored) and hands E over through the
// LDS. The fields are read from one set of buffers and written to another,
// because the neighbouring workgroups read this one's cells as they were.
//
// For grids of which a launch is over in a few microseconds, where a step's
// time is its launches and the chain of dependent loads in each: every load
// of a cell (fields, materials, CPML state and coefficients of both half
// steps) is issued at once, and there is one barrier.
constexpr int kStepThreads = 256;

template <class FS, class MS, typename O, bool OBJS>
__global__ void __launch_bounds__(kStepThreads) k_step(StepArgs<FS, MS> a) {
  using T = typename FS::R;
  using Sample = typename FS::Sample;
  // bytes, because complex values have a constructor
  FDTD_LDS __align__(16) unsigned char lds_bytes[3 * kStepThreads * sizeof(T)];
  T(*const lds)[kStepThreads] = reinterpret_cast<T(*)[kStepThreads]>(lds_bytes);
  const Dims d = a.d;
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  const unsigned nx = a.tiles_yz.of(tile), nxy = a.tiles_z.of(tile);  // x slabs and z rows of tiles before this one
  const int i0 = (int)nx * a.tx, j0 = (int)(nxy - nx * (unsigned)a.nty) * a.ty,
            k0 = (int)(tile - nxy * (unsigned)a.ntz) * a.tz;
  // this work-item's cell: the tile's own cells z fastest, then the halo cells
  // past its last x plane, y row and z column
  const int tid = (int)threadIdx.x, tx = a.tx, ty = a.ty, tz = a.tz, yz = ty * tz;
  // an axis with one tile has no halo
  const int bx = tx * yz, by = bx + (a.ntx > 1 ? yz : 0), bz = by + (a.nty > 1 ? tx * tz : 0),
            end = bz + (a.ntz > 1 ? tx * ty : 0);
  int ii = 0, jj = 0, kk = 0;
  if (tid < by) {
    ii = (int)a.cells_yz.of(tid);
    const int r = tid - ii * yz;
    jj = (int)a.cells_z.of(r);
    kk = r - jj * tz;
  } else if (tid < bz) {
    ii = (int)a.cells_z.of(tid - by);
    jj = ty;
    kk = tid - by - ii * tz;
  } else if (tid < end) {
    ii = (int)a.cells_y.of(tid - bz);
    jj = tid - bz - ii * ty;
    kk = tz;
  }
  const bool live = tid < end && i0 + ii < d.nx && j0 + jj < d.ny && k0 + kk < d.nz, own = live && tid < bx;
  // work-items without a cell read the nearest one
  const int i = min(i0 + ii, d.nx - 1), j = min(j0 + jj, d.ny - 1), k = min(k0 + kk, d.nz - 1);
  const int64_t cell = cell_of(d, i, j, k);
  const uint32_t c32 = (uint32_t)cell, fo = c32 * FS::kCell, mo = c32 * MS::kCell;
  // every load of the cell at once
  const typename FS::Own hown = a.H.template own<false>(0, fo);
  const typename FS::Duo hk = a.H.template duo<0, 1>(0, k > 0 ? fo - FS::kCell : fo);
  const typename FS::Duo hj = a.H.template duo<0, 2>(0, j > 0 ? fo - (uint32_t)d.nz * FS::kCell : fo);
  const typename FS::Duo hi = a.H.template duo<1, 2>(0, i > 0 ? fo - (uint32_t)d.px * FS::kCell : fo);
  const typename MS::Own meps = a.Me.template own<false>(0, mo);
  const typename FS::Own eown = a.E.template own<false>(0, fo);
  const typename MS::Own mmu = a.Mu.template own<false>(0, mo);
  StepAxis<0, T> ax;
  StepAxis<1, T> ay;
  StepAxis<2, T> az;
  ax.load(a.sides, i, d.nx, own, [&](int l, int) { return (l * d.ny + j) * d.nz + k; });
  ay.load(a.sides, j, d.ny, own, [&](int l, int t) { return (i * t + l) * d.nz + k; });
  az.load(a.sides, k, d.nz, own, [&](int l, int t) { return (i * d.ny + j) * t + l; });
  const T zero = T(0);
  // E half step; backward differences, an absent one contributes nothing (grid.py:67-74)
  const T h0 = FS::template value<0>(hown), h1 = FS::template value<1>(hown), h2 = FS::template value<2>(hown);
  Diffs<T> df;
  df.zy = j > 0 ? h2 - FS::template value<0, 2, 2>(hj) : zero;
  df.yz = k > 0 ? h1 - FS::template value<0, 1, 1>(hk) : zero;
  df.xz = k > 0 ? h0 - FS::template value<0, 1, 0>(hk) : zero;
  df.zx = i > 0 ? h2 - FS::template value<1, 2, 2>(hi) : zero;
  df.yx = i > 0 ? h1 - FS::template value<1, 2, 1>(hi) : zero;
  df.xy = j > 0 ? h0 - FS::template value<0, 2, 0>(hj) : zero;
  T e[3] = {FS::template value<0>(eown), FS::template value<1>(eown), FS::template value<2>(eown)};
  T m[3], curl[3], kc[3];
  a.Me.values(meps, m);
  curl[0] = (zero + df.zy) - df.yz;
  curl[1] = (zero + df.xz) - df.zx;
  curl[2] = (zero + df.yx) - df.xy;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    kc[c] = a.sc * m[c];
    e[c] = e[c] + kc[c] * curl[c];
  }
  if (OBJS) objects_update_E<T, O>(a.objs, a.nobjs, a.sc, i, j, k, curl, e);
#pragma nounroll
  for (int n = 0; n < 3; ++n) {
    const int axis = (a.order >> (2 * n)) & 3;
    if (axis == 0 && ax.side >= 0) {
      ax.e.advance(ax.bE, ax.cE, ax.e_in, df.zx, df.yx);
      e[1] = e[1] - kc[1] * ax.e.p0;
      e[2] = e[2] + kc[2] * ax.e.p1;
    } else if (axis == 1 && ay.side >= 0) {
      ay.e.advance(ay.bE, ay.cE, ay.e_in, df.zy, df.xy);
      e[0] = e[0] + kc[0] * ay.e.p0;
      e[2] = e[2] - kc[2] * ay.e.p1;
    } else if (axis == 2 && az.side >= 0) {
      az.e.advance(az.bE, az.cE, az.e_in, df.yz, df.xz);
      e[0] = e[0] - kc[0] * az.e.p0;
      e[1] = e[1] + kc[1] * az.e.p1;
    }
  }
  for (int s = 0; s < a.nsrc; ++s) {
    const cptr<StepSrc> src = cp(a.srcs) + s;
    if (!in_box(&src->box, i, j, k)) continue;
    const int p = src->dense ? dense_index(&src->box, i, j, k) : find_cell(src->cells, src->n, cell);
    if (p < 0) continue;
    const T w = (T)cp(a.wave)[s * a.wave_cap + a.q];
    T v = pick(e, src->compE);
    if (!a.folded) v = FS::rounded(v);
    if (src->kind == FDTD_SRC_POINT) v = v + w;
    else if (src->kind == FDTD_SRC_LINE) v = v + (T)gp(src->profile)[p] * w;
    else v = (T)src->amplitude * w;
    put(e, src->compE, v);
  }
  // the H half step reads the E that is stored
#pragma unroll
  for (int c = 0; c < 3; ++c) e[c] = FS::rounded(e[c]);
#pragma unroll
  for (int c = 0; c < 3; ++c) lds[c][tid] = e[c];
  lds_barrier();
  if (!own) return;
  a.E2.template put_own<false>(0, fo, e);
  // H half step; forward differences (grid.py:42-49). Past the grid's edge
  // the neighbour is not read: its value is this cell's.
  const int sk = k < d.nz - 1 ? (kk + 1 < tz ? tid + 1 : bz + ii * ty + jj) : tid;
  const int sj = j < d.ny - 1 ? (jj + 1 < ty ? tid + tz : by + ii * tz + kk) : tid;
  const int si = i < d.nx - 1 ? tid + yz : tid;  // the x halo follows the tile's last plane
  const T ex_kp = lds[0][sk], ey_kp = lds[1][sk], ex_jp = lds[0][sj], ez_jp = lds[2][sj], ey_ip = lds[1][si],
          ez_ip = lds[2][si];
  Diffs<T> dh;
  dh.zy = j < d.ny - 1 ? ez_jp - e[2] : zero;
  dh.yz = k < d.nz - 1 ? ey_kp - e[1] : zero;
  dh.xz = k < d.nz - 1 ? ex_kp - e[0] : zero;
  dh.zx = i < d.nx - 1 ? ez_ip - e[2] : zero;
  dh.yx = i < d.nx - 1 ? ey_ip - e[1] : zero;
  dh.xy = j < d.ny - 1 ? ex_jp - e[0] : zero;
  T ch[3], h[3] = {h0, h1, h2};
  a.Mu.values(mmu, m);
  ch[0] = (zero + dh.zy) - dh.yz;
  ch[1] = (zero + dh.xz) - dh.zx;
  ch[2] = (zero + dh.yx) - dh.xy;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    kc[c] = a.sc * m[c];
    h[c] = h[c] - kc[c] * ch[c];
  }
#pragma nounroll
  for (int n = 0; n < 3; ++n) {
    const int axis = (a.order >> (2 * n)) & 3;
    if (axis == 0 && ax.side >= 0) {
      ax.h.advance(ax.bH, ax.cH, ax.h_in, dh.zx, dh.yx);
      h[1] = h[1] + kc[1] * ax.h.p0;
      h[2] = h[2] - kc[2] * ax.h.p1;
    } else if (axis == 1 && ay.side >= 0) {
      ay.h.advance(ay.bH, ay.cH, ay.h_in, dh.zy, dh.xy);
      h[0] = h[0] - kc[0] * ay.h.p0;
      h[2] = h[2] + kc[2] * ay.h.p1;
    } else if (axis == 2 && az.side >= 0) {
      az.h.advance(az.bH, az.cH, az.h_in, dh.yz, dh.xz);
      h[0] = h[0] + kc[0] * az.h.p0;
      h[1] = h[1] - kc[1] * az.h.p1;
    }
  }
  ax.store(a.sides);
  ay.store(a.sides);
  az.store(a.sides);
  for (int s = 0; s < a.nsrc; ++s) {
    const cptr<StepSrc> src = cp(a.srcs) + s;
    if (src->kind != FDTD_SRC_PLANE || !in_box(&src->box, i, j, k)) continue;
    if (!src->dense && find_cell(src->cells, src->n, cell) < 0) continue;
    put(h, src->compH, (T)src->amplitude * (T)cp(a.wave)[s * a.wave_cap + a.q]);
  }
  a.H2.template put_own<false>(0, fo, h);
  for (int n = 0; n < a.ndet; ++n) {
    const cptr<StepDet> det = cp(a.dets) + n;
    if (!in_box(&det->box, i, j, k)) continue;
    const int p = det->dense ? dense_index(&det->box, i, j, k) : find_cell(det->cells, det->n, cell);
    if (p < 0) continue;
    const int64_t at = gp(det->order)[p];
    Sample* const bE = reinterpret_cast<Sample*>(det->bufE) + ((a.nE - det->slot0E) * det->n + at) * 3;
    Sample* const bH = reinterpret_cast<Sample*>(det->bufH) + ((a.nH - det->slot0H) * det->n + at) * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      st_stream<false>(bE + c, FS::sampled(e[c]));
      st_stream<false>(bH + c, FS::sampled(h[c]));
    }
  }
}

// Copies the fields and psiE of an odd last step back into the plan's arrays:
// n segments of 4-byte words.
struct CopySeg {
  const uint32_t* src;
  uint32_t* dst;
  int64_t words;
};

__global__ void __launch_bounds__(256) k_copy_back(const CopySeg* segs, int n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int s = 0; s < n; ++s) {
    const uint32_t* const src = cp(segs)[s].src;
    uint32_t* const dst = cp(segs)[s].dst;
    const int64_t words = cp(segs)[s].words;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += stride) gp(dst)[i] = gp(src)[i];
  }
}

}  // namespace fdtd_dev
