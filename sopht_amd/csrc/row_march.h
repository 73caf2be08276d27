// Row-vector columns for the standalone grid operators on gfx950.
//
// A thread owns a 16-byte vector of V neighbouring cells of one row (V = 4 FP32, 2 FP64) and
// walks a chunk of z planes; the z neighbours stay in registers and the x neighbours come from
// the adjacent lanes. The vectors of a plane are dealt to the threads in row order without
// gaps, so any row length keeps every lane busy: 170 cells are 43 vectors, and the next row
// starts at the next lane. The last vector of a row ends at the row's last cell; where the row
// length is no multiple of V it overlaps its neighbour by `skip` cells, which it computes but
// does not store. Rows need no alignment beyond the element's: gfx950 loads 16 bytes from any
// 4-byte address.
#pragma once

#include <cstdlib>

#include "common.h"

namespace sopht {
namespace {

constexpr int kRowThreads = 256;

template <typename T>
struct RowVec {
  static constexpr int V = 16 / int(sizeof(T));
  static constexpr unsigned kAll = (1u << V) - 1u;
  typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};
template <typename T>
using rvec = typename RowVec<T>::type;

template <typename T>
__device__ __forceinline__ rvec<T> rload(const T* p) {
  return *reinterpret_cast<const rvec<T>*>(p);
}
// Stores the vector's cells whose bit is set.
template <typename T>
__device__ __forceinline__ void rstore(T* p, rvec<T> v, unsigned mask) {
  if (mask == RowVec<T>::kAll) {
    *reinterpret_cast<rvec<T>*>(p) = v;
  } else {
#pragma unroll
    for (int k = 0; k < RowVec<T>::V; ++k)
      if (mask >> k & 1u) p[k] = v[k];
  }
}

// The value of the previous / next lane of the wavefront (0 at its ends): a DPP move, which
// needs no LDS traffic. Every lane of the wavefront must call it.
template <int CTRL>
__device__ __forceinline__ float lane_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double lane_shift(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
template <typename T>
__device__ __forceinline__ T from_prev_lane(T v) { return lane_shift<0x138>(v); }  // wave_shr:1
template <typename T>
__device__ __forceinline__ T from_next_lane(T v) { return lane_shift<0x130>(v); }  // wave_shl:1

// Element strides of the rows and planes of a field whose cells are adjacent along x.
struct RowStrides {
  int y, z;
};

struct RowGeo {
  int nz, ny, nx;
  int nv;      // vectors per row
  int tiles;   // workgroups per chunk of planes
  int chunk;   // planes per workgroup
};

// The column of this thread. Threads past the last column repeat it (act = false), so that
// every lane takes part in the lane shifts.
template <typename T>
struct RowCol {
  static constexpr int V = RowVec<T>::V;
  int x, y, ym, yp, z0, z1;
  bool yin;            // the row is inside in y
  bool edge_l, edge_r; // the adjacent lane does not hold the adjacent vector
  unsigned own, inner; // cells to store; those inside in x
  int nx;

  __device__ __forceinline__ RowCol(const RowGeo& g) {
    // contiguous runs of workgroups per XCD, so that rows shared by neighbouring workgroups
    // meet in one L2 (workgroup b runs on XCD b mod 8)
    const int total = int(gridDim.x), per = total / 8, more = total % 8;
    const int xcd = int(blockIdx.x) % 8;
    const int item = xcd * per + (xcd < more ? xcd : more) + int(blockIdx.x) / 8;
    const int tile = item % g.tiles;
    z0 = (item / g.tiles) * g.chunk;
    z1 = z0 + g.chunk < g.nz ? z0 + g.chunk : g.nz;
    int col = tile * kRowThreads + int(threadIdx.x);
    const int cols = g.nv * g.ny;
    const bool act = col < cols;
    col = act ? col : cols - 1;
    y = col / g.nv;
    const int xv = col - y * g.nv;
    nx = g.nx;
    x = xv * V < nx - V ? xv * V : nx - V;
    const int skip = xv * V - x;
    yin = y > 0 && y < g.ny - 1;
    ym = y > 0 ? y - 1 : 0;
    yp = y < g.ny - 1 ? y + 1 : y;
    const int lane = int(threadIdx.x) & 63;
    edge_l = lane == 0 || skip != 0 || !act;
    edge_r = lane == 63 || x + 2 * V > nx || !act;
    own = act ? (RowVec<T>::kAll >> skip) << skip : 0u;
    inner = 0;
#pragma unroll
    for (int k = 0; k < V; ++k) inner |= (x + k > 0 && x + k < nx - 1) ? 1u << k : 0u;
  }
  // The cells left and right of the vector v read from row (row points at the field's cell
  // x = 0); unspecified outside the grid.
  __device__ __forceinline__ void nbrs(rvec<T> v, const T* row, T& left, T& right) const {
    left = from_prev_lane(v[V - 1]);
    right = from_next_lane(v[0]);
    if (edge_l && x > 0) left = row[x - 1];
    if (edge_r && x + V < nx) right = row[x + V];
  }
};

// Workgroups for the columns of an (nz, ny, nx) box. Chunks start at `most` planes and are
// halved (down to 2) while there are fewer than four workgroups per CU: a chunk's first planes
// are read again by the one below it, which costs less than idle CUs.
template <typename T>
inline RowGeo row_geo(int64_t nz, int64_t ny, int64_t nx, int most) {
  RowGeo g;
  g.nz = int(nz);
  g.ny = int(ny);
  g.nx = int(nx);
  g.nv = ceil_div(nx, RowVec<T>::V);
  g.tiles = ceil_div(int64_t(g.nv) * ny, kRowThreads);
  g.chunk = most;
  while (g.chunk > 2 && int64_t(g.tiles) * ceil_div(nz, g.chunk) < 1024) g.chunk /= 2;
  return g;
}
inline unsigned row_blocks(const RowGeo& g) { return unsigned(int64_t(g.tiles) * ceil_div(g.nz, g.chunk)); }

// Whether the row-vector kernels take a field: cells adjacent along x, non-negative row and
// plane strides, 32-bit offsets, and rows of at least one vector.
inline bool row_strides_ok(const int64_t* s, int64_t nz, int64_t ny, int64_t nx) {
  constexpr int64_t lim = int64_t(1) << 31;
  return s[2] == 1 && s[0] >= 0 && s[1] >= 0 && s[0] < lim && s[1] < lim &&
         (nz - 1) * s[0] + (ny - 1) * s[1] + nx < lim;
}
template <typename T>
inline bool row_box_ok(int64_t nz, int64_t ny, int64_t nx) {
  constexpr int64_t lim = int64_t(1) << 31;
  return nx >= RowVec<T>::V && nz < lim && ny < lim && nx < lim &&
         ceil_div(nx, RowVec<T>::V) * ny < lim - kRowThreads &&
         int64_t(ceil_div(int64_t(ceil_div(nx, RowVec<T>::V)) * ny, kRowThreads)) * ceil_div(nz, 2) < lim;
}
inline RowStrides row_strides(const int64_t* s) { return RowStrides{int(s[1]), int(s[0])}; }

// Whether the memory spanned by two fields of one box (strides >= 0) meets.
template <typename T>
inline bool fields_meet(const void* a, const int64_t* as, const void* b, const int64_t* bs, int64_t nz,
                        int64_t ny, int64_t nx) {
  auto span = [&](const int64_t* s) {
    return uintptr_t((nz - 1) * s[0] + (ny - 1) * s[1] + (nx - 1) * s[2] + 1) * sizeof(T);
  };
  const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
  return pa < pb + span(bs) && pb < pa + span(as);
}

// ------------------------------------------------------------------ vorticity stretching

template <typename T>
struct Rows3 {
  T* p[3];
  RowStrides s;
};
template <typename T>
inline Rows3<T> rows3(void* const p[3], const int64_t* s) {
  return Rows3<T>{{static_cast<T*>(p[0]), static_cast<T*>(p[1]), static_cast<T*>(p[2])}, row_strides(s)};
}
template <typename T>
inline Rows3<const T> rows3(const void* const p[3], const int64_t* s) {
  return Rows3<const T>{{static_cast<const T*>(p[0]), static_cast<const T*>(p[1]), static_cast<const T*>(p[2])},
                        row_strides(s)};
}

// Vorticity stretching flux p (w . grad) u, and the time steps built on it
// (vorticity_stretching_flux_3d.py:13-107, vorticity_stretching_timestep_3d.py:10-158).
// The flux takes the vorticity at its own cell only, so a whole time step is pointwise in w:
// the velocity differences are formed once and the stages run in registers. SCHEME 0 writes
// the flux, 1 (Euler) also w + flux, 2 (SSPRK3) runs the three stages and leaves the last
// stage's flux and the mid-step field as the sequence of separate kernels does. Bound by memory: an SSPRK3 step moves 15
// words per cell (6 in, 9 out) where the sequence of 3 fluxes, 3 sums and 2 axpbys with their
// border launches moved 72. 130 x 170 x 250 FP32: one SSPRK3
// step in 62 us (5.3 TB/s) against 562 us for the sequence of kernels.
template <typename T, int SCHEME>
__global__ void __launch_bounds__(kRowThreads)
    k_stretch_rows(RowGeo g, Rows3<const T> u, Rows3<const T> w, Rows3<T> wout, Rows3<T> flux, Rows3<T> mid,
                   T p, T p_last) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T> c(g);
  const int ur = c.y * u.s.y, urm = c.ym * u.s.y, urp = c.yp * u.s.y;
  vec um[3], uc[3];
  {
    const int zm = c.z0 > 0 ? c.z0 - 1 : 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      um[a] = rload(u.p[a] + zm * u.s.z + ur + c.x);
      uc[a] = rload(u.p[a] + c.z0 * u.s.z + ur + c.x);
    }
  }
  for (int z = c.z0; z < c.z1; ++z) {
    const int zp = z < g.nz - 1 ? z + 1 : z;
    vec wv[3], up[3], grad[3][3];  // grad[a][axis]: difference of u_a along x, y, z
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const T* ua = u.p[a] + z * u.s.z;
      up[a] = rload(u.p[a] + zp * u.s.z + ur + c.x);
      wv[a] = rload(w.p[a] + z * w.s.z + c.y * w.s.y + c.x);
      grad[a][1] = rload(ua + urp + c.x) - rload(ua + urm + c.x);
      grad[a][2] = up[a] - um[a];
      T left, right;
      c.nbrs(uc[a], ua + ur, left, right);
#pragma unroll
      for (int k = 0; k < V; ++k)
        grad[a][0][k] = (k < V - 1 ? uc[a][k < V - 1 ? k + 1 : k] : right) - (k > 0 ? uc[a][k > 0 ? k - 1 : k] : left);
    }
    const bool zin = c.yin && z > 0 && z < g.nz - 1;
    auto stage = [&](const vec* v, T q, vec* f) {
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int k = 0; k < V; ++k) {
          const T r = q * (v[0][k] * grad[a][0][k] + v[1][k] * grad[a][1][k] + v[2][k] * grad[a][2][k]);
          f[a][k] = zin && (c.inner >> k & 1u) ? r : T(0);
        }
    };
    vec f[3], m[3], o[3];
    stage(wv, p, f);
    if constexpr (SCHEME >= 1)
#pragma unroll
      for (int a = 0; a < 3; ++a) o[a] = m[a] = wv[a] + f[a];
    if constexpr (SCHEME == 2) {
      stage(m, p, f);
#pragma unroll
      for (int a = 0; a < 3; ++a) m[a] = T(0.75) * wv[a] + T(0.25) * (m[a] + f[a]);
      stage(m, p_last, f);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        m[a] = m[a] + f[a];
        o[a] = T(1.0 / 3.0) * wv[a] + T(2.0 / 3.0) * m[a];
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      rstore(flux.p[a] + z * flux.s.z + c.y * flux.s.y + c.x, f[a], c.own);
      if constexpr (SCHEME >= 1) rstore(wout.p[a] + z * wout.s.z + c.y * wout.s.y + c.x, o[a], c.own);
      if constexpr (SCHEME == 2) rstore(mid.p[a] + z * mid.s.z + c.y * mid.s.y + c.x, m[a], c.own);
      um[a] = uc[a];
      uc[a] = up[a];
    }
  }
}

}  // namespace
}  // namespace sopht
