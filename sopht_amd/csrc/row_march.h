// Row-vector columns for the standalone grid operators on gfx950.
//
// A thread owns a 16-byte vector of V neighbouring cells of one row (V = 4 FP32, 2 FP64) and
// walks a chunk of z planes; the z neighbours stay in registers and the x neighbours come from
// the adjacent lanes. The vectors of a plane are dealt to the lanes in row order without gaps,
// so any row length keeps the lanes busy: 170 cells are 43 vectors, and the next row starts at
// the next lane. A wavefront takes 62 vectors; its first and last lane read the vectors beside
// them for their neighbours and store nothing, which replaces scalar loads at its ends.
// Rows need no alignment beyond the element's (gfx950 loads 16 bytes from any 4-byte address).
// Where the row length is no multiple of V, the row's last vector reads up to V - 1 elements
// past the row's end: into the rows behind it, whose values are not used. The last row of the
// last plane has none behind it, and no vector is read there beyond its end: the operators'
// stencils never reach it from a cell they write, and pointwise operands use rload_own.
#pragma once

#include <cstdlib>

#include "common.h"

namespace sopht {
namespace {

// Visit every cell of the box [z0, z0+bz) x [y0, y0+by) x [x0, x0+bx).
template <typename Fn>
__global__ void __launch_bounds__(256) box_kernel(int64_t z0, int64_t y0, int64_t x0, int64_t bz,
                                                  int64_t by, int64_t bx, Fn fn) {
  const int64_t total = bz * by * bx;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t x = i % bx;
    const int64_t t = i / bx;
    const int64_t y = t % by;
    const int64_t z = t / by;
    fn(z0 + z, y0 + y, x0 + x);
  }
}

template <typename Fn>
int launch_box(int64_t z0, int64_t y0, int64_t x0, int64_t bz, int64_t by, int64_t bx, Fn fn,
               hipStream_t s) {
  const int64_t total = bz * by * bx;
  if (total <= 0) return SOPHT_OK;
  int blocks = ceil_div(total, 256);
  if (blocks > 65536) blocks = 65536;
  box_kernel<<<blocks, 256, 0, s>>>(z0, y0, x0, bz, by, bx, fn);
  SOPHT_CHECK_LAUNCH();
  return SOPHT_OK;
}

constexpr int kRowThreads = 256;
constexpr int kRowLanes = 62;  // lanes of a wavefront that own a column

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

// The column of this lane; lanes outside the plane repeat its first or last one and own no
// cell. H is the operator's reach: stencil operands are read around the row yl, which is the
// own row where the operator writes inside values and the nearest such row elsewhere, so that
// every row read exists.
template <typename T, int H>
struct RowCol {
  static constexpr int V = RowVec<T>::V;
  int x, y, yl, z0, z1;
  bool tail;            // the row's vector that holds cells past its end, on the last row
  bool yin;             // rows the operator writes inside values to
  unsigned own, inner;  // cells to store; those inside in x

  __device__ __forceinline__ RowCol(const RowGeo& g) {
    // rows shared by neighbouring workgroups meet in one L2
    const int item = xcd_run(int(gridDim.x), int(blockIdx.x));
    const int tile = item % g.tiles;
    z0 = (item / g.tiles) * g.chunk;
    z1 = z0 + g.chunk < g.nz ? z0 + g.chunk : g.nz;
    const int lane = int(threadIdx.x) & 63;
    int col = (tile * (kRowThreads / 64) + (int(threadIdx.x) >> 6)) * kRowLanes + lane - 1;
    const int cols = g.nv * g.ny;
    const bool act = lane > 0 && lane <= kRowLanes && col < cols;
    col = col < 0 ? 0 : (col < cols ? col : cols - 1);
    y = col / g.nv;
    x = (col - y * g.nv) * V;
    yin = y >= H && y < g.ny - H;
    yl = y < H ? H : (y < g.ny - H ? y : g.ny - H - 1);
    tail = x + V > g.nx && y == g.ny - 1;
    own = inner = 0;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      own |= act && x + k < g.nx ? 1u << k : 0u;
      inner |= x + k >= H && x + k < g.nx - H ? 1u << k : 0u;
    }
  }
};

// A pointwise operand at the lane's own cells of plane z (p points at the first of them).
template <typename T, int H>
__device__ __forceinline__ rvec<T> rload_own(const RowCol<T, H>& c, const RowGeo& g, const T* p, int z) {
  if (c.tail && z == g.nz - 1) {
    rvec<T> v = {};
#pragma unroll
    for (int k = 0; k < RowVec<T>::V; ++k)
      if (c.x + k < g.nx) v[k] = p[k];
    return v;
  }
  return rload(p);
}

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
  g.tiles = ceil_div(int64_t(g.nv) * ny, kRowLanes * (kRowThreads / 64));
  g.chunk = most;
  while (g.chunk > 2 && int64_t(g.tiles) * ceil_div(nz, g.chunk) < 1024) g.chunk /= 2;
  return g;
}
inline unsigned row_blocks(const RowGeo& g) { return unsigned(int64_t(g.tiles) * ceil_div(g.nz, g.chunk)); }

// Whether the row-vector kernels take a field: cells adjacent along x, rows and planes that
// do not overlap, and 32-bit offsets.
inline bool row_strides_ok(const int64_t* s, int64_t nz, int64_t ny, int64_t nx) {
  constexpr int64_t lim = int64_t(1) << 31;
  return s[2] == 1 && s[0] >= nx && s[1] >= nx && s[0] < lim && s[1] < lim &&
         (s[0] >= (ny - 1) * s[1] + nx || s[1] >= (nz - 1) * s[0] + nx) &&
         (nz - 1) * s[0] + (ny - 1) * s[1] + nx < lim;
}
// ... and a box: one with cells the operator (of reach H) writes inside values to, and with
// vectors and workgroups that 32 bits count.
template <typename T, int H>
inline bool row_box_ok(int64_t nz, int64_t ny, int64_t nx) {
  constexpr int64_t lim = int64_t(1) << 30;
  return nz > 2 * H && ny > 2 * H && nx > 2 * H && nx >= RowVec<T>::V && nz < lim && ny < lim && nx < lim &&
         nz * ny < lim && ny * nx < lim && nz * (ny * nx) / RowVec<T>::V < 62 * lim;
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

// Whether no component's output meets another component's output or operand: such components may
// run in any order. A caller may pass windows of one tensor (out = t[0:3], in = t[1:4]) or a
// component repeated by a zero stride; the components then run one after another, as the
// reference's loop over them does.
template <typename T>
inline bool components_apart(int ncomp, void* const* out, const int64_t* os, const void* const* in,
                             const int64_t* is, int64_t nz, int64_t ny, int64_t nx) {
  for (int a = 0; a < ncomp; ++a)
    for (int b = 0; b < ncomp; ++b) {
      if (a == b) continue;
      if (fields_meet<T>(out[a], os, out[b], os, nz, ny, nx)) return false;
      if (in && fields_meet<T>(out[a], os, in[b], is, nz, ny, nx)) return false;
    }
  return true;
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
  const RowCol<T, 1> c(g);
  const int ur = c.yl * u.s.y + c.x, wr = c.y * w.s.y + c.x;
  vec um[3], uc[3];
  {
    const int zm = c.z0 > 0 ? c.z0 - 1 : 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      um[a] = rload(u.p[a] + zm * u.s.z + ur);
      uc[a] = rload(u.p[a] + c.z0 * u.s.z + ur);
    }
  }
  for (int z = c.z0; z < c.z1; ++z) {
    const bool plane = z > 0 && z < g.nz - 1;
    vec wv[3], up[3], grad[3][3];  // grad[a][axis]: difference of u_a along x, y, z
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const T* ua = u.p[a] + z * u.s.z + ur;
      up[a] = z < g.nz - 1 ? rload(ua + u.s.z) : uc[a];
      wv[a] = rload_own(c, g, w.p[a] + z * w.s.z + wr, z);
      grad[a][1] = plane ? rload(ua + u.s.y) - rload(ua - u.s.y) : vec{};
      grad[a][2] = up[a] - um[a];
      const T left = from_prev_lane(uc[a][V - 1]), right = from_next_lane(uc[a][0]);
#pragma unroll
      for (int k = 0; k < V; ++k)
        grad[a][0][k] = (k < V - 1 ? uc[a][k < V - 1 ? k + 1 : k] : right) - (k > 0 ? uc[a][k > 0 ? k - 1 : k] : left);
    }
    const bool zin = c.yin && plane;
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
    if constexpr (SCHEME >= 1) {
#pragma unroll
      for (int a = 0; a < 3; ++a) o[a] = m[a] = wv[a] + f[a];
    }
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

// ------------------------------------------------------------------ ENO3 advection flux

// The flux through the face between cells 0 and 1 of one axis (advection_flux_3d.py:12-233),
// from the field f and the velocity u at cells -1 .. 2. A cell's front face is its upper
// neighbour's back face, with the same upwind choice and the same terms, so each face is formed
// once. The weighted field values and the smallest of the three products round by themselves,
// the other products only in the sums (written out, so that every kernel of the flux gives the
// same bits): 150 x 201 x 230 FP32, relative error 5.4e-7 against 7.7e-7 with every product
// rounded, in the same time.
template <typename T>
__device__ __forceinline__ T eno3_face(T fm, T f0, T f1, T fp, T um, T u0, T u1, T up) {
  const T c13 = T(1.0 / 3.0), c56 = T(5.0 / 6.0), c16 = T(1.0 / 6.0);
  const bool left = u0 > -u1;
  const T far = c16 * (left ? fm : fp) * (left ? um : up);
  return fma(c56 * (left ? f0 : f1), left ? u0 : u1, fma(c13 * (left ? f1 : f0), left ? u1 : u0, -far));
}

// What k_eno3_rows does with the flux E of [2:-2]^3.
enum EnoMode {
  kEnoAdd,  // out += E on [2:-2]^3
  kEnoSet,  // out = E, 0 on the border cells: spares the clearing and the read of the flux field
  kEnoStep  // out = field + E, the field on the border cells
};

// ENO3 conservative advection flux of one scalar field per gridDim.y.
// A thread forms V + 1 x faces, two rows of y faces and one plane of z faces per plane of V
// cells; its 12 16-byte loads per plane (field rows y-2, y-1, y+1, y+2, u_y rows y-2..y+2, u_x, u_z
// and the field two planes up) come mostly from L1 and L2, and their rate bounds it.
// 150 x 201 x 230 FP32, storing: 29 us (4.7 TB/s of 5 words per cell) against 94 us with one
// cell per thread plus 7 us for the clearing.
template <typename T, int MODE>
__global__ void __launch_bounds__(kRowThreads)
    k_eno3_rows(RowGeo g, Rows3<T> out, Rows3<const T> field, Rows3<const T> u, T inv_dx) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T, 2> c(g);
  T* const flux = out.p[blockIdx.y];
  const T* const f = field.p[blockIdx.y];
  const RowStrides os = out.s, fs = field.s;
  const int fr = c.yl * fs.y + c.x, ur = c.yl * u.s.y + c.x, orow = c.y * os.y + c.x, frow = c.y * fs.y + c.x;
  // planes with a flux: those of the chunk inside [2, nz - 2)
  const int za = c.z0 < 2 ? 2 : c.z0, zb = c.z1 < g.nz - 2 ? c.z1 : g.nz - 2;
  if constexpr (MODE != kEnoAdd) {
    for (int z = c.z0; z < c.z1; ++z)
      if (z < za || z >= zb)
        rstore(flux + z * os.z + orow, MODE == kEnoStep ? rload_own(c, g, f + z * fs.z + frow, z) : vec{}, c.own);
  }
  if (za >= zb) return;  // the same for the whole workgroup
  // along z: the field and u_z at z-1, z, z+1, and the back face
  vec fm = rload(f + (za - 1) * fs.z + fr), wm = rload(u.p[2] + (za - 1) * u.s.z + ur);
  vec f0 = rload(f + za * fs.z + fr), f1 = rload(f + (za + 1) * fs.z + fr);
  vec w0 = rload(u.p[2] + za * u.s.z + ur), w1 = rload(u.p[2] + (za + 1) * u.s.z + ur);
  vec back;
  {
    const vec fmm = rload(f + (za - 2) * fs.z + fr), wmm = rload(u.p[2] + (za - 2) * u.s.z + ur);
#pragma unroll
    for (int k = 0; k < V; ++k) back[k] = eno3_face<T>(fmm[k], fm[k], f0[k], f1[k], wmm[k], wm[k], w0[k], w1[k]);
  }
  const unsigned mask = c.yin ? c.own & c.inner : 0u;
  for (int z = za; z < zb; ++z) {
    const T* fz = f + z * fs.z + fr;
    const T* uxz = u.p[0] + z * u.s.z + ur;
    const T* uyz = u.p[1] + z * u.s.z + ur;
    T* oz = flux + z * os.z + orow;
    const vec f2 = rload(fz + 2 * fs.z), w2 = rload(u.p[2] + (z + 2) * u.s.z + ur);
    const vec ux = rload(uxz);
    vec uy[5], fy[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) {
      uy[r] = rload(uyz + (r - 2) * u.s.y);
      fy[r] = r == 2 ? f0 : rload(fz + (r - 2) * fs.y);
    }
    vec acc = {};
    if constexpr (MODE == kEnoAdd) acc = rload_own(c, g, static_cast<const T*>(oz), z);
    {  // x faces -1/2 .. V - 1/2 of the vector
      T e[V + 4], v[V + 4];  // field and velocity at cells -2 .. V + 1
      e[0] = from_prev_lane(f0[V - 2]);
      e[1] = from_prev_lane(f0[V - 1]);
      e[V + 2] = from_next_lane(f0[0]);
      e[V + 3] = from_next_lane(f0[1]);
      v[0] = from_prev_lane(ux[V - 2]);
      v[1] = from_prev_lane(ux[V - 1]);
      v[V + 2] = from_next_lane(ux[0]);
      v[V + 3] = from_next_lane(ux[1]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        e[k + 2] = f0[k];
        v[k + 2] = ux[k];
      }
      T face[V + 1];
#pragma unroll
      for (int k = 0; k <= V; ++k)
        face[k] = eno3_face<T>(e[k], e[k + 1], e[k + 2], e[k + 3], v[k], v[k + 1], v[k + 2], v[k + 3]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        acc[k] = fma(inv_dx, face[k + 1], acc[k]);
        acc[k] = fma(-inv_dx, face[k], acc[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
      acc[k] = fma(inv_dx, eno3_face<T>(fy[1][k], fy[2][k], fy[3][k], fy[4][k], uy[1][k], uy[2][k], uy[3][k], uy[4][k]), acc[k]);
      acc[k] = fma(-inv_dx, eno3_face<T>(fy[0][k], fy[1][k], fy[2][k], fy[3][k], uy[0][k], uy[1][k], uy[2][k], uy[3][k]), acc[k]);
      const T front = eno3_face<T>(fm[k], f0[k], f1[k], f2[k], wm[k], w0[k], w1[k], w2[k]);
      acc[k] = fma(inv_dx, front, acc[k]);
      acc[k] = fma(-inv_dx, back[k], acc[k]);
      back[k] = front;
    }
    if constexpr (MODE == kEnoAdd) {
      rstore(oz, acc, mask);
    } else {
      vec rest = {};
      if constexpr (MODE == kEnoStep) {
        rest = f0;
        if (!c.yin) rest = rload_own(c, g, f + z * fs.z + frow, z);
        acc = rest + acc;
      }
#pragma unroll
      for (int k = 0; k < V; ++k) acc[k] = mask >> k & 1u ? acc[k] : rest[k];
      rstore(oz, acc, c.own);
    }
    fm = f0;
    f0 = f1;
    f1 = f2;
    wm = w0;
    w0 = w1;
    w1 = w2;
  }
}

// Transpose of the ENO3 flux along one axis with the upwind choices frozen at the velocity, at
// cell m: a and u are the flux adjoint (0 where the forward writes nothing) and the axis'
// velocity at cells m - 2 .. m + 2. The flux at a cell is its front face minus its back face,
// so face (i, i + 1) carries d = a(i) - a(i + 1), and the faces m - 2 .. m + 1 read cell m.
template <typename T>
__device__ __forceinline__ T eno3_gather(const T* a, const T* u) {
  const T c13 = T(1.0 / 3.0), c56 = T(5.0 / 6.0), c16 = T(1.0 / 6.0);
  const T lo = !(u[0] > -u[1]) ? a[0] - a[1] : T(0);
  const T hi = u[3] > -u[4] ? a[3] - a[4] : T(0);
  return (u[1] > -u[2] ? c13 : c56) * (a[1] - a[2]) + (u[2] > -u[3] ? c56 : c13) * (a[2] - a[3]) - c16 * (lo + hi);
}

// The transpose on a whole box: gbar_axis as above where the forward flux reads the cell along
// that axis, then field_adj (+)= sum_axis gbar_axis u_axis, vel_adj[axis] (+)= gbar_axis field.
// SET stores instead of adding, which spares the outputs' clearing and their read (4 of 13
// words per cell). A gather: no atomics, the same bits on every run.
// Bound by memory: 150 x 201 x 230 FP32, storing, 53 us (4.7 TB/s of 9 words per cell) against
// 148 us with one cell per thread, each weighing the 15 fluxes that read it, plus 19 us of clearing.
template <typename T, bool SET>
__global__ void __launch_bounds__(kRowThreads)
    k_eno3_adjoint_rows(RowGeo g, T* fa, RowStrides fas, Rows3<T> va, const T* a, RowStrides as, const T* f,
                        RowStrides fs, Rows3<const T> u, T inv_dx) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T, 2> c(g);
  const int ar = c.yl * as.y + c.x, ur = c.yl * u.s.y + c.x;
  // a plane of the flux adjoint, 0 where the forward writes no plane
  auto a_plane = [&](int q) -> vec {
    return q >= 2 && q < g.nz - 2 ? rload(a + q * as.z + ar) : vec{};
  };
  auto u_plane = [&](int q) -> vec {  // u_z, read where a face of the forward reads it
    const int p = q < 1 ? 1 : (q < g.nz - 1 ? q : g.nz - 2);
    return rload(u.p[2] + p * u.s.z + ur);
  };
  vec az[5], uz[5];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    az[k + 1] = a_plane(c.z0 - 2 + k);
    uz[k + 1] = u_plane(c.z0 - 2 + k);
  }
  // rows y - 2 .. y + 2: the flux adjoint is 0 outside [2, ny - 2); the velocity rows are
  // clamped into the grid (a clamped row's faces carry d = 0)
  int arow[5], urow[5];
  bool ain[5];
#pragma unroll
  for (int r = 0; r < 5; ++r) {
    const int y = c.y + r - 2;
    ain[r] = y >= 2 && y < g.ny - 2;
    arow[r] = (y < 2 ? 2 : (y < g.ny - 2 ? y : g.ny - 3)) * as.y + c.x;
    urow[r] = (y < 1 ? 1 : (y < g.ny - 1 ? y : g.ny - 2)) * u.s.y + c.x;
  }
  for (int z = c.z0; z < c.z1; ++z) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      az[k] = az[k + 1];
      uz[k] = uz[k + 1];
    }
    az[4] = a_plane(z + 2);
    uz[4] = u_plane(z + 2);
    vec gb[3] = {{}, {}, {}};
    if (z >= 2 && z < g.nz - 2) {  // the same for the whole workgroup
      vec ay[5], uy[5];
#pragma unroll
      for (int r = 0; r < 5; ++r) {
        uy[r] = rload(u.p[1] + z * u.s.z + urow[r]);
        ay[r] = r == 2 ? az[2] : rload(a + z * as.z + arow[r]);
      }
      const vec ux = rload(u.p[0] + z * u.s.z + ur);
      T e[V + 4], v[V + 4];
#pragma unroll
      for (int k = 0; k < V; ++k) {
        e[k + 2] = c.inner >> k & 1u ? az[2][k] : T(0);
        v[k + 2] = ux[k];
      }
      e[0] = from_prev_lane(e[V]);
      e[1] = from_prev_lane(e[V + 1]);
      v[0] = from_prev_lane(v[V]);
      v[1] = from_prev_lane(v[V + 1]);
      e[V + 2] = from_next_lane(e[2]);
      e[V + 3] = from_next_lane(e[3]);
      v[V + 2] = from_next_lane(v[2]);
      v[V + 3] = from_next_lane(v[3]);
      if (c.x == 0) e[0] = e[1] = T(0);  // the lane before holds another row's end
#pragma unroll
      for (int k = 0; k < V; ++k) {
        if (c.yin) gb[0][k] = inv_dx * eno3_gather<T>(e + k, v + k);
        const T ac[5] = {ain[0] ? ay[0][k] : T(0), ain[1] ? ay[1][k] : T(0), ain[2] ? ay[2][k] : T(0),
                         ain[3] ? ay[3][k] : T(0), ain[4] ? ay[4][k] : T(0)};
        const T uc[5] = {uy[0][k], uy[1][k], uy[2][k], uy[3][k], uy[4][k]};
        if (c.inner >> k & 1u) gb[1][k] = inv_dx * eno3_gather<T>(ac, uc);
      }
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const T ac[5] = {az[0][k], az[1][k], az[2][k], az[3][k], az[4][k]};
      const T uc[5] = {uz[0][k], uz[1][k], uz[2][k], uz[3][k], uz[4][k]};
      if (c.yin && (c.inner >> k & 1u)) gb[2][k] = inv_dx * eno3_gather<T>(ac, uc);
    }
    if (fa) {
      T* o = fa + z * fas.z + c.y * fas.y + c.x;
      vec r = {};
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) r += gb[ax] * rload_own(c, g, u.p[ax] + z * u.s.z + c.y * u.s.y + c.x, z);
      if (!SET) r += rload_own(c, g, static_cast<const T*>(o), z);
      rstore(o, r, c.own);
    }
    if (va.p[0]) {
      const vec fv = rload_own(c, g, f + z * fs.z + c.y * fs.y + c.x, z);
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        T* o = va.p[ax] + z * va.s.z + c.y * va.s.y + c.x;
        vec r = gb[ax] * fv;
        if (!SET) r += rload_own(c, g, static_cast<const T*>(o), z);
        rstore(o, r, c.own);
      }
    }
  }
}

// ------------------------------------------------------------------ curl, Laplacian, divergence

// What a stencil kernel does with its output field.
enum RowMode {
  kRowInside,  // store the inside cells, leave the border
  kRowReset,   // store the inside cells and zeros on the border
  kRowAdd,     // add to the inside cells
  kRowStep     // (Laplacian) store the operand plus the result, the operand on the border
};

template <typename T, int MODE>
__device__ __forceinline__ void row_out(const RowCol<T, 1>& c, const RowGeo& g, T* p, rvec<T> v, unsigned inside, int z) {
  if constexpr (MODE == kRowAdd) {
    if (inside) rstore(p, rload_own(c, g, static_cast<const T*>(p), z) + v, inside);
  } else if constexpr (MODE == kRowReset) {
#pragma unroll
    for (int k = 0; k < RowVec<T>::V; ++k) v[k] = inside >> k & 1u ? v[k] : T(0);
    rstore(p, v, c.own);
  } else {
    rstore(p, v, inside);
  }
}

// p curl_h(f) (curl_3d.py:13-132) and its accumulating form
// (update_vorticity_from_velocity_forcing_3d.py:12-132). Bound by memory: f0 and f1 are
// differentiated along z and march in registers, so a plane costs 7 16-byte loads per thread.
// 96 x 128 x 192 FP32 with the border reset: 16 us (3.5 TB/s) against 25 us with one cell per
// thread plus six border launches of 2.4 to 5 us.
template <typename T, int MODE>
__global__ void __launch_bounds__(kRowThreads) k_curl_rows(RowGeo g, Rows3<T> o, Rows3<const T> f, T p) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T, 1> c(g);
  const int fr = c.yl * f.s.y + c.x, orow = c.y * o.s.y + c.x;
  const int zm = c.z0 > 0 ? c.z0 - 1 : 0;
  vec xm = rload(f.p[0] + zm * f.s.z + fr), ym = rload(f.p[1] + zm * f.s.z + fr);
  vec xc = rload(f.p[0] + c.z0 * f.s.z + fr), yc = rload(f.p[1] + c.z0 * f.s.z + fr);
  for (int z = c.z0; z < c.z1; ++z) {
    const bool plane = z > 0 && z < g.nz - 1;  // the same for the whole workgroup
    vec r0 = {}, r1 = {}, r2 = {}, xp = xc, yp = yc;
    if (z < g.nz - 1) {
      xp = rload(f.p[0] + (z + 1) * f.s.z + fr);
      yp = rload(f.p[1] + (z + 1) * f.s.z + fr);
    }
    if (plane) {
      const T* f0 = f.p[0] + z * f.s.z + fr;
      const T* f2 = f.p[2] + z * f.s.z + fr;
      const vec zc = rload(f2);
      const vec z_yp = rload(f2 + f.s.y), z_ym = rload(f2 - f.s.y);
      const vec x_yp = rload(f0 + f.s.y), x_ym = rload(f0 - f.s.y);
      const T zl = from_prev_lane(zc[V - 1]), zr = from_next_lane(zc[0]);
      const T yl = from_prev_lane(yc[V - 1]), yr = from_next_lane(yc[0]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        const T z_r = k < V - 1 ? zc[k < V - 1 ? k + 1 : k] : zr, z_l = k > 0 ? zc[k > 0 ? k - 1 : k] : zl;
        const T y_r = k < V - 1 ? yc[k < V - 1 ? k + 1 : k] : yr, y_l = k > 0 ? yc[k > 0 ? k - 1 : k] : yl;
        r0[k] = p * (z_yp[k] - z_ym[k] - yp[k] + ym[k]);
        r1[k] = p * (xp[k] - xm[k] - z_r + z_l);
        r2[k] = p * (y_r - y_l - x_yp[k] + x_ym[k]);
      }
    }
    const unsigned inside = plane && c.yin ? c.own & c.inner : 0u;
    row_out<T, MODE>(c, g, o.p[0] + z * o.s.z + orow, r0, inside, z);
    row_out<T, MODE>(c, g, o.p[1] + z * o.s.z + orow, r1, inside, z);
    row_out<T, MODE>(c, g, o.p[2] + z * o.s.z + orow, r2, inside, z);
    xm = xc;
    xc = xp;
    ym = yc;
    yc = yp;
  }
}

// p lap_h(f) of one scalar field per gridDim.y (diffusion_flux_3d.py:14-115). Bound by memory:
// 130 x 170 x 250 FP32, 10.4 us (4.2 TB/s) against 21 us with one cell per thread plus six
// border launches of 2.2 to 4.6 us.
template <typename T, int MODE>
__global__ void __launch_bounds__(kRowThreads) k_laplacian_rows(RowGeo g, Rows3<T> o, Rows3<const T> in, T p) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T, 1> c(g);
  const T* const f = in.p[blockIdx.y];
  T* const out = o.p[blockIdx.y];
  const int fr = c.yl * in.s.y + c.x, orow = c.y * o.s.y + c.x;
  vec fm = rload(f + (c.z0 > 0 ? c.z0 - 1 : 0) * in.s.z + fr), fc = rload(f + c.z0 * in.s.z + fr);
  for (int z = c.z0; z < c.z1; ++z) {
    const bool plane = z > 0 && z < g.nz - 1;
    const T* fz = f + z * in.s.z + fr;
    vec r = {}, fp = fc;  // r: lap_h(f), times p but for kRowStep
    if (z < g.nz - 1) fp = rload(fz + in.s.z);
    if (plane) {
      const vec yp = rload(fz + in.s.y), ym = rload(fz - in.s.y);
      const T xl = from_prev_lane(fc[V - 1]), xr = from_next_lane(fc[0]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        const T right = k < V - 1 ? fc[k < V - 1 ? k + 1 : k] : xr, left = k > 0 ? fc[k > 0 ? k - 1 : k] : xl;
        const T lap = fp[k] + fm[k] + yp[k] + ym[k] + right + left - T(6) * fc[k];
        r[k] = MODE == kRowStep ? lap : p * lap;
      }
    }
    const unsigned inside = plane && c.yin ? c.own & c.inner : 0u;
    if constexpr (MODE == kRowStep) {
      vec v = fc;
      if (!c.yin) v = rload_own(c, g, f + z * in.s.z + c.y * in.s.y + c.x, z);
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = inside >> k & 1u ? fma(p, r[k], v[k]) : v[k];
      rstore(out + z * o.s.z + orow, v, c.own);
    } else {
      row_out<T, MODE>(c, g, out + z * o.s.z + orow, r, inside, z);
    }
    fm = fc;
    fc = fp;
  }
}

// div_h(f) (divergence_3d.py:13-96). Bound by memory: 130 x 170 x 250 FP32,
// 15 us (5.8 TB/s) against 23 us with one cell per thread plus six border launches.
template <typename T, int MODE>
__global__ void __launch_bounds__(kRowThreads)
    k_divergence_rows(RowGeo g, T* out, RowStrides os, Rows3<const T> f, T inv_dx) {
  constexpr int V = RowVec<T>::V;
  using vec = rvec<T>;
  const RowCol<T, 1> c(g);
  const int fr = c.yl * f.s.y + c.x, orow = c.y * os.y + c.x;
  vec zm = rload(f.p[2] + (c.z0 > 0 ? c.z0 - 1 : 0) * f.s.z + fr), zc = rload(f.p[2] + c.z0 * f.s.z + fr);
  for (int z = c.z0; z < c.z1; ++z) {
    const bool plane = z > 0 && z < g.nz - 1;
    vec r = {}, zp = zc;
    if (z < g.nz - 1) zp = rload(f.p[2] + (z + 1) * f.s.z + fr);
    if (plane) {
      const vec xc = rload(f.p[0] + z * f.s.z + fr);
      const vec yp = rload(f.p[1] + z * f.s.z + fr + f.s.y), ym = rload(f.p[1] + z * f.s.z + fr - f.s.y);
      const T xl = from_prev_lane(xc[V - 1]), xr = from_next_lane(xc[0]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        const T right = k < V - 1 ? xc[k < V - 1 ? k + 1 : k] : xr, left = k > 0 ? xc[k > 0 ? k - 1 : k] : xl;
        r[k] = T(0.5) * inv_dx * (right - left + yp[k] - ym[k] + zp[k] - zm[k]);
      }
    }
    const unsigned inside = plane && c.yin ? c.own & c.inner : 0u;
    row_out<T, MODE>(c, g, out + z * os.z + orow, r, inside, z);
    zm = zc;
    zc = zp;
  }
}

// ------------------------------------------------------------------ pointwise operators

// Whether the fields of a box are dense: their cells follow each other without gaps.
inline bool dense(const int64_t* s, int64_t ny, int64_t nx) { return s[2] == 1 && s[1] == nx && s[0] == ny * nx; }

template <typename T, int N>
struct Flat {
  T* out[3];
  const T* in[N > 0 ? N : 1][3];
  int64_t n;  // cells
  int first;  // component of gridDim.y's first slice
};

// out = fn(comp, in...) over the cells of up to three dense components (gridDim.y from a.first), 16
// bytes a thread. Bound by memory: the sum of two 130 x 170 x 250 FP32 fields takes 10.9 us (6.1 TB/s, most
// of it from the caches) against 18.4 us with one cell per thread and 64-bit divisions.
template <typename T, int N, typename Fn>
__global__ void __launch_bounds__(256) k_flat(Flat<T, N> a, Fn fn) {
  constexpr int V = RowVec<T>::V;
  const int c = a.first + int(blockIdx.y);
  const int64_t i = (blockIdx.x * int64_t(256) + threadIdx.x) * V;
  auto one = [&](const T* v) -> T {
    if constexpr (N == 0) return fn(c);
    else if constexpr (N == 1) return fn(c, v[0]);
    else return fn(c, v[0], v[1]);
  };
  if (i + V <= a.n) {
    rvec<T> in[N > 0 ? N : 1] = {}, o;
#pragma unroll
    for (int q = 0; q < N; ++q) in[q] = rload(a.in[q][c] + i);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      T v[N > 0 ? N : 1] = {};
#pragma unroll
      for (int q = 0; q < N; ++q) v[q] = in[q][k];
      o[k] = one(v);
    }
    *reinterpret_cast<rvec<T>*>(a.out[c] + i) = o;
  } else {
    for (int64_t j = i; j < a.n; ++j) {
      T v[N > 0 ? N : 1] = {};
      for (int q = 0; q < N; ++q) v[q] = a.in[q][c][j];
      a.out[c][j] = one(v);
    }
  }
}

// result = a x b on dense fields (elementwise_ops_3d.py:390-449). 96 x 128 x 192 FP32: 13.4 us
// (6.3 TB/s) against 18 us with one cell per thread.
template <typename T>
__global__ void __launch_bounds__(256) k_cross_flat(Flat<T, 2> f) {
  constexpr int V = RowVec<T>::V;
  const int64_t i = (blockIdx.x * int64_t(256) + threadIdx.x) * V;
  if (i + V <= f.n) {
    rvec<T> a[3], b[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      a[c] = rload(f.in[0][c] + i);
      b[c] = rload(f.in[1][c] + i);
    }
    *reinterpret_cast<rvec<T>*>(f.out[0] + i) = a[1] * b[2] - b[1] * a[2];
    *reinterpret_cast<rvec<T>*>(f.out[1] + i) = a[2] * b[0] - b[2] * a[0];
    *reinterpret_cast<rvec<T>*>(f.out[2] + i) = a[0] * b[1] - b[0] * a[1];
  } else {
    for (int64_t j = i; j < f.n; ++j) {
      const T a0 = f.in[0][0][j], a1 = f.in[0][1][j], a2 = f.in[0][2][j];
      const T b0 = f.in[1][0][j], b1 = f.in[1][1][j], b2 = f.in[1][2][j];
      f.out[0][j] = a1 * b2 - b1 * a2;
      f.out[1][j] = a2 * b0 - b2 * a0;
      f.out[2][j] = a0 * b1 - b0 * a1;
    }
  }
}

template <typename T>
inline dim3 flat_grid(int64_t n, int comps) {
  return dim3(unsigned((n + 256 * RowVec<T>::V - 1) / (256 * RowVec<T>::V)), unsigned(comps));
}

}  // namespace
}  // namespace sopht
