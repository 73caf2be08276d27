// The spectral slab of the free-space Poisson solver and the fields of a solve, shared by its
// passes (poisson_3d.hip, poisson_xy.h).
#pragma once

#include "common.h"
#include "fft_reg.h"

namespace sopht {

// A streaming store of one complex value: the next pass reads it back from HBM, so it need
// not stay in the cache hierarchy.
template <typename T>
__device__ __forceinline__ void store_stream(Cplx<T>* p, Cplx<T> v) {
  typedef T pair __attribute__((ext_vector_type(2)));
  pair w;
  w.x = v.re;
  w.y = v.im;
  __builtin_nontemporal_store(w, reinterpret_cast<pair*>(p));
}

using rfft::LinePlan;
using rfft::region_stride;
using rfft::static_for;
using rfft::team_fft;

// Slab rows (kx = 0..nx) are padded to a whole number of 128-byte lines, so every column
// tile of the y and z passes reads and writes whole cache lines.
template <typename T>
constexpr int kLineCplx = 128 / int(sizeof(Cplx<T>));
#ifndef SOPHT_COL_HALF
#define SOPHT_COL_HALF 1
#endif
#ifndef SOPHT_ROW_PAD
#define SOPHT_ROW_PAD 1
#endif
// Column tiles are half a 128-byte line when SOPHT_COL_HALF is set; the two halves of a line
// then go to workgroups b and b + 8, which the dispatcher sends to the same XCD one after the
// other, so the second half is read from that XCD's L2.
constexpr int kColHalf = SOPHT_COL_HALF;
constexpr int64_t kRowPad = SOPHT_ROW_PAD;
// Columns per slab tile of the three-pass schedule. Measured at 256^3 FP32 (pass A + z pass +
// pass C): 16 columns 1.21 ms, 8 columns 1.20 ms (the z pass faster, passes A and C slower),
// 4 columns 2.2 ms (pass A's writes become 32-byte pieces of lines from four planes, which
// other workgroups write).
#ifndef SOPHT_SLAB_TILE
#define SOPHT_SLAB_TILE 16
#endif
constexpr int kSlabTile = SOPHT_SLAB_TILE;
static_assert(16 % kSlabTile == 0, "slab tiles divide a 128-byte line");

// (row, first kx) of the column tile of workgroup b; false for the padding workgroups.
__device__ __forceinline__ bool col_tile(int64_t b, int64_t ncols, int64_t nrows, int wc,
                                         int64_t& row, int64_t& kx0) {
  if (kColHalf) {
    const int64_t lines = (ncols + 2 * wc - 1) / (2 * wc);
    const int64_t line = (b / 16) * 8 + b % 8;
    const int64_t half = (b / 8) % 2;
    row = line / lines;
    kx0 = ((line % lines) * 2 + half) * wc;
    return row < nrows;
  }
  const int64_t tiles = (ncols + wc - 1) / wc;
  row = b / tiles;
  kx0 = (b % tiles) * wc;
  return row < nrows;
}

// The same with a line split in PARTS tiles: the parts of a line go to workgroups
// b + 8 p (p < PARTS), which the dispatcher sends to one XCD.
template <int PARTS>
__device__ __forceinline__ bool col_tile_parts(int64_t b, int64_t ncols, int64_t nrows, int wc,
                                               int64_t& row, int64_t& kx0) {
  const int64_t lines = (ncols + PARTS * wc - 1) / (PARTS * wc);
  const int64_t line = (b / (8 * PARTS)) * 8 + b % 8;
  const int64_t part = (b / 8) % PARTS;
  row = line / lines;
  kx0 = ((line % lines) * PARTS + part) * wc;
  return row < nrows;
}

inline int64_t col_tile_parts_blocks(int parts, int64_t ncols, int64_t nrows, int wc) {
  const int64_t lines = (ncols + parts * wc - 1) / (parts * wc);
  return 8 * parts * ((lines * nrows + 7) / 8);
}

inline int64_t col_tile_blocks(int64_t ncols, int64_t nrows, int wc) {
  if (kColHalf) {
    const int64_t lines = (ncols + 2 * wc - 1) / (2 * wc);
    return 16 * ((lines * nrows + 7) / 8);
  }
  return (ncols + wc - 1) / wc * nrows;
}

inline int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

struct SlabGeom {
  int64_t nz, ny, nx;  // physical grid
  int64_t rs;          // row stride (complex elements), >= nx + 1
  int64_t gz;          // G^ line stride (elements), >= nz + 1
  int ncomp;
  // H index of (c, z, ky, kx)
  __device__ __forceinline__ int64_t h(int c, int64_t z, int64_t ky, int64_t kx) const {
    return ((int64_t(c) * nz + z) * (2 * ny) + ky) * rs + kx;
  }
  // the same as a 32-bit offset (plan creation checks that the slab has < 2^31 elements):
  // loads then take a uniform base plus one VGPR of offset
  __device__ __forceinline__ int hi(int c, int z, int ky, int kx) const {
    return ((c * int(nz) + z) * (2 * int(ny)) + ky) * int(rs) + kx;
  }
  // The three-pass schedule keeps the slab in column tiles of kSlabTile columns with z inside
  // a tile: (c, ky, kx / kSlabTile, z, kx % kSlabTile). The z pass then reads and writes each
  // tile's z line as one contiguous run; with 16 columns (one 128-byte line per plane) the x/y
  // passes still move whole lines (rs is a multiple of 16 there).
  // (Unsigned arithmetic: the divisions by the power-of-two tile width are shifts.) Moving by
  // dr rows adds dr rs nz; moving by a whole number of tiles, dk columns, adds dk nz.
  __device__ __forceinline__ int ti(int c, int z, int ky, int kx) const {
    const unsigned k = unsigned(kx);
    return int((((unsigned(c) * 2u * unsigned(ny) + unsigned(ky)) * (unsigned(rs) / kSlabTile) + k / kSlabTile) *
                    unsigned(nz) + unsigned(z)) * kSlabTile + k % kSlabTile);
  }
  __device__ __forceinline__ int64_t row_h(int64_t r) const {  // H row of input row r
    const int c = int(r / (nz * ny));
    const int64_t rem = r % (nz * ny);
    return h(c, rem / ny, rem % ny, 0);
  }
};

// Component fields of a solve: up to three pointers by value, or (batched solves over many
// instances of one grid size) a device table of one pointer per component.
struct CompPtrs {
  const void* p[3];
  const void* const* tab;
  int64_t sz, sy, sx;
  __device__ __forceinline__ const void* get(int c) const { return tab ? tab[c] : p[c]; }
};
struct CompPtrsW {
  void* p[3];
  void* const* tab;
  int64_t sz, sy, sx;
  __device__ __forceinline__ void* get(int c) const { return tab ? tab[c] : p[c]; }
};

}  // namespace sopht
