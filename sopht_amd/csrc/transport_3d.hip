// Passive transport step of a scalar or vector field on gfx950. Per component phi,
//   phi_a   = phi + E(phi, u)                  conservative ENO3 advection with -dt/dx on
//                                              [2:-2]^3, E = 0 elsewhere
//                                              (advection_timestep_3d.py:12-99,
//                                              advection_flux_3d.py:12-233)
//   phi_new = phi_a + pD lap_h(phi_a)          on [1:-1]^3, phi_a on the border
//                                              (diffusion_timestep_3d.py:12-80)
// i.e. the reference's advection step followed by its diffusion step, in its operation order.
// Two row-vector sweeps: the advection writes phi_a to a scratch field, the diffusion reads it
// and writes phi_new over phi, so nothing is copied back and no neighbour of a written cell is
// read. Both are bound by memory: 4 words per cell and component, 3 for the velocity (read
// once per component, mostly from the caches). One sweep that keeps phi_a in LDS moves the
// same words once the result has to be copied back, and recomputes the advection on tile
// rings: 200 x 160 x 240 FP32 vector 134 us (90 + 44) against 287 us, 61 x 70 x 83 FP64 scalar
// 11 us against 39 us.
#include <algorithm>

#include "common.h"
#include "row_march.h"

namespace sopht {
namespace {

constexpr int kTransportChunk = 16;

template <typename T>
int transport_launch(int ncomp, void* const field[3], void* const scratch[3], const void* const vel[3],
                     int64_t nz, int64_t ny, int64_t nx, double dt_by_dx, double nu_dt_by_dx2,
                     hipStream_t s) {
  // the reference forms inv_dx = -real_t(dt / dx) and nu dt / dx^2 in real_t
  const T inv_dx = -T(dt_by_dx), pD = T(nu_dt_by_dx2);
  const int64_t st[3] = {ny * nx, nx, 1};
  if (row_box_ok<T, 2>(nz, ny, nx)) {
    Rows3<T> phi{}, next{};
    Rows3<const T> phi_in{}, next_in{};
    phi.s = next.s = phi_in.s = next_in.s = row_strides(st);
    for (int c = 0; c < ncomp; ++c) {
      phi_in.p[c] = phi.p[c] = static_cast<T*>(field[c]);
      next_in.p[c] = next.p[c] = static_cast<T*>(scratch[c]);
    }
    const RowGeo g = row_geo<T>(nz, ny, nx, kTransportChunk);
    const dim3 grid{row_blocks(g), unsigned(ncomp), 1u};
    k_eno3_rows<T, kEnoStep><<<grid, kRowThreads, 0, s>>>(g, next, phi_in, rows3<T>(vel, st), inv_dx);
    SOPHT_CHECK_LAUNCH();
    k_laplacian_rows<T, kRowStep><<<grid, kRowThreads, 0, s>>>(g, phi, next_in, pD);
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  }
  // a box without cells two away from every face is not advected
  for (int c = 0; c < ncomp; ++c) {
    View3<T> f = make_view<T>(field[c], st), o = make_view<T>(scratch[c], st);
    int rc = launch_box(
        0, 0, 0, nz, ny, nx,
        [=] __device__(int64_t z, int64_t y, int64_t x) {
          T v = f(z, y, x);
          if (z > 0 && z < nz - 1 && y > 0 && y < ny - 1 && x > 0 && x < nx - 1)
            v = v + pD * (f(z + 1, y, x) + f(z - 1, y, x) + f(z, y + 1, x) + f(z, y - 1, x) + f(z, y, x + 1) +
                          f(z, y, x - 1) - T(6) * f(z, y, x));
          o(z, y, x) = v;
        },
        s);
    if (!rc)
      rc = launch_box(
          0, 0, 0, nz, ny, nx, [=] __device__(int64_t z, int64_t y, int64_t x) { f(z, y, x) = o(z, y, x); }, s);
    if (rc) return rc;
  }
  return SOPHT_OK;
}

// max over cells of |u0| + |u1| + |u2| (numpy's axis-0 sum order); optionally stores the sum
template <typename T>
__global__ void __launch_bounds__(256) k_abs_sum_max(const T* __restrict__ u0, const T* __restrict__ u1,
                                                     const T* __restrict__ u2, int64_t n,
                                                     T* __restrict__ mag, T* __restrict__ partial) {
  __shared__ T red[256];
  T m = T(0);
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const T v = (fabs(u0[i]) + fabs(u1[i])) + fabs(u2[i]);
    if (mag) mag[i] = v;
    m = v > m ? v : m;
  }
  red[threadIdx.x] = m;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (int(threadIdx.x) < k) red[threadIdx.x] = red[threadIdx.x + k] > red[threadIdx.x] ? red[threadIdx.x + k] : red[threadIdx.x];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

template <typename T>
int abs_sum_max(const void* const vel[3], int64_t n, void* mag, void* partial, int64_t cap, void* out,
                hipStream_t s) {
  const int nb = int(std::min<int64_t>(cap, (n + 255) / 256));
  k_abs_sum_max<T><<<nb, 256, 0, s>>>(static_cast<const T*>(vel[0]), static_cast<const T*>(vel[1]),
                                      static_cast<const T*>(vel[2]), n, static_cast<T*>(mag),
                                      static_cast<T*>(partial));
  SOPHT_CHECK_LAUNCH();
  k_max_final<T><<<1, 1024, 0, s>>>(static_cast<const T*>(partial), nb, static_cast<T*>(out));
  SOPHT_CHECK_LAUNCH();
  return SOPHT_OK;
}

}  // namespace
}  // namespace sopht

using namespace sopht;

extern "C" {

int sopht_passive_transport_step_3d(int dtype, int ncomp, void* const field[3], void* const scratch[3],
                                    const void* const vel[3], int64_t nz, int64_t ny, int64_t nx,
                                    double dt_by_dx, double nu_dt_by_dx2, void* stream) {
  SOPHT_REQUIRE(dtype == SOPHT_F32 || dtype == SOPHT_F64, "dtype must be SOPHT_F32 or SOPHT_F64");
  SOPHT_REQUIRE(ncomp == 1 || ncomp == 3, "ncomp must be 1 (scalar) or 3 (vector)");
  SOPHT_REQUIRE(nz >= 1 && ny >= 1 && nx >= 1, "grid sizes must be positive");
  SOPHT_REQUIRE(nz * ny * nx < (int64_t(1) << 31), "grid too large (nz ny nx must be below 2^31)");
  SOPHT_REQUIRE(field && scratch && vel && vel[0] && vel[1] && vel[2], "null pointer");
  for (int c = 0; c < ncomp; ++c) {
    SOPHT_REQUIRE(field[c] && scratch[c], "null component pointer");
    SOPHT_REQUIRE(field[c] != scratch[c], "the scratch field must not alias the field");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == SOPHT_F32 ? transport_launch<float>(ncomp, field, scratch, vel, nz, ny, nx, dt_by_dx, nu_dt_by_dx2, s)
                            : transport_launch<double>(ncomp, field, scratch, vel, nz, ny, nx, dt_by_dx, nu_dt_by_dx2, s);
}

int sopht_velocity_abs_sum_max_3d(int dtype, const void* const vel[3], int64_t n, void* magnitude,
                                  void* partial, int64_t partial_cap, void* out, void* stream) {
  SOPHT_REQUIRE(dtype == SOPHT_F32 || dtype == SOPHT_F64, "dtype must be SOPHT_F32 or SOPHT_F64");
  SOPHT_REQUIRE(vel && vel[0] && vel[1] && vel[2] && partial && out, "null pointer");
  SOPHT_REQUIRE(n > 0 && partial_cap > 0, "sizes must be positive");
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == SOPHT_F32 ? abs_sum_max<float>(vel, n, magnitude, partial, partial_cap, out, s)
                            : abs_sum_max<double>(vel, n, magnitude, partial, partial_cap, out, s);
}

}  // extern "C"
