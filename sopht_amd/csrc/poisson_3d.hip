// Free-space Poisson solve -lap(psi) = omega on an (nz, ny, nx) grid by Hockney-Eastwood
// domain doubling (UnboundedPoissonSolverPYFFTW3D.py:9-172), as pruned FFT passes on gfx950.
//
// The doubled domain is never materialised. Per component c (all components of a vector
// solve go through each pass in one launch):
//   K1 xr2c : rows (c, z<nz, y<ny): real row (zero-padded to 2nx) -> nx+1 complex, two rows
//             packed per complex FFT and separated through the conjugate pairing.
//   K2 yfwd : columns (c, z<nz, kx): y<ny inputs, zero-padded FFT of length 2ny -> all ky.
//   K3 zconv: pencils (c, ky, kx): z<nz inputs, FFT 2nz, times G^ (real, even: read from the
//             (nz+1)(ny+1)(nx+1) octant), inverse FFT, keep z<nz.
//   K4 yinv : columns: inverse FFT over all ky, keep y<ny.
//   K5 xc2r : rows: Hermitian half-spectra of two rows -> one complex inverse FFT, keep x<nx.
// All of them work in the spectral slab H[c][z<nz][ky<2ny][kx<=nx] (complex, real_t).
// G^ is the DFT of the even-reflected Green's function G = 1/(4 pi r), G(0) = 1/(4 pi dx)
// (:56-83); being real and even per axis it is a separable DCT-I of the octant, evaluated
// here in FP64 on the device, then scaled by dx^3 / (8 nz ny nx) (the dx^3 of :47-49 and the
// 1/(2N)^3 backward normalisation of pyfftw) and stored in real_t.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <new>

#include "common.h"
#include "fft_reg.h"
#include "poisson_xy.h"
#include "poisson_z.h"

struct sopht_poisson3d {
  int dtype;
  int64_t nz, ny, nx;
  double x_range, dx;
  void* slab;       // complex slab, 3 components
  void* ghat;       // real octant
  void* tw[3];      // twiddles for lengths 2nx, 2ny, 2nz (x, y, z)
  int64_t rs;       // slab row stride (complex elements)
  int64_t gz;       // G^ line stride (elements): nz + 1 rounded up to a 128-byte line
  int comps;        // components a solve may take (3, or 3 per instance of a batched class)
  int slab_comps;   // components the slab holds: all of them, or a part of a large class
  int64_t slab_bytes, ghat_bytes;
  int passes;       // 3: x and y passes fused (three-pass schedule), or 5
  int zjobs;        // three-pass z pass: jobs per workgroup, chosen at plan creation
};

namespace sopht {
namespace {

// Row passes (x): one team of T threads per row pair, RowTile::NTEAM teams per workgroup.
template <typename T, int L>
struct RowTile {
  static constexpr int E = LinePlan<L>::E, TT = LinePlan<L>::T;
  static constexpr int NTEAM = TT >= 256 ? 1 : 256 / TT;
  static constexpr int NT = NTEAM * TT;
  static constexpr int S = region_stride<L, false>();
  static constexpr size_t lds = size_t(NTEAM) * S * sizeof(Cplx<T>);
};

// Column passes (y, z): WC neighbouring kx columns per workgroup (one 128-byte line of a
// slab row), one team per column. Loads and stores run with kx fastest (lanes (w, row));
// the transform runs one team per column; LDS region w (S elements) holds column w.
template <typename T, int L>
struct ColTile {
  static constexpr int E = LinePlan<L>::E, TT = LinePlan<L>::T;
  static constexpr int WC = kColHalf ? kLineCplx<T> / 2 : kLineCplx<T>;
  static constexpr int NT = WC * TT;
  static constexpr int S = region_stride<L, true>();
  static constexpr size_t lds = size_t(WC) * S * sizeof(Cplx<T>);
};

// K1: x real-to-complex of zero-padded rows, two rows (ra, rb) per complex FFT of length
// L = 2nx; the pair is separated with A = (Z[k] + conj Z[L-k])/2, B = (Z[k] - conj Z[L-k])/(2i).
template <typename T, int L>
__global__ void __launch_bounds__((RowTile<T, L>::NT)) k1_xr2c(SlabGeom g, CompPtrs in, Cplx<T>* H,
                                                             const Cplx<T>* tw) {
  using RT = RowTile<T, L>;
  constexpr int E = RT::E, TT = RT::TT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int t = threadIdx.x % TT;
  const int team = threadIdx.x / TT;
  const int64_t rows = int64_t(g.ncomp) * g.nz * g.ny;
  const int64_t q = int64_t(blockIdx.x) * RT::NTEAM + team;
  const int64_t ra = 2 * q, rb = 2 * q + 1;
  auto row_ptr = [&](int64_t r) -> const T* {
    const int c = int(r / (g.nz * g.ny));
    const int64_t rem = r % (g.nz * g.ny);
    return static_cast<const T*>(in.get(c)) + (rem / g.ny) * in.sz + (rem % g.ny) * in.sy;
  };
  const T* pa = ra < rows ? row_ptr(ra) : nullptr;
  const T* pb = rb < rows ? row_ptr(rb) : nullptr;
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    if constexpr (e < E / 2) {  // x = t + T e < nx
      const int64_t x = t + TT * e;
      v[e] = Cplx<T>{pa ? pa[x * in.sx] : T(0), pb ? pb[x * in.sx] : T(0)};
    } else {
      v[e] = Cplx<T>{T(0), T(0)};
    }
  });
  Cplx<T>* const line = xb + team * RT::S;
  // the twiddle table in LDS, shared by the workgroup's teams
  Cplx<T>* const twl = xb + RT::NTEAM * RT::S;
  rfft::load_tw_lds<T, L>(twl, tw, threadIdx.x, RT::NT);
  __syncthreads();
  team_fft<T, L, false, true, true>(v, line, twl, t);
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  rfft::wave_sync();
  Cplx<T>* ha = ra < rows ? H + g.row_h(ra) : nullptr;
  Cplx<T>* hb = rb < rows ? H + g.row_h(rb) : nullptr;
  for (int k = t; k <= g.nx; k += TT) {
    const Cplx<T> zk = line[k];
    const Cplx<T> zm = line[(L - k) % L];
    if (ha) store_stream(ha + k, Cplx<T>{T(0.5) * (zk.re + zm.re), T(0.5) * (zk.im - zm.im)});
    if (hb) store_stream(hb + k, Cplx<T>{T(0.5) * (zk.im + zm.im), T(0.5) * (zm.re - zk.re)});
  }
}

// K2 / K4: FFT along y of columns (c, z, kx). Forward: inputs y < ny (zero padding), all
// 2ny outputs stored. Inverse: all 2ny inputs, outputs y < ny stored.
template <typename T, int L, bool INV>
__global__ void __launch_bounds__((ColTile<T, L>::NT)) k_ycols(SlabGeom g, Cplx<T>* H, const Cplx<T>* tw) {
  using CT = ColTile<T, L>;
  constexpr int E = CT::E, TT = CT::TT, WC = CT::WC, S = CT::S;
  constexpr int KIN = INV ? E : E / 2, KOUT = INV ? E / 2 : E;  // rows = TT * K
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int lw = tid % WC, lr = tid / WC;  // load / store role
  const int team = tid / TT, t = tid % TT;  // transform role
  const int64_t ncols = g.nx + 1;
  int64_t cz, kx0;  // cz = c * nz + z
  if (!col_tile(blockIdx.x, ncols, int64_t(g.ncomp) * g.nz, WC, cz, kx0)) return;
  const int c = int(cz / g.nz);
  const int64_t z = cz % g.nz;
  const int64_t kx = kx0 + lw;
  const bool live = kx < ncols;
  // a wavefront whose teams all have kx >= ncols skips its transforms
  const bool wave_live = kx0 + (tid / 64) * (64 / TT) < ncols;
  const int col = g.hi(c, int(z), 0, live ? int(kx) : 0);
  const int ys = int(g.rs);  // stride between consecutive y (or ky)
  // the twiddle table in LDS (one load per thread), read by every stage of the 8 transforms
  Cplx<T>* const twl = xb + WC * S;
  rfft::load_tw_lds<T, L>(twl, tw, tid, CT::NT);
  static_for<0, KIN>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const int y = lr + TT * k;
    xb[lw * S + y] = live ? H[col + y * ys] : Cplx<T>{T(0), T(0)};
  });
  __syncthreads();
  Cplx<T>* const line = xb + team * S;
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    if constexpr (e < KIN) v[e] = line[t + TT * e];
    else v[e] = Cplx<T>{T(0), T(0)};
  });
  rfft::wave_sync();
  if (wave_live) team_fft<T, L, INV, !INV, true>(v, line, twl, t);
  static_for<0, KOUT>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  __syncthreads();
  if (live)
    static_for<0, KOUT>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      const int y = lr + TT * k;
      if constexpr (INV)
        H[col + y * ys] = xb[lw * S + y];
      else
        store_stream(H + col + y * ys, xb[lw * S + y]);
    });
}

// pencil tiles per z-pass workgroup at most (all of them for a 3-component solve)
constexpr int kZconvJobs = 6;

// K3: z pencils (c, ky, kx): zero-padded forward FFT, times G^ (real, even), inverse FFT,
// crop to z < nz. A workgroup owns one kx tile of one |ky| = kyo and runs the pencils of
// every component at ky = kyo and ky = 2ny - kyo (the same G^ line) one after another: G^
// stays in registers, and the next pencil tile's loads are in flight during the transforms.
// G^ is stored [kyo][kx][kz], kz fastest, so a team reads its line contiguously.
template <typename T, int L>
__global__ void __launch_bounds__((ColTile<T, L>::NT)) __attribute__((amdgpu_waves_per_eu(kZconvWavesFor<T, L>))) k3_zconv(SlabGeom g, Cplx<T>* H, const T* ghat,
                                                              const Cplx<T>* tw) {
  using CT = ColTile<T, L>;
  constexpr int E = CT::E, TT = CT::TT, WC = CT::WC, S = CT::S, K = E / 2;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int lw = tid % WC, lr = tid / WC;
  const int team = tid / TT, t = tid % TT;
  const int64_t ncols = g.nx + 1;
  int64_t kyo, kx0;  // kyo = 0..ny
  if (!col_tile(blockIdx.x, ncols, g.ny + 1, WC, kyo, kx0)) return;
  // jobs (component, ky or 2ny - ky) of this workgroup: chunk blockIdx.y of kZconvJobs
  const int alljobs = (kyo == 0 || kyo == g.ny) ? g.ncomp : 2 * g.ncomp;
  const int jbeg = int(blockIdx.y) * kZconvJobs;
  if (jbeg >= alljobs) return;
  const int njobs = alljobs - jbeg < kZconvJobs ? alljobs - jbeg : kZconvJobs;
  const int64_t kx = kx0 + lw;
  const bool live = kx < ncols;
  const bool wave_live = kx0 + (tid / 64) * (64 / TT) < ncols;
  T gv[E];
  {
    const int64_t kxt = kx0 + team;
    const T* gq = ghat + int((kyo * ncols + (kxt < ncols ? kxt : 0)) * g.gz);
    static_for<0, E>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      const int kz = t + TT * e;
      gv[e] = gq[kz <= L / 2 ? kz : L - kz];
    });
  }
  const int zs = 2 * int(g.ny) * int(g.rs);  // stride between consecutive z
  // the twiddles of this thread's butterflies in the second and last stages, the same for
  // every pencil of the workgroup
  using P3 = Plan3<typename LinePlan<L>::R>;
  constexpr int R1 = at_least_1(P3::r1), R2 = at_least_1(P3::r2);
  constexpr int PER2 = at_least_1(E / R1), PER3 = at_least_1(E / R2);
  Cplx<T> w2[PER2][R1], w3[PER3][R2];
  if constexpr (last_twiddles_hoisted<L>()) {
    static_for<0, PER2>([&](auto p_) {
      constexpr int p = decltype(p_)::value;
      rfft::stage_twiddles<T, L, R1, P3::r0>(w2[p], tw, (t + p * TT) % P3::r0);
    });
    static_for<0, PER3>([&](auto p_) {
      constexpr int p = decltype(p_)::value;
      rfft::stage_twiddles<T, L, R2, P3::r0 * R1>(w3[p], tw, (t + p * TT) % (P3::r0 * R1));
    });
  }
  auto column = [&](int jl) -> int {
    const int j = jbeg + jl;
    const int c = j % g.ncomp;
    const int ky = j < g.ncomp ? int(kyo) : 2 * int(g.ny) - int(kyo);
    return g.hi(c, 0, ky, live ? int(kx) : 0);
  };
  Cplx<T> pf[K];
  auto load = [&](int j) {
    const int col = column(j);
    static_for<0, K>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      pf[k] = live ? H[col + (lr + TT * k) * zs] : Cplx<T>{T(0), T(0)};
    });
  };
  Cplx<T>* const line = xb + team * S;
  load(0);
  for (int j = 0; j < njobs; ++j) {
    static_for<0, K>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      const int z = lr + TT * k;
      xb[lw * S + z] = pf[k];
    });
    __syncthreads();
    Cplx<T> v[E];
    static_for<0, E>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      if constexpr (e < K) v[e] = line[t + TT * e];
      else v[e] = Cplx<T>{T(0), T(0)};
    });
    rfft::wave_sync();
    if (j + 1 < njobs) load(j + 1);
    if (wave_live) {
      if constexpr (last_twiddles_hoisted<L>()) {
        constexpr int R0 = P3::r0, NS3 = R0 * R1;
        rfft::stockham_stage<T, L, R0, 1, false, true>(v, line, tw, t);
        rfft::stockham_stage_given<T, L, R1, R0, false>(v, line, w2, t);
        rfft::stockham_stage_given<T, L, R2, NS3, false>(v, line, w3, t);
        static_for<0, E>([&](auto e_) {
          constexpr int e = decltype(e_)::value;
          v[e] = Cplx<T>{v[e].re * gv[e], v[e].im * gv[e]};
        });
        rfft::stockham_stage<T, L, R0, 1, true, false>(v, line, tw, t);
        rfft::stockham_stage_given<T, L, R1, R0, true>(v, line, w2, t);
        rfft::stockham_stage_given<T, L, R2, NS3, true>(v, line, w3, t);
      } else {
        team_fft<T, L, false, true>(v, line, tw, t);
        static_for<0, E>([&](auto e_) {
          constexpr int e = decltype(e_)::value;
          v[e] = Cplx<T>{v[e].re * gv[e], v[e].im * gv[e]};
        });
        team_fft<T, L, true>(v, line, tw, t);
      }
    }
    static_for<0, K>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      line[t + TT * e] = v[e];
    });
    __syncthreads();
    if (live) {
      const int col = column(j);
      static_for<0, K>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        const int z = lr + TT * k;
        store_stream(H + col + z * zs, xb[lw * S + z]);
      });
    }
    __syncthreads();
  }
}

// K5: x complex-to-real of two rows per complex inverse FFT, crop to x < nx. The Hermitian
// half spectra A, B (kx <= nx) of rows ra, rb become Z[k] = A[k] + i B[k],
// Z[L-k] = conj(A[k]) + i conj(B[k]); imaginary parts at kx = 0 and nx are dropped
// (irfft semantics).
template <typename T, int L, bool ACC>
__global__ void __launch_bounds__((RowTile<T, L>::NT)) k5_xc2r(SlabGeom g, const Cplx<T>* H, CompPtrsW out,
                                                             const Cplx<T>* tw) {
  using RT = RowTile<T, L>;
  constexpr int E = RT::E, TT = RT::TT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int t = threadIdx.x % TT;
  const int team = threadIdx.x / TT;
  const int64_t rows = int64_t(g.ncomp) * g.nz * g.ny;
  const int64_t q = int64_t(blockIdx.x) * RT::NTEAM + team;
  const int64_t ra = 2 * q, rb = 2 * q + 1;
  const int64_t nx = g.nx;
  const Cplx<T>* ha = ra < rows ? H + g.row_h(ra) : nullptr;
  const Cplx<T>* hb = rb < rows ? H + g.row_h(rb) : nullptr;
  Cplx<T>* const line = xb + team * RT::S;
  // the twiddle table in LDS, shared by the workgroup's teams (one barrier, below)
  Cplx<T>* const twl = xb + RT::NTEAM * RT::S;
  rfft::load_tw_lds<T, L>(twl, tw, threadIdx.x, RT::NT);
  for (int k = t; k <= nx; k += TT) {
    Cplx<T> a = {T(0), T(0)}, bb = {T(0), T(0)};
    if (ha) a = ha[k];
    if (hb) bb = hb[k];
    if (k == 0 || k == nx) {
      a.im = T(0);
      bb.im = T(0);
    }
    line[k] = Cplx<T>{a.re - bb.im, a.im + bb.re};
    if (k > 0 && k < nx) line[L - k] = Cplx<T>{a.re + bb.im, bb.re - a.im};
  }
  rfft::wave_sync();
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    v[e] = line[t + TT * e];
  });
  __syncthreads();  // the twiddle table is complete
  team_fft<T, L, true, false, true>(v, line, twl, t);
  auto row_ptr = [&](int64_t r) -> T* {
    const int c = int(r / (g.nz * g.ny));
    const int64_t rem = r % (g.nz * g.ny);
    return static_cast<T*>(out.get(c)) + (rem / g.ny) * out.sz + (rem % g.ny) * out.sy;
  };
  T* pa = ra < rows ? row_ptr(ra) : nullptr;
  T* pb = rb < rows ? row_ptr(rb) : nullptr;
  static_for<0, E / 2>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int64_t x = t + TT * e;
    if constexpr (ACC) {  // solution += result (the adjoint adds G psi_bar to omega_bar)
      if (pa) pa[x * out.sx] += v[e].re;
      if (pb) pb[x * out.sx] += v[e].im;
    } else {
      if (pa) __builtin_nontemporal_store(v[e].re, pa + x * out.sx);
      if (pb) __builtin_nontemporal_store(v[e].im, pb + x * out.sx);
    }
  });
}

// ------------------------------------------------------------------ Green's function octant
// g[z][y][x] = 1/(4 pi r dx) on integer offsets, g[0] = 1/(4 pi dx), in FP64.
__global__ void k_green_octant(double* g, int64_t nz1, int64_t ny1, int64_t nx1, double dx) {
  const int64_t n = nz1 * ny1 * nx1;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t x = i % nx1, y = (i / nx1) % ny1, z = i / (nx1 * ny1);
    const double r = sqrt(double(x * x + y * y + z * z)) * dx;
    g[i] = (i == 0) ? 1.0 / (4.0 * M_PI * dx) : 1.0 / (4.0 * M_PI * r);
  }
}

// DCT-I along one axis of the octant (length n+1 per line, doubled period 2n):
// out[k] = g[0] + (-1)^k g[n] + 2 sum_{j=1}^{n-1} g[j] cos(pi j k / n), k = 0..n.
// `stride` is the element stride of the axis, `lines` enumerates all other indices through
// (outer, inner) with inner extent `inner` (= stride).
__global__ void k_dct1_axis(const double* in, double* out, int64_t n, int64_t stride,
                            int64_t inner, int64_t outer, const double* cos_tab) {
  const int64_t total = outer * (n + 1) * inner;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t in_i = i % inner;
    const int64_t k = (i / inner) % (n + 1);
    const int64_t o = i / (inner * (n + 1));
    const double* line = in + o * (n + 1) * inner + in_i;
    double acc = line[0] + ((k & 1) ? -line[n * stride] : line[n * stride]);
    double s = 0.0;
    for (int64_t j = 1; j < n; ++j) s += line[j * stride] * cos_tab[(j * k) % (2 * n)];
    out[i] = acc + 2.0 * s;
  }
}

// scaled, converted to real_t and stored [y][x][z] (z fastest, line stride gz)
template <typename T>
__global__ void k_ghat_store(const double* in, T* out, int64_t nz1, int64_t ny1, int64_t nx1,
                             int64_t gz, double s) {
  const int64_t n = nz1 * ny1 * nx1;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t z = i % nz1, yx = i / nz1;  // output order: consecutive threads, consecutive z
    const int64_t x = yx % nx1, y = yx / nx1;
    out[yx * gz + z] = T(in[(z * ny1 + y) * nx1 + x] * s);
  }
}

// ------------------------------------------------------------------ dispatch on length
#define SOPHT_FFT_LENGTHS(X) \
  X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(768) X(1024)

bool length_supported(int64_t L) {
#define X(n) if (L == n) return true;
  SOPHT_FFT_LENGTHS(X)
#undef X
  return false;
}

template <typename T>
int launch_k1(int64_t L, SlabGeom g, CompPtrs in, Cplx<T>* H, const Cplx<T>* tw, hipStream_t s) {
  const int64_t rows = int64_t(g.ncomp) * g.nz * g.ny;
  const int64_t pairs = (rows + 1) / 2;
#define X(n)                                                                          \
  if (L == n) {                                                                       \
    using RT = RowTile<T, n>;                                                         \
    k1_xr2c<T, n><<<ceil_div(pairs, RT::NTEAM), RT::NT, RT::lds + rfft::tw_lds_size<n>() * sizeof(Cplx<T>), s>>>(g, in, H, tw); \
    SOPHT_CHECK_LAUNCH();                                                             \
    return SOPHT_OK;                                                                  \
  }
  SOPHT_FFT_LENGTHS(X)
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

template <typename T, bool INV>
int launch_ycols(int64_t L, SlabGeom g, Cplx<T>* H, const Cplx<T>* tw, hipStream_t s) {
#define X(n)                                                                          \
  if (L == n) {                                                                       \
    using CT = ColTile<T, n>;                                                         \
    const int64_t nb = col_tile_blocks(g.nx + 1, int64_t(g.ncomp) * g.nz, CT::WC);    \
    k_ycols<T, n, INV><<<nb, CT::NT, CT::lds + rfft::tw_lds_size<n>() * sizeof(Cplx<T>), s>>>(g, H, tw);   \
    SOPHT_CHECK_LAUNCH();                                                             \
    return SOPHT_OK;                                                                  \
  }
  SOPHT_FFT_LENGTHS(X)
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

template <typename T>
int launch_k3(int64_t L, SlabGeom g, Cplx<T>* H, const T* ghat, const Cplx<T>* tw,
              hipStream_t s) {
#define X(n)                                                                          \
  if (L == n) {                                                                       \
    using CT = ColTile<T, n>;                                                         \
    const int64_t nb = col_tile_blocks(g.nx + 1, g.ny + 1, CT::WC);                   \
    const unsigned nch = unsigned((2 * g.ncomp + kZconvJobs - 1) / kZconvJobs);        \
    k3_zconv<T, n><<<dim3(unsigned(nb), nch), CT::NT, CT::lds, s>>>(g, H, ghat, tw);   \
    SOPHT_CHECK_LAUNCH();                                                             \
    return SOPHT_OK;                                                                  \
  }
  SOPHT_FFT_LENGTHS(X)
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

template <typename T>
int launch_k5(int64_t L, SlabGeom g, const Cplx<T>* H, CompPtrsW out, const Cplx<T>* tw,
              hipStream_t s, bool acc) {
  const int64_t rows = int64_t(g.ncomp) * g.nz * g.ny;
  const int64_t pairs = (rows + 1) / 2;
#define X(n)                                                                          \
  if (L == n) {                                                                       \
    using RT = RowTile<T, n>;                                                         \
    if (acc)                                                                          \
      k5_xc2r<T, n, true><<<ceil_div(pairs, RT::NTEAM), RT::NT, RT::lds + rfft::tw_lds_size<n>() * sizeof(Cplx<T>), s>>>(g, H, out, tw); \
    else                                                                              \
      k5_xc2r<T, n, false><<<ceil_div(pairs, RT::NTEAM), RT::NT, RT::lds + rfft::tw_lds_size<n>() * sizeof(Cplx<T>), s>>>(g, H, out, tw); \
    SOPHT_CHECK_LAUNCH();                                                             \
    return SOPHT_OK;                                                                  \
  }
  SOPHT_FFT_LENGTHS(X)
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

SlabGeom slab_geom(const sopht_poisson3d* P, int ncomp) {
  return SlabGeom{P->nz, P->ny, P->nx, P->rs, P->gz, ncomp};
}

// ncomp <= 3 components by value (sol, rhs), or any number from device pointer tables
// (sol_tab, rhs_tab; the slab must hold ncomp components).
template <typename T>
int solve_impl(sopht_poisson3d* P, int ncomp, void* const sol[3], const int64_t* ss,
               const void* const rhs[3], const int64_t* rs, hipStream_t s,
               StageTimer* timer = nullptr, int first_stage = 0, void* const* sol_tab = nullptr,
               const void* const* rhs_tab = nullptr, bool accumulate = false) {
  if (ncomp > P->slab_comps) {
    set_last_error("more components than the Poisson plan's slab holds", __FILE__, __LINE__);
    return SOPHT_ERR_INVALID;
  }
  const SlabGeom g = slab_geom(P, ncomp);
  CompPtrs in;
  CompPtrsW out;
  in.tab = rhs_tab;
  out.tab = sol_tab;
  for (int c = 0; c < 3; ++c) {
    in.p[c] = (!rhs_tab && c < ncomp) ? rhs[c] : nullptr;
    out.p[c] = (!sol_tab && c < ncomp) ? sol[c] : nullptr;
  }
  in.sz = rs[0]; in.sy = rs[1]; in.sx = rs[2];
  out.sz = ss[0]; out.sy = ss[1]; out.sx = ss[2];
  Cplx<T>* H = static_cast<Cplx<T>*>(P->slab);
  const Cplx<T>* twx = static_cast<const Cplx<T>*>(P->tw[0]);
  const Cplx<T>* twy = static_cast<const Cplx<T>*>(P->tw[1]);
  const Cplx<T>* twz = static_cast<const Cplx<T>*>(P->tw[2]);
  int rc;
  auto mark = [&](int i) {
    if (timer) timer->mark(first_stage + i, s);
  };
  if (P->passes == 3) {
    if ((rc = poisson_xy_fwd(2 * P->nx, 2 * P->ny, g, in, H, twx, twy, s))) return rc;
    mark(0);
    if ((rc = poisson_z_rows(2 * P->nz, g, H, static_cast<const T*>(P->ghat), twz, s, P->zjobs))) return rc;
    mark(1);
    rc = accumulate ? poisson_yx_inv_add(2 * P->nx, 2 * P->ny, g, H, out, twx, twy, s)
                    : poisson_yx_inv(2 * P->nx, 2 * P->ny, g, H, out, twx, twy, s);
    mark(2);
    return rc;
  }
  if ((rc = launch_k1<T>(2 * P->nx, g, in, H, twx, s))) return rc;
  mark(0);
  if ((rc = launch_ycols<T, false>(2 * P->ny, g, H, twy, s))) return rc;
  mark(1);
  if ((rc = launch_k3<T>(2 * P->nz, g, H, static_cast<const T*>(P->ghat), twz, s))) return rc;
  mark(2);
  if ((rc = launch_ycols<T, true>(2 * P->ny, g, H, twy, s))) return rc;
  mark(3);
  rc = launch_k5<T>(2 * P->nx, g, H, out, twx, s, accumulate);
  mark(4);
  return rc;
}

// exp(-2 pi i m / L) in FP64 with exact argument reduction to the first octant.
void twiddle_fp64(int64_t L, int64_t m, double& re, double& im) {
  m %= L;
  // angle = 2 pi m / L; use symmetry to keep the argument small
  const long double a = 2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)L;
  re = double(cosl(a));
  im = -double(sinl(a));
}

template <typename T>
int upload_twiddles(int64_t L, void** dst, hipStream_t s) {
  Cplx<T>* host = static_cast<Cplx<T>*>(malloc(sizeof(Cplx<T>) * L));
  if (!host) return SOPHT_ERR_INVALID;
  for (int64_t m = 0; m < L; ++m) {
    double re, im;
    twiddle_fp64(L, m, re, im);
    host[m] = Cplx<T>{T(re), T(im)};
  }
  hipError_t e = hipMalloc(dst, sizeof(Cplx<T>) * L);
  if (e == hipSuccess) e = hipMemcpyAsync(*dst, host, sizeof(Cplx<T>) * L, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  free(host);
  SOPHT_CHECK_HIP(e);
  return SOPHT_OK;
}

int build_ghat(sopht_poisson3d* P, hipStream_t s) {
  const int64_t nz1 = P->nz + 1, ny1 = P->ny + 1, nx1 = P->nx + 1;
  const int64_t n = nz1 * ny1 * nx1;
  double *a = nullptr, *b = nullptr, *ct = nullptr;
  SOPHT_CHECK_HIP(hipMalloc(&a, n * sizeof(double)));
  SOPHT_CHECK_HIP(hipMalloc(&b, n * sizeof(double)));
  const int64_t nmax = std::max(P->nx, std::max(P->ny, P->nz));
  SOPHT_CHECK_HIP(hipMalloc(&ct, 2 * nmax * sizeof(double)));
  double* host = static_cast<double*>(malloc(2 * nmax * sizeof(double)));
  const int blocks = std::min<int64_t>(65536, (n + 255) / 256);
  k_green_octant<<<blocks, 256, 0, s>>>(a, nz1, ny1, nx1, P->dx);
  SOPHT_CHECK_LAUNCH();
  // axis passes: x (stride 1), y (stride nx1), z (stride nx1*ny1)
  struct Ax { int64_t n, stride, inner, outer; } axes[3] = {
      {P->nx, 1, 1, nz1 * ny1},
      {P->ny, nx1, nx1, nz1},
      {P->nz, nx1 * ny1, nx1 * ny1, 1}};
  double* src = a;
  double* dst = b;
  for (const Ax& ax : axes) {
    for (int64_t m = 0; m < 2 * ax.n; ++m)
      host[m] = double(cosl(3.14159265358979323846264338327950288L * (long double)m / (long double)ax.n));
    SOPHT_CHECK_HIP(hipMemcpyAsync(ct, host, 2 * ax.n * sizeof(double), hipMemcpyHostToDevice, s));
    SOPHT_CHECK_HIP(hipStreamSynchronize(s));
    k_dct1_axis<<<blocks, 256, 0, s>>>(src, dst, ax.n, ax.stride, ax.inner, ax.outer, ct);
    SOPHT_CHECK_LAUNCH();
    std::swap(src, dst);
  }
  const double scale = P->dx * P->dx * P->dx / (8.0 * double(P->nz) * double(P->ny) * double(P->nx));
  if (P->dtype == SOPHT_F32)
    k_ghat_store<float><<<blocks, 256, 0, s>>>(src, static_cast<float*>(P->ghat), nz1, ny1, nx1, P->gz, scale);
  else
    k_ghat_store<double><<<blocks, 256, 0, s>>>(src, static_cast<double*>(P->ghat), nz1, ny1, nx1, P->gz, scale);
  SOPHT_CHECK_LAUNCH();
  SOPHT_CHECK_HIP(hipStreamSynchronize(s));
  free(host);
  SOPHT_CHECK_HIP(hipFree(a));
  SOPHT_CHECK_HIP(hipFree(b));
  SOPHT_CHECK_HIP(hipFree(ct));
  return SOPHT_OK;
}

// Jobs per workgroup of the three-pass z pass: the fewer, the more workgroups (and the more
// G^ staging). Each candidate runs once on the plan's own slab (zeroed) and stream, after one run
// that is not timed, and the fastest is kept: five z passes. Choices that one run does not tell
// apart are within 2% of a solve; the wrong end of the range costs up to 60% (48^3).
// SOPHT_POISSON_ZJOBS in the environment fixes the choice instead. Results do
// not depend on it: a pencil's arithmetic is the same in any workgroup.
template <typename T>
int tune_zpass(sopht_poisson3d* P, hipStream_t s) {
  P->zjobs = kZrowJobs;
  if (P->passes != 3) return SOPHT_OK;
  if (const char* forced = std::getenv("SOPHT_POISSON_ZJOBS")) {
    const int j = std::atoi(forced);
    if (j >= 1) P->zjobs = j;
    return SOPHT_OK;
  }
  const SlabGeom g = slab_geom(P, P->slab_comps);
  Cplx<T>* H = static_cast<Cplx<T>*>(P->slab);
  const T* gh = static_cast<const T*>(P->ghat);
  const Cplx<T>* twz = static_cast<const Cplx<T>*>(P->tw[2]);
  SOPHT_CHECK_HIP(hipMemsetAsync(P->slab, 0, size_t(P->slab_bytes), s));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  SOPHT_CHECK_HIP(hipEventCreate(&e0));
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    set_last_error("hipEventCreate failed", __FILE__, __LINE__);
    return SOPHT_ERR_HIP;
  }
  int rc = SOPHT_OK;
  float best = -1.f;
  rc = poisson_z_rows(2 * P->nz, g, H, gh, twz, s, 1);  // warm-up
  for (const int jobs : {1, 2, 3, 6}) {
    if (rc) break;
    if (jobs > 2 * g.ncomp) continue;
    if (hipEventRecord(e0, s) != hipSuccess) { rc = SOPHT_ERR_HIP; break; }
    if ((rc = poisson_z_rows(2 * P->nz, g, H, gh, twz, s, jobs))) break;
    float ms = 0.f;
    if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
      rc = SOPHT_ERR_HIP;
      break;
    }
    if (best < 0.f || ms < best) {
      best = ms;
      P->zjobs = jobs;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc == SOPHT_ERR_HIP) set_last_error("timing the z pass at plan creation failed", __FILE__, __LINE__);
  return rc;
}

}  // namespace

int poisson_stage_count(const sopht_poisson3d* P) { return P->passes; }

int poisson_vector_solve_timed(sopht_poisson3d* P, void* const sol[3], const int64_t* ss,
                               const void* const rhs[3], const int64_t* rs, hipStream_t s,
                               StageTimer* timer, int first_stage) {
  return P->dtype == SOPHT_F32 ? solve_impl<float>(P, 3, sol, ss, rhs, rs, s, timer, first_stage)
                               : solve_impl<double>(P, 3, sol, ss, rhs, rs, s, timer, first_stage);
}

int poisson_vector_solve_accumulate(sopht_poisson3d* P, void* const sol[3], const int64_t* ss,
                                    const void* const rhs[3], const int64_t* rs, hipStream_t s) {
  return P->dtype == SOPHT_F32
             ? solve_impl<float>(P, 3, sol, ss, rhs, rs, s, nullptr, 0, nullptr, nullptr, true)
             : solve_impl<double>(P, 3, sol, ss, rhs, rs, s, nullptr, 0, nullptr, nullptr, true);
}

int poisson_table_solve(sopht_poisson3d* P, int ncomp, void* const* sol_tab, const int64_t* ss,
                        const void* const* rhs_tab, const int64_t* rs, hipStream_t s) {
  SOPHT_REQUIRE(ncomp <= P->comps, "more components than the Poisson plan was created for");
  for (int c = 0; c < ncomp; c += P->slab_comps) {
    const int n = std::min(ncomp - c, P->slab_comps);
    const int rc = P->dtype == SOPHT_F32
                       ? solve_impl<float>(P, n, nullptr, ss, nullptr, rs, s, nullptr, 0, sol_tab + c, rhs_tab + c)
                       : solve_impl<double>(P, n, nullptr, ss, nullptr, rs, s, nullptr, 0, sol_tab + c, rhs_tab + c);
    if (rc) return rc;
  }
  return SOPHT_OK;
}

}  // namespace sopht

using namespace sopht;

extern "C" {

int sopht_poisson3d_create(int dtype, int64_t nz, int64_t ny, int64_t nx, double x_range,
                           void* stream, sopht_poisson3d** out) {
  return sopht::poisson_create(dtype, nz, ny, nx, x_range, 3, stream, out);
}

}  // extern "C"

namespace sopht {

int poisson_create(int dtype, int64_t nz, int64_t ny, int64_t nx, double x_range, int comps,
                   void* stream, sopht_poisson3d** out) {
  SOPHT_REQUIRE(out != nullptr, "plan pointer is null");
  SOPHT_REQUIRE(comps >= 1, "a Poisson plan holds at least one component");
  *out = nullptr;
  SOPHT_REQUIRE(dtype == SOPHT_F32 || dtype == SOPHT_F64, "dtype must be SOPHT_F32 or SOPHT_F64");
  SOPHT_REQUIRE(nz > 0 && ny > 0 && nx > 0 && x_range > 0, "grid sizes and x_range must be positive");
  if (!length_supported(2 * nx) || !length_supported(2 * ny) || !length_supported(2 * nz)) {
    set_last_error("unsupported Poisson grid size: 2*n must be one of 8, 12, 16, 24, 32, 48, 64, "
                   "96, 128, 192, 256, 384, 512, 768, 1024", __FILE__, __LINE__);
    return SOPHT_ERR_UNSUPPORTED;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  sopht_poisson3d* P = new (std::nothrow) sopht_poisson3d();
  SOPHT_REQUIRE(P != nullptr, "out of host memory");
  P->dtype = dtype;
  P->nz = nz; P->ny = ny; P->nx = nx;
  P->x_range = x_range;
  P->dx = x_range / double(nx);
  if (dtype == SOPHT_F32) P->dx = double(float(P->dx));  // the reference's real_t(dx)
  const size_t cs = dtype == SOPHT_F32 ? sizeof(Cplx<float>) : sizeof(Cplx<double>);
  const size_t rsz = dtype == SOPHT_F32 ? sizeof(float) : sizeof(double);
  // the three-pass schedule where its kernels are built (2 nx and 2 ny in SOPHT_XY_LENGTHS of
  // the precision, 2 nz in SOPHT_ZROW_LENGTHS); SOPHT_POISSON_PASSES=5 in the environment
  // keeps the five-pass one. Per vector solve it was never slower at any pair of lengths
  // (five / three passes, ms): FP32 48^3 0.053 / 0.038; nz, ny, nx = 128, 96, 192 0.211 / 0.180;
  // 48, 128, 256 0.171 / 0.153; 256, 128, 256 0.670 / 0.573; 256, 192, 256 1.10 / 0.98; FP64
  // 48^3 0.068 / 0.046; 64^3 0.079 / 0.057; 96^3 0.192 / 0.151; 128^3 0.330 / 0.330; 192, 128,
  // 192 0.897 / 0.826; 192^3 1.485 / 1.194
  const char* forced = std::getenv("SOPHT_POISSON_PASSES");
  const bool five = forced != nullptr && std::atoi(forced) == 5;
  P->passes = (!five && kRowPad && xy_length_supported(dtype, 2 * nx) && xy_length_supported(dtype, 2 * ny) &&
               zrow_length_supported(2 * nz)) ? 3 : 5;
  // rows of whole 128-byte lines, and of whole column tiles of the three-pass slab
  auto row_stride = [&](int passes) -> int64_t {
    const int64_t line = passes == 3 ? std::max<int64_t>(128 / cs, kSlabTile) : int64_t(128 / cs);
    return kRowPad ? round_up(nx + 1, line) : nx + 1;
  };
  // The passes index the slab with 32 bits. FP64 rows of the three-pass slab are padded further than
  // the five-pass ones (192^3: 208 against 200), so some classes of many members (47 and 48 of 192^3)
  // exceed it only for that: they are solved in parts, each member by the schedule it has alone.
  auto elements = [&](int64_t c, int passes) -> int64_t { return c * nz * 2 * ny * row_stride(passes); };
  constexpr int64_t most = (int64_t(1) << 31) - 1;
  P->comps = P->slab_comps = comps;
  if (elements(comps, P->passes) > most && elements(comps, 5) <= most) {
    const int64_t at_once = most / elements(1, P->passes);
    P->slab_comps = ceil_div(comps, ceil_div(comps, at_once));
  }
  const int64_t rs = row_stride(P->passes);
  P->rs = rs;
  P->gz = kRowPad ? round_up(nz + 1, int64_t(128 / rsz)) : nz + 1;
  P->slab_bytes = elements(P->slab_comps, P->passes) * int64_t(cs);
  if (elements(P->slab_comps, P->passes) > most) {
    delete P;
    set_last_error("Poisson grid too large: the spectral slab must have < 2^31 elements", __FILE__, __LINE__);
    return SOPHT_ERR_UNSUPPORTED;
  }
  P->ghat_bytes = (ny + 1) * (nx + 1) * P->gz * int64_t(rsz);
  int rc = SOPHT_OK;
  auto fail = [&](int code) {
    sopht_poisson3d_destroy(P);
    return code;
  };
  if (hipMalloc(&P->slab, P->slab_bytes) != hipSuccess) {
    set_last_error("hipMalloc of the Poisson slab failed", __FILE__, __LINE__);
    return fail(SOPHT_ERR_HIP);
  }
  if (hipMalloc(&P->ghat, P->ghat_bytes) != hipSuccess) {
    set_last_error("hipMalloc of the Green's function failed", __FILE__, __LINE__);
    return fail(SOPHT_ERR_HIP);
  }
  const int64_t Ls[3] = {2 * nx, 2 * ny, 2 * nz};
  for (int a = 0; a < 3; ++a) {
    rc = dtype == SOPHT_F32 ? upload_twiddles<float>(Ls[a], &P->tw[a], s)
                            : upload_twiddles<double>(Ls[a], &P->tw[a], s);
    if (rc) return fail(rc);
  }
  if ((rc = build_ghat(P, s))) return fail(rc);
  rc = dtype == SOPHT_F32 ? tune_zpass<float>(P, s) : tune_zpass<double>(P, s);
  if (rc) return fail(rc);
  *out = P;
  return SOPHT_OK;
}

}  // namespace sopht

extern "C" {

int sopht_poisson3d_destroy(sopht_poisson3d* P) {
  if (!P) return SOPHT_OK;
  if (P->slab) (void)hipFree(P->slab);
  if (P->ghat) (void)hipFree(P->ghat);
  for (int a = 0; a < 3; ++a)
    if (P->tw[a]) (void)hipFree(P->tw[a]);
  delete P;
  return SOPHT_OK;
}

int64_t sopht_poisson3d_scratch_bytes(const sopht_poisson3d* P) {
  return P ? P->slab_bytes + P->ghat_bytes : 0;
}

int sopht_poisson3d_schedule(const sopht_poisson3d* P, int* passes, int* zpass_jobs) {
  SOPHT_REQUIRE(P != nullptr, "plan is null");
  if (passes) *passes = P->passes;
  if (zpass_jobs) *zpass_jobs = P->passes == 3 ? P->zjobs : 0;
  return SOPHT_OK;
}

int sopht_poisson3d_solve(sopht_poisson3d* P, void* sol, const int64_t* ss, const void* rhs,
                          const int64_t* rs, void* stream) {
  SOPHT_REQUIRE(P != nullptr, "plan is null");
  void* const so[3] = {sol, nullptr, nullptr};
  const void* const rh[3] = {rhs, nullptr, nullptr};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return P->dtype == SOPHT_F32 ? solve_impl<float>(P, 1, so, ss, rh, rs, s)
                               : solve_impl<double>(P, 1, so, ss, rh, rs, s);
}

int sopht_poisson3d_vector_solve(sopht_poisson3d* P, void* const sol[3], const int64_t* ss,
                                 const void* const rhs[3], const int64_t* rs, void* stream) {
  SOPHT_REQUIRE(P != nullptr, "plan is null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  return P->dtype == SOPHT_F32 ? solve_impl<float>(P, 3, sol, ss, rhs, rs, s)
                               : solve_impl<double>(P, 3, sol, ss, rhs, rs, s);
}

}  // extern "C"
