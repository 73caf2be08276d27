// Fast diagonalisation by cosine transforms. The eigenbasis of the Neumann second-difference
// matrix is the cell-centred cosines v_k(i) = c_k cos(pi k (i + 1/2) / N), so applying V^T is a
// DCT-II and applying V a DCT-III. A DCT of N reals is an FFT of N complex numbers that carries
// two real lines a + i b at once (Makhoul 1980): with the even cells first and the odd ones
// behind them backwards, V = FFT(v) and w_k = exp(-i pi k / (2 N)),
//   X_k = (w_k V_k + conj(w_k) V_{N-k}) / 2         (X_N-k reads the same two values)
//   V_k = conj(w_k) (X_k - i X_{N-k}),  X_N = 0     (inverse)
// where X = X_a + i X_b: both formulas are linear over the pair, so it is never separated.
//
// Five passes per solve: x rows (two rows per transform), y columns, z columns (transform,
// division by the eigenvalue sum, inverse transform), y columns, x rows. Along y and z two
// neighbouring x cells are the pair, so a field is read as complex numbers as it lies.
// Bound by memory: 10 words per cell and component. 256^3 FP32, three components: 0.39 ms (rows
// 0.071 / 0.076, y columns 0.078 / 0.079, z 0.134, the last by its vector instructions: two
// transforms and the divisions) against 1.44 ms for the six dense products; faster at every size
// from 16^3 (0.026 against 0.041 ms) to 384^3 (1.56 against 6.95 ms).
#include <cmath>
#include <new>
#include <vector>

#include "dct_3d.h"
#include "fft_reg.h"

namespace sopht {

struct DctPlan {
  int dtype;
  int64_t n[3];     // z, y, x
  void* tw[3] = {};   // exp(-2 pi i m / N), m < N
  void* half[3] = {}; // exp(-i pi k / (2 N)), k < N
  void* lam[3] = {};  // eigenvalues, mode k at k
  int64_t plane;      // reals between the planes of the workspace
};

namespace {

using rfft::LinePlan;
using rfft::region_stride;
using rfft::static_for;
using rfft::team_fft;
using rfft::wave_sync;

// Where cell i of a line goes before the transform: even cells first, odd cells backwards.
template <int L>
__device__ __forceinline__ int dct_slot(int i) {
  return i & 1 ? L - 1 - (i >> 1) : i >> 1;
}

template <typename T>
__device__ __forceinline__ Cplx<T> dct_out(Cplx<T> w, Cplx<T> vk, Cplx<T> vm) {
  const Cplx<T> a = cmul(vk, w), b = cmulc(vm, w);
  return Cplx<T>{T(0.5) * (a.re + b.re), T(0.5) * (a.im + b.im)};
}
template <typename T>
__device__ __forceinline__ Cplx<T> dct_in(Cplx<T> w, Cplx<T> xk, Cplx<T> xm) {
  return cmulc(Cplx<T>{xk.re + xm.im, xk.im - xm.re}, w);
}

// Rows: one team per pair of rows (2q, 2q + 1).
template <typename T, int L>
struct DctRows {
  static constexpr int E = LinePlan<L>::E, TT = LinePlan<L>::T;
  static constexpr int NTEAM = 256 / TT, NT = NTEAM * TT;
  static constexpr int S = region_stride<L, false>();
  static constexpr size_t lds = (size_t(NTEAM) * S + rfft::tw_lds_size<L>()) * sizeof(Cplx<T>);
};

template <typename T, int L, bool INV>
__global__ void __launch_bounds__((DctRows<T, L>::NT))
    k_dct_rows(const T* in, T* out, int pairs, int plane_pairs, int64_t in_pad, int64_t out_pad, const Cplx<T>* tw,
               const Cplx<T>* half) {
  using R = DctRows<T, L>;
  constexpr int E = R::E, TT = R::TT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* const xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int t = threadIdx.x % TT, team = threadIdx.x / TT;
  const int q = int(blockIdx.x) * R::NTEAM + team;
  const bool live = q < pairs;
  const int plane = (live ? q : 0) / plane_pairs;
  Cplx<T>* const line = xb + team * R::S;
  Cplx<T>* const twl = xb + R::NTEAM * R::S;
  rfft::load_tw_lds<T, L>(twl, tw, threadIdx.x, R::NT);
  const T* const a = in + (live ? q : 0) * int64_t(2 * L) + plane * in_pad;
  static_for<0, E>([&](auto e_) {
    const int i = t + TT * decltype(e_)::value;
    line[INV ? i : dct_slot<L>(i)] = Cplx<T>{a[i], a[L + i]};
  });
  __syncthreads();
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int k = t + TT * e;
    if constexpr (INV) {
      const Cplx<T> xm = k == 0 ? Cplx<T>{T(0), T(0)} : line[L - k];
      v[e] = dct_in(half[k], line[k], xm);
    } else {
      v[e] = line[k];
    }
  });
  wave_sync();
  team_fft<T, L, INV, false, true>(v, line, twl, t);
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  wave_sync();
  if (!live) return;
  T* const o = out + q * int64_t(2 * L) + plane * out_pad;
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int i = t + TT * e;
    Cplx<T> r;
    if constexpr (INV) r = line[dct_slot<L>(i)];
    else r = dct_out(half[i], line[i], line[(L - i) % L]);
    o[i] = r.re;
    o[L + i] = r.im;
  });
}

// Columns: WC neighbouring pairs of cells per workgroup, one 128-byte line per row where the
// transform leaves a workgroup of at most 512 threads.
template <typename T, int L>
struct DctCols {
  static constexpr int E = LinePlan<L>::E, TT = LinePlan<L>::T;
  static constexpr int FULL = 128 / int(sizeof(Cplx<T>));
  static constexpr int WC = FULL * TT <= 512 ? FULL : 512 / TT;
  static constexpr int NT = WC * TT;
  // a column's cells take neighbouring slots of opposite parity, so two rows of WC columns (half a
  // wavefront) fall in distinct LDS banks at a stride of 2 (mod 32); at 16, which suits the
  // exchanges of teams of 16, the loads and stores meet 8 lanes deep: 128^3 FP32 80 against 63 us,
  // 192^3 FP32 218 against 170 us
  static constexpr int S = L + 2;
  static constexpr size_t lds = (size_t(WC) * S + rfft::tw_lds_size<L>()) * sizeof(Cplx<T>);
};

struct ColGeo {
  int64_t stride;  // complex elements between the cells of a column
  int64_t outer;   // complex elements between the sets of neighbouring columns
  int cols;        // neighbouring columns of a set
  int tiles;       // workgroups per set
};

template <typename T, int L, bool INV>
__global__ void __launch_bounds__((DctCols<T, L>::NT))
    k_dct_cols(ColGeo g, Cplx<T>* f, const Cplx<T>* tw, const Cplx<T>* half) {
  using C = DctCols<T, L>;
  constexpr int E = C::E, TT = C::TT, WC = C::WC, S = C::S;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* const xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int lw = tid % WC, lr = tid / WC;   // load / store role
  const int team = tid / TT, t = tid % TT;  // transform role
  const int col = int(blockIdx.x % g.tiles) * WC + lw;
  const bool live = col < g.cols;
  Cplx<T>* const p = f + int64_t(blockIdx.x / g.tiles) * g.outer + (live ? col : 0);
  Cplx<T>* const twl = xb + WC * S;
  rfft::load_tw_lds<T, L>(twl, tw, tid, C::NT);
  static_for<0, E>([&](auto e_) {
    const int i = lr + TT * decltype(e_)::value;
    xb[lw * S + (INV ? i : dct_slot<L>(i))] = p[i * g.stride];
  });
  __syncthreads();
  Cplx<T>* const line = xb + team * S;
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int k = t + TT * e;
    if constexpr (INV) {
      const Cplx<T> xm = k == 0 ? Cplx<T>{T(0), T(0)} : line[L - k];
      v[e] = dct_in(half[k], line[k], xm);
    } else {
      v[e] = line[k];
    }
  });
  wave_sync();
  team_fft<T, L, INV, false, true>(v, line, twl, t);
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  __syncthreads();
  if (!live) return;
  const Cplx<T>* const own = xb + lw * S;
  static_for<0, E>([&](auto e_) {
    const int i = lr + TT * decltype(e_)::value;
    if constexpr (INV) p[i * g.stride] = own[dct_slot<L>(i)];
    else p[i * g.stride] = dct_out(half[i], own[i], own[(L - i) % L]);
  });
}

// z columns of one (component, ky) row per set: transform, times norm / ((lz + ly) + lx) per mode
// (0 for the constant one), inverse transform.
template <typename T, int L>
__global__ void __launch_bounds__((DctCols<T, L>::NT))
    k_dct_z(ColGeo g, int ny, int64_t comp, Cplx<T>* f, const Cplx<T>* tw, const Cplx<T>* half, const T* lz,
            const T* ly, const T* lx, T norm) {
  using C = DctCols<T, L>;
  constexpr int E = C::E, TT = C::TT, WC = C::WC, S = C::S;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* const xb = reinterpret_cast<Cplx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int lw = tid % WC, lr = tid / WC;
  const int team = tid / TT, t = tid % TT;
  const int set = int(blockIdx.x / g.tiles), ky = set % ny;
  const int col0 = int(blockIdx.x % g.tiles) * WC;
  const bool live = col0 + lw < g.cols;
  Cplx<T>* const p = f + (set / ny) * comp + ky * g.outer + (live ? col0 + lw : 0);
  Cplx<T>* const twl = xb + WC * S;
  rfft::load_tw_lds<T, L>(twl, tw, tid, C::NT);
  static_for<0, E>([&](auto e_) {
    const int i = lr + TT * decltype(e_)::value;
    xb[lw * S + dct_slot<L>(i)] = p[i * g.stride];
  });
  __syncthreads();
  Cplx<T>* const line = xb + team * S;
  Cplx<T> v[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    v[e] = line[t + TT * e];
  });
  wave_sync();
  team_fft<T, L, false, false, true>(v, line, twl, t);
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  wave_sync();
  const int tcol = col0 + team < g.cols ? col0 + team : 0;
  const T lxa = lx[2 * tcol], lxb = lx[2 * tcol + 1], lyk = ly[ky];
  Cplx<T> x[E];
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int k = t + TT * e;
    const Cplx<T> r = dct_out(half[k], v[e], line[(L - k) % L]);
    const T ab = lz[k] + lyk;
    const bool null = k == 0 && ky == 0 && tcol == 0;
    x[e] = Cplx<T>{null ? T(0) : r.re * (norm / (ab + lxa)), r.im * (norm / (ab + lxb))};
  });
  wave_sync();
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = x[e];
  });
  wave_sync();
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    const int k = t + TT * e;
    const Cplx<T> xm = k == 0 ? Cplx<T>{T(0), T(0)} : line[L - k];
    v[e] = dct_in(half[k], x[e], xm);
  });
  wave_sync();
  team_fft<T, L, true, false, true>(v, line, twl, t);
  static_for<0, E>([&](auto e_) {
    constexpr int e = decltype(e_)::value;
    line[t + TT * e] = v[e];
  });
  __syncthreads();
  if (!live) return;
  const Cplx<T>* const own = xb + lw * S;
  static_for<0, E>([&](auto e_) {
    const int i = lr + TT * decltype(e_)::value;
    p[i * g.stride] = own[dct_slot<L>(i)];
  });
}

#define SOPHT_DCT_LENGTHS(X) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

// fn(integral_constant<L>) for a supported length, else an error.
template <typename Fn>
int with_length(int64_t n, Fn&& fn) {
  switch (n) {
#define X(L_) \
  case L_:    \
    return fn(std::integral_constant<int, L_>{});
    SOPHT_DCT_LENGTHS(X)
#undef X
    default: break;
  }
  set_last_error("unsupported cosine-transform length", __FILE__, __LINE__);
  return SOPHT_ERR_UNSUPPORTED;
}

template <typename T, bool INV>
int rows_pass(DctPlan* P, const T* in, T* out, int ncomp, hipStream_t s) {
  return with_length(P->n[2], [&](auto l) -> int {
    constexpr int L = decltype(l)::value;
    using R = DctRows<T, L>;
    const int plane_pairs = int(P->n[1] / 2), pairs = int(ncomp * P->n[0]) * plane_pairs;
    const int64_t pad = P->plane - P->n[1] * P->n[2];
    int rc = allow_lds(k_dct_rows<T, L, INV>, R::lds);
    if (rc) return rc;
    k_dct_rows<T, L, INV><<<ceil_div(pairs, R::NTEAM), R::NT, R::lds, s>>>(
        in, out, pairs, plane_pairs, INV ? pad : 0, INV ? 0 : pad, static_cast<const Cplx<T>*>(P->tw[2]),
        static_cast<const Cplx<T>*>(P->half[2]));
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

template <typename T, bool INV>
int y_pass(DctPlan* P, T* f, int ncomp, hipStream_t s) {
  return with_length(P->n[1], [&](auto l) -> int {
    constexpr int L = decltype(l)::value;
    using C = DctCols<T, L>;
    const int cols = int(P->n[2] / 2);
    const ColGeo g{cols, P->plane / 2, cols, ceil_div(cols, C::WC)};
    int rc = allow_lds(k_dct_cols<T, L, INV>, C::lds);
    if (rc) return rc;
    k_dct_cols<T, L, INV><<<unsigned(g.tiles * ncomp * P->n[0]), C::NT, C::lds, s>>>(
        g, reinterpret_cast<Cplx<T>*>(f), static_cast<const Cplx<T>*>(P->tw[1]),
        static_cast<const Cplx<T>*>(P->half[1]));
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

template <typename T>
int z_pass(DctPlan* P, T* f, int ncomp, hipStream_t s) {
  return with_length(P->n[0], [&](auto l) -> int {
    constexpr int L = decltype(l)::value;
    using C = DctCols<T, L>;
    const int cols = int(P->n[2] / 2), ny = int(P->n[1]);
    const int64_t plane = P->plane / 2;
    const ColGeo g{plane, cols, cols, ceil_div(cols, C::WC)};
    int rc = allow_lds(k_dct_z<T, L>, C::lds);
    if (rc) return rc;
    const T norm = T(1.0 / (double(P->n[0]) * double(P->n[1]) * double(P->n[2])));
    k_dct_z<T, L><<<unsigned(int64_t(g.tiles) * ncomp * ny), C::NT, C::lds, s>>>(
        g, ny, plane * P->n[0], reinterpret_cast<Cplx<T>*>(f), static_cast<const Cplx<T>*>(P->tw[0]),
        static_cast<const Cplx<T>*>(P->half[0]), static_cast<const T*>(P->lam[0]), static_cast<const T*>(P->lam[1]),
        static_cast<const T*>(P->lam[2]), norm);
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

template <typename T>
int solve(DctPlan* P, T* sol, const T* rhs, T* work, int ncomp, hipStream_t s, StageTimer* tm, int first) {
  int rc = rows_pass<T, false>(P, rhs, work, ncomp, s);
  if (rc) return rc;
  if (tm) tm->mark(first, s);
  if ((rc = y_pass<T, false>(P, work, ncomp, s))) return rc;
  if (tm) tm->mark(first + 1, s);
  if ((rc = z_pass<T>(P, work, ncomp, s))) return rc;
  if (tm) tm->mark(first + 2, s);
  if ((rc = y_pass<T, true>(P, work, ncomp, s))) return rc;
  if (tm) tm->mark(first + 3, s);
  if ((rc = rows_pass<T, true>(P, work, sol, ncomp, s))) return rc;
  if (tm) tm->mark(first + 4, s);
  return SOPHT_OK;
}

template <typename T>
int upload(void** dst, const std::vector<T>& h) {
  SOPHT_CHECK_HIP(hipMalloc(dst, h.size() * sizeof(T)));
  SOPHT_CHECK_HIP(hipMemcpy(*dst, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  return SOPHT_OK;
}

template <typename T>
int tables(DctPlan* P, const double* const lam[3]) {
  for (int a = 0; a < 3; ++a) {
    const int64_t n = P->n[a];
    std::vector<T> tw(2 * n), half(2 * n), l(n);
    for (int64_t k = 0; k < n; ++k) {
      const double full = 2.0 * M_PI * double(k) / double(n), h = M_PI * double(k) / (2.0 * double(n));
      tw[2 * k] = T(std::cos(full));
      tw[2 * k + 1] = T(-std::sin(full));
      half[2 * k] = T(std::cos(h));
      half[2 * k + 1] = T(-std::sin(h));
      l[k] = T(lam[a][k]);
    }
    int rc = upload(&P->tw[a], tw);
    if (!rc) rc = upload(&P->half[a], half);
    if (!rc) rc = upload(&P->lam[a], l);
    if (rc) return rc;
  }
  return SOPHT_OK;
}

}  // namespace

bool dct_supported(const int64_t n[3]) {
  for (int a = 0; a < 3; ++a) {
    bool ok = false;
#define X(L_) ok = ok || n[a] == L_;
    SOPHT_DCT_LENGTHS(X)
#undef X
    if (!ok) return false;
  }
  return true;
}

int64_t dct_plane(int dtype, const int64_t n[3]) {
  return n[1] * n[2] + 128 / (dtype == SOPHT_F32 ? 4 : 8);
}

int dct_create(int dtype, const int64_t n[3], const double* const lam[3], DctPlan** out) {
  *out = nullptr;
  DctPlan* P = new (std::nothrow) DctPlan();
  SOPHT_REQUIRE(P != nullptr, "out of host memory");
  P->dtype = dtype;
  for (int a = 0; a < 3; ++a) P->n[a] = n[a];
  P->plane = dct_plane(dtype, n);
  const int rc = dtype == SOPHT_F32 ? tables<float>(P, lam) : tables<double>(P, lam);
  if (rc) {
    dct_destroy(P);
    return rc;
  }
  *out = P;
  return SOPHT_OK;
}

void dct_destroy(DctPlan* P) {
  if (!P) return;
  for (int a = 0; a < 3; ++a)
    for (void* p : {P->tw[a], P->half[a], P->lam[a]})
      if (p) (void)hipFree(p);
  delete P;
}

int dct_solve(DctPlan* P, void* sol, const void* rhs, void* work, int ncomp, hipStream_t s, StageTimer* tm,
              int first) {
  return P->dtype == SOPHT_F32
             ? solve<float>(P, static_cast<float*>(sol), static_cast<const float*>(rhs), static_cast<float*>(work),
                            ncomp, s, tm, first)
             : solve<double>(P, static_cast<double*>(sol), static_cast<const double*>(rhs),
                             static_cast<double*>(work), ncomp, s, tm, first);
}

}  // namespace sopht
