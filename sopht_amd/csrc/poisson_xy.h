// Passes A and C of the three-pass Poisson schedule: the x and y transforms of a plane's row
// class in one kernel. Built for every pair of lengths 2 nx, 2 ny below, one translation unit
// per pass and precision.
#pragma once

#include "poisson_slab.h"

// Line lengths of x and y that have the kernels. (FP64 lines of 512 points leave the passes
// without registers; those plans keep five passes.)
#define SOPHT_XY_LENGTHS_F64(X) X(96) X(128) X(192) X(256) X(384)
#define SOPHT_XY_LENGTHS(X) SOPHT_XY_LENGTHS_F64(X) X(512)

namespace sopht {

inline bool xy_length_supported(int dtype, int64_t L) {
  if (dtype == SOPHT_F64 && L == 512) return false;
#define X(n) if (L == n) return true;
  SOPHT_XY_LENGTHS(X)
#undef X
  return false;
}

// Pass A: fields -> slab rows y1 L2 + k2; pass C: slab rows -> fields, and its adding form.
#define SOPHT_XY_PASSES(T)                                                                             \
  int poisson_xy_fwd(int64_t LX, int64_t LY, SlabGeom g, CompPtrs in, Cplx<T>* H, const Cplx<T>* twx,     \
                     const Cplx<T>* twy, hipStream_t s);                                                 \
  int poisson_yx_inv(int64_t LX, int64_t LY, SlabGeom g, const Cplx<T>* H, CompPtrsW out,                 \
                     const Cplx<T>* twx, const Cplx<T>* twy, hipStream_t s);                             \
  int poisson_yx_inv_add(int64_t LX, int64_t LY, SlabGeom g, const Cplx<T>* H, CompPtrsW out,             \
                         const Cplx<T>* twx, const Cplx<T>* twy, hipStream_t s);
SOPHT_XY_PASSES(float)
SOPHT_XY_PASSES(double)
#undef SOPHT_XY_PASSES

namespace {

// ------------------------------------------------------------------ three-pass schedule
// The y transform (length LY = 2 ny = 4 L2) is split by decimation in time, y = 4 y2 + y1 and
// ky = k2 + L2 k1:
//   Y[k2 + L2 k1] = sum_{y1<4} w4^{y1 k1} * [ w_LY^{y1 k2} * sum_{y2} x[4 y2 + y1] w_L2^{y2 k2} ]
// and its inverse the same way with conjugate roots. Pass A (ka_xy_fwd) runs per (c, z, y1):
// the x transforms of the rows y = 4 y2 + y1, then the inner L2-point sums over y2 and the
// twiddle, stored in slab row y1 L2 + k2. The z pass (k3_zconv4) applies the 4-point sums
// over y1 before its convolution and their inverse after it. Pass C (kc_yx_inv) undoes the
// twiddle and the inner sums and runs the inverse x transforms. So the x-pass outputs
// (K1 -> K2) and the inverse y-pass outputs (K4 -> K5) of the five-pass schedule never reach
// HBM: 24 words per cell fewer.

// Elements of a thread's half spectrum per chunk of the y sums: the most that divide EX / 2 and
// keep the chunk's column teams and staging rows within the workgroup, for chunks of up to 64
// columns (128 where TX = 64 would leave one element; 96 columns of a 384 x 384 FP64 plane would
// not fit the LDS).
constexpr int xy_chunk_elems(int EX, int TX, int T2, int NT, int L2) {
  int best = 1;
  for (int k = 1; k == 1 || k * TX <= (TX == 64 ? 128 : 64); ++k) {
    const int cw = k * TX;
    if ((EX / 2) % k == 0 && cw * T2 <= NT && NT % cw == 0 && L2 % (NT / cw) == 0) best = k;
  }
  return best;
}

// Teams of a workgroup: the most, up to 1024 threads, that share the row pairs evenly; half as
// many, with two pairs each, where more than 512 threads would leave half of them without a
// column in the y sums' chunks (64 columns of T2 threads): two workgroups then fit a CU and
// overlap. 128 x 256 (ny x nx), 256 planes: 0.565 ms per solve against 0.642 with one pair per
// team; 96 x 256: 0.473 against 0.515.
constexpr int xy_teams(int pairs, int TX, int T2) {
  int best = 1;
  for (int k = 1; k <= pairs && k * TX <= 1024; ++k)
    if (pairs % k == 0) best = k;
  if (best * TX > 512 && best % 2 == 0 && best * TX >= 2 * 64 * T2) best /= 2;
  return best;
}

// A workgroup of pass A or C holds the ny / 4 rows of its (c, z, y1) as row pairs (two real
// rows per complex x transform), PPT pairs per team of TX threads. The y sums run on chunks of
// CW = KC TX columns (kx = CW ch + TX kk + t, element KC ch + kk of every x thread; the last
// chunk is kx = nx alone), one team of T2 threads per column, staged through LDS. Lines of
// fewer than 64 x threads take KC > 1, so a chunk still spans a wavefront's width of columns
// and the workgroup passes fewer chunk barriers; so do lines of 64 x threads whose column teams
// are small enough for 128 columns (48 x 256, 256 planes: 0.235 ms per solve against 0.253).
template <typename T, int LX, int LY>
struct XYPass {
  static constexpr int EX = LinePlan<LX>::E, TX = LinePlan<LX>::T;
  static constexpr int L2 = LY / 4;
  static constexpr int E2 = LinePlan<L2>::E, T2 = LinePlan<L2>::T;
  static constexpr int NY2 = L2 / 2;      // rows of a workgroup (y2 < ny / 4)
  static constexpr int NPAIR = NY2 / 2;
  static constexpr int NTEAM = xy_teams(NPAIR, TX, T2);
  static constexpr int PPT = NPAIR / NTEAM;  // row pairs per x team
  static constexpr int NT = NTEAM * TX;
  static constexpr int KC = xy_chunk_elems(EX, TX, T2, NT, L2);
  static constexpr int CW = KC * TX;         // columns per chunk: kx = CW ch + kk TX + t, kk < KC
  static constexpr int NCH = EX / 2 / KC + 1;  // the last chunk is kx = nx alone
  static constexpr int SX = region_stride<LX, false>();
  static constexpr int S2 = region_stride<L2, true>();
  // staging tile [row][P]: the column teams' accesses (T2 rows of LANES / T2 columns) fall in
  // distinct banks when P = LANES / T2 (mod LANES), LANES the lanes served at a time
  static constexpr int LANES = sizeof(T) == 4 ? 32 : 16;
  static constexpr int P = (CW + LANES - 1) / LANES * LANES + (LANES >= T2 ? LANES / T2 : 1);
  static constexpr int TW2 = rfft::tw_lds_size<L2>();                // padded w_L2 table
  static constexpr int XPH = NTEAM * SX + rfft::tw_lds_size<LX>();  // x regions, x table
  static constexpr int CREG = CW * S2;         // column regions
  static constexpr int STG = L2 * P;           // staging tile
  static constexpr int UNION = XPH > CREG ? (XPH > STG ? XPH : STG) : (CREG > STG ? CREG : STG);
  static constexpr size_t lds = size_t(TW2 + L2 + UNION) * sizeof(Cplx<T>);
  // the staging tile moves to and from HBM as rows of CW columns: thread tid takes column
  // tid % CW of the rows tid / CW + q NT / CW
  static constexpr int RSTEP = NT / CW, NQ = L2 / RSTEP;
  static_assert(LY % 8 == 0 && NPAIR % NTEAM == 0 && NTEAM >= T2 && T2 <= 32, "three-pass geometry");
  static_assert(NT % CW == 0 && L2 % RSTEP == 0 && CW * T2 <= NT, "whole staging rows per thread");
};

// Pass A: x real-to-complex of the rows y = 4 y2 + y1 of (c, z) (two rows per complex FFT,
// separated as in k1_xr2c), then per column kx the zero-padded L2-point FFT over y2 times
// w_LY^{y1 k2}, stored in slab row y1 L2 + k2.
template <typename T, int LX, int LY>
__global__ void __launch_bounds__((XYPass<T, LX, LY>::NT)) ka_xy_fwd(SlabGeom g, CompPtrs in, Cplx<T>* H,
                                                                    const Cplx<T>* twx, const Cplx<T>* twy) {
  using F = XYPass<T, LX, LY>;
  constexpr int EX = F::EX, TX = F::TX, L2 = F::L2, E2 = F::E2, T2 = F::T2, PPT = F::PPT, P = F::P;
  constexpr int CW = F::CW, NT = F::NT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* const tw2 = reinterpret_cast<Cplx<T>*>(smem_raw);  // w_L2^m = w_LY^{4m}, padded
  Cplx<T>* const twr = tw2 + F::TW2;                           // w_LY^{y1 k2}
  Cplx<T>* const U = twr + L2;
  const int tid = threadIdx.x;
  const int y1 = int(blockIdx.x & 3);
  const int cz = int(blockIdx.x >> 2);
  const int c = cz / int(g.nz), z = cz % int(g.nz);
  const int team = tid / TX, t = tid % TX;
  for (int i = tid; i < L2; i += NT) {
    tw2[rfft::tw_slot(i)] = twy[4 * i];  // padded (w_L2^m = w_LY^{4m})
    twr[i] = twy[(y1 * i) % LY];
  }
  Cplx<T>* const twxl = U + F::NTEAM * F::SX;
  rfft::load_tw_lds<T, LX>(twxl, twx, tid, NT);
  const T* base = static_cast<const T*>(in.get(c)) + int64_t(z) * in.sz;
  Cplx<T> v[PPT][EX];
  static_for<0, PPT>([&](auto p_) {
    constexpr int p = decltype(p_)::value;
    const int y2 = 2 * (team * PPT + p);
    const T* ra = base + int64_t(4 * y2 + y1) * in.sy + int64_t(t) * in.sx;
    const T* rb = ra + 4 * in.sy;
    static_for<0, EX>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      if constexpr (e < EX / 2) {
        v[p][e] = Cplx<T>{ra[int64_t(TX * e) * in.sx], rb[int64_t(TX * e) * in.sx]};
      } else {
        v[p][e] = Cplx<T>{T(0), T(0)};
      }
    });
  });
  __syncthreads();  // tables complete
  Cplx<T>* const xline = U + team * F::SX;
  // half spectra kx = TX e + t (e <= EX / 2; e = EX / 2 is kx = nx, lane 0 only)
  Cplx<T> A[PPT][EX / 2 + 1], B[PPT][EX / 2 + 1];
  const int mirror_lane = (TX - t) % TX;
  static_for<0, PPT>([&](auto p_) {
    constexpr int p = decltype(p_)::value;
    rfft::team_fft<T, LX, false, true, true>(v[p], xline, twxl, t);
    static_for<0, EX / 2 + 1>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      // Z[LX - k], k = TX e + t: lane TX - t, element EX - 1 - e (t > 0); lane 0: EX - e
      const Cplx<T> zk = v[p][e];
      Cplx<T> zm;
      zm.re = __shfl(v[p][EX - 1 - e].re, mirror_lane, TX);
      zm.im = __shfl(v[p][EX - 1 - e].im, mirror_lane, TX);
      if (t == 0) zm = v[p][(EX - e) % EX];
      A[p][e] = Cplx<T>{T(0.5) * (zk.re + zm.re), T(0.5) * (zk.im - zm.im)};
      B[p][e] = Cplx<T>{T(0.5) * (zk.im + zm.im), T(0.5) * (zm.re - zk.re)};
    });
  });
  __syncthreads();  // x regions free: the chunk phase reuses the area
  const int col = tid / T2, t2 = tid % T2;
  const bool col_role = tid < CW * T2;
  Cplx<T>* const creg = U + col * F::S2;
  // staging rows to HBM: column sc of rows sr + q RSTEP
  const int sc = tid % CW, sr = tid / CW;
  static_for<0, F::NCH>([&](auto ch_) {
    constexpr int ch = decltype(ch_)::value;
    constexpr bool last = ch == F::NCH - 1;  // kx = nx alone
    if constexpr (last) {
      if (t == 0) {
        static_for<0, PPT>([&](auto p_) {
          constexpr int p = decltype(p_)::value;
          const int y2 = 2 * (team * PPT + p);
          U[y2 * P] = A[p][EX / 2];
          U[(y2 + 1) * P] = B[p][EX / 2];
        });
      }
    } else {
      static_for<0, F::KC>([&](auto k_) {
        constexpr int kk = decltype(k_)::value;
        static_for<0, PPT>([&](auto p_) {
          constexpr int p = decltype(p_)::value;
          const int y2 = 2 * (team * PPT + p);
          U[y2 * P + kk * TX + t] = A[p][ch * F::KC + kk];
          U[(y2 + 1) * P + kk * TX + t] = B[p][ch * F::KC + kk];
        });
      });
    }
    __syncthreads();
    const bool live = col_role && (!last || col == 0);
    Cplx<T> w[E2];
    if (live) {
      static_for<0, E2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        if constexpr (e < E2 / 2) w[e] = U[(t2 + T2 * e) * P + col];
        else w[e] = Cplx<T>{T(0), T(0)};
      });
    }
    __syncthreads();
    if (live) {
      rfft::team_fft<T, L2, false, true, true>(w, creg, tw2, t2);
      static_for<0, E2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        w[e] = cmul(w[e], twr[t2 + T2 * e]);
      });
    }
    __syncthreads();
    if (live) {
      static_for<0, E2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        U[(t2 + T2 * e) * P + col] = w[e];
      });
    }
    __syncthreads();
    if (!last || sc == 0) {
      static_for<0, F::NQ>([&](auto q_) {
        constexpr int q = decltype(q_)::value;
        store_stream(H + g.ti(c, z, y1 * L2 + sr + q * F::RSTEP, CW * ch + sc), U[(sr + q * F::RSTEP) * P + sc]);
      });
    }
    __syncthreads();
  });
}

// Pass C: per column kx, w_LY^{-y1 k2} times the slab rows y1 L2 + k2, the inverse L2-point
// FFT over k2 (outputs y2 < ny / 4), then the Hermitian x half spectra of each row pair to one
// complex inverse FFT (as in k5_xc2r), rows y = 4 y2 + y1 stored (ACC: added). The next
// chunk's rows are loaded while the current one is transformed.
template <typename T, int LX, int LY, bool ACC>
__global__ void __launch_bounds__((XYPass<T, LX, LY>::NT)) kc_yx_inv(SlabGeom g, const Cplx<T>* H, CompPtrsW out,
                                                                    const Cplx<T>* twx, const Cplx<T>* twy) {
  using F = XYPass<T, LX, LY>;
  constexpr int EX = F::EX, TX = F::TX, L2 = F::L2, E2 = F::E2, T2 = F::T2, PPT = F::PPT, P = F::P;
  constexpr int CW = F::CW, NT = F::NT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* const tw2 = reinterpret_cast<Cplx<T>*>(smem_raw);
  Cplx<T>* const twr = tw2 + F::TW2;
  Cplx<T>* const U = twr + L2;
  const int tid = threadIdx.x;
  const int y1 = int(blockIdx.x & 3);
  const int cz = int(blockIdx.x >> 2);
  const int c = cz / int(g.nz), z = cz % int(g.nz);
  const int team = tid / TX, t = tid % TX;
  for (int i = tid; i < L2; i += NT) {
    tw2[rfft::tw_slot(i)] = twy[4 * i];  // padded (w_L2^m = w_LY^{4m})
    twr[i] = twy[(y1 * i) % LY];
  }
  const int col = tid / T2, t2 = tid % T2;
  const bool col_role = tid < CW * T2;
  Cplx<T>* const creg = U + col * F::S2;
  const int mirror_lane = (TX - t) % TX;
  // the rows of a chunk: thread tid holds elements tid + NT q of the chunk's L2 x ncol block
  // (addresses formed per load: a hoisted row pointer costs the registers of the prefetch)
  // (kept as separate reals: FP64 pairs moved whole would stay in scratch memory)
  T pre_re[F::NQ] = {}, pre_im[F::NQ] = {};
  auto keep = [&](auto q_, const Cplx<T>& h) {
    pre_re[decltype(q_)::value] = h.re;
    pre_im[decltype(q_)::value] = h.im;
  };
  const int hsrc = g.ti(c, z, y1 * L2 + tid / CW, tid % CW);
  const int rowel = int(g.rs) * int(g.nz);  // elements per slab row
  auto load_chunk = [&](auto ch_) {
    constexpr int ch = decltype(ch_)::value;
    constexpr int ncol = ch == F::NCH - 1 ? 1 : CW;
    static_for<0, F::NQ>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const int i = tid + q * NT;
      if constexpr (ncol == CW && CW % kSlabTile == 0) {
        // row i / CW = tid / CW + q NT / CW, column CW ch + tid % CW
        keep(q_, H[hsrc + q * (NT / CW) * rowel + CW * ch * int(g.nz)]);
      } else if constexpr (q * NT < L2 * ncol) {
        // past the block's end its last element again
        const int k = i < L2 * ncol ? i : L2 * ncol - 1;
        keep(q_, H[g.ti(c, z, y1 * L2 + k / ncol, CW * ch + k % ncol)]);
      }
    });
  };
  load_chunk(std::integral_constant<int, 0>{});
  Cplx<T> v[PPT][EX];
  static_for<0, F::NCH>([&](auto ch_) {
    constexpr int ch = decltype(ch_)::value;
    constexpr bool last = ch == F::NCH - 1;
    constexpr int ncol = last ? 1 : CW;
    static_for<0, F::NQ>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const int i = tid + q * NT;
      if constexpr (q * NT < L2 * ncol) {
        if ((q + 1) * NT <= L2 * ncol || i < L2 * ncol) U[(i / ncol) * P + i % ncol] = Cplx<T>{pre_re[q], pre_im[q]};
      }
    });
    if constexpr (ch + 1 < F::NCH) load_chunk(std::integral_constant<int, ch + 1>{});
    __syncthreads();  // (first chunk: the tables too)
    const bool live = col_role && (!last || col == 0);
    Cplx<T> w[E2];
    if (live) {
      static_for<0, E2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        w[e] = cmulc(U[(t2 + T2 * e) * P + col], twr[t2 + T2 * e]);
      });
    }
    __syncthreads();
    if (live) rfft::team_fft<T, L2, true, false, true>(w, creg, tw2, t2);
    __syncthreads();
    if (live) {
      static_for<0, E2 / 2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        U[(t2 + T2 * e) * P + col] = w[e];
      });
    }
    __syncthreads();
    static_for<0, (last ? 1 : F::KC)>([&](auto k_) {
      constexpr int kk = decltype(k_)::value;
      constexpr int e = last ? EX / 2 : ch * F::KC + kk;  // the element of kx = TX e + t
      static_for<0, PPT>([&](auto p_) {
        constexpr int p = decltype(p_)::value;
        const int y2 = 2 * (team * PPT + p);
        Cplx<T> a = U[y2 * P + kk * TX + t], b = U[(y2 + 1) * P + kk * TX + t];
        if ((e == 0 && t == 0) || last) {  // kx = 0 and kx = nx: imaginary parts dropped
          a.im = T(0);
          b.im = T(0);
        }
        const Cplx<T> zk = {a.re - b.im, a.im + b.re};  // Z[k] = A + i B
        const Cplx<T> zm = {a.re + b.im, b.re - a.im};  // Z[LX - k] = conj(A) + i conj(B)
        if constexpr (last) {
          if (t == 0) v[p][EX / 2] = zk;
        } else {
          Cplx<T> r;
          r.re = __shfl(zm.re, mirror_lane, TX);
          r.im = __shfl(zm.im, mirror_lane, TX);
          v[p][e] = zk;
          // Z[LX - k'] of lane TX - t (k' = TX e + TX - t) is element EX - 1 - e of lane t;
          // lane 0 keeps its own mirror, element EX - e
          if (t != 0) v[p][EX - 1 - e] = r;
          if constexpr (e > 0) {
            if (t == 0) v[p][EX - e] = zm;
          }
        }
      });
    });
    __syncthreads();
  });
  Cplx<T>* const twxl = U + F::NTEAM * F::SX;
  rfft::load_tw_lds<T, LX>(twxl, twx, tid, NT);
  __syncthreads();
  Cplx<T>* const xline = U + team * F::SX;
  T* const base = static_cast<T*>(out.get(c)) + int64_t(z) * out.sz;
  static_for<0, PPT>([&](auto p_) {
    constexpr int p = decltype(p_)::value;
    rfft::team_fft<T, LX, true, false, true>(v[p], xline, twxl, t);
    const int y2 = 2 * (team * PPT + p);
    T* const ra = base + int64_t(4 * y2 + y1) * out.sy + int64_t(t) * out.sx;
    T* const rb = ra + 4 * out.sy;
    static_for<0, EX / 2>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      const int64_t x = int64_t(TX * e) * out.sx;
      if constexpr (ACC) {
        ra[x] += v[p][e].re;
        rb[x] += v[p][e].im;
      } else {
        __builtin_nontemporal_store(v[p][e].re, ra + x);
        __builtin_nontemporal_store(v[p][e].im, rb + x);
      }
    });
  });
}

// fn(integral_constant<LX>, integral_constant<LY>) for the lengths of precision T.
template <typename T, int LX, typename Fn>
int with_xy_y(int64_t LY, Fn&& fn) {
#define X(n) \
  if (LY == n) return fn(std::integral_constant<int, LX>{}, std::integral_constant<int, n>{});
  SOPHT_XY_LENGTHS_F64(X)
  if constexpr (sizeof(T) == 4) {
    X(512)
  }
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}
template <typename T, typename Fn>
int with_xy(int64_t LX, int64_t LY, Fn&& fn) {
#define X(n) if (LX == n) return with_xy_y<T, n>(LY, fn);
  SOPHT_XY_LENGTHS_F64(X)
  if constexpr (sizeof(T) == 4) {
    X(512)
  }
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace sopht
