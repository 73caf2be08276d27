// The z pass of the three-pass Poisson schedule.
#include "poisson_z.h"

namespace sopht {
namespace {

using rfft::wave_sync;

// Build-time choices of the three-pass z pass (measured: ordinary stores beat streaming ones
// there, quarter-line tiles beat half-line ones, six jobs per workgroup beat two or three).
#ifndef SOPHT_ZROW_STREAM
#define SOPHT_ZROW_STREAM 0
#endif
#ifndef SOPHT_ZROW_PARTS
#define SOPHT_ZROW_PARTS 4
#endif
#ifndef SOPHT_ZROW_SLOTS
#define SOPHT_ZROW_SLOTS 2
#endif
#ifndef SOPHT_ZROW_PREFETCH
#define SOPHT_ZROW_PREFETCH 1
#endif
constexpr bool kZrowStream = SOPHT_ZROW_STREAM;
constexpr bool kZrowPrefetch = SOPHT_ZROW_PREFETCH;

// The z pass of the three-pass schedule. A workgroup owns one kx tile (WC columns) of the row
// class k2 (slab rows y1 L2 + k2, y1 < 4) and of its mirror class L2 - k2. Per job (component,
// class) the four rows are loaded, the 4-point DFT over y1 gives the pencils ky = k2 + L2 k1,
// each pencil is convolved along z as in k3_zconv, and the inverse 4-point DFT returns the rows.
// The workgroup has two teams per column and transforms two pencils at a time (two LDS tiles),
// so a thread holds E / 4 values of each row: the next job's rows are loaded during the
// transforms within 128 VGPRs. The G^ lines of the class, |k2 + L2 k1| folded to <= ny for
// k1 < 4, are staged in LDS once per workgroup. Slot s of a column takes pencil k1 = s + 2r in
// round r of a job, and so G^ line s + 2r; in a mirror job it takes pencil 3 - s - 2r, whose
// ky' = L2 - k2 + L2 (3 - s - 2r) has the line of 2 ny - ky' = k2 + L2 (s + 2r): the same.
template <typename T, int L>
struct ZRowTile {
  static constexpr int E = LinePlan<L>::E, TT = LinePlan<L>::T;
  // a quarter of a 128-byte line per workgroup (two workgroups per CU); the four quarters of a
  // line go to workgroups b, b + 8, b + 16, b + 24 (the same XCD), so three come from its L2
  static constexpr int PARTS = sizeof(T) == 4 ? SOPHT_ZROW_PARTS : SOPHT_ZROW_PARTS / 2;  // (FP64: a half)
  static constexpr int SLOTS = SOPHT_ZROW_SLOTS;  // pencils per column transformed at once
  static constexpr int WC = kLineCplx<T> / PARTS;
  static constexpr int NT = SLOTS * WC * TT;
  // tiles [slot][column]: the load role's lanes (column, z) hit distinct banks when the column
  // stride is 8 (mod 32) slots, or 4 (mod 16) of the 16-byte FP64 ones, which are served 16 lanes
  // at a time; FP32 teams of 16 need 16 for their exchanges, shorter ones 9 as elsewhere. (Conflict
  // cycles of the whole pass, by the counters: 26% of its LDS cycles in FP32, 37% at L = 128 and 43% at
  // L = 384 in FP64.)
  static constexpr int S = TT < 16 ? region_stride<L, true>()
                           : sizeof(T) == 8 ? L + 4
                           : TT < 32 ? L + 16 : (WC == 4 ? L + 8 : L + 4);
  static constexpr int KL = E / (2 * SLOTS);  // z values per row per thread (z = lr + SLOTS TT k)
  static constexpr int GL = L / 2 + 1;
  static constexpr size_t lds = size_t(SLOTS * WC * S) * sizeof(Cplx<T>) + size_t(4 * WC * GL) * sizeof(T);
  static_assert(E % (2 * SLOTS) == 0 && 4 % SLOTS == 0, "the z rows split among the slots");
};

template <typename T, int L>
__global__ void __launch_bounds__((ZRowTile<T, L>::NT)) __attribute__((amdgpu_waves_per_eu(kZconvWavesFor<T, L>))) k3_zconv4(SlabGeom g, Cplx<T>* H, const T* ghat,
                                                                  const Cplx<T>* tw, int jobs) {
  using ZT = ZRowTile<T, L>;
  constexpr int E = ZT::E, TT = ZT::TT, WC = ZT::WC, S = ZT::S, KL = ZT::KL, GL = ZT::GL;
  constexpr int SL = ZT::SLOTS, ZSTEP = SL * TT;
  extern __shared__ unsigned char smem_raw[];
  Cplx<T>* xb = reinterpret_cast<Cplx<T>*>(smem_raw);  // tiles [slot][column][z]
  T* const gl = reinterpret_cast<T*>(xb + SL * WC * S);  // G^ lines [k1][column][kz]
  const int tid = threadIdx.x;
  const int lw = tid % WC, lr = tid / WC;  // load role: column, first z
  const int team = tid / TT, t = tid % TT;  // transform role: team = slot * WC + column
  const int tcol = team % WC, slot = team / WC;
  const int64_t ncols = g.nx + 1;
  const int L2 = int(g.ny) / 2;
  int64_t k2, kx0;
  if (!col_tile_parts<ZT::PARTS>(blockIdx.x, ncols, L2 / 2 + 1, WC, k2, kx0)) return;
  const bool self = k2 == 0 || 2 * k2 == L2;
  const int alljobs = self ? g.ncomp : 2 * g.ncomp;
  const int jbeg = int(blockIdx.y) * jobs;
  if (jbeg >= alljobs) return;
  const int njobs = alljobs - jbeg < jobs ? alljobs - jbeg : jobs;
  const int64_t kx = kx0 + lw;
  const bool live = kx < ncols;
  const int first_col = 64 / TT >= WC ? 0 : ((tid / 64) * (64 / TT)) % WC;
  const bool wave_live = kx0 + first_col < ncols;
  {
    // every load in flight before the first LDS write (a loop would wait on each in turn)
    constexpr int NG = 4 * WC * GL, NIT = (NG + ZT::NT - 1) / ZT::NT;
    T gt[NIT];
    static_for<0, NIT>([&](auto i_) {
      constexpr int it = decltype(i_)::value;
      const int i = tid + it * ZT::NT;
      const int kz = i % GL, rest = i / GL;
      const int w = rest % WC, k1 = (rest / WC) & 3;
      const int ky = int(k2) + L2 * k1;
      const int kyo = ky <= int(g.ny) ? ky : 2 * int(g.ny) - ky;
      const int kxt = kx0 + w < ncols ? int(kx0) + w : 0;
      gt[it] = (it + 1 < NIT || i < NG) ? ghat[(kyo * int(ncols) + kxt) * int(g.gz) + kz] : T(0);
    });
    static_for<0, NIT>([&](auto i_) {
      constexpr int it = decltype(i_)::value;
      const int i = tid + it * ZT::NT;
      if (it + 1 < NIT || i < NG) gl[i] = gt[it];
    });
  }
  constexpr int zs = kSlabTile;  // consecutive z of a column tile (ti layout)
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
  auto row_col = [&](int jl, int y1) -> int {
    const int j = jbeg + jl;
    const int cc = j % g.ncomp;
    const int cls = j < g.ncomp ? int(k2) : L2 - int(k2);
    return g.ti(cc, 0, y1 * L2 + cls, live ? int(kx) : 0);
  };
  Cplx<T> pf[4][KL];
  auto load = [&](int j) {
    static_for<0, 4>([&](auto y_) {
      constexpr int y1 = decltype(y_)::value;
      const int colp = row_col(j, y1);
      static_for<0, KL>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        pf[y1][k] = live ? H[colp + (lr + ZSTEP * k) * zs] : Cplx<T>{T(0), T(0)};
      });
    });
  };
  Cplx<T>* const line = xb + team * S;
  if constexpr (kZrowPrefetch) load(0);
  __syncthreads();  // G^ lines staged
  for (int j = 0; j < njobs; ++j) {
    const bool mirror = jbeg + j >= g.ncomp;
    if constexpr (!kZrowPrefetch) load(j);
    Cplx<T> y[4][KL];
    static_for<0, KL>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      Cplx<T> u[4] = {pf[0][k], pf[1][k], pf[2][k], pf[3][k]};
      rfft::dft4<T, false>(u);
      static_for<0, 4>([&](auto q_) { y[decltype(q_)::value][k] = u[decltype(q_)::value]; });
    });
    if constexpr (kZrowPrefetch) {
      if (j + 1 < njobs) load(j + 1);
    }
    static_for<0, 4 / SL>([&](auto r_) {
      constexpr int r = decltype(r_)::value;
      // slot sl takes pencil sl + SL r (a mirror job: 3 - sl - SL r)
      static_for<0, SL>([&](auto s_) {
        constexpr int sl = decltype(s_)::value;
        static_for<0, KL>([&](auto k_) {
          constexpr int k = decltype(k_)::value;
          // selects on values (a select of two array elements' addresses would leave y in
          // scratch memory)
          const Cplx<T> a = y[3 - sl - SL * r][k], b = y[sl + SL * r][k];
          xb[(sl * WC + lw) * S + lr + ZSTEP * k] = Cplx<T>{mirror ? a.re : b.re, mirror ? a.im : b.im};
        });
      });
      __syncthreads();
      Cplx<T> v[E];
      static_for<0, E>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        if constexpr (e < E / 2) v[e] = line[t + TT * e];
        else v[e] = Cplx<T>{T(0), T(0)};
      });
      rfft::wave_sync();
      if (wave_live) {
        const T* const gq = gl + ((slot + SL * r) * WC + tcol) * GL;
        if constexpr (last_twiddles_hoisted<L>()) {
          constexpr int R0 = P3::r0, NS3 = R0 * R1;
          rfft::stockham_stage<T, L, R0, 1, false, true>(v, line, tw, t);
          rfft::stockham_stage_given<T, L, R1, R0, false>(v, line, w2, t);
          rfft::stockham_stage_given<T, L, R2, NS3, false>(v, line, w3, t);
        } else {
          rfft::team_fft<T, L, false, true>(v, line, tw, t);
        }
        static_for<0, E>([&](auto e_) {
          constexpr int e = decltype(e_)::value;
          const int kz = t + TT * e;
          const T gv = gq[kz <= L / 2 ? kz : L - kz];
          v[e] = Cplx<T>{v[e].re * gv, v[e].im * gv};
        });
        if constexpr (last_twiddles_hoisted<L>()) {
          constexpr int R0 = P3::r0, NS3 = R0 * R1;
          rfft::stockham_stage<T, L, R0, 1, true, false>(v, line, tw, t);
          rfft::stockham_stage_given<T, L, R1, R0, true>(v, line, w2, t);
          rfft::stockham_stage_given<T, L, R2, NS3, true>(v, line, w3, t);
        } else {
          rfft::team_fft<T, L, true>(v, line, tw, t);
        }
      }
      static_for<0, E / 2>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        line[t + TT * e] = v[e];
      });
      __syncthreads();
      static_for<0, SL>([&](auto s_) {
        constexpr int sl = decltype(s_)::value;
        static_for<0, KL>([&](auto k_) {
          constexpr int k = decltype(k_)::value;
          const Cplx<T> val = xb[(sl * WC + lw) * S + lr + ZSTEP * k];
          Cplx<T>& a = y[3 - sl - SL * r][k];
          Cplx<T>& b = y[sl + SL * r][k];
          a = Cplx<T>{mirror ? val.re : a.re, mirror ? val.im : a.im};
          b = Cplx<T>{mirror ? b.re : val.re, mirror ? b.im : val.im};
        });
      });
      __syncthreads();
    });
    if (live) {
      static_for<0, KL>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        Cplx<T> u[4] = {y[0][k], y[1][k], y[2][k], y[3][k]};
        rfft::dft4<T, true>(u);
        static_for<0, 4>([&](auto q_) {
          constexpr int y1 = decltype(q_)::value;
          if constexpr (kZrowStream) store_stream(H + row_col(j, y1) + (lr + ZSTEP * k) * zs, u[y1]);
          else H[row_col(j, y1) + (lr + ZSTEP * k) * zs] = u[y1];
        });
      });
    }
  }
}

template <typename T>
int z_rows(int64_t L, SlabGeom g, Cplx<T>* H, const T* ghat, const Cplx<T>* tw,
                   hipStream_t s, int jobs) {
#define X(n)                                                                          \
  if (L == n) {                                                                       \
    using ZT = ZRowTile<T, n>;                                                        \
    const int64_t nb = col_tile_parts_blocks(ZT::PARTS, g.nx + 1, g.ny / 4 + 1, ZT::WC); \
    const unsigned nch = unsigned((2 * g.ncomp + jobs - 1) / jobs);                    \
    static const int lds_ok = allow_lds(k3_zconv4<T, n>, ZT::lds);                    \
    if (lds_ok) return lds_ok;                                                        \
    k3_zconv4<T, n><<<dim3(unsigned(nb), nch), ZT::NT, ZT::lds, s>>>(g, H, ghat, tw, jobs); \
    SOPHT_CHECK_LAUNCH();                                                             \
    return SOPHT_OK;                                                                  \
  }
  SOPHT_ZROW_LENGTHS(X)
#undef X
  return SOPHT_ERR_UNSUPPORTED;
}

}  // namespace

int poisson_z_rows(int64_t LZ, SlabGeom g, Cplx<float>* H, const float* ghat, const Cplx<float>* tw, hipStream_t s,
                   int jobs) {
  return z_rows<float>(LZ, g, H, ghat, tw, s, jobs);
}
int poisson_z_rows(int64_t LZ, SlabGeom g, Cplx<double>* H, const double* ghat, const Cplx<double>* tw, hipStream_t s,
                   int jobs) {
  return z_rows<double>(LZ, g, H, ghat, tw, s, jobs);
}

}  // namespace sopht
