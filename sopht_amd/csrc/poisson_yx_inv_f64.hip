// Pass C of the three-pass Poisson schedule in FP64 for every pair of x and y lengths.
#include "poisson_xy.h"

namespace sopht {

int poisson_yx_inv(int64_t LX, int64_t LY, SlabGeom g, const Cplx<double>* H, CompPtrsW out, const Cplx<double>* twx,
                   const Cplx<double>* twy, hipStream_t s) {
  const unsigned blocks = unsigned(int64_t(g.ncomp) * g.nz * 4);
  return with_xy<double>(LX, LY, [&](auto lx, auto ly) -> int {
    constexpr int NX = decltype(lx)::value, NY = decltype(ly)::value;
    using F = XYPass<double, NX, NY>;
    static const int lds_ok = allow_lds(kc_yx_inv<double, NX, NY, false>, F::lds);
    if (lds_ok) return lds_ok;
    kc_yx_inv<double, NX, NY, false><<<blocks, F::NT, F::lds, s>>>(g, H, out, twx, twy);
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

}  // namespace sopht
