// Pass A of the three-pass Poisson schedule in FP32 for every pair of x and y lengths.
#include "poisson_xy.h"

namespace sopht {

int poisson_xy_fwd(int64_t LX, int64_t LY, SlabGeom g, CompPtrs in, Cplx<float>* H, const Cplx<float>* twx,
                   const Cplx<float>* twy, hipStream_t s) {
  const unsigned blocks = unsigned(int64_t(g.ncomp) * g.nz * 4);
  return with_xy<float>(LX, LY, [&](auto lx, auto ly) -> int {
    constexpr int NX = decltype(lx)::value, NY = decltype(ly)::value;
    using F = XYPass<float, NX, NY>;
    static const int lds_ok = allow_lds(ka_xy_fwd<float, NX, NY>, F::lds);
    if (lds_ok) return lds_ok;
    ka_xy_fwd<float, NX, NY><<<blocks, F::NT, F::lds, s>>>(g, in, H, twx, twy);
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

}  // namespace sopht
