// Pass C of the three-pass Poisson schedule in FP32 that adds to the fields (the adjoint's solve).
#include "poisson_xy.h"

namespace sopht {

int poisson_yx_inv_add(int64_t LX, int64_t LY, SlabGeom g, const Cplx<float>* H, CompPtrsW out,
                       const Cplx<float>* twx, const Cplx<float>* twy, hipStream_t s) {
  const unsigned blocks = unsigned(int64_t(g.ncomp) * g.nz * 4);
  return with_xy<float>(LX, LY, [&](auto lx, auto ly) -> int {
    constexpr int NX = decltype(lx)::value, NY = decltype(ly)::value;
    using F = XYPass<float, NX, NY>;
    static const int lds_ok = allow_lds(kc_yx_inv<float, NX, NY, true>, F::lds);
    if (lds_ok) return lds_ok;
    kc_yx_inv<float, NX, NY, true><<<blocks, F::NT, F::lds, s>>>(g, H, out, twx, twy);
    SOPHT_CHECK_LAUNCH();
    return SOPHT_OK;
  });
}

}  // namespace sopht
