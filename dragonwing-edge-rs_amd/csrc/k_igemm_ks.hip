// Split-K int8 implicit-GEMM instantiations.
#include "igemm_ks.h"

namespace dw {

bool igemm_launch_ks_i8(hipStream_t st, const IgemmArgs& a, const TileCfg& t) {
#define DW_KS(BC, NW) \
  if (t.bc == BC && t.pb == NW) return ig::launch_ks<BC / 16, NW>(st, a), true;
  DW_KS(16, 4) DW_KS(16, 8) DW_KS(16, 16) DW_KS(32, 4) DW_KS(32, 8) DW_KS(32, 16)
#undef DW_KS
  return false;
}

}  // namespace dw
