// In-order fp16 implicit-GEMM instantiations.
#include "igemm_fp.h"

namespace dw {

bool igemm_launch_fp_f16(hipStream_t st, const IgemmArgs& a, const TileCfg& t) {
  switch (t.bc) {
    case 16: return ig::launch_fp<1>(st, a), true;
    case 32: return ig::launch_fp<2>(st, a), true;
    case 64: return ig::launch_fp<4>(st, a), true;
  }
  return false;
}

}  // namespace dw
