// fwd_paged_d256.hip — the fp16/bf16 forward over a paged K/V cache, kernel width 256 (workgroup
// shapes C and CF of launch_fwd_pg in fwd_kernel.hpp).
#include "fwd_kernel.hpp"

namespace fa {

int launch_fwd_paged_d256(const FableFwdParams& p, const FwdPaged& pg, int dtype, bool rot, hipStream_t st, FwdWs& ws) {
  using C = FwdCfg<256, 32, 4, 1>;
  using CF = FwdCfg<256, 32, 4, 1>;
  if (dtype == FA_F16) return launch_fwd_pg<_Float16, C, CF>(p, pg, rot, st, ws);
  return launch_fwd_pg<__bf16, C, CF>(p, pg, rot, st, ws);
}

}  // namespace fa
