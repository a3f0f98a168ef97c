// Scan backward kernels for bf16 I/O.
#include "ltv_scan_launch.hpp"

namespace ltv {
int scan_bwd_launch_bf16(const BwdArgs& a, ScanCfg c, int grid, bool vec, int gm, bool lb, int rm,
                        hipStream_t st) {
  return scan_bwd_launch_t<bf16_t>(a, c, grid, vec, gm, lb, rm, st);
}
int scan_bwd_chain_launch_bf16(const BwdArgs& a, ScanCfg c, int grid, int gm, int rm,
                              hipStream_t st) {
  return scan_bwd_chain_launch_t<bf16_t>(a, c, grid, gm, rm, st);
}
}  // namespace ltv
