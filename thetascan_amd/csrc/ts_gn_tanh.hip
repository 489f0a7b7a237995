// The GN write and read kernels with a tanh hidden layer (see ts_gn_kernels.h).

#include "ts_gn_pick.h"

ts::GnKernel ts::gn_tanh_kernel(bool bf16, bool wide, bool fwd, int d, int m) {
  return gn_kernel<TS_GN_TANH>(bf16, wide, fwd, d, m);
}
ts::GnReadKernel ts::gn_read_tanh_kernel(bool bf16, bool wide, bool fwd, int d, int m) {
  return gn_read_kernel<TS_GN_TANH>(bf16, wide, fwd, d, m);
}
