// Kernel tables of the GN write and read stages for one nonlinearity
// (compile time: the chain then carries no branch per element).
#pragma once

#include "ts_gn_kernels.h"

namespace {

using ts::GnKernel;
using ts::GnReadKernel;

template <int ACT, typename E, bool FWD, int D>
GnKernel gn_pick_m(int m) {
#define TS_GN(MB) \
  return FWD ? (GnKernel)ts::gn_write_fwd_kernel<ACT, E, D, MB> : (GnKernel)ts::gn_write_bwd_kernel<ACT, E, D, MB>;
  switch (m) {
    case 16: TS_GN(1)
    case 32: TS_GN(2)
    case 48: TS_GN(3)
    case 64: TS_GN(4)
    case 80: TS_GN(5)
    case 96: TS_GN(6)
    case 112: TS_GN(7)
    case 128: TS_GN(8)
    case 192: TS_GN(12)
    case 256: TS_GN(16)
  }
#undef TS_GN
  return nullptr;
}

template <int ACT, typename E, bool FWD>
GnKernel gn_pick(int d, int m) {
  switch (d) {
    case 16: return gn_pick_m<ACT, E, FWD, 16>(m);
    case 32: return gn_pick_m<ACT, E, FWD, 32>(m);
    case 64: return gn_pick_m<ACT, E, FWD, 64>(m);
    case 128: return gn_pick_m<ACT, E, FWD, 128>(m);
  }
  return nullptr;
}

template <int ACT, int D>
GnKernel gn_wide_pick_d(int m, bool fwd) {
  switch (m) {
    case 192: return fwd ? (GnKernel)ts::gn_write_fwd_wide_kernel<ACT, D, 12> : (GnKernel)ts::gn_write_bwd_wide_kernel<ACT, D, 12>;
    case 384: return fwd ? (GnKernel)ts::gn_write_fwd_wide_kernel<ACT, D, 24> : (GnKernel)ts::gn_write_bwd_wide_kernel<ACT, D, 24>;
  }
  return nullptr;
}
template <int ACT, typename E, bool FWD, int D>
GnReadKernel gn_read_pick_m(int m) {
#define TS_GNR(MB) \
  return FWD ? (GnReadKernel)ts::gn_read_fwd_kernel<ACT, E, D, MB> : (GnReadKernel)ts::gn_read_bwd_kernel<ACT, E, D, MB>;
  switch (m) {
    case 16: TS_GNR(1)
    case 32: TS_GNR(2)
    case 48: TS_GNR(3)
    case 64: TS_GNR(4)
    case 80: TS_GNR(5)
    case 96: TS_GNR(6)
    case 112: TS_GNR(7)
    case 128: TS_GNR(8)
    case 192: TS_GNR(12)
    case 256: TS_GNR(16)
  }
#undef TS_GNR
  return nullptr;
}

template <int ACT, typename E, bool FWD>
GnReadKernel gn_read_pick(int d, int m) {
  switch (d) {
    case 16: return gn_read_pick_m<ACT, E, FWD, 16>(m);
    case 32: return gn_read_pick_m<ACT, E, FWD, 32>(m);
    case 64: return gn_read_pick_m<ACT, E, FWD, 64>(m);
    case 128: return gn_read_pick_m<ACT, E, FWD, 128>(m);
  }
  return nullptr;
}

template <int ACT, int D>
GnReadKernel gn_read_wide_pick_d(int m, bool fwd) {
  switch (m) {
    case 192: return fwd ? (GnReadKernel)ts::gn_read_fwd_wide_kernel<ACT, D, 12> : (GnReadKernel)ts::gn_read_bwd_wide_kernel<ACT, D, 12>;
    case 384: return fwd ? (GnReadKernel)ts::gn_read_fwd_wide_kernel<ACT, D, 24> : (GnReadKernel)ts::gn_read_bwd_wide_kernel<ACT, D, 24>;
  }
  return nullptr;
}

template <int ACT>
GnKernel gn_kernel(bool bf16, bool wide, bool fwd, int d, int m) {
  if (wide) return d == 32 ? gn_wide_pick_d<ACT, 32>(m, fwd) : gn_wide_pick_d<ACT, 64>(m, fwd);
  if (bf16) return fwd ? gn_pick<ACT, ts::bf16, true>(d, m) : gn_pick<ACT, ts::bf16, false>(d, m);
  return fwd ? gn_pick<ACT, float, true>(d, m) : gn_pick<ACT, float, false>(d, m);
}
template <int ACT>
GnReadKernel gn_read_kernel(bool bf16, bool wide, bool fwd, int d, int m) {
  if (wide) return d == 32 ? gn_read_wide_pick_d<ACT, 32>(m, fwd) : gn_read_wide_pick_d<ACT, 64>(m, fwd);
  if (bf16) return fwd ? gn_read_pick<ACT, ts::bf16, true>(d, m) : gn_read_pick<ACT, ts::bf16, false>(d, m);
  return fwd ? gn_read_pick<ACT, float, true>(d, m) : gn_read_pick<ACT, float, false>(d, m);
}

}  // namespace
