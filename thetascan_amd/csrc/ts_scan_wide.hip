// The one-view scan with keys of more than 128 features (bf16): the key widths
// 192, 256 and 384 of the wide feature maps and the Gauss-Newton memories.
// One workgroup holds the [DK][64] fp32 state of its 64 value columns in the
// accumulators of four waves, so every key block's scores add up in one MFMA
// chain and a wide scan is one summary, one prefix and one main launch.  Cut
// into 128-wide key blocks it took three launches per block, with the partial
// outputs added up in fp32 through memory.
//
// Bound: HBM for the main pass, then LDS bandwidth: a wave of a 384-wide tile
// reads about 125 KB of K and state fragments for about 126 MFMAs.  Whole
// calls (summary, prefix and main pass) against the 128-wide blocks:
//   B8 H8 T4096, 384 x 64 (0.70 GB): plain 202 and 282 us, with the mass
//   column 234 and 592, with a static retention and the mass 266 and 594;
//   B4 H8 T3001, 192 x 192: 89 and 194 us, with both 110 and 333.
// K [64][392], V [64][72] and one state copy [64][392] take 113 KB, so one
// workgroup per CU is resident (192 and 256 wide: two), and the next tile's
// rows are fetched into registers while a tile is computed.

#include "ts_scan_kernel.h"

namespace {

typedef void (*KernelFn)(ts::ScanP);

template <int DK>
KernelFn pick(bool main_kernel, int mode) {
  using namespace ts;
  switch (mode) {
#define TS_MODE(M)                                                        \
  case M:                                                                 \
    return main_kernel ? (KernelFn)ts::scan_kernel<bf16, DK, 1, true, M>  \
                       : (KernelFn)ts::scan_kernel<bf16, DK, 1, false, M>;
    TS_MODE(kPlain)
    TS_MODE(kKeyExt)
    TS_MODE(kValExt)
    TS_MODE(kStatic)
    TS_MODE(kStatic | kValExt)
    TS_MODE(kF32Out)
    TS_MODE(kF32Out | kKeyExt)
    TS_MODE(kF32Out | kStatic)
    TS_MODE(kF32Out | kStatic | kKeyExt)
#undef TS_MODE
  }
  return main_kernel ? (KernelFn)scan_kernel<bf16, DK, 1, true, kGeneral>
                     : (KernelFn)scan_kernel<bf16, DK, 1, false, kGeneral>;
}

}  // namespace

ts::ScanFn ts::pick_wide_scan(int dkp, bool main_kernel, int mode) {
  switch (dkp) {
    case 192: return pick<192>(main_kernel, mode);
    case 256: return pick<256>(main_kernel, mode);
    case 384: return pick<384>(main_kernel, mode);
  }
  return nullptr;
}
