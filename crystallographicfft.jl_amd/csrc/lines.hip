// Launches of the line-matrix chain's kernels (lines.hpp).  Compiled once per
// precision (LINES_PREC) to keep the build parallel.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "lines.hpp"

namespace cfft {

namespace {

template <typename T, int H, int CENT>
void launch_mode(int mode, const LineP& p, const LineEnt& e, hipStream_t s) {
  const dim3 grid((unsigned)(p.batch * H * line_parts(H))), block(64 * LineCent<CENT>::NCH);
#define CFFT_LINES(MODE)                                                                                       \
  case MODE:                                                                                                   \
    hipLaunchKernelGGL((k_lines<T, H, CENT, MODE>), grid, block, 0, s, p.ch, p.mats, p.axv, p.batch, p.step, \
                       p.flags, p.E, p.f0_in, p.f0_out, e);                                                    \
    break;
  switch (mode) {
    CFFT_LINES(kLinesOut)
    CFFT_LINES(kLinesIn)
    CFFT_LINES(kLinesIn | kLinesOut)
    CFFT_LINES(kLinesIn | kLinesOut | kLinesStore)
    default: throw Error{CFFT_ERR_INVALID, "unknown line-chain mode"};
  }
#undef CFFT_LINES
  hip_check(hipGetLastError(), "k_lines");
}

template <typename T, int H>
void launch_cent(int cent, int mode, const LineP& p, const LineEnt& e, hipStream_t s) {
  switch (cent) {
    case CENT_P: launch_mode<T, H, CENT_P>(mode, p, e, s); break;
    case CENT_I: launch_mode<T, H, CENT_I>(mode, p, e, s); break;
    case CENT_C: launch_mode<T, H, CENT_C>(mode, p, e, s); break;
    case CENT_A: launch_mode<T, H, CENT_A>(mode, p, e, s); break;
    case CENT_F: launch_mode<T, H, CENT_F>(mode, p, e, s); break;
    default: throw Error{CFFT_ERR_UNSUPPORTED, "no line-chain kernel for this centring"};
  }
}

}  // namespace

template <typename T>
void launch_lines_prec(int H, int cent, int mode, const LineP& p, const LineEnt& e, hipStream_t s) {
  switch (H) {
    case 8: launch_cent<T, 8>(cent, mode, p, e, s); break;
    case 12: launch_cent<T, 12>(cent, mode, p, e, s); break;
    case 16: launch_cent<T, 16>(cent, mode, p, e, s); break;
    case 24: launch_cent<T, 24>(cent, mode, p, e, s); break;
    case 32: launch_cent<T, 32>(cent, mode, p, e, s); break;
    case 48: launch_cent<T, 48>(cent, mode, p, e, s); break;
    case 64: launch_cent<T, 64>(cent, mode, p, e, s); break;
    default: throw Error{CFFT_ERR_UNSUPPORTED, "no line-chain kernel for this length"};
  }
}

#if LINES_PREC == 64
template void launch_lines_prec<double>(int, int, int, const LineP&, const LineEnt&, hipStream_t);
void launch_lines(int prec, int H, int cent, int mode, const LineP& p, const LineEnt& e, hipStream_t s) {
  if (prec == CFFT_FP64) launch_lines_prec<double>(H, cent, mode, p, e, s);
  else launch_lines_prec<float>(H, cent, mode, p, e, s);
}
#else
template void launch_lines_prec<float>(int, int, int, const LineP&, const LineEnt&, hipStream_t);
#endif

}  // namespace cfft
