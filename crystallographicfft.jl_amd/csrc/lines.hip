// Launches of the line-matrix chain's kernels (lines.hpp).
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "lines.hpp"

namespace cfft {

namespace {

template <typename T, int H, int CENT>
void launch_mode(int mode, const PipeP& p, const PipeBufs& B, int step, int line, int flip, hipStream_t s) {
  const dim3 grid((unsigned)(p.batch * H * line_tiles(H))), block(64 * LineCent<CENT>::NCH);
  switch (mode) {
    case kLinesOut:
      hipLaunchKernelGGL((k_lines<T, H, CENT, kLinesOut>), grid, block, 0, s, p, B, step, line, flip);
      break;
    case kLinesIn:
      hipLaunchKernelGGL((k_lines<T, H, CENT, kLinesIn>), grid, block, 0, s, p, B, step, line, flip);
      break;
    case kLinesIn | kLinesOut:
      hipLaunchKernelGGL((k_lines<T, H, CENT, kLinesIn | kLinesOut>), grid, block, 0, s, p, B, step, line, flip);
      break;
    case kLinesIn | kLinesOut | kLinesStore:
      hipLaunchKernelGGL((k_lines<T, H, CENT, kLinesIn | kLinesOut | kLinesStore>), grid, block, 0, s, p, B, step, line,
                         flip);
      break;
    default: throw Error{CFFT_ERR_INVALID, "unknown line-chain mode"};
  }
  hip_check(hipGetLastError(), "k_lines");
}

template <typename T, int H>
void launch_cent(int cent, int mode, const PipeP& p, const PipeBufs& B, int step, int line, int flip, hipStream_t s) {
  switch (cent) {
    case CENT_P: launch_mode<T, H, CENT_P>(mode, p, B, step, line, flip, s); break;
    case CENT_I: launch_mode<T, H, CENT_I>(mode, p, B, step, line, flip, s); break;
    case CENT_C: launch_mode<T, H, CENT_C>(mode, p, B, step, line, flip, s); break;
    case CENT_A: launch_mode<T, H, CENT_A>(mode, p, B, step, line, flip, s); break;
    case CENT_F: launch_mode<T, H, CENT_F>(mode, p, B, step, line, flip, s); break;
    default: throw Error{CFFT_ERR_UNSUPPORTED, "no line-chain kernel for this centring"};
  }
}

template <typename T>
void launch_len(int H, int cent, int mode, const PipeP& p, const PipeBufs& B, int step, int line, int flip,
                hipStream_t s) {
  switch (H) {
    case 8: launch_cent<T, 8>(cent, mode, p, B, step, line, flip, s); break;
    case 12: launch_cent<T, 12>(cent, mode, p, B, step, line, flip, s); break;
    case 16: launch_cent<T, 16>(cent, mode, p, B, step, line, flip, s); break;
    case 24: launch_cent<T, 24>(cent, mode, p, B, step, line, flip, s); break;
    case 32: launch_cent<T, 32>(cent, mode, p, B, step, line, flip, s); break;
    case 48: launch_cent<T, 48>(cent, mode, p, B, step, line, flip, s); break;
    case 64: launch_cent<T, 64>(cent, mode, p, B, step, line, flip, s); break;
    default: throw Error{CFFT_ERR_UNSUPPORTED, "no line-chain kernel for this length"};
  }
}

}  // namespace

void launch_lines(int prec, int H, int cent, int mode, const PipeP& p, const PipeBufs& B, int step, int line, int flip,
                  hipStream_t s) {
  if (prec == CFFT_FP64) launch_len<double>(H, cent, mode, p, B, step, line, flip, s);
  else launch_len<float>(H, cent, mode, p, B, step, line, flip, s);
}

}  // namespace cfft
