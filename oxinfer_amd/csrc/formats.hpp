// The weight formats as the device code tells them apart.
#pragma once

namespace oxhip {

enum Fmt : int { FMT_Q4 = 0, FMT_Q8_0 = 1, FMT_Q4_K = 2, FMT_Q6_K = 3, FMT_FP8 = 4, FMT_BF16 = 5, FMT_Q4M = 6, FMT_Q8F = 7, FMT_Q40 = 8, FMT_Q5_K = 9, FMT_MXFP4 = 10, FMT_NVFP4 = 11 };

}  // namespace oxhip
