// The mid-size tiled GEMM (gemm_mid.hip) as the entry points of gemm.hip call
// it: one linear or P5 (gate weight w0, up weight w1).
#pragma once

#include "gemm_ks.hpp"

namespace umic {

// Its expected time in nanoseconds on a chip of cus CUs (P5: N gate rows and as
// many up rows), or -1 for a shape it does not take (K must be a multiple of 64).
double mid_time_ns(bool p5, int64_t M, int64_t N, int64_t K, int act, int64_t cus,
                   TileShape* tile = nullptr);

// Launches it on a call of one segment and no residual, for arguments that
// have passed the entry point's checks and whose K is a multiple of 64.
int launch_mid(bool p5, const KsCall& c, hipStream_t st);

}  // namespace umic
