// The wave-split-K GEMM (gemm_ks.hip) as the entry points of gemm.hip call it.
#pragma once

#include "common.hpp"

namespace umic {

// Compute units of the current device (0: no device).
int64_t device_cus();

// Up to kKsMaxSegs linears over one x (P5: one, its gate weight in w0 and up
// weight in w1).  Leading dims in elements.
constexpr int kKsMaxSegs = 3;
struct KsSeg {
  const uint16_t* w0;
  const uint16_t* w1;    // P5 only
  const uint16_t* bias;  // or NULL
  uint16_t* out;
  int64_t N, ldw0, ldw1, ldo;
};
struct KsCall {
  const uint16_t* x;
  const uint16_t* resid;  // out = bf16(resid + bf16(result)), or NULL
  int64_t M, K, ldx, ldr;
  KsSeg seg[kKsMaxSegs];
  int count;
  int act;
};

// The tile a call takes: rows of x, weight rows (P5: gate and up together) and
// waves of a workgroup.
struct TileShape {
  int rows, cols, waves;
};

// Its expected time in nanoseconds for rows x K against N weight rows in all
// (P5: N gate rows and as many up rows) on a chip of cus CUs, or -1 for a shape it
// does not take (K must be a multiple of 64).  For comparison with the other
// kernels.
double ks_time_ns(bool p5, int64_t M, int64_t N, int64_t K, int64_t cus,
                  TileShape* tile = nullptr);

// Launches it (one set of linears, or P5) for arguments that have passed the
// entry point's checks and whose K is a multiple of 64.
int launch_ks(bool p5, const KsCall& c, hipStream_t st);

}  // namespace umic
