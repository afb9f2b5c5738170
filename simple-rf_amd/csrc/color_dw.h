// Weight gradients of the TensoRF colour network (kernel in color_dw.hip): dW = dZ X^T and db = row sums of
// dZ of its four products (W1, W2, W3, basis) over the FP32 tile blocks that the forward and backward store,
// in FP32 (16x16x4 MFMAs) or split BF16 (32x32x16 MFMAs, dZ_hi X_hi + dZ_hi X_lo + dZ_lo X_hi).
//
// What bounds it: per 16 points the FP32 products of the 300^2 network take about 5,600 cycles of a compute
// unit's matrix cores and its rows (55 KB) the same at the HBM's share of one, so both have to run all the
// time.  One block of eight waves is resident per compute unit and reduces one product over a range of
// points; its fragments (16 rows x 16 points, 1 KB) go through a ring of 32-point slots of the product's
// own size, and a wave reads the operands of 16 points while the MFMAs of the previous 16 run.  The ranges
// are cut in the kernel, from the device-side count, so that every block costs about the same and one round
// of the compute units does it (two rounds measure the same).  1.4M rows of the 144-component network in
// FP32: 1.25 ms (2.15 ms by equal chunks of the MLP's FP32 kernel, which read a unit's operands after its
// barrier and kept two waves of eight busy on the basis and one on W3); 300,000 rows of the 72-component
// one, split: 0.21 ms or 4.7 TB/s (0.46 ms in chunks of 3,840, whose second round was nearly empty).
#pragma once

#include "common.h"

namespace srf {
namespace color {

constexpr int kCdwMaxA = 8, kCdwMaxB = 16;  // 16-row tiles: dZ <= 128 rows, X <= 256 rows

struct CdwJob {
  const uint8_t* dz;
  const uint8_t* x;
  int nA, nB;  // 16-row tiles of dZ and X (the tiles of their arrays)
  int M, N;    // valid rows and columns of dW
  float* dw;
  int ld_dw;
  float* db;   // nullable
};

struct CdwArgs {
  CdwJob jobs[4];
  int n_jobs, cols;
  int chunk;               // points of a block, a multiple of 32; 0: equal costs
  int cus;                 // compute units (more than n_jobs)
  // optional device-side point count: only the columns below it, rounded up to whole 256-point blocks, are
  // reduced; the columns up to that bound must hold finite values with dZ = 0 beyond the count, as the
  // forward and backward kernels leave them
  const int32_t* cols_dev;
};

int cdw_launch(const CdwArgs& a, bool split, hipStream_t s);

}  // namespace color
}  // namespace srf
