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
// FP32: 1.28 ms (2.15 ms by equal chunks of the MLP's FP32 kernel, which read a unit's operands after its
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

// Tiles that each wave of a block multiplies, of 16 x 16 (FP32) or 32 x 32 entries (split).  At most two row
// tiles: the eight waves share the columns, column tile w + 8 k or column block w going to wave w.  More: waves
// 2 r and 2 r + 1 (FP32) or r and r + 4 (split) take row tiles 2 r, 2 r + 1 or row block r, and half of the
// columns each.  The kernel has exactly these forms, each without a branch between its products, and the costs
// below are theirs.  (With FP32 forms of 4, 5 and 8 column tiles alone, whatever the product had, but costs of
// its own, the first layer of the network without encoding, two tiles, was charged 800 cycles per 16 points and
// took 2,250, and set the launch's time.  Backward of 1.4M rows of 72 components: 3.05 ms then,
// 2.44 before there were costs, 1.77 here.)
struct CdwForm {
  int rows, cols;
};
template <bool SPLIT>
__host__ __device__ constexpr CdwForm cdw_form(int nA, int nB) {
  if (nA <= 2) return SPLIT ? CdwForm{1, 1} : CdwForm{nA, (nB + 7) / 8};
  return SPLIT ? CdwForm{1, (nB + 3) / 4} : CdwForm{2, (nB + 1) / 2};
}

// Cost of 16 points to a block, in cycles: the MFMAs of its busiest SIMD (two waves) or the reads, and the
// step itself.  The reads' share and the step's were swept (the kernel on 1.4M rows of 144 components and of 72 without
// encoding in FP32, and on 300,000 of 72 split, us): 104 / 200 1370, 993, 212; 80 / 200 1307, 895, 214; 60 / 200
// 1295, 904, 200; 60 / 50 1296, 952, 218; 40 / 100 1406, 988, 208; 60 (split 90) / 200 1280, 897, 208.
template <bool SPLIT>
__host__ __device__ constexpr int cdw_cost(int nA, int nB) {
  const CdwForm f = cdw_form<SPLIT>(nA, nB);
  const int mfma = (SPLIT ? 512 : 256) * f.rows * f.cols, reads = (SPLIT ? 90 : 60) * (nA + nB);
  return (mfma > reads ? mfma : reads) + 200;
}

int cdw_launch(const CdwArgs& a, bool split, hipStream_t s);

}  // namespace color
}  // namespace srf
