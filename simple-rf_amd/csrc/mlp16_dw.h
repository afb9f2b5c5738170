// Weight gradients of the NeRF MLP for 16-bit operands (kernel in mlp16_dw.hip): dW = dZ X^T over all layers in one
// grouped launch, K = points, on 32x32x16 MFMAs.  mlp16.h writes the operands (store_tile16).
//
// What bounds it: every stored row is read from HBM once (10 KB a point of the main model) at 120 FLOP a
// byte, below the chip's balance, so the reads have to stream while the matrix cores and the LDS work behind
// them.  A block of eight waves holds all of a layer's gradient (256 x 256 FP32 in registers, and the
// layer's other inputs or outputs: the skip's encoding, the sigma row, the view layer's extras), so that no
// row is read twice, and reduces a range of points.  Units of 32 points (one 1 KB fragment per 16-row
// tile) go through a ring of as many slots as the job's fragments leave room for; a wave reads the
// operands of a k-step of 16 points while the MFMAs of the previous one run.
//   786,432 points of the main model: 1,598 us by the 16x16x32 kernel it replaces (14 jobs, 8.9 GB: the skip's,
// the sigma row's and the view layer's operands read again; operands read after each unit's barrier, before
// its MFMAs), 1,461 us here: 7.9 GB at 5.4 TB/s, where a 2 GiB copy moves 4.9 TB/s.
//   A block's running FP32 sums end before its range does: after jb.segment points they are added to the gradients
// or, where a wave holds one or two tiles, set aside in registers (mlp.hip, weight_grads16).
#pragma once

#include "mlp_impl.h"

namespace srf {
namespace mlp {

constexpr int kDw16Jobs = 12;
constexpr int kDw16Lds = 160;       // KB of the ring
constexpr int kDw16MaxSlots = 8;

// Kinds of job: 32-row tiles x 32-column tiles a wave holds.  Wave w takes rows wr = w / 2 and columns
// wc = w % 2 as listed; kBias: the row sums of dZ go to db.
enum {
  kDwFull,    // 256 x 256: row tiles 2 wr, 2 wr + 1, column tiles 4 wc .. 4 wc + 3
  kDwWide,    // 256 x (256 + up to 64): as above, and column tile 8 + wc (array x2)
  kDwTall,    // 257 x 256: as kDwFull, and row 256 (16-row tile 16) x column tile 4 wc + wr
  kDwHalf,    // 128 x (256 + up to 96): row tile wr, column tiles 4 wc .. + 3, and 8 + wc, 10 + wc (x2)
  kDwNarrow,  // 256 x up to 64: row tiles 2 wr, 2 wr + 1, column tile wc
  kDwRow      // up to 16 x up to 256: row tile 0, column tile w
};

struct Dw16Job {
  const uint8_t* dz;   // 16-row tiles of dZ, n_dz of them
  const uint8_t* x;    // of the inputs, n_x
  const uint8_t* x2;   // of the extra inputs, n_x2 (columns 256 ..)
  int kind, n_dz, n_x, n_x2;
  int M, N, N2;        // valid rows, columns of x and of x2
  float* dw;           // gradient of the columns of x (first element), of x2, of row 256; row stride
  float* dw2;
  float* dw_row;
  int ld;
  float* db;
  float* db_row;
  int chunk;           // points per block, a multiple of 64
  int segment;         // points after which the block adds its sums to the gradients and begins anew (of 64)
  int first_block;
};

struct Dw16Args {
  Dw16Job jobs[kDw16Jobs];
  int n_jobs, ldP, cols;
};
int dw16_launch(const Dw16Args& a, int blocks, hipStream_t s);

}  // namespace mlp
}  // namespace srf
