// Grouped weight-gradient kernel of the NeRF MLP for 16-bit operands (design notes in mlp16_dw.h).
#include "mlp16.h"
#include "mlp16_dw.h"

namespace srf {
namespace mlp {

template <int RM, int NC, int NX, bool ROW>
__device__ __forceinline__ void dw16_run(const Dw16Args& a, const Dw16Job& jb, int row0, int col0, int colx, bool sums,
                                         uint8_t* ring) {
  constexpr int NB = NC + NX;       // column tiles
  constexpr int NA = RM + (ROW ? 1 : 0);
  const int lane = threadIdx.x & 63, h = lane >> 5, i32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_frag = jb.n_dz + jb.n_x + jb.n_x2;
  const int slots = min(kDw16MaxSlots, kDw16Lds / n_frag);
  const int slot_bytes = n_frag * 1024;
  const int pb = (blockIdx.x - jb.first_block) * jb.chunk;
  const int units = (min(pb + jb.chunk, a.cols) - pb) / 32, seg_units = jb.segment / 32;

  // This wave's fragments of a unit: f = w, w + 8, ...  LDS position l of a fragment (16 B) takes chunk
  // k = (l >> 1) & 1 of record (l & 1, c) with c = 16 (unit % 2) + 8 s + 4 h' + d, where d = l >> 4, h' = (l >> 2)
  // & 1 and s = (l >> 3 ^ f) & 1: operand lane (h', row) of k-step s finds its row at the points c, 32 + c as
  // the dwords d (0 .. 3), 256 B apart.  (s is swapped in odd fragments so that the rows of a tile's two
  // fragments lie in different banks.)
  const int src_lane = ((lane >> 1) & 1) * 1024 +
                       ((lane & 1) * 32 + 8 * (((lane >> 3) ^ w) & 1) + 4 * ((lane >> 2) & 1) + (lane >> 4)) * 16;
  constexpr int kMaxFrags = 5;
  const int n_mine = (n_frag - w + 7) / 8;
  const uint8_t* src[kMaxFrags];
#pragma unroll
  for (int q = 0; q < kMaxFrags; ++q) {
    const int f = min(w + 8 * q, n_frag - 1);
    const uint8_t* base = f < jb.n_dz ? jb.dz : (f < jb.n_dz + jb.n_x ? jb.x : jb.x2);
    const int t = f < jb.n_dz ? f : (f < jb.n_dz + jb.n_x ? f - jb.n_dz : f - jb.n_dz - jb.n_x);
    src[q] = base + (size_t)t * 32 * a.ldP + (size_t)(pb / 64) * 2048;
  }
  const uint32_t lds0 = lds_offset(ring) + 1024u * w;
  uint32_t wr = 0;                  // byte offset of the slot to fill
  int filled = 0;
  auto fill = [&]() SRF_AI {
#pragma unroll
    for (int q = 0; q < kMaxFrags; ++q)
      if (q < n_mine) lds_dma_1k_ahead(src[q] + (filled & 1) * 256, lds0 + wr + 8192u * q, src_lane);
    if (filled & 1)
#pragma unroll
      for (int q = 0; q < kMaxFrags; ++q) src[q] += 2048;
    ++filled;
    wr = wr + slot_bytes == (uint32_t)(slots * slot_bytes) ? 0u : wr + slot_bytes;
  };
  for (int u = 0; u < slots - 1 && u < units; ++u) fill();

  // Sums of few tiles are set aside in registers, those of many added to the gradients, after jb.segment points.
  constexpr bool kAside = RM * NB <= 2;
  f32x16 acc[RM][NB], aside[kAside ? RM : 1][kAside ? NB : 1], row_acc;
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][k][r] = 0.f;
        if constexpr (kAside) aside[i][k][r] = 0.f;
      }
#pragma unroll
  for (int r = 0; r < 16; ++r) row_acc[r] = 0.f;
  float rs[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) rs[i] = 0.f;

  // byte offset in a slot of the lane's row in 32-row tile 0 at k-step 0 (k-step 1: ^ 128)
  const uint32_t at_lane = (i32 >> 4) * 1024 + (((i32 >> 4) & 1) * 32 + h * 16 + (i32 & 15)) * 4;
  const int odd_x = jb.n_dz & 1;    // x's fragments start at an odd one: the swap is the other way round
  const uint32_t ta = row0 * 2048, tx = jb.n_dz * 1024;
  auto operand = [&](uint32_t at) SRF_AI {
    const uint32_t* v = reinterpret_cast<const uint32_t*>(ring + at);
    return u32x4{v[0], v[64], v[128], v[192]};
  };
  auto load = [&](uint32_t slot, int s, u32x4 (&av)[NA], u32x4 (&bv)[NB], u32x4& bx) SRF_AI {
    const uint32_t la = slot + (at_lane ^ (s ? 128u : 0u)), lx = slot + tx + (at_lane ^ ((s ^ odd_x) ? 128u : 0u));
#pragma unroll
    for (int i = 0; i < RM; ++i) av[i] = operand(la + ta + i * 2048);
    if constexpr (ROW) av[RM] = operand(la + 8 * 2048);
#pragma unroll
    for (int k = 0; k < NC; ++k) bv[k] = operand(lx + min(col0 + k, jb.n_x / 2 - 1) * 2048);
#pragma unroll
    for (int k = 0; k < NX; ++k) bv[NC + k] = operand(lx + min(colx + 2 * k, (jb.n_x + jb.n_x2) / 2 - 1) * 2048);
    if constexpr (ROW) bx = operand(lx + (col0 + row0 / 2) * 2048);
  };
  // row sums: of two row tiles, each wave of the pair takes one
  const int my_sum = RM == 2 ? (w & 1) : 0;
  auto add_rows = [&](const u32x4& v, float& s) SRF_AI {
#pragma unroll
    for (int q = 0; q < 4; ++q) s += unpack_lo<kBF16>(v[q]) + unpack_hi<kBF16>(v[q]);
  };
  auto multiply = [&](const u32x4 (&av)[NA], const u32x4 (&bv)[NB], const u32x4& bx) SRF_AI {
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int k = 0; k < NB; ++k) acc[i][k] = mfma32x32<kBF16>(av[i], bv[k], acc[i][k]);
    if constexpr (ROW) row_acc = mfma32x32<kBF16>(av[RM], bx, row_acc);
    if (sums) {
      if constexpr (RM == 2) add_rows(my_sum ? av[1] : av[0], rs[0]);
      else add_rows(av[0], rs[0]);
    }
    if constexpr (ROW)
      if (w == 0) add_rows(av[RM], rs[RM]);
  };

  // adds the block's sums: D register r holds row 8 (r / 4) + 4 h + r % 4, column i32 of a tile
  auto add_sums = [&](bool last) SRF_AI {
    if constexpr (kAside) {
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            aside[i][k][r] += acc[i][k][r];
            acc[i][k][r] = last ? aside[i][k][r] : 0.f;
          }
      if (!last) return;
    }
    const int at = (int)lane_here(), h = at >> 5, i32 = at & 31;
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const int ct = k < NC ? col0 + k : colx + 2 * (k - NC);
        const bool ext = k >= NC;
        const int c = 32 * (ext ? ct - 8 : ct) + i32;
        float* dst = ext ? jb.dw2 : jb.dw;
        const int n = ext ? jb.N2 : jb.N;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int o = 32 * (row0 + i) + 8 * (r >> 2) + 4 * h + (r & 3);
          if (o < jb.M && c < n) unsafeAtomicAdd(dst + (size_t)o * jb.ld + c, acc[i][k][r]);
          acc[i][k][r] = 0.f;
        }
      }
    if constexpr (ROW) {
      if (h == 0) unsafeAtomicAdd(jb.dw_row + 32 * (col0 + row0 / 2) + i32, row_acc[0]);
#pragma unroll
      for (int r = 0; r < 16; ++r) row_acc[r] = 0.f;
    }
    if (sums && last) {
      const float s = rs[0] + __shfl_xor(rs[0], 32, 64);
      const int o = 32 * (row0 + my_sum) + i32;
      if (h == 0 && o < jb.M) unsafeAtomicAdd(jb.db + o, s);
    }
    if constexpr (ROW)
      if (w == 0 && last) {
        const float s = rs[RM] + __shfl_xor(rs[RM], 32, 64);
        if (lane == 0) unsafeAtomicAdd(jb.db_row, s);
      }
  };

  u32x4 a0[NA], b0[NB], x0 = {0u, 0u, 0u, 0u}, a1[NA], b1[NB], x1 = {0u, 0u, 0u, 0u};
  uint32_t rd = 0;
  // unit 0 (and the others of the prologue that every wave has waited for)
  wait_vmem_at_most(max(0, min(15, (min(slots - 1, units) - 1) * n_mine)));
  block_barrier();
  load(0, 0, a0, b0, x0);
#pragma unroll 1
  for (int u = 0, stop = min(seg_units, units); u < units; ++u) {
    // unit u + 1 has landed once only the units copied after it are outstanding; the barrier makes every
    // wave's part visible and frees the slot of unit u - 1, whose operands are all in registers
    const int after = min(slots - 3, units - 2 - u);
    wait_vmem_at_most(max(0, min(15, after * n_mine)));
    block_barrier();
    if (u + slots - 1 < units) fill();
    load(rd, 1, a1, b1, x1);
    multiply(a0, b0, x0);
    __builtin_amdgcn_sched_barrier(0);
    rd = rd + slot_bytes == (uint32_t)(slots * slot_bytes) ? 0u : rd + slot_bytes;
    load(rd, 0, a0, b0, x0);  // (past the last unit: a slot's old contents, unused)
    multiply(a1, b1, x1);
    __builtin_amdgcn_sched_barrier(0);
    if (u + 1 == stop) {
      add_sums(u + 1 == units);
      stop = min(stop + seg_units, units);
      if (!kAside && u + 1 < units) wait_vmem();  // the counted waits above are of copies alone
    }
  }
}

__global__ __launch_bounds__(64 * kDwWaves) void mlp16_dw_kernel(Dw16Args a) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[kDw16Lds * 1024];
  int ji = 0;
#pragma unroll 1
  while (ji + 1 < a.n_jobs && (int)blockIdx.x >= a.jobs[ji + 1].first_block) ++ji;
  const Dw16Job& jb = a.jobs[ji];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = w >> 1, c = w & 1;
  switch (jb.kind) {
    case kDwFull: dw16_run<2, 4, 0, false>(a, jb, 2 * r, 4 * c, 0, true, ring); break;
    case kDwWide: dw16_run<2, 4, 1, false>(a, jb, 2 * r, 4 * c, 8 + c, true, ring); break;
    case kDwTall: dw16_run<2, 4, 0, true>(a, jb, 2 * r, 4 * c, 0, true, ring); break;
    case kDwHalf: dw16_run<1, 4, 2, false>(a, jb, r, 4 * c, 8 + c, c == 0, ring); break;
    case kDwNarrow: dw16_run<2, 1, 0, false>(a, jb, 2 * r, c, 0, true, ring); break;
    default: dw16_run<1, 1, 0, false>(a, jb, 0, w, 0, w == 0, ring); break;
  }
}

int dw16_launch(const Dw16Args& a, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(mlp16_dw_kernel, dim3(blocks), dim3(64 * kDwWaves), 0, s, a);
  return launch_status();
}

}  // namespace mlp
}  // namespace srf
