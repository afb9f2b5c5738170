// Grouped weight-gradient kernel of the TensoRF colour network (design notes in color_dw.h).
#include "color_dw.h"
#include "mlp_impl.h"

namespace srf {
namespace color {
namespace {

using mlp::static_for;

constexpr int kCdwWaves = 8;
constexpr int kCdwRingKB = 160;
constexpr int kCdwMaxSlots = 8;
constexpr int kCdwLeast = 512;     // least points of a block
// 32-point steps after which a wave sets its partial sums aside, in registers, and begins anew: an FP32 sum is
// that much more exact than one over a whole range.  Gradients of 1,000,000 rows with random signs, distance from
// the FP64 sum: W1 and W2 of the 144-component network in FP32 2.0e-6 and 2.3e-6 with sums added to the gradients
// every 16,384 points, 6.5e-7 and 7.6e-7 here; all weights in the BF16 modes 2.3e-6 to 2.9e-6 and 5e-7.  The registers
// are there (252 and 240 of 256).  The row sums, few numbers that many points add up to, are compensated besides.
constexpr int kCdwAside = 32;

typedef float f32x16 __attribute__((ext_vector_type(16)));

// s_waitcnt vmcnt(n) for a wave-uniform n of at most 30.
__device__ __forceinline__ void wait_vmem_le(int n) {
  switch (n) {
#define SRF_WAIT_CASE(k) case k: __builtin_amdgcn_s_waitcnt(mlp::vmcnt_only(k)); break;
    SRF_WAIT_CASE(0) SRF_WAIT_CASE(1) SRF_WAIT_CASE(2) SRF_WAIT_CASE(3) SRF_WAIT_CASE(4) SRF_WAIT_CASE(5)
    SRF_WAIT_CASE(6) SRF_WAIT_CASE(7) SRF_WAIT_CASE(8) SRF_WAIT_CASE(9) SRF_WAIT_CASE(10) SRF_WAIT_CASE(11)
    SRF_WAIT_CASE(12) SRF_WAIT_CASE(13) SRF_WAIT_CASE(14) SRF_WAIT_CASE(15) SRF_WAIT_CASE(16) SRF_WAIT_CASE(17)
    SRF_WAIT_CASE(18) SRF_WAIT_CASE(19) SRF_WAIT_CASE(20) SRF_WAIT_CASE(21) SRF_WAIT_CASE(22) SRF_WAIT_CASE(23)
    SRF_WAIT_CASE(24) SRF_WAIT_CASE(25) SRF_WAIT_CASE(26) SRF_WAIT_CASE(27) SRF_WAIT_CASE(28) SRF_WAIT_CASE(29)
#undef SRF_WAIT_CASE
    default: __builtin_amdgcn_s_waitcnt(mlp::vmcnt_only(30)); break;
  }
}

// The block's stream of one product: points pb .. pb + 32 steps - 1 in 32-point slots, both 16-point halves
// of a slot in the same fragment order (nA dZ tiles, then nB X tiles, 1 KB each).
struct Ring {
  uint8_t* ring;
  int nf, slots, steps, slot_bytes, n_mine;
  const uint8_t* src[3];   // this wave's fragments f = w, w + 8, w + 16 of the next step
  int adv[3];              // bytes to the next step's
  uint32_t lds0, wr, rd;
  int lane_off;

  __device__ SRF_AI Ring(const CdwJob& jb, int pb, int n_steps, uint8_t* r) {
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ring = r;
    nf = jb.nA + jb.nB;
    steps = n_steps;
    slots = min(kCdwMaxSlots, kCdwRingKB / (2 * nf));
    slot_bytes = 2 * nf * 1024;
    n_mine = (nf - w + kCdwWaves - 1) / kCdwWaves;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int f = min(w + kCdwWaves * q, nf - 1);
      const bool is_a = f < jb.nA;
      adv[q] = (is_a ? jb.nA : jb.nB) * 2048;
      src[q] = (is_a ? jb.dz : jb.x) + (size_t)(pb >> 5) * adv[q] + (is_a ? f : f - jb.nA) * 2048;
    }
    // lane (g, j) copies the 16 B of feature j at the four points of lane group g (the record of
    // mlp::store_tile); the second half of the block's points lies 128 B on
    lane_off = (j & 1) * 1024 + (16 * (j >> 2) + 2 * g + ((j >> 1) & 1)) * 16;
    lds0 = lds_offset(r) + 1024u * w;
    wr = rd = 0;
    for (int i = 0; i < slots - 1 && i < steps; ++i) fill();
  }
  __device__ SRF_AI uint32_t next(uint32_t o) const { return o + slot_bytes == (uint32_t)(slots * slot_bytes) ? 0u : o + slot_bytes; }
  __device__ SRF_AI void fill() {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q < n_mine) {
        lds_dma_1k_ahead(src[q], lds0 + wr + 8192u * q, lane_off);
        lds_dma_1k_ahead(src[q] + 128, lds0 + wr + nf * 1024u + 8192u * q, lane_off);
        src[q] += adv[q];
      }
    wr = next(wr);
  }
  // load(slot byte offset of a half, operands) reads one half's operands; multiply(operands) runs its
  // products; put_aside(last) sets the partial sums aside, or with last adds them all to the gradients.
  template <typename Ops, typename Load, typename Mul, typename Aside>
  __device__ SRF_AI void run(Ops& o0, Ops& o1, Load&& load, Mul&& multiply, Aside&& put_aside) {
    wait_vmem_le(min(30, (min(slots - 1, steps) - 1) * 2 * n_mine));
    block_barrier();
    load(rd, o0);
#pragma unroll 1
    for (int st = 0; st < steps; ++st) {
      // step st + 1 has landed once only the steps copied after it are outstanding; the barrier makes every
      // wave's part visible and frees the slot of step st - 1, whose operands are all in registers
      wait_vmem_le(max(0, min(30, min(slots - 3, steps - 2 - st) * 2 * n_mine)));
      block_barrier();
      if (st + slots - 1 < steps) fill();
      load(rd + nf * 1024u, o1);
      multiply(o0);
      __builtin_amdgcn_sched_barrier(0);
      rd = next(rd);
      load(rd, o0);  // (past the last step: a slot's old contents, unused)
      multiply(o1);
      __builtin_amdgcn_sched_barrier(0);
      if ((st + 1) % kCdwAside == 0 || st + 1 == steps) put_aside(st + 1 == steps);
    }
  }
};

// A compensated sum (Kahan).  An infinite sum has nothing to compensate: inf - inf would turn it into NaN at the
// next term.
struct RowSum {
  float sum = 0.f, c = 0.f;
  __device__ SRF_AI void add(float v) {
    const float y = v - c, t = sum + y;
    c = __builtin_isinf(t) ? 0.f : (t - sum) - y;
    sum = t;
  }
};

// FP32: row tiles row0 .. row0 + RM - 1, column tiles col0 + kStride k (16 x 16 each).
template <int RM, int NC, int kStride>
__device__ __forceinline__ void run_f32(const CdwJob& jb, int row0, int col0, bool sums, Ring& ring) {
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  struct Ops { f32x4 a[RM], b[NC]; } o0, o1;
  f32x4 acc[RM][NC], aside[RM][NC];
  RowSum rs[RM];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[i][k] = aside[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  ring.run(
      o0, o1,
      [&](uint32_t at, Ops& o) SRF_AI {
        const uint8_t* fr = ring.ring + at + lane * 16;
#pragma unroll
        for (int i = 0; i < RM; ++i) o.a[i] = *reinterpret_cast<const f32x4*>(fr + min(row0 + i, jb.nA - 1) * 1024);
#pragma unroll
        for (int k = 0; k < NC; ++k)
          o.b[k] = *reinterpret_cast<const f32x4*>(fr + (jb.nA + min(col0 + kStride * k, jb.nB - 1)) * 1024);
      },
      [&](const Ops& o) SRF_AI {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int k = 0; k < NC; ++k) acc[i][k] = mfma32(o.a[i][q], o.b[k][q], acc[i][k]);
        if (sums)
#pragma unroll
          for (int i = 0; i < RM; ++i) rs[i].add((o.a[i][0] + o.a[i][1]) + (o.a[i][2] + o.a[i][3]));
      },
      [&](bool last) SRF_AI {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int k = 0; k < NC; ++k) {
            aside[i][k] += acc[i][k];
            acc[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        if (!last) return;
#pragma unroll
        for (int i = 0; i < RM; ++i) {
#pragma unroll
          for (int k = 0; k < NC; ++k) {
            const int c = 16 * (col0 + kStride * k) + j;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int o = 16 * (row0 + i) + 4 * g + r;
              if (o < jb.M && c < jb.N) unsafeAtomicAdd(jb.dw + (size_t)o * jb.ld_dw + c, aside[i][k][r]);
            }
          }
          if (sums) {
            float s = rs[i].sum;
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            const int o = 16 * (row0 + i) + j;
            if (g == 0 && o < jb.M) unsafeAtomicAdd(jb.db + o, s);
          }
        }
      });
}

// Split BF16: row block rb, column blocks cb0 .. cb0 + NC - 1 (32 x 32 each).
template <int NC>
__device__ __forceinline__ void run_split(const CdwJob& jb, int rb, int cb0, bool sums, Ring& ring) {
  const int lane = threadIdx.x & 63, h = lane >> 5, i32 = lane & 31;
  struct Ops { f32x4 a[2], b[NC][2]; } o0, o1;
  f32x16 acc[NC], aside[NC];
  RowSum rs;
#pragma unroll
  for (int k = 0; k < NC; ++k)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[k][r] = aside[k][r] = 0.f;
  // lane (h, i): its row's eight points, the records of lane groups 2 h and 2 h + 1; a 32-row block's second
  // tile past the product's rows repeats the last (rows past M, columns past N are not stored)
  const int at_lane = (2 * h * 16 + (i32 & 15)) * 16;
  auto planes = [&](const f32x4 (&v)[2], u32x4& hi, u32x4& lo) SRF_AI {
    uint32_t t[4][2];
    split_pair<2>(v[0][0], v[0][1], t[0]);
    split_pair<2>(v[0][2], v[0][3], t[1]);
    split_pair<2>(v[1][0], v[1][1], t[2]);
    split_pair<2>(v[1][2], v[1][3], t[3]);
    hi = u32x4{t[0][0], t[1][0], t[2][0], t[3][0]};
    lo = u32x4{t[0][1], t[1][1], t[2][1], t[3][1]};
  };
  ring.run(
      o0, o1,
      [&](uint32_t at, Ops& o) SRF_AI {
        const uint8_t* fr = ring.ring + at + at_lane;
        const uint8_t* fa = fr + min(2 * rb + (i32 >> 4), jb.nA - 1) * 1024;
        o.a[0] = *reinterpret_cast<const f32x4*>(fa);
        o.a[1] = *reinterpret_cast<const f32x4*>(fa + 256);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
          const uint8_t* fb = fr + (jb.nA + min(2 * (cb0 + k) + (i32 >> 4), jb.nB - 1)) * 1024;
          o.b[k][0] = *reinterpret_cast<const f32x4*>(fb);
          o.b[k][1] = *reinterpret_cast<const f32x4*>(fb + 256);
        }
      },
      [&](const Ops& o) SRF_AI {
        u32x4 ah, al, bh[NC], bl[NC];
        planes(o.a, ah, al);
#pragma unroll
        for (int k = 0; k < NC; ++k) planes(o.b[k], bh[k], bl[k]);
#pragma unroll
        for (int pr = 0; pr < 3; ++pr)
#pragma unroll
          for (int k = 0; k < NC; ++k)
            acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, pr == 0 ? al : ah),
                                                             __builtin_bit_cast(bf16x8, pr == 1 ? bl[k] : bh[k]),
                                                             acc[k], 0, 0, 0);
        if (sums)
          rs.add(((o.a[0][0] + o.a[0][1]) + (o.a[0][2] + o.a[0][3])) + ((o.a[1][0] + o.a[1][1]) + (o.a[1][2] + o.a[1][3])));
      },
      // 32x32 D layout: lane l, register r holds row 8 (r / 4) + 4 (l / 32) + (r mod 4), column l mod 32
      [&](bool last) SRF_AI {
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            aside[k][r] += acc[k][r];
            acc[k][r] = 0.f;
          }
        if (!last) return;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
          const int col = 32 * (cb0 + k) + i32;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int o = 32 * rb + 8 * (r >> 2) + 4 * h + (r & 3);
            if (o < jb.M && col < jb.N) unsafeAtomicAdd(jb.dw + (size_t)o * jb.ld_dw + col, aside[k][r]);
          }
        }
        if (sums) {
          const float s = rs.sum + __shfl_xor(rs.sum, 32, 64);
          const int o = 32 * rb + i32;
          if (h == 0 && o < jb.M) unsafeAtomicAdd(jb.db + o, s);
        }
      });
}

template <bool SPLIT>
__global__ __launch_bounds__(64 * kCdwWaves) void color_dw_kernel(CdwArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kCdwRingKB * 1024];
  const int cols = a.cols_dev ? min(a.cols, (*a.cols_dev + 255) / 256 * 256) : a.cols;
  // the block's product and range of points: product by product, each cut into ranges of equal cost
  int total = 0;
  for (int i = 0; i < a.n_jobs; ++i) total += cdw_cost<SPLIT>(a.jobs[i].nA, a.jobs[i].nB);
  const float per_block = (float)cols * (float)total / (float)(a.cus - a.n_jobs);
  int ji = 0, b = blockIdx.x, chunk = 0;
#pragma unroll 1
  for (; ji < a.n_jobs; ++ji) {
    chunk = a.chunk ? a.chunk : max(kCdwLeast, ((int)(per_block / (float)cdw_cost<SPLIT>(a.jobs[ji].nA, a.jobs[ji].nB)) + 31) / 32 * 32);
    const int n = (cols + chunk - 1) / chunk;
    if (b < n) break;
    b -= n;
  }
  if (ji == a.n_jobs) return;  // uniform over the block
  // (the ranges come from vector instructions; scalar from here on)
  ji = __builtin_amdgcn_readfirstlane(ji);
  b = __builtin_amdgcn_readfirstlane(b);
  chunk = __builtin_amdgcn_readfirstlane(chunk);
  const CdwJob& jb = a.jobs[ji];
  const int pb = b * chunk, steps = (min(pb + chunk, cols) - pb) / 32;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Ring ring(jb, pb, steps, lds);
  const CdwForm form = cdw_form<SPLIT>(jb.nA, jb.nB);
  if (jb.nA <= 2) {
    const bool sums = jb.db && w == 0;
    if constexpr (SPLIT) {
      run_split<1>(jb, 0, w, sums, ring);
    } else {
      switch (2 * form.rows + form.cols) {
        case 3: run_f32<1, 1, 8>(jb, 0, w, sums, ring); break;
        case 4: run_f32<1, 2, 8>(jb, 0, w, sums, ring); break;
        case 5: run_f32<2, 1, 8>(jb, 0, w, sums, ring); break;
        default: run_f32<2, 2, 8>(jb, 0, w, sums, ring); break;
      }
    }
  } else if constexpr (SPLIT) {
    const int rb = w & 3, half = w >> 2;
    const bool sums = jb.db && half == 0;
    switch (form.cols) {
      case 1: run_split<1>(jb, rb, 1 * half, sums, ring); break;
      case 2: run_split<2>(jb, rb, 2 * half, sums, ring); break;
      case 3: run_split<3>(jb, rb, 3 * half, sums, ring); break;
      default: run_split<4>(jb, rb, 4 * half, sums, ring); break;
    }
  } else {
    const int row0 = 2 * (w >> 1), half = w & 1;
    const bool sums = jb.db && half == 0;
    switch (form.cols) {
      case 1: run_f32<2, 1, 1>(jb, row0, 1 * half, sums, ring); break;
      case 2: run_f32<2, 2, 1>(jb, row0, 2 * half, sums, ring); break;
      case 3: run_f32<2, 3, 1>(jb, row0, 3 * half, sums, ring); break;
      case 4: run_f32<2, 4, 1>(jb, row0, 4 * half, sums, ring); break;
      case 5: run_f32<2, 5, 1>(jb, row0, 5 * half, sums, ring); break;
      case 6: run_f32<2, 6, 1>(jb, row0, 6 * half, sums, ring); break;
      case 7: run_f32<2, 7, 1>(jb, row0, 7 * half, sums, ring); break;
      default: run_f32<2, 8, 1>(jb, row0, 8 * half, sums, ring); break;
    }
  }
}

}  // namespace

int cdw_launch(const CdwArgs& a, bool split, hipStream_t s) {
  // equal costs: one round of the compute units, however many points there turn out to be
  const int blocks = a.chunk ? a.n_jobs * ((a.cols + a.chunk - 1) / a.chunk) : a.cus;
  if (split) hipLaunchKernelGGL(color_dw_kernel<true>, dim3(blocks), dim3(64 * kCdwWaves), 0, s, a);
  else hipLaunchKernelGGL(color_dw_kernel<false>, dim3(blocks), dim3(64 * kCdwWaves), 0, s, a);
  return launch_status();
}

}  // namespace color
}  // namespace srf
