// NeRF MLP forward and backward chain for 16-bit operands (BF16 training and inference, FP16
// inference) on 32x32x16 MFMAs.  Plan, workspace and weight gradients are those of mlp_impl.h.
//
// Why 32x32: with one wave per SIMD (the accumulators take the whole AGPR file) a stream of
// independent 16x16x32 MFMAs on random operands reaches 1.40-1.50 PFLOP/s on this chip, the same
// products as 32x32x16 MFMAs 1.79 PFLOP/s (1.58 and 2.49 on zeros: the larger shape also draws less
// power per product).  4,096 rays x 192 samples, main model: training forward 1,705 us on 16x16x32 tiles,
// 1,214 us here; backward chain 1,339 -> 1,078 us; inference of 16,384 x 192 points 3,981 -> 3,444 us.
// Part of it is the epilogue: ReLU by v_med3, masks from packed pairs, tile records without a lane exchange
// (2,700 -> 1,100 vector operations a layer).
//
// Lane layout (lane = 32 h + c, h = 0, 1):
//   A operand (32 x 16): row c, eight reduction slots i = 0 .. 7
//   B operand (16 x 32): column c, the same slots
//   D tile (32 x 32):    register 4 q + r holds row 8 q + 4 h + r (q, r = 0 .. 3) of column c
// k-step 2 T + m of a layer takes feature 32 T + 16 (i / 4) + 8 m + 4 h + i % 4 in slot (h, i): the packed
// registers q = m and q = m + 2 of D tile T are, bit for bit, its B operand.  A 16x16x32 MFMA with the
// slot map of mfma.h adds the eight products of lane group g = 0, 1, 2, 3 after one another, and a
// 32x32x16 MFMA those of h = 0, 1; this map gives groups 0, 1 to m = 0 and 2, 3 to m = 1, so that the sums
// are rounded in the same order and the results are those of the 16x16x32 kernels bit for bit.
// A wave owns 32 NB points (column blocks), one register quad per (k-step, column block).
#pragma once

#include "mlp_impl.h"

namespace srf {
namespace mlp {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int P>
__device__ __forceinline__ f32x16 mfma32x32(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (P == kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

// Weight stage: two buffers of one chunk each.  The packed image of a product lists its 1 KB
// fragments k-step by k-step (all OUT row tiles of k-step 0, then of k-step 1, ...), so a chunk of
// kChunk / OUT k-steps is one linear copy and the wave reads its fragments in the order they lie.
constexpr int kChunk = 32;  // fragments of a chunk (32 KB)
struct Stage16 {
  uint8_t* base;
  uint32_t off;  // byte offset of the buffer that holds the next product's first chunk (0 or 32 KB)
};

// The first chunk of the product that follows: n fragments (0: none) at src.
struct NextChunk {
  const uint8_t* src;
  int n;
};

// Copies n fragments (n <= kChunk, uniform) at src into the buffer at dst, by the block's waves together.
__device__ __forceinline__ void dma_frags(const uint8_t* __restrict__ src, int n, uint8_t* dst) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < kChunk / kWaves; ++i) {
    const int f = w + kWaves * i;
    if (f < n) lds_dma_1k(src + (size_t)f * 1024, dst + f * 1024);
  }
}

__device__ __forceinline__ void block_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc[T][cb] (+)= rows 32 T .. of the image at img times the NK k-steps that fin(s, cb) returns; the
// sum starts from the bias of those rows (kBias), from zero (kZero) or from acc (kAdd).
// On entry the first chunk lies in the stage (st.off); every wave of the block must come here.  While
// a chunk is multiplied the next one is copied, and while the last one is, the first chunk of the
// product that follows (next): its latency hides behind this product's epilogue.
// Deferred stores: side(i), i in [0, NSIDE), issues at least two vector-memory operations each (the
// training copies of the tiles that this product reads).  They are spread over the groups of MFMAs, and
// a chunk waits with vmcnt(operations issued after its copy), since these complete in issue order.
enum { kZero, kBias, kAdd };
template <int P, int NB, int NK, int OUT, int INIT, int NSIDE = 0, typename FIn, typename Side = NoSide>
__device__ __forceinline__ void product(f32x16 (&acc)[OUT][NB], const uint8_t* __restrict__ img, const float* bias,
                                        FIn&& fin, Stage16& st, NextChunk next, Side&& side = Side{}) {
  constexpr int KC = kChunk / OUT < NK ? kChunk / OUT : NK;  // k-steps per chunk
  constexpr int NCH = (NK + KC - 1) / KC;
  constexpr int kPer = (NSIDE + NCH - 1) / NCH;               // side items per chunk
  constexpr int kG = 4;                                       // fragments per group
  const int lane = threadIdx.x & 63;
  const float* bias_h = bias + 4 * (lane >> 5);
  static_for<0, NCH>([&](auto CI) SRF_AI {
    constexpr int c = decltype(CI)::value;
    constexpr int kn = NK - c * KC < KC ? NK - c * KC : KC;
    constexpr int NF = kn * OUT, NG = (NF + kG - 1) / kG;
    const uint8_t* cur = st.base + st.off;
    st.off ^= kChunk * 1024;
    if constexpr (c + 1 < NCH) {
      constexpr int kn1 = NK - (c + 1) * KC < KC ? NK - (c + 1) * KC : KC;
      dma_frags(img + (size_t)(c + 1) * KC * OUT * 1024, kn1 * OUT, st.base + st.off);
    } else if (next.n) {
      dma_frags(next.src, next.n, st.base + st.off);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    constexpr int i0 = c * kPer < NSIDE ? c * kPer : NSIDE;
    constexpr int i1 = (c + 1) * kPer < NSIDE ? (c + 1) * kPer : NSIDE;
    constexpr int per_group = (i1 - i0 + NG - 1) / NG;
    auto read_a = [&](auto GI, u32x4 (&a)[kG]) SRF_AI {
      constexpr int g = decltype(GI)::value;
#pragma unroll
      for (int q = 0; q < kG; ++q)
        if (g * kG + q < NF) a[q] = *reinterpret_cast<const u32x4*>(cur + (g * kG + q) * 1024 + lane * 16);
    };
    // the fragments of group g + 1 are read from LDS while the MFMAs of group g run; the scheduling
    // barriers keep the compiler from hoisting every read of the chunk
    u32x4 a_cur[kG], a_nxt[kG];
    read_a(std::integral_constant<int, 0>{}, a_cur);
    static_for<0, NG>([&](auto GI) SRF_AI {
      constexpr int g = decltype(GI)::value;
      if constexpr (g + 1 < NG) read_a(std::integral_constant<int, g + 1>{}, a_nxt);
      static_for<0, kG>([&](auto QI) SRF_AI {
        constexpr int f = g * kG + decltype(QI)::value;
        if constexpr (f < NF) {
          constexpr int s = c * KC + f / OUT, T = f % OUT;
          f32x16 init;
          if constexpr (s == 0 && INIT == kBias) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4 b = *reinterpret_cast<const f32x4*>(bias_h + 32 * T + 8 * q);
#pragma unroll
              for (int r = 0; r < 4; ++r) init[4 * q + r] = b[r];
            }
          } else if constexpr (s == 0 && INIT == kZero) {
#pragma unroll
            for (int r = 0; r < 16; ++r) init[r] = 0.f;
          }
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) {
            if constexpr (s == 0 && INIT != kAdd) acc[T][cb] = mfma32x32<P>(a_cur[decltype(QI)::value], fin(s, cb), init);
            else acc[T][cb] = mfma32x32<P>(a_cur[decltype(QI)::value], fin(s, cb), acc[T][cb]);
          }
        }
      });
      static_for<0, per_group>([&](auto KI) SRF_AI {
        constexpr int i = i0 + g * per_group + decltype(KI)::value;
        if constexpr (i < i1) side(std::integral_constant<int, i>{});
      });
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kG; ++q) a_cur[q] = a_nxt[q];
    });
    // the copy has landed once at most the 2 (i1 - i0) operations issued after it are outstanding; the
    // barrier also frees the buffer that this chunk read (its reads were consumed by the MFMAs above)
    if (c + 1 < NCH || next.n) {
      constexpr int after = 2 * (i1 - i0);
      __builtin_amdgcn_s_waitcnt(vmcnt_only(after < 63 ? after : 63));
    }
    block_barrier();
  });
}

// Stores 16-feature tile t of the wave's 64 points as the 2 KB block that the weight-gradient GEMM
// reads (mlp_dw_kernel): record (h, c), chunk k at byte 1024 k + 16 (32 h + c), holds features 8 k + 4 h +
// r (r = 0 .. 3, one dword each) at the lane's own points c and 32 + c.  Chunk k comes from quad k of the
// tile's pair (its k-steps 2 (t / 2) + k) in both column blocks.  One byte permutation a dword, no lane
// exchange, and each of the two stores writes 1 KB of whole lines.  Non-temporal, as store_tile's.
template <int T>
__device__ __forceinline__ u32x4 tile_chunk(const u32x4& a, const u32x4& b) {
  constexpr uint32_t kLo = 0x05040100, kHi = 0x07060302;  // the low / high halves of two dwords
  constexpr int d = 2 * (T & 1);
  const uint32_t a0 = a[d], a1 = a[d + 1], b0 = b[d], b1 = b[d + 1];
  return u32x4{__builtin_amdgcn_perm(b0, a0, kLo), __builtin_amdgcn_perm(b0, a0, kHi),
               __builtin_amdgcn_perm(b1, a1, kLo), __builtin_amdgcn_perm(b1, a1, kHi)};
}
template <int T>
__device__ __forceinline__ void store_tile16(Rsrc dst, uint32_t blk, const u32x4 (&q0)[2], const u32x4 (&q1)[2]) {
  const uint32_t rec = lane_here() * 16u;
  store_nt16(dst, rec, blk, tile_chunk<T>(q0[0], q0[1]));
  store_nt16(dst, rec, blk + 1024, tile_chunk<T>(q1[0], q1[1]));
}

// The two quads of 32 rows (one D tile) from their eight packed pairs d[2 q + p].
__device__ __forceinline__ u32x4 quad_of(const uint32_t (&d)[8], int m) { return u32x4{d[2 * m], d[2 * m + 1], d[4 + 2 * m], d[5 + 2 * m]}; }

// Positional encoding straight into B-operand quads (lane = point of the wave).
template <int P, int NB>
struct PeQuads {
  // features [f_lo, f_hi) of PE_L(x) at columns f - shift of the wave's quads
  __device__ static SRF_AI void put(uint8_t* quads, int col, float v) {
    const int pt = (threadIdx.x & 63) % (32 * NB);
    const int step = 2 * (col >> 5) + ((col >> 3) & 1);
    const int at = (step * NB + (pt >> 5)) * 1024 + (((col >> 2) & 1) * 32 + (pt & 31)) * 16 +
                   (((col >> 4) & 1) * 4 + (col & 3)) * 2;
    *reinterpret_cast<uint16_t*>(quads + at) = (uint16_t)(pack2<P>(v, 0.f) & 0xffffu);
  }
  __device__ static SRF_AI void write(uint8_t* quads, const float (&x)[3], int L, int f_lo, int f_hi, int shift) {
    // NB = 1: two lanes per point share its levels
    const int part = (threadIdx.x & 63) / (32 * NB), parts = 2 / NB;
    if (part == 0)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (c >= f_lo && c < f_hi) put(quads, c - shift, x[c]);
    for (int m = part; m < L; m += parts) {
      if (8 + 6 * m < f_lo || 3 + 6 * m >= f_hi) continue;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float sn, cs;
        pe_sincos(ldexpf(x[c], m), &sn, &cs);
        const int fs = 3 + 6 * m + c, fc = 6 + 6 * m + c;
        if (fs >= f_lo && fs < f_hi) put(quads, fs - shift, sn);
        if (fc >= f_lo && fc < f_hi) put(quads, fc - shift, cs);
      }
    }
  }
  // columns [n, 16 steps) are zero
  __device__ static SRF_AI void pad(uint8_t* quads, int n, int steps) {
    for (int col = n; col < 16 * steps; ++col) put(quads, col, 0.f);
  }
};

// ------------------------------------------------------------------------ forward
// Training keeps every layer's input and ReLU mask (64-point waves, NB = 2).
template <int P, bool VD, bool TRAIN, int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mlp16_fwd_kernel(FwdArgs a) {
  static_assert(!TRAIN || NB == 2, "the training layout is that of 64-point waves");
  __shared__ __attribute__((aligned(16))) uint8_t stage[2 * kChunk * 1024];
  // computed input features of each wave's points (trunk PE for layers 0 and 5, then the view layer's
  // [PE_xyz[trunk_pe:], PE_dir]) as B-operand quads, written and read by the wave alone
  __shared__ __attribute__((aligned(16))) u32x4 pe_lds[kWaves][6][NB][64];
  __shared__ __attribute__((aligned(16))) float bias_lds[kMaxBiasFloats];
  const int lane = threadIdx.x & 63, h = lane >> 5, cl = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = blockIdx.x * kWaves + wv;
  const int p0 = wave * 32 * NB;
  const Plan& pl = a.p;
  const int ldP = a.w.ldP;
  Stage16 st{stage, 0};
  uint8_t* quads = reinterpret_cast<uint8_t*>(&pe_lds[wv][0][0][0]);
  using PE = PeQuads<P, NB>;
  auto image = [&](int l, int kstep_frags = 0) SRF_AI { return a.packed + pl.fwd_off[l] + (size_t)kstep_frags * 1024; };

  dma_frags(image(0), kChunk, stage);  // layer 0's only chunk
  {
    const float* src = reinterpret_cast<const float*>(a.packed + pl.bias_off[0]);
    for (int i = threadIdx.x; i < pl.bias_floats; i += 64 * kWaves) bias_lds[i] = src[i];
  }
  auto bias_of = [&](int l) SRF_AI { return bias_lds + (pl.bias_off[l] - pl.bias_off[0]) / 4; };

  // the lane's point (PE): stored, or rays_o[..., None, :] + rays_d[..., None, :] * z[..., :, None] of
  // its ray (src/models/SimpleNeRF17.py:213-215, :266-268; two rounded FP32 operations)
  const int pe_p = p0 + lane % (32 * NB);
  const bool pe_in = pe_p < a.n;
  auto load_xyz = [&](float (&v)[3]) SRF_AI {
    const int r = a.z && pe_in ? pe_p / a.n_samples : 0;
    const float zz = a.z && pe_in ? a.z[pe_p] : 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (!pe_in) v[c] = 0.f;
      else if (a.z) v[c] = __fadd_rn(a.rays_o[3 * r + c], __fmul_rn(a.rays_d[3 * r + c], zz));
      else v[c] = a.pts[3 * pe_p + c];
    }
  };
  // its view direction: stored per point, or its ray's (:429-433)
  auto load_dir = [&](float (&v)[3]) SRF_AI {
    const int r = !pe_in ? 0 : (a.z ? pe_p / a.n_samples : pe_p);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = pe_in ? a.dirs[3 * r + c] : 0.f;
  };
  {
    float x[3];
    load_xyz(x);
    PE::write(quads, x, pl.pts_deg, 0, pl.trunk_pe, 0);
    PE::pad(quads, pl.trunk_pe, 4);
  }

  u32x4 q[16][NB];       // the layer input: quad s, column block cb
  uint32_t mbits[NB][4];  // ReLU mask: word T / 2, see relu_epi
  auto fin_q = [&](int s, int cb) SRF_AI { return q[s][cb]; };
  auto fin_pe = [&](int s, int cb) SRF_AI { return pe_lds[wv][s][cb][lane]; };
  // ReLU, packing and (training) the mask from the packed pairs: both bits of pair 8 (T % 2) + 2 qq + p
  // of word T / 2 lie at 15 minus that in the word's halves (push_nonzero)
  auto relu_epi = [&](auto TI, f32x16(&v)[NB]) SRF_AI {
    constexpr int T = decltype(TI)::value;
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      uint32_t d[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) d[i] = pack2<P>(relu1(v[cb][2 * i]), relu1(v[cb][2 * i + 1]));
      q[2 * T][cb] = quad_of(d, 0);
      q[2 * T + 1][cb] = quad_of(d, 1);
      if constexpr (TRAIN) {
        if ((T & 1) == 0) mbits[cb][T >> 1] = 0;
#pragma unroll
        for (int i = 0; i < 8; i += 2) push_nonzero(mbits[cb][T >> 1], d[i], d[i + 1]);
      }
    }
  };
  // Deferred stores of the tiles that a product reads: NQ quads of q at ws offset q_off, then NPE PE
  // quads at pe_off, then (slot >= 0) the ReLU mask of the layer that produced q.
  constexpr int kT = TRAIN ? 1 : 0;
  auto side_of = [&](auto NQI, size_t q_off, auto NPEI, size_t pe_off, int slot) SRF_AI {
    constexpr int nq = decltype(NQI)::value, npe = decltype(NPEI)::value;
    const Rsrc rq = uniform_rsrc(a.ws + q_off), rpe = uniform_rsrc(a.ws + pe_off);
    const Rsrc rm = uniform_rsrc(a.ws + a.w.mask + (size_t)(slot < 0 ? 0 : slot) * ldP * 32);
    return [&, rq, rpe, rm](auto II) SRF_AI {
      constexpr int i = decltype(II)::value;
      if constexpr (NB == 2) {
        if constexpr (i < nq) {
          store_tile16<i>(rq, tile_block<P>(i, ldP, pl.elem, p0), q[i & ~1], q[i | 1]);
        } else if constexpr (i < nq + npe) {
          constexpr int t = i - nq;
          u32x4 e[2][2];
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) e[k][cb] = pe_lds[wv][(t & ~1) + k][cb][lane];
          store_tile16<t>(rpe, tile_block<P>(t, ldP, pl.elem, p0), e[0], e[1]);
        } else {
#pragma unroll
          for (int cb = 0; cb < 2; ++cb)
            store_nt16(rm, lane_here() * 16u, (uint32_t)wave * 2048u + cb * 1024u,
                       u32x4{mbits[cb][0], mbits[cb][1], mbits[cb][2], mbits[cb][3]});
        }
      }
    };
  };
  using I0 = std::integral_constant<int, 0>;
  using I16 = std::integral_constant<int, 16>;

  wait_vmem();
  __syncthreads();  // layer 0's weights, the biases and the PE quads

  // ---- layer 0: PE(trunk) -> 256 (stores the PE tiles)
  {
    f32x16 acc[8][NB];
    product<P, NB, 4, 8, kBias, 4 * kT>(acc, image(0), bias_of(0), fin_pe, st, NextChunk{image(1), kChunk},
                                        side_of(I0{}, 0, std::integral_constant<int, 4>{}, a.w.x0, -1));
    static_for<0, 8>([&](auto TI) SRF_AI { relu_epi(TI, acc[decltype(TI)::value]); });
  }
  // ---- layers 1..7 in place in q; layer 5 adds the trunk PE (storing layer l - 1's output and mask)
  // (three copies of the layer body: with layer 5's extra product behind a branch in one loop, the
  // accumulators meet at its join and the compiler spills and copies them)
  auto trunk_layer = [&](int l, auto SKIP) SRF_AI {
    constexpr bool skip = decltype(SKIP)::value;
    f32x16 acc[8][NB];
    // what comes after layer 7: the sigma tile (stored behind the feature tiles) or the 4-channel head
    const NextChunk nx = skip ? NextChunk{image(5, 16 * 8), kChunk}
                         : l < 7 ? NextChunk{image(l + 1), kChunk}
                                 : NextChunk{image(8, VD ? 16 * 8 : 0), 16};
    product<P, NB, 16, 8, kBias, 17 * kT>(acc, image(l), bias_of(l), fin_q, st, nx,
                                          side_of(I16{}, a.w.h[l - 1], I0{}, 0, l - 1));
    if constexpr (skip) {
      product<P, NB, 4, 8, kAdd>(acc, image(5, 16 * 8), nullptr, fin_pe, st, NextChunk{image(6), kChunk});
    }
    static_for<0, 8>([&](auto TI) SRF_AI { relu_epi(TI, acc[decltype(TI)::value]); });
  };
#pragma unroll 1
  for (int l = 1; l < 5; ++l) trunk_layer(l, std::false_type{});
  trunk_layer(5, std::true_type{});
#pragma unroll 1
  for (int l = 6; l < 8; ++l) trunk_layer(l, std::false_type{});

  // ---- heads (their rows lie in the lanes h = 0)
  auto head_sigma = [&](int p, float raw) SRF_AI {
    if (a.noise) raw = raw + a.noise[p];
    a.sigma[p] = pl.softplus ? softplusf_(raw) : (raw > 0.f ? raw : 0.f);
  };
  f32x16 hd[1][NB];
  if constexpr (!VD) {
    // 4-channel output: sigma, rgb (src/models/SimpleNeRF17.py:735-750); stores layer 7
    product<P, NB, 16, 1, kBias, 17 * kT>(hd, image(8), bias_of(8), fin_q, st, NextChunk{nullptr, 0},
                                          side_of(I16{}, a.w.h[7], I0{}, 0, 7));
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n) {
        head_sigma(p, hd[0][cb][0]);
#pragma unroll
        for (int c = 0; c < 3; ++c) a.rgb[3 * p + c] = sigmoidf_(hd[0][cb][1 + c]);
      }
    }
  } else {
    product<P, NB, 16, 1, kBias>(hd, image(8, 16 * 8), bias_of(8) + 256, fin_q, st, NextChunk{image(8), kChunk});
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n) head_sigma(p, hd[0][cb][0]);
    }
    {
      // feature rows 0..255 (no activation) in place in q; stores layer 7
      f32x16 acc[8][NB];
      product<P, NB, 16, 8, kBias, 17 * kT>(acc, image(8), bias_of(8), fin_q, st, NextChunk{image(9), kChunk},
                                            side_of(I16{}, a.w.h[7], I0{}, 0, 7));
      static_for<0, 8>([&](auto TI) SRF_AI {
        constexpr int T = decltype(TI)::value;
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          uint32_t d[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) d[i] = pack2<P>(acc[T][cb][2 * i], acc[T][cb][2 * i + 1]);
          q[2 * T][cb] = quad_of(d, 0);
          q[2 * T + 1][cb] = quad_of(d, 1);
        }
      });
    }
    // the view layer's computed inputs [PE_xyz[trunk_pe:], PE_dir]
    {
      const int pts_dim = 3 * (2 * pl.pts_deg + 1), n_hi = pts_dim - pl.trunk_pe;
      float x[3], d[3];
      load_xyz(x);
      load_dir(d);
      if (n_hi > 0) PE::write(quads, x, pl.pts_deg, pl.trunk_pe, pts_dim, pl.trunk_pe);
      PE::write(quads, d, pl.dir_deg, 0, pl.extra - n_hi, -n_hi);
      PE::pad(quads, pl.extra, pl.comp_tiles[9]);
      wave_lds_sync();
    }
    // view layer [feature, extras] -> 128, in place into q[0..7]; stores the feature tiles and the extras
    auto fin_qe = [&](int s, int cb) SRF_AI { return s < 16 ? q[s < 16 ? s : 0][cb] : pe_lds[wv][s < 16 ? 0 : s - 16][cb][lane]; };
    {
      f32x16 acc[4][NB];
      const NextChunk nx{image(10), 8};
      if (pl.comp_tiles[9] == 2)
        product<P, NB, 18, 4, kBias, 18 * kT>(acc, image(9), bias_of(9), fin_qe, st, nx,
                                              side_of(I16{}, a.w.f, std::integral_constant<int, 2>{}, a.w.ex, -1));
      else if (pl.comp_tiles[9] == 4)
        product<P, NB, 20, 4, kBias, 20 * kT>(acc, image(9), bias_of(9), fin_qe, st, nx,
                                              side_of(I16{}, a.w.f, std::integral_constant<int, 4>{}, a.w.ex, -1));
      else
        product<P, NB, 22, 4, kBias, 22 * kT>(acc, image(9), bias_of(9), fin_qe, st, nx,
                                              side_of(I16{}, a.w.f, std::integral_constant<int, 6>{}, a.w.ex, -1));
      static_for<0, 4>([&](auto TI) SRF_AI { relu_epi(TI, acc[decltype(TI)::value]); });
      if constexpr (TRAIN)
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) mbits[cb][2] = mbits[cb][3] = 0;
    }
    // rgb head 128 -> 3, sigmoid (stores the view layer's output and mask)
    product<P, NB, 8, 1, kBias, 9 * kT>(hd, image(10), bias_of(10), fin_q, st, NextChunk{nullptr, 0},
                                        side_of(std::integral_constant<int, 8>{}, a.w.v, I0{}, 0, 8));
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n)
#pragma unroll
        for (int c = 0; c < 3; ++c) a.rgb[3 * p + c] = sigmoidf_(hd[0][cb][c]);
    }
  }
}

// ------------------------------------------------------------------- backward chain
template <int P, bool VD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mlp16_bwd_kernel(BwdArgs a) {
  constexpr int NB = 2;
  __shared__ __attribute__((aligned(16))) uint8_t stage[2 * kChunk * 1024];
  const int lane = threadIdx.x & 63, h = lane >> 5, cl = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = blockIdx.x * kWaves + wv;
  const int p0 = wave * 32 * NB;
  const Plan& pl = a.p;
  const int ldP = a.w.ldP;
  Stage16 st{stage, 0};
  auto image = [&](int l) SRF_AI { return a.packed + pl.bwd_off[l]; };
  dma_frags(image(VD ? 10 : 8), VD ? 4 : 8, stage);  // the first product's only chunk

  float dsr[NB], drr[NB][3];  // head pre-activation gradients
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    const int p = p0 + 32 * cb + cl;
    const bool valid = p < a.n;
    const float ds = valid ? a.d_sigma[p] : 0.f, s = valid ? a.sigma[p] : 0.f;
    dsr[cb] = pl.softplus ? ds * (1.0f - expf(-s)) : (s > 0.f ? ds : 0.f);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float dr = valid ? a.d_rgb[3 * p + c] : 0.f, y = valid ? a.rgb[3 * p + c] : 0.f;
      drr[cb][c] = dr * (1.0f - y) * y;
    }
  }

  // z holds the current layer's pre-activation gradients as B-operand quads; every product writes in
  // place, and the next one stores what it reads for the weight gradients (deferred stores).
  u32x4 z[18][NB];  // (z[17]: zero padding)
  uint32_t mb[NB][4];
  auto fin_z = [&](int s, int cb) SRF_AI { return z[s][cb]; };
  // item 0 (slot >= 0): the ReLU masks of that slot, for the epilogue of the product they are loaded in;
  // then the quads of z as tiles of dZ_l
  auto side_of = [&](auto MI, int slot, int l) SRF_AI {
    constexpr int nm = decltype(MI)::value;
    const Rsrc rz = uniform_rsrc(a.ws + a.w.dz[l]);
    const Rsrc rm = uniform_rsrc(a.ws + a.w.mask + (size_t)(slot < 0 ? 0 : slot) * ldP * 32);
    return [&, rz, rm](auto II) SRF_AI {
      constexpr int i = decltype(II)::value;
      if constexpr (i < nm) {
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rm, lane * 16u, (uint32_t)wave * 2048u + cb * 1024u, 0);
#pragma unroll
          for (int k = 0; k < 4; ++k) mb[cb][k] = v[k];
        }
      } else {
        constexpr int t = i - nm;
        store_tile16<t>(rz, tile_block<P>(t, ldP, pl.elem, p0), z[t & ~1], z[t | 1]);
      }
    };
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  // ReLU-masked gradient into z (the forward's bit order, mlp16_fwd_kernel's relu_epi)
  auto masked_epi = [&](auto TI, f32x16(&v)[NB]) SRF_AI {
    constexpr int T = decltype(TI)::value;
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      uint32_t d[8];
      static_for<0, 8>([&](auto KI) SRF_AI {
        constexpr int i = decltype(KI)::value;
        d[i] = pack2<P>(v[cb][2 * i], v[cb][2 * i + 1]) & half_mask<8 * (T & 1) + i>(mb[cb][T >> 1]);
      });
      z[2 * T][cb] = quad_of(d, 0);
      z[2 * T + 1][cb] = quad_of(d, 1);
    }
  };
  // a head's gradient rows 0..3 as quads s, s + 1
  auto head_quad = [&](int s, int cb, float r0, float r1, float r2, float r3) SRF_AI {
    z[s][cb] = h == 0 ? u32x4{pack2<P>(r0, r1), pack2<P>(r2, r3), 0u, 0u} : u32x4{0u, 0u, 0u, 0u};
    z[s + 1][cb] = u32x4{0u, 0u, 0u, 0u};
  };
  wait_vmem();
  __syncthreads();

  if constexpr (VD) {
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) head_quad(0, cb, drr[cb][0], drr[cb][1], drr[cb][2], 0.f);
    {
      // dV = W10^T dZ10, masked by the view-layer ReLU -> dZ9 (z[0..7]); stores dZ10
      f32x16 acc[4][NB];
      product<P, NB, 1, 4, kZero, 2>(acc, image(10), nullptr, fin_z, st, NextChunk{image(9), kChunk}, side_of(I1{}, 8, 10));
      static_for<0, 4>([&](auto TI) SRF_AI { masked_epi(TI, acc[decltype(TI)::value]); });
    }
    {
      // dF = W9^T dZ9 (feature part, no activation) -> dZ8 rows 0..255 (z[0..15]); stores dZ9
      f32x16 acc[8][NB];
      product<P, NB, 8, 8, kZero, 8>(acc, image(9), nullptr, fin_z, st, NextChunk{image(8), kChunk}, side_of(I0{}, -1, 9));
      static_for<0, 8>([&](auto TI) SRF_AI {
        constexpr int T = decltype(TI)::value;
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          uint32_t d[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) d[i] = pack2<P>(acc[T][cb][2 * i], acc[T][cb][2 * i + 1]);
          z[2 * T][cb] = quad_of(d, 0);
          z[2 * T + 1][cb] = quad_of(d, 1);
        }
      });
    }
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) head_quad(16, cb, dsr[cb], 0.f, 0.f, 0.f);
    f32x16 acc[8][NB];
    product<P, NB, 17, 8, kZero, 18>(acc, image(8), nullptr, fin_z, st, NextChunk{image(7), kChunk}, side_of(I1{}, 7, 8));
    static_for<0, 8>([&](auto TI) SRF_AI { masked_epi(TI, acc[decltype(TI)::value]); });
  } else {
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) head_quad(0, cb, dsr[cb], drr[cb][0], drr[cb][1], drr[cb][2]);
    f32x16 acc[8][NB];
    product<P, NB, 1, 8, kZero, 2>(acc, image(8), nullptr, fin_z, st, NextChunk{image(7), kChunk}, side_of(I1{}, 7, 8));
    static_for<0, 8>([&](auto TI) SRF_AI { masked_epi(TI, acc[decltype(TI)::value]); });
  }
  // trunk: z holds dZ_l; dH_{l-1} = W_l^T dZ_l, masked -> dZ_{l-1}, in place (storing dZ_l)
  for (int l = 7; l >= 1; --l) {
    f32x16 acc[8][NB];
    product<P, NB, 16, 8, kZero, 17>(acc, image(l), nullptr, fin_z, st, NextChunk{image(l > 1 ? l - 1 : 1), l > 1 ? kChunk : 0},
                                     side_of(I1{}, l - 1, l));
    static_for<0, 8>([&](auto TI) SRF_AI { masked_epi(TI, acc[decltype(TI)::value]); });
  }
  // dZ0: no product follows
  const Rsrc rz = uniform_rsrc(a.ws + a.w.dz[0]);
  static_for<0, 16>([&](auto TI) SRF_AI {
    constexpr int t = decltype(TI)::value;
    store_tile16<t>(rz, tile_block<P>(t, ldP, pl.elem, p0), z[t & ~1], z[t | 1]);
  });
}

template <int P, bool VD, bool TRAIN, int NB>
int launch_fwd16(const FwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mlp16_fwd_kernel<P, VD, TRAIN, NB>), dim3(a.w.cols / (kWaves * 32 * NB)), dim3(64 * kWaves), 0, s, a);
  return launch_status();
}

template <int P, bool VD>
int launch_bwd16(const BwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mlp16_bwd_kernel<P, VD>), dim3(a.w.cols / (kWaves * 64)), dim3(64 * kWaves), 0, s, a);
  return launch_status();
}

}  // namespace mlp
}  // namespace srf
