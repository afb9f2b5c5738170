// NeRF MLP forward and backward chain for 16-bit operands (BF16 training and inference, FP16
// inference) on 32x32x16 MFMAs.  Plan and workspace are those of mlp_impl.h; the weight gradients are in
// mlp16_dw.h.
//
// Why 32x32: with one wave per SIMD a stream of
// independent 16x16x32 MFMAs on random operands reaches 1.40-1.50 PFLOP/s on this chip, the same
// products as 32x32x16 MFMAs 1.79 PFLOP/s (1.58 and 2.49 on zeros: the larger shape also draws less
// power per product).  4,096 rays x 192 samples, main model: training forward 1,705 us on 16x16x32 tiles,
// 1,103 us here; backward chain 1,339 -> 894 us; inference of 16,384 x 192 points 3,985 -> 2,956 us.
// The kernels are bound by the MFMAs (a 256 x 256 layer of 256 points: 3.5 us at the full clock, 4.8 us at
// the clock that random operands leave), their operand reads from LDS (half of its rate) and, in training,
// the stores (5.5 and 5.2 KB a point: 630 us at a fill's rate for 786,432 points).
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

// Weight stream.  The packed images of a kernel's products lie in the order of their use, each row tile's
// fragments (1 KB, one per k-step, padded to whole units) together: a product runs row tile by row tile,
// all its k-steps, so that only two tiles' accumulators are live, a tile's epilogue runs between the
// MFMAs of the next one, and the layer's outputs fit the AGPRs beside its inputs.  (The earlier form held
// all eight tiles' accumulators and ran its epilogues, 1,100 vector operations a layer, after them.)
// The stream goes through a ring of units of four fragments, copied global -> LDS by the block's four
// waves (one fragment each) and read by all of them one unit ahead of its use.  Every unit used copies the
// one kAhead units further on, so the copies need no schedule; the last ones of a kernel run past its
// images (into what follows them, or the buffer's pad) and are waited for at its end.
// A group is at most six units between two synchronisations.  At its start (sync) all its units and the
// next one have landed, and the waves have read all earlier units, so that at most kAhead + 6 units of
// the ring are in use.
constexpr int kUnit = 4096;
constexpr int kRingUnits = 24;   // 96 KB
constexpr int kAhead = 16;
static_assert((kAhead + 1) * kUnit <= kPackPad, "the copies past the last image stay in the buffer");
struct Stream16 {
  const uint8_t* src;   // this wave's fragment of the next unit to copy
  const uint8_t* ring;
  uint32_t lds;         // LDS offset of this wave's fragment of the ring's first unit
  uint32_t wr, rd;      // byte offsets of the unit to copy / in a
  u32x4 a[4];           // the fragments of the current unit

  __device__ SRF_AI Stream16(const uint8_t* image, const uint8_t* ring_) {
    const uint32_t frag = 1024u * (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    src = image + frag;
    ring = ring_;
    lds = lds_offset(ring_) + frag;
    wr = rd = 0;
#pragma unroll
    for (int i = 0; i < kAhead; ++i) copy();
  }
  __device__ SRF_AI static uint32_t next(uint32_t o) { return o + kUnit == kRingUnits * kUnit ? 0u : o + kUnit; }
  __device__ SRF_AI void copy() {
    lds_dma_1k_ahead(src, lds + wr, (threadIdx.x & 63) * 16);
    src += kUnit;
    wr = next(wr);
  }
  __device__ SRF_AI u32x4 read(uint32_t off, int i) const {
    return *reinterpret_cast<const u32x4*>(ring + off + i * 1024 + (threadIdx.x & 63) * 16);
  }
  // The first unit, once the prologue has waited for the copies.
  __device__ SRF_AI void begin() {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = read(0, i);
  }
  // Start of a group.  This wave's copies of the group's units and the next one were issued at least nine
  // copies and kStores stores ago, and vector-memory operations complete in issue order.
  template <int kStores>
  __device__ SRF_AI void sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vmcnt_only(kAhead - 7 + kStores));
    block_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  // One unit: f(i, fragment) for its four fragments, reading the next unit's meanwhile.
  template <typename F>
  __device__ SRF_AI void unit(F&& f) {
    rd = next(rd);
    static_for<0, 4>([&](auto II) SRF_AI {
      constexpr int i = decltype(II)::value;
      f(II, a[i]);
      a[i] = read(rd, i);
      if constexpr (i == 1) copy();
      __builtin_amdgcn_sched_barrier(0);
    });
  }
};

// A value in an accumulation register (the MFMAs read their operands from there; vector operations
// cannot).  Its output is not an operand that the register also holds before, as push_nonzero's are (the register
// pressure of that spills hundreds of values), so it may be any accumulation register: what makes that safe is
// that no MFMA of these kernels writes one (-amdgpu-mfma-vgpr-form) and that a tile's quads are read a unit or more
// after they are written.  tests/test_written_out_instructions.py reads both off the built code.
__device__ __forceinline__ uint32_t to_agpr(uint32_t x) {
  uint32_t r;
  asm("v_accvgpr_write_b32 %0, %1" : "=a"(r) : "v"(x));
  return r;
}

// Epilogue of one 32-row tile in 16 pieces (q, i): pair p = i % 2 of registers 4 q .. 4 q + 3 of column
// block i / 2, packed into dword 2 (q / 2) + p of quad q % 2 of the tile.  pack(q, i, v0, v1)
// returns the packed pair (after the ReLU or the mask); done(q, e) gets the four dwords e[cb][p] of q.
struct NoPiece {
  template <typename Q, typename I>
  __device__ SRF_AI void operator()(Q, I) const {}
};
template <int NB, typename Pack, typename Done>
struct TileEpi {
  f32x16 (&v)[NB];
  u32x4 (&lo)[NB];   // quad 2 T
  u32x4 (&hi)[NB];   // quad 2 T + 1
  Pack pack;
  Done done;
  uint32_t (&e)[2][2][2];  // [q % 2]: two pieces may be under way
  template <typename Q, typename I>
  __device__ SRF_AI void operator()(Q QI, I) const {
    constexpr int q = Q::value, cb = I::value >> 1, p = I::value & 1;
    if constexpr (cb < NB) {
      const uint32_t d = pack(QI, I{}, v[cb][4 * q + 2 * p], v[cb][4 * q + 2 * p + 1]);
      e[q & 1][cb][p] = d;
      (q & 1 ? hi : lo)[cb][2 * (q >> 1) + p] = to_agpr(d);
    }
    if constexpr (I::value == 3) done(QI, e[q & 1]);
  }
};

// The pieces that go with k-step i of unit u: kPieces = 1: piece (u, i) in units 0 .. 3; 2: pieces (2 u, i)
// and (2 u + 1, i) in units 0 and 1; 4: pieces (i, 0 .. 3) in unit 0.
template <int kPieces, int u, int i, typename Epi>
__device__ __forceinline__ void pieces(const Epi& epi) {
  using std::integral_constant;
  if constexpr (kPieces == 1 && u < 4) {
    epi(integral_constant<int, u>{}, integral_constant<int, i>{});
  } else if constexpr (kPieces == 2 && u < 2) {
    epi(integral_constant<int, 2 * u>{}, integral_constant<int, i>{});
    epi(integral_constant<int, 2 * u + 1>{}, integral_constant<int, i>{});
  } else if constexpr (kPieces == 4 && u == 0) {
    static_for<0, 4>([&](auto J) SRF_AI { epi(integral_constant<int, i>{}, J); });
  }
}
template <typename Epi>
__device__ __forceinline__ void all_pieces(const Epi& epi) {
  static_for<0, 4>([&](auto Q) SRF_AI { static_for<0, 4>([&](auto I) SRF_AI { epi(Q, I); }); });
}

// Stores 16-feature tile t of the wave's 64 points as the 2 KB block that the weight-gradient kernel
// reads (mlp16_dw.h): record (h, c), chunk k at byte 1024 k + 16 (32 h + c), holds features 8 k + 4 h +
// r (r = 0 .. 3, one dword each) at the lane's own points c and 32 + c.  Chunk k comes from quad k of the
// tile's pair (its k-steps 2 (t / 2) + k) in both column blocks.  One byte permutation a dword, no lane
// exchange, and each of the two stores writes 1 KB of whole lines.  Non-temporal, as store_tile's.
__device__ __forceinline__ u32x4 tile_chunk(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
  constexpr uint32_t kLo = 0x05040100, kHi = 0x07060302;  // the low / high halves of two dwords
  return u32x4{__builtin_amdgcn_perm(b0, a0, kLo), __builtin_amdgcn_perm(b0, a0, kHi),
               __builtin_amdgcn_perm(b1, a1, kLo), __builtin_amdgcn_perm(b1, a1, kHi)};
}
// Chunk k of tile t from its quads 2 (t / 2) + k.
template <int T>
__device__ __forceinline__ void store_tile16(Rsrc dst, uint32_t blk, const u32x4 (&q0)[2], const u32x4 (&q1)[2]) {
  const uint32_t rec = (threadIdx.x & 63) * 16u;
  constexpr int d = 2 * (T & 1);
  store_nt16(dst, rec, blk, tile_chunk(q0[0][d], q0[0][d + 1], q0[1][d], q0[1][d + 1]));
  store_nt16(dst, rec, blk + 1024, tile_chunk(q1[0][d], q1[0][d + 1], q1[1][d], q1[1][d + 1]));
}

// Positional encoding straight into B-operand quads (lane = point of the wave).
template <int P, int NB>
struct PeQuads {
  __device__ static SRF_AI void put(uint8_t* quads, int col, float v) {
    const int pt = (threadIdx.x & 63) % (32 * NB);
    // the point's part of the address, and the column's
    const int at_pt = (pt >> 5) * 1024 + (pt & 31) * 16;
    const int at_col = (2 * (col >> 5) + ((col >> 3) & 1)) * NB * 1024 + ((col >> 2) & 1) * 512 +
                       (((col >> 4) & 1) * 4 + (col & 3)) * 2;
    *reinterpret_cast<uint16_t*>(quads + at_pt + at_col) = (uint16_t)(pack2<P>(v, 0.f) & 0xffffu);
  }
  // features [f_lo, f_hi) of PE_L(x) at columns f - shift of the wave's quads
  __device__ static SRF_AI void write(uint8_t* quads, const float (&x)[3], int L, int f_lo, int f_hi, int shift) {
    // NB = 1: two lanes per point share its levels (NB = 2: m, and so the columns, are uniform)
    const int part = NB == 2 ? 0 : (threadIdx.x & 63) / 32, parts = 2 / NB;
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
  __shared__ __attribute__((aligned(16))) uint8_t ring[kRingUnits * kUnit];
  // computed input features of each wave's points (the trunk PE, then the view layer's [PE_xyz[trunk_pe:],
  // PE_dir]) as B-operand quads, written and read by the wave alone
  __shared__ __attribute__((aligned(16))) u32x4 pe_lds[kWaves][6][NB][64];
  __shared__ __attribute__((aligned(16))) float bias_lds[kMaxBiasFloats];
  const int lane = threadIdx.x & 63, h = lane >> 5, cl = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = blockIdx.x * kWaves + wv;
  const int p0 = wave * 32 * NB;
  const Plan& pl = a.p;
  const int ldP = a.w.ldP;
  uint8_t* quads = reinterpret_cast<uint8_t*>(&pe_lds[wv][0][0][0]);
  using PE = PeQuads<P, NB>;

  Stream16 st(a.packed + pl.fwd_off[0], ring);
  static_assert(kMaxBiasFloats % 256 == 0, "copied as whole fragments");
#pragma unroll
  for (int i = 0; i < (kMaxBiasFloats / 256 + kWaves - 1) / kWaves; ++i)
    if (i * kWaves + wv < kMaxBiasFloats / 256)
      lds_dma_1k_ahead(a.packed + pl.bias_off[0] + (i * kWaves + wv) * 1024,
                       lds_offset(bias_lds) + (i * kWaves + wv) * 1024, lane * 16);

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
  float x[3], vdir[3] = {0.f, 0.f, 0.f};
  load_xyz(x);
  if constexpr (VD) load_dir(vdir);
  PE::write(quads, x, pl.pts_deg, 0, pl.trunk_pe, 0);
  PE::pad(quads, pl.trunk_pe, 4);
  wait_vmem();
  __syncthreads();  // the first units, the biases and the PE quads

  u32x4 qa[16][NB], qb[16][NB];  // a layer's input and output quads (AGPRs), in turns
  u32x4 pe[4][NB];               // the trunk PE's
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) pe[s][cb] = pe_lds[wv][s][cb][lane];
  f32x16 acc[2][NB];      // accumulators of tile T in acc[T % 2], the other one's epilogue running
  uint32_t mbits[NB][4];  // ReLU mask: word T / 2
  uint32_t flag = 0;      // push_nonzero's
  uint32_t e[2][2][2];    // the epilogue pieces' dwords

  // biases of the tiles in the order of the products, one tile ahead
  const float* bp = bias_lds + 4 * h;
  f32x16 bias;
  auto next_bias = [&]() SRF_AI {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(bp + 8 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[4 * q + r] = b[r];
    }
    bp += 32;
  };
  next_bias();
  st.begin();

  constexpr int kSt = TRAIN ? 8 : 0;  // stores of two tiles
  using IC0 = std::integral_constant<int, 0>;
  const Rsrc rmask = uniform_rsrc(a.ws + a.w.mask);
  // The epilogue of tile T: ReLU (or not), packing, the mask from the packed pairs (both bits of pair
  // 8 (T % 2) + 2 q + p of word T / 2 at 15 minus that in the word's halves), and the tile's record.
  auto epi = [&](auto TI, auto RELU, u32x4 (&dst)[16][NB], Rsrc out) SRF_AI {
    constexpr int T = decltype(TI)::value;
    constexpr bool relu = decltype(RELU)::value;
    auto pack = [&](auto QI, auto II, float v0, float v1) SRF_AI {
      constexpr int cb = decltype(II)::value >> 1, p = decltype(II)::value & 1;
      const uint32_t d = relu ? pack2<P>(relu1(v0), relu1(v1)) : pack2<P>(v0, v1);
      if constexpr (TRAIN && relu && p == 1) {
        if constexpr (decltype(QI)::value == 0 && (T & 1) == 0) mbits[cb][T >> 1] = 0;
        push_nonzero(mbits[cb][T >> 1], flag, e[decltype(QI)::value & 1][cb][0], d);
      }
      return d;
    };
    auto done = [&, out](auto QI, const uint32_t (&d)[2][2]) SRF_AI {
      constexpr int q = decltype(QI)::value;
      if constexpr (TRAIN)
        store_nt16(out, lane * 16u, tile_block<P>(2 * T + (q >> 1), ldP, pl.elem, p0) + 1024u * (q & 1),
                   tile_chunk(d[0][0], d[0][1], d[1][0], d[1][1]));
    };
    return TileEpi<NB, decltype(pack), decltype(done)>{acc[T & 1], dst[2 * T], dst[2 * T + 1], pack, done, e};
  };
  auto out_of = [&](size_t off) SRF_AI { return uniform_rsrc(a.ws + off); };
  auto store_mask = [&](int slot) SRF_AI {
    if constexpr (TRAIN)
#pragma unroll
      for (int cb = 0; cb < NB; ++cb)
        store_nt16(rmask, lane * 16u, (uint32_t)slot * (uint32_t)ldP * 32u + (uint32_t)wave * 2048u + cb * 1024u,
                   u32x4{mbits[cb][0], mbits[cb][1], mbits[cb][2], mbits[cb][3]});
  };
  // One unit of tile accumulators ac: k-steps s0 .. s0 + n - 1 with operand quads src, pieces of the
  // previous tile's epilogue in between.
  auto unit = [&](auto UI, auto NI, auto PIECES, f32x16(&ac)[NB], auto&& src, const auto& prev) SRF_AI {
    constexpr int u = decltype(UI)::value, n = decltype(NI)::value;
    st.unit([&](auto II, const u32x4& w) SRF_AI {
      constexpr int i = decltype(II)::value;
      if constexpr (i < n) {
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) ac[cb] = mfma32x32<P>(w, src(4 * u + i, cb), u == 0 && i == 0 ? bias : ac[cb]);
        if constexpr (u == 0 && i == 0) next_bias();
      }
      pieces<decltype(PIECES)::value, u, i>(prev);
    });
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  using Yes = std::true_type;
  using No = std::false_type;
  // the four units of a 256-input tile
  auto tile = [&](auto PIECES, f32x16(&ac)[NB], const u32x4 (&src)[16][NB], const auto& prev) SRF_AI {
    static_for<0, 4>([&](auto UI) SRF_AI {
      unit(UI, I4{}, PIECES, ac, [&](int s, int cb) SRF_AI { return src[s][cb]; }, prev);
    });
  };

  // ---- layer 0: PE(trunk) -> qa
  if constexpr (TRAIN) {
    const Rsrc rx = out_of(a.w.x0);
    static_for<0, 4>([&](auto TI) SRF_AI {
      constexpr int t = decltype(TI)::value;
      store_tile16<t>(rx, tile_block<P>(t, ldP, pl.elem, p0), pe[t & ~1], pe[t | 1]);
    });
  }
  {
    const Rsrc out = out_of(a.w.h[0]);
    static_for<0, 8>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      if constexpr (T == 4) st.template sync<0>();
      auto src = [&](int s, int cb) SRF_AI { return pe[s][cb]; };
      if constexpr (T == 0) unit(IC0{}, I4{}, I4{}, acc[0], src, NoPiece{});
      else unit(IC0{}, I4{}, I4{}, acc[T & 1], src, epi(std::integral_constant<int, T - 1>{}, Yes{}, qa, out));
    });
  }
  // ---- layers 1-7: src -> dst.  The first tile finishes the previous layer's last one (whose quads its
  // last two k-steps read), which leaves out of layer l - 1 stored.
  auto layer = [&](int l, u32x4 (&src)[16][NB], u32x4 (&dst)[16][NB], auto FIVE) SRF_AI {
    const Rsrc prev = out_of(a.w.h[l - 1]), out = out_of(a.w.h[l]);
    static_for<0, 8>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      st.template sync<kSt>();
      if constexpr (T == 0) {
        tile(I2{}, acc[0], src, epi(std::integral_constant<int, 7>{}, Yes{}, src, prev));
        store_mask(l - 1);
      } else {
        tile(I1{}, acc[T & 1], src, epi(std::integral_constant<int, T - 1>{}, Yes{}, dst, out));
      }
      if constexpr (decltype(FIVE)::value)
        if (l == 5)
          unit(I4{}, I4{}, I4{}, acc[T & 1], [&](int s, int cb) SRF_AI { return pe[s & 3][cb]; }, NoPiece{});
    });
  };
#pragma unroll 1
  for (int l = 1;; l += 2) {
    layer(l, qa, qb, Yes{});
    if (l == 7) break;
    layer(l + 1, qb, qa, No{});
  }

  // ---- heads (their rows lie in the lanes h = 0)
  auto head_sigma = [&](int p, float raw) SRF_AI {
    if (a.noise) raw = raw + a.noise[p];
    a.sigma[p] = pl.softplus ? softplusf_(raw) : (raw > 0.f ? raw : 0.f);
  };
  const Rsrc out7 = out_of(a.w.h[7]);
  const auto last7 = epi(std::integral_constant<int, 7>{}, Yes{}, qb, out7);
  if constexpr (!VD) {
    // 4-channel output: sigma, rgb (src/models/SimpleNeRF17.py:735-750)
    st.template sync<kSt>();
    tile(I2{}, acc[0], qb, last7);
    store_mask(7);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n) {
        head_sigma(p, acc[0][cb][0]);
#pragma unroll
        for (int c = 0; c < 3; ++c) a.rgb[3 * p + c] = sigmoidf_(acc[0][cb][1 + c]);
      }
    }
  } else {
    // feature rows 0..255 (no activation) -> qa, then the sigma row
    const Rsrc out = out_of(a.w.f);
    static_for<0, 9>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      st.template sync<kSt>();
      if constexpr (T == 0) {
        tile(I2{}, acc[0], qb, last7);
        store_mask(7);
      } else {
        tile(I1{}, acc[T & 1], qb, epi(std::integral_constant<int, T - 1>{}, No{}, qa, out));
      }
    });
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n) head_sigma(p, acc[0][cb][0]);
    }
    // the view layer's computed inputs [PE_xyz[trunk_pe:], PE_dir]
    const int ct = pl.comp_tiles[9];  // 2, 4 or 6
    {
      const int pts_dim = 3 * (2 * pl.pts_deg + 1), n_hi = pts_dim - pl.trunk_pe;
      if (n_hi > 0) PE::write(quads, x, pl.pts_deg, pl.trunk_pe, pts_dim, pl.trunk_pe);
      PE::write(quads, vdir, pl.dir_deg, 0, pl.extra - n_hi, -n_hi);
      PE::pad(quads, pl.extra, ct);
      wave_lds_sync();
    }
    u32x4 ex[6][NB];
    static_for<0, 6>([&](auto SI) SRF_AI {
      constexpr int s = decltype(SI)::value;
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) ex[s][cb] = s < ct ? pe_lds[wv][s][cb][lane] : u32x4{0u, 0u, 0u, 0u};
    });
    if constexpr (TRAIN) {
      const Rsrc rx = out_of(a.w.ex);
      static_for<0, 6>([&](auto TI) SRF_AI {
        constexpr int t = decltype(TI)::value;
        if (t < ct) store_tile16<t>(rx, tile_block<P>(t, ldP, pl.elem, p0), ex[t & ~1], ex[t | 1]);
      });
    }
    // view layer [feature, extras] -> 128 in qb[0..7].  The fragments that pad a tile to whole units are
    // zero, and so are the extra quads they meet.
    const Rsrc outv = out_of(a.w.v);
    static_for<0, 4>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      st.template sync<0>();
      auto src = [&](int s, int cb) SRF_AI { return s < 16 ? qa[s & 15][cb] : ex[s < 16 ? 0 : s - 16][cb]; };
      auto run = [&](const auto& prev) SRF_AI {
        static_for<0, 4>([&](auto UI) SRF_AI { unit(UI, I4{}, I1{}, acc[T & 1], src, prev); });
      };
      if constexpr (T == 0) run(NoPiece{});
      else run(epi(std::integral_constant<int, T - 1>{}, Yes{}, qb, outv));
      unit(I4{}, I4{}, I1{}, acc[T & 1], src, NoPiece{});
      if (ct > 4) unit(std::integral_constant<int, 5>{}, I2{}, I1{}, acc[T & 1], src, NoPiece{});
    });
    all_pieces(epi(std::integral_constant<int, 3>{}, Yes{}, qb, outv));
    if constexpr (TRAIN) {
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) mbits[cb][2] = mbits[cb][3] = 0;
      store_mask(8);
    }
    // rgb head 128 -> 3, sigmoid
    st.template sync<0>();
    static_for<0, 2>([&](auto UI) SRF_AI {
      unit(UI, I4{}, I1{}, acc[0], [&](int s, int cb) SRF_AI { return qb[s][cb]; }, NoPiece{});
    });
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const int p = p0 + 32 * cb + cl;
      if (h == 0 && p < a.n)
#pragma unroll
        for (int c = 0; c < 3; ++c) a.rgb[3 * p + c] = sigmoidf_(acc[0][cb][c]);
    }
  }
  wait_vmem();  // the copies past the last unit
}

// ------------------------------------------------------------------- backward chain
template <int P, bool VD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mlp16_bwd_kernel(BwdArgs a) {
  constexpr int NB = 2;
  __shared__ __attribute__((aligned(16))) uint8_t ring[kRingUnits * kUnit];
  const int lane = threadIdx.x & 63, h = lane >> 5, cl = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = blockIdx.x * kWaves + wv;
  const int p0 = wave * 32 * NB;
  const Plan& pl = a.p;
  const int ldP = a.w.ldP;

  Stream16 st(a.packed + pl.bwd_off[VD ? 10 : 8], ring);
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
  wait_vmem();
  __syncthreads();
  st.begin();

  u32x4 za[16][NB], zb[16][NB];  // pre-activation gradients as B-operand quads (AGPRs), in turns
  f32x16 acc[2][NB];
  uint32_t e[2][2][2];
  uint32_t mb[NB][4];  // ReLU masks of the layer whose gradient is being computed
  uint32_t mlast[NB];  // the last word of the previous one's, for its last tile
  const Rsrc rmask = uniform_rsrc(a.ws + a.w.mask);
  auto load_masks = [&](int slot) SRF_AI {
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
          rmask, lane * 16u, (uint32_t)slot * (uint32_t)ldP * 32u + (uint32_t)wave * 2048u + cb * 1024u, 0);
#pragma unroll
      for (int k = 0; k < 4; ++k) mb[cb][k] = v[k];
    }
  };
  auto out_of = [&](int l) SRF_AI { return uniform_rsrc(a.ws + a.w.dz[l]); };
  // Epilogue of tile T: packed, masked (kMask 1: by mb, 2: by mlast, 0: not), stored as dZ tiles.
  auto epi = [&](auto TI, auto MASK, u32x4 (&dst)[16][NB], Rsrc out) SRF_AI {
    constexpr int T = decltype(TI)::value, mask = decltype(MASK)::value;
    auto pack = [&](auto QI, auto II, float v0, float v1) SRF_AI {
      constexpr int cb = decltype(II)::value >> 1, k = 8 * (T & 1) + 2 * decltype(QI)::value + (decltype(II)::value & 1);
      const uint32_t d = pack2<P>(v0, v1);
      if constexpr (mask == 1) return d & half_mask<k>(mb[cb][T >> 1]);
      else if constexpr (mask == 2) return d & half_mask<k>(mlast[cb]);
      else return d;
    };
    auto done = [&, out](auto QI, const uint32_t (&d)[2][2]) SRF_AI {
      constexpr int q = decltype(QI)::value;
      store_nt16(out, lane * 16u, tile_block<P>(2 * T + (q >> 1), ldP, pl.elem, p0) + 1024u * (q & 1),
                 tile_chunk(d[0][0], d[0][1], d[1][0], d[1][1]));
    };
    return TileEpi<NB, decltype(pack), decltype(done)>{acc[T & 1], dst[2 * T], dst[2 * T + 1], pack, done, e};
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  using I7 = std::integral_constant<int, 7>;
  using I8 = std::integral_constant<int, 8>;
  auto unit = [&](auto UI, auto NI, auto PIECES, f32x16(&ac)[NB], auto&& src, const auto& prev) SRF_AI {
    constexpr int u = decltype(UI)::value, n = decltype(NI)::value;
    st.unit([&](auto II, const u32x4& w) SRF_AI {
      constexpr int i = decltype(II)::value;
      if constexpr (i < n) {
        f32x16 zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0.f;
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) ac[cb] = mfma32x32<P>(w, src(4 * u + i, cb), u == 0 && i == 0 ? zero : ac[cb]);
      }
      pieces<decltype(PIECES)::value, u, i>(prev);
    });
  };
  auto tile = [&](auto PIECES, f32x16(&ac)[NB], const u32x4 (&src)[16][NB], const auto& prev) SRF_AI {
    static_for<0, 4>([&](auto UI) SRF_AI {
      unit(UI, I4{}, PIECES, ac, [&](int s, int cb) SRF_AI { return src[s][cb]; }, prev);
    });
  };
  // A head's gradient rows 0..3 as the one quad that holds them, and their 16-row tile t of dZ_l
  // (rows 4.. of it are zero).
  u32x4 head[NB];
  auto set_head = [&](auto rows, Rsrc out, int t) SRF_AI {
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const f32x4 v = rows(cb);
      head[cb] = h == 0 ? u32x4{pack2<P>(v[0], v[1]), pack2<P>(v[2], v[3]), 0u, 0u} : u32x4{0u, 0u, 0u, 0u};
    }
    const u32x4 none[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
    store_tile16<0>(out, tile_block<P>(t, ldP, pl.elem, p0), head, none);
  };
  // A product over one k-step (a head's quad): tile T from fragment T, the epilogue of tile T - 1 behind it.
  auto from_head = [&](auto TILES, u32x4 (&dst)[16][NB], Rsrc out) SRF_AI {
    constexpr int tiles = decltype(TILES)::value;
    static_for<0, tiles / 4>([&](auto UI) SRF_AI {
      st.unit([&](auto II, const u32x4& w) SRF_AI {
        constexpr int T = 4 * decltype(UI)::value + decltype(II)::value;
        f32x16 zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0.f;
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) acc[T & 1][cb] = mfma32x32<P>(w, head[cb], zero);
        if constexpr (T > 0) all_pieces(epi(std::integral_constant<int, T - 1>{}, I1{}, dst, out));
      });
    });
  };
  constexpr int kSt = 8;  // stores of two tiles

  if constexpr (VD) {
    // dV = W10^T dZ10, masked by the view layer's ReLU -> dZ9 (zb[0..7])
    load_masks(8);
    set_head([&](int cb) SRF_AI { return f32x4{drr[cb][0], drr[cb][1], drr[cb][2], 0.f}; }, out_of(10), 0);
    const Rsrc out9 = out_of(9), out8 = out_of(8);
    from_head(I4{}, zb, out9);
    all_pieces(epi(std::integral_constant<int, 3>{}, I1{}, zb, out9));
    // dF = W9^T dZ9 (feature part, no activation) -> dZ8 rows 0..255 (za)
    load_masks(7);
    static_for<0, 8>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      if constexpr ((T & 1) == 0) st.template sync<0>();
      static_for<0, 2>([&](auto UI) SRF_AI {
        auto src = [&](int s, int cb) SRF_AI { return zb[s][cb]; };
        if constexpr (T == 0) unit(UI, I4{}, I2{}, acc[0], src, NoPiece{});
        else unit(UI, I4{}, I2{}, acc[T & 1], src, epi(std::integral_constant<int, T - 1>{}, I0{}, za, out8));
      });
    });
    // dH7 = W8^T dZ8 (feature rows and the sigma row), masked -> dZ7 (zb)
    set_head([&](int cb) SRF_AI { return f32x4{dsr[cb], 0.f, 0.f, 0.f}; }, out8, 16);
    const Rsrc out7 = out_of(7);
    static_for<0, 8>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      st.template sync<0>();
      if constexpr (T == 0) tile(I2{}, acc[0], za, epi(I7{}, I0{}, za, out8));
      else tile(I1{}, acc[T & 1], za, epi(std::integral_constant<int, T - 1>{}, I1{}, zb, out7));
      unit(I4{}, I1{}, I4{}, acc[T & 1], [&](int, int cb) SRF_AI { return head[cb]; }, NoPiece{});
    });
  } else {
    // dH7 = W8^T dZ8 (four channels), masked -> dZ7 (zb)
    load_masks(7);
    set_head([&](int cb) SRF_AI { return f32x4{dsr[cb], drr[cb][0], drr[cb][1], drr[cb][2]}; }, out_of(8), 0);
    from_head(I8{}, zb, out_of(7));
  }
  // trunk: dH_{l-1} = W_l^T dZ_l, masked -> dZ_{l-1}
  auto layer = [&](int l, u32x4 (&src)[16][NB], u32x4 (&dst)[16][NB]) SRF_AI {
    const Rsrc prev = out_of(l), out = out_of(l - 1);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) mlast[cb] = mb[cb][3];
    load_masks(l - 1);
    static_for<0, 8>([&](auto TI) SRF_AI {
      constexpr int T = decltype(TI)::value;
      st.template sync<kSt>();
      if constexpr (T == 0) tile(I2{}, acc[0], src, epi(I7{}, I2{}, src, prev));
      else tile(I1{}, acc[T & 1], src, epi(std::integral_constant<int, T - 1>{}, I1{}, dst, out));
    });
  };
#pragma unroll 1
  for (int l = 7;; l -= 2) {
    layer(l, zb, za);
    if (l == 1) break;
    layer(l - 1, za, zb);
  }
  all_pieces(epi(I7{}, I1{}, za, out_of(0)));
  wait_vmem();  // the copies past the last unit
}

template <int P, bool VD, bool TRAIN, int NB>
int launch_fwd16(const FwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mlp16_fwd_kernel<P, VD, TRAIN, NB>), dim3(a.w.cols / (kWaves * 32 * NB)), dim3(64 * kWaves), 0, s, a);
  return launch_status();
}

// Inference of few points takes 128-point blocks while the compute units are enough for all of them: the call
// takes as long as one block then (62 us for 256 points, 42 for 128; 16,384 points).  Beyond, a block streams its
// weights for twice the points.
template <int P, bool VD>
int launch_infer16(const FwdArgs& a, hipStream_t s) {
  return a.w.cols / (kWaves * 32) <= device_compute_units() ? launch_fwd16<P, VD, false, 1>(a, s)
                                                            : launch_fwd16<P, VD, false, 2>(a, s);
}

template <int P, bool VD>
int launch_bwd16(const BwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mlp16_bwd_kernel<P, VD>), dim3(a.w.cols / (kWaves * 64)), dim3(64 * kWaves), 0, s, a);
  return launch_status();
}

}  // namespace mlp
}  // namespace srf
