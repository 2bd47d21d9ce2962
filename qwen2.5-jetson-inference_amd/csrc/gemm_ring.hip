// Prefill Linear kernels whose operands go straight from memory into an LDS
// ring (buffer_load_dwordx4 ... lds): W8A16 group-64 and BF16 GEMMs of some
// tens to a few thousand tokens, as single calls, groups (a layer's q|k|v),
// gate|up pairs with the SiLU-mul, and the q|k|v epilogue with RoPE and the
// KV-cache store.
//
// Y[m, n] = bf16(sum_k X[m, k] W[n, k] + bias[n]), the arithmetic of gemm.hip:
// stages of 64 columns (one quantisation group), v_mfma_f32_32x32x16_bf16,
// int8 weights converted exactly to BF16, the FP32 partial of a stage scaled
// once by the group scale.
//
// What bounds such a GEMM here is not MFMA: a lone 64 x 64 tile of four waves
// spends 490 (BF16) to 760 (W8A16) cycles on a stage whose MFMAs take 128,
// waiting for one thing after the other (barrier, LDS reads, MFMA chain, fold,
// LDS writes), and a CU pulls 20-40 bytes a clock from beyond its L2.  So:
//  - X and W (int8 as it is: half the LDS bytes) are loaded into LDS without
//    passing registers, NB - 1 rounds ahead, one barrier per round; W is
//    converted as its fragments are read (layouts with one wave along M for
//    W8A16, so that each weight is converted once per workgroup).
//  - KG groups of waves take a KG-th of the stages each and are summed in
//    LDS at the end: several independent chains per SIMD where a launch has
//    too few tiles for several workgroups per CU.
//  - Tiles from 64 x 32 to 128 x 64, the smallest ones where a launch would
//    leave CUs idle, and long reductions over several workgroups
//    (ring_layout).
// Measured against the 64 x 64 and skinny kernels of gemm.hip it replaces, us
// per call on weights from the memory-side cache, W8A16 / BF16: 200 tokens q
// 7.7 -> 5.2 / 6.8 -> 4.5, gate 9.9 -> 8.1 / 8.5 -> 7.8; 512 tokens q|k|v 8.2 ->
// 6.9 / 7.1 -> 5.9, gate|up 20.7 -> 17.7 / 17.4 -> 14.9; 1001 tokens gate 21.1
// -> 17.8 / 17.4 -> 14.3, o 8.4 -> 7.9 / 7.5 -> 6.3.  On weights from memory (600 MB
// of them in turn), where rounds take longer and depth counts for more: 200 tokens
// q 7.7 -> 5.5 / 6.4 -> 4.8, gate 9.4 -> 8.4 / 8.8 -> 9.2; 512 tokens gate 13.3 ->
// 12.0 / 12.9 -> 13.7; 1001 tokens q 7.9 -> 7.5 / 6.7 -> 5.8, gate 21.0 -> 18.1 /
// 20.1 -> 18.7.
//
// LDS layout.  A round's slot holds, per K group, BM rows of X and BN rows of W
// (128 bytes, 64 for int8), filled in the order the loads write them (lane l
// of a load at 16 l).  The XOR swizzle that keeps fragment reads off common
// banks is applied to the source columns: chunk c of row r is at position c ^
// ((r >> 1) & 7) (int8: c ^ ((r >> 2) & 3)), so the 16 rows one LDS cycle
// serves cover all 64 banks.  Slots are separate LDS variables and every
// index into them a constant, so the compiler's waits before a slot's reads
// do not cover the loads into the others.
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "device_common.hpp"
#include "linear_kernels.hpp"

namespace qlin {

namespace {

typedef __bf16 ring_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ring_f32x16 __attribute__((ext_vector_type(16)));
typedef float ring_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRingStageK = 64;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t ring_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes),
                                           0x00020000);
}

__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, uint4* dst, uint32_t voffset,
                                           uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16,
                                           voffset, soffset, 0, 0);
}

// 8 int8 -> 8 BF16, exact: the high halves of the integers as FP32.
__device__ __forceinline__ ring_bf16x8 cvt_i8x8(uint32_t a, uint32_t b) {
  const auto pack = [](float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
  };
  return __builtin_bit_cast(
      ring_bf16x8, make_uint4(pack(sbyte0(a), sbyte1(a)), pack(sbyte2(a), sbyte3(a)),
                              pack(sbyte0(b), sbyte1(b)), pack(sbyte2(b), sbyte3(b))));
}

// This wave's loads but the newest VM, and all its LDS reads, are done; then
// the workgroup's barrier.  After it, every wave's part of the round waited
// for is in LDS and the slot read in the round before is free.
template <int VM>
__device__ __forceinline__ void ring_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM) : "memory");
}

template <int N>
struct RingIdx {
  static constexpr int v = N;
};

template <int BM_, int BN_, int WM_, int WN_, int KG_, int NB_, bool W8_>
struct RingCfg {
  static constexpr int BM = BM_, BN = BN_;    // tile
  static constexpr int WM = WM_, WN = WN_;    // waves of a K group
  static constexpr int KG = KG_, NB = NB_;    // K groups, ring slots
  static constexpr bool W8 = W8_;
  static constexpr int WG = WM * WN, THREADS = kWave * WG * KG;
  static constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
  static constexpr int BC = W8 ? 4 : 8;  // 16-byte chunks of a W row
  static constexpr int A_CH = BM * 8, CH = A_CH + BN * BC;
  static constexpr int A_LD = A_CH / kWave / WG, B_LD = BN * BC / kWave / WG;
  static constexpr int VM = A_LD + B_LD + (W8 ? FN : 0);  // loads per wave and round
  // Epilogue: rows of FP32 (padded so that rows 4 apart differ by half the
  // banks) staged in the first slot, FPP of a wave's FM row blocks a pass.
  static constexpr int EPS = BN + 8;
  static constexpr int SLOT = KG * CH * 16;
  static constexpr int ep_bytes(int f) { return KG * WM * f * 32 * EPS * 4; }
  static constexpr int fpp() {
    int f = FM;
    while (f > 1 && ep_bytes(f) > SLOT) f /= 2;
    return f;
  }
  static constexpr int FPP = fpp();
  static constexpr int S0 = (SLOT > ep_bytes(FPP) ? SLOT : ep_bytes(FPP)) / 16;
  static constexpr int LDS = S0 * 16 + (NB - 1) * SLOT;
  static constexpr int PER_CU = 163840 / LDS > 4 ? 4 : 163840 / LDS;
  static constexpr int MIN_WAVES = PER_CU * THREADS / 256 > 4   ? 4
                                   : PER_CU * THREADS / 256 < 1 ? 1
                                                                : PER_CU * THREADS / 256;
  static_assert(A_LD * kWave * WG == A_CH && B_LD * kWave * WG == BN * BC, "whole loads");
  static_assert(LDS <= 163840, "fits a CU");
};

// One BM x BN tile at (m0, n0) (PAIR: BN / 2 columns of gate and of up from
// n0), K part `part` of d.splits.  Returns after the outputs, or in all but
// the last part to arrive after this part's partial tile.
// STAMP (timeline launches): the unit's loop and epilogue times to stamp.
template <class C, bool PAIR, bool ROPE, bool STAMP = false>
__device__ __forceinline__ void ring_tile(const GemmGroupDesc& d, int m0, int n0, int tile,
                                          int part, unsigned long long* stamp = nullptr) {
  constexpr int KG = C::KG, NB = C::NB, FM = C::FM, FN = C::FN, BM = C::BM, BN = C::BN;
  constexpr bool W8 = C::W8;
  __shared__ uint4 s0[C::S0], s1[KG * C::CH], s2[NB > 2 ? KG * C::CH : 1],
      s3[NB > 3 ? KG * C::CH : 1];
  const auto slot_at = [&](auto S) -> uint4* {
    if constexpr (decltype(S)::v == 0) return s0;
    if constexpr (decltype(S)::v == 1) return s1;
    if constexpr (decltype(S)::v == 2) return s2;
    return s3;
  };
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int kg = KG > 1 ? wave / C::WG : 0;
  const int w = KG > 1 ? wave % C::WG : wave;
  const int wm = w % C::WM, wn = w / C::WM;
  const int r = lane & 31, h = lane >> 5;
  const int k = d.k, groups = k / kRingStageK;
  const int n_rows = PAIR ? d.n / 2 : d.n;  // rows of each weight
  // this part's stages, this K group's rounds of them (one stage a round)
  const int sbeg = part * d.split_stages;
  const int scount = d.splits > 1 ? min(d.split_stages, groups - sbeg) : groups;
  const int rounds = (scount + KG - 1) / KG;
  const int mine = KG > 1 ? max(0, min(rounds, scount - kg * rounds)) : rounds;

  const __amdgpu_buffer_rsrc_t xr = ring_rsrc(d.x, static_cast<uint32_t>(d.m) * k * 2u);
  const uint32_t wbytes = static_cast<uint32_t>(n_rows) * k * (W8 ? 1u : 2u);
  const uint32_t sbytes = W8 ? static_cast<uint32_t>(n_rows) * groups * 2u : 0u;
  const __amdgpu_buffer_rsrc_t wr = ring_rsrc(d.w, wbytes);
  const __amdgpu_buffer_rsrc_t wr2 = PAIR ? ring_rsrc(d.w2, wbytes) : wr;
  // Source offsets of this lane's 16 bytes of each load: rows past M or N are
  // past the resource and read as zero.
  uint32_t xo[C::A_LD], wo[C::B_LD], so[FN];
#pragma unroll
  for (int i = 0; i < C::A_LD; ++i) {
    const int p = (w * C::A_LD + i) * kWave + lane, row = p >> 3;
    const int c = (p & 7) ^ ((row >> 1) & 7);
    xo[i] = (static_cast<uint32_t>(m0 + row) * k + c * 8) * 2u;
  }
#pragma unroll
  for (int i = 0; i < C::B_LD; ++i) {
    const int p = (w * C::B_LD + i) * kWave + lane, row = p / C::BC;
    const int c = W8 ? (p & 3) ^ ((row >> 2) & 3) : (p & 7) ^ ((row >> 1) & 7);
    const int wrow = n0 + (PAIR ? row % (BN / 2) : row);
    wo[i] = W8 ? static_cast<uint32_t>(wrow) * k + c * 16
               : (static_cast<uint32_t>(wrow) * k + c * 8) * 2u;
  }
  // PAIR: a 32-column fragment, and the rows of one load, lie in one half
  static_assert(!PAIR || (BN / 2) % 32 == 0, "whole fragments of each weight");
  __amdgpu_buffer_rsrc_t sr[FN];
#pragma unroll
  for (int fn = 0; fn < FN; ++fn) {
    const int col = wn * C::TN + fn * 32;
    const bool up = PAIR && col >= BN / 2;
    sr[fn] = ring_rsrc(up ? d.s2 : d.s, sbytes);
    so[fn] = static_cast<uint32_t>(n0 + (up ? col - BN / 2 : col) + r) * groups * 2u;
  }
  uint32_t sc[NB][FN];  // W8: the group scales of the rounds in flight
  const auto issue = [&](int t, uint4* slot, uint32_t (&xs)[FN]) {
    const uint32_t g = __builtin_amdgcn_readfirstlane(sbeg + kg * rounds + t);
    uint4* base = slot + kg * C::CH;
    if (W8) {
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        xs[fn] = __builtin_amdgcn_raw_buffer_load_b16(sr[fn], so[fn], g * 2u, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < C::A_LD; ++i) {
      load_lds16(xr, base + (w * C::A_LD + i) * kWave, xo[i], g * (kRingStageK * 2u));
    }
#pragma unroll
    for (int i = 0; i < C::B_LD; ++i) {
      const int q = w * C::B_LD + i;  // load of the tile: 64 / BC rows
      load_lds16(PAIR && q * (kWave / C::BC) >= BN / 2 ? wr2 : wr,
                 base + C::A_CH + q * kWave, wo[i], g * (W8 ? 64u : 128u));
    }
  };

  // The bias of tile column tid, before any other load so that the epilogue
  // need not wait for it (buffer loads, zero where there is none, converted
  // there: a branch or conversion here would wait here).
  const int bias_col = PAIR ? tid % (BN / 2) : tid;
  const uint32_t bias_off = tid < BN ? static_cast<uint32_t>(n0 + bias_col) * 2u : 0xFFFFFFF0u;
  const bool bias_up = PAIR && tid >= BN / 2;
  const uint32_t bias_g = __builtin_amdgcn_raw_buffer_load_b16(
      ring_rsrc(d.bias, d.bias ? n_rows * 2u : 0u), bias_up ? 0xFFFFFFF0u : bias_off, 0, 0);
  const uint32_t bias_u = PAIR ? __builtin_amdgcn_raw_buffer_load_b16(
                                     ring_rsrc(d.bias2, d.bias2 ? n_rows * 2u : 0u),
                                     bias_up ? bias_off : 0xFFFFFFF0u, 0, 0)
                               : 0u;
  // So are the (cos, sin) of the rotation pairs this thread writes.
  constexpr int ER = C::WM * C::FPP * 32;  // rows staged per pass of the epilogue
  // row of Y of staged row `row` of pass p
  const auto out_row = [&](int p, int row) {
    return m0 + (row / (32 * C::FPP)) * C::TM + p * C::FPP * 32 + row % (32 * C::FPP);
  };
  constexpr int RIT = (ER * (BN / 64) * 4 + C::THREADS - 1) / C::THREADS;  // per pass
  constexpr bool kRopeAhead = ROPE && BM == 64 && BN % 64 == 0 && RIT * (FM / C::FPP) <= 2;
  ring_f32x4 cs_ahead[kRopeAhead ? RIT * (FM / C::FPP) * 4 : 1];  // two pairs each
  const auto load_cs = [&](int pos, int c0, int j) {
    return gload(reinterpret_cast<const ring_f32x4*>(d.rope + static_cast<size_t>(pos) * 32 + c0) +
                 j);
  };
  if constexpr (kRopeAhead) {
    if (d.rope_kind == 1 || d.rope_kind == 2) {
#pragma unroll
      for (int i = 0; i < RIT * (FM / C::FPP); ++i) {
        const int it = min(i % RIT * C::THREADS + tid, ER * (BN / 64) * 4 - 1);
        const int pos = min(d.rope_start + out_row(i / RIT, it / (BN / 16)), d.max_seq - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) cs_ahead[i * 4 + j] = load_cs(pos, (it % 4) * 8, j);
      }
    }
  }
  ring_f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  // Fragment chunks: lane (r, h) feeds k-step ks with chunk 4 h + ks of its
  // row (int8: 16-byte piece 2 h + ks / 2).
  int ao[4], bo[W8 ? 2 : 4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    ao[ks] = (wm * C::TM + r) * 8 + ((4 * h + ks) ^ ((r >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < (W8 ? 2 : 4); ++i) {
    bo[i] = C::A_CH + (wn * C::TN + r) * C::BC +
            (W8 ? (2 * h + i) ^ ((r >> 2) & 3) : (4 * h + i) ^ ((r >> 1) & 7));
  }
  const auto compute = [&](const uint4* slot, const uint32_t (&xs)[FN], auto&& next) {
    const uint4* base = slot + kg * C::CH;
    uint4 fa[FM][4], fb[FN][W8 ? 2 : 4];
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
      for (int i = 0; i < (W8 ? 2 : 4); ++i) fb[fn][i] = base[bo[i] + fn * 32 * C::BC];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) fa[fm][ks] = base[ao[ks] + fm * 256];
    next();
    ring_bf16x8 b[FN][4];
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      if constexpr (W8) {
        b[fn][0] = cvt_i8x8(fb[fn][0].x, fb[fn][0].y);
        b[fn][1] = cvt_i8x8(fb[fn][0].z, fb[fn][0].w);
        b[fn][2] = cvt_i8x8(fb[fn][1].x, fb[fn][1].y);
        b[fn][3] = cvt_i8x8(fb[fn][1].z, fb[fn][1].w);
      } else {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) b[fn][ks] = __builtin_bit_cast(ring_bf16x8, fb[fn][ks]);
      }
    }
    if constexpr (W8) {
      ring_f32x16 p[FM][FN];
      const ring_f32x16 zero = {};
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            p[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(ring_bf16x8, fa[fm][ks]), b[fn][ks],
                ks == 0 ? zero : p[fm][fn], 0, 0, 0);
          }
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          const float s = bf16_to_f32(xs[fn]);
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[fm][fn][e] = fmaf(p[fm][fn][e], s, acc[fm][fn][e]);
        }
    } else {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
          for (int fn = 0; fn < FN; ++fn) {
            acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(ring_bf16x8, fa[fm][ks]), b[fn][ks], acc[fm][fn], 0, 0, 0);
          }
    }
  };
  // Round t (slot t mod NB): wait for its loads (those of the NB - 2 rounds
  // after it may stay in flight), barrier, read its fragments, issue round t +
  // NB - 1 into the slot read in round t - 1, then its MFMAs.  A K group past
  // its last stage only keeps the barriers.
  const auto step = [&](auto J, int t) {
    constexpr int j = decltype(J)::v, jn = (j + NB - 1) % NB;
    if (NB > 2 && t + NB - 2 < mine) {
      ring_wait_barrier<(NB - 2) * C::VM>();
    } else {
      ring_wait_barrier<0>();
    }
    if (STAMP && t == 0 && tid == 0) stamp[kStampLoop] = __builtin_amdgcn_s_memrealtime();
    const auto next = [&] {
      if (t + NB - 1 < mine) issue(t + NB - 1, slot_at(RingIdx<jn>{}), sc[jn]);
    };
    if (KG == 1 || t < mine) compute(slot_at(RingIdx<j>{}), sc[j], next);
  };
  if (KG == 1 || 0 < mine) issue(0, s0, sc[0]);
  if constexpr (NB > 2) {
    if (1 < mine) issue(1, s1, sc[1]);
  }
  if constexpr (NB > 3) {
    if (2 < mine) issue(2, s2, sc[2]);
  }
  // (The two loop forms measure differently per tile: whole rounds of NB
  // with a tail for the small ones, an exit after every round for 128-row
  // tiles: 128 x 64 at 1001 x 4864 x 896 BF16, 14.3 against 15.7 us.)
  if constexpr (BM == 64) {
    int t = 0;
    for (; t + NB <= rounds; t += NB) {
      step(RingIdx<0>{}, t);
      step(RingIdx<1>{}, t + 1);
      if constexpr (NB > 2) step(RingIdx<2>{}, t + 2);
      if constexpr (NB > 3) step(RingIdx<3>{}, t + 3);
    }
    if (t < rounds) step(RingIdx<0>{}, t);
    if constexpr (NB > 2) {
      if (t + 1 < rounds) step(RingIdx<1>{}, t + 1);
    }
    if constexpr (NB > 3) {
      if (t + 2 < rounds) step(RingIdx<2>{}, t + 2);
    }
  } else {
    for (int t = 0; t < rounds; t += NB) {
      step(RingIdx<0>{}, t);
      if (t + 1 >= rounds) break;
      step(RingIdx<1>{}, t + 1);
      if constexpr (NB > 2) {
        if (t + 2 >= rounds) break;
        step(RingIdx<2>{}, t + 2);
      }
      static_assert(NB <= 3, "128-row tiles have at most three slots");
    }
  }

  // ---- epilogue ----
  if (STAMP && tid == 0) stamp[kStampEpilogue] = __builtin_amdgcn_s_memrealtime();
  // Element e of a 32 x 32 fragment is row 8 (e / 4) + 4 h + e % 4, column r.
  // Staged as FP32 rows, one copy per K group, summed in group order; a
  // thread takes 8 columns of a row (PAIR: of both halves; rope: 8 rotation
  // pairs).
  float* ep = reinterpret_cast<float*>(s0);
  const auto stage = [&](int p) {
    __syncthreads();
    // (in the padding of the staged rows: column c at row c / 8)
    if (p == 0 && tid < BN) {
      ep[tid / 8 * C::EPS + BN + tid % 8] = bf16_to_f32(static_cast<uint16_t>(bias_g | bias_u));
    }
#pragma unroll
    for (int f = 0; f < C::FPP; ++f)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = (wm * C::FPP + f) * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
          ep[(kg * ER + row) * C::EPS + wn * C::TN + fn * 32 + r] = acc[p * C::FPP + f][fn][e];
        }
    __syncthreads();
  };
  // 8 columns of a staged row
  const auto staged8 = [&](int row, int col, float (&f)[8]) {
#pragma unroll
    for (int g = 0; g < KG; ++g) {
      const float* src = ep + (g * ER + row) * C::EPS + col;
      const ring_f32x4 a = *reinterpret_cast<const ring_f32x4*>(src);
      const ring_f32x4 b = *reinterpret_cast<const ring_f32x4*>(src + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[j] = g == 0 ? a[j] : f[j] + a[j];
        f[4 + j] = g == 0 ? b[j] : f[4 + j] + b[j];
      }
    }
  };
  const auto add_bias = [&](const uint16_t* bias, int col, float (&f)[8]) {
    if (!bias) return;  // (a zero added would change the sign of -0)
    const float* src = ep + col / 8 * C::EPS + BN;
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] += src[j];
  };
  const bool vec = (n_rows % 8) == 0 && (reinterpret_cast<uintptr_t>(d.y) & 15u) == 0;
  const auto write8 = [&](int m, int n, const float (&f)[8]) {
    uint16_t* dst = d.y + static_cast<size_t>(m) * n_rows + n;
    if (vec) {
      store_global16(dst, make_uint4(pack2_bf16(f[0], f[1]), pack2_bf16(f[2], f[3]),
                                     pack2_bf16(f[4], f[5]), pack2_bf16(f[6], f[7])));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (n + j < n_rows) gstore(dst + j, f32_to_bf16(f[j]));
      }
    }
  };

  if constexpr (!PAIR) {
    if (d.splits > 1) {
      // A part's FP32 tile to its place, device-coherent; the last part to
      // arrive (an agent-scope count after its own stores are complete) sums
      // all of them in part order, its own read back too.  Nothing waits on
      // another workgroup.
      // Lanes store and load consecutive 16-byte pieces: whole lines, which
      // write-through stores need (every other piece per store took three
      // times as long).
      constexpr int CPR = BN / 4;
      const __amdgpu_buffer_rsrc_t pr = coherent_rsrc(
          d.partial + static_cast<size_t>(tile) * d.splits * (BM * BN),
          static_cast<uint32_t>(d.splits) * (BM * BN * 4u));
#pragma unroll
      for (int p = 0; p < FM / C::FPP; ++p) {
        stage(p);
        for (int it = tid; it < ER * CPR; it += C::THREADS) {
          const int row = it / CPR, col = (it % CPR) * 4;
          ring_f32x4 f;
#pragma unroll
          for (int g = 0; g < KG; ++g) {
            const ring_f32x4 v =
                *reinterpret_cast<const ring_f32x4*>(ep + (g * ER + row) * C::EPS + col);
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = g == 0 ? v[j] : f[j] + v[j];
          }
          const uint32_t off = part * (BM * BN * 4u) +
                               static_cast<uint32_t>((out_row(p, row) - m0) * BN + col) * 4u;
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f), pr, off, 0,
                                                 kCoherentPolicy);
        }
      }
      __builtin_amdgcn_s_waitcnt(0);  // this thread's stores are complete
      int* last = reinterpret_cast<int*>(s0);
      __syncthreads();
      if (tid == 0) {
        *last = __hip_atomic_fetch_add(d.counters + tile, 1, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) == d.splits - 1;
      }
      __syncthreads();
      if (!*last) return;
      const bool vec4 = (n_rows % 4) == 0 && (reinterpret_cast<uintptr_t>(d.y) & 7u) == 0;
      constexpr int IT = BM * CPR / C::THREADS;  // pieces of a thread, their loads issued at once
      ring_f32x4 f[IT];
      for (int p = 0; p < d.splits; ++p) {
        ring_f32x4 v[IT];
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          v[i] = __builtin_bit_cast(
              ring_f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                              pr, p * (BM * BN * 4u) + (i * C::THREADS + tid) * 16u, 0,
                              kCoherentPolicy));
        }
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) f[i][j] = p == 0 ? v[i][j] : f[i][j] + v[i][j];
      }
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int row = (i * C::THREADS + tid) / CPR, col = (i * C::THREADS + tid) % CPR * 4;
        const int m = m0 + row, n = n0 + col;
        if (m >= d.m || n >= d.n) continue;
        if (d.bias) {
          const float* src = ep + col / 8 * C::EPS + BN + col % 8;
#pragma unroll
          for (int j = 0; j < 4; ++j) f[i][j] += src[j];
        }
        uint16_t* dst = d.y + static_cast<size_t>(m) * d.n + n;
        if (vec4) {
          store_global8(dst, make_uint2(pack2_bf16(f[i][0], f[i][1]),
                                        pack2_bf16(f[i][2], f[i][3])));
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (n + j < d.n) gstore(dst + j, f32_to_bf16(f[i][j]));
          }
        }
      }
      if (tid == 0) {  // ready for the next launch
        __hip_atomic_store(d.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      return;
    }
  }
#pragma unroll
  for (int p = 0; p < FM / C::FPP; ++p) {
    stage(p);
    if constexpr (PAIR) {
      constexpr int CPR = BN / 16;
      for (int it = tid; it < ER * CPR; it += C::THREADS) {
        const int row = it / CPR, col = (it % CPR) * 8;
        const int m = out_row(p, row), n = n0 + col;
        if (m >= d.m || n >= n_rows) continue;
        float g[8], u[8];
        staged8(row, col, g);
        staged8(row, col + BN / 2, u);
        add_bias(d.bias, col, g);
        add_bias(d.bias2, col + BN / 2, u);
#pragma unroll
        for (int j = 0; j < 8; ++j) {  // the two GEMMs' BF16 outputs
          g[j] = bf16_to_f32(f32_to_bf16(g[j]));
          u[j] = bf16_to_f32(f32_to_bf16(u[j]));
        }
        if (d.exact_silu) {
#pragma unroll
          for (int j = 0; j < 8; ++j) g[j] = silu_mul(g[j], u[j]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) g[j] = silu_mul_fast(g[j], u[j]);
        }
        write8(m, n, g);
      }
    } else if (ROPE && BN % 64 == 0 && d.rope_kind != 0) {
      // One head of 64 columns per 64 of the tile: 8 rotation pairs (c, c +
      // 32) of a row per thread, on the BF16 outputs (GemmGroupDesc).
      constexpr int IPR = BN / 64 * 4;
#pragma unroll
      for (int i = 0; i < RIT; ++i) {
        const int it = i * C::THREADS + tid;
        const int row = it / IPR, head = (it % IPR) / 4, c0 = (it % 4) * 8;
        const int m = out_row(p, row), n = n0 + head * 64, pos = d.rope_start + m;
        if (it >= ER * IPR || m >= d.m || pos >= d.max_seq || n + 64 > d.n) continue;
        float lo[8], hi[8];
        staged8(row, head * 64 + c0, lo);
        staged8(row, head * 64 + c0 + 32, hi);
        add_bias(d.bias, head * 64 + c0, lo);
        add_bias(d.bias, head * 64 + c0 + 32, hi);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          lo[j] = bf16_to_f32(f32_to_bf16(lo[j]));
          hi[j] = bf16_to_f32(f32_to_bf16(hi[j]));
        }
        if (d.rope_kind != 3) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const ring_f32x4 cs = kRopeAhead ? cs_ahead[kRopeAhead ? (p * RIT + i) * 4 + j : 0]
                                             : load_cs(pos, c0, j);
            rope_pair(lo[2 * j], hi[2 * j], make_float2(cs[0], cs[1]));
            rope_pair(lo[2 * j + 1], hi[2 * j + 1], make_float2(cs[2], cs[3]));
          }
        }
        uint16_t* dst =
            d.rope_kind == 1
                ? d.y + static_cast<size_t>(m) * d.n + n
                : d.kv_cache + (static_cast<size_t>(n / 64) * d.max_seq + pos) * 64;
        store_global16(dst + c0, make_uint4(pack2_bf16(lo[0], lo[1]), pack2_bf16(lo[2], lo[3]),
                                            pack2_bf16(lo[4], lo[5]), pack2_bf16(lo[6], lo[7])));
        store_global16(dst + 32 + c0,
                       make_uint4(pack2_bf16(hi[0], hi[1]), pack2_bf16(hi[2], hi[3]),
                                  pack2_bf16(hi[4], hi[5]), pack2_bf16(hi[6], hi[7])));
      }
    } else {
      constexpr int CPR = BN / 8;
      for (int it = tid; it < ER * CPR; it += C::THREADS) {
        const int row = it / CPR, col = (it % CPR) * 8;
        const int m = out_row(p, row), n = n0 + col;
        if (m >= d.m || n >= n_rows) continue;
        float f[8];
        staged8(row, col, f);
        add_bias(d.bias, col, f);
        write8(m, n, f);
      }
    }
  }
}

// Workgroup -> unit: workgroup b runs on XCD b mod 8, so XCD x takes the run of
// units [x per, (x + 1) per): neighbouring tiles (same W rows, M fastest, and
// a tile's parts) share that XCD's L2.  Unit u of a descriptor is part u %
// splits of tile u / splits.
__device__ __forceinline__ int ring_unit(int blocks) {
  const int per = (blocks + kXcds - 1) / kXcds;
  return static_cast<int>(blockIdx.x % kXcds) * per + static_cast<int>(blockIdx.x / kXcds);
}

template <class C, bool PAIR, bool ROPE, bool STAMP = false>
__device__ __forceinline__ void ring_run(const GemmGroupDesc& d, int u,
                                         unsigned long long* stamp = nullptr) {
  int tile = u, part = 0;
  if (!PAIR && d.splits > 1) {
    tile = u / d.splits;
    part = u % d.splits;
  }
  const int tn = tile / d.tiles_m, tm = tile - tn * d.tiles_m;
  ring_tile<C, PAIR, ROPE, STAMP>(d, tm * C::BM, tn * (PAIR ? C::BN / 2 : C::BN), tile, part,
                                  stamp);
}

// One GEMM (or pair): its descriptor alone in the kernel arguments, 0.5 to 1 us
// a launch less than choosing among kInlineGroupMax of them (512 x 896 x 896
// BF16: 6.1 -> 5.6 us).
template <class C, bool PAIR>
__global__ __launch_bounds__(C::THREADS, C::MIN_WAVES) void gemm_ring_lone_kernel(GemmGroupDesc d,
                                                                                 int blocks) {
  const int b = ring_unit(blocks);
  if (b < blocks) ring_run<C, PAIR, false>(d, b);
}

template <class C>
__global__ __launch_bounds__(C::THREADS, C::MIN_WAVES) void gemm_ring_group_kernel(RingArgs a) {
  const int b = ring_unit(a.blocks);
  if (b >= a.blocks) return;
  int lo = 0;
#pragma unroll
  for (int i = 1; i < kInlineGroupMax; ++i) {
    if (i < a.count && a.d[i].block_begin <= b) lo = i;
  }
  ring_run<C, false, true>(a.d[lo], b - a.d[lo].block_begin);
}

template <class C>
__global__ __launch_bounds__(C::THREADS, C::MIN_WAVES) void gemm_ring_table_kernel(
    const GemmGroupDesc* __restrict__ table, int count, int blocks) {
  const int b = ring_unit(blocks);
  if (b >= blocks) return;
  int lo = 0, hi = count - 1;
  while (lo < hi) {  // last descriptor whose block_begin <= b
    const int mid = (lo + hi + 1) >> 1;
    if (table[mid].block_begin <= b) lo = mid; else hi = mid - 1;
  }
  ring_run<C, false, false>(table[lo], b - table[lo].block_begin);
}

// A plan's launch with a timeline (a measurement launch): the plan's units and
// their arithmetic, with the clocks read around them.
template <class C>
__global__ __launch_bounds__(C::THREADS, C::MIN_WAVES) void gemm_ring_timeline_kernel(
    const GemmGroupDesc* __restrict__ table, int count, int blocks,
    unsigned long long* __restrict__ stamps) {
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  const unsigned long long c0 = __builtin_amdgcn_s_memtime();
  const int b = ring_unit(blocks);
  if (b >= blocks) return;
  int lo = 0, hi = count - 1;
  while (lo < hi) {  // last descriptor whose block_begin <= b
    const int mid = (lo + hi + 1) >> 1;
    if (table[mid].block_begin <= b) lo = mid; else hi = mid - 1;
  }
  const GemmGroupDesc& d = table[lo];
  const int u = b - d.block_begin, groups = d.k / kRingStageK;
  unsigned long long* stamp = stamps + static_cast<size_t>(b) * kStampSlots;
  if (threadIdx.x == 0) {
    unsigned xcc, hwid;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hwid));
    const int stages =
        d.splits > 1 ? min(d.split_stages, groups - u % d.splits * d.split_stages) : groups;
    stamp[kStampEntry] = t0;
    stamp[kStampXcc] = xcc;
    stamp[kStampHwId] = hwid;
    stamp[kStampUnit] = static_cast<unsigned long long>(b) |
                        (static_cast<unsigned long long>(stages) << 16) |
                        (static_cast<unsigned long long>(d.splits > 1) << 24);
  }
  ring_run<C, false, false, true>(d, u, stamp);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    stamp[kStampEnd] = __builtin_amdgcn_s_memrealtime();
    stamp[kStampCycles] = __builtin_amdgcn_s_memtime() - c0;
  }
}

template <bool W8>
struct RingSet;
// BF16: waves 2 x 2 (the fewest fragment bytes); W8A16: one wave along M up to
// 64 rows, so that a weight is converted once.
template <>
struct RingSet<false> {
  using Small = RingCfg<64, 32, 2, 1, 2, 4, false>;
  using SmallLong = Small;
  using Mid2 = RingCfg<64, 64, 2, 2, 2, 3, false>;
  using Mid2Long = Mid2;
  using Mid = RingCfg<64, 64, 2, 2, 1, 3, false>;
  using MidDeep = RingCfg<64, 64, 2, 2, 1, 4, false>;
  using Large = RingCfg<128, 64, 2, 2, 1, 2, false>;
  using Pair = RingCfg<64, 64, 2, 2, 2, 2, false>;
};
template <>
struct RingSet<true> {
  using Small = RingCfg<64, 32, 1, 1, 4, 2, true>;
  using SmallLong = RingCfg<64, 32, 1, 1, 4, 3, true>;
  using Mid2 = RingCfg<64, 64, 1, 2, 2, 2, true>;
  using Mid2Long = RingCfg<64, 64, 1, 2, 2, 4, true>;
  using Mid = RingCfg<64, 64, 1, 2, 1, 2, true>;
  using Large = RingCfg<128, 64, 2, 2, 1, 2, true>;
  using Pair = RingCfg<64, 64, 1, 2, 4, 2, true>;
};

template <class C, bool PAIR>
void launch_cfg(const RingArgs& a, hipStream_t stream) {
  const dim3 grid((a.blocks + kXcds - 1) / kXcds * kXcds), block(C::THREADS);
  if constexpr (!PAIR) {
    if (a.table) {
      hipLaunchKernelGGL((gemm_ring_table_kernel<C>), grid, block, 0, stream, a.table, a.count,
                         a.blocks);
      return;
    }
    if (a.count > 1) {
      hipLaunchKernelGGL((gemm_ring_group_kernel<C>), grid, block, 0, stream, a);
      return;
    }
  }
  hipLaunchKernelGGL((gemm_ring_lone_kernel<C, PAIR>), grid, block, 0, stream, a.d[0], a.blocks);
}

template <bool W8, bool PAIR>
void launch_set(const RingArgs& a, int tile, hipStream_t stream) {
  using S = RingSet<W8>;
  if constexpr (!PAIR) {
    if (tile == kRingSmall) return launch_cfg<typename S::Small, false>(a, stream);
    if (tile == kRingSmallLong) return launch_cfg<typename S::SmallLong, false>(a, stream);
  }
  if constexpr (PAIR) {
    if (tile == kRingPair) return launch_cfg<typename S::Pair, true>(a, stream);
  }
  if constexpr (!PAIR && !W8) {
    if (tile == kRingMidDeep) return launch_cfg<typename S::MidDeep, false>(a, stream);
  }
  if (tile == kRingMid2Long) return launch_cfg<typename S::Mid2Long, PAIR>(a, stream);
  if (tile == kRingMid2) return launch_cfg<typename S::Mid2, PAIR>(a, stream);
  if (tile == kRingMid) return launch_cfg<typename S::Mid, PAIR>(a, stream);
  launch_cfg<typename S::Large, PAIR>(a, stream);
}

template <class C>
void launch_cfg_timeline(const RingArgs& a, unsigned long long* stamps, hipStream_t stream) {
  const dim3 grid((a.blocks + kXcds - 1) / kXcds * kXcds), block(C::THREADS);
  hipLaunchKernelGGL((gemm_ring_timeline_kernel<C>), grid, block, 0, stream, a.table, a.count,
                     a.blocks, stamps);
}

template <bool W8>
void launch_set_timeline(const RingArgs& a, int tile, unsigned long long* stamps,
                         hipStream_t stream) {
  using S = RingSet<W8>;
  if constexpr (!W8) {
    if (tile == kRingMidDeep) {
      return launch_cfg_timeline<typename S::MidDeep>(a, stamps, stream);
    }
  }
  switch (tile) {
    case kRingSmall: return launch_cfg_timeline<typename S::Small>(a, stamps, stream);
    case kRingSmallLong: return launch_cfg_timeline<typename S::SmallLong>(a, stamps, stream);
    case kRingMid2: return launch_cfg_timeline<typename S::Mid2>(a, stamps, stream);
    case kRingMid2Long: return launch_cfg_timeline<typename S::Mid2Long>(a, stamps, stream);
    case kRingMid: return launch_cfg_timeline<typename S::Mid>(a, stamps, stream);
    default: return launch_cfg_timeline<typename S::Large>(a, stamps, stream);
  }
}

int ring_rows(int tile) { return tile == kRingLarge ? 128 : 64; }
int ring_cols(int tile) { return tile <= kRingSmallLong ? 32 : 64; }

// Workgroups of the tile's kernel that share a CU (its LDS).
int ring_per_cu(bool w8, int tile) {
  switch (tile) {
    case kRingSmall: return w8 ? RingSet<true>::Small::PER_CU : RingSet<false>::Small::PER_CU;
    case kRingSmallLong:
      return w8 ? RingSet<true>::SmallLong::PER_CU : RingSet<false>::SmallLong::PER_CU;
    case kRingMid2Long:
      return w8 ? RingSet<true>::Mid2Long::PER_CU : RingSet<false>::Mid2Long::PER_CU;
    case kRingMid2: return w8 ? RingSet<true>::Mid2::PER_CU : RingSet<false>::Mid2::PER_CU;
    case kRingPair: return w8 ? RingSet<true>::Pair::PER_CU : RingSet<false>::Pair::PER_CU;
    case kRingMidDeep: return RingSet<false>::MidDeep::PER_CU;
    case kRingMid: return w8 ? RingSet<true>::Mid::PER_CU : RingSet<false>::Mid::PER_CU;
    default: return w8 ? RingSet<true>::Large::PER_CU : RingSet<false>::Large::PER_CU;
  }
}

}  // namespace

int ring_layout(bool w8, GemmGroupDesc* d, int count, int cus, bool heads, bool may_split,
                int* blocks_out, size_t* partial_floats, size_t* counters) {
  const bool pair = d[0].w2 != nullptr;
  long long t64 = 0, t32 = 0;
  int min_stages = 1 << 30, max_stages = 0;
  for (int i = 0; i < count; ++i) {
    const long long tm = (d[i].m + 63) / 64;
    t32 += tm * ((d[i].n + 31) / 32);
    t64 += tm * ((d[i].n + 63) / 64);
    min_stages = std::min(min_stages, d[i].k / kRingStageK);
    max_stages = std::max(max_stages, d[i].k / kRingStageK);
  }
  const bool small_ok = !pair && !heads, long_k = max_stages > 16;
  // (A lone int8 GEMM of more tiles than CUs is bound by the loads of each CU,
  // not by the length of a unit: 800 x 1536 x 8960 whole 50.0 us, in two parts 54.9.)
  const bool split_ok = may_split && small_ok && long_k && !(w8 && count == 1 && t64 > cus);
  // The launch's length on `tile` with parts of t stages, in stages of a
  // unit: rounds of workgroups (whole ones where the units are equal) times
  // the stages of a unit, to which a hand-off adds the time of about 14 stages
  // and 3 per part (some 3.5 us at two parts; without it 700 x 1536 x 8960
  // BF16 takes two rounds of parts, 50 against 40 us).
  const auto length = [&](int tile, int t) {
    const int bm = ring_rows(tile), bn = ring_cols(tile);
    long long units = 0;
    for (int i = 0; i < count; ++i) {
      const int stages = d[i].k / kRingStageK;
      units += static_cast<long long>((d[i].m + bm - 1) / bm) * ((d[i].n + bn - 1) / bn) *
               ((stages + t - 1) / t);
    }
    const double rounds =
        static_cast<double>(units) / (static_cast<double>(ring_per_cu(w8, tile)) * cus);
    const int parts = (max_stages + t - 1) / t;
    return (min_stages == max_stages ? std::ceil(rounds) : std::max(1.0, rounds)) *
           (t + (parts > 1 ? 14.0 + 3.0 * parts : 0.0));
  };
  const auto split_tiles = [&](int tile, int t) {
    const int bm = ring_rows(tile), bn = ring_cols(tile);
    long long tiles = 0;
    for (int i = 0; i < count; ++i) {
      if (d[i].k / kRingStageK <= t) continue;
      tiles += static_cast<long long>((d[i].m + bm - 1) / bm) * ((d[i].n + bn - 1) / bn);
    }
    return tiles;
  };
  // The best part length on `tile`; *len receives its launch length.
  const auto best_part = [&](int tile, double* len) {
    int target = max_stages;
    *len = length(tile, target);
    for (int parts = 2; split_ok && parts <= kRingMaxParts; ++parts) {
      const int t = (max_stages + parts - 1) / parts;
      if (t < 8 || (min_stages < max_stages && t < min_stages)) break;
      if (split_tiles(tile, t) > kRingMaxSplitTiles) continue;
      const double l = length(tile, t);
      // (equal lengths: an int8 row of tiles in more parts, 32 x 896 x 4864 in 4 / 5
      // 8.6, 8.9 / 8.4, 8.7 on weights from memory, cached)
      if (l < *len || (l == *len && w8 && count == 1 && d[0].m <= 64)) {
        *len = l;
        target = t;
      }
    }
    return target;
  };
  // The smallest tile that does not need more than a round of workgroups;
  // us per call (64 x 32 / 64 x 64 with two K groups / 64 x 64 / 128 x 64), BF16:
  // 200 x 1152 x 896 (144 tiles of 64 x 32) 4.6 / 5.7 / -, 1001 x 896 x 896 (224
  // of 64 x 64) - / 6.2 / 7.4, 512 x 4864 x 896 (608) - / 12.0 / 10.3 / 11.0, 1001
  // x 4864 x 896 (1216) - / 20.6 / 15.7 / 14.3; W8A16: 512 x 1152 x 896 (288 of
  // 64 x 32) 6.8 / 7.4, 300 x 4864 x 896 (380 of 64 x 64) - / 8.5 / 9.8, 512 x 4864
  // x 896 (608) - / 11.1 / 11.5, 1001 x 4864 x 896 (1216) - / 17.7 / 17.8 / 18.0,
  // 2000 x 4864 x 896 (2432) - / 34.5 / 32.5 / 31.3.
  int tile, target, fixed = 0;  // fixed: part length, 0: best_part's
  double len = 0.0;
  if (pair) {
    // The two GEMMs' values are those of their own whole calls on the ring (not of
    // those the skinny kernel takes: few rows, K over 1024): the stages summed in
    // the same K groups (W8A16: four in 64 x 32 tiles).  Over a BF16
    // pair per CU, two slots instead of three, so that two workgroups share a
    // CU: 32 x 17920 x 1536 (280 tiles) 17.9 -> 13.4 us, 32 x 9728 x 896 (152) 6.4 with
    // three, 8.1 with two.
    GemmGroupDesc half = d[0];
    half.w2 = nullptr;
    half.n /= 2;
    int b = 0;
    size_t pf = 0, cc = 0;
    const int lone = ring_layout(w8, &half, 1, cus, false, false, &b, &pf, &cc);
    if (lone <= kRingMid2Long) {
      tile = (w8 ? lone <= kRingSmallLong : t64 > cus) ? kRingPair : kRingMid2;
    } else {
      tile = (w8 ? t64 <= 5 * cus : t64 <= 3 * cus) ? kRingMid : kRingLarge;
    }
  } else if (!long_k && small_ok && t32 <= cus) {
    tile = kRingSmall;
  } else if (long_k && small_ok && t64 <= cus) {
    // One workgroup per CU, of either tile, whichever gives the shorter
    // launch (200 x 1536 x 8960 BF16, 64 x 32 whole / 64 x 64 in two parts: 25.2 /
    // 18.8 us; 40 x 1536 x 8960, 5 parts / 10 parts: 11.6 / 13.0).
    double mid = 0.0;
    best_part(kRingSmallLong, &len);
    best_part(kRingMid2Long, &mid);
    // (An int8 row of tiles is bound by its weights: 64 x 64 saves no loads there; 2
    // x 4096 x 4096 in 2 narrow / 4 wide parts 10.3 / 11.5, 64 rows 10.2 / 11.2.)
    const double lead = w8 && count == 1 && d[0].m <= 64 ? 1.25 : 1.05;
    tile = len <= lead * mid ? kRingSmallLong : kRingMid2Long;
    // Of equal lengths the wider tile where X is most of the loads (two or more
    // tiles of rows to one of columns), its rows a multiple of 1 KB apart (they
    // share few L2 channels) and the narrow tile, which reads X twice as often,
    // nearly fills the CUs: 2000 x 256 x 1536 BF16 10.2 -> 7.0 us, W8A16 11.1 -> 9.8;
    // but 1200 x 256 x 1536 (152 narrow tiles) 6.1 / 7.2, 1500 x 320 x 1536 W8A16 (240)
    // 8.9 / 9.8, 2500 x 192 x 1088 5.7 / 6.0, 1001 x 512 x 2048 (as many of rows as of
    // columns) 7.3 / 8.9.
    if (len == mid && count == 1 && d[0].k % 512 == 0 &&
        (d[0].m + 63) / 64 >= 2 * ((d[0].n + 31) / 32) && 16 * t32 > (w8 ? 15 : 10) * cus) {
      tile = kRingMid2Long;
    }
    // A lone int8 one with a workgroup for a third of the CUs or more in as many
    // parts as give two workgroups per CU (their rounds share a CU's loads well, a
    // third one's no more: 600 x 896 x 4864, 140 tiles, us in 2 / 3 / 4 / 6 parts 19.1 /
    // 16.7 / 20.6 / 22.2, 512 tokens 19.0 / 16.2 / 14.8 / 18.2), three where a part
    // would be over 40 stages, whose rounds of loads a third one hides (512 x 1536 x
    // 8960, weights from memory, in 2 / 4 parts 48.3 / 38.1).  Up to five sixths of
    // the CUs, or all of them if two parts are enough: 1001 x 896 x 4864 (224) whole
    // 24.3, in two 22.4.  Up to 40 stages the launch's length decides.
    const bool lone_w8 = w8 && count == 1 && split_ok && 3 * t64 > cus;
    const int two = static_cast<int>(2 * cus / t64);
    const bool whole = max_stages <= 40 * two;  // parts of up to 40 stages
    if (lone_w8 && (6 * t64 <= 5 * cus || (whole && max_stages >= 40))) {
      tile = kRingMid2;
      const int parts = whole ? two : static_cast<int>(3 * cus / t64);
      if (max_stages >= 40) fixed = (max_stages + parts - 1) / parts;
    }
    // An int8 group mostly of short GEMMs: two workgroups per CU (a layer's seven
    // at 2 to 64 tokens 12.3-12.9 -> 10.8-11.7 us), where that is about one round of
    // them: a unit's stages and at most the hand-offs of the most parts, 14 + 3 x 15.
    if (w8 && min_stages <= 16) {
      const int t = best_part(kRingSmall, &len);
      if (len < t + 60) tile = kRingSmall;
    }
  } else if (t64 <= (w8 ? 2 : 1) * cus) {
    tile = kRingMid2;
  } else if (!w8 && t64 <= 2 * cus && (max_stages > 64 || (count == 1 && d[0].m < d[0].n)) &&
             best_part(kRingMid, &len) == max_stages) {
    // Whole reductions of up to two workgroups per CU: a fourth slot, two rounds in
    // flight behind the one awaited.  Weights from memory / from the memory-side
    // cache, us, three slots / four / the 64 x 64 register tile: 65 x 8960 x 1536
    // 15.7, 10.3 / 13.9, 10.1 / 13.8, 12.5; 700 x 1536 x 8960 69.1, 50.2 / 54.8, 39.6 /
    // 56.9, 50.8; 512 x 4096 x 4096 38.7, 27.0 / 35.8, 26.9 / 33.5, 28.8; 256 x 4864 x 896
    // 11.3, 7.0 / 10.8, 7.2 / 9.1, 8.2; but, more rows than columns, 1200 x 896 x 896 7.7,
    // 6.9 / 7.4, 7.4 and 2500 x 512 x 2048 16.2, 16.7 / 17.6, 18.1.  (The
    // register tile's lead on weights from memory, 14.4 against 17.7 at 128 x 8960 x
    // 1536, is its order of tiles, neighbouring columns on different XCDs, with
    // which the ring takes 15.0 there and 14.9 instead of 10.6 on cached weights.)
    tile = kRingMidDeep;
  } else if (w8 ? t64 <= 5 * cus : t64 <= 3 * cus) {
    tile = kRingMid;
  } else {
    tile = kRingLarge;
  }
  target = fixed ? fixed : best_part(tile, &len);
  const int bm = ring_rows(tile), bn = ring_cols(tile);
  for (int i = 0; i < count; ++i) {
    d[i].tiles_m = (d[i].m + bm - 1) / bm;
    d[i].splits = 1;
    d[i].split_stages = d[i].k / kRingStageK;
    d[i].partial = nullptr;
    d[i].counters = nullptr;
  }
  size_t pf = 0, cc = 0;
  for (int i = 0; i < count; ++i) {
    const int s = d[i].k / kRingStageK, parts = (s + target - 1) / target;
    if (parts <= 1) continue;
    d[i].split_stages = (s + parts - 1) / parts;
    d[i].splits = (s + d[i].split_stages - 1) / d[i].split_stages;  // no empty part
    const size_t tiles = static_cast<size_t>(d[i].tiles_m) * ((d[i].n + bn - 1) / bn);
    pf += tiles * d[i].splits * bm * bn;
    cc += tiles;
  }
  std::stable_sort(d, d + count, [](const GemmGroupDesc& a, const GemmGroupDesc& b) {
    return a.split_stages > b.split_stages;  // longest units first
  });
  long long blocks = 0;
  const int bn_out = pair ? bn / 2 : bn;
  for (int i = 0; i < count; ++i) {
    d[i].block_begin = static_cast<int>(blocks);
    const int n = pair ? d[i].n / 2 : d[i].n;
    blocks += static_cast<long long>(d[i].tiles_m) * ((n + bn_out - 1) / bn_out) * d[i].splits;
  }
  *blocks_out = blocks > 0x7FFFFFF0 ? -1 : static_cast<int>(blocks);
  *partial_floats = pf;
  *counters = cc;
  return tile;
}

void ring_bind(GemmGroupDesc* d, int count, int tile, float* partial, int* counters) {
  const int bm = ring_rows(tile), bn = ring_cols(tile);
  for (int i = 0; i < count; ++i) {
    if (d[i].splits <= 1) continue;
    const size_t tiles = static_cast<size_t>(d[i].tiles_m) * ((d[i].n + bn - 1) / bn);
    d[i].partial = partial;
    d[i].counters = counters;
    partial += tiles * d[i].splits * bm * bn;
    counters += tiles;
  }
}

void launch_gemm_ring(bool w8, const RingArgs& a, int tile, hipStream_t stream) {
  const bool pair = !a.table && a.d[0].w2 != nullptr;
  if (w8) {
    pair ? launch_set<true, true>(a, tile, stream) : launch_set<true, false>(a, tile, stream);
  } else {
    pair ? launch_set<false, true>(a, tile, stream) : launch_set<false, false>(a, tile, stream);
  }
}

void launch_gemm_ring_timeline(bool w8, const RingArgs& a, int tile, unsigned long long* stamps,
                               hipStream_t stream) {
  if (w8) {
    launch_set_timeline<true>(a, tile, stamps, stream);
  } else {
    launch_set_timeline<false>(a, tile, stamps, stream);
  }
}

void launch_gemm_lone(bool w8, const GemmArgs& g, int cus, hipStream_t stream) {
  // BF16, long K whole, between 11/8 and two 64 x 64 tiles per CU: the register
  // tile; us, weights from memory / cached, against four ring slots: 1001 x 1536 x
  // 8960 58.3, 52.2 / 70.4, 56.9, 1200 60.5, 54.7 / 65.8, 56.8, 2000 x 896 x 4864 34.7,
  // 33.6 / 36.4, 33.6; but 850 x 1536 x 8960 (336 tiles) 57.7, 51.8 / 54.9, 41.7, 400 x
  // 4096 x 4096 29.9, 26.2 / 31.5, 24.0.
  const long long t64 = static_cast<long long>((g.m + 63) / 64) * ((g.n + 63) / 64);
  if (!w8 && g.k > 4096 && 8 * t64 > 11 * cus && t64 <= 2 * cus) {
    return launch_gemm_mfma(kGemmTile64x64, w8, g, stream);
  }
  if (!gemm_wide_preferred(w8, g.m, g.n, g.k, cus)) {
    RingArgs a{};
    a.d[0] = GemmGroupDesc{g.w, g.s, g.bias, g.x, g.y, g.m, g.n, g.k, 0, 0, 1, g.k / kRingStageK,
                           nullptr, nullptr};
    a.count = 1;
    size_t pf = 0, cc = 0;
    const int tile = ring_layout(w8, a.d, 1, cus, false, false, &a.blocks, &pf, &cc);
    if (a.blocks > 0) return launch_gemm_ring(w8, a, tile, stream);
  }
  launch_gemm_mfma(kGemmTile256x128, w8, g, stream);
}

}  // namespace qlin
