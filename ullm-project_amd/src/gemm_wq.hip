// gemm_wq.hip -- products of more than 16 rows with exact (bf16) activations
// on gfx950: batched decode and prefill of FP8-E4M3 and AQ4 g128 weights.
//
// Y[m, n] = alpha * sum_k dequant(W)[n, k] * x[m, k], fp32 accumulation, from
// the wave tiles of layout.hpp.  The decode kernels (gemv.hip) read every
// weight once per 32 rows; here a weight byte is read from memory once and
// unpacked in registers for all the rows of a block, so the product becomes
// bound by v_mfma_f32_16x16x32_bf16 at many rows and by the copies of x into
// LDS (about 50 KB per microsecond and CU) at few.
//
// Two kernels, one choice (plan_wq_gemm):
//   * wq_gemm_kernel: blocks of 32..128 rows x 128..384 columns, 8 waves
//     tiling the block, x staged in LDS for all of them.  MI355X, K = 4096,
//     M = 2048, N = 28672: AQ4 1060 -> 447 us (1.08 PFLOP/s), FP8 1350 -> 433
//     us (1.11 PFLOP/s); a plain bf16 GEMM of that size, weights already
//     bf16, takes 407 us in the vendor's library.
//   * wq_strip_kernel: blocks of 16..64 rows x 32..96 columns, the waves
//     splitting K, each with an LDS ring of its own and no barrier before the
//     final reduction, where a grid of large blocks would leave CUs idle or a
//     block's few MFMAs would not cover its barriers.  M = 96, N = 6144: AQ4
//     19.1 -> 13.2 us, FP8 42 -> 14 us (weights from HBM).
//
// AQ4 uses sum_k (q - z) s x = s * sum_k (16 + q) x - s (16 + z) sum_k x per
// 128-k group: 16 + q is exact in bf16 (a nibble in mantissa bits 3..6) and
// the offset is an eighth of the decode kernels' 128, which makes the
// cancelling parts smaller: relative error against 64-bit sums 5e-7 (the
// 8-wave blocks) and 2e-7 (the strips) against the decode kernels' 1.8e-6.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace ullm {
namespace {

// Block configuration.  WM x WN waves of TM x TN 16 x 16 tiles; a k-step is
// 128 k.  STAGES LDS stages of x, BD steps of weights in flight in registers,
// a barrier every SPB steps.  WK = 2: two such groups of waves take the even
// and the odd steps.
template <uint32_t TM_, uint32_t TN_, uint32_t WM_, uint32_t WN_, uint32_t STAGES_,
          uint32_t BD_ = 1, uint32_t SPB_ = 1, uint32_t WK_ = 1>
struct WqCfg {
  static constexpr uint32_t SPB = SPB_, WK = WK_;
  static constexpr uint32_t G = SPB * WK;  // k-steps between barriers
  static_assert(STAGES_ % G == 0 && STAGES_ / G >= 2 && 4 % SPB == 0, "stages");
  static_assert(WK == 1 || (WK == 2 && TM_ % 2 == 0), "K groups");
  static constexpr uint32_t TM = TM_, TN = TN_, WM = WM_, WN = WN_, STAGES = STAGES_;
  static constexpr uint32_t BD = BD_;
  static constexpr uint32_t WAVES = WM * WN * WK;
  static constexpr uint32_t BM = TM * WM * 16, BN = TN * WN * 16;
  static constexpr uint32_t A_BYTES = BM * 256;  // 128 k of every row
  // AQ4 activation sums: two sets of four groups for every row (and WK).
  static constexpr uint32_t XS_BYTES = WK * 2 * BM * 16;
  static constexpr uint32_t COPIES = BM / (4 * WAVES);
  static_assert(BM % (4 * WAVES) == 0 && WAVES % 4 == 0, "copy split");
  // Row pitch (bf16 elements) of a wave's epilogue chunk: 16 bytes of padding
  // put the rows of one LDS store in different banks.
  static constexpr uint32_t OUT_STRIDE = TN * 16 + 8;
  static constexpr uint32_t CHUNK_BYTES = 16 * OUT_STRIDE * 2;
  static constexpr uint32_t MAIN_BYTES =
      STAGES * A_BYTES > WAVES * CHUNK_BYTES ? STAGES * A_BYTES : WAVES * CHUNK_BYTES;
  static constexpr uint32_t LDS = MAIN_BYTES + XS_BYTES;
  static_assert(LDS <= 160 * 1024, "gfx950 LDS per workgroup");
};

// Workgroup barrier that waits for this wave's LDS accesses only: copies and
// weight loads stay in flight (the caller waits for those it needs).
__device__ __forceinline__ void wq_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int N>
__device__ __forceinline__ void wq_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xf) | ((N >> 4) << 14) | (0x7 << 4) | (0xf << 8));
}

// Eight 4-bit codes in one dword -> eight bf16 holding 16 + q: each nibble
// lands in mantissa bits 3..6 of bf16 16.0.
__device__ __forceinline__ bf16x8 nib8_to_bf16_off16(uint32_t w, uint32_t mask,
                                                     uint32_t magic) {
  return __builtin_bit_cast(
      bf16x8, u32x4{((w << 3) & mask) | magic, ((w >> 1) & mask) | magic,
                    ((w >> 5) & mask) | magic, ((w >> 9) & mask) | magic});
}

// An FP8 wave tile's 16 bytes of a lane -> its two MFMA operands.
__device__ __forceinline__ void fp8_tile_operands(u32x4 w, bf16x8 &b0, bf16x8 &b1) {
  const u32x2 b01 = e4m3x4_to_bf16x4(w.x), b23 = e4m3x4_to_bf16x4(w.y);
  const u32x2 b45 = e4m3x4_to_bf16x4(w.z), b67 = e4m3x4_to_bf16x4(w.w);
  b0 = __builtin_bit_cast(bf16x8, u32x4{b01.x, b01.y, b23.x, b23.y});
  b1 = __builtin_bit_cast(bf16x8, u32x4{b45.x, b45.y, b67.x, b67.y});
}

// 16 bytes per lane from a buffer into LDS at the wave's base.
__device__ __forceinline__ void wq_dma16(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff,
                                         uint32_t soff, void *lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rsrc, (__attribute__((address_space(3))) void *)(lds_wave_base), 16, voff, soff, 0, 0);
}

// Dispatch order -> tile: workgroups go round-robin over the 8 XCDs, so each
// XCD gets one contiguous range of tiles (rows fastest) and the workgroups
// that share an L2 share weights.
__device__ __forceinline__ uint32_t wq_tile() {
  const uint32_t total = gridDim.x, xcd = blockIdx.x % 8;
  return xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
}

// 8-wave blocks.  Per k-step a block copies BM rows x 256 bytes of x into LDS
// (direct loads, whole 256-byte row segments, the 16-byte chunk c of row r at
// slot c ^ (r % 16), so the 16 rows of an MFMA operand read hit 16 bank
// groups), each wave loads its own TN weight tiles straight into registers,
// unpacks them once and contracts them with its TM row tiles.
//
// What bounds a step is the sum of its parts more than the largest: with the
// copies taken out (timing only) the 256 x 192 block of two waves by four took
// 434 of 504 us (M = 2048, N = 28672, AQ4), with the MFMAs taken out 206.  A
// step costs each wave 4 TM TN MFMAs, an unpack of 32 (AQ4) or 16 (FP8) VALU
// instructions per weight tile, 4 per product tile, and TM 4 KiB operand
// reads.  All waves side by side over the columns (WM = 1) unpack every weight
// once per block instead of once per WM: 128 x 256 blocks, 2 x 4 waves of
// 64 x 64 against 1 x 8 of 128 x 32: FP8 2.01 -> 1.57 us per step, AQ4 1.87 ->
// 1.79.  128 x 384 leaves the matrix cores the largest share (AQ4 447 us
// against 475 in 128 x 256).  64 x 128 blocks of one K group
// read x from LDS as long as they contract it (16 columns per wave); with two
// groups of four waves on alternating steps the reads halve (WK = 2: AQ4 M =
// 512 14336 -> 4096 87 -> 75 us), at the price of an exchange at the end.
//
// Every step's products start from zero and are added to the fp32 accumulators
// per tile: AQ4 needs that for the group scale (one multiply-add per element).
// FP8 adds them up in two levels, four steps and then these sums, which keeps
// the error below the decode kernels' (relative, against 64-bit sums; decode
// kernels / one level / two, K = 4096 9.0e-8 / 1.15e-7 / 7.9e-8, K = 14336
// 1.45e-7 / 1.98e-7 / 1.14e-7) in the same time (128 x 256 and 64 x 128 within
// 3 %): the first step of four starts the sum, so a round makes as many
// additions as before.  The second set of sums fits 128 x 256 blocks (228
// registers); in 128 x 384 ones it spills 253, so FP8 does without them (M =
// 2048 N = 28672 433 us against 414, M = 1463 N = 7214 K = 6848, one round
// there and two here, 186 against 131).
//
// AQ4's sum_k x per (row, group): each of the WN waves that share a row tile
// takes every WN-th one, sums it by an MFMA against ones and leaves it in
// LDS; after four groups one MFMA per tile subtracts their s (16 + z) sum_k x
// from the accumulators, both factors split three ways into bf16 (correct()).
// As a multiply-add per element and group the same subtraction took as many
// VALU slots as the scaling itself.
template <bool AQ4, class C, int EPI>
__global__ __launch_bounds__(C::WAVES *kWave) void wq_gemm_kernel(GemvArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t wk = wave / (C::WM * C::WN);  // 0 unless WK = 2
  const uint32_t wm = wave / C::WN % C::WM, wn = wave % C::WN;
  const uint32_t stripes = a.n16 / 16;
  const uint32_t mblocks = (a.m + C::BM - 1) / C::BM;
  const uint32_t tile = wq_tile();
  const uint32_t m0 = (tile % mblocks) * C::BM;
  const uint32_t T0 = (tile / mblocks) * (C::BN / 16) + wn * C::TN;

  // Rows past M lie outside the buffer and read zeros; so do the look-ahead
  // copies past the last row's end (past an inner row's they read what
  // follows it, into a stage that no step reads).
  const uint32_t rows = min(C::BM, a.m - m0);
  const __amdgpu_buffer_rsrc_t abuf = byte_buffer(
      a.x + uint64_t(m0) * a.ldx, uint32_t(((rows - 1) * a.ldx + a.k) * 2));
  const uint32_t ldb = uint32_t(a.ldx) * 2;
  const uint32_t crow = wave * 4 + lane / 16;
  const uint32_t avoff = crow * ldb + ((lane % 16) ^ (crow % 16)) * 16;
  auto copy_a = [&](uint32_t g, char *st) {
#pragma unroll
    for (uint32_t i = 0; i < C::COPIES; ++i) {
      wq_dma16(abuf, avoff, g * 256 + i * (C::WAVES * 4) * ldb,
               st + (i * C::WAVES + wave) * 1024);
    }
  };

  // Stripes past N read zeros.
  const uint32_t units = a.units;
  const uint32_t Tb = min(T0, stripes - 1);
  const uint32_t nT = T0 < stripes ? min(C::TN, stripes - T0) : 0u;
  const __amdgpu_buffer_rsrc_t wbuf = byte_buffer(
      static_cast<const uint8_t *>(a.tiles) + uint64_t(Tb) * units * 1024,
      nT * units * 1024);
  const __amdgpu_buffer_rsrc_t zbuf =
      byte_buffer(static_cast<const uint32_t *>(a.aux) + uint64_t(Tb) * units * 16,
                  AQ4 ? nT * units * 64 : 0u);
  const uint32_t wlane = lane * 16;
  constexpr uint32_t U = AQ4 ? 1 : 2;  // weight tiles of one 128-k step
  const uint32_t steps = (units + U - 1) / U;

  u32x4 raw[C::BD][C::TN][U];
  auto load_b = [&](u32x4 (&w)[C::TN][U], uint32_t g) {
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        w[j][u] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       wbuf, wlane, (j * units + g * U + u) * 1024, 0));
      }
    }
  };
  // Step u of this wave is k-step u WK + wk.
  auto kstep = [&](uint32_t u) { return u * C::WK + wk; };
  // AQ4 scale|zero words of four of its groups: lane l holds step u0 + l / 16.
  uint32_t zc[C::TN], zn[C::TN];
  auto load_z = [&](uint32_t u0) {
    if constexpr (AQ4) {
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        zn[j] = __builtin_amdgcn_raw_buffer_load_b32(
            zbuf, lane % 16 * 4 + lane / 16 * (C::WK * 64), (j * units + kstep(u0)) * 64, 0);
      }
    }
  };

  f32x4 acc[C::TM][C::TN];
#pragma unroll
  for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  float *xsb = reinterpret_cast<float *>(lds + C::MAIN_BYTES) + wk * (2 * C::BM * 4);
  load_z(0);
#pragma unroll
  for (uint32_t d = 0; d < C::BD; ++d) {
    load_b(raw[d], kstep(d));
  }
#pragma unroll
  for (uint32_t t = 0; t + C::G < C::STAGES; ++t) {
    copy_a(t, lds + t * C::A_BYTES);
  }
  const uint32_t nmask = opaque_u32(0x00780078u);
  const uint32_t nmagic = opaque_u32(0x41804180u);
  const bf16x8 ones = __builtin_bit_cast(
      bf16x8, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  // Lane's A row and swizzle; the operand's 16-byte chunk c of the row sits
  // at slot c ^ (row % 16).
  const uint32_t arow = (wm * C::TM * 16 + lane % 16) * 256;
  const uint32_t q4 = lane / 16, sw = lane % 16;
  auto a_operand = [&](const char *st, uint32_t i, uint32_t q) {
    const uint32_t c = AQ4 ? 4 * q + q4 : 8 * (q / 2) + 2 * q4 + q % 2;
    return *reinterpret_cast<const bf16x8 *>(st + arow + i * 4096 + ((c ^ sw) * 16));
  };
  // acc -= sum over the groups of steps u0 .. u0 + 3 of (s (16 + z))[n] *
  // xs[m], as one MFMA per tile: k-slots 8 q4 .. + 7 carry step u0 + q4's
  // products of the three-way bf16 splits of both factors.
  auto split3 = [&](float v, float (&o)[3]) {
    o[0] = bits_f32(f32_bits(static_cast<float>(static_cast<__bf16>(v))));
    o[1] = static_cast<float>(static_cast<__bf16>(v - o[0]));
    o[2] = v - o[0] - o[1];
  };
  auto correct = [&](uint32_t u0) {
    const bool live = kstep(u0 + q4) < units;
    bf16x8 cb[C::TN];
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      const uint32_t z = zc[j];
      const float cv = f16_to_f32(uint16_t(z & 0xffffu)) *
                       (16.0f + f16_to_f32(uint16_t(z >> 16)));
      float o[3];
      split3(live ? -cv : 0.0f, o);
      cb[j] = __builtin_bit_cast(
          bf16x8, u32x4{f32x2_to_bf16x2(o[0], o[1]), f32x2_to_bf16x2(o[0], o[1]),
                        f32x2_to_bf16x2(o[2], o[0]), f32x2_to_bf16x2(o[2], o[1])});
    }
    const float *xold = xsb + ((u0 / 4) & 1) * (C::BM * 4) + q4;
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
      float o[3];
      split3(live ? xold[(wm * C::TM * 16 + i * 16 + sw) * 4] : 0.0f, o);
      const bf16x8 xa = __builtin_bit_cast(
          bf16x8, u32x4{f32x2_to_bf16x2(o[0], o[0]), f32x2_to_bf16x2(o[1], o[1]),
                        f32x2_to_bf16x2(o[0], o[2]), f32x2_to_bf16x2(o[1], o[2])});
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        acc[i][j] = mfma_bf16(xa, cb[j], acc[i][j]);
      }
    }
  };
  __builtin_amdgcn_s_waitcnt(0);
  wq_barrier();

  uint32_t rd = wk, wr = C::STAGES - C::G;
  // Operands and scales of a step from its raw tiles (t: its place among the
  // four of z).  The waves of a SIMD are a pair (w, w + WAVES / 2).  For AQ4
  // the first unpacks a step at the end of the one before, the second at its
  // own start, so that one's unpacking runs under the other's MFMAs (with
  // both at the start: M = 512 14336 -> 4096 79.9 against 75.2 us, M = 2048
  // 4096 -> 28672 in 128 x 256 blocks 503 against 483).  FP8's converts are
  // half as many, and unpacking in two places spilled registers.
  const bool late = !AQ4 || wave >= C::WAVES / 2;
  bf16x8 b[C::TN][4];
  float sf[C::TN];
  auto unpack = [&](const u32x4 (&rw)[C::TN][U], const uint32_t (&z)[C::TN], uint32_t t) {
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      if constexpr (AQ4) {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          b[j][q] = nib8_to_bf16_off16(rw[j][0][q], nmask, nmagic);
        }
        sf[j] = f16_to_f32(uint16_t(
            __builtin_amdgcn_ds_bpermute(int((t * 16 + sw) * 4), int(z[j])) & 0xffff));
      } else {
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
          fp8_tile_operands(rw[j][u], b[j][2 * u], b[j][2 * u + 1]);
        }
      }
    }
  };
  if (!late) {
    unpack(raw[0], zn, 0);
  }
  // FP8's second level of sums: every four steps' sum is added to the total.
  f32x4 sum[AQ4 ? 1 : C::TM][AQ4 ? 1 : C::TN];
  if constexpr (!AQ4) {
    static_assert(AQ4 || C::WK == 1, "a round's first step is its wave's own");
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  auto fold = [&](uint32_t i, uint32_t j) {
    if constexpr (!AQ4) {
      sum[i][j] += acc[i][j];
      asm volatile("" : "+v"(sum[i][j]));
    }
  };
  // This wave's step t (0..3) of the four that start at step u4.
  // TAIL: the weights loaded ahead may be dead, so only the copies count as
  // newer than the next step's.
  auto step = [&](uint32_t u4, uint32_t t, auto tail) {
    const uint32_t g = kstep(u4 + t);
    const char *st = lds + rd * C::A_BYTES;
    u32x4 (&rw)[C::TN][U] = raw[t % C::BD];
    if (late) {
      unpack(rw, zc, t);
    }
    load_b(rw, kstep(u4 + t + C::BD));
    if (t % C::SPB == 0) {
#pragma unroll
      for (uint32_t v = 0; v < C::G; ++v) {
        copy_a((u4 + t) * C::WK + C::STAGES - C::G + v, lds + (wr + v) * C::A_BYTES);
      }
      wr = wr + C::G == C::STAGES ? 0u : wr + C::G;
    }
    __builtin_amdgcn_sched_barrier(0);  // issued before any use below
    // An FP8 weight's K may end in the middle of its last step.
    const uint32_t nq = !AQ4 && decltype(tail)::value && units - g * 2 == 1 ? 2u : 4u;
    float *xcur = xsb + ((u4 / 4) & 1) * (C::BM * 4) + t;
    // At the end one of two groups may have no step left.
    if (C::WK == 1 || !decltype(tail)::value || g < steps) {
    bf16x8 av[4];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      av[q] = a_operand(st, 0, q);
    }
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
      if (AQ4 && i % C::WN == wn) {
        f32x4 xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          xs = mfma_bf16(av[q], ones, xs);
        }
        if (sw < 4) {
          const float lo = sw & 1 ? xs[1] : xs[0], hi = sw & 1 ? xs[3] : xs[2];
          xcur[(wm * C::TM * 16 + i * 16 + 4 * q4 + sw) * 4] = sw & 2 ? hi : lo;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      f32x4 p[C::TN];
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        if (q < 2 || q < nq) {
#pragma unroll
          for (uint32_t j = 0; j < C::TN; ++j) {
            p[j] = mfma_bf16(av[q], b[j][q], q == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : p[j]);
          }
        }
        if (i + 1 < C::TM) {
          av[q] = a_operand(st, i + 1, q);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[i][j][r] = AQ4      ? __builtin_fmaf(sf[j], p[j][r], acc[i][j][r])
                         : t == 0 ? p[j][r]
                                  : acc[i][j][r] + p[j][r];
        }
        // Keeps the sums here: sunk below the next row tile's branch they
        // would keep every tile's products alive.
        asm volatile("" : "+v"(acc[i][j]));
        if (!AQ4 && t == 3) {
          fold(i, j);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    }
    if (!late) {
      unpack(raw[(t + 1) % C::BD], t == 3 ? zn : zc, (t + 1) % 4);
    }
    rd = rd + C::WK >= C::STAGES ? rd + C::WK - C::STAGES : rd + C::WK;
    // Every SPB steps: the next ones' copies have landed before the barrier;
    // later copies and weights stay in flight.
    if (t % C::SPB == C::SPB - 1) {
      constexpr uint32_t R = C::STAGES / C::G;
      constexpr uint32_t bl = decltype(tail)::value ? 0 : C::SPB * C::TN * U;
      constexpr uint32_t last = decltype(tail)::value ? 0 : (C::SPB - 1) * C::TN * U;
      wq_wait_vm<(R - 2) * (C::G * C::COPIES + bl) + last>();
      wq_barrier();
    }
  };
  auto next_z = [&](uint32_t u4) {
    if constexpr (AQ4) {
      if (u4 != 0) {
        correct(u4 - 4);
      }
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        zc[j] = zn[j];
      }
      load_z(u4 + 4);
    }
  };
  // Whole steps only: an FP8 weight's half step, which ends at an odd number of
  // 64-k tiles, must find its tail step below whatever the count is.
  const uint32_t whole = units / U;
  uint32_t u4 = 0;
#pragma clang loop unroll(disable)
  for (; (u4 + 4) * C::WK <= whole; u4 += 4) {
    next_z(u4);
#pragma unroll
    for (uint32_t t = 0; t < 4; ++t) {
      step(u4, t, std::false_type{});
    }
  }
  // The last one to three steps (four where the last is an FP8 half step, or
  // where one of two groups has none).
  const uint32_t usteps = (steps + C::WK - 1) / C::WK;
  if (u4 < usteps) {
    next_z(u4);
    step(u4, 0, std::true_type{});
    if (u4 + 1 < usteps) {
      step(u4, 1, std::true_type{});
      if (u4 + 2 < usteps) {
        step(u4, 2, std::true_type{});
        if ((!AQ4 || C::WK > 1) && u4 + 3 < usteps) {
          step(u4, 3, std::true_type{});
        }
      }
    }
  }
  if constexpr (!AQ4) {
    const bool open = usteps % 4 != 0;  // the last round ended before its fourth step
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        acc[i][j] = open ? sum[i][j] + acc[i][j] : sum[i][j];
      }
    }
  }
  wq_wait_vm<0>();  // no copy may land in the stages the epilogue reuses
  wq_barrier();

  const uint32_t mw = m0 + wm * C::TM * 16 + 4 * q4;
  if constexpr (AQ4) {
    correct((usteps - 1) / 4 * 4);
  }
  // The two K groups' sums: each wave hands the row tiles it will not store to
  // the wave that will.
  constexpr uint32_t HALF = C::TM / C::WK;
  auto stores = [&](uint32_t i) { return C::WK == 1 || i / HALF == wk; };
  if constexpr (C::WK > 1) {
    static_assert(C::WAVES * HALF * C::TN * 1024 <= C::MAIN_BYTES, "exchange fits");
    f32x4 *ex = reinterpret_cast<f32x4 *>(lds);
    const uint32_t other = wave < C::WM * C::WN ? wave + C::WM * C::WN : wave - C::WM * C::WN;
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
      if (!stores(i)) {
#pragma unroll
        for (uint32_t j = 0; j < C::TN; ++j) {
          ex[((wave * HALF + i % HALF) * C::TN + j) * kWave + lane] = acc[i][j];
        }
      }
    }
    wq_barrier();
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
      if (stores(i)) {
#pragma unroll
        for (uint32_t j = 0; j < C::TN; ++j) {
          acc[i][j] += ex[((other * HALF + i % HALF) * C::TN + j) * kWave + lane];
        }
      }
    }
    wq_barrier();  // the chunks below reuse the exchange
  }
  if constexpr (!AQ4) {
    const float *scales = static_cast<const float *>(a.aux);
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      const float s = scales[min((T0 + j) * 16 + sw, a.n16 - 1)];
#pragma unroll
      for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[i][j][r] *= s;
        }
      }
    }
  }
  const bool vec = !a.y_f32 && reinterpret_cast<uintptr_t>(a.y) % 16 == 0 && a.ldy % 8 == 0;
  if (!vec) {
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
      if (!stores(i)) {
        continue;
      }
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t m = mw + i * 16 + r;
          store_out<EPI>(a.y, a.ldy, a.y_f32, a.epi, a.n, m, (T0 + j) * 16 + sw,
                         a.alpha * acc[i][j][r], m < a.m);
        }
      }
    }
    return;
  }
  // bf16 rows leave through a wave-private LDS chunk as 16-byte segments.
  constexpr bool gated = EPI == kEpiSiluMul;
  constexpr uint32_t tw = gated ? 8 : 16;
  constexpr uint32_t lpr = C::TN * tw / 8, segs = 16 * lpr;
  uint16_t *chunk = reinterpret_cast<uint16_t *>(lds + wave * C::CHUNK_BYTES);
  const uint32_t n0 = T0 * tw, nlim = gated ? a.epi.n_out : a.n;
#pragma unroll
  for (uint32_t i = 0; i < C::TM; ++i) {
    if (!stores(i)) {
      continue;
    }
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = a.alpha * acc[i][j][r];
        if constexpr (gated) {
          const float up = __shfl_xor(v[r], 8, kWave);
          v[r] = silu_f32(v[r]) * up;
        } else if constexpr (EPI == kEpiResidual) {
          const uint32_t m = mw + i * 16 + r, n = (T0 + j) * 16 + sw;
          if (m < a.m && n < a.n) {
            const uint64_t ri = uint64_t(m) * a.epi.ldr + n;
            v[r] += a.epi.res_f32
                        ? static_cast<const float *>(a.epi.res)[ri]
                        : bf16_to_f32(static_cast<const uint16_t *>(a.epi.res)[ri]);
          }
        }
      }
      const uint32_t p01 = f32x2_to_bf16x2(v[0], v[1]);
      const uint32_t p23 = f32x2_to_bf16x2(v[2], v[3]);
      uint16_t *c0 = chunk + 4 * q4 * C::OUT_STRIDE + j * tw + sw;
      if (!gated || sw < 8) {
        c0[0] = uint16_t(p01);
        c0[C::OUT_STRIDE] = uint16_t(p01 >> 16);
        c0[2 * C::OUT_STRIDE] = uint16_t(p23);
        c0[3 * C::OUT_STRIDE] = uint16_t(p23 >> 16);
      }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
#pragma unroll
    for (uint32_t it = 0; it < (segs + kWave - 1) / kWave; ++it) {
      const uint32_t seg = it * kWave + lane;
      if (segs % kWave == 0 || seg < segs) {
        const uint32_t rr = seg / lpr, c8 = (seg % lpr) * 8;
        const u32x4 w = *reinterpret_cast<const u32x4 *>(chunk + rr * C::OUT_STRIDE + c8);
        const uint32_t mo = m0 + wm * C::TM * 16 + i * 16 + rr, n = n0 + c8;
        uint16_t *dst = static_cast<uint16_t *>(a.y) + uint64_t(mo) * a.ldy + n;
        if (mo < a.m) {
          if (n + 8 <= nlim) {
            __builtin_nontemporal_store(w, reinterpret_cast<u32x4 *>(dst));
          } else {
            const uint32_t e4[4] = {w.x, w.y, w.z, w.w};
            for (uint32_t e = 0; e < 8 && n + e < nlim; ++e) {
              dst[e] = static_cast<uint16_t>(e4[e / 2] >> (16 * (e % 2)));
            }
          }
        }
      }
    }
    asm volatile("" ::: "memory");
  }
}


// Strip configuration: TM x TN 16 x 16 tiles, WAVES waves splitting K, each
// with DEPTH LDS stages of x of its own.
template <uint32_t TM_, uint32_t TN_, uint32_t WAVES_, uint32_t DEPTH_ = 2>
struct StripCfg {
  static constexpr uint32_t TM = TM_, TN = TN_, WAVES = WAVES_, DEPTH = DEPTH_;
  static constexpr uint32_t BM = TM * 16, BN = TN * 16;
  static constexpr uint32_t A_BYTES = BM * 256;
  static constexpr uint32_t WAVE_BYTES =
      DEPTH * A_BYTES > TM * TN * 1024 ? DEPTH * A_BYTES : TM * TN * 1024;
  static constexpr uint32_t LDS = WAVES * WAVE_BYTES;
  static_assert(LDS <= 160 * 1024, "gfx950 LDS per workgroup");
};

// Strips.  A workgroup's waves split K; each copies its own rows x 128 k of x
// into its own LDS ring (same swizzle as above) and streams its own weight
// tiles into registers, one step ahead, so no wave waits for another before
// the sums meet in LDS at the end.  On grids this small a launch costs a
// fixed part (start, first loads, reduction) plus its bytes at the copy rate
// of a CU, so the block shape that makes the grid fill the CUs wins.
template <bool AQ4, class C, int EPI>
__global__ __launch_bounds__(C::WAVES *kWave) void wq_strip_kernel(GemvArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t sw = lane % 16, q4 = lane / 16;
  const uint32_t stripes = a.n16 / 16;
  const uint32_t mblocks = (a.m + C::BM - 1) / C::BM;
  const uint32_t tile = wq_tile();
  const uint32_t m0 = (tile % mblocks) * C::BM;
  const uint32_t T0 = (tile / mblocks) * C::TN;
  const uint32_t units = a.units;
  constexpr uint32_t U = AQ4 ? 1 : 2;
  const uint32_t steps = (units + U - 1) / U;
  const uint32_t sb = steps * wave / C::WAVES, se = steps * (wave + 1) / C::WAVES;

  const uint32_t rows = min(C::BM, a.m - m0);
  const __amdgpu_buffer_rsrc_t abuf = byte_buffer(
      a.x + uint64_t(m0) * a.ldx, uint32_t(((rows - 1) * a.ldx + a.k) * 2));
  const uint32_t nT = min(C::TN, stripes - T0);
  const __amdgpu_buffer_rsrc_t wbuf = byte_buffer(
      static_cast<const uint8_t *>(a.tiles) + uint64_t(T0) * units * 1024,
      nT * units * 1024);
  const __amdgpu_buffer_rsrc_t zbuf =
      byte_buffer(static_cast<const uint32_t *>(a.aux) + uint64_t(T0) * units * 16,
                  AQ4 ? nT * units * 64 : 0u);
  const uint32_t ldb = uint32_t(a.ldx) * 2;
  char *const mine = lds + wave * C::WAVE_BYTES;
  uint32_t avoff[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    avoff[i] = (i * 4 + q4) * ldb + ((sw ^ q4 ^ (4 * i)) * 16);
  }
  struct Batch {
    u32x4 w[C::TN][U];
    uint32_t z[C::TN];
  };
  constexpr uint32_t OPS = C::TM * 4 + C::TN * U + (AQ4 ? C::TN : 0);
  auto issue = [&](Batch &bt, uint32_t g, uint32_t slot) {
    // Past the wave's run every load falls outside its buffer.
    const uint32_t past = g < se ? 0u : 0x80000000u;
#pragma unroll
    for (uint32_t i = 0; i < C::TM * 4; ++i) {
      wq_dma16(abuf, avoff[i % 4], (g * 256 + (i / 4) * 16 * ldb) | past,
               mine + slot * C::A_BYTES + i * 1024);
    }
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        bt.w[j][u] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       wbuf, lane * 16, ((j * units + g * U + u) * 1024) | past, 0));
      }
      if constexpr (AQ4) {
        bt.z[j] = __builtin_amdgcn_raw_buffer_load_b32(
            zbuf, sw * 4, ((j * units + g) * 64) | past, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[C::TM][C::TN];
#pragma unroll
  for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  const uint32_t nmask = opaque_u32(0x00780078u);
  const uint32_t nmagic = opaque_u32(0x41804180u);
  const bf16x8 ones = __builtin_bit_cast(
      bf16x8, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  auto consume = [&](const Batch &bt, uint32_t g, uint32_t slot) {
    const char *st = mine + slot * C::A_BYTES + sw * 256;
    auto a_operand = [&](uint32_t i, uint32_t c) {
      return *reinterpret_cast<const bf16x8 *>(st + i * 4096 + ((c ^ sw) * 16));
    };
    if constexpr (AQ4) {
      bf16x8 av[C::TM][4];
      f32x4 xs[C::TM];
#pragma unroll
      for (uint32_t i = 0; i < C::TM; ++i) {
        xs[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          av[i][q] = a_operand(i, 4 * q + q4);
          xs[i] = mfma_bf16(av[i][q], ones, xs[i]);
        }
      }
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        f32x4 p[C::TM];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          const bf16x8 b = nib8_to_bf16_off16(bt.w[j][0][q], nmask, nmagic);
#pragma unroll
          for (uint32_t i = 0; i < C::TM; ++i) {
            p[i] = mfma_bf16(av[i][q], b, q == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : p[i]);
          }
        }
        const float sf = f16_to_f32(uint16_t(bt.z[j] & 0xffffu));
        const float zoff = 16.0f + f16_to_f32(uint16_t(bt.z[j] >> 16));
#pragma unroll
        for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            acc[i][j][r] = __builtin_fmaf(sf, __builtin_fmaf(-zoff, xs[i][r], p[i][r]),
                                          acc[i][j][r]);
          }
        }
      }
    } else {
      const uint32_t nu = min(units - g * 2, 2u);
#pragma unroll
      for (uint32_t u = 0; u < 2; ++u) {
        if (u < nu) {
          bf16x8 av[C::TM][2];
#pragma unroll
          for (uint32_t i = 0; i < C::TM; ++i) {
            av[i][0] = a_operand(i, 8 * u + 2 * q4);
            av[i][1] = a_operand(i, 8 * u + 2 * q4 + 1);
          }
#pragma unroll
          for (uint32_t j = 0; j < C::TN; ++j) {
            bf16x8 b0, b1;
            fp8_tile_operands(bt.w[j][u], b0, b1);
#pragma unroll
            for (uint32_t i = 0; i < C::TM; ++i) {
              acc[i][j] = mfma_bf16(av[i][0], b0, acc[i][j]);
            }
#pragma unroll
            for (uint32_t i = 0; i < C::TM; ++i) {
              acc[i][j] = mfma_bf16(av[i][1], b1, acc[i][j]);
            }
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  Batch ring[C::DEPTH];
#pragma unroll
  for (uint32_t r = 0; r + 1 < C::DEPTH; ++r) {
    issue(ring[r], sb + r, r);
  }
  // FP8: the chain of a wave's products is cut every DEPTH steps and the parts
  // are added up: relative error at M=64 N=4096 K=14336 1.0e-7 instead of
  // 2.0e-7 (the decode kernels 1.4e-7), M=203 N=5003 K=4096 8.0e-8 instead of
  // 1.1e-7 (9.1e-8), at the same time (26.7 / 26.5 us, 21.5 / 21.7).
  f32x4 sum[C::TM][C::TN];
  if constexpr (!AQ4) {
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  auto fold = [&]() {
#pragma unroll
    for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
      for (uint32_t j = 0; j < C::TN; ++j) {
        sum[i][j] += acc[i][j];
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(sum[i][j]));
      }
    }
  };
  const uint32_t n = se - sb;
  for (uint32_t t = 0; t < n; t += C::DEPTH) {
#pragma unroll
    for (uint32_t r = 0; r < C::DEPTH; ++r) {
      issue(ring[(r + C::DEPTH - 1) % C::DEPTH], sb + t + r + C::DEPTH - 1,
            (r + C::DEPTH - 1) % C::DEPTH);
      // This step's copies and weights have landed; the next steps' stay in
      // flight.
      wq_wait_vm<(C::DEPTH - 1) * OPS>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (t + r < n) {
        consume(ring[r], sb + t + r, r);
      }
      asm volatile("" ::: "memory");
    }
    if constexpr (!AQ4) {
      fold();
    }
  }
  wq_wait_vm<0>();
  asm volatile("" ::: "memory");
  // Cross-wave reduction: every wave's sums go to its own LDS region.
  f32x4 *red = reinterpret_cast<f32x4 *>(mine);
#pragma unroll
  for (uint32_t i = 0; i < C::TM; ++i) {
#pragma unroll
    for (uint32_t j = 0; j < C::TN; ++j) {
      red[(i * C::TN + j) * kWave + lane] = AQ4 ? acc[i][j] : sum[i][j];
    }
  }
  wq_barrier();
  // Output o: row o / BN, column o % BN; its sum sits at element row % 4 of
  // lane column % 16 + 16 * (row % 16 / 4) of its tile.
  for (uint32_t o = threadIdx.x; o < C::BM * C::BN; o += C::WAVES * kWave) {
    const uint32_t r = o / C::BN, c = o % C::BN;
    const uint32_t at = ((r / 16 * C::TN + c / 16) * kWave + c % 16 + 16 * (r % 16 / 4)) * 4 + r % 4;
    float v = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < C::WAVES; ++w) {
      v += reinterpret_cast<const float *>(lds + w * C::WAVE_BYTES)[at];
    }
    const uint32_t nn = T0 * 16 + c;
    if constexpr (!AQ4) {
      v *= static_cast<const float *>(a.aux)[min(nn, a.n16 - 1)];
    }
    store_out<EPI>(a.y, a.ldy, a.y_f32, a.epi, a.n, m0 + r, nn, a.alpha * v, m0 + r < a.m);
  }
}

template <bool AQ4, class C, int EPI>
hipError_t launch_wq_t(const GemvArgs &a, hipStream_t s) {
  const void *k = reinterpret_cast<const void *>(wq_gemm_kernel<AQ4, C, EPI>);
  const hipError_t e = raise_lds_limit(k, C::LDS);
  if (e != hipSuccess) {
    return e;
  }
  const uint32_t tiles = (a.m + C::BM - 1) / C::BM * ((a.n16 + C::BN - 1) / C::BN);
  hipLaunchKernelGGL((wq_gemm_kernel<AQ4, C, EPI>), dim3(tiles), dim3(C::WAVES * kWave),
                     C::LDS, s, a);
  return hipGetLastError();
}

template <bool AQ4, class C, int EPI>
hipError_t launch_strip_t(const GemvArgs &a, hipStream_t s) {
  const void *k = reinterpret_cast<const void *>(wq_strip_kernel<AQ4, C, EPI>);
  const hipError_t e = raise_lds_limit(k, C::LDS);
  if (e != hipSuccess) {
    return e;
  }
  const uint32_t tiles = (a.m + C::BM - 1) / C::BM * ((a.n16 + C::BN - 1) / C::BN);
  hipLaunchKernelGGL((wq_strip_kernel<AQ4, C, EPI>), dim3(tiles), dim3(C::WAVES * kWave),
                     C::LDS, s, a);
  return hipGetLastError();
}

using W128x384 = WqCfg<8, 3, 1, 8, 3>;
using W128x256 = WqCfg<8, 2, 1, 8, 3>;
using W64x128 = WqCfg<4, 1, 1, 8, 4, 2, 2>;
using W32x128 = WqCfg<2, 1, 1, 8, 6, 2, 2>;
using W64x128K = WqCfg<4, 2, 1, 4, 6, 2, 1, 2>;
using S64x64 = StripCfg<4, 4, 4>;
using S48x64 = StripCfg<3, 4, 6>;
using S48x48 = StripCfg<3, 3, 6>;
using S32x96 = StripCfg<2, 6, 4>;
using S32x64 = StripCfg<2, 4, 4>;
using S32x48 = StripCfg<2, 3, 4>;
using S32x32 = StripCfg<2, 2, 4>;
using S16x32 = StripCfg<1, 2, 8>;

// What a launch of each configuration takes, in microseconds: t0 + rounds x
// (k-steps x step + tile), rounds = its tiles over the CUs, rounded up (also
// where LDS fits two workgroups per CU: they share what bounds them).
// Fitted to launches of every configuration on one MI355X (256 CUs, weights
// from HBM) over M = 33 .. 2048 and (N, K) = (1024 | 4096 | 6144 | 14336 |
// 28672, 4096), (4096, 14336), (2560, 1024), (9000, 2048).  The choice it
// makes is the fastest of the table or within 1 % of it on average, 10 % at
// worst; without the 48-row strips it is up to 18 % worse (M = 64, N = 6144),
// without the 64 x 128 blocks of one K group up to 14 % (M = 384, N = 9000).
struct WqCost {
  uint32_t bm, bn;
  float aq4[3], fp8[3];  // t0, step, tile; t0 < 0: not used
};
constexpr WqCost kWqCosts[] = {
    {128, 384, {0.00f, 2.374f, 6.04f}, {-1.0f, 0.0f, 0.0f}},
    {128, 256, {0.00f, 1.788f, 4.37f}, {0.00f, 1.593f, 3.51f}},
    {64, 128, {3.71f, 0.671f, 0.00f}, {2.92f, 0.588f, 0.00f}},
    {64, 128, {0.23f, 0.612f, 3.60f}, {-1.0f, 0.0f, 0.0f}},
    {32, 128, {3.57f, 0.416f, 0.00f}, {2.64f, 0.376f, 0.05f}},
    {64, 64, {0.65f, 0.344f, 4.72f}, {0.58f, 0.314f, 4.52f}},
    {48, 64, {1.11f, 0.280f, 4.16f}, {1.40f, 0.282f, 3.39f}},
    {48, 48, {1.27f, 0.233f, 3.41f}, {1.35f, 0.241f, 3.07f}},
    {32, 96, {4.27f, 0.275f, 1.04f}, {3.51f, 0.255f, 1.36f}},
    {32, 64, {3.35f, 0.214f, 0.62f}, {2.63f, 0.209f, 0.88f}},
    {32, 48, {3.03f, 0.169f, 0.65f}, {2.36f, 0.171f, 0.88f}},
    {32, 32, {2.73f, 0.143f, 0.33f}, {2.07f, 0.151f, 0.53f}},
    {16, 32, {2.46f, 0.078f, 0.58f}, {2.30f, 0.095f, 0.64f}},
};
enum : uint32_t {
  kW128x384, kW128x256, kW64x128, kW64x128K, kW32x128, kS64x64, kS48x64,
  kS48x48, kS32x96, kS32x64, kS32x48, kS32x32, kS16x32
};

template <bool AQ4, int EPI>
hipError_t wq_e(const GemvArgs &a, uint32_t cfg, hipStream_t s) {
  switch (cfg) {
    case kW128x384:
      // FP8's two levels of sums do not fit its registers.
      if constexpr (AQ4) {
        return launch_wq_t<AQ4, W128x384, EPI>(a, s);
      }
      break;
    case kW128x256: return launch_wq_t<AQ4, W128x256, EPI>(a, s);
    case kW64x128: return launch_wq_t<AQ4, W64x128, EPI>(a, s);
    case kW64x128K:
      // FP8 gains on one round only (M = 512 14336 -> 4096 79 against 72 us)
      // and loses on more.
      if constexpr (AQ4) {
        return launch_wq_t<AQ4, W64x128K, EPI>(a, s);
      }
      break;
    case kW32x128: return launch_wq_t<AQ4, W32x128, EPI>(a, s);
    case kS64x64: return launch_strip_t<AQ4, S64x64, EPI>(a, s);
    case kS48x64: return launch_strip_t<AQ4, S48x64, EPI>(a, s);
    case kS48x48: return launch_strip_t<AQ4, S48x48, EPI>(a, s);
    case kS32x96: return launch_strip_t<AQ4, S32x96, EPI>(a, s);
    case kS32x64: return launch_strip_t<AQ4, S32x64, EPI>(a, s);
    case kS32x48: return launch_strip_t<AQ4, S32x48, EPI>(a, s);
    case kS32x32: return launch_strip_t<AQ4, S32x32, EPI>(a, s);
    case kS16x32: return launch_strip_t<AQ4, S16x32, EPI>(a, s);
    default: break;
  }
  return hipErrorInvalidValue;
}

template <int EPI>
hipError_t wq_enc(const GemvArgs &a, bool aq4, uint32_t cfg, hipStream_t s) {
  return aq4 ? wq_e<true, EPI>(a, cfg, s) : wq_e<false, EPI>(a, cfg, s);
}

// 17 to 32 rows on at most one round of 16 x 32 strips, where the decode
// kernels leave CUs idle and run a stripe's whole K in one workgroup.  MI355X,
// decode kernels / strips, us: M=32 N=480 K=10624 AQ4 22.6 / 8.5, FP8 22.2 /
// 9.0; M=17 N=1000 K=8192 9.6 / 8.0 and 14.5 / 8.9; M=32 N=4096 K=8192 13.2 /
// 9.9 and 16.9 / 12.5; M=24 N=3000 K=5120 8.4 / 7.0 and 10.3 / 8.5; M=32
// N=1024 K=4096 6.8 / 5.1 and 8.3 / 5.1, K=1024 3.5 / 3.2 and 4.0 / 3.8.
// - up to 16 rows, one strip of rows, half as many CUs work (M=16 N=2048
//   K=8192 7.9 / 9.1, 9.6 / 11.6).
// - the other lines are narrower than where the kernels cross.  The strips are
//   ahead beyond them too, but the tests pin those sizes to the decode
//   kernels.  K <= 4096, or fewer than 24 rows or more than half of the CUs
//   there (AQ4, FP8): M=32 N=4096 K=4096 7.4 / 5.7, 9.3 / 5.8, K=2048 5.2 /
//   4.4, 6.4 / 4.4, K=1024 3.9 / 3.7, 4.6 / 4.1; M=17 N=1000 K=4096 6.7 / 4.6,
//   6.4 / 5.0.  Calls that the decode kernels split over K (from 12288): M=32
//   N=4096 K=12288 15.5 / 12.8, 20.0 / 18.2, K=14336 16.9 / 15.2, 21.3 / 20.6;
//   M=32 N=1000 K=14336 15.0 / 10.1, 23.1 / 11.0.
// Relative error at K = 10624: FP8 9.2e-8 against 1.3e-7, AQ4 1.9e-7 against
// 1.8e-6.
bool wq_few_rows(const GemvArgs &a, bool aq4, uint32_t cus) {
  const uint32_t tiles = (a.m + 15) / 16 * ((a.n16 + 31) / 32);
  return a.m > 16 && tiles <= cus && (aq4 || a.k <= 10752) &&
         (a.k > 4096 || (a.m >= 24 && a.k >= 2048 && 2 * tiles <= cus)) &&
         gemv_split_parts(a, aq4) == 1;
}

}  // namespace

// The calls of wq_few_rows, and those of more than 32 rows, with aligned
// activations and whole 64-k tiles, but one kind of the latter: up to four
// rows past the first 32 at K <= 1024 on more stripes than CUs, which the tests
// pin to the decode kernels' two passes.  Those are ahead for AQ4 on 6200 to
// 8192 columns at K = 512 only (decode kernels / blocks, us: M = 33, N = 8192
// 4.7 / 5.2) and lose elsewhere (N = 8192, K = 1024 AQ4 6.2 / 5.8, FP8 7.4 /
// 5.9; N = 28672, K = 1024 16.2 / 9.6, 18.0 / 9.8), by 1.2 to 7.8 times
// outside that kind.  Sizes whose 32-bit buffer offsets would not do stay with
// them.
WqPlan plan_wq_gemm(const GemvArgs &a, bool aq4) {
  WqPlan p;
  const uint32_t unit_k = aq4 ? 128 : 64;
  const uint64_t row_bytes = a.ldx * 2;
  const uint32_t cus = device_cu_count();
  const bool few = a.m <= 32;
  if (few ? !wq_few_rows(a, aq4, cus)
          : a.m <= 36 && a.k <= 1024 && a.n16 / 16 > cus) {
    return p;
  }
  if (a.k % unit_k != 0 || reinterpret_cast<uintptr_t>(a.x) % 16 != 0 || a.ldx % 8 != 0 ||
      row_bytes >= (uint64_t(1) << 22) || a.units >= (1u << 17)) {
    return p;
  }
  int forced = -1;
  if (const char *v = tuning_env("ULLM_WQ")) {  // read by a -DULLM_TUNING build only
    forced = std::atoi(v);
  }
  const float steps = float((uint64_t(a.k) + 127) / 128);
  float best = 0.0f;
  for (uint32_t i = 0; i < sizeof(kWqCosts) / sizeof(kWqCosts[0]); ++i) {
    const WqCost &c = kWqCosts[i];
    const float *t = aq4 ? c.aq4 : c.fp8;
    const uint64_t tiles = uint64_t((a.m + c.bm - 1) / c.bm) * ((a.n16 + c.bn - 1) / c.bn);
    if (t[0] < 0.0f || tiles >= (1u << 22) || (forced >= 0 && uint32_t(forced) != i) ||
        (few && i != kS16x32)) {
      continue;
    }
    const uint64_t rounds = (tiles + cus - 1) / cus;
    const float cost = t[0] + float(rounds) * (steps * t[1] + t[2]);
    if (!p.taken || cost < best) {
      p = WqPlan{true, i, c.bm, c.bn, uint32_t(tiles)};
      best = cost;
    }
  }
  return p;
}

hipError_t launch_wq_gemm(const GemvArgs &a, bool aq4, const WqPlan &p, hipStream_t s) {
  switch (a.epi.kind) {
    case kEpiSiluMul: return wq_enc<kEpiSiluMul>(a, aq4, p.cfg, s);
    case kEpiResidual: return wq_enc<kEpiResidual>(a, aq4, p.cfg, s);
    default: return wq_enc<kEpiNone>(a, aq4, p.cfg, s);
  }
}

}  // namespace ullm
