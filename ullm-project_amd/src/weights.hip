// weights.hip -- quantization, repacking, export and dequantization of
// device-resident weights, and per-token activation quantization.
//
// These kernels run once per weight (creation) or are parity/debug tools; the
// activation quantizer is on the prefill path and is HBM-bound (2 bytes read,
// 1 byte written per element).  All arithmetic that defines a quantized value
// is written with FMA contraction off so it matches the format definitions
// bit for bit: q = enc(w / s), dequant = dec(q) * s, AQ4 dequant = (q - z) * s.
#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace ullm {
namespace {

constexpr int kBlock = 256;

template <int BLOCK = kBlock>
__device__ float block_max(float v, float *red) {
  v = wave_max(v);
  const int wave = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) {
    red[wave] = v;
  }
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < BLOCK / kWave; ++i) {
    r = fmaxf(r, red[i]);
  }
  return r;
}

// ------------------------------------------------------------ weight tiles
// Every kernel below moves whole 1 KiB wave tiles, one wave per tile (the FP8
// quantizer, which needs row maxima, a workgroup per four rows of a stripe).
// Encoded values keep the tile's order, lane l = physical row l % 16 and
// 16-byte slot l / 16 of it: the tile side of a copy is one 16-byte access
// per lane and the canonical side runs of 64 bytes of 16 rows, with the
// tile's place in the matrix a wave-uniform division instead of one per
// element.  They are bound by memory.  Padding rows and columns
// are written as zeros, so the buffers need no clearing first.  MI355X, N =
// 14336, K = 4096, sources from HBM (element-wise kernels with byte or word
// accesses before): FP8 quantize 174 -> 61 us and decode 162 -> 55 us, AQ4
// quantize 118 -> 50 us and decode 127 -> 59 us.

// Calls f(tile index, stripe, unit) for each of this wave's tiles (of
// stripes x units; more than one only past kMaxTileBlocks workgroups).
constexpr unsigned kMaxTileBlocks = 1u << 23;
template <class F>
__device__ __forceinline__ void for_tiles(uint64_t stripes, uint64_t units, F f) {
  constexpr uint64_t per = kBlock / kWave;
  for (uint64_t i = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) + blockIdx.x * per;
       i < stripes * units; i += gridDim.x * per) {
    f(i, i / units, i % units);
  }
}

__device__ __forceinline__ bool aligned16(const void *p) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

// --------------------------------------------------------------- FP8 rows
// Floats go the other way round: four rows x 16 lanes an instruction, 16 bytes
// a lane, so that each row's 64 columns of a tile are one 256-byte run (a lane
// per 16-byte slot, four 16-byte accesses 64 bytes apart, took 322 us to
// decode N = 14336, K = 4096 and this takes 50).  The tile side is then one
// dword a lane: row r, columns 4 c .. + 3 at dword (r + 16 (c / 4)) * 4 + c % 4.

// Four weights of a row at column c (zeros past K).
__device__ __forceinline__ f32x4 load_row4(const float *row, uint64_t c, uint64_t k,
                                           bool vec) {
  if (vec && c + 4 <= k) {
    return *reinterpret_cast<const f32x4 *>(row + c);
  }
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = c + e < k ? row[c + e] : 0.0f;
  }
  return v;
}

// E4M3 codes of v / s.  Quotients of a finite scale are at most one rounding
// past 448, where the hardware convert rounds to nearest even and saturates
// exactly like f32_to_e4m3; anything else (NaN, an infinite or subnormal
// scale) takes the software encode.
__device__ __forceinline__ uint32_t encode4(f32x4 v, float s) {
  if (s == 0.0f) {
    return 0u;
  }
  float q[4];
  bool plain = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    q[e] = v[e] / s;
    plain = plain && fabsf(q[e]) < 449.0f;
  }
  if (plain) {
    s16x2 r = {0, 0};
    r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, q[0], q[1], 1.0f, false);
    r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, q[2], q[3], 1.0f, true);
    return __builtin_bit_cast(uint32_t, r);
  }
  uint32_t w = 0u;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    w |= f32_to_e4m3(q[e]) << (8 * e);
  }
  return w;
}

// One workgroup per four rows of a stripe: s = max|w| / 448 of each row, q =
// e4m3(w / s).  Wave w takes tiles w, w + W, ...; up to NB of them (K <= 64 W
// NB) stay in registers between the row maximum and the encode, so the floats
// are read from memory once; NB = 0 reads them twice, for any K.  Four rows,
// not the stripe's 16, so that several workgroups share a CU and one's loads
// run under another's encode (76 against 93 us for whole
// stripes); the four workgroups of a stripe sit on one XCD, where their
// 64-byte pieces of a tile line meet in L2.
template <int W, int NB>
__global__ __launch_bounds__(W *kWave) void fp8_quantize_kernel(
    const float *__restrict__ w, Fp8Layout L, uint8_t *__restrict__ tiles,
    float *__restrict__ scales) {
  __shared__ float red[W][4];
  const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const uint32_t r0 = lane / 16, c = lane % 16;
  // Workgroups go round-robin over the 8 XCDs: stripe T's four are 8 apart.
  const uint64_t T = uint64_t(blockIdx.x / 32) * 8 + blockIdx.x % 8;
  if (T >= L.n16 / 16) {
    return;  // the last group of 8 stripes is partly filled
  }
  const uint32_t r = r0 + 4 * (blockIdx.x / 8 % 4);  // row of the stripe
  const uint64_t n = canonical_row(T * 16 + r, L.n, L.gate);
  const float *row = w + (n < L.n ? n : 0) * L.k;
  const uint64_t kk = n < L.n ? L.k : 0;  // columns to read: 0 for padding
  const bool vec = aligned16(w) && L.k % 4 == 0;
  const uint32_t units = uint32_t(L.blocks_per_stripe());
  f32x4 v[NB > 0 ? NB : 1];
  float amax = 0.0f;
  auto take = [&](uint32_t u) {
    return load_row4(row, uint64_t(u) * 64 + 4 * c, u < units ? kk : 0, vec);
  };
  auto fold = [&](f32x4 x) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      amax = fmaxf(amax, fabsf(x[e]));
    }
  };
  if constexpr (NB > 0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      v[b] = take(wave + b * W);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      fold(v[b]);
    }
  } else {
    for (uint32_t u = wave; u < units; u += W) {
      fold(take(u));
    }
  }
#pragma unroll
  for (int off = 1; off < 16; off *= 2) {
    amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
  }
  if (c == 0) {
    red[wave][r0] = amax;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < W; ++j) {
    amax = fmaxf(amax, red[j][r0]);
  }
  const float s = amax / 448.0f;
  if (threadIdx.x < kWave && c == 0) {
    scales[T * 16 + r] = s;
  }
  uint32_t *out = reinterpret_cast<uint32_t *>(tiles) + T * units * 256 +
                  (r + 16 * (c / 4)) * 4 + c % 4;
  if constexpr (NB > 0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (wave + b * W < units) {
        out[uint64_t(wave + b * W) * 256] = encode4(v[b], s);
      }
    }
  } else {
    for (uint32_t u = wave; u < units; u += W) {
      out[uint64_t(u) * 256] = encode4(take(u), s);
    }
  }
}

__global__ __launch_bounds__(kBlock) void fp8_pack_kernel(
    const uint8_t *__restrict__ q, const float *__restrict__ s_in, Fp8Layout L,
    uint8_t *__restrict__ tiles, float *__restrict__ scales) {
  for_tiles(L.n16 / 16, L.blocks_per_stripe(), [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t lane = threadIdx.x % kWave;
    const uint64_t p = stripe * 16 + lane % 16, n = canonical_row(p, L.n, L.gate);
    const uint64_t c = unit * 64 + 16 * (lane / 16);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (n < L.n) {
      const uint8_t *src = q + n * L.k + c;
      if (c + 16 <= L.k && L.k % 16 == 0 && aligned16(q)) {
        v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src));
      } else {
        uint32_t b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          b[i / 4] |= (c + i < L.k ? uint32_t(src[i]) : 0u) << (8 * (i % 4));
        }
        v = u32x4{b[0], b[1], b[2], b[3]};
      }
    }
    reinterpret_cast<u32x4 *>(tiles)[index * kWave + lane] = v;
    if (unit == 0 && lane < 16) {
      scales[p] = n < L.n ? s_in[n] : 0.0f;
    }
  });
}

__global__ __launch_bounds__(kBlock) void fp8_export_kernel(
    const uint8_t *__restrict__ tiles, const float *__restrict__ scales,
    Fp8Layout L, uint8_t *__restrict__ q, float *__restrict__ s_out) {
  for_tiles(L.n16 / 16, L.blocks_per_stripe(), [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t lane = threadIdx.x % kWave;
    const uint64_t p = stripe * 16 + lane % 16, n = canonical_row(p, L.n, L.gate);
    const uint64_t c = unit * 64 + 16 * (lane / 16);
    if (n >= L.n) {
      return;
    }
    const u32x4 v = reinterpret_cast<const u32x4 *>(tiles)[index * kWave + lane];
    uint8_t *dst = q + n * L.k + c;
    if (c + 16 <= L.k && L.k % 16 == 0 && aligned16(q)) {
      *reinterpret_cast<u32x4 *>(dst) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (c + i < L.k) {
          dst[i] = uint8_t(v[i / 4] >> (8 * (i % 4)));
        }
      }
    }
    if (unit == 0 && lane < 16) {
      s_out[n] = scales[p];
    }
  });
}

// Four floats to columns c .. c + 3 of a row of k columns.
__device__ __forceinline__ void store_row4(float *row, uint64_t c, uint64_t k, bool vec,
                                           f32x4 v) {
  if (vec && c + 4 <= k) {
    *reinterpret_cast<f32x4 *>(row + c) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (c + e < k) {
        row[c + e] = v[e];
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void fp8_dequant_kernel(
    const uint8_t *__restrict__ tiles, const float *__restrict__ scales,
    Fp8Layout L, float *__restrict__ out) {
  const bool vec = aligned16(out) && L.k % 4 == 0;
  const uint32_t lane = threadIdx.x % kWave, r0 = lane / 16, c = lane % 16;
  for_tiles(L.n16 / 16, L.blocks_per_stripe(),
            [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t *src = reinterpret_cast<const uint32_t *>(tiles) + index * 256 +
                          (r0 + 16 * (c / 4)) * 4 + c % 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t p = stripe * 16 + r0 + 4 * i, n = canonical_row(p, L.n, L.gate);
      if (n < L.n) {
        const uint32_t v = src[16 * i];
        const float s = scales[p];
        f32x4 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[e] = e4m3_to_f32((v >> (8 * e)) & 0xffu) * s;
        }
        store_row4(out + n * L.k, unit * 64 + 4 * c, L.k, vec, f);
      }
    }
  });
}

// ---------------------------------------------------------------- AQ4 g128
// A lane's four dwords j of tile (T, g) hold columns 128 g + 32 j + 8 (l / 16)
// .. + 7 of its row, so a group's 128 columns lie in the four lanes of a row.

__global__ __launch_bounds__(kBlock) void aq4_quantize_kernel(
    const float *__restrict__ w, Aq4Layout L, uint32_t *__restrict__ tiles,
    uint32_t *__restrict__ sz) {
  for_tiles(L.n16 / 16, L.groups, [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t lane = threadIdx.x % kWave;
    const uint64_t n = canonical_row(stripe * 16 + lane % 16, L.n, L.gate);
    const bool live = n < L.n;
    const float *src = w + (live ? n : 0) * L.k + unit * 128 + 8 * (lane / 16);
    const bool vec = aligned16(w);
    float v[4][8];
    float lo = 0.0f, hi = 0.0f;  // set by the first element
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 f;
        if (vec) {
          f = *reinterpret_cast<const f32x4 *>(src + 32 * j + 4 * h);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f[e] = src[32 * j + 4 * h + e];
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[j][4 * h + e] = f[e];
          lo = j + h + e == 0 ? f[e] : fminf(lo, f[e]);
          hi = j + h + e == 0 ? f[e] : fmaxf(hi, f[e]);
        }
      }
    }
#pragma unroll
    for (int off = 16; off <= 32; off *= 2) {
      lo = fminf(lo, __shfl_xor(lo, off, kWave));
      hi = fmaxf(hi, __shfl_xor(hi, off, kWave));
    }
    uint16_t s16 = f32_to_f16((hi - lo) / 15.0f);
    float sf = f16_to_f32(s16);
    uint16_t z16 = sf != 0.0f ? f32_to_f16(-lo / sf) : uint16_t(0);
    if (sf == 0.0f || !__builtin_isfinite(f16_to_f32(z16))) {
      s16 = 0x3c00u;  // 1.0
      z16 = f32_to_f16(-lo);
      sf = 1.0f;
    }
    const float zf = f16_to_f32(z16);
    u32x4 out = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float u = fminf(fmaxf(__builtin_rintf(v[j][e] / sf + zf), 0.0f), 15.0f);
        out[j] |= uint32_t(u) << (4 * aq4_nibble_pos(e));
      }
    }
    reinterpret_cast<u32x4 *>(tiles)[index * kWave + lane] =
        live ? out : u32x4{0u, 0u, 0u, 0u};
    if (lane < 16) {
      sz[index * 16 + lane] = live ? uint32_t(s16) | (uint32_t(z16) << 16) : 0u;
    }
  });
}

// Nibbles of a canonical word (code t at nibble t) to a device word (code t
// at nibble aq4_nibble_pos(t)) and back.
__device__ __forceinline__ uint32_t aq4_to_device(uint32_t w) {
  uint32_t r = 0;
#pragma unroll
  for (uint32_t t = 0; t < 8; ++t) {
    r |= ((w >> (4 * t)) & 0xfu) << (4 * aq4_nibble_pos(t));
  }
  return r;
}
__device__ __forceinline__ uint32_t aq4_to_canonical(uint32_t w) {
  uint32_t r = 0;
#pragma unroll
  for (uint32_t t = 0; t < 8; ++t) {
    r |= ((w >> (4 * aq4_nibble_pos(t))) & 0xfu) << (4 * t);
  }
  return r;
}

__global__ __launch_bounds__(kBlock) void aq4_pack_kernel(
    const uint32_t *__restrict__ packed, const uint16_t *__restrict__ scales,
    const uint16_t *__restrict__ zeros, Aq4Layout L,
    uint32_t *__restrict__ tiles, uint32_t *__restrict__ sz) {
  for_tiles(L.n16 / 16, L.groups, [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t lane = threadIdx.x % kWave;
    const uint64_t n = canonical_row(stripe * 16 + lane % 16, L.n, L.gate);
    const bool live = n < L.n;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (live) {
      const uint32_t *src = packed + n * (L.k / 8) + unit * 16 + lane / 16;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = aq4_to_device(src[4 * j]);
      }
    }
    reinterpret_cast<u32x4 *>(tiles)[index * kWave + lane] = v;
    if (lane < 16) {
      const uint64_t si = n * L.groups + unit;
      sz[index * 16 + lane] =
          live ? uint32_t(scales[si]) | (uint32_t(zeros[si]) << 16) : 0u;
    }
  });
}

__global__ __launch_bounds__(kBlock) void aq4_export_kernel(
    const uint32_t *__restrict__ tiles, const uint32_t *__restrict__ sz,
    Aq4Layout L, uint32_t *__restrict__ packed, uint16_t *__restrict__ scales,
    uint16_t *__restrict__ zeros) {
  for_tiles(L.n16 / 16, L.groups, [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t lane = threadIdx.x % kWave;
    const uint64_t n = canonical_row(stripe * 16 + lane % 16, L.n, L.gate);
    if (n >= L.n) {
      return;
    }
    const u32x4 v = reinterpret_cast<const u32x4 *>(tiles)[index * kWave + lane];
    uint32_t *dst = packed + n * (L.k / 8) + unit * 16 + lane / 16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dst[4 * j] = aq4_to_canonical(v[j]);
    }
    if (lane < 16) {
      const uint32_t z = sz[index * 16 + lane];
      scales[n * L.groups + unit] = uint16_t(z & 0xffffu);
      zeros[n * L.groups + unit] = uint16_t(z >> 16);
    }
  });
}

__global__ __launch_bounds__(kBlock) void aq4_dequant_kernel(
    const uint32_t *__restrict__ tiles, const uint32_t *__restrict__ sz,
    Aq4Layout L, float *__restrict__ out) {
  // Two rows x 32 lanes an instruction: lane c of a row decodes half h = c % 2
  // of the word of columns 8 (c / 2) .. + 7.
  const bool vec = aligned16(out);
  const uint32_t lane = threadIdx.x % kWave, r0 = lane / 32, c = lane % 32;
  const uint32_t q4 = (c / 2) % 4, j = c / 8, h = c % 2;
  for_tiles(L.n16 / 16, L.groups, [&](uint64_t index, uint64_t stripe, uint64_t unit) {
    const uint32_t *src = tiles + index * 256 + (r0 + 16 * q4) * 4 + j;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint64_t n = canonical_row(stripe * 16 + r0 + 2 * i, L.n, L.gate);
      if (n < L.n) {
        const uint32_t v = src[8 * i] >> (8 * h);  // codes 4 h, 4 h + 2: nibbles 2 h, 2 h + 1
        const uint32_t z = sz[index * 16 + r0 + 2 * i];
        const float sf = f16_to_f32(uint16_t(z & 0xffffu));
        const float zf = f16_to_f32(uint16_t(z >> 16));
        f32x4 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[e] = (float((v >> (4 * aq4_nibble_pos(e))) & 0xfu) - zf) * sf;
        }
        store_row4(out + n * L.k, unit * 128 + 4 * c, L.k, vec, f);
      }
    }
  });
}

// ------------------------------------------------------ activation quant
// Optional fused addend: the quantized activations are x + b, each element
// the fp32 sum of the two bf16 values rounded to bf16 (round to nearest
// even), also written to `sum` when it is not null (`sum` may be x or b
// itself: every element is read before the same thread writes it).
struct AddIn {
  const uint16_t *b = nullptr;  // null: no addend
  uint64_t ldb = 0;
  uint16_t *sum = nullptr;
  uint64_t lds = 0;
};

__device__ __forceinline__ uint16_t add_bf16(uint16_t x, uint16_t y) {
  return f32_to_bf16(bf16_to_f32(x) + bf16_to_f32(y));
}

// One workgroup per token row: a = max|x| / 448, xq = e4m3(x / a).
template <bool ADD>
__global__ __launch_bounds__(kBlock) void act_quant_kernel(
    const uint16_t *x, uint64_t ldx, uint64_t k, uint8_t *__restrict__ xq,
    float *__restrict__ xs, AddIn add) {
  __shared__ float red[kBlock / kWave];
  const uint64_t row = blockIdx.x;
  const uint16_t *src = x + row * ldx;
  const uint16_t *bsrc = ADD ? add.b + row * add.ldb : nullptr;
  uint16_t *sdst = ADD && add.sum != nullptr ? add.sum + row * add.lds : nullptr;
  float amax = 0.0f;
  for (uint64_t c = threadIdx.x; c < k; c += kBlock) {
    uint16_t h = src[c];
    if constexpr (ADD) {
      h = add_bf16(h, bsrc[c]);
      if (sdst != nullptr) {
        sdst[c] = h;
      }
    }
    amax = fmaxf(amax, fabsf(bf16_to_f32(h)));
  }
  amax = block_max(amax, red);
  const float a = amax / 448.0f;
  if (threadIdx.x == 0) {
    xs[row] = a;
  }
  for (uint64_t c = threadIdx.x; c < k; c += kBlock) {
    // The sum written above is read back (it may have replaced x or b);
    // without a sum output it is formed again.
    const uint16_t h = !ADD ? src[c] : sdst != nullptr ? sdst[c] : add_bf16(src[c], bsrc[c]);
    const uint32_t q = a == 0.0f ? 0u : f32_to_e4m3(bf16_to_f32(h) / a);
    xq[row * k + c] = static_cast<uint8_t>(q);
  }
}

// Vectorized activation quantization for 16-byte aligned rows with K a
// multiple of 8: each thread keeps CH chunks of 8 bf16 of its row in
// registers (one 16-byte load each), so the row is read once, and writes 8
// codes per store.  The per-element arithmetic is that of act_quant_kernel.
// Workgroups of 256 threads, or 512 with the residual add (two input
// streams): measured on MI355X at M = 2048, K = 4096, the plain quantize
// takes 7.4 us with 256 threads against 8.3 with 512 and 8.1 with 128; the
// fused add 14.0 us with 512 against 14.8 with 256.
constexpr int kAddBlock = 512;
template <int CH, bool ADD>
__global__ __launch_bounds__(ADD ? kAddBlock : kBlock) void act_quant_vec_kernel(
    const uint16_t *x, uint64_t ldx, uint64_t k, uint8_t *__restrict__ xq,
    float *__restrict__ xs, AddIn add) {
  constexpr int kT = ADD ? kAddBlock : kBlock;
  __shared__ float red[kT / kWave];
  const uint64_t row = blockIdx.x;
  const uint16_t *src = x + row * ldx;
  u32x4 v[CH];
  // Row maximum of the bf16 magnitudes as integers: for non-NaN values the
  // bit order is the value order, and any inf or NaN shows as >= 0x7f80.
  u16x2 mx = {0, 0};
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint64_t idx = (uint64_t(c) * kT + threadIdx.x) * 8;
    v[c] = idx < k ? *reinterpret_cast<const u32x4 *>(src + idx)
                   : u32x4{0u, 0u, 0u, 0u};
    if constexpr (ADD) {
      if (idx < k) {
        const u32x4 b = *reinterpret_cast<const u32x4 *>(add.b + row * add.ldb + idx);
        u32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          r[e] = f32x2_to_bf16x2(bits_f32(v[c][e] << 16) + bits_f32(b[e] << 16),
                                 bits_f32(v[c][e] & 0xffff0000u) +
                                     bits_f32(b[e] & 0xffff0000u));
        }
        v[c] = r;
        if (add.sum != nullptr) {
          *reinterpret_cast<u32x4 *>(add.sum + row * add.lds + idx) = r;
        }
      }
    }
    const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      mx = __builtin_elementwise_max(
          mx, __builtin_bit_cast(u16x2, w[e] & 0x7fff7fffu));
    }
  }
  const uint32_t mb = mx.x > mx.y ? mx.x : mx.y;
  float amax = block_max<kT>(mb >= 0x7f80u ? __builtin_inff() : bits_f32(mb << 16), red);
  const bool finite = amax != __builtin_inff();
  if (!finite) {
    // A row holding inf or NaN: max|x| over the non-NaN values, as fmaxf.
    __syncthreads();
    float am = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        am = fmaxf(am, fabsf(bf16_to_f32(uint16_t(w[e] & 0xffffu))));
        am = fmaxf(am, fabsf(bf16_to_f32(uint16_t(w[e] >> 16))));
      }
    }
    amax = block_max<kT>(am, red);
  }
  const float a = amax / 448.0f;
  if (threadIdx.x == 0) {
    xs[row] = a;
  }
  // x / a through the row's reciprocal: q0 = x * r, then one residual step
  // q = q0 + (x - q0 a) r with fused multiply-adds (r = 1 / a correctly
  // rounded, once per row).  For a >= 2^-100 this gives the same E4M3 code
  // as the correctly rounded quotient for every bf16 x with |x| <= max|x|:
  // checked exhaustively over every finite bf16 row maximum and every such
  // x (tests/test_act_quant_division.py).  The quotients that differ in the
  // last fp32 bit lie far below the smallest E4M3 code, and an exact zero
  // keeps its sign (q0).  Rows with a smaller scale divide.
  const float rcp = 1.0f / a;
  const bool via_rcp = a >= 0x1p-100f;
  auto quot = [&](float x) {
    if (!via_rcp) {
      return x / a;
    }
    const float q0 = x * rcp;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, a, x), rcp, q0);
    return q0 == 0.0f ? q0 : q1;
  };
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint64_t idx = (uint64_t(c) * kT + threadIdx.x) * 8;
    if (idx < k) {
      const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
      uint32_t out[2] = {0u, 0u};
      if (finite && a != 0.0f) {
        // Every quotient is finite with |x / a| <= 448 (one rounding of
        // 448 at most above it), where the hardware E4M3 convert rounds to
        // nearest even exactly like f32_to_e4m3; scale 1.0 leaves it plain.
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          float f[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t ww = w[2 * d + e / 2];
            f[e] = quot(bf16_to_f32(uint16_t(e % 2 ? ww >> 16 : ww & 0xffffu)));
          }
          s16x2 r = {0, 0};
          r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, f[0], f[1], 1.0f, false);
          r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, f[2], f[3], 1.0f, true);
          out[d] = __builtin_bit_cast(uint32_t, r);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint16_t h = uint16_t(e % 2 ? w[e / 2] >> 16 : w[e / 2] & 0xffffu);
          const uint32_t q = a == 0.0f ? 0u : f32_to_e4m3(bf16_to_f32(h) / a);
          out[e / 4] |= q << (8 * (e % 4));
        }
      }
      *reinterpret_cast<u32x2 *>(xq + row * k + idx) = u32x2{out[0], out[1]};
    }
  }
}

// Workgroups of one wave per tile.
unsigned tile_grid(uint64_t tiles) {
  constexpr uint64_t per = kBlock / kWave;
  return static_cast<unsigned>(std::min<uint64_t>((tiles + per - 1) / per, kMaxTileBlocks));
}

}  // namespace

hipError_t launch_fp8_quantize(const float *w, const Fp8Layout &L,
                               uint8_t *tiles, float *scales, hipStream_t s) {
  const uint64_t u = L.blocks_per_stripe();
  const dim3 grid(static_cast<unsigned>((L.n16 / 16 + 7) / 8 * 32));
  auto launch = [&](auto kernel, unsigned waves) {
    hipLaunchKernelGGL(kernel, grid, dim3(waves * kWave), 0, s, w, L, tiles, scales);
    return hipGetLastError();
  };
  return u <= 16    ? launch(fp8_quantize_kernel<4, 4>, 4)
         : u <= 32  ? launch(fp8_quantize_kernel<4, 8>, 4)
         : u <= 64  ? launch(fp8_quantize_kernel<4, 16>, 4)
         : u <= 128 ? launch(fp8_quantize_kernel<8, 16>, 8)
         : u <= 256 ? launch(fp8_quantize_kernel<8, 32>, 8)
                    : launch(fp8_quantize_kernel<8, 0>, 8);
}

hipError_t launch_fp8_pack(const uint8_t *q, const float *scales_in,
                           const Fp8Layout &L, uint8_t *tiles, float *scales,
                           hipStream_t s) {
  hipLaunchKernelGGL(fp8_pack_kernel, dim3(tile_grid(L.bytes() / 1024)), dim3(kBlock),
                     0, s, q, scales_in, L, tiles, scales);
  return hipGetLastError();
}

hipError_t launch_fp8_export(const uint8_t *tiles, const float *scales,
                             const Fp8Layout &L, uint8_t *q, float *s_out,
                             hipStream_t s) {
  hipLaunchKernelGGL(fp8_export_kernel, dim3(tile_grid(L.bytes() / 1024)),
                     dim3(kBlock), 0, s, tiles, scales, L, q, s_out);
  return hipGetLastError();
}

hipError_t launch_fp8_dequant(const uint8_t *tiles, const float *scales,
                              const Fp8Layout &L, float *out, hipStream_t s) {
  hipLaunchKernelGGL(fp8_dequant_kernel, dim3(tile_grid(L.bytes() / 1024)),
                     dim3(kBlock), 0, s, tiles, scales, L, out);
  return hipGetLastError();
}

hipError_t launch_aq4_quantize(const float *w, const Aq4Layout &L,
                               uint32_t *tiles, uint32_t *sz, hipStream_t s) {
  hipLaunchKernelGGL(aq4_quantize_kernel, dim3(tile_grid(L.words() / 256)), dim3(kBlock),
                     0, s, w, L, tiles, sz);
  return hipGetLastError();
}

hipError_t launch_aq4_pack(const uint32_t *packed, const uint16_t *scales,
                           const uint16_t *zeros, const Aq4Layout &L,
                           uint32_t *tiles, uint32_t *sz, hipStream_t s) {
  hipLaunchKernelGGL(aq4_pack_kernel, dim3(tile_grid(L.words() / 256)),
                     dim3(kBlock), 0, s, packed, scales, zeros, L, tiles, sz);
  return hipGetLastError();
}

hipError_t launch_aq4_export(const uint32_t *tiles, const uint32_t *sz,
                             const Aq4Layout &L, uint32_t *packed,
                             uint16_t *scales, uint16_t *zeros, hipStream_t s) {
  hipLaunchKernelGGL(aq4_export_kernel, dim3(tile_grid(L.words() / 256)),
                     dim3(kBlock), 0, s, tiles, sz, L, packed, scales, zeros);
  return hipGetLastError();
}

hipError_t launch_aq4_dequant(const uint32_t *tiles, const uint32_t *sz,
                              const Aq4Layout &L, float *out, hipStream_t s) {
  hipLaunchKernelGGL(aq4_dequant_kernel, dim3(tile_grid(L.words() / 256)),
                     dim3(kBlock), 0, s, tiles, sz, L, out);
  return hipGetLastError();
}

namespace {

template <bool ADD>
hipError_t launch_act_quant_t(const uint16_t *x, uint64_t ldx, uint64_t m,
                              uint64_t k, uint8_t *xq, float *xs,
                              const AddIn &add, hipStream_t s) {
  auto a16 = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  bool vec = a16(x) && ldx % 8 == 0 && k % 8 == 0 &&
             reinterpret_cast<uintptr_t>(xq) % 8 == 0;
  if (ADD) {
    vec = vec && a16(add.b) && add.ldb % 8 == 0 &&
          (add.sum == nullptr || (a16(add.sum) && add.lds % 8 == 0));
  }
  const int threads = ADD ? kAddBlock : kBlock;
  const uint64_t chunks = (k / 8 + threads - 1) / threads;  // per thread
  if (vec && chunks <= 8) {
    auto kernel = chunks <= 1   ? act_quant_vec_kernel<1, ADD>
                  : chunks <= 2 ? act_quant_vec_kernel<2, ADD>
                  : chunks <= 4 ? act_quant_vec_kernel<4, ADD>
                                : act_quant_vec_kernel<8, ADD>;
    hipLaunchKernelGGL(kernel, dim3(m), dim3(threads), 0, s, x, ldx, k, xq, xs, add);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(act_quant_kernel<ADD>, dim3(m), dim3(kBlock), 0, s, x, ldx,
                     k, xq, xs, add);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_act_quant(const uint16_t *x, uint64_t ldx, uint64_t m,
                            uint64_t k, uint8_t *xq, float *xs, hipStream_t s) {
  return launch_act_quant_t<false>(x, ldx, m, k, xq, xs, AddIn{}, s);
}

hipError_t launch_add_act_quant(const uint16_t *x, uint64_t ldx,
                                const uint16_t *b, uint64_t ldb, uint16_t *sum,
                                uint64_t lds, uint64_t m, uint64_t k,
                                uint8_t *xq, float *xs, hipStream_t s) {
  AddIn add;
  add.b = b;
  add.ldb = ldb;
  add.sum = sum;
  add.lds = lds;
  return launch_act_quant_t<true>(x, ldx, m, k, xq, xs, add, s);
}

}  // namespace ullm
