// f32 values as three bf16 pieces, and the pack that writes an f32 operand
// as pieces in MFMA lane order (see gemm_f32x6.hip for the arithmetic).
#pragma once
#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// x = out[0] + ... + out[P - 1] + what is left over, each piece rounded to
// nearest.  P = 3 leaves nothing from 2^-110 up to the largest bf16, whose
// lowest bits end at bf16's smallest denormal (smaller values leave nothing
// when their lower bits are zeros; infinities and NaN leave NaN).  Returns
// the OR of the eight remainders' bits: zero if all are +0.
template <int P> TA_DEVICE uint32_t split_bf16(const float (&x)[8], bf16x8 (&out)[P]) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    r[i] = x[i];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      bf16x2 a = {(__bf16)r[i], (__bf16)r[i + 1]};
      asm("" : "+v"(a)); // widen from the packed pair
      out[p][i] = a[0];
      out[p][i + 1] = a[1];
      const uint32_t w = __builtin_bit_cast(uint32_t, a);
      r[i] -= __uint_as_float(w << 16);
      r[i + 1] -= __uint_as_float(w & 0xffff0000u);
    }
  uint32_t left = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    left |= __float_as_uint(r[i]);
  return left;
}

// One workgroup of a pack job: four waves of 4 k-steps each.  ROWS: A's 32
// rows (lane = row, k half: 8 consecutive k of a row per step, the row's
// 128-byte lines shared by the wave's steps), else B's 64 columns (lane =
// column, 8 strided k per half step, 256 contiguous bytes per load).
template <bool ROWS> TA_DEVICE void pack_job(const PackX3Job &p, uint32_t group, uint32_t *or_sh) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t per_plane = (ROWS ? p.blocks : p.blocks / 2) * p.chunks;
  const uint32_t plane = group / per_plane, in = group % per_plane;
  const uint32_t blk = in / p.chunks, chunk = in % p.chunks;
  const uint32_t row = ROWS ? blk * 32u + (lane & 31u) : blk * 64u + lane;
  const uint32_t block = ROWS ? blk : blk * 2u + (lane >> 5);
  const bool ok = row < p.rows;
  const float *src = p.src + (uint64_t)plane * p.stride +
                     (ROWS ? (uint64_t)min(row, p.rows - 1u) * p.k : (uint64_t)min(row, p.rows - 1u));
  bf16x8 *dst = reinterpret_cast<bf16x8 *>(p.dst) +
                ((uint64_t)plane * p.blocks + block) * p.ksteps * (TA_X6_STEP_BYTES / 16u);
  const uint32_t step0 = chunk * TA_X6_CHUNK_STEPS + wave * 4u;
  // 8 values of one k half of one step: A: half = lane / 32 of step i;
  // B: half i % 2 of step i / 2 (two trips).
  uint32_t bits = 0;
#pragma unroll
  for (int trip = 0; trip < (ROWS ? 1 : 2); ++trip) {
    float x[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t step = step0 + (ROWS ? i : trip * 2 + i / 2);
      const uint32_t half = ROWS ? lane >> 5 : i % 2;
      const uint32_t k = step * 16u + half * 8u;
      if (ROWS && ok && k + 8u <= p.k && (p.k & 3u) == 0u) {
        const f32x4 u = *reinterpret_cast<const f32x4 *>(src + k);
        const f32x4 v = *reinterpret_cast<const f32x4 *>(src + k + 4u);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[i][e] = u[e];
          x[i][4 + e] = v[e];
        }
      } else {
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e)
          x[i][e] = ok && k + e < p.k ? (ROWS ? src[k + e] : src[(uint64_t)(k + e) * p.rows]) : 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t step = step0 + (ROWS ? i : trip * 2 + i / 2);
      const uint32_t half = ROWS ? lane >> 5 : i % 2;
      if (step < p.ksteps) { // zeros past it
        bf16x8 o[3];
        bits |= split_bf16(x[i], o);
#pragma unroll
        for (int q = 0; q < 3; ++q)
          dst[((uint64_t)step * 3u + q) * 64u + half * 32u + (lane & 31u)] = o[q];
      }
    }
  }
  or_sh[threadIdx.x] = bits;
  __syncthreads();
  if (wave == 0) {
    for (uint32_t w = 1; w < 4; ++w)
      bits |= or_sh[w * 64u + lane];
    if (ROWS) {
      bits |= or_sh[(lane ^ 32u)] | or_sh[64u + (lane ^ 32u)] | or_sh[128u + (lane ^ 32u)] |
              or_sh[192u + (lane ^ 32u)];
      if (lane >= 32u)
        return;
    }
    p.bits[((uint64_t)plane * p.chunks + chunk) * p.blocks * 32u + row] = bits;
  }
}

} // namespace
