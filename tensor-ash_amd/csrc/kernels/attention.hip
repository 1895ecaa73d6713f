// Fused causal prefill attention for gfx950 (the reference's
// run_flash_attention: src/executor/elementwise/flash.rs:13-250,
// shaders/attention_flash_kernel.glsl).  out = softmax_causal(q K^T *
// scale) V in one launch with an online softmax; score tiles stay in
// registers and tiles past a workgroup's causal frontier are never read.
//
// Work split.  A workgroup is QB*KP waves over 32*QB query rows of one
// head: wave w takes query block w % QB (32 rows) and key part w / QB (32
// keys) of every 32*KP-key tile, keeping its own running max / sum /
// output; the KP key parts of a query block merge through LDS at the end,
// in part order.  QB = 2 (64-row tiles).  Head dim 64: KP = 4 (8 waves;
// each wave's walk over the keys is half as long as with 2 parts: 10%
// faster on a 512-token prompt; 32-row tiles with 4 parts, twice the
// workgroups, were 10-20% slower).  Head dim 128: KP = 2 (a 128-key f32
// K/V tile would take 128 KiB of LDS).
//
// Operands (all v_mfma_f32_32x32x2_f32, f32 in f32 accumulate, so f16
// caches widen exactly and the result is f32-accurate):
//  * scores are computed transposed, S^T = K Q^T (m = key, n = query,
//    k = head dim): each lane then owns one query row, so the row max is
//    a register reduction plus one exchange between the lane halves.
//    MFMA step s pairs head-dim lanes s and s + dh/2 (lane half h takes
//    d = s + h*dh/2), so every lane keeps its query row's q values for
//    its half of the head dim in registers;
//  * O^T += V^T P^T (m = head dim, n = query, k = key): in the score
//    accumulator lane (j, h) holds keys 8q + 4h + r at register 4q + r,
//    so step (q, r), which pairs keys 8q + r and 8q + 4 + r, takes its
//    P operand straight from register 4q + r in both lane halves; no
//    data moves between the two products.
// K and V tiles are staged in LDS as [d][key] and [key][d] (the cache
// layouts), so each MFMA operand read is 32 consecutive floats per lane
// half.  Cache rows at or past min(t_max, the workgroup's frontier) are
// staged as zeros, so unwritten cache memory never reaches the sums.
#include "common.h"

#include <type_traits>

namespace {

template <int DH> constexpr int flash_parts() { return ta_flash_parts(DH); }     // KP
template <int DH> constexpr int flash_qblocks() { return ta_flash_qblocks(DH); } // QB
constexpr float kNegMax = -3.402823466e38f;
constexpr float kMasked = -__builtin_inff();
constexpr float kMinScale = 1.17549435e-38f; // 2^-126
// f16-cache kernels: a row's probabilities stay below 2^kSlack and are scaled
// by kProbScale, so that they use the range of their f16 pieces.  (A
// reference point 11 below the maximum would scale them too, but rounds the
// exponents of the largest ones to 2^-21: 2.2e-7 off instead of 1.9e-7.)
constexpr float kSlack = 4.0f, kProbScale = 2048.0f;
// What the first piece of an f32 operand leaves over is scaled by kLowScale
// before it becomes f16, and its products are summed apart.
constexpr float kLowScale = 2048.0f;

template <bool F16> TA_DEVICE void store4(void *base, uint64_t i, f32x4 v) {
  if constexpr (F16) {
    *reinterpret_cast<f16x4 *>(static_cast<_Float16 *>(base) + i) =
        f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  } else {
    *reinterpret_cast<f32x4 *>(static_cast<float *>(base) + i) = v;
  }
}

// (head, query tile) of this workgroup.  Consecutive workgroups go to the 8
// XCDs in turn; with a multiple of 8 heads, all tiles of a head run on one
// XCD (its L2 keeps that head's K/V).  Tiles start longest first over all
// heads of an XCD: the last tile of a causal prompt has q_tiles times the
// first one's keys, and head by head the second half of the heads started
// its longest tiles when the first had drained.  That counts for more than an
// XCD's own heads where 8 does not divide them (us, head by head in one run
// per XCD / longest first; 2048 tokens, dh 128: 12 heads f32 215 / 192, f16
// 52.7 / 45.7; 4 heads 186.5 / 186.9, 30.9 / 31.4).
TA_DEVICE void flash_work(const FlashArgs &p, uint32_t &head, uint32_t &tile) {
  uint32_t i = blockIdx.x, first = 0, count = p.heads;
  if (p.heads % 8u == 0u) {
    count = p.heads >> 3;
    first = (i & 7u) * count;
    i >>= 3;
  }
  head = first + i % count;
  tile = p.q_tiles - 1u - i / count;
}

// Maximum over the two lanes (halves of the wave) that share a query row.
TA_DEVICE float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// One wave's 32 query rows on the f32 MFMAs, for rows whose result is not
// finite: an infinite operand must not meet the zero pieces of a split one
// (inf * 0), so these rows are computed again with whole values, from the
// caches as they lie in memory.  Blocks of 32 keys that some row does not
// attend to in full add their values row by row: a masked probability is a
// zero too.  With an infinite value in every head: 2048 tokens, 32 heads / 8
// KV, dh 128, f16 863 us; 512 tokens at 512, 32 / 8, dh 64, f32 q 211 us (a
// lane per key and column: 15300 and 5200).  Two loops, not a branch in one:
// the joined registers cost the split form a wave per SIMD.
template <int DH, bool IO16>
TA_DEVICE void flash_rows_whole(const FlashArgs &p, uint32_t head, uint32_t kv_head, uint32_t row0,
                                uint32_t lane) {
  constexpr int HALF = DH / 2, DB = DH / 32;
  const uint32_t j = lane & 31u, h = lane >> 5, row = row0 + j;
  const bool live = row < p.t_q;
  const _Float16 *kt = static_cast<const _Float16 *>(p.kt) + (uint64_t)kv_head * DH * p.t_max;
  const _Float16 *vv = static_cast<const _Float16 *>(p.v) + (uint64_t)kv_head * p.t_max * DH;
  const uint32_t keys = min(p.kv_len, p.t_max);
  const uint32_t valid = live ? min(keys, p.pos_base + row + 1u) : 0u;
  const uint32_t any = min(keys, p.pos_base + min(row0 + 32u, p.t_q));
  const uint32_t all = min(keys, p.pos_base + row0 + 1u);
  const uint64_t qbase = (uint64_t)head * p.q_head_stride + (uint64_t)min(row, p.t_q - 1u) * p.q_row_stride;
  const float scale2 = p.scale * 1.44269504088896340736f;
  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    o[b] = f32x16{};
  float m_run = kNegMax, l_run = 0.0f;
  f32x16 s;
  // Register e of s: the probability of key k0 + 4 h + 8 (e / 4) + e % 4.
  auto block = [&](uint32_t k0) __attribute__((always_inline)) {
    s = f32x16{};
    const uint32_t key = min(k0 + j, any - 1u); // keys past the rows' are masked
#pragma unroll 4
    for (uint32_t i = 0; i < (uint32_t)HALF; ++i) {
      const uint32_t d = h * HALF + i;
      const float q = IO16 ? (float)static_cast<const _Float16 *>(p.q)[qbase + d]
                           : static_cast<const float *>(p.q)[qbase + d];
      s = __builtin_amdgcn_mfma_f32_32x32x2f32((float)kt[(uint64_t)d * p.t_max + key], q, s, 0, 0, 0);
    }
    const uint32_t kbase = k0 + 4u * h;
    float m_new = m_run;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = kbase + 8u * (e / 4) + e % 4 < valid ? s[e] * scale2 : kNegMax;
      m_new = fmaxf(m_new, s[e]);
    }
    m_new = fmaxf(m_new, __shfl_xor(m_new, 32));
    const float corr = exp2f(m_run - m_new);
    m_run = m_new;
    float psum = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = kbase + 8u * (e / 4) + e % 4 < valid ? exp2f(s[e] - m_new) : 0.0f;
      psum += s[e];
    }
    l_run = l_run * corr + psum;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        o[b][e] *= corr;
  };
  uint32_t k0 = 0;
  for (; k0 + 32u <= all; k0 += 32u) {
    block(k0);
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
      for (int b = 0; b < DB; ++b)
        o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(
            (float)vv[(uint64_t)(k0 + 4u * h + 8u * (e / 4) + e % 4) * DH + b * 32 + j], s[e], o[b], 0, 0, 0);
  }
  for (; k0 < any; k0 += 32u) {
    block(k0);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float other = __shfl_xor(s[e], 32);
#pragma unroll
      for (uint32_t half = 0; half < 2u; ++half) {
        const uint32_t at = k0 + 4u * half + 8u * (e / 4) + e % 4;
        const float w = half == h ? s[e] : other;
        const _Float16 *v = vv + (uint64_t)min(at, any - 1u) * DH + 4u * h;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f16x4 x = *reinterpret_cast<const f16x4 *>(v + b * 32 + 8 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              o[b][4 * q + r] = at < valid ? fmaf(w, (float)x[r], o[b][4 * q + r]) : o[b][4 * q + r];
          }
      }
    }
  }
  const float l = l_run + __shfl_xor(l_run, 32);
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  if (live) {
    const uint64_t obase = (uint64_t)head * p.o_head_stride + (uint64_t)row * p.o_row_stride + 4u * h;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        store4<IO16>(p.out, obase + b * 32 + 8 * q,
                     f32x4{o[b][4 * q] * inv, o[b][4 * q + 1] * inv, o[b][4 * q + 2] * inv, o[b][4 * q + 3] * inv});
  }
}

template <int DH> TA_DEVICE void flash_body(const FlashArgs &p) {
  constexpr int KP = flash_parts<DH>();  // key parts
  constexpr int QB = flash_qblocks<DH>(); // 32-row query blocks
  constexpr int kBQ = 32 * QB;           // query rows per workgroup
  constexpr int kFlashThreads = 64 * QB * KP;
  constexpr int kBK = 32 * KP;           // keys per tile
  constexpr int KC = kBK / 4;            // four-key chunks per K row
  constexpr int HALF = DH / 2; // MFMA k-steps of the score product
  constexpr int DB = DH / 32;  // 32-row head-dim blocks of the output
  constexpr int REGS = DB * 16 + 2; // merge record per lane: o, m, l
  constexpr int LDS_TILES = 2 * DH * kBK, LDS_MERGE = QB * (KP - 1) * REGS * 64;
  __shared__ float lds[LDS_TILES > LDS_MERGE ? LDS_TILES : LDS_MERGE];
  float *ksh = lds;            // [DH][kBK]
  float *vsh = lds + DH * kBK; // [kBK][DH]

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t qb = wave % QB, kh = wave / QB;
  const uint32_t j = lane & 31u, h = lane >> 5;

  uint32_t head, tile;
  flash_work(p, head, tile);

  const uint32_t q0 = tile * kBQ;
  const uint32_t qrow = q0 + qb * 32u + j;
  const bool live = qrow < p.t_q;
  const uint32_t kv_head = head / p.group_size;
  const uint32_t valid_row = live ? min(p.kv_len, p.pos_base + qrow + 1u) : 0u;
  const uint32_t last_row = min(q0 + (uint32_t)kBQ, p.t_q) - 1u;
  const uint32_t valid_max = min(p.kv_len, p.pos_base + last_row + 1u);
  const uint32_t stage_end = min(valid_max, p.t_max);
  const uint32_t n_tiles = (valid_max + kBK - 1u) / kBK;

  // This lane's q values: Q[qrow][h*HALF + s], s < HALF.
  float qreg[HALF];
  {
    const uint64_t qbase = (uint64_t)head * p.q_head_stride +
                           (uint64_t)min(qrow, p.t_q - 1u) * p.q_row_stride + h * HALF;
#pragma unroll
    for (int s = 0; s < HALF; s += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(p.q) + qbase + s);
      qreg[s] = v[0];
      qreg[s + 1] = v[1];
      qreg[s + 2] = v[2];
      qreg[s + 3] = v[3];
    }
  }

  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    o[b] = f32x16{};
  float m_run = kNegMax, l_run = 0.0f;

  const uint64_t kt_base = (uint64_t)kv_head * DH * p.t_max;
  const uint64_t v_base = (uint64_t)kv_head * p.t_max * DH;
  const bool kt_vec = (p.t_max & 3u) == 0u;

  // K/V of the next tile are loaded into registers while the current one
  // is computed: ksh[d][c] = Kt[d][k0 + c] in KC four-key chunks per row,
  // vsh[r][d] = V[k0 + r][d].
  constexpr int NCH = DH * kBK / 4 / kFlashThreads;
  const float *kt = static_cast<const float *>(p.kt), *vv = static_cast<const float *>(p.v);
  f32x4 kreg[NCH], vreg[NCH];
  auto load_tile = [&](uint32_t k0) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint32_t c = tid + i * kFlashThreads;
      const uint32_t d = c / KC, key = k0 + (c % KC) * 4u;
      const uint64_t src = kt_base + (uint64_t)d * p.t_max + key;
      if (kt_vec && key + 3u < stage_end) {
        kreg[i] = *reinterpret_cast<const f32x4 *>(kt + src);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          kreg[i][e] = key + e < stage_end ? kt[src + e] : 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint32_t c = tid + i * kFlashThreads;
      const uint32_t key = k0 + c / (DH / 4), dc = (c % (DH / 4)) * 4u;
      vreg[i] = key < stage_end ? *reinterpret_cast<const f32x4 *>(vv + v_base + (uint64_t)key * DH + dc) : f32x4{};
    }
  };
  if (n_tiles > 0)
    load_tile(0);

  // Softmax in base 2: scores are scaled by scale * log2(e) once, so each
  // probability is one native exp2.
  const float scale2 = p.scale * 1.44269504088896340736f;

  for (uint32_t t = 0; t < n_tiles; ++t) {
    const uint32_t k0 = t * kBK;
    __syncthreads(); // the previous tile's LDS reads are done
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint32_t c = tid + i * kFlashThreads;
      *reinterpret_cast<f32x4 *>(ksh + (c / KC) * kBK + (c % KC) * 4u) = kreg[i];
      *reinterpret_cast<f32x4 *>(vsh + (c / (DH / 4)) * DH + (c % (DH / 4)) * 4u) = vreg[i];
    }
    __syncthreads();
    if (t + 1 < n_tiles)
      load_tile(k0 + kBK);

    // S^T block: keys kh*32 + m (m < 32) against this wave's 32 queries.
    f32x16 s = f32x16{};
    {
      const float *kp = ksh + h * HALF * kBK + kh * 32u + j;
#pragma unroll
      for (int st = 0; st < HALF; ++st)
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(kp[st * kBK], qreg[st], s, 0, 0, 0);
    }

    // Online softmax over this wave's keys (per query row = per lane pair).
    const uint32_t kbase = k0 + kh * 32u + 4u * h;
    float tmax = kNegMax;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t key = kbase + 8u * q + r;
        const float v = key < valid_row ? s[4 * q + r] * scale2 : kNegMax;
        s[4 * q + r] = v;
        tmax = fmaxf(tmax, v);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m_run, tmax);
    const float corr = exp2f(m_run - m_new);
    float psum = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t key = kbase + 8u * q + r;
        const float pv = key < valid_row ? exp2f(s[4 * q + r] - m_new) : 0.0f;
        s[4 * q + r] = pv;
        psum += pv;
      }
    l_run = l_run * corr + psum;
    m_run = m_new;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        o[b][e] *= corr;

    // O^T += V^T P^T over this wave's 32 keys.
    {
      const float *vp = vsh + (kh * 32u + 4u * h) * DH + j;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(vp[(8 * q + r) * DH + b * 32], s[4 * q + r],
                                                        o[b], 0, 0, 0);
    }
  }

  // Merge the key parts of each query block: parts 1..KP-1 leave their
  // state as [register][lane] records in LDS, part 0 rescales all KP to
  // the common maximum and sums them in part order.
  __syncthreads();
  float *mb = lds + qb * ((KP - 1) * REGS * 64);
  if (kh != 0u) {
    float *rec = mb + (kh - 1u) * (REGS * 64);
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        rec[(b * 16 + e) * 64 + lane] = o[b][e];
    rec[(DB * 16) * 64 + lane] = m_run;
    rec[(DB * 16 + 1) * 64 + lane] = l_run;
  }
  __syncthreads();
  if (kh == 0u) {
    float mp[KP], a[KP];
    mp[0] = m_run;
    float m = m_run;
#pragma unroll
    for (int k = 1; k < KP; ++k) {
      mp[k] = mb[((k - 1) * REGS + DB * 16) * 64 + lane];
      m = fmaxf(m, mp[k]);
    }
    float l = 0.0f;
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      a[k] = exp2f(mp[k] - m);
      const float lk = k == 0 ? l_run : mb[((k - 1) * REGS + DB * 16 + 1) * 64 + lane];
      l = k == 0 ? lk * a[k] : l + lk * a[k];
    }
    l += __shfl_xor(l, 32);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    if (live) {
      const uint64_t obase =
          (uint64_t)head * p.o_head_stride + (uint64_t)qrow * p.o_row_stride + 4u * h;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int e = b * 16 + 4 * q + r;
            float acc = o[b][4 * q + r] * a[0];
#pragma unroll
            for (int k = 1; k < KP; ++k)
              acc += mb[((k - 1) * REGS + e) * 64 + lane] * a[k];
            v[r] = acc * inv;
          }
          store4<false>(p.out, obase + b * 32 + 8 * q, v);
        }
    }
  }
}

// ---------------------------------------------------------------------
// f16 caches: both products on v_mfma_f32_32x32x16_f16 (16 times the f32
// rate), with the f32 operands split into f16 pieces whose products with the
// f16 cache values are exact in the f32 accumulator:
//  * q: as it is when f16; f32 rows are scaled by a power of two (largest
//    value into [2^14, 2^15)) and split into three pieces: exactly down to
//    2^-26 of the row's largest value, to 2^-50 of it below that;
//  * probabilities: two pieces, within 2^-23 of every value down to 2^-23 of
//    the row's largest, and to 2^-47 of that below; the row sum takes the f32
//    values.
// The pieces after the first are scaled by kLowScale and summed apart: in one
// sum they end at f16's smallest step, 2^-36 of a row's largest probability
// and 2^-40 of its largest q, and results that come from keys of 2^-26 alone
// were 8e-4 off (now 6e-7).  Where the registers are there (dh 64; dh 128 with
// f16 q and 64 rows) their sums stay apart to the end: 2048 tokens, 16 / 4
// heads of dh 64 32.9 us (in one sum 32.3), the size below 78 (76).  Else they
// are added tile by tile, 64 FMAs at dh 128 (f32 q 113 us for 106; kept apart
// it spills, 170).
// Measured against f64 (normal inputs): 1.2e-7 .. 2.1e-7 (in one sum 1.5e-7 ..
// 2.7e-7).  An infinite operand would meet zero pieces (inf * 0); rows
// that come out non-finite are computed again by flash_rows_whole.
//
// Layout.  K and V tiles stay in LDS as they lie in the caches ([d][key],
// [key][d]), and both reach the matrix cores through ds_read_b64_tr_b16.
// Scores are computed transposed (m = key, n = query), so a lane owns one
// query row and the PV product takes P straight from the score registers:
// step u pairs registers 8u .. 8u+7 with V rows 16u + 4h + {0..3, 8..11}.
// Tiles arrive by direct global -> LDS loads into two buffers with one
// barrier per tile.  The q registers are pinned before the loop: the
// compiler's own wait for q's loads inside it also waited for the tile in
// flight (112 -> 94 us at the size below).
//
// Split.  Four waves: 2 query blocks x 2 key parts of 32 keys, or 1 x 4
// for short prompts (twice the workgroups, a quarter of the keys per
// wave; ta_flash16_rows).  Tiles of 128 rows x 64 keys were slower (102
// against 94 us): fewer, longer workgroups leave CUs idle at the end.
//
// 2048 tokens, 32 heads / 8 KV, dh 128, f16: 437 us on the f32 MFMAs, 78 us
// here (440 TFLOP/s), kv16 434 -> 113 us; 512 tokens, 4 KV heads, dh 64,
// f16: 28 -> 10.9 us.  MFMAs are busy 32% (kv16 37%) and CUs 75%; a wave's
// scores, softmax and PV product follow each other and overlap only with its
// SIMD's other wave.
template <int DH, bool IO16, bool DIRECT, int QB, int KP, int BKW> struct FlashH16 {
  static constexpr int T = 64 * QB * KP;
  static constexpr int BQ = 32 * QB;         // query rows per workgroup
  static constexpr int BK = KP * BKW;        // keys per tile
  static constexpr int KB = BKW / 32;        // 32-key score blocks per wave
  static constexpr int KS = DH / 16;         // MFMA k-steps of the score product
  static constexpr int DB = DH / 32;         // 32-row head-dim blocks of the output
  static constexpr int QP = IO16 ? 1 : 3;    // f16 pieces of q
  static constexpr int K_BYTES = DH * BK * 2, STAGE = 2 * K_BYTES;
  static constexpr int CK = BK / 8, CV = DH / 8; // 16-byte chunks per K / V row
  static constexpr int LD = K_BYTES / 16 / T;    // direct loads per thread, per operand
  static constexpr int REGS = DB * 16 + 2;       // merge record per lane: o, m, l
  static constexpr int MERGE = QB * (KP - 1) * REGS * 64 * 4;
  static constexpr int SMEM = 2 * STAGE > MERGE ? 2 * STAGE : MERGE;
  static_assert(LD * T * 16 == K_BYTES && CK >= 8 && CV >= 8, "stages split evenly");
  static_assert(SMEM <= 160 * 1024, "LDS");

  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

  static TA_DEVICE uint32_t swz(uint32_t row, int chunks) {
    return chunks >= 16 ? (0xACA60u >> (4u * (row & 3u))) & 15u : 2u * (row & 3u);
  }
  // `base` and `lds` are the same in every lane.
  static TA_DEVICE void load16s(const void *src, uint32_t off, uint32_t lds) {
    const uint64_t a = reinterpret_cast<uint64_t>(src);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const uint64_t base = (uint64_t)lo | (uint64_t)hi << 32;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
                 : "memory", "m0");
  }
  // Two transpose reads: rows r .. r + 3 (`lo`) and r' .. r' + 3 (`hi`) of
  // this lane's column.
  static TA_DEVICE f16x8 tr(uint32_t lo, uint32_t hi) {
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)hi);
    return __builtin_bit_cast(f16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
  }

  static TA_DEVICE void run(const FlashArgs &p) {
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t qb = wave % QB, kh = wave / QB;
    const uint32_t j = lane & 31u, h = lane >> 5;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;

    uint32_t head, tile;
    flash_work(p, head, tile);
    const uint32_t q0 = tile * BQ, qw0 = q0 + qb * 32u, qrow = qw0 + j;
    const bool live = qrow < p.t_q;
    const uint32_t kv_head = head / p.group_size;
    const uint32_t valid_row = live ? min(p.kv_len, p.pos_base + qrow + 1u) : 0u;
    const uint32_t last_row = min(q0 + (uint32_t)BQ, p.t_q) - 1u;
    const uint32_t valid_max = min(p.kv_len, p.pos_base + last_row + 1u);
    const uint32_t stage_end = min(valid_max, p.t_max);
    const uint32_t n_tiles = (valid_max + BK - 1u) / BK;
    // keys every row of this wave attends to / any row of it does
    const uint32_t wave_all = min(p.kv_len, p.pos_base + qw0 + 1u);
    const uint32_t wave_any = qw0 < p.t_q ? min(p.kv_len, p.pos_base + min(qw0 + 32u, p.t_q)) : 0u;

    // This lane's q operand: Q[qrow][16 s + 8 h .. + 7] of every step s.
    f16x8 qf[QP][KS];
    const float s2 = p.scale * 1.44269504088896340736f, sign = s2 < 0.0f ? -1.0f : 1.0f;
    float scale2 = s2 * sign; // the sign goes to q
    {
      const uint64_t qbase = (uint64_t)head * p.q_head_stride +
                             (uint64_t)min(qrow, p.t_q - 1u) * p.q_row_stride + h * 8u;
      if constexpr (IO16) {
#pragma unroll
        for (int s = 0; s < KS; ++s)
          qf[0][s] = *reinterpret_cast<const f16x8 *>(static_cast<const _Float16 *>(p.q) + qbase + 16 * s) *
                     (_Float16)sign;
      } else {
        const float *src = static_cast<const float *>(p.q) + qbase;
        float qmax = 0.0f;
        f32x4 raw[KS][2];
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            raw[s][i] = *reinterpret_cast<const f32x4 *>(src + 16 * s + 4 * i);
#pragma unroll
            for (int c = 0; c < 4; ++c)
              qmax = fmaxf(qmax, fabsf(raw[s][i][c]));
          }
        qmax = fmaxf(qmax, __shfl_xor(qmax, 32));
        // largest |q| of the row into [2^14, 2^15); the factor ends at 2^127,
        // which leaves rows below 2^-112 as exact (f32's denormals end there)
        int e = 15 - __builtin_amdgcn_frexp_expf(qmax);
        e = qmax > 0.0f ? min(e, 127) : 0;
        const float up = ldexpf(sign, e);
        scale2 = scale2 * ldexpf(1.0f, -e);
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            float x = raw[s][i / 4][i % 4] * up;
#pragma unroll
            for (int q = 0; q < QP; ++q) {
              qf[q][s][i] = (_Float16)x;
              x = (x - (float)qf[q][s][i]) * (q == 0 ? kLowScale : 1.0f);
            }
          }
      }
    }

    // A scale that underflows (or 0) keeps every finite score at 0 and a
    // masked one (-inf) at -inf.
    scale2 = scale2 < kMinScale ? kMinScale : scale2;
    // The loads of q end here: the compiler places its waits before the
    // first use, and one inside the loop would also wait for the tile in
    // flight.
#pragma unroll
    for (int q = 0; q < QP; ++q)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        asm volatile("" : "+v"(qf[q][s]));

    // The smaller pieces' sums: kept apart to the end, or added tile by tile
    // where there are no registers for that (the two round alike, not the
    // same: f16 q and the same q in f32 may differ in an f16 result's last bit).
    constexpr bool APART = DH == 64 || (QB == 2 && IO16);
    f32x16 o[DB], o_low[APART ? DB : 1];
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      o[b] = f32x16{};
      if constexpr (APART)
        o_low[b] = f32x16{};
    }
    float m_run = kNegMax, l_run = 0.0f;

    const _Float16 *kt = static_cast<const _Float16 *>(p.kt) + (uint64_t)kv_head * DH * p.t_max;
    const _Float16 *vv = static_cast<const _Float16 *>(p.v) + (uint64_t)kv_head * p.t_max * DH;
    // Stage tile t: K as [d][key], V as [key][d], 16-byte chunks swizzled
    // within a row.  Whole tiles go through a uniform base and fixed lane
    // offsets; a tile that runs past the cache clamps every address (its
    // keys past t_max are masked, its V rows zeroed below).
    uint32_t koff[LD], voff[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const uint32_t q = i * T + tid;
      uint32_t row = q / CK, c = (q % CK) ^ swz(row, CK);
      koff[i] = row * p.t_max + 8u * c;
      row = q / CV, c = (q % CV) ^ swz(row, CV);
      voff[i] = row * DH + 8u * c;
    }
    // K rows that are not whole 16-byte pieces go through registers:
    // fetched before a tile's compute, written to LDS after it.
    f16x8 kreg[DIRECT ? 1 : LD];
    const uint64_t k_left = (uint64_t)(p.heads / p.group_size - kv_head) * DH * p.t_max;
    auto issue = [&](uint32_t t) __attribute__((always_inline)) {
      const uint32_t k0 = t * BK;
      const uint32_t base = __builtin_amdgcn_readfirstlane(lds0 + (t & 1u) * STAGE + wave * 1024u);
      const _Float16 *ks = kt + k0, *vs = vv + (uint64_t)k0 * DH;
      const bool whole = k0 + BK <= p.t_max;
      if constexpr (DIRECT) {
        if (whole) {
#pragma unroll
          for (int i = 0; i < LD; ++i)
            load16s(ks, koff[i] * 2u, base + i * T * 16u);
        } else {
#pragma unroll
          for (int i = 0; i < LD; ++i) {
            const uint32_t row = (i * T + tid) / CK, key = k0 + koff[i] - row * p.t_max;
            load16s(kt, (row * p.t_max + min(key, p.t_max - 8u)) * 2u, base + i * T * 16u);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < LD; ++i) {
          typedef f16x8 f16x8u __attribute__((aligned(2)));
          const uint32_t q = i * T + tid, row = q / CK, c = (q % CK) ^ swz(row, CK);
          const uint64_t at = (uint64_t)row * p.t_max + k0 + 8u * c;
          if (at + 8u <= k_left) {
            kreg[i] = *reinterpret_cast<const f16x8u *>(kt + at);
          } else {
#pragma unroll
            for (int x = 0; x < 8; ++x)
              kreg[i][x] = at + x < k_left ? kt[at + x] : (_Float16)0.0f;
          }
        }
      }
      if (whole) {
#pragma unroll
        for (int i = 0; i < LD; ++i)
          load16s(vs, voff[i] * 2u, base + K_BYTES + i * T * 16u);
      } else {
#pragma unroll
        for (int i = 0; i < LD; ++i) {
          const uint32_t row = (i * T + tid) / CV;
          load16s(vs, (voff[i] + (min(k0 + row, p.t_max - 1u) - k0 - row) * DH) * 2u,
                  base + K_BYTES + i * T * 16u);
        }
      }
    };
    auto commit = [&](uint32_t t) __attribute__((always_inline)) {
      if constexpr (!DIRECT) {
#pragma unroll
        for (int i = 0; i < LD; ++i)
          *reinterpret_cast<f16x8 *>(smem + (t & 1u) * STAGE + (i * T + tid) * 16u) = kreg[i];
      }
    };

    // Per-lane LDS read offsets (transpose reads: group g of 16 lanes, t).
    const uint32_t g = lane >> 4, t16 = lane & 15u;
    uint32_t k_off[KB], v_off[DB];
    {
      const uint32_t row = 8u * (g >> 1) + (t16 >> 2);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const uint32_t col = kh * BKW + kb * 32u + 16u * (g & 1u) + 4u * (t16 & 3u);
        k_off[kb] = row * (BK * 2) + 16u * ((col >> 3) ^ swz(row, CK)) + (col & 7u) * 2u;
      }
      const uint32_t vrow = kh * BKW + 4u * (g >> 1) + (t16 >> 2);
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const uint32_t col = b * 32u + 16u * (g & 1u) + 4u * (t16 & 3u);
        v_off[b] = K_BYTES + vrow * (DH * 2) + 16u * ((col >> 3) ^ swz(vrow, CV)) + (col & 7u) * 2u;
      }
    }

    if (n_tiles > 0) {
      issue(0);
      commit(0);
    }
    for (uint32_t t = 0; t < n_tiles; ++t) {
      const uint32_t k0 = t * BK;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads(); // tile t landed; every wave is done with tile t - 1
      if (t + 1 < n_tiles)
        issue(t + 1);
      if (k0 + BK > stage_end) {
        // rows of V at or past the frontier become zeros (unwritten cache
        // memory may hold anything, and 0 * inf is not 0)
        const uint32_t first = stage_end - min(stage_end, k0);
        char *vs = smem + (t & 1u) * STAGE + K_BYTES;
        for (uint32_t i = first * (DH * 2 / 16) + tid; i < (uint32_t)(BK * DH * 2 / 16); i += T)
          *reinterpret_cast<f32x4 *>(vs + i * 16u) = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        __syncthreads();
      }
      const uint32_t kw0 = k0 + kh * BKW;
      if (kw0 >= wave_any) { // no row of this wave attends to these keys
        if (t + 1 < n_tiles)
          commit(t + 1);
        continue;
      }
      const uint32_t st = lds0 + (t & 1u) * STAGE;

      f32x16 s[KB], low[KB]; // low: the smaller pieces of q
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        s[kb] = low[kb] = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const uint32_t at = st + k_off[kb] + ks * 16 * (BK * 2);
          const f16x8 a = tr(at, at + 4 * (BK * 2));
#pragma unroll
          for (int q = 0; q < QP; ++q) {
            f32x16 &c = q ? low[kb] : s[kb];
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[q][ks], c, 0, 0, 0);
          }
        }
      if constexpr (QP > 1) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            s[kb][e] = fmaf(low[kb][e], 1.0f / kLowScale, s[kb][e]);
      }

      float tmax = kNegMax;
      if (kw0 + BKW > wave_all) {
        const uint32_t kbase = kw0 + 4u * h;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const uint32_t key = kbase + kb * 32u + 8u * (e / 4) + (e % 4);
            s[kb][e] = key < valid_row ? s[kb][e] : kMasked;
          }
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          tmax = fmaxf(tmax, s[kb][e]);
      tmax = fmaxf(half_max(tmax) * scale2, kNegMax);
      // The reference point moves only when a row's maximum has outgrown it
      // by 2^kSlack (probabilities stay below 2^kSlack): with 32 rows in a
      // wave some row finds a new maximum in nearly every tile, and scaling
      // the output for it was a third of the softmax's instructions.
      if (__any(tmax > m_run + kSlack)) {
        const float m_new = fmaxf(m_run, tmax);
        const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= corr;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            o[b][e] *= corr;
            if constexpr (APART)
              o_low[b][e] *= corr;
          }
      }
      float psum = 0.0f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float pv = __builtin_amdgcn_exp2f(fmaf(s[kb][e], scale2, -m_run));
          psum += pv;
          s[kb][e] = pv * kProbScale;
        }
      l_run += psum;

      // O^T += V^T P^T: step u of a 32-key block pairs P registers 8u..8u+7
      // (keys 16u + 4h + 0..3 and 16u + 8 + 4h + 0..3) with the same V rows.
      f16x8 hi[KB][2], lo[KB][2];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
            const float x = s[kb][8 * u + e], y = s[kb][8 * u + e + 1];
            f16x2 a = {(_Float16)x, (_Float16)y};
            asm("" : "+v"(a)); // widen from the packed pair
            hi[kb][u][e] = a[0];
            hi[kb][u][e + 1] = a[1];
            lo[kb][u][e] = (_Float16)fmaf((float)a[0], -kLowScale, x * kLowScale);
            lo[kb][u][e + 1] = (_Float16)fmaf((float)a[1], -kLowScale, y * kLowScale);
          }
      auto v_at = [&](int b, int kb, int u) __attribute__((always_inline)) {
        const uint32_t at = st + v_off[b] + (kb * 32 + u * 16) * (DH * 2);
        return tr(at, at + 8 * (DH * 2));
      };
      if constexpr (APART) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int b = 0; b < DB; ++b) {
              const f16x8 a = v_at(b, kb, u);
              o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, hi[kb][u], o[b], 0, 0, 0);
              o_low[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, lo[kb][u], o_low[b], 0, 0, 0);
            }
      } else {
#pragma unroll
        for (int b = 0; b < DB; ++b) {
          f32x16 low = f32x16{};
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const f16x8 a = v_at(b, kb, u);
              o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, hi[kb][u], o[b], 0, 0, 0);
              low = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, lo[kb][u], low, 0, 0, 0);
            }
#pragma unroll
          for (int e = 0; e < 16; ++e)
            o[b][e] = fmaf(low[e], 1.0f / kLowScale, o[b][e]);
        }
      }
      if (t + 1 < n_tiles)
        commit(t + 1);
    }
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        o[b][e] = (APART ? fmaf(o_low[APART ? b : 0][e], 1.0f / kLowScale, o[b][e]) : o[b][e]) *
                  (1.0f / kProbScale);

    float m = m_run, l = l_run, a0 = 1.0f;
    float mp[KP], a[KP];
    float *mb = reinterpret_cast<float *>(smem) + qb * ((KP - 1) * REGS * 64);
    if constexpr (KP > 1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (kh != 0u) {
        float *rec = mb + (kh - 1u) * (REGS * 64);
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            rec[(b * 16 + e) * 64 + lane] = o[b][e];
        rec[(DB * 16) * 64 + lane] = m_run;
        rec[(DB * 16 + 1) * 64 + lane] = l_run;
      }
      __syncthreads();
      if (kh != 0u)
        return;
#pragma unroll
      for (int k = 1; k < KP; ++k) {
        mp[k] = mb[((k - 1) * REGS + DB * 16) * 64 + lane];
        m = fmaxf(m, mp[k]);
      }
      a0 = __builtin_amdgcn_exp2f(m_run - m);
      l = l_run * a0;
#pragma unroll
      for (int k = 1; k < KP; ++k) {
        a[k] = __builtin_amdgcn_exp2f(mp[k] - m);
        l += mb[((k - 1) * REGS + DB * 16 + 1) * 64 + lane] * a[k];
      }
    }
    l += __shfl_xor(l, 32);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    bool finite = true;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float acc = o[b][e] * a0;
        if constexpr (KP > 1) {
#pragma unroll
          for (int k = 1; k < KP; ++k)
            acc += mb[((k - 1) * REGS + b * 16 + e) * 64 + lane] * a[k];
        }
        o[b][e] = acc * inv;
        finite = finite && __builtin_isfinite(o[b][e]);
      }
    if (live) {
      const uint64_t obase =
          (uint64_t)head * p.o_head_stride + (uint64_t)qrow * p.o_row_stride + 4u * h;
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          store4<IO16>(p.out, obase + b * 32 + 8 * q,
                       f32x4{o[b][4 * q], o[b][4 * q + 1], o[b][4 * q + 2], o[b][4 * q + 3]});
    }
    if (__any(live && !finite))
      flash_rows_whole<DH, IO16>(p, head, kv_head, qw0, lane);
  }
};

} // namespace

#define TA_FLASH(DH)                                                                        \
  extern "C" __global__ __launch_bounds__(ta_flash_threads(DH)) void                         \
  ta_flash_attention_dh##DH(FlashArgs p) {                                                   \
    flash_body<DH>(p);                                                                       \
  }
TA_FLASH(64)
TA_FLASH(128)

// f16 caches (kv16: f32 q/out, io16: f16 q/out): 64-row and 32-row query
// tiles, and `_any` forms for caches whose K rows are not whole 16-byte
// pieces.  At least two waves per SIMD share the registers.
#define TA_FLASH_H16(SYM, DH, IO16, ROWS, DIRECT)                                            \
  extern "C" __global__ __launch_bounds__(256, 2) void SYM(FlashArgs p) {                    \
    FlashH16<DH, IO16, DIRECT, ROWS / 32, 128 / ROWS, 32>::run(p);                           \
  }
#define TA_FLASH_H16_FAMILY(DH, ROWS)                                                        \
  TA_FLASH_H16(ta_flash_attention_kv16_dh##DH##_r##ROWS, DH, false, ROWS, true)              \
  TA_FLASH_H16(ta_flash_attention_kv16_dh##DH##_r##ROWS##_any, DH, false, ROWS, false)       \
  TA_FLASH_H16(ta_flash_attention_io16_dh##DH##_r##ROWS, DH, true, ROWS, true)               \
  TA_FLASH_H16(ta_flash_attention_io16_dh##DH##_r##ROWS##_any, DH, true, ROWS, false)
TA_FLASH_H16_FAMILY(64, 64)
TA_FLASH_H16_FAMILY(64, 32)
TA_FLASH_H16_FAMILY(128, 64)
TA_FLASH_H16_FAMILY(128, 32)
