// Few rows of f32 A on f16 weights, for gfx950 (CDNA4): prompts of up to 64
// tokens, and batches of a few rows, where the weights' bytes are the work.
//
// The arithmetic is the f32 widening of B that smaller shapes always had
// (A is not rounded to f16): A arrives as three exact bf16 pieces in MFMA
// lane order (ta_pack_f32x3), each f16 weight is split in registers into two
// bf16 pieces (8 + 3 bits, exact), and of the six piece products the five
// largest are summed on v_mfma_f32_32x32x16_bf16; the sixth is below 2^-27
// of the product.  A result that is not finite (an infinite operand meets
// zero pieces), or a row with a value that is not exactly its three pieces
// (nonzero below 2^-110), makes its tile compute whole f32 products instead.
//
// Split.  A workgroup owns 32 or 64 rows x 64 columns and a run of 64-deep K
// stages; several share a tile's K so that two workgroups per CU stream
// weights (A's panel comes from the L2), and the last to arrive sums their
// partials in split order (the protocol of gemm_f16.hip's split-K tiles).
// Eight waves: two column blocks x four k-steps of a stage; a wave's chain of
// LDS read, split and products is long, so what counts is how many waves
// take turns (four waves on 128-column tiles, one workgroup per CU: 53 us
// against 41 below).  B is staged as it lies in memory and reaches the
// matrix cores through ds_read_b64_tr_b16; A's pieces are whole KiB.
// Whole f32 products (see above) run on the FP32 MFMAs from operands as they
// lie in memory: every workgroup over its own stages where A's words say so
// before the second stage, the last one over all of K where a sum comes out
// non-finite.  With such a value in every row: 16 x 4096 x 14336 104 us, 24 x
// 3648 x 2816 42 (a dot product per thread: 6800 and 2010).
//
// Kernel time: 16 x 4096 x 14336 41 us = 2.9 TB/s (FP32-MFMA tiles without
// split-K: 1140 us), 24 x 3648 x 2816 17.5 us (217); each op adds a 5 us pack
// unless its A is packed already.  Against f64: 1e-7 (1e-6).
#include "split3.h"

namespace {

template <int FM, int NS, bool ALIGNED> struct GemmW3 {
  static constexpr int BM = 32 * FM, BN = (int)TA_W3_BN, BK = (int)TA_W3_BK, KS = BK / 16;
  static constexpr int W = 8, T = 64 * W, KG = 4; // waves: 2 column blocks x KG k-step groups
  static constexpr int FN = BN / 64;               // column blocks per wave
  static constexpr int A_KB = FM * KS * 3, B_KB = BK * BN * 2 / 1024;
  // Wave loads of 1 KiB per stage; A's may not divide by the waves, then
  // the first A_KB % W waves issue one more.
  static constexpr int A_LD = (A_KB + W - 1) / W, B_LD = B_KB / W, LD = A_LD + B_LD;
  static constexpr int A_MORE = A_KB % W;
  static constexpr int STAGE = (A_KB + B_KB) * 1024, SMEM = NS * STAGE;
  static_assert(B_LD * W == B_KB && KS == KG, "B splits evenly over the waves, one k-step per group");
  static_assert(2 * (KG - 1) * FM * FN * 4096 <= SMEM && SMEM <= 160 * 1024 - 1024, "LDS");
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;

  static constexpr uint32_t CPR = BN / 8; // 16-byte chunks per B row
  static_assert(CPR == 8, "the swizzle separates the 4 rows of a transpose read in 8-chunk rows");
  static TA_DEVICE uint32_t swz(uint32_t row) { return 2u * (row & 3u); }

  static TA_DEVICE void run(const GemmW3Args &q) {
    const GemmArgs &p = q.g;
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];
    constexpr int RW = (BM + 63) / 64;
    __shared__ uint32_t last_flag, whole_sh[RW];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kg = wave >> 1, wn = wave & 1u;
    const uint32_t tn = blockIdx.x % p.tiles_n, tm = blockIdx.x / p.tiles_n;
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t batch = blockIdx.z, split = blockIdx.y, S = p.k_splits;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const uint32_t steps = q.ksteps / KS, per = steps / S, extra = steps % S;
    const uint32_t slo = split * per + min(split, extra);
    const uint32_t kts = per + (split < extra ? 1u : 0u);
    const _Float16 *B = static_cast<const _Float16 *>(p.b) + (uint64_t)batch * p.stride_b;
    const char *A = reinterpret_cast<const char *>(q.pa + batch * q.plane_a);
    constexpr uint32_t STEP = TA_X6_STEP_BYTES;

    // A: load i of wave w is KiB i * W + w of the stage ([row block][step][piece])
    const char *asrc[A_LD];
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      const uint32_t idx = i * W + wave, f = idx / (KS * 3), e = idx % (KS * 3);
      asrc[i] = A + ((uint64_t)(tm * FM + f) * q.ksteps + (uint64_t)slo * KS) * STEP + e * 1024u;
    }
    const uint32_t lo = lane * 16u;
    f16x8 breg[ALIGNED ? 1 : B_LD];
    const uint64_t b_left = (uint64_t)p.k * p.n; // elements of this plane
    auto issue = [&](uint32_t s, uint32_t st) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < A_LD; ++i) {
        if (i * W + W > A_KB && wave >= (uint32_t)A_MORE)
          continue;
        const uint32_t l = lds0 + st * STAGE + (i * W + wave) * 1024u;
        const char *a = asrc[i];
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lo), "s"(a), "s"(l)
                     : "memory", "m0");
        asrc[i] += KS * STEP;
      }
#pragma unroll
      for (int i = 0; i < B_LD; ++i) {
        // rows past K are met by zeros of A
        const uint32_t c16 = i * T + tid, row = c16 / CPR, c = (c16 % CPR) ^ swz(row);
        const uint64_t k = min((slo + s) * (uint32_t)BK + row, p.k - 1u);
        if constexpr (ALIGNED) {
          const char *src =
              reinterpret_cast<const char *>(B + k * p.n + min(n0 + 8u * c, p.n - 8u));
          const uint32_t l = lds0 + st * STAGE + A_KB * 1024u + (i * T + wave * 64u) * 16u;
          asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(l)
                       : "memory", "m0");
        } else {
          typedef f16x8 f16x8u __attribute__((aligned(2)));
          const uint64_t at = k * p.n + n0 + 8u * c; // columns past N reach into the next row
          if (at + 8u <= b_left) {
            breg[i] = *reinterpret_cast<const f16x8u *>(B + at);
          } else {
#pragma unroll
            for (int x = 0; x < 8; ++x)
              breg[i][x] = at + x < b_left ? B[at + x] : (_Float16)0.0f;
          }
        }
      }
    };
    auto commit = [&](uint32_t st) __attribute__((always_inline)) {
      if constexpr (!ALIGNED) {
#pragma unroll
        for (int i = 0; i < B_LD; ++i)
          *reinterpret_cast<f16x8 *>(smem + st * STAGE + A_KB * 1024 + (i * T + tid) * 16u) = breg[i];
      }
    };

    // Transpose-read offsets of this wave's column blocks (k-step 0).
    const uint32_t g = lane >> 4, t16 = lane & 15u;
    const uint32_t brow = 8u * (g >> 1) + (t16 >> 2);
    uint32_t boff[FN];
#pragma unroll
    for (int x = 0; x < FN; ++x) {
      const uint32_t bcol = (wn * FN + x) * 32u + 16u * (g & 1u) + 4u * (t16 & 3u);
      boff[x] = A_KB * 1024u + brow * (BN * 2) + 16u * ((bcol >> 3) ^ swz(brow)) + (bcol & 7u) * 2u;
    }

    f32x16 acc[FM][FN], acc2[FM][FN];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int x = 0; x < FN; ++x)
        acc[f][x] = acc2[f][x] = f32x16{};

    constexpr int AHEAD = ALIGNED ? NS - 1 : 1; // stages in flight
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
      if (s < (int)kts) {
        issue(s, s);
        commit(s);
      }

    // Rows that are not exactly their pieces (while the first stages load):
    // every workgroup of the tile reads the same words and takes whole values.
    bool whole = false;
    for (uint32_t r = tid; r < (uint32_t)BM; r += T) {
      const uint32_t rows = q.blocks_a * 32u;
      const uint32_t *from = q.bits_a + (q.plane_a ? (uint64_t)batch * q.chunks * rows : 0) + m0 + r;
      uint32_t bits = 0;
      for (uint32_t c = 0; c < q.chunks; ++c)
        bits |= from[(uint64_t)c * rows];
      whole = whole || bits != 0u;
    }
    // (the words of the waves that hold rows are read after the first stage's
    // barrier)
    whole = __any(whole);
    if (wave < RW && lane == 0)
      whole_sh[wave] = whole;

    uint32_t st = 0;
    for (uint32_t kt = 0; kt < kts; ++kt) {
      if (ALIGNED && NS > 2 && kt + NS - 2 < kts) {
        if (A_MORE == 0 || wave < (uint32_t)A_MORE)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LD) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * (LD - 1)) : "memory");
      } else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads(); // stage kt landed; every wave is done with stage kt - 1
      if (kt == 0) {
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < RW; ++w)
          any |= whole_sh[w];
        whole = __builtin_amdgcn_readfirstlane(any) != 0u;
        if (whole)
          break;
      }
      const uint32_t ahead = st + AHEAD < NS ? st + AHEAD : st + AHEAD - NS;
      if (kt + AHEAD < kts)
        issue(kt + AHEAD, ahead);
      const uint32_t base = lds0 + st * STAGE;
      {
        const uint32_t ks = kg;
        bf16x8 b[FN][2];
#pragma unroll
        for (int x = 0; x < FN; ++x) {
          const uint32_t at = base + boff[x] + ks * 16u * (BN * 2);
          const s16x4 blo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)at);
          const s16x4 bhi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)(at + 4u * (BN * 2)));
          const f16x8 bh = __builtin_bit_cast(f16x8, __builtin_shufflevector(blo, bhi, 0, 1, 2, 3, 4, 5, 6, 7));
          float w[8];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            w[e] = (float)bh[e];
          split_bf16(w, b[x]);
        }
#pragma unroll
        for (int f = 0; f < FM; ++f) {
          bf16x8 a[3];
#pragma unroll
          for (int c = 0; c < 3; ++c)
            a[c] = *(lds_bf16x8 *)(uintptr_t)(base + lo + ((f * KS + ks) * 3 + c) * 1024u);
          constexpr int PA[5] = {0, 0, 1, 1, 2}, PB[5] = {0, 1, 0, 1, 0};
#pragma unroll
          for (int t = 0; t < 5; ++t)
#pragma unroll
            for (int x = 0; x < FN; ++x) {
              f32x16 &c = t ? acc2[f][x] : acc[f][x];
              c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA[t]], b[x][PB[t]], c, 0, 0, 0);
            }
        }
      }
      if (kt + AHEAD < kts)
        commit(ahead);
      st = st + 1 == NS ? 0 : st + 1;
    }
    // Flat block index from here: block i is rows 32 (i / FN), columns 32 (i % FN)
    // of the wave's part.
    constexpr int NB = FM * FN;
    f32x16 sum[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
      sum[i] = acc[i / FN][i % FN] + acc2[i / FN][i % FN];

    // This wave's part of stages [from, to) in whole f32 products, with A and
    // B as they lie in memory (lane half h takes k = 8 h .. 8 h + 7 of a step).
    const uint32_t lr = lane & 31u, lg = lane >> 5;
    auto whole_stages = [&](uint32_t from, uint32_t to) __attribute__((always_inline)) {
      const float *Af = static_cast<const float *>(p.a) + (uint64_t)batch * p.stride_a;
#pragma unroll
      for (int i = 0; i < NB; ++i)
        sum[i] = f32x16{};
#pragma unroll 2
      for (uint32_t stage = from; stage < to; ++stage) {
        const uint32_t k0 = stage * (uint32_t)BK + kg * 16u + lg * 8u;
        float a[FM][8], b[FN][8];
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
          const uint32_t k = min(k0 + e, p.k - 1u);
          const bool in = k0 + e < p.k;
#pragma unroll
          for (int f = 0; f < FM; ++f) {
            const float v = Af[(uint64_t)min(m0 + f * 32u + lr, p.m - 1u) * p.k + k];
            a[f][e] = in ? v : 0.0f;
          }
#pragma unroll
          for (int x = 0; x < FN; ++x) {
            const float v = (float)B[(uint64_t)k * p.n + min(n0 + (wn * FN + x) * 32u + lr, p.n - 1u)];
            b[x][e] = in ? v : 0.0f;
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int i = 0; i < NB; ++i)
            sum[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i / FN][e], b[i % FN][e], sum[i], 0, 0, 0);
      }
    };
    // The k-step groups meet in LDS, in group order; waves 0 and 1 go on.
    float *red = reinterpret_cast<float *>(smem);
    auto meet = [&]() __attribute__((always_inline)) {
      if (kg > 0) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            red[(((kg - 1) * 2 + wn) * NB + i) * 1024 + r * 64 + lane] = sum[i][r];
      }
      __syncthreads();
      if (kg == 0) {
#pragma unroll
        for (int k = 1; k < KG; ++k)
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              sum[i][r] += red[(((k - 1) * 2 + wn) * NB + i) * 1024 + r * 64 + lane];
      }
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // loads of a loop that was left
    if (whole)
      whole_stages(slo, slo + kts);
    __syncthreads(); // every wave is done with the stages' LDS
    meet();
    if (S > 1) {
      const uint64_t tile_id = (uint64_t)batch * p.tiles_m * p.tiles_n + blockIdx.x;
      constexpr uint32_t SLOT = NB * 16 * 128; // words of one partial tile
      uint32_t *slots = reinterpret_cast<uint32_t *>(p.partial) + tile_id * S * SLOT;
      if (kg == 0) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float v = sum[i][r];
            __hip_atomic_store(slots + (uint64_t)split * SLOT + (i * 16 + r) * 128 + tid, __float_as_uint(v),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
      }
      // Publication and reads as in gemm_f16.hip's split-K tiles: agent-scope
      // stores completed before the barrier, then the count; the last to
      // arrive reads the partials after the count's result.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      uint32_t *counter = p.counters + tile_id * TA_GEMV_COUNTER_STRIDE;
      if (tid == 0)
        last_flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
      __syncthreads();
      if (!last_flag)
        return;
      if (tid == 0)
        __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (kg == 0) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          // in split order, four splits' loads in flight at a time
          f32x16 tot = f32x16{};
          for (uint32_t j0 = 0; j0 < S; j0 += 4u) {
            uint32_t w[4][16];
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j)
#pragma unroll
              for (int r = 0; r < 16; ++r)
                w[j][r] = __hip_atomic_load(slots + (uint64_t)min(j0 + j, S - 1u) * SLOT + (i * 16 + r) * 128 + tid,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j)
              if (j0 + j < S) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                  tot[r] += __uint_as_float(w[j][r]);
              }
          }
          sum[i] = tot;
        }
      }
    }
    // Lane l holds column l % 32 of its block, register r row 8 * (r / 4) + 4 *
    // (l / 32) + r % 4.
    auto row_of = [&](int i, int r) { return m0 + (i / FN) * 32u + 8u * (r / 4) + 4u * (lane >> 5) + (r % 4); };
    auto col_of = [&](int i) { return n0 + (wn * FN + i % FN) * 32u + (lane & 31u); };
    // An infinite weight or a sum past f32: this workgroup computes the tile
    // again, over all of K.
    if (!whole) {
      bool wrong = false;
      if (kg == 0) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            wrong = wrong || (row_of(i, r) < p.m && col_of(i) < p.n && !__builtin_isfinite(sum[i][r]));
      }
      if (__syncthreads_or(wrong)) {
        whole_stages(0, steps);
        meet();
      }
    }
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (row_of(i, r) < p.m && col_of(i) < p.n) {
            const uint64_t at = (uint64_t)batch * p.stride_c + (uint64_t)row_of(i, r) * p.n + col_of(i);
            p.c[at] = ta_epilogue(sum[i][r], p, at, col_of(i), batch);
          }
    }
  }
};

} // namespace

#define TA_GEMM_W3(ROWS, NS)                                                                  \
  extern "C" __global__ __launch_bounds__(512, 4) void ta_gemm_f16w3_r##ROWS(GemmW3Args p) {     \
    GemmW3<ROWS / 32, NS, true>::run(p);                                                      \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(512, 4) void ta_gemm_f16w3_r##ROWS##_any(GemmW3Args p) { \
    GemmW3<ROWS / 32, NS, false>::run(p);                                                     \
  }
TA_GEMM_W3(32, 3)
TA_GEMM_W3(64, 2)
