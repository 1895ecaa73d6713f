// f32 GEMM on the bf16 matrix cores, for gfx950 (CDNA4).
//
// v_mfma_f32_32x32x16_bf16 runs 16 times as many products per second as the
// FP32 MFMAs.  An f32 value is exactly the sum of three bf16 pieces (8 + 8 +
// 8 significant bits, each rounded to nearest, so |mid| <= 2^-9 |x| and |lo|
// <= 2^-18 |x|), products of pieces are exact in the f32 accumulator, and of
// the nine piece products the six largest are summed:
//   hi hi, hi mid, mid hi, mid mid, hi lo, lo hi.
// The three left out are at most 2^-26 |a b| together, a quarter of the
// rounding of one f32 product: a single product is thus off by up to 1.25
// times that rounding.  Measured against f64 (normal inputs): K =
// 4096 9.0e-7 (256 x 256 tile) and 5.1e-7 (128 x 128), against 1.1e-6 of the
// FP32 MFMAs; K = 777 2e-7 against 5e-7.  Ceiling: a sixth of the bf16 rate.
//
// bf16 has f32's exponent range, so no scaling is needed.  Values that are
// not exactly their three pieces (nonzero below 2^-110, where the lowest bits
// fall under bf16's smallest denormal; past the largest bf16; infinities and
// NaN, whose lower pieces are NaN) send their tiles to the FP32 MFMAs
// (GemmF32) in the same launch: the pack leaves a word per row and column that
// says whether any of its values is one, and a sum that comes out non-finite
// says the same.  A tile of the first kind leaves before its second stage, one
// of the second costs both forms.  With a value of the first kind in every row:
// 4096^3 1414 us, 2048^3 196, 1000^3 91 (split products 770, 104, 32; FP32
// MFMA 965, 188, 50, whose kernel picks its own tile).  Denormals are kept
// throughout by the conversions and the MFMAs.
#include "gemm_f32_tile.h"
#include "split3.h"

namespace {

// BM x BN tile of 16 k-steps' pieces at a time: the waves are G groups of
// WGM x WGN; a stage is G k-steps, group g multiplies step g, and the groups'
// sums meet in LDS at the end, in group order.  Operands are in MFMA lane
// order in memory, so a stage's direct global -> LDS loads and the LDS reads
// are whole contiguous KiB (no swizzle, no bank conflicts), and six products
// share three operand reads: a CU moves 16 B/clk from the L2 and 47 B/clk
// from LDS (256 x 256 tile), a fraction of what either gives.
// TWO: the five smaller products have an accumulator of their own, so the
// large sums take one addition per 16 k instead of six.
template <int BM, int BN, int WGM, int WGN, int G, int NS, bool TWO> struct GemmF32X6 {
  static constexpr int WT = WGM * WGN, W = WT * G, T = 64 * W;
  static constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 32, FN = WTN / 32;
  static constexpr int STEP = (int)TA_X6_STEP_BYTES;
  static constexpr int A_KB = BM / 32 * 3 * G, B_KB = BN / 32 * 3 * G; // KiB per stage
  static constexpr int LD = (A_KB + B_KB) / W;                         // loads per wave and stage
  static constexpr int STAGE = (A_KB + B_KB) * 1024;
  static constexpr int MERGE = (G - 1) * WT * FM * FN * 4096, CSTAGE = WT * 32 * (WTN + 4) * 4;
  static constexpr int SMEM = NS * STAGE;
  static_assert(LD * W == A_KB + B_KB, "stages split evenly over the waves");
  static_assert(MERGE <= SMEM && CSTAGE <= SMEM && SMEM <= 160 * 1024 - 1024, "LDS");
  static_assert(NS >= 2 && (NS - 2) * LD <= 63, "vmcnt range");
  // the FP32 form: 64 x 64 in 4 waves, or pieces of 128 x 128 in 8
  static constexpr int PT = BM == 64 ? 64 : 128, PW = BM == 64 ? 4 : 8;
  typedef GemmF32<PT, PT, 2, PW / 2, false, false, 16> Plain;
  static_assert(Plain::SMEM_FLOATS * 4 <= SMEM, "the FP32 form's LDS fits");
  typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;

  static TA_DEVICE void run(const GemmX6Args &q) {
    const GemmArgs &p = q.g;
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];
    __shared__ uint32_t inexact_sh[W];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kg = wave / WT, w2 = wave % WT, wm = w2 / WGN, wn = w2 % WGN;
    uint32_t tm, tn;
    ta_tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    const uint32_t batch = blockIdx.z;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const char *A = reinterpret_cast<const char *>(q.pa + batch * q.plane_a) +
                    (uint64_t)tm * (BM / 32) * q.ksteps * STEP;
    const char *B = reinterpret_cast<const char *>(q.pb + batch * q.plane_b) +
                    (uint64_t)tn * (BN / 32) * q.ksteps * STEP;
    const uint32_t kts = q.ksteps / G;

    const char *src[LD]; // wave-uniform, advanced per stage
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const uint32_t idx = i * W + wave, e = idx < A_KB ? idx : idx - A_KB;
      src[i] = (idx < A_KB ? A : B) + (uint64_t)(e / (3 * G)) * q.ksteps * STEP + (e % (3 * G)) * 1024;
    }
    const uint32_t lo = lane * 16u;
    auto issue = [&](uint32_t st) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const uint32_t l = lds0 + st * STAGE + (i * W + wave) * 1024u;
        const char *s = src[i];
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lo), "s"(s), "s"(l)
                     : "memory", "m0");
        src[i] += G * STEP;
      }
    };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
      if (s < (int)kts)
        issue(s);

    // Rows and columns that are not exactly their pieces (while the first stages load).
    bool inexact = false;
    {
      const uint32_t ra = q.blocks_a * 32u, rb = q.blocks_b * 32u;
      const uint32_t *ba = q.bits_a + (q.plane_a ? (uint64_t)batch * q.chunks * ra : 0) + tm * BM;
      const uint32_t *bb = q.bits_b + (q.plane_b ? (uint64_t)batch * q.chunks * rb : 0) + tn * BN;
      for (uint32_t r = tid; r < (uint32_t)(BM + BN); r += T) {
        const uint32_t *from = r < (uint32_t)BM ? ba + r : bb + (r - BM);
        const uint32_t step = r < (uint32_t)BM ? ra : rb;
        uint32_t bits = 0;
        for (uint32_t c = 0; c < q.chunks; ++c)
          bits |= from[(uint64_t)c * step];
        inexact = inexact || bits != 0u;
      }
    }
    // (one word per wave, read after the first stage's barrier)
    inexact = __any(inexact);
    if (lane == 0)
      inexact_sh[wave] = inexact;

    f32x16 acc[FM][FN], acc2[TWO ? FM : 1][TWO ? FN : 1];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) {
        acc[f][g] = f32x16{};
        if constexpr (TWO)
          acc2[f][g] = f32x16{};
      }
    uint32_t st = 0, nst = NS - 1;
    for (uint32_t kt = 0; kt < kts; ++kt) {
      if (kt + NS - 2 < kts)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LD) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads(); // stage kt landed; every wave is done with stage kt - 1
      if (kt == 0) {
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < W; ++w)
          any |= inexact_sh[w];
        inexact = __builtin_amdgcn_readfirstlane(any) != 0u;
        if (inexact)
          break;
      }
      if (kt + NS - 1 < kts)
        issue(nst);
      const uint32_t ab = lds0 + st * STAGE + lo + wm * FM * (G * STEP) + kg * STEP;
      const uint32_t bb = lds0 + st * STAGE + A_KB * 1024 + lo + wn * FN * (G * STEP) + kg * STEP;
      bf16x8 a[3][FM], b[3][FN];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int f = 0; f < FM; ++f)
          a[c][f] = *(lds_bf16x8 *)(uintptr_t)(ab + f * (G * STEP) + c * 1024);
#pragma unroll
        for (int g = 0; g < FN; ++g)
          b[c][g] = *(lds_bf16x8 *)(uintptr_t)(bb + g * (G * STEP) + c * 1024);
      }
      constexpr int PA[6] = {0, 0, 1, 1, 0, 2}, PB[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
          for (int g = 0; g < FN; ++g) {
            f32x16 &c = TWO && t > 0 ? acc2[TWO ? f : 0][TWO ? g : 0] : acc[f][g];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA[t]][f], b[PB[t]][g], c, 0, 0, 0);
          }
      st = st + 1 == NS ? 0 : st + 1;
      nst = nst + 1 == NS ? 0 : nst + 1;
    }
    if constexpr (TWO) {
#pragma unroll
      for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int g = 0; g < FN; ++g)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[f][g][r] += acc2[f][g][r];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // loads of a loop that was left
    __syncthreads();
    if constexpr (G > 1) {
      float *red = reinterpret_cast<float *>(smem);
      if (kg > 0) {
#pragma unroll
        for (int f = 0; f < FM * FN; ++f)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            red[(((kg - 1) * WT + w2) * FM * FN + f) * 1024 + r * 64 + lane] = acc[f / FN][f % FN][r];
      }
      __syncthreads();
      if (kg == 0) {
#pragma unroll
        for (int k = 1; k < G; ++k)
#pragma unroll
          for (int f = 0; f < FM * FN; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              acc[f / FN][f % FN][r] += red[(((k - 1) * WT + w2) * FM * FN + f) * 1024 + r * 64 + lane];
      }
    }
    bool whole = inexact;
    if (kg == 0) {
#pragma unroll
      for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int g = 0; g < FN; ++g)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            whole = whole || !__builtin_isfinite(acc[f][g][r]);
    }
    if (__syncthreads_or(whole)) {
      // waves past the FP32 form's leave (a barrier counts the rest)
      if (wave < (uint32_t)PW)
        for (uint32_t m = tm * BM; m < min((tm + 1) * BM, p.m); m += PT)
          for (uint32_t n = tn * BN; n < min((tn + 1) * BN, p.n); n += PT)
            Plain::run_tile(p, reinterpret_cast<float *>(smem), m, n);
      return;
    }
    ta_store_tile<WTM, WTN, FM, FN, 64 * WT, false>(reinterpret_cast<float *>(smem), SMEM / 4, acc, p,
                                                    lane, w2, wm, wn, tm * BM, tn * BN, batch, 0, kg == 0);
  }
};

} // namespace

extern "C" __global__ __launch_bounds__(256) void ta_pack_f32x3(PackX3Args p) {
  __shared__ uint32_t or_sh[256];
  if (blockIdx.x < p.a.groups)
    pack_job<true>(p.a, blockIdx.x, or_sh);
  else
    pack_job<false>(p.b, blockIdx.x - p.a.groups, or_sh);
}

#define TA_GEMM_X6(TILE, WGM, WGN, NS, TWO)                                                   \
  extern "C" __global__ __launch_bounds__(ta_x6_threads(TILE), TILE == 64 ? 4 : 2) void       \
  ta_gemm_f32x6_m##TILE##n##TILE(GemmX6Args p) {                                              \
    typedef GemmF32X6<TILE, TILE, WGM, WGN, (int)ta_x6_groups(TILE), NS, TWO> Gemm;           \
    static_assert(Gemm::T == (int)ta_x6_threads(TILE), "host launch width");                  \
    Gemm::run(p);                                                                             \
  }
TA_GEMM_X6(256, 2, 4, 3, false)
TA_GEMM_X6(128, 2, 2, 3, true)
TA_GEMM_X6(64, 2, 2, 3, true)
