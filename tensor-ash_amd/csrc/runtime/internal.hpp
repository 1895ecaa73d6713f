// Internal declarations of the host runtime (not part of the public API).
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../kernels/kernel_args.h"
#include "tensor_ash.hpp"

namespace tensor_ash {

[[noreturn]] void fail(const std::string &msg);
std::string fmt_shape(const std::vector<uint32_t> &shape); // "[a, b, c]"
void hip_check(hipError_t err, const char *what);

// Every device and pinned-host allocation the library makes goes through
// these two, which count the calls (allocation_count) so a caller can
// check that an entry point allocated nothing.
hipError_t device_malloc(void **ptr, size_t bytes);
hipError_t host_malloc(void **ptr, size_t bytes, unsigned int flags);
uint64_t allocation_count();

struct DeviceBuffer {
  std::shared_ptr<Context> ctx;
  void *ptr = nullptr;
  uint64_t bytes = 0;
  ~DeviceBuffer();
};

// src/matmul/resolution.rs:10-76.
struct MatrixShape {
  uint32_t batch, rows, cols;
  static MatrixShape from_tensor_shape(const std::vector<uint32_t> &shape);
  uint32_t batch_stride(const char *label) const;
};

// src/matmul/resolution.rs:80-442.
struct ResolvedMatmul {
  uint32_t m = 0, n = 0, k = 0, batch = 0;
  uint32_t batch_stride_a = 0, batch_stride_b = 0, batch_stride_c = 0;
  uint64_t total_flops = 0;
  bool b_f16 = false;
  bool a_f16 = false;
  bool packed_b = false;

  static ResolvedMatmul from_shapes(const std::vector<uint32_t> &a,
                                    const std::vector<uint32_t> &b,
                                    const std::vector<uint32_t> &c);
  static ResolvedMatmul from_call(const MatmulCall &call);
  static ResolvedMatmul from_op(const MatmulOp &op);
  void validate_bias_shape(const std::vector<uint32_t> &shape) const;
  void validate_epilogue(const MatmulOp &op) const;
  void validate_normed_a(const MatmulOp &op) const;
  void validate_store(const MatmulOp &op) const;
  bool operator==(const ResolvedMatmul &o) const;
};
uint64_t total_flops(const std::vector<ResolvedMatmul> &resolved);

// Largest rows a decode GEMV launch handles (register-resident X rows).
constexpr uint32_t kGemvMaxRows = 8;

// ---- routing (src/pipeline/mod.rs:293-535, selection.rs:89-172) ----
size_t heuristic_kernel_index(uint32_t cus, uint32_t batch, uint32_t m, uint32_t n, uint32_t k,
                              bool b_f16, bool packed_b, bool a_f16 = false);
bool kernel_supports(const KernelSpec &spec, const ResolvedMatmul &dims);
bool gemm_lds_ok(const ResolvedMatmul &dims);
bool f32_mi16_ok(const ResolvedMatmul &dims, uint32_t tile_m, uint32_t tile_n, uint32_t planes);
uint32_t mi16_threads(uint32_t tile_m);
bool f32_groups_ok(uint32_t cus, const ResolvedMatmul &dims, const KernelSpec &spec, uint32_t planes);
bool f16_dual_tile(const KernelSpec &spec);
std::vector<size_t> tune_candidate_indices(const ResolvedMatmul &dims);
size_t registry_index(const char *name);

// ---- split-K (src/executor/splitk2.rs) ----
constexpr uint32_t kReduceThreads = 256;
constexpr uint64_t kAutoScratchCapBytes = 256ull << 20;
const KernelSpec &splitk_stage1_spec(uint32_t m, uint32_t n, uint32_t k);
uint32_t gemm_threads(const KernelSpec &s);
uint32_t h16sk_splits(uint32_t cus, uint32_t batch, uint32_t m, uint32_t n, uint32_t k,
                      uint32_t tile_m, uint32_t tile_n);
uint32_t splitk_sub_splits(uint32_t cus, const ResolvedMatmul &dims, uint32_t splits);
std::optional<uint32_t> heuristic_splits(uint32_t cus, uint32_t batch, uint32_t m, uint32_t n,
                                         uint32_t k);
uint32_t splitk_reduce_groups(uint32_t cus, uint64_t quads, uint32_t planes);
uint32_t default_num_k_splits(uint32_t cus, uint32_t batch, uint32_t m, uint32_t n, uint32_t k);
bool auto_route_fits(uint32_t batch, uint32_t m, uint32_t n, uint32_t k, uint32_t splits);
void validate_scratch_geometry(uint32_t batch, uint32_t m, uint32_t n, uint32_t k,
                               uint32_t splits);
std::optional<uint64_t> checked_auto_scratch_end(uint64_t offset, uint64_t bytes);

// ---- GEMV geometry ----
// Layout of one f32 op on the split-product route (ta_pack_f32x3 +
// ta_gemm_f32x6_<tile>): packed A, packed B, then their row / column bits,
// in one scratch region of `bytes`.
struct F32X6Plan {
  uint32_t blocks_a, blocks_b, ksteps, chunks;
  uint64_t planes_a, planes_b;
  uint64_t b_off, bits_a_off, bits_b_off, bytes;
};
F32X6Plan f32x6_plan(const ResolvedMatmul &dims, uint32_t tile);
// Tile (256, 128, 64) of the split-product route when it is the faster one
// for this shape, else 0.  `fp32`, `splits`: the route it would replace.
uint32_t f32x6_tile(uint32_t cus, const ResolvedMatmul &dims, const KernelSpec &fp32,
                    std::optional<uint32_t> splits);
constexpr uint64_t kF32X6ScratchCapBytes = 1ull << 30;

// An op of few rows on f16 weights on the split-product route
// (ta_gemm_f16w3_r<rows>): packed A, K splits and scratch.
struct W3Plan {
  uint32_t rows; // 32 or 64 per workgroup
  uint32_t blocks, ksteps, chunks, tiles_m, tiles_n, splits;
  uint64_t planes, bits_off, pack_bytes;
  uint64_t partial_bytes, counters;
};
W3Plan w3_plan(uint32_t cus, const ResolvedMatmul &dims);
bool w3_ok(const ResolvedMatmul &dims);
uint32_t w3_group(const ResolvedMatmul &dims);
constexpr uint64_t kW3ScratchCapBytes = 256ull << 20;

struct GemvPlan {
  uint32_t tw = 64, mr = 1, tiles = 0, kchunk = 0, kchunks = 1;
  uint64_t partial_bytes = 0; // 0 when kchunks == 1
};
uint32_t gemv_unit(uint32_t tw, bool f32_weights, bool dual, uint32_t rows);
GemvPlan plan_gemv(uint32_t cus, uint32_t rows, uint32_t n, uint32_t k, uint32_t tw, bool dual,
                   uint32_t unit);

// ---- copies of A kept within a submission ----
// f16 copies of A that pre-passes (or a dual launch's f16 output copy) of a
// submission left behind: a later f16w GEMM with the same A (same buffer,
// same elements) reuses one unless an op in between wrote that buffer, or
// wrote the split-K region the copy lives in (record() and launch_gemm()
// drop such entries).  Two entries, so a layer that converts x for QKV and
// then the attention output for O still finds x for its up/gate pair.
// Pre-pass copies go to the half of the split-K region the other live copy
// does not use (scratch_need reserves two halves, each as large as the op's
// A).
// A's packed pieces (ta_pack_f32x3) are kept the same way.  An f16 copy has
// A's own order, whatever shape an alias gives the buffer; the pieces lie
// in blocks of 32 rows that start anew in every plane, so they are the same
// only for the same planes of the same rows (n then fixes K).
struct CvtEntry {
  const void *buffer = nullptr;
  const void *src = nullptr;
  uint64_t n = 0;             // elements of A
  void *base = nullptr;       // where the copy lives
  size_t producer = SIZE_MAX; // op whose epilogue wrote it, if any
  int half = -1;              // split-K region half, -1 = elsewhere
  uint64_t planes = 0;        // packed pieces: planes and rows of each;
  uint32_t rows = 0;          // f16 copy: 0
  uint64_t age = 0;
};
struct CvtCache {
  CvtEntry e[2];
  uint64_t clock = 0;
  CvtEntry *find(const void *buffer, const void *src, uint64_t n, uint64_t planes = 0,
                 uint32_t rows = 0) {
    for (auto &x : e)
      if (x.buffer && x.buffer == buffer && x.src == src && x.n == n && x.planes == planes &&
          x.rows == rows)
        return &x;
    return nullptr;
  }
  // The entry to replace: an empty one, else the older.
  CvtEntry &victim() {
    if (!e[0].buffer)
      return e[0];
    if (!e[1].buffer)
      return e[1];
    return e[0].age <= e[1].age ? e[0] : e[1];
  }
  // A copy written at `v.base` replaces whatever entry that memory held
  // (every dual launch writes its f16 output copy to the same scratch).
  void put(CvtEntry &slot, CvtEntry v) {
    for (auto &x : e)
      if (&x != &slot && x.buffer && x.base == v.base)
        x = CvtEntry{};
    v.age = ++clock;
    slot = v;
  }
  // An op wrote `buffer`: copies of it are stale (except the one that
  // op's own epilogue produced).
  void wrote(const void *buffer, size_t op) {
    for (auto &x : e)
      if (x.buffer && x.buffer == buffer && x.producer != op)
        x = CvtEntry{};
  }
  void drop_region() { // the split-K region was overwritten
    for (auto &x : e)
      if (x.half >= 0)
        x = CvtEntry{};
  }
};

// ---- f16w A conversions converted up front ----
// One op of a submission as the paired up-front conversion sees it: its A
// (buffer, device pointer, values converted), whether its route converts A
// to f16, and the buffers it writes.
struct CvtCandidate {
  const void *a_buffer = nullptr;
  const void *a_ptr = nullptr;
  uint64_t n = 0;
  bool converts = false;
  const void *writes[2] = {nullptr, nullptr};
};
// Indices of the ops whose A is converted at submission start: the first
// two distinct A's that take the conversion and that no earlier op writes
// (fewer than two: nothing is paired).
std::vector<size_t> paired_conversion_picks(const std::vector<CvtCandidate> &ops);

// ---- tuner (src/executor/tuning.rs:300-313, pipeline/tuning.rs) ----
std::optional<uint64_t> median(std::vector<uint64_t> samples);
size_t candidate_at(size_t len, uint32_t round, size_t offset);

struct TuneKey {
  uint32_t batch, m, n, k;
  bool b_f16;
  bool operator<(const TuneKey &o) const;
};
struct TuneEntry {
  size_t kernel;
  std::optional<uint32_t> splitk2_splits;
};
// The route a shape takes untuned, as measured: `kernel` as it is, its
// split-product form, or split-K.
struct TuneBase {
  size_t kernel = 0;
  std::optional<uint32_t> splits;
  bool split_products = false;
  std::optional<uint64_t> ns;
};
// What the tuner stores: the untuned route unless a kernel, or a split
// count, is more than 2% faster.  Nothing measured: nothing.
std::optional<TuneEntry> tune_pick(const TuneBase &base,
                                   const std::vector<std::pair<size_t, uint64_t>> &kernels,
                                   const std::vector<std::pair<uint32_t, uint64_t>> &split_counts);
std::string tune_store_path(const Context &ctx);
std::string tune_header_line(const Context &ctx);
std::map<TuneKey, TuneEntry> parse_tune_store(const std::string &text, const std::string &header);
std::string format_tune_store(const std::map<TuneKey, TuneEntry> &map, const std::string &header);

// Fixed device scratch (fixed_scratch.hip): the array's address on
// `device` (the current device), resolved once per device, and the mutex
// that serialises its users on that device.
hipError_t fixed_scratch_address(int device, void **out);
std::mutex &fixed_scratch_mutex(int device);

} // namespace tensor_ash
