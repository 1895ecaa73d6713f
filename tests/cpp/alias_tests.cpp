// One buffer read by several ops of a submission under different shapes
// (Tensor::alias_with_shape): few rows of f32 A on f16 weights, whose packed
// pieces of A are kept between ops.  Run by tests/test_gemm_f16w3_gpu.py.
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "../../tensor-ash_amd/csrc/runtime/tensor_ash.hpp"

using namespace tensor_ash;

static std::vector<float> fill(size_t n, uint32_t seed) {
  std::vector<float> v(n);
  for (auto &x : v) {
    seed = seed * 1664525u + 1013904223u;
    x = (float)((int)(seed >> 20) - 2048) / 2048.0f; // exact in f16
  }
  return v;
}

struct View {
  uint32_t planes, rows, k;
};

int main() {
  const uint32_t n = 96, len = 32 * 512;
  auto ctx = Context::create(false, "index:0");
  ExecutorConfig cfg;
  cfg.tune = false;
  Executor ex(ctx, KernelSelection{}, cfg);
  const std::vector<float> ha = fill(len, 1);
  const std::vector<View> views = {{1, 32, 512}, {2, 16, 512}, {1, 16, 1024}, {4, 16, 256}};
  int bad = 0;
  for (size_t i = 0; i < views.size(); ++i)
    for (size_t j = 0; j < views.size(); ++j)
      for (int graph = 0; graph < 2; ++graph) {
        const View order[2] = {views[i], views[j]};
        std::printf("views %zu %zu graph %d\n", i, j, graph);
        std::fflush(stdout);
        Tensor a = Tensor::uninit_device(ctx, {len});
        ex.upload(ha.data(), ha.size(), a);
        std::vector<Tensor> as, bs, cs;
        std::vector<std::vector<float>> hb;
        for (const View &v : order) {
          const bool flat = v.planes == 1;
          as.push_back(a.alias_with_shape(flat ? std::vector<uint32_t>{v.rows, v.k}
                                               : std::vector<uint32_t>{v.planes, v.rows, v.k}));
          hb.push_back(fill((size_t)v.planes * v.k * n, 7));
          bs.push_back(Tensor::uninit_device_f16(ctx, flat ? std::vector<uint32_t>{v.k, n}
                                                           : std::vector<uint32_t>{v.planes, v.k, n}));
          ex.upload(hb.back().data(), hb.back().size(), bs.back());
          cs.push_back(Tensor::uninit_device(ctx, flat ? std::vector<uint32_t>{v.rows, n}
                                                       : std::vector<uint32_t>{v.planes, v.rows, n}));
        }
        std::vector<MatmulOp> ops;
        for (int o = 0; o < 2; ++o)
          ops.emplace_back(MatmulCall{&as[o], &bs[o], &cs[o], 1.0f, false});
        graph ? ex.run_op_graph(ops) : ex.run_ops(ops);
        for (int o = 0; o < 2; ++o) {
          const View &v = order[o];
          std::vector<float> got((size_t)v.planes * v.rows * n);
          ex.download(cs[o], got.data(), got.size());
          for (uint32_t p = 0; p < v.planes; ++p)
            for (uint32_t r = 0; r < v.rows; ++r)
              for (uint32_t c = 0; c < n; ++c) {
                double s = 0, mag = 0;
                for (uint32_t k = 0; k < v.k; ++k) {
                  const double t = (double)ha[((size_t)p * v.rows + r) * v.k + k] *
                                   hb[o][((size_t)p * v.k + k) * n + c];
                  s += t;
                  mag += std::fabs(t);
                }
                // f32 sums of K products in any order
                const double tol = v.k * std::ldexp(1.0, -24) * mag;
                if (!(std::fabs(got[((size_t)p * v.rows + r) * n + c] - s) <= tol))
                  ++bad;
              }
        }
        if (bad) {
          std::printf("FAIL: %d wrong values\n", bad);
          return 1;
        }
      }
  std::printf("OK\n");
  return 0;
}
