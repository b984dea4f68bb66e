// For a model's products, some at the edges of the kernels' choice and some at random: every launch of at most
// `rows` sequences fits the workspace sized for `rows`.  Plans only, no GPU.
#include <algorithm>
#include <array>
#include <cstdio>
#include <random>
#include <vector>

#include "gemv.h"

using namespace efh;

int main() {
  ctx().cu_count = 256;
  ctx().lds_per_block = 160 * 1024;
  std::mt19937 rng(7);
  struct Shape {
    int epi;
    std::vector<std::array<size_t, 2>> mats;  // rows, type
    size_t K;
  };
  const size_t q4 = EF_QTYPE_Q4_0, q8 = EF_QTYPE_Q8_0;
  std::vector<Shape> shapes = {
      {kEpiStore, {{2048, q4}, {256, q4}, {256, q8}}, 2048}, {kEpiResidual, {{2048, q4}}, 2048},
      {kEpiSwiglu, {{5632, q4}}, 2048},  {kEpiResidual, {{2048, q4}}, 5632}, {kEpiStore, {{32000, q8}}, 2048},
      {kEpiResidual, {{1000, q4}}, 4000}, {kEpiResidual, {{512, q4}}, 14336}, {kEpiSwiglu, {{14336, q4}}, 512},
      {kEpiStore, {{256, q8}}, 5632},     {kEpiSwiglu, {{96, q4}}, 8192}};
  for (int i = 0; i < 20; ++i) {
    const size_t K = 32 * (1 + rng() % 448);
    shapes.push_back({static_cast<int>(rng() % 3), {{64 + rng() % 6000, rng() % 2 ? q4 : q8}}, K});
  }
  int checked = 0, bad = 0;
  for (const Shape& s : shapes) {
    std::vector<ef_hip_weight_s> w(s.mats.size());
    std::vector<GemvJob> jobs(s.mats.size());
    for (size_t j = 0; j < w.size(); ++j) {
      w[j].rows = s.mats[j][0];
      w[j].cols = s.K;
      w[j].qtype = static_cast<int>(s.mats[j][1]);
      w[j].row_bytes = s.K / 32 * (w[j].qtype == EF_QTYPE_Q4_0 ? 18 : 34);
      jobs[j] = GemvJob{&w[j], s.epi == kEpiSwiglu ? &w[j] : nullptr, nullptr, nullptr, s.K, w[j].rows};
    }
    const int n = static_cast<int>(jobs.size());
    for (const int rows : {40, 500, 1023, 1500, 2047, 4096}) {
      const size_t need = gemv_mfma_workspace_upto(jobs.data(), n, s.epi, rows, s.K);
      for (int r = 2; r <= rows; r += 1 + static_cast<int>(rng() % 5)) {
        // a launch takes the plan of its whole 16-sequence tiles where its own wants more
        const size_t own = std::min(gemv_mfma_workspace_bytes(jobs.data(), n, s.epi, r, s.K),
                                    gemv_mfma_workspace_bytes(jobs.data(), n, s.epi, (r + 15) / 16 * 16, s.K));
        ++checked;
        if (own > need) {
          if (bad++ < 10)
            std::printf("epi %d rows %zu K %zu: %d of %d sequences want %zu of %zu bytes\n", s.epi, w[0].rows, s.K, r,
                        rows, own, need);
        }
      }
    }
  }
  std::printf("%d launches checked, %d too large\n", checked, bad);
  return bad ? 1 : 0;
}
