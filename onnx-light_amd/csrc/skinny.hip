// Decode GEMM instantiations (skinny_gemm.hpp).
#include <algorithm>

#include "igemm_fast.hpp"
#include "kernels.hpp"
#include "skinny_gemm.hpp"

namespace onnxl_amd {
namespace {

template <int KIND, int OUT, bool ZP, int CW, int W, int MT, bool GRP>
void Go(const sk::Args &q, int64_t entries, hipStream_t s) {
  const int64_t blocks = (q.g.N + 16 * CW - 1) / (16 * CW) * entries;
  hipLaunchKernelGGL((sk::SkinnyKernel<KIND, OUT, ZP, CW, W, MT, GRP>), dim3((unsigned)blocks), dim3(64 * W), 0, s, q);
}

// 64-column tiles of 16 waves while they fit one round of the chip, else
// 128-column tiles of 8 waves, which read whole 128-byte lines but are half as
// many (u8[8,4096] x s8[4096,N]: N = 4096 7.4 against 12.1 us, N = 28672 25.5
// against 21.4 us; the two meet at N = 14336, 224 of the narrow ones).  Grouped:
// by the most units that the pairs can make (64 tokens, 4 experts [4096, 4096] of
// about one unit each, by the groups 36.4 us, by the units 24.0).
bool Wide(const mg::GemmArgs &g, int64_t entries) { return (g.N + 63) / 64 * entries > 256; }

template <int KIND, int OUT, bool ZP> void Dense(const mg::GemmArgs &g, hipStream_t s) {
  sk::Args q{};
  q.g = g;
  if (g.M + (ZP ? 1 : 0) > 16) Go<KIND, OUT, ZP, 4, 16, 2, false>(q, g.batch, s);
  else if (Wide(g, g.batch)) Go<KIND, OUT, ZP, 8, 8, 1, false>(q, g.batch, s);
  else Go<KIND, OUT, ZP, 4, 16, 1, false>(q, g.batch, s);
}

}  // namespace

void LaunchIGemmSkinny(const IGemmParams &p, hipStream_t s) {
  const mg::GemmArgs g = ToGemmArgs(p);
  const bool zp = p.need_ra || p.need_cb;
  if (p.epilogue == kEpiInt32) {
    if (zp) Dense<mg::kI8, mg::kOutI32, true>(g, s);
    else Dense<mg::kI8, mg::kOutI32, false>(g, s);
  } else {
    if (zp) Dense<mg::kI8, mg::kOutQ8, true>(g, s);
    else Dense<mg::kI8, mg::kOutQ8, false>(g, s);
  }
}

void LaunchF8Skinny(const mg::GemmArgs &g, hipStream_t s) { Dense<mg::kBf16F8, mg::kOutBf16, false>(g, s); }

void LaunchF8SkinnyGrouped(const mg::GemmArgs &g, const void *idx, int idx64, hipStream_t s) {
  sk::Args q{};
  q.g = g;
  q.idx = idx;
  q.idx64 = idx64;
  // two 16-row operands per workgroup once an expert's average share of the
  // pairs nears one (8 experts of [4096, 14336]: 32 tokens, 8 rows each, 100.7
  // with one against 106.1 us with two; 64 tokens 161.5 against 114.8)
  const int64_t P = g.M * g.grp_sel;
  const bool two = P > 12 * (int64_t)g.grp_count;
  // the most units of R pairs that P pairs in at most that many groups make
  const int64_t R = two ? 32 : 16, most = std::min<int64_t>(P, g.grp_count), units = std::min(P, (P + (R - 1) * most) / R);
  if (Wide(g, units)) {
    if (two) Go<mg::kBf16F8, mg::kOutBf16, false, 8, 8, 2, true>(q, units, s);
    else Go<mg::kBf16F8, mg::kOutBf16, false, 8, 8, 1, true>(q, units, s);
  } else {
    if (two) Go<mg::kBf16F8, mg::kOutBf16, false, 4, 16, 2, true>(q, units, s);
    else Go<mg::kBf16F8, mg::kOutBf16, false, 4, 16, 1, true>(q, units, s);
  }
}

}  // namespace onnxl_amd
