// Pipelined int8 GEMM instantiations for single device-resident zero points
// (MatMulInteger): the kernel reads them and drops the sums they do not need.
#include "igemm_fast.hpp"

namespace onnxl_amd {
namespace {

template <int MB> void Tile(const IGemmParams &p, hipStream_t s) {
  const mg::GemmArgs g = ToGemmArgs(p);
  switch ((p.a_u8 ? 2 : 0) | (p.b_u8 ? 1 : 0)) {
  case 0: mg::Launch<mg::kI8, mg::kOutI32, true, false, false, 2, false, MB, true>(g, s); break;
  case 1: mg::Launch<mg::kI8, mg::kOutI32, true, false, true, 2, false, MB, true>(g, s); break;
  case 2: mg::Launch<mg::kI8, mg::kOutI32, true, true, false, 2, false, MB, true>(g, s); break;
  default: mg::Launch<mg::kI8, mg::kOutI32, true, true, true, 2, false, MB, true>(g, s); break;
  }
}

}  // namespace

void LaunchIGemmFastDev(const IGemmParams &p, bool half, hipStream_t s) {
  if (half) Tile<2>(p, s);
  else Tile<4>(p, s);
}

}  // namespace onnxl_amd
