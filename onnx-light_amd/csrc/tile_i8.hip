// Small-tile int8 GEMM instantiations (tile_gemm.hpp): MatMulInteger,
// QLinearMatMul and the convolutions' GEMM over im2col columns.
#include "igemm_fast.hpp"
#include "tile_gemm.hpp"

namespace onnxl_amd {

void LaunchIGemmTile(const IGemmParams &p, bool big, hipStream_t s) {
  const mg::GemmArgs g = ToGemmArgs(p);
  const bool zp = p.need_ra || p.need_cb;
  if (p.epilogue == kEpiQuant8Row) {  // convolutions: a zero point on x is the rule
    tg::Launch<mg::kI8, tg::kSrcRow, mg::kOutQ8Row, true>(g, big, s);
  } else if (p.epilogue == kEpiInt32) {
    if (zp) tg::Launch<mg::kI8, tg::kSrcRow, mg::kOutI32, true>(g, big, s);
    else tg::Launch<mg::kI8, tg::kSrcRow, mg::kOutI32, false>(g, big, s);
  } else {
    if (zp) tg::Launch<mg::kI8, tg::kSrcRow, mg::kOutQ8, true>(g, big, s);
    else tg::Launch<mg::kI8, tg::kSrcRow, mg::kOutQ8, false>(g, big, s);
  }
}

}  // namespace onnxl_amd
