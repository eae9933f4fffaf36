// Small-tile 16-bit GEMM instantiations (tile_gemm.hpp): FLOAT16 / BFLOAT16
// MatMul, B given transposed, and float8e4m3fn weights under bf16 activations.
#include "kernels.hpp"
#include "tile_gemm.hpp"

namespace onnxl_amd {

void LaunchHTile(const mg::GemmArgs &g, bool bf16, bool big, hipStream_t s) {
  if (bf16) tg::Launch<mg::kH16, tg::kSrcRow, mg::kOutBf16, false>(g, big, s);
  else tg::Launch<mg::kH16, tg::kSrcRow, mg::kOutF16, false>(g, big, s);
}

void LaunchHTileBT(const mg::GemmArgs &g, bool bf16, bool big, hipStream_t s) {
  if (bf16) tg::Launch<mg::kH16, tg::kSrcT, mg::kOutBf16, false>(g, big, s);
  else tg::Launch<mg::kH16, tg::kSrcT, mg::kOutF16, false>(g, big, s);
}

void LaunchF8Tile(const mg::GemmArgs &g, bool chain, bool big, hipStream_t s) {
  if (chain) tg::Launch<mg::kBf16F8, tg::kSrcF8Chain, mg::kOutBf16, false>(g, big, s);
  else tg::Launch<mg::kBf16F8, tg::kSrcF8, mg::kOutBf16, false>(g, big, s);
}

}  // namespace onnxl_amd
