// Dequantize-fused MatMul dispatch and the FLOAT16 / BFLOAT16 MatMul.
//
//  - int4 / uint4 weights with FLOAT16 scales, M <= 16 (decode): the
//    bandwidth-bound GEMV, on the ONNX packing (gemv_q4.hip) or on the tiled
//    layout of a prepared weight (gemv_q4_tiled.hip, also more rows in slabs).
//  - prepared int4 / uint4 weights, FLOAT16 activations and scales, more rows:
//    the pipelined MFMA core with the weight decoded as its fragments are read
//    from LDS (mfma_gemm.hpp, kF16I4).
//  - float8e4m3fn weights, FLOAT scales per column or per tensor, Cast to
//    BFLOAT16, bf16 activations (prefill): the pipelined MFMA core with the
//    weight decoded exactly to bf16 as it is read from LDS and the scale
//    applied to the fp32 sums (mfma_gemm.hpp, kBf16F8); the decode GEMM
//    (skinny_gemm.hpp) for a few rows; the small-tile GEMM for few outputs, and
//    for the shapes and alignments the core does not take, there with each
//    weight rounded as the chain rounds it.
//  - anything else the C ABI accepts: the weight is dequantised into scratch
//    with the chain's exact rounding, then multiplied by the 16-bit MatMul.
#include <algorithm>

#include "common.hpp"
#include "device_codecs.hpp"
#include "kernels.hpp"
#include "mfma_gemm.hpp"
#include "skinny_gemm.hpp"
#include "tile_gemm.hpp"

namespace onnxl_amd {

bool GemvQ4Eligible(const DqMatMulParams &p);
bool GemvQ4TiledEligible(const DqMatMulParams &p);
void LaunchGemvQ4Tiled(const DqMatMulParams &p, hipStream_t stream);
size_t GemvQ4ScratchBytes(const DqMatMulParams &p);
size_t GemvQ4Counters(const DqMatMulParams &p);
void LaunchGemvQ4(const DqMatMulParams &p, void *scratch, unsigned *counters, hipStream_t stream);
void LaunchHTile(const mg::GemmArgs &g, bool bf16, bool big, hipStream_t s);
void LaunchHTileBT(const mg::GemmArgs &g, bool bf16, bool big, hipStream_t s);
void LaunchF8Skinny(const mg::GemmArgs &g, hipStream_t s);
void LaunchF8Tile(const mg::GemmArgs &g, bool chain, bool big, hipStream_t s);

namespace {

mg::GemmArgs HArgs(const HMatMulParams &p) {
  mg::GemmArgs g{};
  g.A = p.A;
  g.B = p.B;
  g.Y = p.Y;
  g.M = p.M;
  g.N = p.N;
  g.K = p.K;
  g.batch = p.batch;
  g.bm = p.bm;
  return g;
}

// ---------------------------------------------------------------------------
// Weight dequantisation into a 16-bit [K, N] scratch matrix with the unfused
// chain's rounding: DequantizeLinear computes (x - zp) * scale in fp32 and
// stores the scale's dtype (FLOAT16: round to nearest even); an optional Cast
// rounds FLOAT to BFLOAT16 / FLOAT16
// (kq/kernel_dequantizelinear.cc:57-63,259-285; kernel_cast.cc:360-370).
__device__ __forceinline__ float DecodeWeight(const uint8_t *w, int dt, int64_t i) {
  switch (dt) {
  case kInt4: return (float)Int4ToInt((w[i >> 1] >> (4 * (i & 1))) & 0xfu);
  case kUint4: return (float)((w[i >> 1] >> (4 * (i & 1))) & 0xfu);
  case kInt8: return (float)(int8_t)w[i];
  case kUint8: return (float)w[i];
  default: return Fp8E4M3ToF32(w[i]);
  }
}

// Element (k, n) of a 4-bit weight in the tiled layout (kernels.hpp).
__device__ __forceinline__ float DecodeTiled(const uint8_t *w, int dt, int64_t ngroups, int64_t k, int64_t n) {
  const int64_t t = n >> 4, i = n & 15, q = k >> 7, c = (k >> 5) & 3, g = (k >> 3) & 3, j = k & 7;
  const uint32_t word = reinterpret_cast<const uint32_t *>(w)[((t * ngroups + q) * 64 + g * 16 + i) * 4 + c];
  const uint32_t u = (word >> ((j & 1) ? 16 + 4 * (j >> 1) : 4 * (j >> 1))) & 15u;
  return dt == kInt4 ? (float)((int)u - 8) : (float)u;
}

// The dequantised value as the chain stores it: DequantizeLinear's FLOAT16, or
// a Cast's BFLOAT16 / FLOAT16.
__device__ __forceinline__ uint16_t WeightBits(const DqMatMulParams &p, float v) {
  return !p.deq_round_f16 && p.cast_round == 16 ? F32ToBf16(v) : F32ToF16(v);
}

__global__ __launch_bounds__(256) void DequantWeightKernel(const DqMatMulParams p, uint16_t *out) {
  const int64_t total = p.K * p.N;
  const int64_t ngroups = (p.K + 127) / 128;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t k = i / p.N, n = i % p.N;
    int64_t si = 0;
    if (p.mode == 1) si = n;
    else if (p.mode == 2) si = (k / p.block) * p.N + n;
    const float s = p.scale_f16 ? F16ToF32(static_cast<const uint16_t *>(p.scale)[si])
                                : static_cast<const float *>(p.scale)[si];
    const float z = p.zp ? DecodeWeight(p.zp, p.w_dtype, si) : 0.f;
    const float x = p.w_tiled ? DecodeTiled(p.W, p.w_dtype, ngroups, k, n) : DecodeWeight(p.W, p.w_dtype, i);
    out[i] = WeightBits(p, (x - z) * s);
  }
}

__device__ __forceinline__ float ScaleAt(const DqMatMulParams &p, int64_t si) {
  return p.scale_f16 ? F16ToF32(static_cast<const uint16_t *>(p.scale)[si]) : static_cast<const float *>(p.scale)[si];
}

// The same values from a tiled 4-bit weight, scale rows of a multiple of 8 rows
// (or one): a thread reads 16 bytes (32 rows of a column) and one scale and zero
// point per 8 rows, a wave stores 128 bytes of a row at a time.  The kernel above
// pays two 64-bit divisions, a scale and a code load for every value.  [4096,
// 11006]: 157 -> 47 us (23 at the copy rate; 2-byte stores bound it).
__global__ __launch_bounds__(256) void DequantTiledKernel(const DqMatMulParams p, uint16_t *out) {
  const int64_t n = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63), q = blockIdx.y;
  const int g = threadIdx.x >> 6;
  if (n >= p.N) return;
  const int64_t ngroups = (p.K + 127) / 128;
  unsigned w[4];
  __builtin_memcpy(w, p.W + (((n >> 4) * ngroups + q) * 64 + g * 16 + (n & 15)) * 16, 16);
  float s[4], z[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t k = 128 * q + 32 * c + 8 * g;
    const int64_t kb = p.mode == 2 ? (unsigned)(k < p.K ? k : 0) / (unsigned)p.block : 0;
    const int64_t si = p.mode == 0 ? 0 : kb * p.N + n;
    s[c] = ScaleAt(p, si);
    z[c] = p.zp ? DecodeWeight(p.zp, p.w_dtype, si) : 0.f;
  }
  const unsigned flip = p.w_dtype == kInt4 ? 8u : 0u;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t k = 128 * q + 32 * c + 8 * g;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (k + j >= p.K) return;
      const int u = (int)((w[c] >> ((j & 1) ? 16 + 4 * (j >> 1) : 4 * (j >> 1))) & 15u) - (int)flip;
      out[(k + j) * p.N + n] = WeightBits(p, ((float)u - z[c]) * s[c]);
    }
  }
}

// The same from row-major weights, N a multiple of E (8 or 2): E values of a row
// per step, the codes, scales and zero points of kRowUnits steps on their way
// before the first is decoded.  With the product, 8 rows of bf16, [4096, 11008]:
// int4 131 -> 53 us, uint8 with zero points 147 -> 63.
constexpr int kRowUnits = 2;
template <int E>
__global__ __launch_bounds__(256) void DequantRowsKernel(const DqMatMulParams p, unsigned units, uint16_t *out) {
  const bool four = p.w_dtype == kInt4 || p.w_dtype == kUint4;
  const unsigned per_row = (unsigned)(p.N / E);
  uint8_t w[kRowUnits][E], zb[kRowUnits][E];
  uint16_t s16[kRowUnits][E];
  float s32[kRowUnits][E];
  auto unit = [&](int t) { return (blockIdx.x * kRowUnits + t) * 256u + threadIdx.x; };
  auto bytes = [&](uint8_t(&to)[E], const uint8_t *from, int64_t i) {
    if (four) __builtin_memcpy(to, from + i / 2, E / 2);
    else __builtin_memcpy(to, from + i, E);
  };
#pragma unroll
  for (int t = 0; t < kRowUnits; ++t) {
    const unsigned u = unit(t) < units ? unit(t) : units - 1, k = u / per_row;
    bytes(w[t], p.W, (int64_t)u * E);
    if (p.mode == 0) continue;
    const int64_t si = (p.mode == 2 ? (int64_t)(k / (unsigned)p.block) * p.N : 0) + (u - k * per_row) * E;
    if (p.scale_f16) __builtin_memcpy(s16[t], static_cast<const uint16_t *>(p.scale) + si, 2 * E);
    else __builtin_memcpy(s32[t], static_cast<const float *>(p.scale) + si, 4 * E);
    if (p.zp) bytes(zb[t], p.zp, si);
  }
  const float s0 = p.mode == 0 ? ScaleAt(p, 0) : 0.f, z0 = p.mode == 0 && p.zp ? DecodeWeight(p.zp, p.w_dtype, 0) : 0.f;
#pragma unroll
  for (int t = 0; t < kRowUnits; ++t) {
    if (unit(t) >= units) return;
    unsigned o[E / 2];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float s = p.mode == 0 ? s0 : (p.scale_f16 ? F16ToF32(s16[t][e]) : s32[t][e]);
      const float z = p.mode == 0 || !p.zp ? z0 : DecodeWeight(zb[t], p.w_dtype, e);
      const unsigned b = WeightBits(p, (DecodeWeight(w[t], p.w_dtype, e) - z) * s);
      o[e / 2] = e & 1 ? o[e / 2] | b << 16 : b;
    }
    __builtin_memcpy(out + (int64_t)unit(t) * E, o, 2 * E);
  }
}

// Weights of up to this many values give the vector kernels too few threads to
// hide their longer chains: the value-per-thread kernel takes them.  With the
// product, 32 rows, value per thread -> vector: uint8 256 x 512 with zero points 7.1 ->
// 10.2 us, 512 x 1024 9.1 -> 11.5, 1024 x 1024 13.3 -> 14.3, 1024 x 2048 15.6 -> 15.6,
// 2048 x 2048 26.2 -> 22.8; int4 tiled 512 x 512 8.4 -> 10.4, 1024 x 1024 13.7 -> 13.8,
// 1024 x 2048 16.2 -> 14.9.  Pairs of columns make four times the threads of eights
// (uint8 256 x 514 7.6 -> 8.4, 512 x 1026 10.0 -> 10.1, 1024 x 2050 18.4 -> 15.1).
constexpr int64_t kSmallWeight = int64_t(1) << 20;

void LaunchDequantWeight(const DqMatMulParams &p, uint16_t *out, hipStream_t stream) {
  const int64_t total = p.K * p.N, cols = (p.N + 63) / 64, ngroups = (p.K + 127) / 128;
  const bool k32 = p.K <= 0x7fffffff && p.block <= 0x7fffffff;
  if (p.w_tiled && k32 && total > kSmallWeight && (p.mode != 2 || p.block % 8 == 0) && ngroups <= 65535 && cols <= 0x7fffffff) {
    hipLaunchKernelGGL(DequantTiledKernel, dim3((unsigned)cols, (unsigned)ngroups), dim3(256), 0, stream, p, out);
  } else if (!p.w_tiled && k32 && p.N % 2 == 0 && total > kSmallWeight / (p.N % 8 == 0 ? 1 : 4) &&
             total <= (int64_t(1) << 32)) {
    const unsigned units = (unsigned)(total / (p.N % 8 == 0 ? 8 : 2)), per = 256 * kRowUnits;
    const dim3 grid((units + per - 1) / per);
    if (p.N % 8 == 0) hipLaunchKernelGGL(DequantRowsKernel<8>, grid, dim3(256), 0, stream, p, units, out);
    else hipLaunchKernelGGL(DequantRowsKernel<2>, grid, dim3(256), 0, stream, p, units, out);
  } else {
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(DequantWeightKernel, dim3(blocks), dim3(256), 0, stream, p, out);
  }
}

bool Fp8Eligible(const DqMatMulParams &p) {
  return p.w_dtype == kFloat8E4M3FN && p.a_bf16 && p.cast_round == 16 && !p.scale_f16 &&
         (p.mode == 0 || p.mode == 1) && p.zp == nullptr;
}

// Compute units of the current device, queried once per device.
int64_t DeviceCUs() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// The fp8 GEMM in 256 x 256 tiles, except that when those tiles leave a last,
// partly filled round of workgroups, the trailing columns go to a second
// launch in 256 x 128 tiles.  C4 (4096 x 14336): 896 tiles are 3.5 rounds on
// 256 CUs; 768 tiles (12288 columns) make 3 whole rounds and the last 2048
// columns are 256 half-size tiles, one round of half the time.
void LaunchFp8Gemm(const mg::GemmArgs &g, hipStream_t stream) {
  const int64_t cus = DeviceCUs();
  const int64_t nbm = (g.M + 255) / 256, nbn = (g.N + 255) / 256;
  if (nbm * nbn < 512 || g.K % 64 != 0) {  // 256 x 256 tiles take whole K steps only
    if (mg::PrefersHalfTile<mg::kBf16F8>(g)) mg::Launch<mg::kBf16F8, mg::kOutBf16, false, false, false, 2, false, 2>(g, stream);
    else mg::Launch<mg::kBf16F8, mg::kOutBf16, false, false, false, 2>(g, stream);
    return;
  }
  int64_t nb = nbn;  // tile-columns in 256 x 256 tiles
  if ((nbm * nbn) % cus != 0 && g.N % 256 == 0) {
    int64_t c = nbn - 1;
    while (c > 0 && (nbm * c) % cus != 0) --c;
    if (c > 0 && nbm * (nbn - c) * 2 <= cus) nb = c;
  }
  if (nb == nbn) {
    mg::Launch<mg::kBf16F8, mg::kOutBf16, false, false, false, 4>(g, stream);
    return;
  }
  const int64_t n0 = nb * 256;
  mg::GemmArgs g1 = g, g2 = g;
  g1.N = n0;
  g1.ldb = g.N;
  g1.ldy = g.N;
  g2.N = g.N - n0;
  g2.ldb = g.N;
  g2.ldy = g.N;
  g2.B = static_cast<const uint8_t *>(g.B) + n0;
  g2.Y = static_cast<uint16_t *>(g.Y) + n0;
  if (g.scale_per_col) g2.scale = static_cast<const float *>(g.scale) + n0;
  mg::Launch<mg::kBf16F8, mg::kOutBf16, false, false, false, 4>(g1, stream);
  mg::Launch<mg::kBf16F8, mg::kOutBf16, false, false, false, 2>(g2, stream);
}

mg::GemmArgs Fp8Args(const DqMatMulParams &p) {
  mg::GemmArgs g{};
  g.A = p.A;
  g.B = p.W;
  g.Y = p.Y;
  g.M = p.M;
  g.N = p.N;
  g.K = p.K;
  g.batch = 1;
  g.scale = p.scale;
  g.scale_f16 = 0;
  g.scale_per_col = p.mode == 1;
  return g;
}

// Prepared 4-bit weights past the GEMV's rows, decoded inside the GEMM: fp16
// activations and scales, one scale row per 32 or more rows of k (a power of
// two) or one for all.  Dequantising the whole weight first costs a pass over
// it and over its fp16 form for every call (K = 4096, N = 11008: 20 us if it
// ran at the copy rate, 128 us as it was), more than the decode adds to the
// GEMM (M = 1000: fp16 weight 94 us, this 104 us).
mg::GemmArgs Int4Args(const DqMatMulParams &p) {
  mg::GemmArgs g{};
  g.A = p.A;
  g.B = p.W;
  g.Y = p.Y;
  g.M = p.M;
  g.N = p.N;
  g.K = p.K;
  g.batch = 1;
  g.scale = p.scale;
  g.scale_rows = p.mode == 2 ? p.K / p.block : 1;
  g.blk_shift = p.mode == 2 ? __builtin_ctzll((unsigned long long)p.block) : 31;
  g.zp4 = p.zp;
  g.w_signed = p.w_dtype == kInt4;
  return g;
}

bool Int4GemmEligible(const DqMatMulParams &p) {
  if (!p.w_tiled || p.a_bf16 || !p.scale_f16 || !p.deq_round_f16 || p.cast_round != 0) return false;
  if (p.mode == 2 ? p.block < 32 || (p.block & (p.block - 1)) != 0 : p.mode != 1) return false;
  return mg::EligibleI4(Int4Args(p));
}

void LaunchInt4Gemm(const DqMatMulParams &p, hipStream_t stream) {
  const mg::GemmArgs g = Int4Args(p);
  const bool half = mg::PrefersHalfTile<mg::kF16I4>(g);
  if (p.zp != nullptr) {
    if (half) mg::Launch<mg::kF16I4, mg::kOutF16, true, false, false, 2, false, 2>(g, stream);
    else mg::Launch<mg::kF16I4, mg::kOutF16, true, false, false>(g, stream);
  } else {
    if (half) mg::Launch<mg::kF16I4, mg::kOutF16, false, false, false, 2, false, 2>(g, stream);
    else mg::Launch<mg::kF16I4, mg::kOutF16, false, false, false>(g, stream);
  }
}

// A 4-bit weight in the ONNX packing past its GEMV's rows: tiled into scratch,
// then as a prepared one.  Never more scratch than the dequantised weight of
// the general path.  K = 4096, N = 11008: the pass takes 10 us (dequantising it 128),
// 17 rows 125 -> 22.6 us, 1000 rows 204 -> 119.  A small weight whose last columns
// or rows the pass would gather byte by byte is dequantised instead (32 rows,
// dequantised -> tiled: 64 x 64 7.3 -> 11.2 us, 256 x 514 7.6 -> 11.5, 512 x 1026
// 10.0 -> 12.0; 1024 x 2050 18.2 -> 12.9; whole ones 512 x 512 8.3 -> 7.4).
DqMatMulParams WithTiledWeight(const DqMatMulParams &p, const void *scratch) {
  DqMatMulParams t = p;
  t.W = static_cast<const uint8_t *>(scratch);
  t.w_tiled = 1;
  return t;
}

bool TilesFirst(const DqMatMulParams &p) {
  if (p.w_tiled || (p.w_dtype != kInt4 && p.w_dtype != kUint4) || p.K == 0 || p.N % 2 != 0 ||
      TiledInt4Bytes(p.K, p.N) > p.K * p.N * 2 ||
      (p.K * p.N <= kSmallWeight && (p.N % 8 != 0 || p.K % 128 != 0)))
    return false;
  const DqMatMulParams t = WithTiledWeight(p, reinterpret_cast<const void *>(uintptr_t(256)));
  return GemvQ4TiledEligible(t) || Int4GemmEligible(t);
}

}  // namespace

void LaunchHMatMul(const HMatMulParams &p, hipStream_t stream) {
  if (p.M == 0 || p.N == 0 || p.batch == 0) return;
  const mg::GemmArgs g = HArgs(p);
  const bool core = mg::Eligible<mg::kH16>(g), small = tg::PrefersSmallTile(g, core);
  const bool half = mg::PrefersHalfTile<mg::kH16>(g);
  if (small || !core) LaunchHTile(g, p.bf16, !small, stream);
  else if (half && p.bf16) mg::Launch<mg::kH16, mg::kOutBf16, false, false, false, 2, false, 2>(g, stream);
  else if (half) mg::Launch<mg::kH16, mg::kOutF16, false, false, false, 2, false, 2>(g, stream);
  else if (p.bf16) mg::Launch<mg::kH16, mg::kOutBf16, false, false, false>(g, stream);
  else mg::Launch<mg::kH16, mg::kOutF16, false, false, false>(g, stream);
}

// Y = A @ B^T for B given as [N, K] (batch 1).
void LaunchHMatMulBT(const HMatMulParams &p, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return;
  const mg::GemmArgs g = HArgs(p);
  const bool core = mg::EligibleBT(g), small = tg::PrefersSmallTile(g, core);
  const bool half = mg::PrefersHalfTile<mg::kH16>(g);
  if (small || !core) LaunchHTileBT(g, p.bf16, !small, stream);
  else if (half && p.bf16) mg::LaunchBT<mg::kOutBf16, 2>(g, stream);
  else if (half) mg::LaunchBT<mg::kOutF16, 2>(g, stream);
  else if (p.bf16) mg::LaunchBT<mg::kOutBf16>(g, stream);
  else mg::LaunchBT<mg::kOutF16>(g, stream);
}

size_t DqMatMulScratchBytes(const DqMatMulParams &p) {
  if (GemvQ4TiledEligible(p) || Int4GemmEligible(p) || Fp8Eligible(p)) return 0;
  if (GemvQ4Eligible(p)) return GemvQ4ScratchBytes(p);
  if (TilesFirst(p)) return (size_t)TiledInt4Bytes(p.K, p.N);
  return (size_t)(p.K * p.N) * sizeof(uint16_t);
}

// The bytes that the no-allocation entry point counts a call with, against its
// fixed array: the scratch of the GEMVs, none for an fp8 weight of the pipelined
// GEMM's shapes, and for every other call its dequantised weight, whatever kernel
// takes it.  So the calls it accepts depend on sizes and types alone: a line between
// two kernels that moves (PrefersGemv, TilesFirst) turns no captured call away.
// Never less than DqMatMulScratchBytes.
size_t DqMatMulFixedScratchBytes(const DqMatMulParams &p) {
  if (p.M <= 16 && GemvQ4TiledEligible(p)) return 0;
  if (GemvQ4Eligible(p)) return GemvQ4ScratchBytes(p);
  if (Fp8Eligible(p) && mg::Eligible<mg::kBf16F8>(Fp8Args(p))) return 0;
  return (size_t)(p.K * p.N) * sizeof(uint16_t);
}

size_t DqMatMulCounters(const DqMatMulParams &p) {
  return GemvQ4Eligible(p) ? GemvQ4Counters(p) : 0;
}

bool LaunchDqMatMul(const DqMatMulParams &p, void *scratch, size_t scratch_bytes, unsigned *counters,
                    size_t n_counters, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return true;
  if (GemvQ4TiledEligible(p)) {
    LaunchGemvQ4Tiled(p, stream);
    return true;
  }
  if (GemvQ4Eligible(p)) {
    if (scratch_bytes < GemvQ4ScratchBytes(p) || n_counters < GemvQ4Counters(p)) return false;
    LaunchGemvQ4(p, scratch, counters, stream);
    return true;
  }
  if (Int4GemmEligible(p)) {
    LaunchInt4Gemm(p, stream);
    return true;
  }
  if (Fp8Eligible(p)) {
    const mg::GemmArgs g = Fp8Args(p);
    const bool core = mg::Eligible<mg::kBf16F8>(g), small = tg::PrefersSmallTile(g, core);
    if (core && sk::PrefersSkinny(g, false, false)) LaunchF8Skinny(g, stream);
    else if (core && !small) LaunchFp8Gemm(g, stream);
    else LaunchF8Tile(g, /*chain=*/!core, !small, stream);
    return true;
  }
  if (TilesFirst(p)) {
    if (scratch_bytes < (size_t)TiledInt4Bytes(p.K, p.N)) return false;
    const DqMatMulParams t = WithTiledWeight(p, scratch);
    LaunchTileInt4(p.W, p.K, p.N, p.w_dtype == kInt4, static_cast<uint32_t *>(scratch), stream);
    if (GemvQ4TiledEligible(t)) LaunchGemvQ4Tiled(t, stream);
    else LaunchInt4Gemm(t, stream);
    return true;
  }
  // general path: dequantise into scratch, then the 16-bit MatMul (K == 0
  // leaves nothing to dequantise and the MatMul writes zeros)
  if (scratch_bytes < (size_t)(p.K * p.N) * sizeof(uint16_t)) return false;
  uint16_t *w16 = static_cast<uint16_t *>(scratch);
  if (p.K > 0) LaunchDequantWeight(p, w16, stream);
  HMatMulParams h{};
  h.A = static_cast<const uint16_t *>(p.A);
  h.B = w16;
  h.Y = static_cast<uint16_t *>(p.Y);
  h.M = p.M;
  h.N = p.N;
  h.K = p.K;
  h.batch = 1;
  h.bf16 = p.a_bf16;
  LaunchHMatMul(h, stream);
  return true;
}

}  // namespace onnxl_amd
