// Small-tile MFMA GEMM for the shapes the 256-row core (mfma_gemm.hpp) cannot
// take or leaves most of the chip idle on: any M, N and K, any alignment of
// the operands and of the output rows, and problems with few rows.
//
// Workgroup: 4 waves (2 x 2), tile (64 MB) x (64 WB), each wave MB x WB blocks
// of 32 x 32.  MB = WB = 2 (128 x 128) where those tiles fill the chip, else
// MB = WB = 1 (64 x 64), which puts four times the workgroups on it, or MB = 1,
// WB = 2 between the two (PrefersWideTile).
//
// Memory path.  Both operands go global -> registers -> LDS.  The core's
// direct loads need 16-byte aligned rows; a register load does not, so a row
// pitch of any length is read in 16-byte pieces where it lies, with no padded
// copy in memory.  D K steps are held in registers (D = 4 for the 64 x 64
// tile, whose step multiplies for only ~300 cycles against a ~2 us load), two
// in LDS; the LDS layouts (chunk swizzles, transposing reads of a row-major B)
// are the core's.  Only the last K step, where a row's end or the matrix's end
// can fall inside a piece, takes the guarded loads (LoadTail).
//  - UINT8 operands are flipped (x ^ 0x80) on the way into LDS, so one loop
//    serves every operand type; the flip leaves K padding at zero.
//  - fp8 weights become bf16 on the way into LDS, once per workgroup (in the
//    core's fragments each of the two waves sharing columns decodes them).
#pragma once

#include "mfma_gemm.hpp"
#include "tile_steps.hpp"

namespace onnxl_amd {
namespace tg {

using mg::GemmArgs;
using mg::v16f;
using mg::v16i;
using mg::v2f;
using mg::v2i;
using mg::v4f;
using mg::v4i;
using mg::v4s;
using mg::v8bf;
using mg::v8h;

// Where B comes from: the MFMA's type as [K, N] rows, or given transposed
// ([N, K]), or float8e4m3fn [K, N] rows.  kSrcF8 multiplies the codes' exact
// bf16 values and scales the sums, as the core does; kSrcF8Chain rounds each
// scaled weight to bf16 as the DequantizeLinear -> Cast chain does (the shapes
// the core does not take have always been computed so).
enum Src : int { kSrcRow = 0, kSrcF8 = 1, kSrcT = 2, kSrcF8Chain = 3 };

constexpr int kGroupRows = 8;  // tile rows that share a pass over B's columns

// A 16-byte piece at any address.
__device__ __forceinline__ v4i LoadPiece(const char *p) {
  v4i v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// A piece of which only the first `valid` bytes count (the rest become the
// bytes of `fill`), in a matrix of `total` bytes from `base`.  Nothing past
// the matrix is read: where p's piece crosses its end the last whole piece is
// loaded instead, TailBack bytes before p, and TailFix moves p's byte first.
__device__ __forceinline__ int64_t TailBack(const char *base, int64_t total, const char *p) {
  const int64_t s = p - (base + total - 16);
  return s > 0 ? s : 0;
}
__device__ __forceinline__ v4i TailMask(const unsigned (&r)[4], int64_t valid, unsigned fill) {
  v4i w;
  const int n = valid < 16 ? (int)(valid < 0 ? 0 : valid) : 16;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int k = n - 4 * e;  // valid bytes of this dword
    const unsigned m = k >= 4 ? ~0u : (k <= 0 ? 0u : (1u << (8 * k)) - 1u);
    w[e] = (int)((r[e] & m) | (fill & ~m));
  }
  return w;
}
__device__ __forceinline__ v4i TailFix(v4i v, int64_t back, int64_t valid, unsigned fill) {
  const int s = back < 16 ? (int)back : 0;  // 16 or more: no valid byte
  const uint64_t lo = (uint64_t)(unsigned)v.x | (uint64_t)(unsigned)v.y << 32;
  const uint64_t hi = (uint64_t)(unsigned)v.z | (uint64_t)(unsigned)v.w << 32;
  const int b = 8 * (s & 7);
  const uint64_t l1 = s & 8 ? hi : lo, h1 = s & 8 ? 0 : hi;
  const uint64_t l = b ? l1 >> b | h1 << (64 - b) : l1, h = h1 >> b;
  const unsigned r[4] = {(unsigned)l, (unsigned)(l >> 32), (unsigned)h, (unsigned)(h >> 32)};
  return TailMask(r, valid, fill);
}
// The same in a matrix of fewer than 16 bytes, byte by byte.
__device__ __forceinline__ v4i TailBytes(const char *base, int64_t total, const char *p, int64_t valid, unsigned fill) {
  unsigned r[4] = {0, 0, 0, 0};
#pragma unroll 1
  for (int e = 0; e < 16 && e < valid && p + e < base + total; ++e) {
    const unsigned x = (unsigned)(uint8_t)p[e] << (8 * (e & 3));
#pragma unroll
    for (int d = 0; d < 4; ++d) r[d] |= (e >> 2) == d ? x : 0u;
  }
  return TailMask(r, valid, fill);
}

// Orders this wave's LDS accesses before the workgroup barrier.  Loads into
// registers stay in flight across it (a __syncthreads() would wait for them).
__device__ __forceinline__ void LdsBarrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// G groups of 4 waves: each multiplies its share of the K steps
// (PrefersTwoGroups).
template <int KIND, int SRC, int OUT, bool ZP, int MB, int WB, int D, int G>
__global__ __launch_bounds__(256 * G, G == 1 ? 2 : 1) void TileGemmKernel(const GemmArgs p) {
  constexpr bool I8 = KIND == mg::kI8;
  constexpr bool BT = SRC == kSrcT, F8 = SRC == kSrcF8 || SRC == kSrcF8Chain;
  static_assert(I8 ? SRC == kSrcRow : !ZP, "int8 B is row-major; zero points are int8's");
  static_assert(D % 2 == 0, "the LDS stage is a constant after unrolling by D");
  constexpr int BM = 64 * MB, BN = 64 * WB, kWN = 32 * WB;
  constexpr int kKStep = I8 ? 128 : 64;             // k values per step: 128 bytes of A
  constexpr int kAsz = I8 ? 1 : 2;                  // bytes of an A element
  constexpr int kBsz = I8 || F8 ? 1 : 2; // bytes of a B element in memory
  constexpr int kBP = I8 ? BN : 2 * BN;             // bytes of a row-major B row in LDS
  constexpr int kASt = BM * 128, kBSt = BN * 128;   // bytes of a stage
  constexpr int kStage = kASt + kBSt;
  constexpr int NA = BM / 32;                            // 16-byte pieces per thread and step
  constexpr int NB = F8 ? BN / 64 : BN / 32;
  constexpr int kPpr = BN * kBsz / 16;              // pieces per row-major B row
  constexpr int kOsz = OUT == mg::kOutI32 ? 4 : (OUT == mg::kOutQ8 || OUT == mg::kOutQ8Row ? 1 : 2);
  constexpr int kPitch = kWN * kOsz + 16;           // staged output row
  static_assert(4 * 32 * kPitch <= 2 * kStage, "output staging fits the two stages");
  using Acc = std::conditional_t<I8, v16i, v16f>;
  __shared__ __align__(16) char sm[G * 2 * kStage];
  __shared__ int32_t zsum[ZP ? 4 * 2 * kWN : 1];

  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  char *const sg = sm + grp * 2 * kStage;  // this group's stages
  const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, lg = lane >> 5;
  const int64_t M = p.M, N = p.N, K = p.K;

  // each XCD a contiguous run of tiles, kGroupRows tile rows high
  const int64_t nbm = (M + BM - 1) / BM, nbn = (N + BN - 1) / BN, tiles = nbm * nbn, total = tiles * p.batch;
  const int64_t pid = blockIdx.x, xcd = pid % mg::kXcds, per = total / mg::kXcds, extra = total % mg::kXcds;
  const int64_t t_all = xcd * per + mg::MinI64(xcd, extra) + pid / mg::kXcds;
  const int64_t bt = t_all / tiles, tt = t_all % tiles;
  const int64_t first_m = tt / (kGroupRows * nbn) * kGroupRows;
  const int64_t gsize = mg::MinI64(nbm - first_m, kGroupRows);
  const int64_t row0 = (first_m + (tt % (kGroupRows * nbn)) % gsize) * BM;
  const int64_t col0 = (tt % (kGroupRows * nbn)) / gsize * BN;

  int64_t a_off, b_off;
  BatchOffsets(p.bm, bt, a_off, b_off);
  const char *Ab = static_cast<const char *>(p.A) + a_off * kAsz;
  const char *Bb = static_cast<const char *>(p.B) + b_off * kBsz;
  const int64_t KA = K * kAsz;                    // bytes of an A row
  const int64_t NB8 = BT ? K * kBsz : N * kBsz;   // bytes of a B row as it lies in memory
  const int64_t a_total = M * KA, b_total = (BT ? N : K) * NB8;
  const int nk = (int)((K + kKStep - 1) / kKStep);
  // Steps read with plain loads.  The others, at most two, are multiplied
  // first, while the loads of the first plain steps are on their way.
  const int nsafe = PlainSteps(K, kKStep, !BT, NB8);
  // this group's plain steps, and the most that one of them has
  const int s0 = (int)((int64_t)grp * nsafe / G), steps = (int)((int64_t)(grp + 1) * nsafe / G) - s0;
  const int rounds = (nsafe + G - 1) / G;
  const unsigned aflip = I8 && p.a_u8 ? mg::kFlip : 0u, bflip = I8 && p.b_u8 ? mg::kFlip : 0u;

  // ---- addresses of this thread's pieces (K step 0) ----
  const int pr = tid >> 3, pc = tid & 7;  // row (of 32) and piece of a 128-byte row
  const char *pa[NA], *pb[NB];
  int wb[NB];  // LDS offset of B piece q
#pragma unroll
  for (int q = 0; q < NA; ++q) pa[q] = Ab + mg::MinI64(row0 + 32 * q + pr, M - 1) * KA + 16 * pc;
  const int wa = pr * 128 + 16 * (pc ^ (pr & 7) ^ ((pr >> 3) & 1));  // + 4096 q
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    if constexpr (BT) {
      pb[q] = Bb + mg::MinI64(col0 + 32 * q + pr, N - 1) * NB8 + 16 * pc;
      wb[q] = wa + 4096 * q;
    } else {
      const int id = tid + 256 * q, kr = id / kPpr, cc = id % kPpr;
      const int64_t cb = col0 * kBsz + 16 * cc;
      pb[q] = Bb + kr * NB8 + (cb < NB8 ? cb : 0);  // columns past N: any bytes, never stored
      if constexpr (I8) {
        const int sw = BN >= 128 ? kr & 7 : (kr >> 1) & 3;
        wb[q] = kr * kBP + 16 * (cc ^ sw);
      } else if constexpr (F8) {
        wb[q] = kr * kBP + 16 * ((2 * cc) ^ (2 * (kr & 3)));  // the second half: 16 bytes on (the XOR is even)
      } else {
        wb[q] = kr * kBP + 16 * (cc ^ (2 * (kr & 3)));
      }
    }
  }
  const int64_t stepA = 128, stepB = BT ? 128 : (int64_t)kKStep * NB8;

  // kSrcF8Chain: the scales of the 16 columns of each of this thread's pieces
  float wsc[SRC == kSrcF8Chain ? NB : 1][16];
  if constexpr (SRC == kSrcF8Chain) {
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t col = col0 + 16 * ((tid + 256 * q) % kPpr) + e;
        wsc[q][e] = static_cast<const float *>(p.scale)[p.scale_per_col ? mg::MinI64(col, N - 1) : 0];
      }
  }

  v4i fa[D][NA], fb[D][NB];
  // Step min(s0 + t, the last plain step) into register set d: always issued, so
  // that the compiler's waits count exact numbers of younger loads (with a
  // branch around the loads past the end every wait drained them all).
  auto load = [&](int t, int d) __attribute__((always_inline)) {
    const int64_t tc = s0 + t < nsafe ? s0 + t : nsafe - 1;
#pragma unroll
    for (int q = 0; q < NA; ++q) fa[d][q] = LoadPiece(pa[q] + tc * stepA);
#pragma unroll
    for (int q = 0; q < NB; ++q) fb[d][q] = LoadPiece(pb[q] + tc * stepB);
  };
  // `left(q)`: bytes of B piece q that lie inside K (kSrcF8Chain: its padding
  // becomes 0 after the scaling, which an infinite scale would make a NaN).
  auto store = [&](const v4i(&a)[NA], const v4i(&b)[NB], char *st, auto left) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NA; ++q) *reinterpret_cast<v4i *>(st + wa + 4096 * q) = a[q] ^ (int)aflip;
    char *sb = st + kASt;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      if constexpr (F8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int x = b[q][2 * h], y = b[q][2 * h + 1];
          v4i w;
          if constexpr (SRC == kSrcF8Chain) {
            const v2f f0 = __builtin_amdgcn_cvt_pk_f32_fp8(x, false), f1 = __builtin_amdgcn_cvt_pk_f32_fp8(x, true);
            const v2f f2 = __builtin_amdgcn_cvt_pk_f32_fp8(y, false), f3 = __builtin_amdgcn_cvt_pk_f32_fp8(y, true);
            const float *s = wsc[q] + 8 * h;
            w = v4i{(int)mg::PackBf16(f0.x * s[0], f0.y * s[1]), (int)mg::PackBf16(f1.x * s[2], f1.y * s[3]),
                    (int)mg::PackBf16(f2.x * s[4], f2.y * s[5]), (int)mg::PackBf16(f3.x * s[6], f3.y * s[7])};
            if (left(q) == 0) w = v4i{0, 0, 0, 0};
          } else {
            w = v4i{mg::Fp8PairLo(x), mg::Fp8PairHi(x), mg::Fp8PairLo(y), mg::Fp8PairHi(y)};
          }
          *reinterpret_cast<v4i *>(sb + wb[q] + 16 * h) = w;
        }
      } else {
        *reinterpret_cast<v4i *>(sb + wb[q]) = b[q] ^ (int)bflip;
      }
    }
  };

  // ---- fragments (the core's lane layouts) ----
  int a_rd[4], b_rd[WB];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) a_rd[kk] = (wm * 32 * MB + lr) * 128 + 16 * ((2 * kk + lg) ^ (lr & 7) ^ ((lr >> 3) & 1));
  const int s16 = lane & 15, g16 = lane >> 4;
#pragma unroll
  for (int j = 0; j < WB; ++j) {
    if constexpr (BT) {
      b_rd[j] = (wn * kWN + j * 32) * 128;
    } else if constexpr (I8) {
      const int kr = 16 * (g16 >> 1) + (s16 >> 1), col = wn * kWN + j * 32 + 16 * (g16 & 1) + 8 * (s16 & 1);
      b_rd[j] = kr * kBP + 16 * ((col >> 4) ^ (BN >= 128 ? kr & 7 : (kr >> 1) & 3)) + (col & 15);
    } else {
      const int kr = 8 * (g16 >> 1) + (s16 >> 2), col = wn * kWN + j * 32 + 16 * (g16 & 1) + 4 * (s16 & 3);
      b_rd[j] = kr * kBP + 16 * ((col >> 3) ^ (2 * (kr & 3))) + ((2 * col) & 15);
    }
  }
  int bt_rd[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) bt_rd[kk] = lr * 128 + 16 * ((2 * kk + lg) ^ (lr & 7) ^ ((lr >> 3) & 1));

  Acc acc[MB][WB];
  int rsum[MB], csum[WB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    rsum[i] = 0;
#pragma unroll
    for (int j = 0; j < WB; ++j) acc[i][j] = Acc{0};
  }
#pragma unroll
  for (int j = 0; j < WB; ++j) csum[j] = 0;

  auto compute = [&](const char *sa) __attribute__((always_inline)) {
    const char *sb = sa + kASt;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      v4i av[MB], bv[WB];
#pragma unroll
      for (int j = 0; j < WB; ++j) {
        if constexpr (BT) {
          bv[j] = *reinterpret_cast<const v4i *>(sb + b_rd[j] + bt_rd[kk]);
        } else if constexpr (I8) {
          const char *b = sb + kk * 32 * kBP + b_rd[j];
          const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((mg::lds_v2i_t)b);
          const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((mg::lds_v2i_t)(b + 8 * kBP));
          bv[j] = v4i{lo.x, lo.y, hi.x, hi.y};
        } else {
          const char *b = sb + kk * 16 * kBP + b_rd[j];
          const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((mg::lds_v4s_t)b));
          const v2i hi =
              __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((mg::lds_v4s_t)(b + 4 * kBP)));
          bv[j] = v4i{lo.x, lo.y, hi.x, hi.y};
        }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) av[i] = *reinterpret_cast<const v4i *>(sa + a_rd[kk] + i * 4096);
      if constexpr (ZP) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int i = 0; i < MB; ++i) rsum[i] = __builtin_amdgcn_sdot4(av[i][e], 0x01010101, rsum[i], false);
#pragma unroll
          for (int j = 0; j < WB; ++j) csum[j] = __builtin_amdgcn_sdot4(bv[j][e], 0x01010101, csum[j], false);
        }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j) {
          if constexpr (I8)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv[j], av[i], acc[i][j], 0, 0, 0);
          else if constexpr (OUT == mg::kOutBf16)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, bv[j]),
                                                                __builtin_bit_cast(v8bf, av[i]), acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, bv[j]),
                                                               __builtin_bit_cast(v8h, av[i]), acc[i][j], 0, 0, 0);
        }
    }
  };

  // ---- K loop: step t is multiplied from LDS stage t % 2 while step t + 1
  // goes from its registers into the other stage (whose last reads ended at
  // the barrier before) and steps t + 2 .. t + D are on their way ----
  auto tail = [&]() __attribute__((always_inline)) {
#pragma unroll 1
    for (int t = nsafe; t < nk; ++t) {
      if (G > 1 && grp != 0) {  // the first group's
        LdsBarrier();
        LdsBarrier();
        continue;
      }
      v4i a[NA], b[NB];
      const int64_t ka = KA - (int64_t)t * 128 - 16 * pc;  // bytes of the row left at this thread's piece
      int64_t nb[NB];                                      // valid bytes of each B piece
#pragma unroll
      for (int q = 0; q < NB; ++q) nb[q] = BT ? ka : ((int64_t)t * kKStep + (tid + 256 * q) / kPpr < K ? 16 : 0);
      if (a_total >= 16 && b_total >= 16) {
        const char *qa[NA], *qb[NB];
#pragma unroll
        for (int q = 0; q < NA; ++q) {
          qa[q] = pa[q] + t * stepA;
          a[q] = LoadPiece(qa[q] - TailBack(Ab, a_total, qa[q]));
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          qb[q] = pb[q] + t * stepB;
          b[q] = LoadPiece(qb[q] - TailBack(Bb, b_total, qb[q]));
        }
#pragma unroll
        for (int q = 0; q < NA; ++q) a[q] = TailFix(a[q], TailBack(Ab, a_total, qa[q]), ka, aflip);
#pragma unroll
        for (int q = 0; q < NB; ++q) b[q] = TailFix(b[q], TailBack(Bb, b_total, qb[q]), nb[q], bflip);
      } else {
#pragma unroll
        for (int q = 0; q < NA; ++q) a[q] = TailBytes(Ab, a_total, pa[q] + t * stepA, ka, aflip);
#pragma unroll
        for (int q = 0; q < NB; ++q) b[q] = TailBytes(Bb, b_total, pb[q] + t * stepB, nb[q], bflip);
      }
      store(a, b, sm, [&](int q) { return nb[q]; });
      LdsBarrier();
      compute(sm);
      LdsBarrier();
    }
  };
  if (nsafe > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d);
    tail();
    auto whole = [](int) { return 16; };
    store(fa[0], fb[0], sg, whole);
    load(D, 0);
    LdsBarrier();
    for (int t = 0; t < rounds; t += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (t + d >= rounds) break;
        const int n = (d + 1) % D;
        store(fa[n], fb[n], sg + ((d + 1) & 1) * kStage, whole);
        load(t + d + 1 + D, n);
        if (G == 1 || t + d < steps) compute(sg + (d & 1) * kStage);
        LdsBarrier();
      }
    }
  } else {
    tail();
  }

  // ---- the groups' sums, added in order by the first through the stages ----
  if constexpr (G > 1) {
    static_assert(MB == 1 && WB == 1 && !I8, "one block of fp32 sums per wave");
    v4f *part = reinterpret_cast<v4f *>(sg) + wave * 4 * 64 + lane;
    if (grp != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[64 * e] = v4f{acc[0][0][4 * e], acc[0][0][4 * e + 1], acc[0][0][4 * e + 2], acc[0][0][4 * e + 3]};
    }
    __syncthreads();
    if (grp != 0) return;
#pragma unroll
    for (int g = 1; g < G; ++g) {
      const v4f *o = part + g * (2 * kStage / 16);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[0][0][e] += o[64 * (e / 4)][e % 4];
    }
  }

  // ---- zero-point terms (mod 2^32): Y = sum a'b' + beta_j RA_i + alpha_i Q_j, Q_j = CB_j + K beta_j ----
  QResolved qv{p.alpha_scalar, p.beta_scalar, p.cs, p.zy};
  if constexpr (I8) qv = ResolveQ(p.dev, p.a_u8, p.b_u8, p.y_signed, p.alpha_scalar, p.beta_scalar, p.cs, p.zy);
  if constexpr (OUT == mg::kOutQ8) qv = FiniteScale(qv);
  int32_t *zc = zsum + (ZP ? wave * 2 * kWN : 0);
  if constexpr (ZP) {
#pragma unroll
    for (int j = 0; j < WB; ++j) {
      const int64_t col = col0 + wn * kWN + j * 32 + lr;
      const int v = csum[j] + __shfl_xor(csum[j], 32);
      int be = qv.beta;
      if (p.b_zp) {
        const uint8_t z = p.b_zp[col < N ? col : N - 1];
        be = p.b_u8 ? 128 - (int)z : -(int)(int8_t)z;
      }
      if (lg == 0) {
        zc[j * 32 + lr] = (int)((unsigned)v + (unsigned)K * (unsigned)be);
        zc[kWN + j * 32 + lr] = be;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // ---- epilogue: lane (lr, lg) of block (i, j) holds row 32 i + lr and, in
  // registers 4 g .. 4 g + 3, columns 32 j + 8 g + 4 lg + 0..3; each wave
  // stages 32 rows at a time in its own LDS area and writes row pieces ----
  char *stg = sm + wave * 32 * kPitch;
  const float q_bias = p.y_signed ? 128.f : 0.f;
  const float q_zy = qv.zy + q_bias, q_lo = p.qmin + q_bias, q_hi = p.qmax + q_bias;
  const unsigned q_flip = p.y_signed ? 0x80808080u : 0u;
  const int64_t cw = col0 + wn * kWN;  // first column of the wave
  char *Y = static_cast<char *>(p.Y) + bt * M * N * kOsz;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int64_t br = row0 + (wm * MB + i) * 32;
    const int64_t row = mg::MinI64(br + lr, M - 1);
    int32_t ra_r = 0, al_r = 0;
    if constexpr (ZP) {
      ra_r = rsum[i] + __shfl_xor(rsum[i], 32);
      al_r = qv.alpha;
      if (p.a_zp) al_r = p.a_u8 ? 128 - (int)p.a_zp[row] : -(int)(int8_t)p.a_zp[row];
    }
    float cs_r = qv.cs;
    double bias_r = 0.0;
    if constexpr (OUT == mg::kOutQ8Row) {
      cs_r = p.row_xs * p.row_wscale[p.row_wscale_per ? row : 0] / p.row_ys;
      if (p.row_bias) bias_r = (double)p.row_bias[row];
    }
#pragma unroll
    for (int j = 0; j < WB; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int cl = j * 32 + g * 8 + lg * 4;
        char *dst = stg + lr * kPitch + cl * kOsz;
        if constexpr (I8) {
          unsigned v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = (unsigned)acc[i][j][4 * g + e];
            if constexpr (ZP)
              v[e] += (unsigned)zc[kWN + cl + e] * (unsigned)ra_r + (unsigned)al_r * (unsigned)zc[cl + e];
          }
          if constexpr (OUT == mg::kOutI32) {
            *reinterpret_cast<v4i *>(dst) = v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
          } else {
            // ties-to-even before the zero point, then saturation (signed
            // outputs biased by 128, exact on these integers)
            unsigned packed = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float f;
              if constexpr (OUT == mg::kOutQ8Row) {
                f = __builtin_rintf((float)((double)(int32_t)v[e] + bias_r) * cs_r) + q_zy;
                if (f != f) f = q_bias;
              } else {
                f = __builtin_rintf((float)(int32_t)v[e] * qv.cs) + q_zy;
              }
              packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(f, q_lo, q_hi), e, packed);
            }
            *reinterpret_cast<unsigned *>(dst) = packed ^ q_flip;
          }
        } else {
          float f[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f[e] = acc[i][j][4 * g + e];
            if constexpr (SRC == kSrcF8) {  // the column's dequantization scale
              const int64_t si = p.scale_per_col ? mg::MinI64(cw + cl + e, N - 1) : 0;
              f[e] *= static_cast<const float *>(p.scale)[si];
            }
          }
          if constexpr (OUT == mg::kOutBf16) {
            *reinterpret_cast<v2i *>(dst) = v2i{(int)mg::PackBf16(f[0], f[1]), (int)mg::PackBf16(f[2], f[3])};
          } else {
            typedef _Float16 v4h __attribute__((ext_vector_type(4)));
            *reinterpret_cast<v4h *>(dst) = v4h{(_Float16)f[0], (_Float16)f[1], (_Float16)f[2], (_Float16)f[3]};
          }
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int kPc = kWN * kOsz / 16;  // pieces per staged row
    constexpr int kPl = 32 * kPc / 64;    // pieces per lane
    v4i piece[kPl];
#pragma unroll
    for (int c = 0; c < kPl; ++c) {
      const int id = c * 64 + lane;
      piece[c] = *reinterpret_cast<const v4i *>(stg + (id / kPc) * kPitch + (id % kPc) * 16);
    }
#pragma unroll
    for (int c = 0; c < kPl; ++c) {
      const int id = c * 64 + lane, rr = id / kPc, cc = id % kPc;
      const int64_t left = (N - cw) * kOsz - 16 * cc;  // bytes of the row from this piece on
      if (br + rr >= M || left <= 0) continue;
      char *out = Y + ((br + rr) * N + cw) * kOsz + 16 * cc;
      if (left >= 16) {
        __builtin_memcpy(out, &piece[c], 16);
      } else {
#pragma unroll
        for (int e = 0; e < 16 / kOsz; ++e)
          if (e * kOsz < left) {
            const unsigned w = (unsigned)piece[c][e * kOsz / 4] >> (8 * (e * kOsz & 3));
            if constexpr (kOsz == 4) *reinterpret_cast<unsigned *>(out + 4 * e) = w;
            else if constexpr (kOsz == 2) *reinterpret_cast<uint16_t *>(out + 2 * e) = (uint16_t)w;
            else out[e] = (char)w;
          }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

inline int64_t Tiles(const GemmArgs &p, int side) {
  return (p.M + side - 1) / side * ((p.N + side - 1) / side) * p.batch;
}

// Whether p goes to 64 x 64 tiles.  Where the core takes p as well (`core`), up
// to one of them per CU: at K = 4096, int8 / fp8 / fp16, 256 x 4096 outputs (256
// small tiles) take 14.1 / 24.0 / 23.7 us here and 15.5 / 25.6 / 24.2 us in the
// core's 128 x 128 tiles; 512 x 4096 (512 small tiles) 21.4 / 35.4 / 34.3 against
// 16.7 / 26.6 / 25.6 us: a small tile reads each operand byte for half as many
// products as the core's.  The shapes the core does not take go on to two per CU, then to
// 128 x 128 tiles of this kernel (1024 x 4096: 39.4 -> 30.0 us int8, 67.1 -> 51.0 us
// fp16; at 688 small tiles the two tie).
inline bool PrefersSmallTile(const GemmArgs &p, bool core) { return Tiles(p, 64) <= (core ? 256 : 512); }

// Whether the 64 x 64 tile takes two groups of waves per workgroup, each half of
// the K steps: with at most one tile per CU, one group's step is a chain of LDS
// writes, a barrier, LDS reads and four dependent MFMAs; two groups fill part of
// its waits (fp16 150 x 4096 x 4096 with two: the waves still wait half of their
// time, the LDS is 30% and the matrix cores are 14% busy).  The exchange at the end costs about 1 us, so it pays for long K: fp16,
// one -> two groups, 150 x 4096 outputs at K = 1536 9.5 -> 9.6 us, 2048 11.2 ->
// 11.2, 3072 16.1 -> 15.3, 4096 22.6 -> 19.4, 8192 40.8 -> 32.9; fp8, whose
// decode lengthens the chain, 1536 10.4 -> 9.9, 4096 21.4 -> 18.5 us.  int8
// steps are twice as deep: 4096 12.8 -> 13.4 us.  Four groups were within 0.6 us
// of two from K = 2048 to 4096 and lost up to 1.4 us below.  With rows of both
// operands off 16 bytes the loads bound it (fp16 150 x 4097 at K = 4089 29.8 ->
// 32.7 us).
template <int KIND, int SRC> inline bool PrefersTwoGroups(const GemmArgs &p) {
  if (KIND == mg::kI8 || Tiles(p, 64) > 256) return false;
  if (SRC == kSrcF8 || SRC == kSrcF8Chain) return p.K >= 1536;
  return p.K >= 3072 && (p.K % 8 == 0 || (SRC == kSrcRow && p.N % 8 == 0));
}

// Whether 64 x 128 tiles take a problem of more 64 x 64 tiles than CUs: at most
// one per CU, they keep any CU from two of the small ones: twice the outputs for
// one chain of steps and half again the LDS traffic (72 KB a step against 48).
// Neither unit is near full then (u8 335 x 3001, K = 1001: LDS 7%, matrix cores 4%,
// 0.6 waves per SIMD): the chain's latency bounds it.  335 x 3001
// outputs, 64 x 64 -> 64 x 128: int8 K = 513 11.2 -> 8.8 us, 1001 13.0 -> 10.4, 4090
// 29.3 -> 25.2; fp16 11.3 -> 10.2, 15.3 -> 13.1, 42.5 -> 35.2.  Steps in flight: two
// for int8 (four: 9.9, 11.5, 25.0), four for fp16 (two: 9.7, 12.7, 39.2).  fp8 weights
// stay with the small tile (K = 1001 14.6 -> 14.9, 4090 38.1 -> 40.7).  Two of them
// per CU also beat two rounds of 128 x 128 ones, which rows or columns left over
// fill badly: 300 x 11007, 128 x 128 -> 64 x 128, int8 K = 1001 21.9 -> 16.1 us, 4090
// 59.6 -> 41.8, fp16 31.8 -> 22.7 and 82.5 -> 61.1; against one round they lose (1000 x
// 3001 at K = 4090 37.9 -> 41.3, 57.2 -> 60.1), three rounds against two too (1500 x
// 4001 60.7 -> 66.9).
inline int64_t WideTiles(const GemmArgs &p) { return (p.M + 63) / 64 * ((p.N + 127) / 128) * p.batch; }
inline bool PrefersWideTile(const GemmArgs &p) {
  const int64_t wide = WideTiles(p);
  return (Tiles(p, 64) > 256 && wide <= 256) || (Tiles(p, 128) > 256 && wide <= 512);
}

template <int KIND, int SRC, int OUT, bool ZP> inline void Launch(const GemmArgs &p, bool big, hipStream_t s) {
  if constexpr (SRC == kSrcRow || SRC == kSrcT) {
    if (PrefersWideTile(p)) {
      hipLaunchKernelGGL((TileGemmKernel<KIND, SRC, OUT, ZP, 1, 2, KIND == mg::kI8 ? 2 : 4, 1>),
                         dim3((unsigned)WideTiles(p)), dim3(256), 0, s, p);
      return;
    }
  }
  if (big) {
    hipLaunchKernelGGL((TileGemmKernel<KIND, SRC, OUT, ZP, 2, 2, 2, 1>), dim3((unsigned)Tiles(p, 128)), dim3(256), 0, s, p);
    return;
  }
  const dim3 grid((unsigned)Tiles(p, 64));
  if constexpr (KIND != mg::kI8) {
    if (PrefersTwoGroups<KIND, SRC>(p)) {
      hipLaunchKernelGGL((TileGemmKernel<KIND, SRC, OUT, ZP, 1, 1, 4, 2>), grid, dim3(512), 0, s, p);
      return;
    }
  }
  hipLaunchKernelGGL((TileGemmKernel<KIND, SRC, OUT, ZP, 1, 1, 4, 1>), grid, dim3(256), 0, s, p);
}

}  // namespace tg
}  // namespace onnxl_amd
