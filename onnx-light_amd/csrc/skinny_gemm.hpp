// Decode GEMM for gfx950: a few rows of A (one or two 16-row MFMA operands)
// times a one-byte weight B [K, N], int8 / uint8 or float8e4m3fn, and the same
// for every expert of a small grouped call.
//
// Bound by reading B once.  A tile GEMM leaves that to as many workgroups as
// N has tiles, each walking all of K behind a barrier per step; here
//  - a workgroup owns 16 CW columns over all of K, its W waves take every W-th
//    chunk of KC rows, and their sums meet in LDS once at the end: no barrier
//    in the loop and no workspace;
//  - a lane loads CW bytes of each of its KC / 4 rows (16 lanes read 16 CW
//    consecutive bytes of a row; CW = 8 a whole 128-byte line), two chunks in
//    flight per wave, and transposes 4 x 4 bytes in registers: column CW i + c
//    of lane i is then the MFMA's weight operand of tile c, whose order over k
//    is the order of the activations' 16-byte loads.  B never touches LDS.
//  - the weights are the MFMA's row operand, the rows of A its columns, so the
//    idle part of a 16-row product costs only matrix-core time, of which a
//    decode has plenty.
//  - int8 zero points: a row of ones behind the last row of A makes the column
//    sums of B one more row of the product.
//  - grouped (GRP): a workgroup counts the (token, selection) pairs of every
//    expert and finds its own 16 MT of one expert by itself, so a call is one
//    launch with no routing pass before it.  An expert with more pairs has more
//    workgroups, not longer ones: 32 tokens, top 2 of 8 experts [4096, 14336], all
//    pairs to one expert 214.8 us where one workgroup per column tile walked its
//    expert's pairs, 40.8 now (the routed core 85.8); skewed 202 -> 113 (167); even 99.5.
#pragma once

#include "mfma_gemm.hpp"
#include "tile_gemm.hpp"

namespace onnxl_amd {
namespace sk {

using mg::v2i;
using mg::v4f;
using mg::v4i;
using mg::v8bf;

constexpr int kMaxPairs = 1024;   // (token, selection) pairs a grouped call may have
constexpr int kMaxGroups = 4096;  // and groups

struct Args {
  mg::GemmArgs g;
  const void *idx;  // grouped: [M, grp_sel] INT32 / INT64 group of each pair
  int idx64;
};

// 4 x 4 byte transpose: d[c] = byte c of r0, r1, r2, r3.
__device__ __forceinline__ void Transpose4(unsigned r0, unsigned r1, unsigned r2, unsigned r3, unsigned (&d)[4]) {
  const unsigned a = __builtin_amdgcn_perm(r1, r0, 0x05010400u), b = __builtin_amdgcn_perm(r3, r2, 0x05010400u);
  const unsigned c = __builtin_amdgcn_perm(r1, r0, 0x07030602u), e = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
  d[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
  d[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  d[2] = __builtin_amdgcn_perm(e, c, 0x05040100u);
  d[3] = __builtin_amdgcn_perm(e, c, 0x07060302u);
}

// Sum over this lane and those before it, by DPP: the six exchanges through LDS
// that __shfl_up takes cost 0.5 us at the start of every workgroup.
__device__ __forceinline__ int WaveScan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // lane 15 of rows 0 and 2 to rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // lane 31 to rows 2 and 3
  return v;
}

template <int KIND, int OUT, bool ZP, int CW, int W, int MT, bool GRP>
__global__ __launch_bounds__(64 * W, CW == 8 && MT == 2 ? 2 : 4) void SkinnyKernel(const Args q) {
  const mg::GemmArgs &p = q.g;
  constexpr bool I8 = KIND == mg::kI8;
  // A chunk is KC rows of B, 64 bytes of each row of A; lane group g4 owns rows
  // (KC / 4) g4 .. of it and reads them 8 at a time (int8: in two halves), one
  // MFMA operand of 8 consecutive k each time.
  constexpr int KC = I8 ? 64 : 32, H = KC / 32, RPL = KC / 4;
  constexpr int COLS = 16 * CW, NW = CW / 4;      // columns of the workgroup, dwords per loaded row
  constexpr int kAsz = I8 ? 1 : 2;
  constexpr int kOsz = OUT == mg::kOutI32 ? 4 : (OUT == mg::kOutQ8 ? 1 : 2);
  constexpr int PITCH = COLS + 4;
  using Acc = std::conditional_t<I8, v4i, v4f>;
  using El = std::conditional_t<I8, int, float>;
  __shared__ __align__(16) El red[W][16][PITCH];
  __shared__ int rsums[ZP ? W : 1][ZP ? 16 * MT : 1];
  __shared__ int csums[ZP ? COLS : 1];
  __shared__ int pairs[GRP ? 16 * MT : 1];  // this workgroup's (token, selection) pairs

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t M = p.M, N = p.N, K = p.K;
  // each XCD a contiguous run of column tiles (grouped: about one unit each);
  // 32-bit and made scalar, so that B's addresses are a scalar base and one
  // 32-bit offset per lane
  const unsigned nbn = (unsigned)((N + COLS - 1) / COLS), pid = blockIdx.x;
  auto tile_of = [&](unsigned total) __attribute__((always_inline)) {
    const unsigned xcd = pid % mg::kXcds, extra = total % mg::kXcds;
    return xcd * (total / mg::kXcds) + (xcd < extra ? xcd : extra) + pid / mg::kXcds;
  };
  unsigned t = 0;
  int64_t a_off = 0, b_off = 0, rbase = 0;
  int grp = 0, tr = (int)M;  // rows of this workgroup
  if constexpr (GRP) {
    // A unit of work is up to R pairs of one group: count them, find this one.
    constexpr int R = 16 * MT;
    static_assert(sizeof(red) >= (kMaxGroups + kMaxPairs) * sizeof(int), "both lists, before the sums need it");
    int *cnt = reinterpret_cast<int *>(red), *sel = cnt + p.grp_count;  // pairs per group, group of each pair
    const int P = (int)M * p.grp_sel, G = p.grp_count;
    for (int g = tid; g < G; g += 64 * W) cnt[g] = 0;
    __syncthreads();
    for (int i = tid; i < P; i += 64 * W) {
      const int64_t v = q.idx64 ? static_cast<const int64_t *>(q.idx)[i]
                                : (int64_t) static_cast<const int32_t *>(q.idx)[i];
      const bool in = v >= 0 && v < G;
      sel[i] = in ? (int)v : -1;
      if (in) atomicAdd(&cnt[v], 1);
      // a pair outside the groups gets a NaN row, a column tile of it from each
      // of the first workgroups
      if (!in && pid < nbn)
        for (int64_t n = (int64_t)pid * COLS; n < mg::MinI64((int64_t)(pid + 1) * COLS, N); ++n)
          static_cast<uint16_t *>(p.Y)[i * N + n] = 0x7fc0u;
    }
    __syncthreads();
    // units of the groups b .. b + lane
    auto units = [&](int b) __attribute__((always_inline)) {
      return WaveScan(b + lane < G ? (cnt[b + lane] + R - 1) / R : 0);
    };
    int v = units(0);
    int all = __builtin_amdgcn_readlane(v, 63);
    for (int b = 64; b < G; b += 64) all += __builtin_amdgcn_readlane(units(b), 63);
    if (pid >= (unsigned)all * nbn) return;
    t = tile_of((unsigned)all * nbn);
    int unit = __builtin_amdgcn_readfirstlane((int)(t / nbn));  // below `all`, so that a group is found
    for (int sum; unit >= (sum = __builtin_amdgcn_readlane(v, 63)); v = units(grp)) {
      unit -= sum;
      grp += 64;
    }
    const int l = __builtin_ctzll(__ballot(v > unit));
    unit -= l > 0 ? __builtin_amdgcn_readlane(v, l - 1) : 0;
    grp += l;
    tr = __builtin_amdgcn_readfirstlane(min(cnt[grp] - unit * R, R));
    // the group's pairs from unit * R on, in the order of their indices (the same
    // in every workgroup)
    if (wave == 0) {
      for (int b = 0, rank = -unit * R; b < P && rank < R; b += 256) {
        int g[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = b + 64 * e + lane < P ? sel[b + 64 * e + lane] : -1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint64_t hit = __ballot(g[e] == grp);
          const int r = rank + __popcll(hit & ((uint64_t(1) << lane) - 1));
          if (g[e] == grp && r >= 0 && r < R) pairs[r] = b + 64 * e + lane;
          rank += __popcll(hit);
        }
      }
    }
    __syncthreads();
    b_off = grp * p.grp_b_stride;
  } else {
    t = tile_of(gridDim.x);
    const int entry = __builtin_amdgcn_readfirstlane((int)(t / nbn));  // batch entry
    BatchOffsets(p.bm, entry, a_off, b_off);
    rbase = entry * M;  // first row of this batch entry in Y
  }
  const int64_t n0 = (int64_t)__builtin_amdgcn_readfirstlane((int)(t % nbn)) * COLS;
  const char *Ab = static_cast<const char *>(p.A) + a_off * kAsz;
  const char *Bb = static_cast<const char *>(p.B) + b_off;
  const int64_t KA = K * kAsz;
  // chunks read with plain loads; the one after them, if any, holds k past K
  // or a row whose last columns a whole load would cross the matrix's end at
  const int nch = (int)((K + KC - 1) / KC);
  const int nfull = K % KC == 0 && N % CW == 0 ? nch : nch - 1;
  const int nj = wave < nfull ? (nfull - wave + W - 1) / W : 0;  // this wave's plain chunks
  const unsigned aflip = I8 && p.a_u8 ? mg::kFlip : 0u;
  const bool bflip = I8 && p.b_u8;

  const int i16 = lane & 15, g4 = lane >> 4;
  const int64_t col = n0 + CW * i16;
  const unsigned bvo = (unsigned)(RPL * g4 * N + (col < N ? col : 0));
  const char *pa[MT];
  bool one[MT];  // ZP: this lane's row is the row of ones
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    int64_t row = min(16 * m + i16, tr - 1);
    if constexpr (GRP) row = pairs[row] / p.grp_sel;
    pa[m] = Ab + row * KA + 16 * g4;
    one[m] = ZP && 16 * m + i16 == tr;
  }
  Acc acc[CW][MT];
  int rs[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    rs[m] = 0;
#pragma unroll
    for (int c = 0; c < CW; ++c) acc[c][m] = Acc{0, 0, 0, 0};
  }
  unsigned fb[2][8][NW];
  v4i fa[2][MT];
  // Chunk j of this wave (past the end: the last one again, so that the
  // waits count exact numbers of younger loads).
  auto chunk = [&](int j) __attribute__((always_inline)) -> int64_t {
    return wave + (int64_t)(j < nj ? j : nj - 1) * W;
  };
  auto load_a = [&](int j, int d) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MT; ++m) fa[d][m] = tg::LoadPiece(pa[m] + chunk(j) * 64);
  };
  auto load_b = [&](int j, int h, int d) __attribute__((always_inline)) {
    const char *b = Bb + (chunk(j) * KC + 8 * h) * N;
#pragma unroll
    for (int r = 0; r < 8; ++r) __builtin_memcpy(fb[d][r], b + r * N + bvo, CW);
    __builtin_amdgcn_sched_barrier(0);
  };
  // A's operands as they enter the products (once per chunk)
  auto ready_a = [&](v4i(&a)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if constexpr (I8) a[m] ^= (int)aflip;
      if constexpr (ZP) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          rs[m] = __builtin_amdgcn_sdot4(a[m][e], 0x01010101, rs[m], false);
          a[m][e] = one[m] ? 0x01010101 : a[m][e];  // rows of B past K are zero
        }
      }
    }
  };
  auto process = [&](const unsigned(&b)[8][NW], const v4i(&a)[MT], int h) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      unsigned d0[4], d1[4];
      Transpose4(b[0][w], b[1][w], b[2][w], b[3][w], d0);
      Transpose4(b[4][w], b[5][w], b[6][w], b[7][w], d1);
      if (bflip) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          d0[c] ^= mg::kFlip;
          d1[c] ^= mg::kFlip;
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (I8) {
          const long x = __builtin_bit_cast(long, v2i{(int)d0[c], (int)d1[c]});
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[4 * w + c][m] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                x, __builtin_bit_cast(long, v2i{a[m][2 * h], a[m][2 * h + 1]}), acc[4 * w + c][m], 0, 0, 0);
        } else {
          const v4i x = {mg::Fp8PairLo((int)d0[c]), mg::Fp8PairHi((int)d0[c]), mg::Fp8PairLo((int)d1[c]),
                         mg::Fp8PairHi((int)d1[c])};
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[4 * w + c][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(v8bf, x), __builtin_bit_cast(v8bf, a[m]), acc[4 * w + c][m], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // one chunk of parity z, and the loads that take its registers' place
  auto step = [&](int j, int z, bool more) __attribute__((always_inline)) {
    ready_a(fa[z]);
    if constexpr (H == 2) {
      process(fb[0], fa[z], 0);
      if (more) {
        load_a(j + 1, 1 - z);
        load_b(j + 1, 0, 0);
      }
      process(fb[1], fa[z], 1);
      if (more) load_b(j + 1, 1, 1);
    } else {
      process(fb[z], fa[z], 0);
      if (more) {
        load_a(j + 2, z);
        load_b(j + 2, 0, z);
      }
    }
  };
  if (nj > 0) {
    load_a(0, 0);
    load_b(0, 0, 0);
    if constexpr (H == 1) load_a(1, 1);
    load_b(H == 1 ? 1 : 0, H - 1, 1);
    for (int j = 0; j + 2 <= nj; j += 2) {
      step(j, 0, true);
      step(j + 1, 1, true);
    }
    if (nj & 1) step(0, 0, false);
  }
  if (nfull < nch && nfull % W == wave) {  // the guarded chunk
    v4i a[MT];
    const char *bend = Bb + K * N - CW;  // the last whole load of the matrix
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const char *at = pa[m] + (int64_t)nfull * 64;
      const int64_t s = tg::TailBack(Ab, M * KA, at);
      a[m] = tg::TailFix(tg::LoadPiece(at - s), s, KA - (int64_t)nfull * 64 - 16 * g4, aflip);
    }
    ready_a(a);
#pragma unroll
    for (int h = 0; h < H; ++h) {
      unsigned b[8][NW];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int64_t k = (int64_t)nfull * KC + RPL * g4 + 8 * h + r;
        const char *at = Bb + mg::MinI64(k, K - 1) * N + (col < N ? col : 0);
        const int back = at > bend ? (int)(at - bend) : 0;
        uint64_t v = 0;
        __builtin_memcpy(&v, at - back, CW);
        v >>= 8 * back;
        if (k >= K) v = bflip ? ~uint64_t(0) / 255 * 128 : 0;
        __builtin_memcpy(b[r], &v, CW);
      }
      process(b, a, h);
    }
  }

  // ---- the waves' sums: lane (i16, g4) of tile c holds row i16 and, in
  // register r, column CW (4 g4 + r) + c ----
  if constexpr (ZP) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      int v = rs[m] + __shfl_xor(rs[m], 16);
      v += __shfl_xor(v, 32);
      if (g4 == 0) rsums[wave][16 * m + i16] = v;
    }
  }
  QResolved qv{p.alpha_scalar, p.beta_scalar, p.cs, p.zy};
  if constexpr (I8) qv = ResolveQ(p.dev, p.a_u8, p.b_u8, p.y_signed, p.alpha_scalar, p.beta_scalar, p.cs, p.zy);
  if constexpr (OUT == mg::kOutQ8) qv = FiniteScale(qv);
  const int mone = tr / 16;  // ZP: the operand that holds the row of ones (tr < 16 MT)
#pragma unroll
  for (int m = MT - 1; m >= 0; --m) {
    if (16 * m >= tr && !(ZP && m == mone)) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < NW; ++h) {
        Acc v;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = acc[4 * h + c][m][r];
        *reinterpret_cast<Acc *>(&red[wave][i16][CW * (4 * g4 + r) + 4 * h]) = v;
      }
    __syncthreads();
    auto sum = [&](int row, int n4) __attribute__((always_inline)) {
      Acc v = *reinterpret_cast<const Acc *>(&red[0][row][4 * n4]);
#pragma unroll
      for (int w = 1; w < W; ++w) v += *reinterpret_cast<const Acc *>(&red[w][row][4 * n4]);
      return v;
    };
    if constexpr (ZP) {
      if (m == mone && tid < COLS / 4) *reinterpret_cast<Acc *>(&csums[4 * tid]) = sum(tr % 16, tid);
      __syncthreads();
    }
    for (int id = tid; id < 16 * (COLS / 4); id += 64 * W) {
      const int mr = id / (COLS / 4), n4 = id % (COLS / 4);
      const int row = 16 * m + mr;  // row of this workgroup
      const int64_t n = n0 + 4 * n4;
      if (row >= tr || n >= N) continue;
      const Acc s = sum(mr, n4);
      const int64_t yrow = GRP ? (int64_t)pairs[row] : rbase + row;
      char *y = static_cast<char *>(p.Y) + (yrow * N + n) * kOsz;
      const int left = (int)mg::MinI64(N - n, 4);
      if constexpr (I8) {
        unsigned v[4];
        int ra = 0, al = 0;
        if constexpr (ZP) {
#pragma unroll
          for (int w = 0; w < W; ++w) ra += rsums[w][row];
          al = qv.alpha;
          if (p.a_zp) al = p.a_u8 ? 128 - (int)p.a_zp[row] : -(int)(int8_t)p.a_zp[row];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = (unsigned)s[e];
          if constexpr (ZP) {
            int be = qv.beta;
            if (p.b_zp) {
              const uint8_t z = p.b_zp[mg::MinI64(n + e, N - 1)];
              be = p.b_u8 ? 128 - (int)z : -(int)(int8_t)z;
            }
            v[e] += (unsigned)be * (unsigned)ra +
                    (unsigned)al * ((unsigned)csums[4 * n4 + e] + (unsigned)K * (unsigned)be);
          }
        }
        if constexpr (OUT == mg::kOutI32) {
          if (left == 4) __builtin_memcpy(y, v, 16);
          else
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (e < left) reinterpret_cast<unsigned *>(y)[e] = v[e];
        } else {
          const float bias = p.y_signed ? 128.f : 0.f;
          unsigned packed = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f = __builtin_rintf((float)(int32_t)v[e] * qv.cs) + qv.zy + bias;
            packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(f, p.qmin + bias, p.qmax + bias), e,
                                                    packed);
          }
          packed ^= p.y_signed ? 0x80808080u : 0u;
          if (left == 4) __builtin_memcpy(y, &packed, 4);
          else
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (e < left) y[e] = (char)(packed >> (8 * e));
        }
      } else {
        unsigned o[2];
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t si = grp * p.scale_grp_stride + (p.scale_per_col ? mg::MinI64(n + e, N - 1) : 0);
          f[e] = s[e] * static_cast<const float *>(p.scale)[si];
        }
        if constexpr (GRP) {
          if (p.grp_bias) {  // MatMul, then Add: the sum rounded, the bias added, rounded again
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint16_t b = static_cast<const uint16_t *>(p.grp_bias)[grp * N + mg::MinI64(n + e, N - 1)];
              f[e] = __builtin_bit_cast(float, (mg::PackBf16(f[e], 0.f) & 0xffffu) << 16) +
                     __builtin_bit_cast(float, (unsigned)b << 16);
            }
          }
        }
        o[0] = mg::PackBf16(f[0], f[1]);
        o[1] = mg::PackBf16(f[2], f[3]);
        if (left == 4) __builtin_memcpy(y, o, 8);
        else
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (e < left) reinterpret_cast<uint16_t *>(y)[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
      }
    }
    __syncthreads();
  }
}

// Whether a dense product goes here.  Up to 16 rows (15 with zero points, which
// need a row of ones) whenever K gives the 16 waves a few chunks: at K = 256
// 3.8 against the small tile's 4.1 us, at K = 4096 int8 / fp8 with 8 rows
// N = 4096 7.4 against 12.4 / 8.2 against 20.8 us, N = 11008 11.8 against 15.0 /
// 12.4 against 24.1 us.  Up to 32 rows two operands share a pass over B; the
// small tile wastes less there, so only deep products with few column tiles
// come here (K = 4096, 24 rows, int8: N = 4096 10.1 against 12.5 us, N = 8192 15.7
// against 14.7 us; fp8: N = 4096 13.3 against 20.8 us, N = 14336 19.9 against
// 24.7 us; K = 1024 ties).
inline bool PrefersSkinny(const mg::GemmArgs &p, bool i8, bool zp) {
  if (p.K < 256 || p.N < 64 || p.N > (int64_t(1) << 26)) return false;  // 48 N fits the 32-bit lane offsets
  const int64_t rows = p.M + (zp ? 1 : 0);
  if (rows <= 16) return true;
  return rows <= 32 && p.K >= 2048 && (p.N + 63) / 64 * p.batch <= (i8 ? 64 : 256);
}

// Whether a grouped call goes here instead of the routed core, whose tiles are
// nearly empty then: by the average number of pairs per expert and the columns
// of all experts.  bf16 x fp8 experts, K = 4096, evenly routed, here against the
// core's 128-row tiles: 8 x N = 14336 with 8 / 12 / 16 / 32 pairs per expert 100 / 109 /
// 117 / 164 against 107 / 109 / 110 / 115 us; 8 x N = 4096 with 16 / 32 pairs 26.6 / 49.3
// against 34.1 / 38.2; 8 x N = 1024 with 32 / 64 / 128 pairs 21.1 / 22.6 / 41.4 against
// 30.9 / 31.6 / 31.8 (the line is below what 64 would allow).  Skewed routing, where
// busy experts' columns are read once per 16 pairs: 8 x 14336 with 12 pairs 122 against 113,
// 8 x 4096 with 16 pairs 41.4 against 34.6.
inline bool PrefersSkinnyGrouped(const mg::GemmArgs &p) {
  const int64_t pairs = p.M * p.grp_sel, cols = p.grp_count * p.N;
  const int64_t most = cols <= 16384 ? 32 : (cols <= 65536 ? 16 : 12);
  return pairs <= kMaxPairs && pairs <= most * p.grp_count && p.N >= 64 && p.N <= (int64_t(1) << 26) && p.K >= 32;
}

}  // namespace sk
}  // namespace onnxl_amd
