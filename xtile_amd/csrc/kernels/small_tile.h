// The wave-private tiles of gemm_small.hip and conv_tiles.hip: a workgroup of
// four waves that split K between them (stage s of kStageK bytes belongs to wave
// s % 4).  Each wave fills a ring of its own in LDS, multiplies the whole BM x BN
// tile and meets the others once, at the end.
//
// Stage layout: A [BM rows][128 B], then B [128 / ES k rows][BN * ES B].  An
// instruction fills 1 KB, lane L at byte 16 L; the chunk each lane fetches
// swizzles the tile: A row r keeps its 16-byte chunk c at c ^ ((r >> 1) & 7), so
// 16 consecutive rows of a fragment read hit 16 bank groups; a B row of 128 B
// (16-bit, BN = 64) keeps it at c ^ 4 ((k >> 1) & 1), a B row of 64 B of bytes at
// c ^ 2 ((k >> 2) & 1), so the rows a half-wave's transposing read covers fill
// 256 B of banks; narrower B rows fill them as they are.
#pragma once

#include <type_traits>

#include "gemm_common.h"

namespace xtk {
namespace {

constexpr int kStageK = 128;  // K bytes per stage: a whole cache line of every A row

template <int ELEM, int BM, int BN>
struct SmallTile {
  typedef typename Acc<ELEM>::type acc_t;
  typedef typename std::conditional<ELEM == kI8, int, float>::type num_t;
  typedef num_t num4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) unsigned char lds_t;
  static constexpr int ES = ELEM == kI8 ? 1 : 2;
  static constexpr int STAGE = (BM + BN) * kStageK;
  static constexpr int NS = BM + BN == 128 ? 2 : BM + BN == 96 ? 3 : 4;  // stages of a wave's ring
  static constexpr int RING = NS * STAGE;
  static constexpr int LDC = BN + 8;  // floats per row of a partial tile: half-waves, four rows apart, in distinct banks
  static constexpr int LDS = 4 * RING;
  static_assert(4 * BM * LDC * 4 <= LDS, "the partial tiles reuse the rings");
  static constexpr int MI = BM / 32, NJ = BN / 32;
  static constexpr int AB = BM * kStageK;   // A bytes per stage
  static constexpr int BR = BN * ES;        // bytes of a B row
  static constexpr int KR = kStageK / ES;   // B rows per stage
  static constexpr int KSR = 32 / ES;       // B rows per MFMA step
  static constexpr int STEPS = kStageK / 32;
  static constexpr int PA = BM / 8, PB = BN / 8, PER = PA + PB;  // instructions per stage
  static constexpr int CPR = BR / 16, RPI = 1024 / BR;
  static_assert((NS - 1) * PER < 64 && NS <= 4, "vmcnt is six bits");

  static __device__ __forceinline__ int bsw(int k) {
    return BR == 128 ? 4 * ((k >> 1) & 1) : ES == 1 && BR == 64 ? 2 * ((k >> 2) & 1) : 0;
  }
  // what a lane fetches: A row 8 i + lane / 8, chunk a_chunk(lane, i); B row RPI i + lane / CPR, chunk b_chunk(lane)
  static __device__ __forceinline__ int a_chunk(int lane, int i) { return (lane & 7) ^ ((4 * i + (lane >> 4)) & 7); }
  static __device__ __forceinline__ int b_chunk(int lane) { return (lane % CPR) ^ bsw(lane / CPR); }

  int lane, lrow, hi;
  int aoff[MI], asw[MI], boff[NJ][2];
  acc_t acc[MI][NJ];
  uint4v af[STEPS][MI], bf[STEPS][NJ];  // the fragments of a stage

  __device__ __forceinline__ void begin(int l) {
    lane = l;
    lrow = l & 31;
    hi = l >> 5;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = i * 32 + lrow;
      aoff[i] = r * kStageK;
      asw[i] = (r >> 1) & 7;
    }
    const int g = lane >> 4, li = lane & 15;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = ES == 2 ? 8 * (g >> 1) + 4 * h + (li >> 2) : 16 * (g >> 1) + 8 * h + (li >> 1);
        const int cb = ES == 2 ? (j * 32 + 16 * (g & 1) + 4 * (li & 3)) * 2 : j * 32 + 16 * (g & 1) + 8 * (li & 1);
        boff[j][h] = AB + k * BR + (((cb >> 4) ^ bsw(k)) << 4) + (cb & 15);
      }
  }

  __device__ __forceinline__ void read_stage(const unsigned char* S) {
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
        af[ks][i] = *reinterpret_cast<const uint4v*>(S + aoff[i] + (((ks * 2 + hi) ^ asw[i]) << 4));
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        lds_t* const f = (lds_t*)(S + ks * KSR * BR);
        uint2v lo, up;
        if constexpr (ES == 2) {
          lo = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                              reinterpret_cast<short4v __attribute__((address_space(3)))*>(f + boff[j][0])));
          up = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                              reinterpret_cast<short4v __attribute__((address_space(3)))*>(f + boff[j][1])));
        } else {
          lo = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                              reinterpret_cast<int2v __attribute__((address_space(3)))*>(f + boff[j][0])));
          up = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                              reinterpret_cast<int2v __attribute__((address_space(3)))*>(f + boff[j][1])));
        }
        bf[ks][j] = uint4v{lo[0], lo[1], up[0], up[1]};
      }
    }
  }

  __device__ __forceinline__ void multiply() {
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma<ELEM>(af[ks][i], bf[ks][j], acc[i][j]);
  }

  // At most `ahead` (<= NS - 1) later stages of this wave are outstanding.
  static __device__ __forceinline__ void landed(int ahead) {
    switch (ahead) {
      case 0: XTK_WAIT_VM(0); break;
      case 1: XTK_WAIT_VM(PER); break;
      case 2: XTK_WAIT_VM(2 * PER); break;
      default: XTK_WAIT_VM(3 * PER); break;
    }
    asm volatile("" ::: "memory");
  }

  // This wave's `mine` (a scalar) stages through its ring by DMA: issue(q, slot
  // address, i) is instruction i (of PER) of its stage q.
  template <typename F>
  __device__ __forceinline__ void run(unsigned char* ring, int mine, F issue) {
    const unsigned at = lds_addr(ring);
#pragma unroll
    for (int q = 0; q < NS; ++q)
      if (q < mine)
#pragma unroll
        for (int i = 0; i < PER; ++i) issue(q, at + q * STAGE, i);
    int slot = 0;
    for (int q = 0; q < mine; ++q) {
      landed(min(mine - 1 - q, NS - 1));
      read_stage(ring + slot * STAGE);
      // every fragment is in registers before the DMA that reuses the slot
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (q + NS < mine)
#pragma unroll
        for (int i = 0; i < PER; ++i) issue(q + NS, at + slot * STAGE, i);
      multiply();
      slot = slot + 1 == NS ? 0 : slot + 1;
    }
  }

  // The waves' partial tiles summed through LDS, in a fixed order; out(m, n0, x)
  // takes columns n0 .. n0 + 3 of row m.  Accumulator register v of tile (i, j)
  // holds row 8 (v / 4) + 4 hi + v % 4, column lane % 32.
  template <typename F>
  __device__ __forceinline__ void finish(unsigned char* lds, int wave, F out) const {
    __syncthreads();
    num_t* const part = reinterpret_cast<num_t*>(lds);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          part[(wave * BM + i * 32 + (v >> 2) * 8 + hi * 4 + (v & 3)) * LDC + j * 32 + lrow] = acc[i][j][v];
    __syncthreads();
    constexpr int TPR = BN / 4;  // threads per output row
    const int tid = wave * 64 + lane, n0 = 4 * (tid % TPR);
#pragma unroll
    for (int m = tid / TPR; m < BM; m += 256 / TPR) {
      num4 x = *reinterpret_cast<const num4*>(part + m * LDC + n0);
#pragma unroll
      for (int w = 1; w < 4; ++w) x += *reinterpret_cast<const num4*>(part + (w * BM + m) * LDC + n0);
      out(m, n0, x);
    }
  }
};

}  // namespace
}  // namespace xtk
