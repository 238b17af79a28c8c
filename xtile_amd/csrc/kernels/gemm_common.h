// What the GEMM kernels share: launch arguments, the MFMA of each element
// type, the workgroup -> tile mapping and the epilogue's arithmetic.
#pragma once

#include <algorithm>

#include "../plan.h"
#include "common.h"

namespace xtk {

struct GemmArgs {
  const unsigned char* a;
  const unsigned char* b;
  void* c;
  const float* scale;
  const float* bias;
  TileOff ta, tb, tc, ts, tbias;  // element offsets
  long long lda, ldb, ldc;        // row pitches in elements
  int nk;                         // K slices
  int vgx, vgy;                   // virtual grid (fused axes divided by their factor)
  int mul[3];                     // block id = virtual id * mul (fused axes)
  int sub_m, sub_n;               // workgroup tiles per (fused) Block along M and N
  int nwg;
  int group;
  int has_scale, has_bias;
  // K split (DMA kernel, f32 results without an epilogue): nwg = tiles *
  // ksplit workgroups, K range r covering stages [r S / ksplit, (r + 1) S /
  // ksplit) of the S = 2 nk stages of 64 K bytes (ranges differ by at most
  // one stage; kstages = the shortest); ksplit = 1, tiles = nwg otherwise
  int tiles, ksplit, kstages;
  // gemm_small_kernel: K values of the product; `edge`: the tiles cover one
  // M x N region and the last ones may reach past it; `cvec`: every output
  // row of a tile starts on a 4-element boundary
  int M, N, K, edge, cvec;
  // the tile mapping's divisors (divide()): an integer division by a kernel
  // argument costs ~30 dependent instructions, and a tile takes six of them
  Div31 d_tiles, d_subs, d_subn, d_plane, d_group, d_gsize, d_glast;
  void divide() {
    d_tiles = div31(tiles);
    d_subs = div31(sub_m * sub_n);
    d_subn = div31(sub_n);
    d_plane = div31(vgx * vgy);
    d_group = div31(group * vgy);
    d_gsize = div31(std::min(group, vgx));
    d_glast = div31(vgx % group ? vgx % group : std::min(group, vgx));
  }
};

// gemm_small.hip: bm, bn in {32, 64}; `dma` says the operands may take LDS DMA.
hipError_t run_gemm_small(xt::Elem elem, bool out_i8, int bm, int bn, bool dma, const GemmArgs& a, hipStream_t s);

namespace {

enum { kF16 = 0, kBF16 = 1, kI8 = 2 };

typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int16v __attribute__((ext_vector_type(16)));

template <int ELEM>
struct Acc {
  typedef float16v type;
};
template <>
struct Acc<kI8> {
  typedef int16v type;
};

template <int ELEM>
__device__ __forceinline__ typename Acc<ELEM>::type mfma(uint4v a, uint4v b, typename Acc<ELEM>::type c) {
  if constexpr (ELEM == kI8)
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(int4v, a), __builtin_bit_cast(int4v, b), c,
                                                 0, 0, 0);
  else if constexpr (ELEM == kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c,
                                                  0, 0, 0);
}

// Workgroup -> tile origins.  Contiguous runs per XCD, then GROUP-wide column
// groups over the virtual grid.
struct TilePtrs {
  const unsigned char* A;
  const unsigned char* B;
  long long c_off;  // element offset of the C tile
  const float* S;
  const float* Bias;
};

// The workgroup's linear id with contiguous runs per XCD: the K range is
// gemm_lin / tiles, the tile gemm_lin % tiles.
__device__ __forceinline__ int gemm_lin(const GemmArgs& p) {
  return xcd_contiguous(blockIdx.x, p.nwg);
}

// tx, ty: the tile's virtual block id along the grid's first two axes.
template <int ELEM, int BM, int BN, bool KS = false>
__device__ __forceinline__ TilePtrs gemm_tile_of(const GemmArgs& p, int& tx, int& ty) {
  constexpr int ES = ELEM == kI8 ? 1 : 2;
  int L = gemm_lin(p);
  if constexpr (KS) L -= (int)p.d_tiles(L) * p.tiles;
  int blk = p.d_subs(L);
  const int s = L - blk * p.sub_m * p.sub_n;
  const int sm = p.d_subn(s);
  const int sn = s - sm * p.sub_n;
  const int per_plane = p.vgx * p.vgy;
  const int vz = p.d_plane(blk);
  blk -= vz * per_plane;
  const int gid = p.d_group(blk);
  const int first = gid * p.group;
  const int r = blk - gid * p.group * p.vgy;
  const bool last = first + p.group >= p.vgx;
  const int gsize = last ? p.vgx - first : p.group;
  ty = last ? p.d_glast(r) : p.d_gsize(r);
  tx = first + r - ty * gsize;
  const int x = tx * p.mul[0];
  const int y = ty * p.mul[1];
  const int z = vz * p.mul[2];
  TilePtrs t;
  t.A = p.a + (p.ta.at(x, y, z) + (long long)sm * BM * p.lda) * ES;
  t.B = p.b + p.tb.at(x, y, z) * ES + (long long)sn * BN * ES;
  t.c_off = p.tc.at(x, y, z) + (long long)sm * BM * p.ldc + (long long)sn * BN;
  t.S = p.scale + p.ts.at(x, y, z) + sn * BN;
  t.Bias = p.bias + p.tbias.at(x, y, z) + sn * BN;
  return t;
}

// x * s + b as two separately rounded f32 operations.
__device__ __forceinline__ float scale_bias(float x, float s, float b, bool hs, bool hb) {
#pragma clang fp contract(off)
  float t = hs ? x * s : x;
  return hb ? t + b : t;
}

// The same conversion in three instructions: v_rndne_f32 (half to even),
// v_cvt_i32_f32 (saturates out-of-range values and infinities, converts NaN
// to 0; issued as assembly because a C++ cast of such values is undefined),
// v_med3_i32 (clamp to [-128, 127]).
__device__ __forceinline__ int ftoi_i8_fast(float v) {
  int i;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(__builtin_rintf(v)));
  return min(max(i, -128), 127);
}

// Low bytes of four ints packed into one word (byte e from q[e]).
__device__ __forceinline__ unsigned pack_i8x4(const int (&q)[4]) {
  const unsigned lo = __builtin_amdgcn_perm((unsigned)q[1], (unsigned)q[0], 0x0c0c0400u);  // q0 q1 0 0
  const unsigned hi = __builtin_amdgcn_perm((unsigned)q[3], (unsigned)q[2], 0x04000c0cu);  // 0 0 q2 q3
  return lo | hi;
}

}  // namespace
}  // namespace xtk
