// GEMM tiles of 64 x 64 down to 32 x 32, with ragged edges.
//
// For products whose 128-wide tiles leave CUs idle (decoding a few dozen
// rows, 1024^3), whose M or N no 128-wide tile divides, or whose sizes or
// alignment the DMA kernel of gemm.hip does not take at all.
//
// What bounds such a launch is how fast one CU gets its operands, behind the
// start and end of a launch, against little matrix work: beyond about 6 us the
// time grows by 72 KB of operands a us and CU at 64 x 64 tiles of f16, by 36 at
// 32 x 32 of i8, whose 32-byte rows of B make four requests of a line (1024^3:
// 0.52 M requests to L2, matrix pipes busy 0.11 of its cycles;
// 64 x 4096 x 4096 i8: 1.31 M requests, 0.80 of them B's, busy 0.04;
// profiles/small_gemm_rates.txt, matmul_*_gemm_small.txt).  So the kernel keeps as many bytes in flight as LDS holds, and
// nothing waits for anything else: the workgroup's four waves split K between
// them (stage s of 64 K bytes belongs to wave s % 4), each wave fills its own
// LDS ring, waits for its own loads and multiplies the whole BM x BN tile, so
// the K loop has no barrier and no other wave's latency in it.  Splitting K
// also halves the LDS reads a product needs against splitting the tile.  The
// four partial tiles meet once, in LDS, and leave as 16-byte stores.  The
// order of the sums is fixed: results are the same run to run.
//
// Measured (graph replay, us a launch, before -> now; "before" are 64 x 64 tiles
// of register-staged slices two deep, 128 x 128 tiles with an atomic K split
// behind a zero fill, or, for sizes 64 does not divide, the staged kernel's
// whole panels in LDS): 64 x 4096 x 4096 i8 28.4 -> 11.6, 1024^3 f16 15.7 ->
// 9.5, 384 x 896 x 3712 i8 20.3 -> 10.3, 256 x 320 x 640 i8 7.7 -> 3.8, 1000^3
// f16 in 40 x 40 Blocks 235 -> 10.2, 114 x 630 x 371 f16 88 -> 4.8.  Stages of
// 64 K bytes (half lines of A), 64 x 64 tiles: 1024^3 9.1, 1024 x 1024 x 4096
// 23+, 1984 x 1408 x 8064 95 against 84; DMA issued between the MFMAs instead
// of in one burst before them: 10.8 on 1024^3.
//
// Layouts and the loop are in small_tile.h.
//
// DMA (LOAD = kDma): buffer_load ... lds, NS - 1 stages ahead.  Rows past M
// and column chunks past N are clamped to ones that exist (their results are
// never stored); K positions past the end get an offset past the descriptor's
// records and read as zeros on both sides.  Needs 16-byte aligned rows and K
// a whole number of 16-byte chunks.
// Registers (LOAD = kRegs): any element alignment, K and N of at least 16
// bytes.  16-byte loads at element alignment (gfx950 takes unaligned global
// accesses), kAhead stages held in registers, written to the same LDS layout.
// A stage that holds K's end or B's last bytes takes each chunk from a load
// that ends where its elements end, shifted into place, zeros past K.
#include "launch.h"
#include "small_tile.h"

namespace xtk {
namespace {

enum { kDma = 0, kRegs = 1 };

// Sixteen bytes at element alignment.
template <int ES>
__device__ __forceinline__ uint4v load16(const unsigned char* q) {
  if constexpr (ES == 2) {
    typedef short v8 __attribute__((ext_vector_type(8), aligned(2)));
    return __builtin_bit_cast(uint4v, (short8)(*reinterpret_cast<const v8*>(q)));
  } else {
    typedef unsigned u4 __attribute__((ext_vector_type(4), aligned(1)));
    return (uint4v)(*reinterpret_cast<const u4*>(q));
  }
}

// The first n (<= 0: none) of the 16 / ES elements at q, zeros after them, from
// one 16-byte load that ends where those elements end (so q - 16 + n ES must
// be readable); `safe` is read, and dropped, when there are none.
template <int ES>
__device__ __forceinline__ uint4v load_part(const unsigned char* q, int n, const unsigned char* safe) {
  const int back = n >= 16 / ES ? 0 : 16 - n * ES;  // bytes
  uint4v v = load16<ES>(n > 0 ? q - back : safe);
  if (back & 4) v = uint4v{v[1], v[2], v[3], 0u};
  if (back & 8) v = uint4v{v[2], v[3], 0u, 0u};
  const unsigned r = (back & 3) * 8;
  v = uint4v{__builtin_amdgcn_alignbit(v[1], v[0], r), __builtin_amdgcn_alignbit(v[2], v[1], r),
             __builtin_amdgcn_alignbit(v[3], v[2], r), v[3] >> r};
  return n > 0 ? v : uint4v{0u, 0u, 0u, 0u};
}

template <int ELEM, bool OUT_I8, int BM, int BN, int LOAD>
__global__ __launch_bounds__(256, 1) void gemm_small_kernel(GemmArgs p) {
  typedef SmallTile<ELEM, BM, BN> T;
  constexpr int ES = T::ES, AB = T::AB, BR = T::BR, KR = T::KR, PA = T::PA, PB = T::PB, PER = T::PER, RPI = T::RPI;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[T::LDS];

  int tx, ty;
  const TilePtrs t = gemm_tile_of<ELEM, BM, BN>(p, tx, ty);
  const int mleft = p.edge ? min(BM, p.M - ty * BM) : BM;
  const int nleft = p.edge ? min(BN, p.N - tx * BN) : BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* const ring = lds + wave * T::RING;

  const int arow = lane >> 3, brow = lane / T::CPR;
  auto ach = [&](int i) { return T::a_chunk(lane, i); };
  int bch = T::b_chunk(lane);
  if (bch * (16 / ES) >= nleft) bch = 0;
  const int ns = (p.K * ES + kStageK - 1) / kStageK;  // stages; this wave's: wave, wave + 4, ...
  const int mine = (ns - wave + 3) >> 2;

  T t4;
  t4.begin(lane);

  if constexpr (LOAD == kDma) {
    // K past the end: offsets at 2^31, past the records of a descriptor that
    // ends there (a launch without a K tail may span up to 4 GiB)
    const bool tail = (p.K * ES) % kStageK != 0;
    const i32x4 ra = raw_rsrc(t.A, tail ? 0x80000000u : 0xFFFFFFFFu), rb = raw_rsrc(t.B, tail ? 0x80000000u : 0xFFFFFFFFu);
    const unsigned lda = (unsigned)(p.lda * ES), ldb = (unsigned)(p.ldb * ES);
    unsigned va[PA];
#pragma unroll
    for (int i = 0; i < PA; ++i) va[i] = (unsigned)min(8 * i + arow, mleft - 1) * lda + (unsigned)ach(i) * 16;
    const unsigned vb = (unsigned)brow * ldb + (unsigned)bch * 16;
    t4.run(ring, mine, [&](int q, unsigned at, int i) {
      const int s = __builtin_amdgcn_readfirstlane(4 * q + wave);
      const bool last = tail && s + 1 == ns;
      if (i < PA) {
        const bool in = !last || ach(i) * 16 < p.K * ES - s * kStageK;
        dma16(ra, at + i * 1024, in ? va[i] : 0x80000000u, __builtin_amdgcn_readfirstlane((unsigned)s * kStageK));
      } else {
        const int k = s * KR + RPI * (i - PA);
        const bool in = !last || k + brow < p.K;
        dma16(rb, at + AB + (i - PA) * 1024, in ? vb : 0x80000000u, __builtin_amdgcn_readfirstlane((unsigned)k * ldb));
      }
    });
  } else {
    constexpr int kAhead = 2;
    uint4v reg[kAhead][PER];
    const long long lda = p.lda * ES, ldb = p.ldb * ES;
    const long long b_end = (long long)(p.K - 1) * ldb + (long long)nleft * ES;  // past the last B byte this tile may read
    const unsigned char* pa[PA];
#pragma unroll
    for (int i = 0; i < PA; ++i) pa[i] = t.A + (long long)min(8 * i + arow, mleft - 1) * lda + ach(i) * 16;
    const unsigned char* const pb = t.B + (long long)brow * ldb + bch * 16;
    auto fetch = [&](int q, uint4v(&r)[PER]) {
      const int s = 4 * q + wave;
      const unsigned char* const bs = pb + (long long)(s * KR) * ldb;
      // every chunk of the stage lies inside its row / inside B
      if ((s + 1) * kStageK <= p.K * ES && (long long)((s + 1) * KR - 1) * ldb + BR <= b_end) {
#pragma unroll
        for (int i = 0; i < PA; ++i) r[i] = load16<ES>(pa[i] + s * kStageK);
#pragma unroll
        for (int i = 0; i < PB; ++i) r[PA + i] = load16<ES>(bs + (long long)(RPI * i) * ldb);
      } else {
        const int kleft = p.K - s * KR;  // K values from this stage's start
#pragma unroll
        for (int i = 0; i < PA; ++i) r[i] = load_part<ES>(pa[i] + s * kStageK, kleft - ach(i) * (16 / ES), t.A);
#pragma unroll
        for (int i = 0; i < PB; ++i)
          r[PA + i] = load_part<ES>(bs + (long long)(RPI * i) * ldb,
                                    RPI * i + brow < kleft ? nleft - bch * (16 / ES) : 0, t.B - (nleft < 16 / ES ? 16 : 0));
      }
    };
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
      if (q < mine) fetch(q, reg[q]);
    for (int q0 = 0; q0 < mine; q0 += kAhead)
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int q = q0 + u;
        if (q >= mine) break;
        unsigned char* const S = ring + (q & 1) * T::STAGE;
#pragma unroll
        for (int i = 0; i < PER; ++i) *reinterpret_cast<uint4v*>(S + i * 1024 + lane * 16) = reg[u][i];
        if (q + kAhead < mine) fetch(q + kAhead, reg[u]);
        t4.read_stage(S);
        t4.multiply();
      }
  }

  const bool hs = p.has_scale, hb = p.has_bias;
  float sv[4] = {1.f, 1.f, 1.f, 1.f}, bv[4] = {0.f, 0.f, 0.f, 0.f};
  const int col = 4 * (tid % (BN / 4));  // this thread's output columns
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (col + e < nleft) {
      if (hs) sv[e] = t.S[col + e];
      if (hb) bv[e] = t.Bias[col + e];
    }
  t4.finish(lds, wave, [&](int m, int n0, typename T::num4 x) {
    if (m >= mleft || n0 >= nleft) return;
    const long long off = t.c_off + (long long)m * p.ldc + n0;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = scale_bias((float)x[e], sv[e], bv[e], hs, hb);
    const bool whole = p.cvec && n0 + 4 <= nleft;
    if constexpr (OUT_I8) {
      int q[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) q[e] = ftoi_i8_fast(y[e]);
      signed char* const c = static_cast<signed char*>(p.c) + off;
      if (whole) {
        *reinterpret_cast<unsigned*>(c) = pack_i8x4(q);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n0 + e < nleft) c[e] = (signed char)q[e];
      }
    } else {
      float* const c = static_cast<float*>(p.c) + off;
      if (whole) {
        *reinterpret_cast<float4v*>(c) = float4v{y[0], y[1], y[2], y[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n0 + e < nleft) c[e] = y[e];
      }
    }
  });
}

template <int ELEM, bool OUT_I8, int LOAD>
void launch_tile(int bm, int bn, const GemmArgs& a, hipStream_t s) {
  const dim3 grid(a.nwg), block(256);
  if (bm == 64 && bn == 64)
    hipLaunchKernelGGL((gemm_small_kernel<ELEM, OUT_I8, 64, 64, LOAD>), grid, block, 0, s, a);
  else if (bn == 64)
    hipLaunchKernelGGL((gemm_small_kernel<ELEM, OUT_I8, 32, 64, LOAD>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((gemm_small_kernel<ELEM, OUT_I8, 32, 32, LOAD>), grid, block, 0, s, a);
}

template <int ELEM, bool OUT_I8>
void launch_load(int bm, int bn, bool dma, const GemmArgs& a, hipStream_t s) {
  dma ? launch_tile<ELEM, OUT_I8, kDma>(bm, bn, a, s) : launch_tile<ELEM, OUT_I8, kRegs>(bm, bn, a, s);
}

}  // namespace

hipError_t run_gemm_small(xt::Elem elem, bool out_i8, int bm, int bn, bool dma, const GemmArgs& a, hipStream_t s) {
  switch (elem) {
    case xt::Elem::I8: out_i8 ? launch_load<kI8, true>(bm, bn, dma, a, s) : launch_load<kI8, false>(bm, bn, dma, a, s); break;
    case xt::Elem::BF16:
      out_i8 ? launch_load<kBF16, true>(bm, bn, dma, a, s) : launch_load<kBF16, false>(bm, bn, dma, a, s);
      break;
    default:
      out_i8 ? launch_load<kF16, true>(bm, bn, dma, a, s) : launch_load<kF16, false>(bm, bn, dma, a, s);
      break;
  }
  return hipGetLastError();
}

}  // namespace xtk
