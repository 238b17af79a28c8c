// Tile matmul C = epilogue(A @ B) on the gfx950 matrix cores.
//
// Semantics: xt.matmul over one Block's tiles, the whole K extent of the tile
// (kernels/matmul.py:11-16,35; lib/xt/XTOps.cpp:218-253): f16 x f16 and
// bf16 x bf16 accumulate in f32 (the narrow-float extension); i8 x i8
// accumulates exactly in i32 and the result is f32.  The optional epilogue is
// the one of kernels/matmul.py:15-17: t * scale + bias with (1, TN) row tiles
// broadcast over the rows (two separately rounded f32 operations, never fused),
// then astype(int8) = xt.ftoi (round half to even, saturate to [-128, 127],
// NaN -> 0; the reference fixes no rule, this is the oracle's).
//
// Workgroup tiles are decoupled from xt Block tiles.  A Block's TM x TN output
// tile is split into (TM/BM) x (TN/BN) workgroup tiles when it is larger, and
// neighbouring Blocks are fused into one workgroup tile when it is smaller and
// the planner's affine addresses show them to be contiguous (the next Block
// along one grid axis continues the same A rows / B columns / C tile / scale
// and bias columns).  Blocks are independent (README.md:85-89), so both are
// pure scheduling choices.
//
// 256 x 256, 256 x 128, 128 x 256 and 128 x 128 workgroup tiles run on
// gemm_dma_kernel (operands landed in LDS by DMA; described where it is
// defined), whatever the element type and result: 256 x 256 when the Blocks map
// onto it and its tiles fill the CUs (or are few enough to split K), else the
// first smaller tile whose tiles fill them.  Where none does, the rest compete
// by estimated time (tile_us): the fullest of those tiles, 128 x 128 and 256 x
// 256 tiles over the whole M x N region with the last ones reaching past it,
// and gemm_small.hip's 64 x 64, 32 x 64 and 32 x 32 tiles, which also take the
// products of any size and alignment (launch_gemm_ragged).
//   * For an f32 result a half-wave stores one whole 128-byte line per
//     accumulator register.
//   * Workgroups are dispatched round-robin over the 8 XCDs; the linear id is
//     remapped so that each XCD receives a contiguous run of tiles, and tiles
//     are ordered in groups of GROUP tile columns so that concurrently resident
//     workgroups share A and B panels in their XCD's L2.
#include <algorithm>
#include <type_traits>

#include "gemm_common.h"
#include "launch.h"

namespace xtk {
namespace {

constexpr int SLICE = 128;  // bytes of K per LDS row and K slice
// K stages of gemm_dma_kernel in LDS: a stage's DMA has two stages of compute
// to land; three and five stages measured no faster on C3 (bench.py: four
// and five both 129.7 us before the DMA was spread over the MFMA slots)
constexpr int kDmaStages = 4;
constexpr int kTileGroup = 8;  // tile columns per group of the workgroup order

// Waves of gemm_dma_kernel: 4 (one per SIMD, 128 x 128 each) or 8 (two per
// SIMD, 128 x 64 each: half an LDS read more per MFMA, but a second wave to
// issue MFMAs while one waits).  Measured in one call (bench.py, 2000
// launches): C3 (f16) 122.6 us with 4 and 124.0 with 8, C5 (bf16) 319.9 and
// 317.2, C6 (i8) 72.6 and 71.2.
template <int ELEM>
constexpr int dma_waves() { return ELEM == kF16 ? 4 : 8; }

// ---------------------------------------------------------------------------
// 256 x 256 GEMM whose operands reach LDS by DMA (buffer_load ... lds): no
// VGPR staging, no register transposes, no LDS stores.  f16 / bf16 or i8
// operands; an f32 result, or (OUT_I8) the i8 result of the epilogue.
//   * NW = 4 waves of 128 x 128 (4 x 4 tiles of v_mfma_f32_32x32x16_{f16,bf16}
//     or v_mfma_i32_32x32x32_i8), one per SIMD, or NW = 8 waves of 128 x 64
//     (4 x 2 tiles), two per SIMD.  A stage is 64 bytes of K
//     (32 f16 / bf16 or 64 i8 values): A [256 rows][64 B] and B [KR k][BR B]
//     (32 x 512 B, or 64 x 256 B for i8), 16 KB each, in one of NS LDS
//     buffers (each its own LDS variable, so that reading one while DMA into
//     others is in flight needs no wait).
//   * A DMA instruction fills 1 KB of LDS, lane L at byte 16 L.  The layouts
//     are swizzled by choosing which global chunk each lane fetches: A row r
//     keeps its 16-byte chunk c at position c ^ ((r >> 2) & 3), so a
//     16-lane phase of fragment reads (16 consecutive rows) hits 16 distinct
//     16-byte bank groups.  16-bit B row k keeps chunk c at c ^ 4 (k & 3), so
//     the four rows a half-wave reads with ds_read_b64_tr_b16 fall in four
//     different 64-byte bank groups; i8 B row k keeps it at c ^ 2 (k & 7), so
//     the eight rows a half-wave reads with ds_read_b64_tr_b8 fall in eight
//     different 32-byte bank groups.
//   * B fragments come straight from the [k][n] layout through the
//     transposing reads: lane l receives column l % 32 and the 16 bytes of K
//     16 (l / 32) .. + 15 (bytes), 8 from each of two reads, the operand
//     layout of the MFMA.  A 16-lane group of ds_read_b64_tr_b16 reads a
//     4 (k) x 16 (n) block, lane i at row i / 4 and columns 4 (i % 4) .. + 3;
//     of ds_read_b64_tr_b8 an 8 x 16 block, lane i at row i / 2 and columns
//     8 (i % 2) .. + 7.
//   * For an i8 result the MFMAs compute D = B^T-fragment x A-fragment, so
//     each lane holds runs of four consecutive output columns of one row and
//     writes them as one 4-byte store.
//   * Barrier B_s opens stage s.  Before it each wave waits for its own DMA
//     of stages s and s + 1 and for its LDS reads; so after it every wave's
//     DMA of both stages has landed and every wave is done with stage s - 1.
//     Then the DMA of stage s + NS - 1 goes into stage s - 1's buffer, the
//     stage's two K steps run (32 MFMAs a wave), and the first fragments of
//     stage s + 1 are read before B_{s+1}, so no barrier is followed by an
//     LDS round trip.  A stage's DMA has NS - 2 stages of compute to land.
//     The barrier is a bare s_barrier: __syncthreads' release fence would
//     also wait for the DMA that should stay in flight.
//   * EDGE: the tiles cover one M x N region whose size no tile divides.  Rows
//     past M and column chunks past N are clamped to ones that exist, and
//     their results are not stored.  (Odd multiples of 64, which had run on 64
//     x 64 tiles: bf16 4864 x 2112 x 1280 73 -> 37 us, 1984 x 1408 x 8064 96 ->
//     69, f16 3776 x 6656 x 256 97 -> 37, i8 4224 x 2752 x 2176 90 -> 37.)
template <int ELEM, int NS, bool OUT_I8, bool EPI, int NW, bool KS = false, int BMT = 256, int BNT = 256, bool EDGE = false>
__global__ __launch_bounds__(64 * NW, BMT * BNT <= 128 * 128 ? 2 : 1) void gemm_dma_kernel(GemmArgs p) {
  static_assert(!KS || (!EPI && !OUT_I8 && !EDGE), "K split only without an epilogue");
  static_assert(NS >= 3 && NS <= 5, "stages");
  static_assert(NW == 4 || NW == 8, "waves");
  static_assert((BMT == 256 || BMT == 128) && (BNT == 256 || BNT == 128) && (NW == 4 || BMT * BNT == 65536),
                "tiles");
  // NW = 4: 2 x 2 waves of (BM / 2) x (BN / 2); NW = 8 (256 x 256 only): 2 x 4
  // waves of 128 x 64 (two waves per SIMD)
  constexpr int BM = BMT, BN = BNT, WM = BM / 2, WN = 2 * BN / NW, MI = WM / 32, NI = WN / 32;
  constexpr int ES = ELEM == kI8 ? 1 : 2;  // bytes per element
  constexpr int KB = 64;            // K bytes per A row and stage
  constexpr int AB = BM * KB;       // A bytes per stage
  constexpr int BR = BN * ES;       // B bytes per k row
  constexpr int KR = KB / ES;       // B k rows per stage
  constexpr int RPI = 1024 / BR;    // B k rows per DMA instruction
  constexpr int KSR = 32 / ES;      // B k rows per MFMA K step
  constexpr int STAGE = AB + KR * BR;
  constexpr int PA = BM / 16 / NW;  // A DMA instructions (16 rows each) per wave and stage
  constexpr int PB = KR * BR / 1024 / NW;  // B DMA instructions per wave and stage
  constexpr int PER = PA + PB;      // DMA instructions per wave and stage
  typedef typename Acc<ELEM>::type acc_t;
  typedef __attribute__((address_space(3))) unsigned char lds_t;
  __shared__ __attribute__((aligned(1024))) unsigned char S0[STAGE];
  __shared__ __attribute__((aligned(1024))) unsigned char S1[STAGE];
  __shared__ __attribute__((aligned(1024))) unsigned char S2[STAGE];
  __shared__ __attribute__((aligned(1024))) unsigned char S3[NS > 3 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) unsigned char S4[NS > 4 ? STAGE : 16];
  unsigned char* const buf[5] = {S0, S1, S2, S3, S4};

  int tx, ty;
  const TilePtrs t = gemm_tile_of<ELEM, BM, BN, KS>(p, tx, ty);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / (NW / 2), wn = wave % (NW / 2);
  static_assert(WM * 2 == BM && WN * (NW / 2) == BN, "wave layout");
  const int mleft = EDGE ? min(BM, p.M - ty * BM) : BM, nleft = EDGE ? min(BN, p.N - tx * BN) : BN;
  const i32x4 ra = raw_rsrc(t.A), rb = raw_rsrc(t.B);
  const unsigned lda = (unsigned)(p.lda * ES), ldb = (unsigned)(p.ldb * ES);
  // this workgroup's stages of 64 K bytes: [kbase, kbase + nk)
  const int krange = KS ? (int)p.d_tiles(gemm_lin(p)) : 0;
  const int kbase = KS ? (int)((long long)krange * (p.nk * 2) / p.ksplit) : 0;
  const int nk = KS ? (int)((long long)(krange + 1) * (p.nk * 2) / p.ksplit) - kbase : p.nk * 2;

  // B row k keeps its 16-byte chunk c at c ^ bsw(k) (rows of 128-byte i8:
  // (k / 2) % 4, so the eight rows a half-wave's tr_b8 read covers still
  // fall in distinct 16-byte bank groups)
  auto bsw = [](int k) { return ES == 2 ? 4 * (k & 3) : BR == 128 ? (k >> 1) & 3 : 2 * (k & 7); };
  // DMA lane offsets.  A instruction i (rows 16i .. 16i+15): lane L holds
  // row 16i + L/4 at position L%4, i.e. chunk (L%4) ^ ((L/16) & 3).  B
  // instruction i (k rows RPI i .. + RPI - 1, CPR chunks each): lane
  // (h, pc) = (L / CPR, L % CPR) holds chunk pc ^ bsw(RPI i + h), which
  // depends on i only through i & 1.
  constexpr int CPR = BR / 16;
  const unsigned ach = (unsigned)(((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  const unsigned va = (unsigned)(lane >> 2) * lda + ach;
  unsigned va_edge[EDGE ? PA : 1];  // with the rows of this wave's instructions, clamped
  if constexpr (EDGE)
#pragma unroll
    for (int q = 0; q < PA; ++q) va_edge[q] = (unsigned)min(16 * (wave * PA + q) + (lane >> 2), mleft - 1) * lda + ach;
  unsigned vb[2];
  {
    const int h = lane / CPR, pc = lane % CPR;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = pc ^ bsw(RPI * q + h);
      vb[q] = (unsigned)h * ldb + (unsigned)((EDGE && c * (16 / ES) >= nleft ? 0 : c) << 4);
    }
  }
  // this wave's share of stage kt: A instructions PA w .. + PA - 1 (q < PA),
  // B instructions PB w .. + PB - 1 (q >= PA)
  auto dma_one = [&](int kt, unsigned char* S, int q) {
    const int kg = kt + kbase;
    if (q < PA) {
      const int i = wave * PA + q;
      if constexpr (EDGE) dma16(ra, lds_addr(S + i * 1024), va_edge[q], (unsigned)kg * KB);
      else dma16(ra, lds_addr(S + i * 1024), va, (unsigned)(16 * i) * lda + (unsigned)kg * KB);
    } else {
      const int i = wave * PB + (q - PA);
      dma16(rb, lds_addr(S + AB + i * 1024), vb[i & 1], (unsigned)(kg * KR + RPI * i) * ldb);
    }
  };
  auto dma = [&](int kt, unsigned char* S) {
#pragma unroll
    for (int q = 0; q < PER; ++q) dma_one(kt, S, q);
  };

  // fragment offsets: A row r at r * 64, chunk c at c ^ ((r >> 2) & 3); B per
  // (tile j, read h) an offset in the stage's first K step, plus KSR rows for
  // the second
  const int lrow = lane & 31, hi = lane >> 5;
  int arow[MI], asw[MI], boff[NI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = wm * WM + i * 32 + lrow;
    arow[i] = r * KB;
    asw[i] = (r >> 2) & 3;
  }
  {
    const int g = lane >> 4, li = lane & 15;
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int k, cb;
        if constexpr (ES == 2) {
          k = 8 * (g >> 1) + 4 * h + (li >> 2);
          cb = (wn * WN + j * 32 + 16 * (g & 1) + 4 * (li & 3)) * 2;
        } else {
          k = 16 * (g >> 1) + 8 * h + (li >> 1);
          cb = wn * WN + j * 32 + 16 * (g & 1) + 8 * (li & 1);
        }
        boff[j][h] = AB + k * BR + (((cb >> 4) ^ bsw(k)) << 4) + (cb & 15);
      }
  }
  acc_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
  uint4v af[2][MI], bfr[2][NI];
  auto read_a = [&](const unsigned char* S, int ks, int set, int i) {
    af[set][i] = *reinterpret_cast<const uint4v*>(S + arow[i] + (((ks * 2 + hi) ^ asw[i]) << 4));
  };
  auto read_b = [&](const unsigned char* S, int ks, int set, int j) {
    lds_t* const f = (lds_t*)(S + ks * KSR * BR);
    uint2v l2, h2;
    if constexpr (ES == 2) {
      l2 = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                          reinterpret_cast<short4v __attribute__((address_space(3)))*>(f + boff[j][0])));
      h2 = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                          reinterpret_cast<short4v __attribute__((address_space(3)))*>(f + boff[j][1])));
    } else {
      l2 = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                          reinterpret_cast<int2v __attribute__((address_space(3)))*>(f + boff[j][0])));
      h2 = __builtin_bit_cast(uint2v, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                          reinterpret_cast<int2v __attribute__((address_space(3)))*>(f + boff[j][1])));
    }
    bfr[set][j] = uint4v{l2[0], l2[1], h2[0], h2[1]};
  };
  auto read_frags = [&](const unsigned char* S, int ks, int set) {
#pragma unroll
    for (int i = 0; i < MI; ++i) read_a(S, ks, set, i);
#pragma unroll
    for (int j = 0; j < NI; ++j) read_b(S, ks, set, j);
  };
  // D = A x B, or D^T = B^T x A^T for an i8 result
  auto mma = [&](int set, int i, int j) {
    if constexpr (OUT_I8) acc[i][j] = mfma<ELEM>(bfr[set][j], af[set][i], acc[i][j]);
    else acc[i][j] = mfma<ELEM>(af[set][i], bfr[set][j], acc[i][j]);
  };
  // MFMA n of a K step.  NW = 4: in shells of max(i, j) (shell k holds
  // n = k^2 .. k^2 + 2k: (0, k) .. (k-1, k), then (k, 0) .. (k, k)), the
  // fragments of A row i and B column j being read in slot max(i, j) of the
  // step before; NW = 8: (0,0) (1,0) (0,1) (1,1) (2,0) (3,0) (2,1) (3,1), the
  // step before reading A0, B0, A1 in its first slot and B1, A2, A3 in its
  // second.  Either way the first MFMAs of a step need only the earliest
  // reads.
  auto mma_n = [&](int set, int n) {
    if constexpr (NW == 4 && MI == 4 && NI == 4) {
      const int k = n < 1 ? 0 : n < 4 ? 1 : n < 9 ? 2 : 3, r = n - k * k;
      if (r < k) mma(set, r, k);
      else mma(set, k, r - k);
    } else if constexpr (NW == 4) {
      // the same shells over an MI x NI grid (MI, NI in {2, 4})
      int c = 0, mi = 0, mj = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int r = 0; r < k; ++r)
          if (r < MI && k < NI) {
            if (c == n) mi = r, mj = k;
            ++c;
          }
#pragma unroll
        for (int r = 0; r <= k; ++r)
          if (k < MI && r < NI) {
            if (c == n) mi = k, mj = r;
            ++c;
          }
      }
      mma(set, mi, mj);
    } else {
      mma(set, 2 * (n >> 2) + (n & 1), (n >> 1) & 1);
    }
  };
  // the fragment reads of slot g (of MI * NI / 4 slots) of a K step
  auto slot_reads = [&](const unsigned char* S, int ks, int set, int g) {
    if constexpr (NW == 4 && MI == 4 && NI == 4) {
      read_a(S, ks, set, g);
      read_b(S, ks, set, g);
    } else if constexpr (NW == 4) {
      // slot 0: A0 B0 A1 B1 (the first four MFMAs' shells); slot 1 of a
      // 4 x 2 or 2 x 4 grid: the rest (A2 A3 or B2 B3)
      if (g == 0) {
        read_a(S, ks, set, 0);
        read_b(S, ks, set, 0);
        read_a(S, ks, set, 1);
        read_b(S, ks, set, 1);
      } else if constexpr (MI == 4) {
        read_a(S, ks, set, 2);
        read_a(S, ks, set, 3);
      } else {
        read_b(S, ks, set, 2);
        read_b(S, ks, set, 3);
      }
    } else if (g == 0) {
      read_a(S, ks, set, 0);
      read_b(S, ks, set, 0);
      read_a(S, ks, set, 1);
    } else {
      read_b(S, ks, set, 1);
      read_a(S, ks, set, 2);
      read_a(S, ks, set, 3);
    }
  };

  // The LDS reads need no wait before a barrier: those of the stage whose
  // buffer the next DMA overwrites were consumed by its MFMAs, and the
  // prefetched reads target a buffer no DMA touches until later.
#define XT_WAIT_VM(n) XTK_WAIT_VM(n)
  // prologue: stages 0 .. NS-2 in flight; 0 and 1 landed before B_0
#pragma unroll
  for (int q = 0; q < NS - 1; ++q)
    if (q < nk) dma(q, buf[q]);
  if (nk >= NS - 1) XT_WAIT_VM(PER * (NS - 3));
  else XT_WAIT_VM(0);
  asm volatile("s_barrier" ::: "memory");
  read_frags(buf[0], 0, 0);

  // A stage is 2 MI NI / 4 slots of four MFMAs (8 with four waves, 4 with
  // eight).  Slot g issues, in this order (sched_barrier fences keep the
  // compiler from moving anything across): MFMA, this wave's DMA instruction
  // g of stage s + NS - 1, MFMA, the slot's first fragment read(s), MFMA, the
  // rest, MFMA.  The first half of the slots runs K step 0 on fragment set 0
  // and reads set 1; the second half runs step 1 and reads the next stage's
  // set 0.  Spread out this way the DMA never queues more than one
  // instruction per wave ahead of the MFMAs; issued as a burst after the
  // barrier, it held every wave's issue (C3: ~330 cycles a stage).
  constexpr int SLOTS = MI * NI / 2, HALF = SLOTS / 2;
  // one DMA instruction per slot, two in the first slots of a tile smaller
  // than 256 x 256 (6 for 4 slots, 4 for 2)
  static_assert(PER >= SLOTS && PER <= 2 * SLOTS, "DMA instructions per slot");
  // `more` (a stage NS - 1 ahead exists) is std::true_type in the steady
  // state, so the DMA of each slot is issued with no test in front of it
  // (a test per instruction cost C3 ~70 scalar instructions a stage), and
  // a bool in the last stages.
  auto stage = [&](auto more_c, int s, unsigned char* S, const unsigned char* Snext, unsigned char* Sfree) {
    const bool more = more_c;
#pragma unroll
    for (int g = 0; g < SLOTS; ++g) {
      const int set = g < HALF ? 0 : 1, n0 = 4 * (g % HALF);
      __builtin_amdgcn_sched_barrier(0);
      mma_n(set, n0);
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        dma_one(s + NS - 1, Sfree, g);
        if (g + SLOTS < PER) dma_one(s + NS - 1, Sfree, g + SLOTS);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma_n(set, n0 + 1);
      __builtin_amdgcn_sched_barrier(0);
      // the last stage's reads of Snext fetch a buffer it never uses: kept
      // unconditional so that the waits for this step's fragments do not
      // cover them
      if (g < HALF) slot_reads(S, 1, 1, g);
      else slot_reads(Snext, 0, 0, g - HALF);
      __builtin_amdgcn_sched_barrier(0);
      mma_n(set, n0 + 2);
      __builtin_amdgcn_sched_barrier(0);
      mma_n(set, n0 + 3);
    }
    __builtin_amdgcn_sched_barrier(0);
    // B_{s+1}: this wave's DMA of stage s + 2 landed (stages s+3 .. s+NS-1
    // may stay in flight), its reads done
    if (more) XT_WAIT_VM(PER * (NS - 3));
    else XT_WAIT_VM(0);
    asm volatile("s_barrier" ::: "memory");
  };
  int s0 = 0;
  // steady state: every stage of the group has a stage NS - 1 ahead
  for (; s0 + 2 * NS - 2 < nk; s0 += NS) {
#pragma unroll
    for (int q = 0; q < NS; ++q)
      stage(std::true_type{}, s0 + q, buf[q], buf[(q + 1) % NS], buf[(q + NS - 1) % NS]);
  }
  for (; s0 < nk; s0 += NS) {
#pragma unroll
    for (int q = 0; q < NS; ++q)
      if (s0 + q < nk)
        stage(s0 + q + NS - 1 < nk, s0 + q, buf[q], buf[(q + 1) % NS], buf[(q + NS - 1) % NS]);
  }
#undef XT_WAIT_VM

  const bool hs = p.has_scale, hb = p.has_bias;
  if constexpr (OUT_I8) {
    // D^T = B^T x A^T per 32x32 tile: lane l holds output row m = l%32 of
    // tile i and register v output column 8*(v/4) + 4*(l/32) + v%4 of tile j,
    // so four consecutive columns pack into one 4-byte store.  Without a
    // scale or bias the factors are 1 and 0: x * 1 = x exactly, and x + 0
    // differs from x only for -0, which ftoi maps to 0 like +0.
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n0 = wn * WN + j * 32 + 8 * g + 4 * hi;
        float4v sv = {1.f, 1.f, 1.f, 1.f}, bv = {0.f, 0.f, 0.f, 0.f};
        if (EDGE && n0 >= nleft) continue;
        if (hs) sv = *reinterpret_cast<const float4v*>(t.S + n0);
        if (hb) bv = *reinterpret_cast<const float4v*>(t.Bias + n0);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          if (EDGE && wm * WM + i * 32 + lrow >= mleft) continue;
          const long long off = t.c_off + (long long)(wm * WM + i * 32 + lrow) * p.ldc + n0;
          int q[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) q[e] = ftoi_i8_fast(scale_bias((float)acc[i][j][4 * g + e], sv[e], bv[e], true, true));
          // a plain store: the L2 merges the 8-byte pieces of a row into
          // whole lines (non-temporal stores of them measured 120 us on C6
          // against 78 us for the same GEMM with f32 results)
          *reinterpret_cast<unsigned*>(static_cast<signed char*>(p.c) + off) = pack_i8x4(q);
        }
      }
  } else {
    // D = A x B per 32x32 tile: lane l holds output column l%32 of tile j and
    // register v row 8*(v/4) + 4*(l/32) + v%4 of tile i; a half-wave writes
    // one whole 128-byte line per register.  EPI = false: no scale or bias,
    // so no instructions are spent on them.
    const int orow = hi * 4;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = wn * WN + j * 32 + lrow;
      if (EDGE && n >= nleft) continue;
      const float sv = EPI && hs ? t.S[n] : 1.f, bv = EPI && hb ? t.Bias[n] : 0.f;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = wm * WM + i * 32 + (v >> 2) * 8 + orow + (v & 3);
          if (EDGE && m >= mleft) continue;
          const long long off = t.c_off + (long long)m * p.ldc + n;
          const float x = (float)acc[i][j][v];
          float* const o = static_cast<float*>(p.c) + off;
          // K split (never with an epilogue): the ranges' partial sums meet
          // in the zero-filled output, in an order that varies
          if constexpr (KS) __hip_atomic_fetch_add(o, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          else __builtin_nontemporal_store(EPI ? scale_bias(x, sv, bv, hs, hb) : x, o);
        }
    }
  }
}

TileOff to_off(const xt::TileAddr& a) { return TileOff{a.c0, a.sx, a.sy, a.sz}; }

bool offs_multiple(const xt::TileAddr& a, long long m) {
  return a.c0 % m == 0 && a.sx % m == 0 && a.sy % m == 0 && a.sz % m == 0;
}

// Zero-fills rows x (4 cols4) floats at pitch ld (a kernel, not
// hipMemsetAsync, so that a captured graph replays it correctly).
__global__ __launch_bounds__(256) void gemm_zero_kernel(float* __restrict__ c, long long ld, int rows, int cols4) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long r = i / cols4;
  if (r >= rows) return;
  const long long q = i - r * cols4;
  __builtin_nontemporal_store(float4v{0.f, 0.f, 0.f, 0.f}, reinterpret_cast<float4v*>(c + r * ld) + q);
}

template <int ELEM, bool OUT_I8, int BMT, int BNT, bool EDGE>
void launch_dma(const GemmArgs& a, hipStream_t s) {
  constexpr int NW = BMT * BNT != 65536 ? 4 : EDGE ? 8 : dma_waves<ELEM>();  // EDGE with four waves spills
  const dim3 grid(a.nwg), block(64 * NW);
  if constexpr (OUT_I8) {
    hipLaunchKernelGGL((gemm_dma_kernel<ELEM, kDmaStages, true, true, NW, false, BMT, BNT, EDGE>), grid, block, 0, s, a);
  } else if (a.has_scale || a.has_bias) {
    hipLaunchKernelGGL((gemm_dma_kernel<ELEM, kDmaStages, false, true, NW, false, BMT, BNT, EDGE>), grid, block, 0, s, a);
  } else if (a.ksplit > 1) {
    // the split is taken at square tiles without edges only
    if constexpr (BMT == BNT && !EDGE)
      hipLaunchKernelGGL((gemm_dma_kernel<ELEM, kDmaStages, false, false, NW, true, BMT, BNT>), grid, block, 0, s, a);
  } else {
    hipLaunchKernelGGL((gemm_dma_kernel<ELEM, kDmaStages, false, false, NW, false, BMT, BNT, EDGE>), grid, block, 0, s, a);
  }
}

template <int ELEM, bool OUT_I8>
void launch_t(int bm, int bn, const GemmArgs& a, hipStream_t s) {
  if (bm == 256 && bn == 256)
    a.edge ? launch_dma<ELEM, OUT_I8, 256, 256, true>(a, s) : launch_dma<ELEM, OUT_I8, 256, 256, false>(a, s);
  else if (bm == 256)
    launch_dma<ELEM, OUT_I8, 256, 128, false>(a, s);
  else if (bn == 256)
    launch_dma<ELEM, OUT_I8, 128, 256, false>(a, s);
  else
    a.edge ? launch_dma<ELEM, OUT_I8, 128, 128, true>(a, s) : launch_dma<ELEM, OUT_I8, 128, 128, false>(a, s);
}

}  // namespace

// gemm_small.hip's tiles.  64 x 32 is not one: its 64-byte B rows are half cache
// lines, and it measured behind 32 x 64 on every 16-bit product tried.
static constexpr int kSmallTiles[3][2] = {{64, 64}, {32, 64}, {32, 32}};

static int cu_count() {
  int cus = 256, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    return 256;
  return cus;
}

// Estimated microseconds of a launch of `tiles` bm x bn tiles (K in `ks`
// ranges), fitted to graph-replay times of 30 products from 256 x 320 x 640 to
// 3776 x 6656 x 256: a round of one tile a CU costs its start and end, its K
// loop at the operand rate one CU reached, and its output at its share of HBM.
// (64 x 64: 1024^3 f16 9.5 us measured, 9.2 estimated; 1024 x 1024 x 4096 21.0,
// 20.1.  32 x 64: 256 x 2048 x 5632 18.9, 19.1.  32 x 32: 512^3 4.1, 4.7.
// 128 x 128: 1536^2 x 4096 35.1, 37.  30 other products, of the kernel each
// chose: 0.71 to 1.53 of the estimate, median 1.01; profiles/tile_estimates.txt.)
static double tile_us(int bm, int bn, long long tiles, long long ks, long long kbytes, long long es, int out_bytes, int cus) {
  const double n = double(tiles) * ks / cus;
  // K split: start, end and the zero fill, a range's operands, the atomic sums;
  // 1075 products of 256 x 256 to 1536 x 1280 outputs, 2 to 16 ranges: 0.90 to 1.18
  // of it (256 x 512 x 8192 in 16 ranges 15.1 us, 32 x 32 tiles 22.3;
  // profiles/dispatch_rules.txt)
  if (ks > 1)
    return 3.65 + std::ceil(n) * (bm + bn) * kbytes / ks / 1024 / 59 + 3.9 * ks * double(tiles) * bm * bn / (1 << 20);
  const bool bytes = es == 1;
  double start, rate;  // us a round; KB of operands a us
  if (bm >= 128) start = bm == 256 ? 3 : 2.5, rate = bm == 256 ? 50 : 62;
  else if (bm == 64) start = 3.2, rate = bytes ? 60 : 70;
  else if (bn == 64) start = 2.1, rate = bytes ? 55 : 70;
  else start = 1.5, rate = bytes ? 36 : 50;  // a row of B is a quarter or half of a cache line
  const double round = start + double(bm + bn) * kbytes / 1024 / rate + double(bm) * bn * out_bytes / 1024 / 30;
  // 128 x 128 tiles run two to a CU, the others one
  const double rounds = bm >= 128 && bm + bn < 512 && n > 2 ? n : std::ceil(n);
  return 1.8 + rounds * round;
}

// Tiles of bm x bn over the plan's whole M x N region, columns along x, rows
// along y.
static void region_tiles(const xt::Plan& p, long long M, long long N, int bm, int bn, GemmArgs& a) {
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(N);
  a.mul[0] = a.mul[1] = a.mul[2] = 1;
  a.sub_m = a.sub_n = 1;
  a.vgx = static_cast<int>((N + bn - 1) / bn);
  a.vgy = static_cast<int>((M + bm - 1) / bm);
  a.ta = TileOff{p.a.addr.c0, 0, bm * p.a.ld, 0};
  a.tb = TileOff{p.b.addr.c0, bn, 0, 0};
  a.tc = TileOff{p.c.addr.c0, bn, bm * p.c.ld, 0};
  a.ts = TileOff{p.gemm_scale ? p.scale.addr.c0 : 0, bn, 0, 0};
  a.tbias = TileOff{p.gemm_bias ? p.bias.addr.c0 : 0, bn, 0, 0};
}

hipError_t launch_gemm(const xt::Plan& p, void* const* bufs, hipStream_t s, std::string& why) {
  const bool i8 = p.a.elem == xt::Elem::I8;
  const long long es = i8 ? 1 : 2;
  GemmArgs a = {};
  a.a = static_cast<const unsigned char*>(bufs[p.a.arg]);
  a.b = static_cast<const unsigned char*>(bufs[p.b.arg]);
  a.c = bufs[p.c.arg];
  a.scale = p.gemm_scale ? static_cast<const float*>(bufs[p.scale.arg]) : nullptr;
  a.bias = p.gemm_bias ? static_cast<const float*>(bufs[p.bias.arg]) : nullptr;
  a.has_scale = p.gemm_scale;
  a.has_bias = p.gemm_bias;
  a.ta = to_off(p.a.addr);
  a.tb = to_off(p.b.addr);
  a.tc = to_off(p.c.addr);
  a.ts = p.gemm_scale ? to_off(p.scale.addr) : TileOff{0, 0, 0, 0};
  a.tbias = p.gemm_bias ? to_off(p.bias.addr) : TileOff{0, 0, 0, 0};
  a.lda = p.a.ld;
  a.ldb = p.b.ld;
  a.ldc = p.c.ld;
  const long long kbytes = p.gemm_k * es;
  const long long TM = p.a.rows, TN = p.b.cols;
  if (kbytes % SLICE || TM % 64 || TN % 64) {
    why = i8 ? "i8 matmul tile must have M, N multiples of 64 and K a multiple of 128"
             : "matmul tile must have M, N, K multiples of 64";
    return hipErrorInvalidValue;
  }
  a.nk = static_cast<int>(kbytes / SLICE);
  for (const void* ptr : {bufs[p.a.arg], bufs[p.b.arg], bufs[p.c.arg]})
    if (reinterpret_cast<uintptr_t>(ptr) % 16) {
      why = "matmul buffers must be 16-byte aligned";
      return hipErrorInvalidValue;
    }
  if ((a.lda * es) % 16 || (a.ldb * es) % 16 || !offs_multiple(p.a.addr, 16 / es) ||
      !offs_multiple(p.b.addr, 16 / es)) {
    why = "matmul input tiles must start on 16-byte boundaries";
    return hipErrorInvalidValue;
  }
  // the staging addresses each workgroup's A and B panels with 32-bit offsets
  if (TM * a.lda * es >= (1LL << 32) || p.gemm_k * a.ldb * es >= (1LL << 32)) {
    why = "matmul A and B tile panels must each span less than 4 GiB";
    return hipErrorInvalidValue;
  }
  if (p.c.ld % 4 || !offs_multiple(p.c.addr, 4)) {
    why = "matmul output tiles must start on 4-element boundaries";
    return hipErrorInvalidValue;
  }
  for (int e = 0; e < 2; ++e) {
    const bool on = e == 0 ? p.gemm_scale : p.gemm_bias;
    const xt::Access2D& v = e == 0 ? p.scale : p.bias;
    if (on && (reinterpret_cast<uintptr_t>(bufs[v.arg]) % 16 || !offs_multiple(v.addr, 4))) {
      why = "matmul scale / bias tiles must start on 16-byte boundaries";
      return hipErrorInvalidValue;
    }
  }
  const int cus = cu_count();
  const bool out_i8 = p.c.elem == xt::Elem::I8;
  int64_t M = 0, N = 0;
  float* const cbase = static_cast<float*>(bufs[p.c.arg]) + p.c.addr.c0;
  const bool region = xt::gemm_region(p, M, N) && M < (1LL << 31) && N < (1LL << 31);
  const bool can_split = ksplit_allowed() && !i8 && !out_i8 && !p.gemm_scale && !p.gemm_bias && region && N % 4 == 0 &&
                         p.c.ld % 4 == 0 && reinterpret_cast<uintptr_t>(cbase) % 16 == 0 && M < (1LL << 31);
  // a result over A's or B's bytes: see gemm_tile
  const bool over_a = accesses_meet(p, bufs, p.c, p.a), over_b = accesses_meet(p, bufs, p.c, p.b);
  // Workgroup tile, all on the DMA kernel: 256 x 256 when the Blocks map onto
  // it and its tiles fill the CUs, or are few enough for the K split below;
  // else the first of 256 x 128, 128 x 256, 128 x 128 whose tiles fill the
  // CUs, else the one with the most tiles (a 2048^3 f16 GEMM: 64 tiles of
  // 256 x 256, 256 of 128 x 128).
  struct Cand {
    int bm = 0, bn = 0;
    xt::GemmCover cm, cn;
    long long tiles = 0;
    bool edge = false;  // tiles of the whole region, the last ones reaching past it
  };
  auto try_tile = [&](int bmv, int bnv, Cand& c) {
    c.bm = bmv;
    c.bn = bnv;
    c.cm = xt::gemm_cover(p, bmv, true);
    c.cn = xt::gemm_cover(p, bnv, false);
    if (!xt::gemm_tile(c.cm, c.cn, over_a, over_b)) return false;
    long long g[3] = {p.grid[0], p.grid[1], p.grid[2]};
    if (c.cm.axis >= 0) g[c.cm.axis] /= c.cm.factor;
    if (c.cn.axis >= 0) g[c.cn.axis] /= c.cn.factor;
    c.tiles = g[0] * g[1] * g[2] * c.cm.sub * c.cn.sub;
    return true;
  };
  Cand pick, c256, c128;
  const bool has256 = try_tile(256, 256, c256);
  // A GEMM of at most CUs / 8 tiles of 256 x 256 that can split K takes 128
  // x 128 tiles with the split (1024 x 1024 x 4096 f16: 42.3 us on 16 tiles
  // of 256 x 256 in 8 K ranges, 28.2 on 64 of 128 x 128 in 4; hipBLASLt 25.1)
  const bool tiny = can_split && has256 && c256.tiles * 8 <= cus;
  if (tiny && try_tile(128, 128, c128)) {
    pick = c128;
  } else if (has256 && (c256.tiles >= cus || tiny)) {
    pick = c256;
  } else {
    Cand most = has256 ? c256 : Cand{};
    bool found = false;
    const int shapes[3][2] = {{256, 128}, {128, 256}, {128, 128}};
    for (const auto& sh : shapes) {
      Cand c;
      if (!try_tile(sh[0], sh[1], c)) continue;
      if (c.tiles >= cus) {
        pick = c;
        found = true;
        break;
      }
      if (c.tiles > most.tiles) most = c;
    }
    if (!found) pick = most;
  }
  // K ranges of the split below, 1 for none
  auto ranges = [&](const Cand& c) {
    const bool few = c.bm == 256 ? c.tiles * 8 <= cus : tiny && c.bm == 128 && c.tiles * 2 <= cus;
    if (!can_split || c.edge || c.bm != c.bn || c.bm < 128 || !few) return 1LL;
    return std::max(1LL, std::min<long long>(cus / c.tiles, a.nk * 2LL / 16));
  };
  // Where those tiles leave CUs idle, or none maps, the small tiles and the
  // 128 x 128 and 256 x 256 tiles with edges compete by estimated time.
  if (pick.bm == 0 || pick.tiles < cus) {
    double best = pick.bm == 0 ? 1e30 : tile_us(pick.bm, pick.bn, pick.tiles, ranges(pick), kbytes, es, out_i8 ? 1 : 4, cus);
    // a K split has to be 2 us ahead, the most that small tiles took below their
    // estimate (821 products with both measured: 0.17% behind the better of the two
    // on average, 0.83% without it; 256 x 256 x 2560 7.8 us on 32 x 32, split 9.9)
    if (ranges(pick) > 1) best += 2;
    auto offer = [&](const Cand& c) {
      const double us = tile_us(c.bm, c.bn, c.tiles, 1, kbytes, es, out_i8 ? 1 : 4, cus);
      if (us < best && grid_fits(c.tiles, 512)) {
        best = us;
        pick = c;
      }
    };
    for (const auto& sh : kSmallTiles) {
      Cand c;
      if (try_tile(sh[0], sh[1], c)) offer(c);
    }
    for (int t : {128, 256}) {
      Cand c;
      if (!region || (over_a && N > t) || (over_b && M > t) || try_tile(t, t, c) || t * a.lda * es >= (1LL << 32)) continue;
      c = Cand{};
      c.bm = c.bn = t;
      c.edge = true;
      c.tiles = (M + t - 1) / t * ((N + t - 1) / t);
      offer(c);
    }
    if (pick.bm == 0) {
      why = over_a || over_b ? "a matmul over the bytes of its own operand needs Blocks that workgroup tiles cover whole"
                             : "matmul Blocks cannot be mapped onto workgroup tiles in one launch";
      return hipErrorInvalidValue;
    }
  }
  const int bm = pick.bm, bn = pick.bn;
  const xt::GemmCover cm = pick.cm, cn = pick.cn;
  a.mul[0] = a.mul[1] = a.mul[2] = 1;
  int vg[3] = {p.grid[0], p.grid[1], p.grid[2]};
  if (cm.axis >= 0) {
    a.mul[cm.axis] = cm.factor;
    vg[cm.axis] /= cm.factor;
  }
  if (cn.axis >= 0) {
    a.mul[cn.axis] = cn.factor;
    vg[cn.axis] /= cn.factor;
  }
  a.vgx = vg[0];
  a.vgy = vg[1];
  a.sub_m = cm.sub;
  a.sub_n = cn.sub;
  a.edge = pick.edge;
  if (pick.edge) region_tiles(p, M, N, bm, bn, a);
  long long nwg = pick.edge ? (long long)a.vgx * a.vgy : (long long)vg[0] * vg[1] * vg[2] * a.sub_m * a.sub_n;
  if (!grid_fits(nwg, bm == 256 && bn == 256 ? 512 : 256)) {
    why = "matmul grid of " + std::to_string(nwg) + " workgroup tiles exceeds one launch";
    return hipErrorInvalidValue;
  }
  a.nwg = static_cast<int>(nwg);
  a.group = kTileGroup;
  a.tiles = a.nwg;
  a.ksplit = 1;
  a.kstages = a.nk * 2;
  // K split: when the 256 x 256 tiles fill at most an eighth of the CUs, f32
  // results of f16 / bf16 products without an epilogue split K into ranges
  // of at least 16 stages (spread evenly: lengths differ by at most one),
  // one workgroup each, adding their partial sums atomically into the
  // zero-filled output (the f32 addition order, and so the last bits, vary
  // between runs; i8 sums stay exact and whole).  XTILE_AMD_KSPLIT=0 turns
  // the split off (run-to-run reproducible results).
  // Measured (f16, 30 launches): 1024 x 1024 x 4096 (16 tiles) 79.2 us whole,
  // 42.8 in 8 ranges; 2048^3 (64 tiles) 47.3 whole, 71.4 in 4; 1024 x 8192 x
  // 8192 (128 tiles) 155.9 whole, 164.4 in 2.
  if (const long long ks = ranges(pick); ks > 1) {
    a.kstages = (int)(a.nk * 2LL / ks);
    a.ksplit = (int)ks;
    a.nwg = (int)(nwg * ks);
    const long long n4 = M * (N / 4);
    hipLaunchKernelGGL(gemm_zero_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, cbase, p.c.ld,
                       (int)M, (int)(N / 4));
  }
  a.divide();
  if (bm <= 64) {
    a.K = static_cast<int>(p.gemm_k);
    a.cvec = reinterpret_cast<uintptr_t>(static_cast<char*>(bufs[p.c.arg])) % 16 == 0;
    return run_gemm_small(p.a.elem, out_i8, bm, bn, true, a, s);
  }
  switch (p.a.elem) {
    case xt::Elem::I8: out_i8 ? launch_t<kI8, true>(bm, bn, a, s) : launch_t<kI8, false>(bm, bn, a, s); break;
    case xt::Elem::BF16:
      out_i8 ? launch_t<kBF16, true>(bm, bn, a, s) : launch_t<kBF16, false>(bm, bn, a, s);
      break;
    default: out_i8 ? launch_t<kF16, true>(bm, bn, a, s) : launch_t<kF16, false>(bm, bn, a, s); break;
  }
  return hipGetLastError();
}

bool launch_gemm_ragged(const xt::Plan& p, void* const* bufs, hipStream_t s, hipError_t& e) {
  const bool i8 = p.a.elem == xt::Elem::I8, out_i8 = p.c.elem == xt::Elem::I8;
  const long long es = i8 ? 1 : 2;
  int64_t M, N;
  if (!xt::gemm_region(p, M, N) || M >= (1LL << 31) || N >= (1LL << 31) || p.gemm_k >= (1LL << 17)) return false;
  // a result over its operands stays staged, one workgroup a Block; over the
  // epilogue's rows it may lie where it is one row, which the thread that
  // stores a column read at that column before
  if (accesses_meet(p, bufs, p.c, p.a) || accesses_meet(p, bufs, p.c, p.b) ||
      (M > 1 && ((p.gemm_scale && accesses_meet(p, bufs, p.c, p.scale)) ||
                 (p.gemm_bias && accesses_meet(p, bufs, p.c, p.bias)))))
    return false;
  auto origin = [&](const xt::Access2D& v, long long b) { return static_cast<unsigned char*>(bufs[v.arg]) + v.addr.c0 * b; };
  auto aligned = [](const void* q, long long n) { return reinterpret_cast<uintptr_t>(q) % n == 0; };
  const unsigned char *A = origin(p.a, es), *B = origin(p.b, es), *C = origin(p.c, out_i8 ? 1 : 4);
  if (!aligned(A, es) || !aligned(B, es) || (!out_i8 && !aligned(C, 4))) return false;
  GemmArgs a = {};
  a.a = static_cast<unsigned char*>(bufs[p.a.arg]);
  a.b = static_cast<unsigned char*>(bufs[p.b.arg]);
  a.c = bufs[p.c.arg];
  if (p.gemm_scale) a.scale = static_cast<const float*>(bufs[p.scale.arg]);
  if (p.gemm_bias) a.bias = static_cast<const float*>(bufs[p.bias.arg]);
  if (!aligned(a.scale, 4) || !aligned(a.bias, 4)) return false;
  a.has_scale = p.gemm_scale;
  a.has_bias = p.gemm_bias;
  a.lda = p.a.ld;
  a.ldb = p.b.ld;
  a.ldc = p.c.ld;
  a.K = static_cast<int>(p.gemm_k);
  a.edge = 1;
  a.cvec = a.ldc % 4 == 0 && aligned(C, out_i8 ? 4 : 16);
  const int cus = cu_count();
  int bm = 0, bn = 0;
  double best = 1e30;
  for (const auto& sh : kSmallTiles) {
    const double us = tile_us(sh[0], sh[1], (M + sh[0] - 1) / sh[0] * ((N + sh[1] - 1) / sh[1]), 1, p.gemm_k * es, es,
                              out_i8 ? 1 : 4, cus);
    if (us < best) best = us, bm = sh[0], bn = sh[1];
  }
  region_tiles(p, M, N, bm, bn, a);
  const long long nwg = (long long)a.vgx * a.vgy;
  if (!grid_fits(nwg, 256)) return false;
  a.nwg = a.tiles = static_cast<int>(nwg);
  a.ksplit = 1;
  a.group = kTileGroup;
  a.divide();
  // LDS DMA: 16-byte rows and K chunks, and panels whose offsets stay below
  // 2^31, where the K tail's out-of-range offsets begin
  const bool dma = aligned(A, 16) && aligned(B, 16) && (a.lda * es) % 16 == 0 && (a.ldb * es) % 16 == 0 &&
                   (a.K * es) % 16 == 0 && bm * a.lda * es < (1LL << 31) && a.K * a.ldb * es < (1LL << 31);
  // the register path's loads of partial chunks reach back up to 16 bytes in a row
  if (!dma && (a.K * es < 16 || N * es < 16)) return false;
  e = run_gemm_small(p.a.elem, out_i8, bm, bn, dma, a, s);
  return true;
}

}  // namespace xtk
