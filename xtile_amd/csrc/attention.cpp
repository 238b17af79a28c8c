// Attention Blocks: softmax(Q K^T) V programs whose staged kernel would walk
// its phases one after another, turned into the source of one HIP kernel that
// keeps the scores in registers.  Host code; the runtime compiles it like every
// staged kernel (kernels/fused_jit.cpp).
//
// What bounds the program is the f32 product P V (P and V are f32 in the
// program and stay so): 64 heads x 512 queries x 256 keys x 64 is 6.8 us of
// v_mfma_f32_16x16x4_f32 at the rate of the chip, against 3 us of memory
// traffic.  The staged kernel of the same program (one Block a CU, scores and
// probabilities through LDS, a barrier between phases) took 51.3 us a launch,
// this one 15.6; 256 heads x 512 x 160 x 128 308 -> 58, 9 x 96 x 232 x 64 21.4 ->
// 5.7, 1024 x 64 x 64 x 64 15.2 -> 12.7, and none of 30 drawn sizes slower
// (profiles/attention_staged_compare.txt).  The matrix pipes are busy 0.59 of the
// first one's cycles (profiles/attention_256_xt_attend.txt).  Raising
// half of the waves' priority, to set softmax against products, changed nothing.
//
//   * A workgroup holds one head's K (16 bits) and V (f32) in LDS, fetched once
//     by LDS DMA, V behind the scores' products.  Its waves each take 16 query
//     rows, or (DS > 1, where there are too few rows to fill the chip) a 1 / DS
//     share of V's columns of the same rows; query tiles of one head that the
//     grid walks are one row range, so the program's own query tile does not
//     set the work of a wave.
//   * Scores are computed transposed, S^T = K Q^T (v_mfma_f32_16x16x32): lane l
//     then holds, for query l % 16, the keys 16 b + 4 (l / 16) + r in register
//     r of block b.  That is an A operand of v_mfma_f32_16x16x4_f32 if step r of
//     a block multiplies the keys 16 b + {r, 4 + r, 8 + r, 12 + r}: P goes from
//     the softmax into the second product without leaving its lane.
//   * The row maximum and sum are per lane over its registers, then over the
//     four lanes of a query (two shuffles).
//   * V's rows are stored in the order the steps read them (row 16 b + 4 r + g
//     holds key 16 b + 4 g + r), so the four lane groups of a read take four
//     consecutive rows: no bank conflicts at any width.  A lane reads adjacent
//     columns for up to four products and stores them as one vector.
//   * K's 16-byte chunks are swizzled by row so that the 16 rows of a fragment
//     read meet in different banks.
// Keys past nk (nk is padded to 16) score -inf, so their probability is 0, and
// their K and V rows read as zeros.
#include <algorithm>
#include <cmath>
#include <map>
#include <sstream>

#include "fused_common.h"
#include "plan.h"

namespace xt {
namespace {

constexpr int kCus = 256;
constexpr long long kLds = 160 * 1024;

struct Form {
  const VmAccess *q = nullptr, *k = nullptr, *v = nullptr, *o = nullptr;
  int iq = 0, ik = 0, iv = 0, io = 0;  // access indices
  int tq = 0, nk = 0, d = 0;
};

// The program as store(matmul(e * recip(sum(e)), V)), e = exp(s - max(s)),
// s = matmul(Q, transpose(K)), each part read by nothing else.
bool match(const VmPlan& vm, Form& f) {
  if (vm.inst.size() != 13) return false;
  std::map<int, int> cur;  // slot -> the instruction that wrote it last
  struct In {
    int a = -1, b = -1;
  };
  std::vector<In> from(vm.inst.size());
  for (size_t i = 0; i < vm.inst.size(); ++i) {
    const VmInst& in = vm.inst[i];
    auto at = [&](int slot) {
      auto it = cur.find(slot);
      return it == cur.end() ? -1 : it->second;
    };
    if (in.op != VmOp::Load) from[i].a = at(in.a);
    if (in.op == VmOp::Binary || in.op == VmOp::Matmul) from[i].b = at(in.b);
    if (in.op != VmOp::Store) cur[in.dst] = static_cast<int>(i);
  }
  auto is = [&](int i, VmOp op, int kind = -1) {
    return i >= 0 && vm.inst[i].op == op && (kind < 0 || vm.inst[i].kind == kind);
  };
  const int st = static_cast<int>(vm.inst.size()) - 1;
  if (!is(st, VmOp::Store)) return false;
  const int pv = from[st].a;
  if (!is(pv, VmOp::Matmul) || vm.inst[pv].c >= 0 || vm.inst[pv].aux[1]) return false;
  const int p = from[pv].a, v = from[pv].b;
  if (!is(p, VmOp::Binary, static_cast<int>(VmBinary::Mul)) || !is(v, VmOp::Load)) return false;
  int e = from[p].a, r = from[p].b;
  if (is(e, VmOp::Unary, static_cast<int>(VmUnary::Recip))) std::swap(e, r);
  if (!is(e, VmOp::Unary, static_cast<int>(VmUnary::Exp)) || !is(r, VmOp::Unary, static_cast<int>(VmUnary::Recip)))
    return false;
  const int sum = from[r].a, sub = from[e].a;
  if (!is(sum, VmOp::Reduce, static_cast<int>(VmReduce::Sum)) || from[sum].a != e || vm.inst[sum].aux[0] != 1 ||
      !is(sub, VmOp::Binary, static_cast<int>(VmBinary::Sub)))
    return false;
  const int s = from[sub].a, mx = from[sub].b;
  if (!is(s, VmOp::Matmul) || vm.inst[s].c >= 0 || vm.inst[s].aux[1] ||
      !is(mx, VmOp::Reduce, static_cast<int>(VmReduce::Max)) || from[mx].a != s || vm.inst[mx].aux[0] != 1)
    return false;
  const int q = from[s].a, kt = from[s].b;
  if (!is(q, VmOp::Load) || !is(kt, VmOp::Permute)) return false;
  const int* perm = vm.inst[kt].aux;
  const int k = from[kt].a;
  if (perm[0] != 0 || perm[1] != 2 || perm[2] != 1 || !is(k, VmOp::Load)) return false;
  f.tq = vm.inst[s].dims[1];
  f.nk = vm.inst[s].dims[2];
  f.d = vm.inst[s].aux[0];
  auto tile = [&](int i, int rows, int cols) {
    const int* n = vm.inst[i].dims;
    return n[0] == 1 && n[1] == rows && n[2] == cols;
  };
  if (!tile(q, f.tq, f.d) || !tile(k, f.nk, f.d) || !tile(v, f.nk, f.d) || !tile(st, f.tq, f.d) || vm.inst[s].dims[0] != 1 ||
      vm.inst[pv].dims[1] != f.tq || vm.inst[pv].dims[2] != f.d || vm.inst[pv].aux[0] != f.nk)
    return false;
  f.iq = vm.inst[q].kind;
  f.ik = vm.inst[k].kind;
  f.iv = vm.inst[v].kind;
  f.io = vm.inst[st].kind;
  f.q = &vm.access[f.iq];
  f.k = &vm.access[f.ik];
  f.v = &vm.access[f.iv];
  f.o = &vm.access[f.io];
  return true;
}

bool multiple(const VmAccess& a, long long n) {
  return a.stride[2] == 1 && a.stride[1] % n == 0 && a.addr.c0 % n == 0 && a.addr.sx % n == 0 && a.addr.sy % n == 0 &&
         a.addr.sz % n == 0;
}

long long step(const VmAccess& a, int axis) { return axis == 0 ? a.addr.sx : axis == 1 ? a.addr.sy : a.addr.sz; }

const char* kBody = R"(
typedef int xi4v __attribute__((ext_vector_type(4)));
typedef unsigned xu4v __attribute__((ext_vector_type(4)));
typedef _Float16 xh8 __attribute__((ext_vector_type(8)));
typedef __bf16 xb8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ xi4v xrsrc(const void* p) {
  const unsigned long long b = reinterpret_cast<unsigned long long>(p);
  return xi4v{(int)(unsigned)b, (int)(unsigned)(b >> 32) & 0xFFFF, (int)0x80000000u, 0x00020000};
}
// 16 bytes a lane from offset voff (zeros from 2^31 on) to LDS lds + 16 lane; waited for by count
__device__ __forceinline__ void xdma(xi4v r, unsigned lds, unsigned voff) {
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(voff), "s"(r), "{m0}"(lds) : "memory");
}
__device__ __forceinline__ xf4 xmm16(xu4v a, xu4v b, xf4 c) {
  if constexpr (BF) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(xb8, a), __builtin_bit_cast(xb8, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(xh8, a), __builtin_bit_cast(xh8, b), c, 0, 0, 0);
}
constexpr int KB = (NK + 15) / 16;             // key blocks
constexpr int KROW = D * 2, VROW = D * 4;      // LDS row bytes
constexpr int KBYTES = KB * 16 * KROW, VBYTES = KB * 16 * VROW;
constexpr int DW = D / DS, NB = DW / 16;       // a wave's columns, its products a step
constexpr int VW = NB >= 4 ? 4 : NB;           // columns of one LDS read and store
extern "C" __global__ void __launch_bounds__(64 * NW) xt_attend(FusedArgs a) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(1024))) unsigned char L[KBYTES + VBYTES];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  // workgroups go round-robin over 8 XCDs: a head's workgroups to one XCD's L2
  const int per = WGS / 8, rem = WGS % 8, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int id = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
  const int head = id / WPH, first = id % WPH;
  const int ha = head % GA, hb = head / GA;
  const unsigned short* const Q = static_cast<const unsigned short*>(a.p[IQ]) + (QC + ha * QA + hb * QB);
  const unsigned short* const K = static_cast<const unsigned short*>(a.p[IK]) + (KC + ha * KA + hb * KBS);
  const float* const V = static_cast<const float*>(a.p[IV]) + (VC + ha * VA + hb * VBS);
  float* const O = static_cast<float*>(a.p[IO]) + (OC + ha * OA + hb * OB);
  const unsigned lbase = (unsigned)reinterpret_cast<unsigned long long>((__attribute__((address_space(3))) unsigned char*)L);
  // the chunk that row `row` of K keeps at position c
  auto swz = [](int row) { return D == 32 ? (row >> 2) & 3 : D == 64 ? (row >> 1) & 7 : row & 15; };
  {
    const xi4v rk = xrsrc(K);
    constexpr int RPI = 1024 / KROW, CPR = KROW / 16;
#pragma unroll
    for (int i = wave; i < KBYTES / 1024; i += NW) {
      const int row = i * RPI + lane / CPR, c = (lane % CPR) ^ swz(row);
      xdma(rk, lbase + i * 1024, row < NK ? (unsigned)row * (LDK * 2) + c * 16 : 0x80000000u);
    }
  }
  const int rt = wave / DS, col0 = (wave % DS) * DW;
  xu4v qf[D / 32];
  auto load_q = [&](int tile) {
    const int row = min(tile * (16 * RT) + rt * 16 + n16, M - 1);
#pragma unroll
    for (int s = 0; s < D / 32; ++s)
      qf[s] = *reinterpret_cast<const xu4v*>(Q + (long long)row * LDQ + s * 32 + g * 8);
  };
  load_q(first);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): K and Q
  asm volatile("s_barrier" ::: "memory");
  {
    const xi4v rv = xrsrc(V);
    constexpr int RPI = 1024 / VROW, CPR = VROW / 16;
#pragma unroll
    for (int i = wave; i < VBYTES / 1024; i += NW) {
      const int s = i * RPI + lane / CPR;
      const int key = (s & ~15) + 4 * (s & 3) + ((s >> 2) & 3);
      xdma(rv, lbase + KBYTES + i * 1024, key < NK ? (unsigned)key * (LDV * 4) + (lane % CPR) * 16 : 0x80000000u);
    }
  }
#pragma unroll 1
  for (int it = 0; it < ITERS; ++it) {
    const int tile = first + it * WPH, row0 = tile * (16 * RT) + rt * 16;
    const bool active = tile < TILES && row0 < M;
    xf4 s[KB];
    if (active) {
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        xf4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
          const int row = 16 * b + n16;
          const xu4v kf = *reinterpret_cast<const xu4v*>(L + row * KROW + (((4 * c + g) ^ swz(n16)) << 4));
          acc = xmm16(kf, qf[c], acc);
        }
        s[b] = acc;
      }
      if constexpr (NK % 16 != 0)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * (KB - 1) + 4 * g + r >= NK) s[KB - 1][r] = -__builtin_huge_valf();
      float m = -__builtin_huge_valf();
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, s[b][r]);
      m = fmaxf(m, __shfl_xor(m, 16, 64));
      m = fmaxf(m, __shfl_xor(m, 32, 64));
      xf4 sums = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = s[b][r] - m;
          const float e = __builtin_amdgcn_exp2f(x * 1.44269504088896340736f);
          s[b][r] = e;
          sums[r] += e;
        }
      float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      const float inv = 1.0f / sum;
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[b][r] *= inv;
    }
    if (it == 0) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): V
      asm volatile("s_barrier" ::: "memory");
    }
    if (!active) continue;
    if (it + 1 < ITERS) load_q(tile + WPH);
    xf4 o[2][NB];  // even and odd key blocks: shorter sums, smaller rounding errors
#pragma unroll
    for (int n = 0; n < NB; ++n) o[0][n] = o[1][n] = xf4{0.f, 0.f, 0.f, 0.f};
    float v[2][4][NB];
    auto read_v = [&](int b, int set) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < NB; n += VW) {
          const unsigned char* at = L + KBYTES + (16 * b + 4 * r + g) * VROW + (col0 + n * 16 + VW * n16) * 4;
          if constexpr (VW == 4) {
            const xf4 x = *reinterpret_cast<const xf4*>(at);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[set][r][n + e] = x[e];
          } else if constexpr (VW == 2) {
            const xf2 x = *reinterpret_cast<const xf2*>(at);
            v[set][r][n] = x[0];
            v[set][r][n + 1] = x[1];
          } else {
            v[set][r][n] = *reinterpret_cast<const float*>(at);
          }
        }
    };
    read_v(0, 0);
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      if (b + 1 < KB) read_v(b + 1, (b + 1) & 1);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < NB; ++n) o[b & 1][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[b][r], v[b & 1][r][n], o[b & 1][n], 0, 0, 0);
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) o[0][n] += o[1][n];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 4 * g + r;
      if (row < M)
#pragma unroll
        for (int n = 0; n < NB; n += VW) {
          float* const at = O + (long long)row * LDO + col0 + n * 16 + VW * n16;
          if constexpr (VW == 4) __builtin_nontemporal_store(xf4{o[0][n][r], o[0][n + 1][r], o[0][n + 2][r], o[0][n + 3][r]}, reinterpret_cast<xf4*>(at));
          else if constexpr (VW == 2) __builtin_nontemporal_store(xf2{o[0][n][r], o[0][n + 1][r]}, reinterpret_cast<xf2*>(at));
          else __builtin_nontemporal_store(o[0][n][r], at);
        }
    }
  }
}
}  // namespace xatt
)";

}  // namespace

bool attend_vm(const VmPlan& vm, const int32_t grid[3], FusedPlan& fp) {
  Form f;
  if (!match(vm, f)) return false;
  // Several workgroups read a head's K and V while others store its rows: O is a
  // memref of its own (buffers that meet: launch_fused).  A Block that updates
  // its own tile in place stays with the staged kernel, one workgroup a Block.
  if (f.o->arg == f.v->arg || f.o->arg == f.k->arg || f.o->arg == f.q->arg) return false;
  if ((f.q->elem != Elem::F16 && f.q->elem != Elem::BF16) || f.k->elem != f.q->elem || f.v->elem != Elem::F32 ||
      f.o->elem != Elem::F32)
    return false;
  if (f.d != 32 && f.d != 64 && f.d != 128) return false;
  if (!multiple(*f.q, 8) || !multiple(*f.k, 8) || !multiple(*f.v, 4) || !multiple(*f.o, 4)) return false;
  const long long ldk = f.k->stride[1], ldv = f.v->stride[1];
  const int kp = (f.nk + 15) / 16 * 16;
  const long long lds = (long long)kp * f.d * 6;
  // the kernel holds every pitch in an int
  if (f.q->stride[1] >= (1LL << 31) || f.o->stride[1] >= (1LL << 31)) return false;
  if (lds > kLds || f.nk > 512 || ldk * 2 * f.nk >= (1LL << 31) || ldv * 4 * f.nk >= (1LL << 31)) return false;
  // the grid axis whose Blocks continue the query rows of one head
  int rows_axis = -1;
  for (int ax = 0; ax < 3 && rows_axis < 0; ++ax)
    if (grid[ax] > 1 && step(*f.q, ax) == f.tq * f.q->stride[1] && step(*f.o, ax) == f.tq * f.o->stride[1] &&
        step(*f.k, ax) == 0 && step(*f.v, ax) == 0)
      rows_axis = ax;
  const long long m = (long long)f.tq * (rows_axis < 0 ? 1 : grid[rows_axis]);
  if (m >= (1LL << 30)) return false;
  // a head's index counts the remaining axes longer than 1, of which there may be two
  int axes[3], na = 0;
  for (int ax = 0; ax < 3; ++ax)
    if (ax != rows_axis && grid[ax] > 1) axes[na++] = ax;
  if (na > 2) return false;
  const long long ga = na > 0 ? grid[axes[0]] : 1, gb = na > 1 ? grid[axes[1]] : 1, heads = ga * gb;
  // Waves: up to eight 16-row tiles a workgroup while that leaves most CUs a
  // workgroup; then, while there are fewer than two waves a SIMD, V's columns
  // shared by up to four waves of the same rows (the scores are computed again,
  // a 16th of the work).  225 heads x 32 x 224 keys x 64: 2 x 4 waves 8.4 us, 1
  // x 4 in twice the workgroups 10.1; 1024 x 64 x 64 x 64: 4 x 1 12.7 us, 4 x 2
  // 12.9.
  const long long row_tiles = (m + 15) / 16;
  int rt = 8;
  while (rt > 1 && (rt / 2 >= row_tiles || heads * ((row_tiles + rt - 1) / rt) < kCus * 3 / 4)) rt /= 2;
  int ds = 1;
  while (ds < std::min({4, f.d / 16, 8 / rt}) && heads * ((row_tiles + rt - 1) / rt) * rt * ds < kCus * 8) ds *= 2;
  const int nw = rt * ds;
  const long long tiles = (row_tiles + rt - 1) / rt;
  // several tiles a workgroup where one each would take more than a round
  const long long held = kCus * std::max(1LL, std::min<long long>(kLds / lds, 8 / nw));
  const long long iters = std::max(1LL, std::min(tiles, heads * tiles / held));
  const long long wph = (tiles + iters - 1) / iters;
  const long long wgs = heads * wph;
  if (wgs < 1 || wgs > 0x7fffffffLL || wgs * 64 * nw >= (1LL << 32)) return false;
  std::ostringstream k;
  auto c = [&](const char* name, long long v) { k << "constexpr int " << name << " = " << v << ";\n"; };
  auto o = [&](const char* base, const VmAccess& a, const char* na_, const char* nb_) {
    k << "constexpr long long " << base << " = " << a.addr.c0 << "LL, " << na_ << " = " << (na > 0 ? step(a, axes[0]) : 0)
      << "LL, " << nb_ << " = " << (na > 1 ? step(a, axes[1]) : 0) << "LL;\n";
  };
  k << "constexpr bool BF = " << (f.q->elem == Elem::BF16 ? "true" : "false") << ";\n";
  c("NK", f.nk), c("D", f.d), c("M", m), c("NW", nw), c("DS", ds), c("RT", rt), c("TILES", tiles), c("ITERS", iters);
  c("WPH", wph), c("WGS", wgs), c("GA", ga), c("IQ", f.iq), c("IK", f.ik), c("IV", f.iv), c("IO", f.io);
  c("LDQ", f.q->stride[1]), c("LDK", ldk), c("LDV", ldv), c("LDO", f.o->stride[1]);
  o("QC", *f.q, "QA", "QB"), o("KC", *f.k, "KA", "KBS"), o("VC", *f.v, "VA", "VBS"), o("OC", *f.o, "OA", "OB");
  // before the staged kernel, in the same program
  const std::string head = fused_preamble();
  fp.source = head + "namespace xatt {\n" + k.str() + kBody + fp.source.substr(head.size());
  fp.attend_threads = 64 * nw;
  fp.attend_workgroups = static_cast<int>(wgs);
  std::ostringstream lay;
  lay << " attention waves=" << nw << " rows=" << 16 * rt << " columns=" << f.d / ds << " workgroups=" << wgs;
  fp.layout += lay.str();
  return true;
}

}  // namespace xt
