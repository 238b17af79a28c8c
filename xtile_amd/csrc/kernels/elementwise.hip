// Bandwidth-bound tile programs: elementwise binary ops and row softmax.
//
// Consecutive lanes touch consecutive 16-byte chunks, so each wave instruction
// covers whole 64-byte segments; how Blocks and rows map to workgroups is
// described at each kernel.
//
// Semantics follow the reference DSL: add/sub/mul are plain IEEE f32 ops
// (xtile/dsl.py:321-325,351-352); softmax is x - max(x), exp, sum, then
// multiply by reciprocal(sum) exactly as `x / r` is traced
// (xtile/dsl.py:354-357, kernels/softmax.py:13-18).  exp is exp_fast
// (common.h: relative error below 5.3e-6 for normal results, against the
// 1e-5 relative bar of the f32 softmax), and full-wave reductions use DPP
// (wave_reduce); together they took C2 from 43.0 to 41.9 us a launch.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace xtk {
namespace {

struct EwArgs {
  const float* a;
  const float* b;
  float* c;
  TileOff ta, tb, tc;
  long long lda, ldb, ldc;
  int rows, cols;
  BlockDecode grid;  // y fastest when that makes neighbouring workgroups neighbours in memory
  int cv_shift;      // log2(cols / VW) when that is a power of two, else -1
};

template <int OP>
__device__ __forceinline__ float ew_apply(float x, float y) {
  if constexpr (OP == 0) return x + y;
  else if constexpr (OP == 1) return x - y;
  else return x * y;
}

// Streaming accesses: tiles are read and written exactly once per launch, so
// loads and stores are non-temporal (they do not displace reusable lines).
template <typename T>
__device__ __forceinline__ T ld_nt(const T* p) { return __builtin_nontemporal_load(p); }
template <typename T>
__device__ __forceinline__ void st_nt(T v, T* p) { __builtin_nontemporal_store(v, p); }

// Four floats at element alignment.
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4v ld_nt4(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const float4u*>(p));
}
__device__ __forceinline__ void st_nt4(float4v v, float* p) {
  __builtin_nontemporal_store(v, reinterpret_cast<float4u*>(p));
}

// Each thread handles U vectors per step; U is the smallest of 1, 2, 4 that
// covers the tile in one step (4 when it takes several).  All U loads are
// issued before any is consumed; indices past the end of the tile (only in a
// tile's last step) are clamped to element 0 and their results discarded, so a
// step costs one memory round trip, not U.  POW2: the row length in vectors is
// a power of two and row/column come from a shift and a mask.
template <int OP, int VW, int U, bool POW2>
__global__ __launch_bounds__(256) void ew_binary_kernel(EwArgs p) {
  int x, y, z;
  p.grid(blockIdx.x, x, y, z);
  const float* A = p.a + p.ta.at(x, y, z);
  const float* B = p.b + p.tb.at(x, y, z);
  float* C = p.c + p.tc.at(x, y, z);
  const int cv = p.cols / VW;
  const int n = p.rows * cv;
  for (int base = threadIdx.x; base < n; base += 256 * U) {
    long long offa[U], offb[U], offc[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u * 256;
      ok[u] = i < n;
      const int ic = ok[u] ? i : 0;
      const int r = POW2 ? (ic >> p.cv_shift) : ic / cv;
      const int col = (POW2 ? (ic & (cv - 1)) : ic - r * cv) * VW;
      offa[u] = r * p.lda + col;
      offb[u] = r * p.ldb + col;
      offc[u] = r * p.ldc + col;
    }
    if constexpr (VW == 4) {
      float4v va[U], vb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        va[u] = ld_nt(reinterpret_cast<const float4v*>(A + offa[u]));
        vb[u] = ld_nt(reinterpret_cast<const float4v*>(B + offb[u]));
      }
      issue_fence();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float4v vc;
        vc.x = ew_apply<OP>(va[u].x, vb[u].x);
        vc.y = ew_apply<OP>(va[u].y, vb[u].y);
        vc.z = ew_apply<OP>(va[u].z, vb[u].z);
        vc.w = ew_apply<OP>(va[u].w, vb[u].w);
        if (ok[u]) st_nt(vc, reinterpret_cast<float4v*>(C + offc[u]));
      }
    } else {
      float va[U], vb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        va[u] = ld_nt(A + offa[u]);
        vb[u] = ld_nt(B + offb[u]);
      }
      issue_fence();
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) st_nt(ew_apply<OP>(va[u], vb[u]), C + offc[u]);
    }
  }
}

// The flat form of a program whose Blocks' tiles cover one contiguous run in
// every operand at the same relative positions: c[i] = a[i] op b[i] over the
// run, 512 float4 per workgroup (two per thread, all four loads issued before
// the first use), the last n % 4 elements by the thread whose vector they would
// be.  One Block's work is then spread over several workgroups and one
// workgroup covers parts of several Blocks; both are pure scheduling, since
// Blocks are independent.  Bound by HBM: for C1 (1024 x 1024, 32 x 64 tiles)
// this measured 3.43-3.45 us per launch against 4.05 us for the tiled kernel
// with its Block decode and 32 separate rows per workgroup.  The vectors are
// loaded at element alignment (gfx950 takes unaligned 16-byte accesses), so
// neither the tile's width nor the run's length or start sets the access:
// 18963 x 1020 in 43 x 30 tiles 91.9 -> 37.4 us, which the tiled kernel read a
// float at a time, 875 x 2340 in 35 x 30 12.2 -> 5.4.
template <int OP>
__global__ __launch_bounds__(256) void ew_flat_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                      float* __restrict__ c, long long n) {
  const long long base = (long long)blockIdx.x * 512 + threadIdx.x, nv = n >> 2;
  float4v va[2], vb[2];
  bool ok[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const long long i = base + u * 256;
    ok[u] = i < nv;
    va[u] = ld_nt4(a + 4 * (ok[u] ? i : 0));
    vb[u] = ld_nt4(b + 4 * (ok[u] ? i : 0));
  }
  issue_fence();
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const long long i = base + u * 256;
    float4v vc;
    vc.x = ew_apply<OP>(va[u].x, vb[u].x);
    vc.y = ew_apply<OP>(va[u].y, vb[u].y);
    vc.z = ew_apply<OP>(va[u].z, vb[u].z);
    vc.w = ew_apply<OP>(va[u].w, vb[u].w);
    if (ok[u]) st_nt4(vc, c + 4 * i);
    else if (i == nv)
      for (long long e = 4 * nv; e < n; ++e) c[e] = ew_apply<OP>(a[e], b[e]);
  }
}

struct SoftmaxArgs {
  const float* x;
  float* y;
  TileOff tx, ty;
  long long ldx, ldy;
  int rows, cols;
  long long total;  // rows of all Blocks
  Div31 d_rows;  // by `rows`
  BlockDecode grid;
};

// Row `id` of all Blocks' rows: its first element in x and y.  MANY: more rows
// than one launch's 2^32 threads or 2^31 indices take, so workgroups walk them
// (the walk and its 64-bit division cost an ordinary launch 0.25 us).
template <bool MANY>
__device__ __forceinline__ void softmax_row(const SoftmaxArgs& p, long long id, const float*& xr, float*& yr) {
  const int blk = MANY ? (int)(id / p.rows) : (int)p.d_rows((unsigned)id);
  const int r = (int)(id - (long long)blk * p.rows);
  int x, y, z;
  p.grid(blk, x, y, z);
  xr = p.x + p.tx.at(x, y, z) + r * p.ldx;
  yr = p.y + p.ty.at(x, y, z) + r * p.ldy;
}

// Row reduction across the TPR threads that share a row.  For TPR <= 64 the
// group lies inside one wave and a butterfly suffices; 256 threads combine the
// per-wave partials through LDS with a single barrier (max and sum in slots of
// their own).
template <bool IS_MAX, int TPR>
__device__ __forceinline__ float row_reduce(float v, float* lds) {
  if constexpr (TPR >= 64) {
    v = wave_reduce<IS_MAX>(v);
  } else {
#pragma unroll
    for (int o = TPR >> 1; o > 0; o >>= 1) {
      const float t = __shfl_xor(v, o, 64);
      v = IS_MAX ? fmaxf(v, t) : v + t;
    }
  }
  if constexpr (TPR <= 64) {
    return v;
  } else {
    static_assert(TPR == 256, "a row takes part of a wave, a wave or the workgroup");
    float* slot = lds + (IS_MAX ? 0 : 4);
    if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
    __syncthreads();
    return IS_MAX ? fmaxf(fmaxf(slot[0], slot[1]), fmaxf(slot[2], slot[3])) : (slot[0] + slot[1]) + (slot[2] + slot[3]);
  }
}

// Rows of any length and alignment: TPR threads a row, NV float4 a thread, the
// rows of all Blocks dealt over the grid (Blocks are independent, and so are
// their rows), each thread group taking one.  Bound by HBM, so what counts is
// rows in flight: rows up to 2048 floats take one wave, which needs no barrier,
// and every row of a Block its own wave, where one 256-thread group had walked a
// Block's rows one after another (5000 x 1000, 8 rows a Block: 13.8 -> 8.2 us;
// 7976 x 1674 24.0 -> 20.6; 1152 x 395 5.6 -> 3.1).  Longer rows take the
// workgroup.  Vectors are loaded at element alignment; a row's last cols % 4
// elements are loaded and stored one by one.
template <int NV, int TPR, bool MANY>
__global__ __launch_bounds__(256) void row_softmax_kernel(SoftmaxArgs p) {
  __shared__ float lds[8];
  const int lane = threadIdx.x & (TPR - 1);
  for (long long first = (long long)blockIdx.x * (256 / TPR); first < p.total; first += (long long)gridDim.x * (256 / TPR)) {
    const long long id = first + threadIdx.x / TPR;
    const bool live = id < p.total;  // the whole workgroup's where TPR is 256
    const float* xr;
    float* yr;
    softmax_row<MANY>(p, live ? id : 0, xr, yr);
    float v[NV][4];
    int have[NV];  // elements of the vector inside the row
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int col = (lane + j * TPR) * 4;
      have[j] = live ? min(4, p.cols - col) : 0;
      // absent vectors read the row's first one (of rows up to 8 floats, which
      // may have none, nothing)
      float4v t = {0.f, 0.f, 0.f, 0.f};
      if (TPR > 1 || have[j] == 4) t = ld_nt4(xr + (have[j] == 4 ? col : 0));
      v[j][0] = t.x;
      v[j][1] = t.y;
      v[j][2] = t.z;
      v[j][3] = t.w;
    }
    issue_fence();
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (have[j] < 4 && have[j] > 0)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (k < have[j]) v[j][k] = xr[(lane + j * TPR) * 4 + k];
#pragma unroll
      for (int k = 0; k < 4; ++k) m = k < have[j] ? fmaxf(m, v[j][k]) : m;
    }
    m = row_reduce<true, TPR>(m, lds);
    // a tree within the thread: as a chain of 4 * NV terms the row's sum had the
    // larger error (7.5e-8 of 1000 columns' result against 7.3e-8)
    float part[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[j][k] = k < have[j] ? exp_fast(v[j][k] - m) : 0.0f;
      part[j] = (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
    }
#pragma unroll
    for (int o = 1; o < NV; o *= 2)
#pragma unroll
      for (int j = 0; j + o < NV; j += 2 * o) part[j] += part[j + o];
    const float s = row_reduce<false, TPR>(part[0], lds);
    const float inv = 1.0f / s;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      float* const o = yr + (lane + j * TPR) * 4;
      if (have[j] == 4) {
        st_nt4(float4v{v[j][0] * inv, v[j][1] * inv, v[j][2] * inv, v[j][3] * inv}, o);
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (k < have[j]) st_nt(v[j][k] * inv, o + k);
      }
    }
    if constexpr (!MANY) break;
  }
}

// One row of TPB * NV float4 by a TPB-thread workgroup, from this thread's first
// vector of it.
template <int TPB, int NV>
__device__ __forceinline__ void full_row_softmax(const float4v* __restrict__ xr, float4v* __restrict__ yr) {
  constexpr int NW = TPB / 64;
  __shared__ float lds[2][NW];
  const int w = threadIdx.x >> 6;
  float4v v[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) v[j] = ld_nt(xr + j * TPB);
  issue_fence();
  float m = fmaxf(fmaxf(v[0].x, v[0].y), fmaxf(v[0].z, v[0].w));
#pragma unroll
  for (int j = 1; j < NV; ++j) m = fmaxf(m, fmaxf(fmaxf(v[j].x, v[j].y), fmaxf(v[j].z, v[j].w)));
  m = wave_reduce<true>(m);
  if ((threadIdx.x & 63) == 0) lds[0][w] = m;
  __syncthreads();
  m = lds[0][0];
#pragma unroll
  for (int k = 1; k < NW; ++k) m = fmaxf(m, lds[0][k]);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    v[j].x = exp_fast(v[j].x - m);
    v[j].y = exp_fast(v[j].y - m);
    v[j].z = exp_fast(v[j].z - m);
    v[j].w = exp_fast(v[j].w - m);
    s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  s = wave_reduce<false>(s);
  if ((threadIdx.x & 63) == 0) lds[1][w] = s;
  __syncthreads();
  s = lds[1][0];
#pragma unroll
  for (int k = 1; k < NW; ++k) s += lds[1][k];
  const float inv = 1.0f / s;
#pragma unroll
  for (int j = 0; j < NV; ++j) st_nt(v[j] * inv, yr + j * TPB);
}

// Full-row softmax: a TPB-thread workgroup owns one row, each thread NV float4
// of it (cols == TPB * NV * 4 exactly, row starts 16-byte aligned).  The row's
// loads are one instruction per float4 with compile-time offsets, max/sum are
// trees within the thread, then a wave butterfly, then one LDS exchange across
// the TPB/64 waves.  On gfx950 a 512-thread group with two float4 per thread
// keeps the HBM read/write stream at the rate of a plain device copy for
// 4096-wide rows.
template <int TPB, int NV, bool MANY>
__global__ __launch_bounds__(TPB) void row_softmax_wide_kernel(SoftmaxArgs p) {
  // the max slot and the sum slot are distinct, so each row's barriers also
  // order the reads of one row before the next row's writes
  for (long long id = blockIdx.x; id < p.total; id += gridDim.x) {
    const float* x0;
    float* y0;
    softmax_row<MANY>(p, id, x0, y0);
    full_row_softmax<TPB, NV>(reinterpret_cast<const float4v*>(x0) + threadIdx.x, reinterpret_cast<float4v*>(y0) + threadIdx.x);
    if constexpr (!MANY) break;
  }
}

// The same full-row softmax for the common case of one row per Block on a
// 1-D grid: Block x's row starts x * step float4 vectors past the row of
// Block 0, so the prologue is one multiply-add (no Block decode, no row loop,
// a four-argument kernarg segment).
template <int TPB, int NV>
__global__ __launch_bounds__(TPB) void row_softmax_1d_kernel(const float4v* __restrict__ x, float4v* __restrict__ y,
                                                             long long xstep, long long ystep) {
  full_row_softmax<TPB, NV>(x + blockIdx.x * xstep + threadIdx.x, y + blockIdx.x * ystep + threadIdx.x);
}

TileOff to_off(const xt::TileAddr& a) { return TileOff{a.c0, a.sx, a.sy, a.sz}; }

bool aligned4(const xt::Access2D& a, const void* base) {
  return (reinterpret_cast<uintptr_t>(base) % 16) == 0 && a.ld % 4 == 0 && a.cols % 4 == 0 &&
         a.addr.c0 % 4 == 0 && a.addr.sx % 4 == 0 && a.addr.sy % 4 == 0 && a.addr.sz % 4 == 0;
}

}  // namespace

hipError_t launch_ew_binary(const xt::Plan& p, void* const* bufs, hipStream_t s, std::string& why) {
  EwArgs a;
  a.a = static_cast<const float*>(bufs[p.a.arg]);
  a.b = static_cast<const float*>(bufs[p.b.arg]);
  a.c = static_cast<float*>(bufs[p.c.arg]);
  a.ta = to_off(p.a.addr);
  a.tb = to_off(p.b.addr);
  a.tc = to_off(p.c.addr);
  a.lda = p.a.ld;
  a.ldb = p.b.ld;
  a.ldc = p.c.ld;
  a.rows = static_cast<int>(p.c.rows);
  a.cols = static_cast<int>(p.c.cols);
  if (p.a.rows != p.c.rows || p.b.rows != p.c.rows || p.a.cols != p.c.cols ||
      p.b.cols != p.c.cols) {
    why = "elementwise operand tiles differ in shape";
    return hipErrorInvalidValue;
  }
  const bool vec = aligned4(p.a, a.a) && aligned4(p.b, a.b) && aligned4(p.c, a.c);
  // the run as one stream of vectors; of tiles that are not whole aligned
  // vectors, only where the tiled kernel could take the grid
  auto element = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 4 == 0; };
  const bool flat = p.ew_flat >= 4 && element(a.a) && element(a.b) && element(a.c);
  const bool whole = flat && vec && p.ew_flat % 4 == 0;
  const int vw = vec ? 4 : 1;
  const long long cv = a.cols / vw;
  const long long nvec = static_cast<long long>(a.rows) * cv;
  if (!whole && nvec >= (1LL << 30)) {
    why = "elementwise tile too large";
    return hipErrorInvalidValue;
  }
  a.cv_shift = -1;
  if (cv > 0 && (cv & (cv - 1)) == 0) a.cv_shift = __builtin_ctzll(static_cast<unsigned long long>(cv));
  const int u = nvec <= 256 ? 1 : nvec <= 512 ? 2 : 4;
  const long long sx = p.c.addr.sx < 0 ? -p.c.addr.sx : p.c.addr.sx;
  const long long sy = p.c.addr.sy < 0 ? -p.c.addr.sy : p.c.addr.sy;
  a.grid = block_decode(p.grid[0], p.grid[1], p.grid[1] > 1 && (sx == 0 || (sy != 0 && sy < sx)));
  const long long blocks = grid_blocks(p);
  if (!whole && !grid_fits(blocks, 256)) {
    why = "elementwise grid of " + std::to_string(blocks) + " Blocks exceeds one launch (2^24 workgroups of 256)";
    return hipErrorInvalidValue;
  }
  if (flat) {
    const long long wgs = ((p.ew_flat + 3) / 4 + 511) / 512;  // whole vectors, and one for the rest
    if (!grid_fits(wgs, 256)) {
      why = "elementwise run of " + std::to_string(p.ew_flat) + " elements exceeds one launch";
      return hipErrorInvalidValue;
    }
    const float *fa = a.a + p.a.addr.c0, *fb = a.b + p.b.addr.c0;
    float* fc = a.c + p.c.addr.c0;
    const dim3 grid(static_cast<unsigned>(wgs)), block(256);
    switch (p.ew_op) {
      case xt::EwOp::Add: hipLaunchKernelGGL(ew_flat_kernel<0>, grid, block, 0, s, fa, fb, fc, p.ew_flat); break;
      case xt::EwOp::Sub: hipLaunchKernelGGL(ew_flat_kernel<1>, grid, block, 0, s, fa, fb, fc, p.ew_flat); break;
      default: hipLaunchKernelGGL(ew_flat_kernel<2>, grid, block, 0, s, fa, fb, fc, p.ew_flat); break;
    }
    return hipGetLastError();
  }
  dim3 grid(static_cast<unsigned>(blocks)), block(256);
  const int op = static_cast<int>(p.ew_op);
  const bool pow2 = a.cv_shift >= 0;
  // kernel variant index: op (3) x vector width (2) x U (3) x pow2 (2)
#define XT_EW(OPV, VWV, UV, P2) \
  hipLaunchKernelGGL((ew_binary_kernel<OPV, VWV, UV, P2>), grid, block, 0, s, a)
#define XT_EW_P2(OPV, VWV, UV) \
  do { if (pow2) XT_EW(OPV, VWV, UV, true); else XT_EW(OPV, VWV, UV, false); } while (0)
#define XT_EW_U(OPV, VWV)                \
  do {                                   \
    if (u == 1) XT_EW_P2(OPV, VWV, 1);   \
    else if (u == 2) XT_EW_P2(OPV, VWV, 2); \
    else XT_EW_P2(OPV, VWV, 4);          \
  } while (0)
#define XT_EW_OP(VWV)                  \
  do {                                 \
    if (op == 0) XT_EW_U(0, VWV);      \
    else if (op == 1) XT_EW_U(1, VWV); \
    else XT_EW_U(2, VWV);              \
  } while (0)
  if (vw == 4) XT_EW_OP(4);
  else XT_EW_OP(1);
#undef XT_EW_OP
#undef XT_EW_U
#undef XT_EW_P2
#undef XT_EW
  return hipGetLastError();
}

hipError_t launch_row_softmax(const xt::Plan& p, void* const* bufs, hipStream_t s,
                              std::string& why) {
  SoftmaxArgs a;
  a.x = static_cast<const float*>(bufs[p.a.arg]);
  a.y = static_cast<float*>(bufs[p.c.arg]);
  a.tx = to_off(p.a.addr);
  a.ty = to_off(p.c.addr);
  a.ldx = p.a.ld;
  a.ldy = p.c.ld;
  a.rows = static_cast<int>(p.a.rows);
  a.cols = static_cast<int>(p.a.cols);
  a.grid = block_decode(p.grid[0], p.grid[1], false);
  if (p.c.rows != p.a.rows || p.c.cols != p.a.cols) {
    why = "softmax input and output tiles differ in shape";
    return hipErrorInvalidValue;
  }
  const bool vec = aligned4(p.a, a.x) && aligned4(p.c, a.y);
  const long long blocks = grid_blocks(p), total = blocks * a.rows;
  const bool wide = vec && a.cols % 2048 == 0 && a.cols <= 8 * 2048;
  // threads a row: a power of two up to a wave for rows up to 2048 floats, else,
  // and where there are so few that a wave's eight float4 are latency (64 x 2000
  // 4.0 us a wave each, 3.7 a workgroup; 1024 x 2000 5.0 either way; to 1024
  // floats no different), the workgroup; two float4 a thread where that makes it less than a wave and
  // there are rows to fill the chip all the same (100000 x 100: 43.7 -> 17.0 us;
  // 64 x 256 2.5 with two, 2.3 with one)
  int tpr = 256;
  if (a.cols <= 1024 || (a.cols <= 2048 && total > 512))
    for (tpr = 1; tpr < 64 && tpr * (total > 4096 ? 8 : 4) < a.cols; tpr *= 2) {
    }
  const int threads = wide ? 512 : 256;
  if (!grid_fits(blocks, threads)) {
    why = "softmax grid of " + std::to_string(blocks) + " Blocks exceeds one launch";
    return hipErrorInvalidValue;
  }
  const long long most = (1LL << 32) / threads - 1;
  const long long need = wide ? total : (total + 256 / tpr - 1) / (256 / tpr), wgs = std::min(need, most);
  const bool many = need > most || total >= (1LL << 31);
  a.total = total;
  a.d_rows = div31(static_cast<unsigned>(a.rows));
  dim3 grid(static_cast<unsigned>(wgs));
  if (wide && a.rows == 1 && p.grid[1] == 1 && p.grid[2] == 1) {
    // one row per Block on a 1-D grid (aligned4 makes every offset a float4 multiple)
    const float4v* x4 = reinterpret_cast<const float4v*>(a.x + p.a.addr.c0);
    float4v* y4 = reinterpret_cast<float4v*>(a.y + p.c.addr.c0);
    const long long xs = p.a.addr.sx / 4, ys = p.c.addr.sx / 4;
    switch (a.cols / 2048) {
#define XT_SM1(NVV) \
  case NVV: hipLaunchKernelGGL((row_softmax_1d_kernel<512, NVV>), grid, dim3(512), 0, s, x4, y4, xs, ys); break
      XT_SM1(1); XT_SM1(2); XT_SM1(3); XT_SM1(4); XT_SM1(5); XT_SM1(6); XT_SM1(7); XT_SM1(8);
#undef XT_SM1
    }
    return hipGetLastError();
  }
  if (wide) {
    switch (a.cols / 2048) {
#define XT_SMW(NVV)                                                                                             \
  case NVV:                                                                                                    \
    if (many) hipLaunchKernelGGL((row_softmax_wide_kernel<512, NVV, true>), grid, dim3(512), 0, s, a);         \
    else hipLaunchKernelGGL((row_softmax_wide_kernel<512, NVV, false>), grid, dim3(512), 0, s, a);             \
    break
      XT_SMW(1); XT_SMW(2); XT_SMW(3); XT_SMW(4); XT_SMW(5); XT_SMW(6); XT_SMW(7); XT_SMW(8);
#undef XT_SMW
    }
    return hipGetLastError();
  }
  const int nv = (a.cols + 4 * tpr - 1) / (4 * tpr);
  dim3 block(256);
#define XT_SM(NVV, TPRV)                                                                            \
  do {                                                                                              \
    if (many) hipLaunchKernelGGL((row_softmax_kernel<NVV, TPRV, true>), grid, block, 0, s, a);      \
    else hipLaunchKernelGGL((row_softmax_kernel<NVV, TPRV, false>), grid, block, 0, s, a);          \
  } while (0)
#define XT_SM_NV(TPRV)             \
  switch (nv) {                    \
    case 1: XT_SM(1, TPRV); break; \
    case 2: XT_SM(2, TPRV); break; \
    case 3: XT_SM(3, TPRV); break; \
    case 4: XT_SM(4, TPRV); break; \
    case 5: XT_SM(5, TPRV); break; \
    case 6: XT_SM(6, TPRV); break; \
    case 7: XT_SM(7, TPRV); break; \
    default: XT_SM(8, TPRV); break; \
  }
#define XT_SM_SUB(TPRV)            \
  if (nv == 1) XT_SM(1, TPRV);     \
  else XT_SM(2, TPRV)
  switch (tpr) {
    case 1: XT_SM_SUB(1); break;
    case 2: XT_SM_SUB(2); break;
    case 4: XT_SM_SUB(4); break;
    case 8: XT_SM_SUB(8); break;
    case 16: XT_SM_SUB(16); break;
    case 32: XT_SM_SUB(32); break;
    case 64: XT_SM_NV(64); break;
    default: XT_SM_NV(256); break;
  }
#undef XT_SM_SUB
#undef XT_SM_NV
#undef XT_SM
  return hipGetLastError();
}

}  // namespace xtk
