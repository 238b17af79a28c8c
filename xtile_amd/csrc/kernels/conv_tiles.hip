// xt.load_conv2d as an implicit GEMM of 64 x 64 to 32 x 32 tiles: the path for
// launches whose larger tiles (conv_igemm.hip) leave most CUs without one -
// single images, small layers, few output channels.
//
// Semantics and conditions are conv_igemm.hip's: M = images * OH * OW output
// pixels, N = Cout, K = KH * KW * Cin in the filter's (kh, kw, c) order.
//
// What bounds such a launch is latency: one workgroup's operands at what one CU
// can fetch (gemm_small.hip).  So it is that kernel's loop - four waves split K,
// each with a ring of its own, no barrier until the partial tiles meet - with
// A's rows gathered by the DMA: K is counted in 16-byte chunks (tap, channels),
// each lane fetches one chunk position of every stage, finds that chunk's tap
// with two multiplications and each of its pixel rows' source position at the
// tap (zeros outside the image).  Chunks run through the taps without padding,
// so few channels cost no idle stages.  Sums are in a fixed order and, for i8,
// exact.
//
// PART (i8 with Cin a multiple of 4 but not of 16): a tap's last chunk starts
// 16 bytes before its last channel's end, so every chunk lies inside its pixel;
// the filter rows of the channels it shares with the chunk before are zeros
// (whole numbers: a product with zero adds nothing).
#include "launch.h"
#include "small_tile.h"

namespace xtk {
namespace {

constexpr unsigned kCtOutOfRange = 0x80000000u;  // the input and the filter are < 2 GiB

struct CtArgs {
  const unsigned char* src;   // NHWC input
  const unsigned char* filt;  // [K][CO]
  float* out;                 // [M][CO]
  unsigned src_bytes, filt_bytes;
  int H, W, C, KW, CO, K;
  int OW, OHW;
  int pad_t, pad_l, sh, sw, dh, dw;
  int M;
  int chunks;  // 16-byte chunks of K: KH * KW * cc
  int cc;      // chunks a tap: C * esize / 16, rounded up
  int ntiles;  // channel tiles
  int nwg;
  Div31 d_ohw, d_ow, d_nt, d_cc, d_kw;
};

template <int ELEM, int BM, int BN, bool PART>
__global__ __launch_bounds__(256, 1) void conv_tiles_kernel(CtArgs p) {
  typedef SmallTile<ELEM, BM, BN> T;
  constexpr int ES = T::ES, AB = T::AB, KR = T::KR, PA = T::PA, RPI = T::RPI;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[T::LDS];
  // neighbouring tiles share input rows and filter columns: contiguous runs per XCD
  const int L = xcd_contiguous(blockIdx.x, p.nwg);
  const int mt = p.d_nt(L), m0 = mt * BM, n0 = (L - mt * p.ntiles) * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const i32x4 ra = raw_rsrc(p.src, p.src_bytes), rb = raw_rsrc(p.filt, p.filt_bytes);

  // this lane's pixel rows 8 i + lane / 8: source origin of the window, and its
  // byte offset (valid taps bring the sum inside the image)
  int ih0[PA], iw0[PA];
  unsigned base[PA];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int pix = m0 + 8 * i + (lane >> 3);
    const int n = p.d_ohw(min(pix, p.M - 1)), rem = min(pix, p.M - 1) - n * p.OHW;
    const int oh = p.d_ow(rem), ow = rem - oh * p.OW;
    ih0[i] = pix < p.M ? oh * p.sh - p.pad_t : -(1 << 30);  // past M: never inside the image
    iw0[i] = ow * p.sw - p.pad_l;
    base[i] = (unsigned)(((n * p.H + oh * p.sh - p.pad_t) * p.W + iw0[i]) * p.C) * (unsigned)ES;
  }
  const unsigned ldb = (unsigned)(p.CO * ES);
  const int brow = lane / T::CPR, bch = T::b_chunk(lane);
  const bool bin = n0 * ES + bch * 16 < p.CO * ES;
  const unsigned vcol = (unsigned)(n0 * ES) + (unsigned)bch * 16, vb = (unsigned)brow * ldb + vcol;

  T t4;
  t4.begin(lane);
  const int ns = (p.chunks + 7) >> 3, mine = (ns - wave + 3) >> 2;
  // the two chunk positions of this lane (even and odd instructions) at the
  // stage being issued: byte offset and rows, columns of the tap, from the origin
  unsigned toff[2];
  int dih[2], diw[2];
  t4.run(lds + wave * T::RING, mine, [&](int q, unsigned at, int i) {
    const int s = 4 * q + wave;
    if (i == 0)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int k = 8 * s + T::a_chunk(lane, e);
        const int tap = p.d_cc(k), kh = p.d_kw(tap), kw = tap - kh * p.KW;
        dih[e] = k < p.chunks ? kh * p.dh : 1 << 29;  // past K: outside every image, rows past M included
        diw[e] = kw * p.dw;
        const int c16 = (k - tap * p.cc) * 16;
        toff[e] = (unsigned)((kh * p.dh * p.W + diw[e]) * p.C * ES + (PART ? min(c16, p.C - 16) : c16));
      }
    if (i < PA) {
      const bool in = ((unsigned)(ih0[i] + dih[i & 1]) < (unsigned)p.H) & ((unsigned)(iw0[i] + diw[i & 1]) < (unsigned)p.W);
      dma16(ra, at + i * 1024, in ? base[i] + toff[i & 1] : kCtOutOfRange, 0);
    } else {
      const int k = s * KR + RPI * (i - PA);
      if constexpr (PART) {
        const int chunk = (k + brow) >> 4, tap = p.d_cc(chunk), c16 = (chunk - tap * p.cc) * 16;
        const int ch = min(c16, p.C - 16) + ((k + brow) & 15);
        const bool in = bin & (chunk < p.chunks) & (ch >= c16);
        dma16(rb, at + AB + (i - PA) * 1024, in ? (unsigned)(tap * p.C + ch) * ldb + vcol : kCtOutOfRange, 0);
      } else
        dma16(rb, at + AB + (i - PA) * 1024, bin & (k + brow < p.K) ? vb + (unsigned)k * ldb : kCtOutOfRange, 0);
    }
  });
  t4.finish(lds, wave, [&](int m, int n, typename T::num4 x) {
    // Cout is a multiple of 8 (16-byte filter rows): four channels are in or out together
    if (m0 + m < p.M && n0 + n < p.CO)
      *reinterpret_cast<float4v*>(p.out + (long long)(m0 + m) * p.CO + n0 + n) =
          float4v{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
  });
}

template <int ELEM, bool PART = false>
void launch_tiles(int bm, int bn, const CtArgs& a, hipStream_t s) {
  const dim3 grid(a.nwg), block(256);
  if (bm == 64) hipLaunchKernelGGL((conv_tiles_kernel<ELEM, 64, 64, PART>), grid, block, 0, s, a);
  else if (bn == 64) hipLaunchKernelGGL((conv_tiles_kernel<ELEM, 32, 64, PART>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((conv_tiles_kernel<ELEM, 32, 32, PART>), grid, block, 0, s, a);
}

}  // namespace

bool run_conv_tiles(const xt::Plan& p, void* const* bufs, long long images, int bm, int bn, hipStream_t s, hipError_t& e) {
  const xt::ConvPlan& c = p.conv;
  const int es = c.elem == xt::Elem::I8 ? 1 : 2;
  const long long M = images * c.out_H * c.out_W, K = c.KH * c.KW * c.C;
  CtArgs a;
  a.src = static_cast<const unsigned char*>(bufs[c.src_arg]);
  a.filt = static_cast<const unsigned char*>(bufs[c.filt_arg]) + c.filt_addr.c0 * es;
  a.out = static_cast<float*>(bufs[c.out_arg]);
  a.src_bytes = static_cast<unsigned>(images * c.H * c.W * c.C * es);
  a.filt_bytes = static_cast<unsigned>(K * c.CO * es);
  a.H = (int)c.H;
  a.W = (int)c.W;
  a.C = (int)c.C;
  a.KW = (int)c.KW;
  a.CO = (int)c.CO;
  a.K = (int)K;
  a.OW = (int)c.out_W;
  a.OHW = (int)(c.out_H * c.out_W);
  a.pad_t = (int)c.pad_top;
  a.pad_l = (int)c.pad_left;
  a.sh = (int)c.stride_h;
  a.sw = (int)c.stride_w;
  a.dh = (int)c.dil_h;
  a.dw = (int)c.dil_w;
  a.M = (int)M;
  a.cc = (int)((c.C * es + 15) / 16);
  a.chunks = (int)(c.KH * c.KW) * a.cc;
  a.ntiles = (int)((c.CO + bn - 1) / bn);
  const long long nwg = (M + bm - 1) / bm * a.ntiles;
  if (!grid_fits(nwg, 256)) return false;
  a.nwg = (int)nwg;
  a.d_ohw = div31((unsigned)a.OHW);
  a.d_ow = div31((unsigned)a.OW);
  a.d_nt = div31((unsigned)a.ntiles);
  a.d_cc = div31((unsigned)a.cc);
  a.d_kw = div31((unsigned)a.KW);
  switch (c.elem) {
    case xt::Elem::I8: c.C % 16 ? launch_tiles<kI8, true>(bm, bn, a, s) : launch_tiles<kI8>(bm, bn, a, s); break;
    case xt::Elem::BF16: launch_tiles<kBF16>(bm, bn, a, s); break;
    default: launch_tiles<kF16>(bm, bn, a, s); break;
  }
  e = hipGetLastError();
  return true;
}

}  // namespace xtk
