// conv(1x1) -> cast|relu -> conv(3x3, stride 1, pad 1) with at most 64 channels everywhere on NCHW tensors, fp16 / bf16: tiles of
// whole output rows, any image width from 8 pixels on, weights as MFMA fragments straight from L2.
//
// For the shapes the row pipeline (conv_rows.h) does not take: image rows that are no multiple of 8 pixels ran on the general
// kernel (six stages of W2 through LDS, two-byte loads and stores; 18 us whatever the batch), rows of more than 64 pixels on the
// persistent kernel (conv_chain_resident.h), whose workgroups first fetch 72 KB of W2 each and then sit one to a compute unit.
// A workgroup here owns TH whole output rows of one image and all channels:
//   - halo rows of X into LDS, channel fastest (stage_halo_rows, as in conv_tiles.h);
//   - the first convolution IN PLACE: a wave reads the input channels of 16 pixels, one or two MFMA steps by four channel
//     tiles, and writes the 64 intermediate channels where the pixel's input was: no second buffer, and no barrier among them;
//   - the second convolution straight from there, 18 steps unrolled, pixel fragments one step and weight fragments four steps
//     ahead; 72-element pixels put the 16 pixels of a fragment on all 64 banks for any tap;
//   - the output through LDS once, so that a channel's run of pixels leaves in 16-byte stores at element alignment.
// Two waves split the output channels and two or four pairs the pixels: every fragment, of either kind, feeds at least two
// MFMAs.
//
// Bound: load, compute and store phases one after the other, overlapped only by the other workgroups of the compute unit
// (49 KB of LDS each at 112 pixels).  Measured, us per launch with prepared weights (2.4 of them the launch), before -> here:
// 32 x 64 x 20 x 20 -> 64 -> 64 24.4 -> 5.4, 4 x 64 x 46 x 46 19.5 -> 5.9, 8 x 64 x 99 x 99 34.9 -> 17.0, 32 x 64 x 99 x 99
// 107 -> 51, 8 x 64 x 112 x 112 20.3 -> 15.2 (three times the input rows are fetched with one output row per workgroup,
// twice with two).
#pragma once
#include "conv_tiles.h"

namespace ditto {

struct Conv13TilesArgs {
  const void* x;
  const void* w1f;  // W1 as fragments: [k step][4 tiles][64 lanes][8]
  const void* w2f;  // W2 as fragments: [half of the output channels][tap, k step][2 tiles][64 lanes][8]
  void* y;
  int N, C0, H, W, C1, C2;
  int TH, tiles_h;  // output rows per workgroup, workgroups per image
  int wp;           // pairs of waves of a workgroup
  int c0p;          // input channels padded to 32 or 64
  int relu_mid, relu_out, out_f32;
  float inv_cg, inv_ng, inv_w;  // 8 / c0p, 1 / ceil(W / 8), 1 / W
};

constexpr int kC13Stride = conv_tiles_stride(64);  // elements per pixel in LDS, of X and of the intermediate image alike
constexpr int kC13Taps = 9, kC13Steps = 2 * kC13Taps;
constexpr int kC13W1Bytes = 2 * 4 * 1024, kC13W2Bytes = kC13Steps * 4 * 1024;
constexpr int kC13Pairs = 4;  // most pairs of waves
inline int conv13_tiles_slots(int wp) { return 64 * wp; }
inline int conv13_tiles_lds_bytes(int TH, int W, int wp) {
  const int x = (TH + 2) * (W + 2) * kC13Stride * 2, out = 64 * (conv13_tiles_slots(wp) + 8) * 2;
  return x > out ? x : out;
}

// 2 x WP waves: two split the output channels, WP the pixels (PT tiles of 16 each).
template <typename T, int WP, int PT>
__global__ __launch_bounds__(128 * WP) void conv13_tiles_kernel(Conv13TilesArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Elem<T>::v8 V8;
  typedef typename Elem<T>::v4 V4;
  constexpr int NW = 2 * WP, NT = 64 * NW, CS = kC13Stride, OS = 64 * WP + 8, D = 4;
  extern __shared__ __attribute__((aligned(16))) char smem_13[];
  T* const Xs = reinterpret_cast<T*>(smem_13);  // [TH + 2][W + 2][CS]: X, then the intermediate image in its place, then the output
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave & 1, wp = wave >> 1;
  const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
  const int n = lid / (unsigned)p.tiles_h, p0 = (lid - n * (unsigned)p.tiles_h) * p.TH;
  const int W = p.W, cols = W + 2, rows = p.TH + 2, npx = min(p.TH, p.H - p0) * W;
  const long long hw = (long long)p.H * W;
  const int npm = rows * W, in0 = p0 == 0 ? W : 0, in1 = min(npm, (p.H - p0 + 1) * W);  // halo pixels, those inside the image

  V8 w1[2][4];
  const T* const w1f = reinterpret_cast<const T*>(p.w1f);
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int m = 0; m < 4; ++m) w1[k][m] = *reinterpret_cast<const V8*>(w1f + ((32 * k < p.c0p ? k : 0) * 4 + m) * 512 + lane * 8);

  stage_halo_rows<NT>(Xs, reinterpret_cast<const T*>(p.x) + (long long)n * p.C0 * hw, p0 - 1, 1, rows, cols, CS, p.c0p / 8, 8, p.C0, p.H, W,
                      p.inv_cg, p.inv_ng, tid);
  if (p.c0p < 64)  // of the rows outside the image: the channels beyond the staged zeros
    for (int t = tid; t < 4 * (in0 + npm - in1); t += NT) {
      const int slot = t / 4 < in0 ? t / 4 : in1 - in0 + t / 4, ri = div_by(slot, p.inv_w);
      *reinterpret_cast<i32x4*>(Xs + (ri * cols + slot - ri * W + 1) * CS + 32 + 8 * (t & 3)) = i32x4{0, 0, 0, 0};
    }
  const T* const w2 = reinterpret_cast<const T*>(p.w2f) + (size_t)wc * (kC13Steps * 2 * 512) + lane * 8;
  V8 wf[D][2];
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int m = 0; m < 2; ++m) wf[d][m] = *reinterpret_cast<const V8*>(w2 + (2 * d + m) * 512);
  wg_sync();

  // ---- first convolution, in place: a wave turns the input channels of its 16 pixels into their 64 intermediate ones.  A row
  // outside the image stays zero whatever the weights: only the pixels of the rows inside are computed.
  for (int s0 = in0 + 16 * wave; s0 < in1; s0 += 16 * NW) {
    const int slot = s0 + c < in1 ? s0 + c : in0, ri = div_by(slot, p.inv_w);
    T* const px = Xs + (ri * cols + slot - ri * W + 1) * CS;
    f32x4 acc[4];
    const V8 x0 = *reinterpret_cast<const V8*>(px + 8 * q);
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = Elem<T>::mfma16(w1[0][m], x0, f32x4{0.f, 0.f, 0.f, 0.f});
    if (p.c0p > 32) {
      const V8 x1 = *reinterpret_cast<const V8*>(px + 32 + 8 * q);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m] = Elem<T>::mfma16(w1[1][m], x1, acc[m]);
    }
    if (s0 + c < in1) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (p.relu_mid)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][r] = fmaxf(acc[m][r], 0.f);
        const typename Elem<T>::v2 lo = cvt2<T>(acc[m][0], acc[m][1]), hi = cvt2<T>(acc[m][2], acc[m][3]);
        const V4 v = {lo[0], lo[1], hi[0], hi[1]}, none = {0, 0, 0, 0};
        *reinterpret_cast<V4*>(px + 16 * m + 4 * q) = 16 * m + 4 * q < p.C1 ? v : none;  // (an infinite input has no part beyond C1)
      }
    }
  }
  wg_sync();

  // ---- second convolution, MFMA row = pixel, column = output channel: step = tap, 32 intermediate channels
  int xb[PT];
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    int slot = 16 * (wp * PT + t) + c;
    slot = slot < npx ? slot : 0;
    const int ph = div_by(slot, p.inv_w);
    xb[t] = (ph * cols + slot - ph * W) * CS + 8 * q;
  }
  f32x4 acc[2][PT];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < PT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  V8 xf[2][PT];
  auto load_x = [&](int b, int st) __attribute__((always_inline)) {
    const int tap = st >> 1, off = (tap / 3 * cols + tap % 3) * CS + 32 * (st & 1);
#pragma unroll
    for (int t = 0; t < PT; ++t) xf[b][t] = *reinterpret_cast<const V8*>(Xs + xb[t] + off);
  };
  load_x(0, 0);
#pragma unroll
  for (int st = 0; st < kC13Steps; ++st) {
    if (st + 1 < kC13Steps) load_x((st + 1) & 1, st + 1);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int t = 0; t < PT; ++t) acc[m][t] = Elem<T>::mfma16(xf[st & 1][t], wf[st % D][m], acc[m][t]);
    if (st + D < kC13Steps)
#pragma unroll
      for (int m = 0; m < 2; ++m) wf[st % D][m] = *reinterpret_cast<const V8*>(w2 + (2 * (st + D) + m) * 512);
    __builtin_amdgcn_sched_barrier(0);  // one step of reads ahead, not all of them (registers)
  }

  T* const yt = reinterpret_cast<T*>(p.y) + (long long)n * p.C2 * hw + (long long)p0 * W;
  if (p.out_f32) {  // a lane's four pixels of a channel from the registers
    float* const yf = reinterpret_cast<float*>(p.y) + (long long)n * p.C2 * hw + (long long)p0 * W;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c2 = 32 * wc + 16 * m + c, px = 16 * (wp * PT + t) + 4 * q + r;
          if (c2 < p.C2 && px < npx) yf[c2 * hw + px] = p.relu_out ? fmaxf(acc[m][t][r], 0.f) : acc[m][t][r];
        }
    return;
  }
  // ---- the output turns around in LDS, [channel][pixel], and leaves as one run of pixels per channel
  wg_sync();
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < PT; ++t) {
      f32x4 v = acc[m][t];
      if (p.relu_out)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f);
      const typename Elem<T>::v2 lo = cvt2<T>(v[0], v[1]), hi = cvt2<T>(v[2], v[3]);
      *reinterpret_cast<V4*>(Xs + (32 * wc + 16 * m + c) * OS + 16 * (wp * PT + t) + 4 * q) = V4{lo[0], lo[1], hi[0], hi[1]};
    }
  wg_sync();
  typedef __attribute__((ext_vector_type(8), aligned(2))) T V8u;  // 16 bytes at any element's address
  const int nv = (npx + 7) / 8;
  const float inv_nv = 1.f / (float)nv;
  auto store = [&](auto ragged) __attribute__((always_inline)) {
    for (int i = tid; i < p.C2 * nv; i += NT) {
      const int c2 = div_by(i, inv_nv), v = 8 * (i - c2 * nv);
      const T* const src = Xs + c2 * OS + v;
      T* const dst = yt + c2 * hw + v;
      const V8 o = *reinterpret_cast<const V8*>(src);
      if (decltype(ragged)::value == 0 || v + 8 <= npx) *reinterpret_cast<V8u*>(dst) = o;
      else store_some(dst, o, npx - v);
    }
  };
  // (rows of whole vectors pay 0.1 us for the test of their ends)
  if ((npx & 7) == 0) store(CtInt<0>());
  else store(CtInt<1>());
#else
  (void)p;
#endif
}

template <typename T, int WP, int PT>
hipError_t launch_conv13_tiles_as(const Conv13TilesArgs& a, hipStream_t stream) {
  auto kern = conv13_tiles_kernel<T, WP, PT>;
  static thread_local int configured_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)a.N * (unsigned)a.tiles_h), dim3(128 * WP), conv13_tiles_lds_bytes(a.TH, a.W, WP), stream, a);
  return hipGetLastError();
}
template <typename T, int WP>
hipError_t launch_conv13_tiles_rows(const Conv13TilesArgs& a, hipStream_t stream) {
  switch ((a.TH * a.W + 16 * WP - 1) / (16 * WP)) {
    case 1: return launch_conv13_tiles_as<T, WP, 1>(a, stream);
    case 2: return launch_conv13_tiles_as<T, WP, 2>(a, stream);
    case 3: return launch_conv13_tiles_as<T, WP, 3>(a, stream);
    case 4: return launch_conv13_tiles_as<T, WP, 4>(a, stream);
  }
  return hipErrorInvalidValue;
}
template <typename T>
hipError_t launch_conv13_tiles(const Conv13TilesArgs& a, hipStream_t stream) {
  return a.wp == 2 ? launch_conv13_tiles_rows<T, 2>(a, stream) : a.wp == 4 ? launch_conv13_tiles_rows<T, 4>(a, stream) : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_pack_conv13_tiles(const Conv13TilesArgs& a, const void* w1, const void* w2, void* w1f, void* w2f, hipStream_t stream) {
  const ConvFragments f1 = {w1, w1f, a.C1, a.C0, a.c0p, 1, 4, (unsigned)(a.c0p / 32 * 4 * 512)};
  const ConvFragments f2 = {w2, w2f, a.C2, a.C1, 64, kC13Taps, 2, (unsigned)(kC13W2Bytes / 2)};
  const unsigned blocks1 = (f1.total + 255) / 256, blocks2 = (f2.total + 255) / 256;
  hipLaunchKernelGGL(pack_conv_fragments_kernel<T>, dim3(blocks1 + blocks2), dim3(256), 0, stream, f1, f2, blocks1);
  return hipGetLastError();
}

}  // namespace ditto
