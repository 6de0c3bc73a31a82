// conv(RxS, any stride) -> cast|relu -> conv(1x1) on NCHW tensors, fp16 / bf16: tiles of whole output rows, any image
// width from 8 pixels on, weights as MFMA fragments straight from L2.
//
// For the shapes the general kernel (conv_chain.h) is bad at: it stages halo tile and weights through LDS in chunks of 32
// channels, four barriers and two exposed memory latencies each, computes 256 pixel slots whatever the tile holds, reads
// image rows that are not whole 16-byte vectors two bytes at a time, and stores two bytes at a time where a tile is not a
// run of such rows.  A workgroup here
//   - owns TH whole output rows (at most 128 pixels) of one image and all channels: one contiguous run of every channel plane;
//   - stages the halo rows of ALL input channels once, with 16-byte loads at element alignment (the hardware takes them at
//     any address) and an 8x8 transposition in registers;
//   - runs the first convolution without a barrier: W1 comes as ready fragments, 1 KB per wave and instruction, each by the
//     one wave (or two, see conv_tiles_split) that owns those channels, four k steps ahead;
//   - puts the cast result into LDS once and takes the second convolution's pixels in the order PO j + t (column j of tile t),
//     which leaves a lane with 8 consecutive pixels of 4 channels: 16-byte stores, 256 contiguous bytes per 16 lanes.
// Three barriers in all; several workgroups share a compute unit and cover one another's loads.
//
// Bound: for few pixels the stream of W1 through one compute unit (64 bytes per clock), otherwise load, compute and
// store phases one after the other, which only other workgroups on the compute unit overlap.  Measured, us per launch with
// prepared weights, general kernel -> this one: 8 x 32 x 147 x 147 stride 2 -> 64 -> 80 21.5 -> 9.8 (2.4 of them
// the launch); one image 128 x 28 x 28 -> 256 -> 128 45.6 -> 9.2 (28 compute units, each streaming 590 KB of W1);
// 21 x 64 x 106 x 106 stride 2 -> 192 -> 128 109 -> 31 (520 TFLOP/s); 32 x 128 x 28 x 28 -> 256 -> 128 46 -> 20.5 (800 TFLOP/s);
// 32 x 256 x 56 x 56 1x1 -> 256 -> 64 83 -> 31.  Tried and left out: columns kept by remainder modulo the stride, so that a
// strided tap reads neighbouring pixels without bank conflicts (level at 147 x 147, 0.3 us slower on small images: the
// index arithmetic); W2 fragments fetched ahead of the first convolution (level).
#pragma once
#include "common.h"

namespace ditto {

struct ConvTilesArgs {
  const void* x;
  const void* w1f;  // W1 as fragments (pack_conv_fragments): [wave][k step][tile of the wave][64 lanes][8]
  const void* w2f;  // W2 as fragments: [output tile][k step][64 lanes][8]
  void* y;
  int N, C0, H, W, C1, C2;
  int R, S, pad, stride;
  int P, Q;           // output extent
  int TH, tiles_h;    // output rows per workgroup, workgroups per image
  int rows_in, cols_in;  // halo rows and columns of a full tile
  int c0p;               // input channels padded to 32
  int relu_mid, relu_out, out_f32;
  float inv_cg, inv_ng, inv_q;  // 1 / (c0p / 8), 1 / ceil(W / 8), 1 / Q
};

template <int V>
struct CtInt {
  static constexpr int value = V;
};

constexpr int kCtMaxTiles = 8;  // tiles of 16 output pixels per workgroup

// element stride of a pixel's channel vector in LDS: the 8 elements beyond the channels spread consecutive pixels over
// the banks
__host__ __device__ constexpr int conv_tiles_stride(int channels) { return channels + 8; }
// Elements between the intermediate pixels of one lane of the second convolution, `po` of them, and the next lane's.  A 16-byte read of
// lanes (pixels c, 16-byte chunk q) takes 4 cycles where the lanes' pixels lie an odd multiple of 32 bytes apart, 8 at odd multiples of 16
// or 64 bytes and 16 at odd multiples of 128 (measured, eight waves at once), which is where eight pixels of an odd number of 16-byte
// chunks put them.  us per launch without / with the gap: 8 x 32 x 147 x 147 stride 2 -> 64 -> 80 10.75 / 9.83, 4 x 256 x 112 x 112 1x1 -> 256 -> 64
// 16.2 / 13.4, 4 x 128 x 93 x 93 -> 256 -> 128 34.8 / 28.6; over 230 random calls 0.87 - 0.97 by channels at five pixel tiles a workgroup
// and more, level below.  (16 elements behind the channels of the halo pixels, for the first convolution's reads, changed nothing
// beyond that: 1x1 -> 3x3 1.00, whose pixels are written as often as read.)
__host__ __device__ constexpr int conv_tiles_gap(int po) { return po == 2 ? 0 : 16; }
__host__ __device__ inline int conv_tiles_lds_bytes(int rows_in, int cols_in, int c0p, int c1p, int slots) {  // slots: 16 po
  const int x = rows_in * cols_in * conv_tiles_stride(c0p) * 2, mid = (slots * conv_tiles_stride(c1p) + 16 * conv_tiles_gap(slots / 16)) * 2;
  return x > mid ? x : mid;
}

// Both weight tensors in one launch, each W[rows][cols][taps] -> [group of `per` row tiles][k step][tile][lane][8], zero padded: element e of lane l of tile t
// is row 16 t + l % 16, column 32 (step % (colsp / 32)) + 8 (l / 16) + e, tap step / (colsp / 32)
struct ConvFragments {
  const void* w;
  void* out;
  int rows, cols, colsp, taps, per;
  unsigned total;  // elements of `out`
};
template <typename T>
__global__ void pack_conv_fragments_kernel(ConvFragments w1, ConvFragments w2, unsigned blocks1) {
  const bool first = blockIdx.x < blocks1;
  const ConvFragments& a = first ? w1 : w2;
  const unsigned i = (blockIdx.x - (first ? 0 : blocks1)) * blockDim.x + threadIdx.x;
  if (i >= a.total) return;
  const int e = i & 7, l = (i >> 3) & 63;
  const unsigned f = i >> 9;
  const int cb = a.colsp / 32, steps = a.taps * cb;
  const int m = f % (unsigned)a.per, step = f / (unsigned)a.per % (unsigned)steps, grp = f / (unsigned)a.per / (unsigned)steps;
  const int row = 16 * (grp * a.per + m) + (l & 15), col = 32 * (step % cb) + 8 * (l >> 4) + e, tap = step / cb;
  static_cast<T*>(a.out)[i] =
      row < a.rows && col < a.cols ? static_cast<const T*>(a.w)[((long long)row * a.cols + col) * a.taps + tap] : (T)0.f;
}

// Halo rows of one image into LDS, channel fastest: [rows_in][cols_in][CHS], image column 0 at column `pad`.  A task is 8 pixels
// x 8 channels of one image row: eight 16-byte loads (at element alignment: rows of any length), an 8x8 transposition in
// registers, eight 16-byte writes.  The last group of a row starts at W - 8 and repeats pixels of the one before it.  Two
// tasks of a thread are in flight together.
// Neighbouring lanes take neighbouring pixels: the address unit takes four lanes at a time and spends a cycle on every line
// they touch, so four lanes on four channels' planes cost it four times what four lanes on 64 contiguous bytes do.  Where rows
// are whole 16-byte vectors lanes 2 i, 2 i + 1 are neighbours and a group of eight lanes writes eight different 16-byte columns of
// the LDS banks; elsewhere four lanes are, whose loads straddle lines less often, at the price of writing two by two.  us per
// launch, channels on neighbouring lanes / pairs / fours: 8 x 32 x 147 x 147 stride 2 -> 64 -> 80 12.9 / 11.9 / 10.8, 5 x 64 x 97 x 97
// 1x1 -> 64 -> 3x3 64 10.6 / 9.8 / 9.2; 12 x 64 x 112 x 112 -> 128 -> 64 33.7 / 32.6 / 34.5, 20 x 64 x 56 x 56 -> 128 -> 64 17.1 / 16.8 / 18.7.
// The last one to three groups of pixels, which fill no four, are neighbours among themselves: with lanes left idle for the missing
// ones one pass over the threads became two (1 x 192 x 66 x 66 1x1 -> 64 -> 16 5.46 us, 4.76 here, 4.97 with channels on neighbouring
// lanes; 3 x 192 x 22 x 22 stride 2 -> 64 -> 64 8.26 / 7.54 / 7.65).  Not with eight waves, whose threads hardly ever miss the tasks by so
// few: idle lanes cost them less than the index (100 random calls of 256 channels 1.007 with it, the worst 1.05).
// cg: groups of 8 channels staged, a multiple of 4; zg: groups zeroed in the columns left and right.
template <int NT, typename T>
__device__ __forceinline__ void stage_halo_rows(T* Xs, const T* Xg, int h0, int pad, int rows_in, int cols_in, int CHS, int cg, int zg,
                                                int C0, int H, int W, float inv_cg, float inv_ng, int tid) {
  typedef typename Elem<T>::v8 V8;
  typedef __attribute__((ext_vector_type(8), aligned(2))) T V8u;  // 16 bytes at any element's address
  const int row_step = cols_in * CHS, ng = (W + 7) / 8, groups = rows_in * ng;
  constexpr bool kTail = NT == 256;
  const int tail = groups & 3, body = (groups - tail) * cg, tasks = body + (tail == 0 ? 0 : kTail ? tail : 4) * cg;
  const float inv_tail = tail == 1 ? 1.f : tail == 2 ? 1.f / 2 : 1.f / 3;
  const bool whole = W % 8 == 0;
  const int low = whole ? 4 : 2, per = whole ? cg >> 2 : cg;  // lane bits below `rest`, values of it
  const float inv_per = whole ? 4.f * inv_cg : inv_cg;
  const long long hw = (long long)H * W;
  auto stage = [&](auto both, int t0) __attribute__((always_inline)) {
    constexpr int U = decltype(both)::value;
    i32x4 xr[U][8];
    int col[U];
    bool in[U];
    T* dst[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * NT, hi = t >> low, quad = div_by(hi, inv_per), rest = hi - quad * per;
      int chg = whole ? 4 * rest + ((t >> 1) & 3) : rest, grp = 4 * quad + (whole ? (t & 1) + ((t >> 2) & 2) : t & 3);
      if (kTail && t >= body) chg = div_by(t - body, inv_tail), grp = groups - tail + (t - body) - chg * tail;
      const int ri = div_by(grp, inv_ng);
      const int w = min(8 * (grp - ri * ng), W - 8), h = h0 + ri;
      col[u] = w + pad;
      dst[u] = Xs + ri * row_step + (w + pad) * CHS + 8 * chg;
      in[u] = t < tasks && (kTail || grp < groups);
      const bool live = in[u] && h >= 0 && h < H;
      const T* const src = Xg + (long long)(8 * chg) * hw + (long long)h * W + w;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        i32x4 v = {0, 0, 0, 0};
        if (live && 8 * chg + k < C0) v = __builtin_bit_cast(i32x4, (V8)*reinterpret_cast<const V8u*>(src + k * hw));
        xr[u][k] = v;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!in[u]) break;
#pragma unroll
      for (int px = 0; px < 8; ++px) {
        i32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          o[k] = __builtin_amdgcn_perm(xr[u][2 * k + 1][px >> 1], xr[u][2 * k][px >> 1], (px & 1) ? 0x07060302 : 0x05040100);
        if (col[u] + px < cols_in) *reinterpret_cast<i32x4*>(dst[u] + px * CHS) = o;
      }
    }
  };
  int t0 = tid;
  for (; t0 - tid + NT < tasks; t0 += 2 * NT) stage(CtInt<2>(), t0);
  if (t0 - tid < tasks) stage(CtInt<1>(), t0);
  // the columns left and right of the image
  const int right = max(0, cols_in - W - pad), nz = pad + right;
  if (nz > 0) {
    const float inv_nz = 1.f / (float)nz, inv_zg = zg == cg ? inv_cg : 1.f / (float)zg;
    for (int t = tid; t < rows_in * nz * zg; t += NT) {
      const int rest = div_by(t, inv_zg), chg = t - rest * zg, ri = div_by(rest, inv_nz), z = rest - ri * nz;
      *reinterpret_cast<i32x4*>(Xs + ri * row_step + (z < pad ? z : W + z) * CHS + 8 * chg) = i32x4{0, 0, 0, 0};
    }
  }
}

// Waves of a SIMD that the compiler is held to where its own choice misses them by a few registers: 256 channels on 8 pixel tiles, two
// workgroups of eight waves; 128 on 7 and 192 on 5 take 170, and three workgroups to a compute unit 168 (19 x 64 x 56 x 56 -> 128 -> 64 18.4 us against 16.4).
// 8 pixel tiles would spill (6 x 64 x 57 x 57 -> 128 -> 64 12.9 against 10.6).
constexpr int conv_tiles_min_waves(int WC, int WP, int MC, int PT) {
  return WC == 8 && PT == 8 ? 4 : WC == 4 && WP == 1 && ((MC == 2 && PT == 7) || (MC == 3 && PT == 5)) ? 3 : 1;
}
// WC x WP waves: WC of them split the intermediate channels (MC tiles of 16 each), WP the pixels (PT tiles of 16 each).
template <typename T, int WC, int WP, int MC, int PT>
__global__ __launch_bounds__(64 * WC * WP, conv_tiles_min_waves(WC, WP, MC, PT)) void conv_tiles_kernel(ConvTilesArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Elem<T>::v8 V8;
  typedef typename Elem<T>::v4 V4;
  constexpr int NW = WC * WP, NT = 64 * NW, C1P = 16 * WC * MC, MS = conv_tiles_stride(C1P);
  constexpr int PO = WP * PT <= 2 ? 2 : WP * PT <= 4 ? 4 : 8;  // consecutive output pixels of a lane
  constexpr int D = NW == 8 ? 2 : 4;                 // W1 fragments in flight per tile
  extern __shared__ __attribute__((aligned(16))) char smem_ct[];
  T* const Xs = reinterpret_cast<T*>(smem_ct);  // [rows_in][cols_in][CHS]
  T* const Ms = Xs;                             // [slot][MS], once everyone is done with Xs
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % WC, wp = wave / WC;
  const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
  const int n = lid / (unsigned)p.tiles_h, p0 = (lid - n * (unsigned)p.tiles_h) * p.TH;
  const int npx = min(p.TH, p.P - p0) * p.Q;
  const int h0 = p0 * p.stride - p.pad;
  const int gap = NW == 8 || p.C2 > 16 ? conv_tiles_gap(PO) : 0;  // (one tile of output channels, one wave's: the writes would lose what the reads gain)
  const int CHS = conv_tiles_stride(p.c0p), cg = p.c0p / 8;
  const long long hw = (long long)p.H * p.W;

  const int cb = p.c0p / 32, KS = p.R * p.S * cb;
  const T* const w1 = reinterpret_cast<const T*>(p.w1f) + (size_t)wc * KS * MC * 512;
  V8 wf[D][MC];
  auto load_w = [&](int d, int ks) __attribute__((always_inline)) {
    const T* const src = w1 + (size_t)min(ks, KS - 1) * MC * 512;
#pragma unroll
    for (int m = 0; m < MC; ++m) wf[d][m] = *reinterpret_cast<const V8*>(src + m * 512 + lane * 8);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load_w(d, d);

  const int row_step = p.cols_in * CHS;
  stage_halo_rows<NT>(Xs, reinterpret_cast<const T*>(p.x) + (long long)n * p.C0 * hw, h0, p.pad, p.rows_in, p.cols_in, CHS, cg, cg, p.C0, p.H,
                      p.W, p.inv_cg, p.inv_ng, tid);

  int xb[PT];  // element offset of this lane's pixel of tile t at tap (0, 0)
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    int slot = 16 * (wp * PT + t) + c;
    slot = slot < npx ? slot : 0;
    const int ph = div_by(slot, p.inv_q), pw = slot - ph * p.Q;
    xb[t] = (ph * p.cols_in + pw) * p.stride * CHS + 8 * q;
  }
  f32x4 acc[MC][PT];
#pragma unroll
  for (int m = 0; m < MC; ++m)
#pragma unroll
    for (int t = 0; t < PT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  wg_sync();

  // ---- first convolution: k step = 32 channels of one tap
  {
    int kb = 0, ts = 0, off = 0;  // of the next pixel fragments to fetch: channel block, tap column, element offset
    constexpr int XB = NW == 8 ? 1 : 2;  // (eight waves: four per SIMD hide the LDS latency, and registers are what they lack)
    V8 xf[XB][PT];
    auto load_x = [&](int d) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < PT; ++t) xf[d][t] = *reinterpret_cast<const V8*>(Xs + xb[t] + off);
      off += 32;
      if (++kb == cb) {
        kb = 0, off += CHS - p.c0p;
        if (++ts == p.S) ts = 0, off += row_step - p.S * CHS;
      }
    };
    if (XB == 2) load_x(0);
    for (int ks = 0; ks < KS; ks += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (ks + d >= KS) break;
        if (XB == 1) load_x(0);
        else if (ks + d + 1 < KS) load_x((d + 1) & 1);
#pragma unroll
        for (int m = 0; m < MC; ++m)
#pragma unroll
          for (int t = 0; t < PT; ++t) acc[m][t] = Elem<T>::mfma16(wf[d][m], xf[d & (XB - 1)][t], acc[m][t]);
        load_w(d, ks + d + D);
      }
    }
  }

  // ---- second convolution (1x1): column j of output tile t is pixel PO j + t, so a lane ends with PO consecutive pixels
  // of four channels
  constexpr int KS2 = C1P / 32;
  const int tiles2 = (p.C2 + 15) / 16;
  V8 vf[KS2];
  auto load_w2 = [&](int ct) __attribute__((always_inline)) {
    const T* const src = reinterpret_cast<const T*>(p.w2f) + (size_t)min(ct, tiles2 - 1) * KS2 * 512;
#pragma unroll
    for (int k = 0; k < KS2; ++k) vf[k] = *reinterpret_cast<const V8*>(src + k * 512 + lane * 8);
  };
  load_w2(wave);
  wg_sync();  // the halo rows are no longer read
  // The channels that C1 is padded by are zero also under an infinite pixel, which meets zero weights there.  Where they are
  // rare as one branch here; eight waves mask every store instead, which costs them less (one image of 128 x 28 x 28 -> 256 ->
  // 128 8.9 us, 9.0 with the branch; masking stores costs the other splits up to 1 %).
  constexpr bool kMaskStores = NW == 8;
  if (!kMaskStores && p.C1 < C1P)
#pragma unroll
    for (int m = 0; m < MC; ++m)
      if (16 * (wc * MC + m) + 4 * q >= p.C1)
#pragma unroll
        for (int t = 0; t < PT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  T* const ms = Ms + (16 * wp * PT + c) * MS + (16 * wp * PT + c) / PO * gap + 16 * wc * MC + 4 * q;
#pragma unroll
  for (int m = 0; m < MC; ++m)
#pragma unroll
    for (int t = 0; t < PT; ++t) {
      f32x4 v = acc[m][t];
      if (p.relu_mid)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f);
      const typename Elem<T>::v2 lo = cvt2<T>(v[0], v[1]), hi = cvt2<T>(v[2], v[3]);
      const int c1 = 16 * (wc * MC + m) + 4 * q;
      V4 x = {lo[0], lo[1], hi[0], hi[1]};
      if (kMaskStores && c1 >= p.C1) x = V4{0, 0, 0, 0};
      *reinterpret_cast<V4*>(PO == 2 ? Ms + (16 * (wp * PT + t) + c) * MS + c1 : ms + t * (16 * MS + 16 / PO * gap) + 16 * m) = x;
    }
  wg_sync();
  const T* const mb = Ms + c * (PO * MS + gap) + 8 * q;
  const long long plane = (long long)p.P * p.Q;
  const int valid = npx - PO * c;  // of this lane's pixels
  for (int ct = wave; ct < tiles2; ct += NW) {
    f32x4 o[PO];
#pragma unroll
    for (int t = 0; t < PO; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    V8 mf[2][PO];
#pragma unroll
    for (int t = 0; t < PO; ++t) mf[0][t] = *reinterpret_cast<const V8*>(mb + t * MS);
#pragma unroll
    for (int k = 0; k < KS2; ++k) {
      if (k + 1 < KS2)
#pragma unroll
        for (int t = 0; t < PO; ++t) mf[(k + 1) & 1][t] = *reinterpret_cast<const V8*>(mb + t * MS + 32 * (k + 1));
#pragma unroll
      for (int t = 0; t < PO; ++t) o[t] = Elem<T>::mfma16(vf[k], mf[k & 1][t], o[t]);
      __builtin_amdgcn_sched_barrier(0);  // one step of reads ahead, not all of them (registers)
    }
    load_w2(ct + NW);
    if (p.relu_out)
#pragma unroll
      for (int t = 0; t < PO; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[t][r] = fmaxf(o[t][r], 0.f);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c2 = 16 * ct + 4 * q + r;
      if (c2 >= p.C2) continue;
      const long long at = ((long long)n * p.C2 + c2) * plane + (long long)p0 * p.Q + PO * c;
      if (p.out_f32) {
        float* const dst = reinterpret_cast<float*>(p.y) + at;
#pragma unroll
        for (int t = 0; t < PO; ++t)
          if (t < valid) dst[t] = o[t][r];
        continue;
      }
      typedef __attribute__((ext_vector_type(PO))) T VP;
      typedef __attribute__((ext_vector_type(PO), aligned(2))) T VPu;
      VP v;
#pragma unroll
      for (int t = 0; t < PO; t += 2) {
        const typename Elem<T>::v2 two = cvt2<T>(o[t][r], o[t + 1][r]);
        v[t] = two[0], v[t + 1] = two[1];
      }
      T* const dst = reinterpret_cast<T*>(p.y) + at;
      if (valid >= PO) {
        *reinterpret_cast<VPu*>(dst) = v;
      } else if constexpr (NW == 8) {
        // (the pieces' offsets and tests take sixteen registers, and past 128 only one workgroup of eight waves fits a compute
        // unit: 6 x 128 x 71 x 71 -> 256 -> 128 31.3 us against 33.7)
#pragma unroll
        for (int t = 0; t < PO; ++t)
          if (t < valid) dst[t] = v[t];
      } else if (valid > 0) {
        store_some(dst, v, valid);
      }
    }
  }
#else
  (void)p;
#endif
}

template <typename T, int WC, int WP, int MC, int PT>
hipError_t launch_conv_tiles_as(const ConvTilesArgs& a, hipStream_t stream) {
  auto kern = conv_tiles_kernel<T, WC, WP, MC, PT>;
  static thread_local int configured_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  constexpr int slots = WP * PT <= 2 ? 32 : WP * PT <= 4 ? 64 : 128;
  const int lds = conv_tiles_lds_bytes(a.rows_in, a.cols_in, a.c0p, 16 * WC * MC, slots);
  hipLaunchKernelGGL(kern, dim3((unsigned)a.N * (unsigned)a.tiles_h), dim3(64 * WC * WP), lds, stream, a);
  return hipGetLastError();
}

template <typename T, int WC, int WP, int MC>
hipError_t launch_conv_tiles_rows(const ConvTilesArgs& a, hipStream_t stream) {
  const int tiles = (a.TH * a.Q + 15) / 16, pt = (tiles + WP - 1) / WP;
  if (tiles > kCtMaxTiles) return hipErrorInvalidValue;
  if (pt == 1) return launch_conv_tiles_as<T, WC, WP, MC, WP == 1 ? 2 : 1>(a, stream);
  if (pt == 2) return launch_conv_tiles_as<T, WC, WP, MC, 2>(a, stream);
  if (pt == 3) return launch_conv_tiles_as<T, WC, WP, MC, 3>(a, stream);
  if (pt == 4) return launch_conv_tiles_as<T, WC, WP, MC, 4>(a, stream);
  if constexpr (WP == 1) {
    if (pt == 5) return launch_conv_tiles_as<T, WC, WP, MC, 5>(a, stream);
    if (pt == 6) return launch_conv_tiles_as<T, WC, WP, MC, 6>(a, stream);
    if (pt == 7) return launch_conv_tiles_as<T, WC, WP, MC, 7>(a, stream);
    if (pt == 8) return launch_conv_tiles_as<T, WC, WP, MC, 8>(a, stream);
  }
  return hipErrorInvalidValue;
}

// How the waves of a workgroup split the C1 x pixels product of the first convolution: wc of them the channels (mc tiles
// of 16 each), wp the pixels.  Splitting channels alone reads every weight fragment once per workgroup and every pixel
// fragment wc times out of LDS; at 64 channels that makes LDS the bound of a long contraction, and two waves by two halve
// its reads for twice the weight fetches: 32 x 64 x 56 x 56 3x3 -> 64 -> 64 17.4 -> 15.7 us, -> 256 24.5 -> 22.7; with 9 k steps
// (32 input channels) the weights are what counts: 32 x 32 x 147 x 147 stride 2 31.4 against 32.7 us.
struct ConvTilesSplit {
  int wc, wp, mc;
};
inline ConvTilesSplit conv_tiles_split(int C1, int k_steps) {
  if (C1 <= 64) return k_steps >= 12 ? ConvTilesSplit{2, 2, 2} : ConvTilesSplit{4, 1, 1};
  return C1 <= 128 ? ConvTilesSplit{4, 1, 2} : C1 <= 192 ? ConvTilesSplit{4, 1, 3} : ConvTilesSplit{8, 1, 2};
}
inline int conv_tiles_c1p(int C1) { return (C1 + 63) / 64 * 64; }
inline size_t conv_tiles_w1_bytes(int C1, int c0p, int taps) { return (size_t)conv_tiles_c1p(C1) / 16 * taps * (c0p / 32) * 1024; }
inline size_t conv_tiles_w2_bytes(int C2, int c1p) { return (size_t)((C2 + 15) / 16) * (c1p / 32) * 1024; }

template <typename T>
hipError_t launch_conv_tiles(const ConvTilesArgs& a, hipStream_t stream) {
  const ConvTilesSplit w = conv_tiles_split(a.C1, a.R * a.S * a.c0p / 32);
  if (w.wp == 2) return launch_conv_tiles_rows<T, 2, 2, 2>(a, stream);
  if (w.wc == 8) return launch_conv_tiles_rows<T, 8, 1, 2>(a, stream);
  if (w.mc == 1) return launch_conv_tiles_rows<T, 4, 1, 1>(a, stream);
  if (w.mc == 2) return launch_conv_tiles_rows<T, 4, 1, 2>(a, stream);
  return launch_conv_tiles_rows<T, 4, 1, 3>(a, stream);
}

template <typename T>
hipError_t launch_pack_conv_tiles(const ConvTilesArgs& a, const void* w1, const void* w2, void* w1f, void* w2f, hipStream_t stream) {
  const int c1p = conv_tiles_c1p(a.C1), taps = a.R * a.S;
  const ConvFragments f1 = {w1, w1f, a.C1, a.C0, a.c0p, taps, conv_tiles_split(a.C1, taps * a.c0p / 32).mc,
                            (unsigned)(conv_tiles_w1_bytes(a.C1, a.c0p, taps) / 2)};
  const ConvFragments f2 = {w2, w2f, a.C2, a.C1, c1p, 1, 1, (unsigned)(conv_tiles_w2_bytes(a.C2, c1p) / 2)};
  const unsigned blocks1 = (f1.total + 255) / 256, blocks2 = (f2.total + 255) / 256;
  hipLaunchKernelGGL(pack_conv_fragments_kernel<T>, dim3(blocks1 + blocks2), dim3(256), 0, stream, f1, f2, blocks1);
  return hipGetLastError();
}

}  // namespace ditto
