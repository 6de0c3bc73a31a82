// depthwise 3x3 (pad 1, any stride, 1 or 16 outputs per input channel) -> cast|relu -> conv 1x1 on NCHW tensors, fp16 /
// bf16: tiles of whole output rows of any length.
#pragma once
#include "common.h"

namespace ditto {

struct DwTilesArgs {
  const void* x;
  const void* w1;
  const void* w2;
  void* y;
  int N, C0, H, W, C2;
  int P, Q, stride;
  int TH, tiles_h;  // output rows per workgroup, workgroups per image
  int rows_in;      // input rows a full tile reads
  int relu_mid, relu_out, out_f32;
  float inv_blocks, inv_rows, inv_q;  // 1 / (16-byte blocks per row), 1 / rows_in, 1 / Q
  float inv_group;                    // 1 / (blocks of eight channels and their padding)
  int groups;                         // of waves that share out a chunk's channels: 1, or 2 or 4 with one tile a wave
};

constexpr int kDtWaves = 8;
constexpr int kDtMaxTiles = 16;  // tiles of 16 output pixels per workgroup

__host__ __device__ constexpr int dw_tiles_chunk(int mult) { return mult == 16 ? 16 : 32; }  // input channels per chunk
// An image row in LDS: one block of 8 zeros (its last is the pixel left of the row, its first the pixel right of the row
// before), then the row in blocks of 8, zeros behind its end.  Behind eight channels a few more blocks of zeros: the lanes
// that read channels 8 q .. + 7 (one output per channel) then start in four different quarters of the banks.
__host__ __device__ inline int dw_tiles_row_blocks(int W) { return 1 + (W + 7) / 8; }
__host__ __device__ inline int dw_tiles_group_blocks(int rows_in, int W) { return 8 * rows_in * dw_tiles_row_blocks(W) + 4; }
__host__ __device__ inline int dw_tiles_lds_bytes(int mult, int rows_in, int W, int nt, int groups) {
  const int x = dw_tiles_chunk(mult) / 8 * dw_tiles_group_blocks(rows_in, W) * 16;
  const int chunk = x + (mult == 16 ? 256 * 18 + 8 * nt * 1024 : 32 * 32 + nt * 1024);
  const int sums = (kDtWaves - kDtWaves / groups) * nt * 1024;  // of all groups of waves but the first
  return chunk > sums ? chunk : sums;
}

template <typename T>
__device__ __forceinline__ f32x4 mfma16x16x16(i32x2 a, i32x2 b, f32x4 c) {
  if constexpr (Elem<T>::is_bf16)
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
}

// 16 bytes shifted towards the end by `s` 16-bit elements (0..7), zeros behind: element i of the result is element i + s
__device__ __forceinline__ i32x4 drop_elements(i32x4 v, int s) {
  i32x4 r = v;
  if (s & 4) r = i32x4{r[2], r[3], 0, 0};
  if (s & 2) r = i32x4{r[1], r[2], r[3], 0};
  if (s & 1)
    r = i32x4{(int)__builtin_amdgcn_alignbit(r[1], r[0], 16), (int)__builtin_amdgcn_alignbit(r[2], r[1], 16),
              (int)__builtin_amdgcn_alignbit(r[3], r[2], 16), (int)((unsigned)r[3] >> 16)};
  return r;
}

// A workgroup owns TH whole output rows of an image: image rows of any length keep 16-byte loads (the last block of a row is
// loaded from W - 8 and shifted in registers), halo rows are fetched once per TH rows, and a tile is never padded to a
// rectangle's width.  Input channels go by in chunks of 16 (32) through LDS.  A wave owns RT tiles of 16 output pixels and all
// C2 <= 16 NT output channels; pixel RT j + t of the wave's is column j of tile t, so a lane ends with RT consecutive pixels
// of four channels of every output tile.  The depthwise results never leave the registers: in both forms a lane holds its
// part of the 1x1 convolution's operand as it computes it.
// What bounds it: on a full grid, times 16, vector ALU (14 us), LDS reads (12) and matrix cores (9) of 33 us under the
// tracer, taking turns more than overlapping (32 x 64 x 56 x 56 -> 64: 29.5 us untraced, the tensors need 5; the general
// kernel, which walks padded rectangles one after another and waits for each chunk, took 52.5); times 1 the vector ALU (40 of
// 54 us at 32 x 64 x 112 x 112); on small grids the chain of a chunk's load, barrier and products, 2 us per 16 channels (one
// image of 32 x 37 x 37 times 16: 8.6 us, before 25.3; 32 x 16 x 147 x 147 times 16 stride 2: 19 us, before 127).
// Rows of at most 64 pixels on few images leave waves without a tile, and the chain above is theirs who have one: two or four
// waves share out the channels of a chunk then (G) and their sums meet at the end (4 x 64 x 28 x 28 times 16: 13.6 -> 9.1 us,
// 3 x 64 x 62 x 62 13.3 -> 10.7, 4 x 32 x 57 x 57 9.6 -> 7.9; times 1, whose sums are shorter: 4 x 64 x 28 x 28 6.5 -> 5.8).
// Eight waves of two tiles instead of four of four: half the blocks for a thread to stage, and two workgroups share a
// compute unit (32.4 -> 29.5 us).  Filters are loaded as they lie in memory, by 16-byte blocks: one 18-byte filter per lane
// cost 0.4 us per chunk in misaligned loads.
template <typename T, int MULT, int RT, int NT, int G>
__global__ __launch_bounds__(64 * kDtWaves, MULT == 1 && RT == 2 ? 2 : 4) void dw_tiles_kernel(DwTilesArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Elem<T>::v8 V8;
  typedef typename Elem<T>::v4 V4;
  typedef typename Elem<T>::v2 V2;
  typedef __attribute__((ext_vector_type(8), aligned(2))) T V8u;
  constexpr int CC = dw_tiles_chunk(MULT), THREADS = 64 * kDtWaves, WP = kDtWaves / G;
  static_assert(G == 1 || RT == 1, "");
  extern __shared__ __attribute__((aligned(16))) char smem_dt[];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // its pixel tiles, its share of the channels.  (With one group the share is said to be the first: from `wave / 8` the compiler
  // does not see the loop's start, unrolls it otherwise, and 25 x 16 x 112 x 112 times 16 stride 2 takes 9.95 us instead of 9.50.)
  const int wp = G == 1 ? wave : wave % WP, wg = G == 1 ? 0 : wave / WP;
  const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
  const int n = lid / (unsigned)p.tiles_h, p0 = (lid - n * (unsigned)p.tiles_h) * p.TH;
  const int npx = min(p.TH, p.P - p0) * p.Q, h0 = p0 * p.stride - 1;
  const int blocks = 1 + (p.W + 7) / 8, plane = p.rows_in * blocks * 4;  // dwords of a channel's rows
  const int C1 = p.C0 * MULT;
  const int hw = p.H * p.W;
  const int group = 8 * p.rows_in * blocks + 4, xblocks = CC / 8 * group;
  const unsigned* const Xs = reinterpret_cast<const unsigned*>(smem_dt);
  char* const w1_lds = smem_dt + xblocks * 16;
  // w1_lds: the filters as they lie in memory (MULT 16); three rows of three taps and a zero, 32 bytes each (MULT 1).
  // W2s: MFMA fragments, [output tile][lane][8], of each pair of channels (MULT 16) or of the chunk (MULT 1)
  T* const W2s = reinterpret_cast<T*>(w1_lds + (MULT == 16 ? 256 * 18 : 32 * 32));
  const unsigned thr = relu_packed_threshold(p.relu_mid != 0);
  const T* const Xg = reinterpret_cast<const T*>(p.x) + (long long)n * p.C0 * hw;
  const T* const W1g = reinterpret_cast<const T*>(p.w1);
  const T* const W2g = reinterpret_cast<const T*>(p.w2);

  // this lane's three taps of a filter row: two dwords from xd[t], shifted down by sh[t].  MULT 16: filter row q (lanes with
  // q = 3 read the zeros a channel starts with); MULT 1: from filter row 0 on
  int xd[RT], sh[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    int slot = 16 * RT * wp + RT * c + t;
    slot = slot < npx ? slot : 0;
    const int ph = div_by(slot, p.inv_q), pw = slot - ph * p.Q;
    const int e = 7 + pw * p.stride;
    xd[t] = MULT == 16 && q == 3 ? 0 : (ph * p.stride + (MULT == 16 ? q : 0)) * blocks * 4 + (e >> 1);
    sh[t] = (e & 1) * 16;
  }
  f32x4 acc[RT][NT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // What this thread brings of a chunk: 16-byte blocks of the input rows (blocks tid + THREADS u of the LDS image; off < 0 where
  // it is zeros), a filter, blocks of W2.  The loads of the next chunk are in flight while one is computed.
  constexpr int KX = 2, K2 = MULT == 16 ? NT : 1;
  auto locate = [&](int b, int& off, int& drop) {
    const int gr = div_by(b, p.inv_group), at = b - gr * group;
    const int cr = div_by(at, p.inv_blocks), ch = div_by(cr, p.inv_rows);
    const int g = at - cr * blocks - 1, h = h0 + cr - ch * p.rows_in;
    drop = max(0, 8 * g + 8 - p.W);  // the row's last block is loaded from W - 8
    off = b < xblocks && ch < 8 && g >= 0 && h >= 0 && h < p.H ? (8 * gr + ch) * hw + h * p.W + 8 * g - drop : -1;
  };
  // (its blocks of W2: row c, eight channels w2g - the order in which a wave's LDS writes meet no bank twice)
  const int w2g = 4 * wave + 2 * (q & 1) + (q >> 1);
  int xoff[KX], xdrop[KX];
#pragma unroll
  for (int u = 0; u < KX; ++u) locate(tid + THREADS * u, xoff[u], xdrop[u]);
  V8 xv[KX], w1v, w2v[K2];  // (rows of W2 behind its last one: anything, their results are not stored)
  T w1last;
  auto load_block = [&](int c0, int off) {  // (off < 0 or a channel behind the last one: anything in bounds)
    return *reinterpret_cast<const V8u*>(Xg + (long long)c0 * hw + (off >= 0 && off < (p.C0 - c0) * hw ? off : 0));
  };
  auto store_block = [&](int c0, int b, V8 v, int off, int drop) {
    i32x4 w = __builtin_bit_cast(i32x4, v);
    if (p.W & 7) w = drop_elements(w, drop);
    if (off < 0 || off >= (p.C0 - c0) * hw) w = i32x4{0, 0, 0, 0};
    reinterpret_cast<i32x4*>(smem_dt)[b] = w;
  };
  auto load_chunk = [&](int c0) {
#pragma unroll
    for (int u = 0; u < KX; ++u) xv[u] = load_block(c0, xoff[u]);
    if constexpr (MULT == 16) {
      w1v = *reinterpret_cast<const V8u*>(W1g + min(c0 * 144 + 8 * tid, C1 * 9 - 8));
    } else {
      const T* const filter = W1g + 9 * min(c0 + tid, C1 - 1);
      w1v = *reinterpret_cast<const V8u*>(filter);
      w1last = filter[8];
    }
    const int c1 = min(MULT == 16 ? c0 * 16 + 8 * w2g : c0 + 8 * q, C1 - 8);
#pragma unroll
    for (int u = 0; u < K2; ++u)
      w2v[u] = *reinterpret_cast<const V8u*>(W2g + (long long)min(16 * (MULT == 16 ? u : wave) + c, p.C2 - 1) * C1 + c1);
  };
  load_chunk(0);

  for (int c0 = 0; c0 < p.C0; c0 += CC) {
    if (c0 > 0) wg_sync();  // everyone is done with the previous chunk
#pragma unroll
    for (int u = 0; u < KX; ++u)
      if (tid + THREADS * u < xblocks) store_block(c0, tid + THREADS * u, xv[u], xoff[u], xdrop[u]);
    for (int b = tid + THREADS * KX; b < xblocks; b += THREADS) {
      int off, drop;
      locate(b, off, drop);
      store_block(c0, b, load_block(c0, off), off, drop);
    }
    // (filters behind the last one are zeros like their input channels: zero times an infinite weight is NaN)
    if constexpr (MULT == 16) {
      if (c0 + CC > p.C0 && c0 * 144 + 8 * tid >= C1 * 9) w1v = V8{0, 0, 0, 0, 0, 0, 0, 0};
      if (tid < 256 * 9 / 8) reinterpret_cast<V8*>(w1_lds)[tid] = w1v;
      // lane q of a fragment holds outputs 4 q .. + 3 of the pair's first channel, then of its second
#pragma unroll
      for (int u = 0; u < K2; ++u) {
        const V8 v = c0 * 16 + 8 * w2g < C1 ? w2v[u] : V8{0, 0, 0, 0, 0, 0, 0, 0};
        T* const dst = W2s + (((w2g >> 2) * NT + u) * 64 + (w2g & 1) * 32 + c) * 8 + 4 * ((w2g >> 1) & 1);
        *reinterpret_cast<V4*>(dst) = V4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<V4*>(dst + 16 * 8) = V4{v[4], v[5], v[6], v[7]};
      }
    } else {
      if (tid < CC) {
        if (c0 + tid >= C1) w1v = V8{0, 0, 0, 0, 0, 0, 0, 0}, w1last = 0;
        reinterpret_cast<V8*>(w1_lds)[2 * tid] = V8{w1v[0], w1v[1], w1v[2], 0, w1v[3], w1v[4], w1v[5], 0};
        reinterpret_cast<V8*>(w1_lds)[2 * tid + 1] = V8{w1v[6], w1v[7], w1last, 0, 0, 0, 0, 0};
      }
      if (wave < NT)
        reinterpret_cast<V8*>(W2s)[tid] = c0 + 8 * q < C1 ? w2v[0] : V8{0, 0, 0, 0, 0, 0, 0, 0};  // C0 is a multiple of 8
    }
    wg_sync();
    if (c0 + CC < p.C0) load_chunk(c0 + CC);

    if constexpr (MULT == 16) {
      // The sixteen filters of a channel as one 16x16x16 MFMA: k = 4 r + s is tap (r, s), lane (c, q) holds filter c's row q
      // and pixel c's row q; the products for s = 3 and r = 3 meet zero weights.  Its result - outputs 4 q .. + 3 of pixel c
      // - is half an operand of the 1x1 convolution as it comes.
      const unsigned* const W1s = reinterpret_cast<const unsigned*>(w1_lds);
      const int o1 = 9 * c + 3 * min(q, 2), w1d = o1 >> 1, w1sh = (o1 & 1) * 16;
      const unsigned keep = q < 3 ? 0xffffffffu : 0u;
#pragma unroll 2
      for (int pr = wg; pr < 8; pr += G) {
        i32x2 a[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const unsigned lo = W1s[(2 * pr + u) * 72 + w1d], hi = W1s[(2 * pr + u) * 72 + w1d + 1];
          a[u] = i32x2{(int)(__builtin_amdgcn_alignbit(hi, lo, w1sh) & keep), (int)((hi >> w1sh) & 0xffffu & keep)};
        }
        V8 w2[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) w2[j] = *reinterpret_cast<const V8*>(W2s + ((pr * NT + j) * 64 + lane) * 8);
        V8 pf[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          f32x4 m[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const unsigned* const x = Xs + (pr >> 2) * 16 + (2 * pr + u) * plane + xd[t];
            const unsigned lo = x[0], hi = x[1];
            m[u] = mfma16x16x16<T>(a[u], i32x2{(int)__builtin_amdgcn_alignbit(hi, lo, sh[t]), (int)__builtin_amdgcn_ubfe(hi, sh[t], 16)}, f32x4{0.f, 0.f, 0.f, 0.f});
          }
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
              const V2 two = cvt2<T>(m[u][r], m[u][r + 1]);
              pf[t][4 * u + r] = two[0];
              pf[t][4 * u + r + 1] = two[1];
            }
          pf[t] = relu_packed(pf[t], thr);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int t = 0; t < RT; ++t) acc[t][j] = Elem<T>::mfma16(w2[j], pf[t], acc[t][j]);
      }
    } else {
      // One output per channel: lane (c, q) computes channels 8 q .. + 7 of pixel c, its share of the 1x1 convolution's
      // operand, as six two-element dot products per channel (three taps of a row: a pair, and one against zero)
      // (with several groups of waves: 8 / G of them, the rest of the operand zeros)
      constexpr int KG = 8 / G;
      const int k0 = KG * wg;
      V8 pf[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) pf[t] = V8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < KG; k += 2) {
        float m[RT][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const i32x2* const w = reinterpret_cast<const i32x2*>(w1_lds) + (8 * q + k0 + k + u) * 4;
#pragma unroll
          for (int t = 0; t < RT; ++t) m[t][u] = 0.f;
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            const i32x2 taps = w[r];
            const int taps01 = taps[0], tap2 = taps[1];  // (a bit cast of a vector's element takes element 0)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              const unsigned* const x = Xs + q * group * 4 + (k0 + k + u) * plane + r * blocks * 4 + xd[t];
              const unsigned lo = x[0], hi = x[1];
              m[t][u] = Elem<T>::dot2(__builtin_bit_cast(V2, __builtin_amdgcn_alignbit(hi, lo, sh[t])), __builtin_bit_cast(V2, taps01), m[t][u]);
              m[t][u] = Elem<T>::dot2(__builtin_bit_cast(V2, __builtin_amdgcn_ubfe(hi, sh[t], 16)), __builtin_bit_cast(V2, tap2), m[t][u]);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const V2 two = cvt2<T>(m[t][0], m[t][1]);
          pf[t][k] = two[0];
          pf[t][k + 1] = two[1];
        }
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) pf[t] = relu_packed(pf[t], thr);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        V8 w2;
        if constexpr (G == 1) {
          w2 = reinterpret_cast<const V8*>(W2s)[j * 64 + lane];
        } else {
          typedef __attribute__((ext_vector_type(KG))) T VG;
          const VG own = *reinterpret_cast<const VG*>(W2s + (j * 64 + lane) * 8 + k0);
          w2 = V8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < KG; ++e) w2[e] = own[e];
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t][j] = Elem<T>::mfma16(w2, pf[t], acc[t][j]);
      }
    }
  }

  if constexpr (G > 1) {
    // the groups' sums meet in LDS, which nobody needs any more, and are added in the order of the groups
    f32x4* const sums = reinterpret_cast<f32x4*>(smem_dt) + wp * NT * 64 + lane;
    wg_sync();
    if (wg > 0)
#pragma unroll
      for (int j = 0; j < NT; ++j) sums[((wg - 1) * WP * NT + j) * 64] = acc[0][j];
    wg_sync();
    if (wg > 0) return;
#pragma unroll
    for (int g = 1; g < G; ++g)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[0][j] += sums[((g - 1) * WP * NT + j) * 64];
  }

  const int first = 16 * RT * wp + RT * c, valid = npx - first;  // of this lane's pixels
  const long long out_plane = (long long)p.P * p.Q;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c2 = 16 * j + 4 * q + r;
      if (c2 >= p.C2) continue;
      const long long at = ((long long)n * p.C2 + c2) * out_plane + (long long)p0 * p.Q + first;
      float v[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) v[t] = p.relu_out ? fmaxf(acc[t][j][r], 0.f) : acc[t][j][r];
      if (p.out_f32) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
          if (t < valid) reinterpret_cast<float*>(p.y)[at + t] = v[t];
        continue;
      }
      T* const dst = reinterpret_cast<T*>(p.y) + at;
      if constexpr (RT > 1) {
        typedef __attribute__((ext_vector_type(RT))) T VP;
        typedef __attribute__((ext_vector_type(RT), aligned(2))) T VPu;
        VP o;
#pragma unroll
        for (int t = 0; t < RT; t += 2) {
          const V2 two = cvt2<T>(v[t], v[t + 1]);
          o[t] = two[0], o[t + 1] = two[1];
        }
        if (valid >= RT) {
          *reinterpret_cast<VPu*>(dst) = o;
        } else {
#pragma unroll
          for (int t = 0; t < RT; ++t)
            if (t < valid) dst[t] = o[t];
        }
      } else if (valid > 0) {
        dst[0] = cvt2<T>(v[0], v[0])[0];
      }
    }
#else
  (void)p;
#endif
}

template <typename T, int MULT, int RT, int NT, int G = 1>
hipError_t launch_dw_tiles_as(const DwTilesArgs& a, hipStream_t stream) {
  auto kern = dw_tiles_kernel<T, MULT, RT, NT, G>;
  static thread_local int configured_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  const int lds = dw_tiles_lds_bytes(MULT, a.rows_in, a.W, NT, a.groups);
  hipLaunchKernelGGL(kern, dim3((unsigned)a.N * (unsigned)a.tiles_h), dim3(64 * kDtWaves), lds, stream, a);
  return hipGetLastError();
}
template <typename T, int MULT>
hipError_t launch_dw_tiles_mult(const DwTilesArgs& a, hipStream_t stream) {
  const int tiles = (a.TH * a.Q + 15) / 16;
  if (tiles > kDtMaxTiles || a.C2 > 64) return hipErrorInvalidValue;
  const bool one = tiles <= kDtWaves;
  if (a.groups > 1 && tiles * a.groups > kDtWaves) return hipErrorInvalidValue;
  if (a.groups == 2) return a.C2 <= 32 ? launch_dw_tiles_as<T, MULT, 1, 2, 2>(a, stream) : launch_dw_tiles_as<T, MULT, 1, 4, 2>(a, stream);
  if (a.groups == 4) return a.C2 <= 32 ? launch_dw_tiles_as<T, MULT, 1, 2, 4>(a, stream) : launch_dw_tiles_as<T, MULT, 1, 4, 4>(a, stream);
  if (a.C2 <= 32)
    return one ? launch_dw_tiles_as<T, MULT, 1, 2>(a, stream) : launch_dw_tiles_as<T, MULT, 2, 2>(a, stream);
  return one ? launch_dw_tiles_as<T, MULT, 1, 4>(a, stream) : launch_dw_tiles_as<T, MULT, 2, 4>(a, stream);
}
// mult: 1 or 16
template <typename T>
hipError_t launch_dw_tiles(int mult, const DwTilesArgs& a, hipStream_t stream) {
  return mult == 16 ? launch_dw_tiles_mult<T, 16>(a, stream) : launch_dw_tiles_mult<T, 1>(a, stream);
}

}  // namespace ditto
