// Fused two-contraction chain  F = epilogue(inter(A.B).C)  for fp16 / bf16 with head sizes that fill neither 64 nor 128
// columns: K and N are padded to 80.  (See bmm_chain_fp.h for the chain and the transposed formulation, bmm_chain_fp8m16.h for
// the operand layouts of v_mfma_f32_16x16x32 and the hand-over between the contractions.)
//
// The kernels padded to 128 columns spend 1.6 times the matrix instructions, LDS traffic and LDS on a head of 80, and start
// slowly: 197 keys were two to three of their steps of a pipeline several steps deep.  Here a wave owns 32 rows (every LDS
// fragment feeds two MFMAs), four or eight waves share a ring of three 24 KB tiles of 64 keys, and two workgroups fit a compute
// unit, one loading while the other computes.  A last tile of at most 32 keys costs half a step, a wave without rows only its
// share of the loads.  Rows in LDS are padded to 13 and 10 16-byte chunks, which spreads both kinds of fragment reads over
// all 64 banks without a swizzle (10-chunk rows: 16 lanes cover 4 rows x 32 bytes at banks 0, 40, 16, 56; 13-chunk rows:
// strides of 52 banks), so all of a tile's fragment addresses are constants from two registers.
//
// Bound: matrix and vector pipes about evenly from a thousand keys on (32 x 4096 x 4096 187 us, 0.92 PFLOP/s counted without the
// padding); below that the chain start -> first tile -> L / 64 steps of 0.85 us.  Measured, us per launch with softmax (2.4 of
// them the launch), padded to 128 -> here, four | eight waves: 256 x 197 x 197 14.3 -> 10.6 | 10.3, 640 x 49 x 49
// 22.9 -> 8.8 | 12.0, 80 x 400 x 400 23.2 -> 13.4 | 12.9, 96 x 700 x 700 44.8 -> 28.7 | 35.9, 32 x 4096 x 4096 206 -> 191 | 187.
// The same kernel at 64 columns (without softmax, large grids) and at 128 (up to about 500 keys) is ahead of the others by its
// start: 512 x 197 x 197 x 64 16.8 -> 12.2, x 128 with softmax 33.2 -> 27.8.
//
// At 64 columns a row of B or C is 128 bytes and needs no padding if it is swizzled: tiles of 16 KB instead of 20, four direct
// loads a wave and tile instead of five, and three workgroups of four waves to a compute unit instead of two.  With two waves on
// a SIMD its pipes were 72 % busy (vector ALU 41, of which v_exp_f32 two thirds, matrix 30); the third takes the waits of the
// other two: 1152 x 512 x 512 with softmax 115 -> 107 us, 830 x 1024 x 1024 291 -> 258, 1249 x 256 x 256 41.6 -> 36.2, and one
// round more of workgroups fits (329 x 197 x 128 9.6 -> 7.8).
#pragma once
#include "bmm_chain_fp4m16.h"
#include "bmm_chain_fp8m16.h"
#include "common.h"

namespace ditto {

constexpr int kRowsRing = 3;

// One tile of 64 keys in LDS: B, then C, filled by direct loads of 64 16-byte chunks each that are dealt to the waves in
// order; rows are padded to chunk counts that spread the reads of 16 lanes over all banks, no swizzle.  Heads of 64 columns
// fill 128-byte rows: those are swizzled (see swz4m16_rows), a tile is 16 KB and three workgroups of four waves fit a compute unit.
// DT: column tiles of 16 that K and N are padded to; the contraction over K runs in steps of 32.
template <int DT, bool B_KL>
struct RowsTiles {
  static constexpr int KS = (DT + 1) / 2;
  static constexpr bool SWZ = DT == 4;
  static constexpr int B_CPR = B_KL || SWZ ? 8 : 4 * KS + 1;  // [64 l][32 KS k], or [32 KS k][64 l] with swizzled 128-byte rows
  static constexpr int B_ROWS = B_KL ? 32 * KS : kBN;
  static constexpr int C_CPR = SWZ ? 8 : DT == 8 ? 18 : 10;
  static constexpr int B_LOADS = (B_ROWS * B_CPR + 63) / 64, C_LOADS = (kBN * C_CPR + 63) / 64;
  static constexpr int C_OFF = B_LOADS * 1024;
  // a wave's 32 rows of A on their way to its registers
  static constexpr int A_CPR = SWZ ? 8 : 2 * DT + 1, A_LOADS = (32 * A_CPR + 63) / 64;
};
template <int DT, bool B_KL, int NW>
__host__ __device__ constexpr int bmm_chain_rows_tile_bytes() {
  return (RowsTiles<DT, B_KL>::B_LOADS + RowsTiles<DT, B_KL>::C_LOADS + NW - 1) / NW * NW * 1024;
}
template <int DT, bool B_KL, int NW>
__host__ __device__ constexpr int bmm_chain_rows_lds() {
  // the first two tiles with A behind them, or all tiles; the flag of the optimistic walk
  return 2 * bmm_chain_rows_tile_bytes<DT, B_KL, NW>() + 64 +
         (bmm_chain_rows_tile_bytes<DT, B_KL, NW>() > NW * RowsTiles<DT, B_KL>::A_LOADS * 1024 ? bmm_chain_rows_tile_bytes<DT, B_KL, NW>()
                                                                                             : NW * RowsTiles<DT, B_KL>::A_LOADS * 1024);
}

inline int bmm_chain_rows_lds(int dt, int nw, bool kl) {
  if (dt == 4 && nw == 4) return kl ? bmm_chain_rows_lds<4, true, 4>() : bmm_chain_rows_lds<4, false, 4>();
  if (dt == 4) return kl ? bmm_chain_rows_lds<4, true, 8>() : bmm_chain_rows_lds<4, false, 8>();
  if (dt == 5 && nw == 4) return kl ? bmm_chain_rows_lds<5, true, 4>() : bmm_chain_rows_lds<5, false, 4>();
  if (dt == 5) return kl ? bmm_chain_rows_lds<5, true, 8>() : bmm_chain_rows_lds<5, false, 8>();
  return kl ? bmm_chain_rows_lds<8, true, 8>() : bmm_chain_rows_lds<8, false, 8>();
}

template <typename T, int DT, int NW, int INTER, bool B_KL, typename Args>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DT == 4 && NW == 4 ? 3 : 2))) void bmm_chain_rows_kernel(Args p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Elem<T>::v8 V8;
  typedef typename Elem<T>::v4 V4;
  typedef typename Elem<T>::v2 V2;
  typedef RowsTiles<DT, B_KL> S;
  constexpr int RT = 2, KS = S::KS, NR = kRowsRing;
  constexpr int TB = bmm_chain_rows_tile_bytes<DT, B_KL, NW>(), NLD = TB / 1024 / NW;
  constexpr bool kSoftmax = INTER == kInterSoftmax;
  // a row's partial sum above which its reference exponent is raised
  constexpr float kLimit = Elem<T>::is_bf16 ? kSumLimitBf16 : kSumLimitF16;
  extern __shared__ __attribute__((aligned(1024))) char smem_rw[];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
  const int bz = lid / (unsigned)p.mblocks, m0 = (lid - bz * (unsigned)p.mblocks) * (16 * RT * NW) + 16 * RT * w;
  const BatchEntry be = batch_entry(p, bz);
  const T* __restrict__ Ag = reinterpret_cast<const T*>(p.a) + be.a;
  const T* const Bg = reinterpret_cast<const T*>(p.b) + be.b;
  const T* const Cg = reinterpret_cast<const T*>(p.c) + be.c;
  const int M = p.M, N = p.N, K = p.K, L = p.L;
  const bool busy = m0 < M;  // a wave without rows loads its share of the tiles and keeps the barriers

  // A fragments (operand column = row of A); with B stored [K][L] in the contraction order its transposing reads give.  Rows past
  // M repeat the last one, columns past K are loaded from column 0 and replaced by zeros.
  V8 af[RT][KS];
  // A goes through LDS, into the third tile's slot and what is kept behind it: loaded in the order the matrix instruction wants it
  // every lane's 16 bytes lie in another row, for each of which the address unit spends a cycle, and the first tile queues behind
  // (us per launch: 16 x 3328 x 144 x 128 without softmax 12.8 -> 10.4, 54 x 976 x 288 x 128 17.1 -> 14.9, packed 24 x 16 heads of 135 x
  // 80 14.4 -> 13.5).  Three workgroups of 64 columns to a compute unit cover one another's starts and do as well without the
  // detour (12 layers of [96 heads, 512 rows] 111.1 with it, 110.8 without).
  constexpr bool kStagedA = DT != 4 || NW != 4;
  if constexpr (kStagedA) {
    const unsigned a_lds = (unsigned)(size_t)(DITTO_LDS char*)smem_rw + 2 * TB + 1024 * S::A_LOADS * w;
#pragma unroll
    for (int i = 0; i < S::A_LOADS; ++i) {
      const int ch = 64 * i + lane, row = min(ch / S::A_CPR, 31), pc = ch - row * S::A_CPR, lc = S::SWZ ? pc ^ swz4m16_rows(row) : pc;
      lds_dma_16_from(Ag + (long long)min(m0 + row, M - 1) * p.a_rs + (8 * lc < K ? 8 * lc : 0), a_lds + 1024 * i);
    }
  } else {
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const T* const row = Ag + (long long)min(m0 + 16 * j + c, M - 1) * p.a_rs;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if constexpr (B_KL) {
          const int k = 32 * s + 4 * q;
          const V4 lo = *reinterpret_cast<const V4*>(row + (k < K ? k : 0)), hi = *reinterpret_cast<const V4*>(row + (k + 16 < K ? k + 16 : 0));
          const V4 none = {0, 0, 0, 0};
          af[j][s] = concat4<V4, V8>(k < K ? lo : none, k + 16 < K ? hi : none);
        } else {
          const int k = 32 * s + 8 * q;
          const V8 v = *reinterpret_cast<const V8*>(row + (k < K ? k : 0)), none = {0, 0, 0, 0, 0, 0, 0, 0};
          af[j][s] = k < K ? v : none;
        }
      }
    }
  }

  // the wave's direct loads of a tile: source offset of the lane's chunk, its first key within the tile (a key past L, like a
  // chunk past K or N, is asked for out of range and reads as zero)
  const int b_bytes = (int)((B_KL ? (long long)(K - 1) * p.b_rs + L : (long long)(L - 1) * p.b_rs + K) * 2);
  const int c_bytes = (int)(((long long)(L - 1) * p.c_rs + N) * 2);
  const i32x4 b_rsrc = make_rsrc(Bg, (unsigned)b_bytes), c_rsrc = make_rsrc(Cg, (unsigned)c_bytes);
  constexpr int kNever = 0x7fffffff;
  int voff[NLD], key[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int ld = NLD * w + i;
    if (ld < S::B_LOADS) {
      const int ch = 64 * ld + lane, row = ch / S::B_CPR, pc = ch - row * S::B_CPR;
      const int lc = B_KL ? pc ^ swz4m16_tr(row) : S::SWZ ? pc ^ swz4m16_rows(row) : pc;
      const bool in = B_KL ? row < K : row < kBN && 8 * lc < K;
      key[i] = !in ? kNever : B_KL ? 8 * lc : row;
      voff[i] = (row * p.b_rs + 8 * lc) * 2;
    } else {
      const int ch = 64 * (ld - S::B_LOADS) + lane, row = ch / S::C_CPR, pc = ch - row * S::C_CPR;
      const int lc = S::SWZ ? pc ^ swz4m16_tr(row) : pc;
      key[i] = row < kBN && 8 * lc < N ? row : kNever;
      voff[i] = (row * p.c_rs + 8 * lc) * 2;
    }
  }
  const unsigned lds_wave = (unsigned)(size_t)(DITTO_LDS char*)smem_rw + 1024 * NLD * w;
  auto load_tile = [&](int tile, int slot) __attribute__((always_inline)) {
    const int bo = tile * (kBN * 2) * (B_KL ? 1 : p.b_rs), co = tile * (kBN * 2) * p.c_rs, left = L - tile * kBN;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const bool is_b = NLD * w + i < S::B_LOADS;
      const int vo = key[i] < left ? voff[i] + (is_b ? bo : co) : kNever;
      lds_dma_16_at(is_b ? b_rsrc : c_rsrc, (unsigned)vo, lds_wave + slot * TB, 1024 * i);
    }
  };

  // LDS read addresses: B fragment of key tile kt (16 keys), k step s; C^T fragment of 32-key half h, column tile j
  const int tr_row = 4 * q + (c >> 2), tr_half = (c & 3) >> 1, tr_byte = 8 * (c & 1);
  constexpr int NBA = B_KL ? 4 : S::SWZ ? KS : 1, NCA = S::SWZ ? DT : 1;
  int b_ad[NBA], c_ad[NCA];
#pragma unroll
  for (int i = 0; i < NBA; ++i)
    b_ad[i] = B_KL     ? tr_row * 128 + (((2 * i + tr_half) ^ swz4m16_tr(tr_row)) * 16) + tr_byte
              : S::SWZ ? c * 128 + (((4 * i + q) ^ swz4m16_rows(c)) * 16)
                       : c * (S::B_CPR * 16) + q * 16;
#pragma unroll
  for (int j = 0; j < NCA; ++j)
    c_ad[j] = tr_row * (S::C_CPR * 16) + (S::SWZ ? (2 * j + tr_half) ^ swz4m16_tr(tr_row) : tr_half) * 16 + tr_byte + S::C_OFF;
  auto b_frag = [&](const char* tile, int kt, int s) __attribute__((always_inline)) -> V8 {
    if constexpr (B_KL) {
      const char* const a = tile + b_ad[kt % NBA] + 32 * s * 128;
      return concat4<V4, V8>(lds_read_tr4<T>(reinterpret_cast<const T*>(a)), lds_read_tr4<T>(reinterpret_cast<const T*>(a + 16 * 128)));
    } else {
      return *reinterpret_cast<const V8*>(tile + b_ad[s % NBA] + kt * 16 * (S::B_CPR * 16) + (S::SWZ ? 0 : s * 64));
    }
  };
  auto c_frag = [&](const char* tile, int h, int j) __attribute__((always_inline)) -> V8 {
    const char* const a = tile + c_ad[j % NCA] + 32 * h * (S::C_CPR * 16) + (S::SWZ ? 0 : j * 32);
    return concat4<V4, V8>(lds_read_tr4<T>(reinterpret_cast<const T*>(a)),
                           lds_read_tr4<T>(reinterpret_cast<const T*>(a + 16 * (S::C_CPR * 16))));
  };

  load_tile(0, 0);
  if constexpr (kStagedA) {
    load_tile(1, 1);
    // (the barrier in front of the third tile's loads waits for these reads)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NLD) : "memory");
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const int row = 16 * j + c, swz = S::SWZ ? swz4m16_rows(row) : 0;
      const char* const at = smem_rw + 2 * TB + 1024 * S::A_LOADS * w + row * (S::A_CPR * 16);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if constexpr (B_KL) {
          const int k = 32 * s + 4 * q, ch = 4 * s + (q >> 1);
          const V4 lo = *reinterpret_cast<const V4*>(at + (ch ^ swz) * 16 + 8 * (q & 1));
          const V4 hi = *reinterpret_cast<const V4*>(at + ((ch + 2) ^ swz) * 16 + 8 * (q & 1)), none = {0, 0, 0, 0};
          af[j][s] = concat4<V4, V8>(k < K ? lo : none, k + 16 < K ? hi : none);
        } else {
          const int k = 32 * s + 8 * q;
          const V8 v = *reinterpret_cast<const V8*>(at + ((4 * s + q) ^ swz) * 16), none = {0, 0, 0, 0, 0, 0, 0, 0};
          af[j][s] = k < K ? v : none;
        }
      }
    }
  } else {
    // the wait for A falls between the first and the second tile's loads
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(af[j][s]));
    load_tile(1, 1);
  }

  // accumulators of F^T: o[j][t][r] = F^T[16 t + 4 q + r][16 j + c]; ls: the row sums, by the matrix pipe against ones
  f32x4 o[RT][DT], ls[RT];
  float ref[RT];  // reference exponent of the lane's row (exp2 domain)
  V8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (T)1.0f;
  asm volatile("" : "+v"(ones));
  const float c2 = p.scale_log2;
  const int ntiles = (L + kBN - 1) / kBN;
  int* const flag = reinterpret_cast<int*>(smem_rw + bmm_chain_rows_lds<DT, B_KL, NW>() - 64);

  // One tile, its first NH halves of 32 keys (a last tile of at most 32 keys has one).
  auto tile_step = [&](int it, const char* tile, auto nh_c, auto safe_c) __attribute__((always_inline)) {
    constexpr int NH = decltype(nh_c)::value;
    constexpr bool SAFE = decltype(safe_c)::value;
    f32x4 s[RT][2 * NH];
#pragma unroll
    for (int st = 0; st < KS; ++st)
#pragma unroll
      for (int kt = 0; kt < 2 * NH; ++kt) {
        const V8 bf = b_frag(tile, kt, st);
#pragma unroll
        for (int j = 0; j < RT; ++j) s[j][kt] = Elem<T>::mfma16(bf, af[j][st], st == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[j][kt]);
      }
    if constexpr (kSoftmax) {
      if (it * kBN + 32 * NH > L) {
        const int left = L - it * kBN - 4 * q;  // keys left, counted from the lane's first
#pragma unroll
        for (int kt = 0; kt < 2 * NH; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int gone = (left - (16 * kt + r) - 1) >> 31;
#pragma unroll
            for (int j = 0; j < RT; ++j) s[j][kt][r] = neg_inf_where(s[j][kt][r], gone);
          }
      }
      if (SAFE || it == 0) {
        float mx[RT];
        bool raise = it == 0;
#pragma unroll
        for (int j = 0; j < RT; ++j) {
          mx[j] = s[j][0][0];
#pragma unroll
          for (int kt = 0; kt < 2 * NH; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[j] = fmaxf(mx[j], s[j][kt][r]);
          mx[j] *= c2;
          raise = raise || mx[j] > ref[j] + kLazy;
        }
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
          // the first tile sets the reference (nothing is accumulated yet); in the exact walk it then follows the running
          // maximum, lazily, and a first tile of scores of minus infinity alone leaves it at the lowest value (the optimistic
          // walk ends with a NaN sum on such a row: the test there would cost it 1 % at 2000 keys)
#pragma unroll
          for (int j = 0; j < RT; ++j) {
            const float m = quad_max(mx[j]);
            const float up = it > 0 ? fmaxf(ref[j], m) : SAFE ? fmaxf(kNoKeyYet, m) : m;
            const float alpha = it == 0 ? 1.f : __builtin_amdgcn_exp2f(ref[j] - up);
            ref[j] = up;
            ls[j] *= alpha;
#pragma unroll
            for (int t = 0; t < DT; ++t) o[j][t] *= alpha;
          }
        }
      }
    }
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      // element e of the operand is key 4 q + e of the half's first 16 (e < 4) or of its second; the sum is taken over the
      // rounded values, exactly what enters the product
      V8 pf[RT];
#pragma unroll
      for (int j = 0; j < RT; ++j) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          float x = s[j][2 * h + (e >> 2)][e & 3], y = s[j][2 * h + (e >> 2)][(e & 3) + 1];
          if constexpr (kSoftmax) {
            x = __builtin_amdgcn_exp2f(__builtin_fmaf(x, c2, -ref[j]));
            y = __builtin_amdgcn_exp2f(__builtin_fmaf(y, c2, -ref[j]));
          } else if (p.relu) {
            x = fmaxf(x, 0.f);
            y = fmaxf(y, 0.f);
          }
          const V2 two = cvt2<T>(x, y);
          pf[j][e] = two[0];
          pf[j][e + 1] = two[1];
        }
        if constexpr (kSoftmax) ls[j] = Elem<T>::mfma16(ones, pf[j], ls[j]);
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const V8 cf = c_frag(tile, h, t);
#pragma unroll
        for (int j = 0; j < RT; ++j) o[j][t] = Elem<T>::mfma16(cf, pf[j], o[j][t]);
      }
    }
    if constexpr (kSoftmax && !SAFE) {
      // optimistic walk: once per tile, lower the scale of a row whose sum has passed the limit (an infinite or NaN sum is
      // left as it is: that is what the end of the walk looks for)
      if (__builtin_amdgcn_ballot_w64(fmaxf(ls[0][0], ls[1][0]) > kLimit) != 0) {
#pragma unroll
        for (int j = 0; j < RT; ++j) {
          const float sum = ls[j][0];
          const int e = (sum > kLimit && sum < INFINITY) ? ((__builtin_bit_cast(int, sum) >> 23) & 255) - 127 : 0;
          const float alpha = __builtin_bit_cast(float, (127 - e) << 23);  // 2^-e, exact
          ref[j] += (float)e;
          ls[j] *= alpha;
#pragma unroll
          for (int t = 0; t < DT; ++t) o[j][t] *= alpha;
        }
      }
    }
  };

  // (tiles 0 and 1 are in flight: issued by the caller)
  auto walk = [&](auto safe_c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      ref[j] = 0.f;
      ls[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < DT; ++t) o[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int slot = 0;
    for (int it = 0; it < ntiles; ++it) {
      // tile `it` has landed (the next one's loads may stay in flight) and every wave is done with tile it - 1, whose slot
      // the loads below fill
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLD) : "memory");
      wg_sync();
      load_tile(it + 2, slot == 0 ? 2 : slot - 1);  // a tile past the last one: zeros
      const char* const tile = smem_rw + slot * TB;
      if (busy) {
        if (it * kBN + 32 < L) tile_step(it, tile, IntC<2>{}, safe_c);
        else tile_step(it, tile, IntC<1>{}, safe_c);
      }
      slot = slot == 2 ? 0 : slot + 1;
    }
    // no direct load still on its way into LDS, every wave done with the tiles
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (kSoftmax && !decltype(safe_c)::value) {
      // a sum that is not finite sends the workgroup through the exact walk (the tiles are its common property)
      // (by its bits: a comparison may be compiled as if there were no NaN)
      auto not_finite = [](float x) { return (__builtin_bit_cast(int, x) & 0x7f800000) == 0x7f800000; };
      const bool bad = busy && (not_finite(ls[0][0]) || not_finite(ls[1][0]));
      if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) *flag = 1;
    }
    wg_sync();
  };
  if (tid == 0) *flag = 0;
  walk(BoolC<false>{});
  if constexpr (kSoftmax) {
    if (__builtin_amdgcn_readfirstlane(*flag)) {
      load_tile(0, 0);
      load_tile(1, 1);
      walk(BoolC<true>{});
    }
  }
  if (!busy) return;

  // ---- normalise (softmax), cast, store the wave's 32 rows: 16-bit rows of whole 16-byte vectors through LDS (see
  // store_tile_rows), else 4 columns per lane from registers
  const bool by_rows = !p.out_f32 && (N & 7) == 0 && (p.f_rs & 7) == 0 && (p.f_bs & 7) == 0 && (p.f_bs2 & 7) == 0 &&
                       (reinterpret_cast<size_t>(p.f) & 15) == 0;  // wave-uniform
  constexpr int D = 16 * DT, kRowBytes = tile_row_bytes<D>();
  static_assert(NW * 16 * RT * kRowBytes <= NR * TB, "the parked rows need the staged tiles' LDS");
  static_assert(16 * RT * D / 8 % 64 == 0, "whole waves of 16-byte stores");
  char* const tw = smem_rw + w * (16 * RT * kRowBytes);
  const long long f0 = be.f + (long long)m0 * p.f_rs;
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    const float inv = kSoftmax ? 1.f / ls[j][0] : 1.f;
    if (!by_rows && m0 + 16 * j + c >= M) continue;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int n = 16 * t + 4 * q;
      f32x4 x = o[j][t] * inv;
      if (!kSoftmax && p.relu_out)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = fmaxf(x[r], 0.f);
      const V2 lo = cvt2<T>(x[0], x[1]), hi = cvt2<T>(x[2], x[3]);
      const V4 v = {lo[0], lo[1], hi[0], hi[1]};
      if (by_rows) {
        *reinterpret_cast<V4*>(tw + (16 * j + c) * kRowBytes + n * 2) = v;
      } else if (n < N) {
        const long long at = f0 + (long long)(16 * j + c) * p.f_rs + n;
        if (p.out_f32) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.f) + at) = x;
        else *reinterpret_cast<V4*>(reinterpret_cast<T*>(p.f) + at) = v;
      }
    }
  }
  if (by_rows) store_tile_rows<T, D, 16 * RT>(tw, reinterpret_cast<T*>(p.f) + f0, p.f_rs, M - m0, N, lane);
#else
  (void)p;
#endif
}

template <typename T, int DT, int NW, int INTER, bool B_KL, typename Args>
hipError_t launch_bmm_chain_rows(const Args& args, hipStream_t stream) {
  constexpr int lds = bmm_chain_rows_lds<DT, B_KL, NW>();
  auto kern = bmm_chain_rows_kernel<T, DT, NW, INTER, B_KL, Args>;
  static thread_local int configured_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)args.mblocks * (unsigned)args.batch), dim3(64 * NW), lds, stream, args);
  return hipGetLastError();
}

}  // namespace ditto
