// Fused two-contraction chain  F = epilogue(inter(A.B).C)  for fp16 / bf16 on few rows: a workgroup of eight waves owns
// 16 RT rows and its waves split the KEYS (the L axis): wave w takes the steps w, w + 8, ... of 32 keys, and the eight
// partial results of a row meet once, in LDS, at the end (with the softmax: each wave has its own reference exponent and
// sum).
//
// The other kernels give a workgroup 64 to 384 rows and walk all keys: with a dozen heads of a few hundred rows that is a
// few dozen workgroups on 256 compute units, each a chain of L / 64 steps of 0.8 us.  Here the chain is L / 256 steps, the
// rows spread over four to eight times as many compute units, and no wave waits for another before the merge: every wave
// loads its own 32 rows of B and of C into its own LDS (direct loads; the next step's B while the second product runs, the
// next C during the first), so the loop has no barrier.  The price is that a workgroup pulls all of B and C of its head for
// 16 or 32 rows, which is what bounds it from about a thousand keys on, and the merge (0.5 us per 16 rows at 128 columns).
// K and N are padded to 64, 80 or 128, not to powers of two.
//
// Measured, us per launch (2.4 of them the launch), other kernel -> this one: 16 x 176 x 176 x 80 8.4 -> 4.9,
// 8 x 461 x 461 x 80 12.7 -> 5.9, 2 x 2392 x 2392 x 80 38.5 -> 13.1, 2 x 4096 x 4096 x 128 60.9 -> 28.4,
// 8 x 512 x 2048 x 64 17.5 -> 8.8, the chain 1 x 512 x 256 x 64 without softmax 4.7 -> 4.05 (with its columns shared out the
// kernel takes 3.72 of 4.45 in a trace; the call, which the launch bounds, the same 4.1 - 4.3).
//
// Where two or more workgroups to a row block still leave each a compute unit, they share out the columns of F (CT of the DT
// tiles each) and repeat the first product: a workgroup then pulls all of B and its columns of C.  21 x 25 x 944 x 128 with softmax
// 8.8 -> 7.0 us (6.4 with A through LDS), 1 x 1463 x 2296 x 128 13.1 -> 10.5 (10.0), 1 x 710 x 1408 x 80 8.2 -> 7.2, 11 x 67 x 2128 x 64 7.05 -> 5.97.
#pragma once
#include "bmm_chain_fp.h"
#include "common.h"

namespace ditto {

constexpr int kSplitWaves = 8;

// LDS of one wave: a tile of 32 rows of C and one of B (32 keys), filled by direct loads of 64 16-byte chunks each.
// DT: column tiles of 16 that K and N are padded to; the contraction over K runs in steps of 32.
// CT: column tiles of C that the workgroup owns.
template <int DT, bool B_KL, int CT = DT>
struct SplitTiles {
  static constexpr int KS = (DT + 1) / 2;
  static constexpr bool POW2 = DT == 4 || DT == 8;
  static constexpr int C_CPR = 2 * CT;                       // chunks per row of the C tile
  static constexpr int C_LOADS = 32 * C_CPR / 64;
  // B stored [L][K]: rows of keys, KS * 32 columns; an odd number of chunks per row where the swizzle has no power of two
  // to work in.  B stored [K][L]: KS * 32 rows of 32 keys.
  static constexpr int B_CPR = B_KL ? 4 : POW2 ? 4 * KS : 4 * KS + 1;
  static constexpr int B_ROWS = B_KL ? 32 * KS : 32;
  static constexpr int B_LOADS = (B_ROWS * B_CPR + 63) / 64;
  static constexpr int C_OFF = B_LOADS * 1024;
  static constexpr int BYTES = C_OFF + C_LOADS * 1024;       // per wave
};
// The workgroup's rows of A on their way to its registers, behind the waves' tiles: rows as of a B stored [L][K].
template <int DT, int RT>
struct SplitRows {
  static constexpr int CPR = SplitTiles<DT, false>::B_CPR, LOADS = (16 * RT * CPR + 63) / 64;
  static_assert(LOADS <= kSplitWaves, "a wave brings 64 chunks");
};
inline int bmm_chain_split_rows_lds(int dt, int rt) {
  const int one = dt == 4 ? SplitRows<4, 1>::LOADS : dt == 5 ? SplitRows<5, 1>::LOADS : SplitRows<8, 1>::LOADS;
  const int two = dt == 4 ? SplitRows<4, 2>::LOADS : dt == 5 ? SplitRows<5, 2>::LOADS : SplitRows<8, 2>::LOADS;
  return 1024 * (rt == 1 ? one : two);
}
// LDS of a workgroup of ct of the column tiles of C: its waves' tiles, or the merge's partial results and their exponents and sums
inline int bmm_chain_split_lds(int dt, int ct, int rt, bool kl) {
  const int whole = (dt == 4   ? (kl ? SplitTiles<4, true>::BYTES : SplitTiles<4, false>::BYTES)
                                   : dt == 5 ? (kl ? SplitTiles<5, true>::BYTES : SplitTiles<5, false>::BYTES)
                                             : (kl ? SplitTiles<8, true>::BYTES : SplitTiles<8, false>::BYTES));
  const int tiles = kSplitWaves * (whole - 1024 * (dt - ct)) + bmm_chain_split_rows_lds(dt, rt), merge = kSplitWaves * 16 * rt * (16 * ct + 4 + 2) * 4;
  return tiles > merge ? tiles : merge;
}

template <typename T, int DT, int RT, int INTER, bool B_KL, typename Args, int CT = DT>
__global__ __launch_bounds__(64 * kSplitWaves) void bmm_chain_split_kernel(Args p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Elem<T>::v8 V8;
  typedef typename Elem<T>::v4 V4;
  typedef typename Elem<T>::v2 V2;
  typedef SplitTiles<DT, B_KL, CT> S;
  constexpr int KS = S::KS, ORS = 16 * CT + 4;
  constexpr bool kSoftmax = INTER == kInterSoftmax;
  // swizzles of the 16-byte chunks of a row: plain row reads (lanes = 16 rows), transposing reads (lanes = 4 rows x 32 bytes)
  auto swz_rows = [](int row) { return DT == 4 ? (row >> 1) & 7 : DT == 8 ? row & 15 : 0; };
  auto swz_tr = [](int row) { return CT == 2 ? 2 * ((row >> 2) & 1) : CT == 4 ? 2 * ((row >> 1) & 3) : CT == 8 ? 2 * (row & 7) : 0; };
  extern __shared__ __attribute__((aligned(1024))) char smem_sp[];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned lid = xcd_remap(blockIdx.x, gridDim.x);
  int col0 = 0;  // the workgroup's first column of F
  if constexpr (CT < DT) {
    const unsigned rows = lid / ((unsigned)(p.N + 16 * CT - 1) / (16u * CT));
    col0 = 16 * CT * (int)(lid - rows * ((unsigned)(p.N + 16 * CT - 1) / (16u * CT)));
    lid = rows;
  }
  const int bz = lid / (unsigned)p.mblocks, m0 = (lid - bz * (unsigned)p.mblocks) * 16 * RT;
  const BatchEntry be = batch_entry(p, bz);
  const T* __restrict__ Ag = reinterpret_cast<const T*>(p.a) + be.a;
  const T* const Bg = reinterpret_cast<const T*>(p.b) + be.b;
  const T* const Cg = reinterpret_cast<const T*>(p.c) + be.c;
  const int M = p.M, N = p.N, K = p.K, L = p.L;

  // A goes through LDS, each row fetched once: every wave needs all of them, and read by the rows the MFMA's lanes want every lane's
  // 16 bytes lie in another line, for each of which the address unit spends a cycle, in front of the first keys (20 x 304 x 752 x 128
  // with softmax 12.8 -> 10.1 us, 5 x 1248 x 624 x 128 12.6 -> 9.3, 2 x 77 x 77 x 128 4.7 -> 4.0, at 64 columns 0.95 of the time).  Rows past M
  // repeat the last one; columns past K are loaded from column 0 and replaced by zeros below.
  // Not 16 rows of 65 to 80 columns with B [L][K] and no softmax, whose short start the detour through LDS and the barrier make longer
  // by more than ten 16-byte pieces a row save: 53 x 133 x 372 x 80 8.49 us through LDS, 7.87 direct, 1 x 105 x 956 x 80 5.27 / 4.92; 175
  // random shapes 1.017 - 1.06 by keys (rows a packed tensor apart 0.95 - 1.00; with softmax 0.98 - 1.01, packed 0.94 - 0.97).
  constexpr bool kStagedA = !(DT == 5 && RT == 1 && !B_KL && !kSoftmax);
  typedef SplitRows<DT, RT> R;
  char* const rows_of_a = smem_sp + kSplitWaves * S::BYTES;
  if (kStagedA && w < R::LOADS) {
    const int ch = 64 * w + lane, row = min(ch / R::CPR, 16 * RT - 1), pc = ch - row * R::CPR, lc = S::POW2 ? pc ^ swz_rows(row) : pc;
    lds_dma_16_from(Ag + (long long)min(m0 + row, M - 1) * p.a_rs + (8 * lc < K ? 8 * lc : 0),
                    (unsigned)(size_t)(DITTO_LDS char*)rows_of_a + 1024 * w);
  }
  // A fragments (operand column = row of A); with B stored [K][L] in the contraction order its transposing reads give
  V8 af[RT][KS];
  if constexpr (!kStagedA) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int k = 32 * s + 8 * q;
        const V8 none = {0, 0, 0, 0, 0, 0, 0, 0};
        const V8 v = *reinterpret_cast<const V8*>(Ag + (long long)min(m0 + 16 * rt + c, M - 1) * p.a_rs + (k < K ? k : 0));
        af[rt][s] = k < K ? v : none;
      }
  }

  // source offsets of the lane's chunks relative to the step's first key; what is not there reads as zero (out of range)
  constexpr int kNone = -16;  // as an unsigned offset beyond any range
  const unsigned b_bytes = (unsigned)((B_KL ? (long long)(K - 1) * p.b_rs + L : (long long)(L - 1) * p.b_rs + K) * 2);
  const unsigned c_bytes = (unsigned)(((long long)(L - 1) * p.c_rs + N) * 2);
  int b_voff[S::B_LOADS], b_key[S::B_LOADS], c_voff[S::C_LOADS];
#pragma unroll
  for (int i = 0; i < S::B_LOADS; ++i) {
    const int ch = 64 * i + lane, row = ch / S::B_CPR, pc = ch - row * S::B_CPR;
    if constexpr (B_KL) {
      const int lc = pc ^ (2 * ((row >> 2) & 1));
      b_key[i] = 8 * lc;
      b_voff[i] = row < K ? (row * p.b_rs + 8 * lc) * 2 : kNone;
    } else {
      const int lc = S::POW2 ? pc ^ swz_rows(row) : pc;
      b_key[i] = 0;
      b_voff[i] = row < 32 && 8 * lc < K ? (row * p.b_rs + 8 * lc) * 2 : kNone;
    }
  }
#pragma unroll
  for (int i = 0; i < S::C_LOADS; ++i) {
    const int ch = 64 * i + lane, row = ch / S::C_CPR, lc = (ch - row * S::C_CPR) ^ swz_tr(row);
    c_voff[i] = col0 + 8 * lc < N ? (row * p.c_rs + col0 + 8 * lc) * 2 : kNone;
  }
  char* const tile = smem_sp + w * S::BYTES;
  const unsigned lds = (unsigned)(size_t)(DITTO_LDS char*)smem_sp + w * S::BYTES;
  const int nsteps = (L + 31) / 32;
  auto load_b = [&](int step) __attribute__((always_inline)) {
    const unsigned at = 64u * (unsigned)step * (B_KL ? 1u : (unsigned)p.b_rs);
    const i32x4 rsrc = make_rsrc_uniform(reinterpret_cast<const char*>(Bg) + at, step < nsteps ? b_bytes - at : 0u);
#pragma unroll
    for (int i = 0; i < S::B_LOADS; ++i) {
      int vo = b_voff[i];
      if (B_KL) vo = 32 * step + b_key[i] < L ? vo : kNone;  // keys past L lie inside the buffer (the next row)
      lds_dma_16_at(rsrc, (unsigned)vo, lds, 1024 * i);
    }
  };
  auto load_c = [&](int step) __attribute__((always_inline)) {
    const unsigned at = 64u * (unsigned)step * (unsigned)p.c_rs;
    const i32x4 rsrc = make_rsrc_uniform(reinterpret_cast<const char*>(Cg) + at, step < nsteps ? c_bytes - at : 0u);
#pragma unroll
    for (int i = 0; i < S::C_LOADS; ++i) lds_dma_16_at(rsrc, (unsigned)c_voff[i], lds, S::C_OFF + 1024 * i);
  };

  // LDS read addresses: B fragment of key tile kt, k step s; C fragment of column tile j
  const int tr_row = 4 * q + (c >> 2), tr_half = (c & 3) >> 1, tr_byte = 8 * (c & 1);
  auto b_frag = [&](int kt, int s) __attribute__((always_inline)) -> V8 {
    if constexpr (B_KL) {
      const char* const a = tile + (32 * s + tr_row) * 64 + (((2 * kt + tr_half) ^ (2 * (q & 1))) * 16) + tr_byte;
      return concat4<V4, V8>(lds_read_tr4<T>(reinterpret_cast<const T*>(a)), lds_read_tr4<T>(reinterpret_cast<const T*>(a + 16 * 64)));
    } else {
      const int row = 16 * kt + c, lc = 4 * s + q;
      return *reinterpret_cast<const V8*>(tile + row * S::B_CPR * 16 + (S::POW2 ? lc ^ swz_rows(c) : lc) * 16);
    }
  };
  auto c_frag = [&](int j) __attribute__((always_inline)) -> V8 {
    const char* const a = tile + S::C_OFF + tr_row * (16 * S::C_CPR) + (((2 * j + tr_half) ^ swz_tr(tr_row)) * 16) + tr_byte;
    return concat4<V4, V8>(lds_read_tr4<T>(reinterpret_cast<const T*>(a)),
                           lds_read_tr4<T>(reinterpret_cast<const T*>(a + 16 * 16 * S::C_CPR)));
  };

  f32x4 o[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < CT; ++j) o[rt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // softmax in the exp2 domain: a row's reference exponent is its maximum over the wave's first keys, raised when a later
  // score exceeds it by more than 2^kLazy; a wave whose keys so far all score minus infinity has none yet (it may be one of
  // eight that has met any key of the row)
  float ref[RT], lsum[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) ref[rt] = kNoKeyYet, lsum[rt] = 0.f;
  const float c2 = p.scale_log2;

  load_b(w);
  if constexpr (kStagedA) {
    load_c(w);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::B_LOADS + S::C_LOADS) : "memory");
    lds_barrier();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const char* const row = rows_of_a + (16 * rt + c) * (16 * R::CPR);
      const int swz = S::POW2 ? swz_rows(c) : 0;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if constexpr (B_KL) {
          const int k = 32 * s + 4 * q, ch = 4 * s + (q >> 1), half = 8 * (q & 1);
          const V4 lo = *reinterpret_cast<const V4*>(row + (ch ^ swz) * 16 + half), hi = *reinterpret_cast<const V4*>(row + ((ch + 2) ^ swz) * 16 + half);
          const V4 none = {0, 0, 0, 0};
          af[rt][s] = concat4<V4, V8>(k < K ? lo : none, k + 16 < K ? hi : none);
        } else {
          const int k = 32 * s + 8 * q;
          const V8 v = *reinterpret_cast<const V8*>(row + ((4 * s + q) ^ swz) * 16), none = {0, 0, 0, 0, 0, 0, 0, 0};
          af[rt][s] = k < K ? v : none;
        }
      }
    }
  } else {
    // the fragments are named between the first direct loads: the compiler's wait for them then falls here, once, and not at their
    // first use inside the loop, where it would wait for the prefetches as well
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(af[rt][s]));
    load_c(w);
  }
  for (int step = w; step < nsteps; step += kSplitWaves) {
    // this step's B tile has landed (its C tile, requested after it, may still be on its way)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::C_LOADS) : "memory");
    V8 bf[2][KS];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int s = 0; s < KS; ++s) bf[kt][s] = b_frag(kt, s);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    load_b(step + kSplitWaves);  // into the tile just read; past the end: zeros
    f32x4 st[RT][2];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          st[rt][kt] = Elem<T>::mfma16(bf[kt][s], af[rt][s], s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : st[rt][kt]);
    if constexpr (kSoftmax) {
      const int left = L - 32 * step - 4 * q;  // keys left, counted from the lane's first
      bool raise = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = st[rt][kt][r] * c2;
            if (32 * step + 32 > L) x = neg_inf_where(x, (left - (16 * kt + r) - 1) >> 31);
            st[rt][kt][r] = x;
            raise |= x > ref[rt] + kLazy;
          }
      if (__builtin_amdgcn_ballot_w64(raise) != 0) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          float mx = st[rt][0][0];
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[rt][kt][r]);
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          mx = fmaxf(mx, __shfl_xor(mx, 32));
          const float up = fmaxf(ref[rt], mx), alpha = __builtin_amdgcn_exp2f(ref[rt] - up);
          ref[rt] = up;
          lsum[rt] *= alpha;
#pragma unroll
          for (int j = 0; j < CT; ++j) o[rt][j] *= alpha;
        }
      }
    }
    // element e of the second operand is key 4 q + e of the first tile (e < 4) or of the second
    V8 pf[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          float x = st[rt][kt][r], y = st[rt][kt][r + 1];
          if constexpr (kSoftmax) {
            x = __builtin_amdgcn_exp2f(x - ref[rt]);
            y = __builtin_amdgcn_exp2f(y - ref[rt]);
          } else if (p.relu) {
            x = fmaxf(x, 0.f);
            y = fmaxf(y, 0.f);
          }
          const V2 two = cvt2<T>(x, y);
          if constexpr (kSoftmax) lsum[rt] = Elem<T>::add_pair(two, lsum[rt]);
          pf[rt][4 * kt + r] = two[0];
          pf[rt][4 * kt + r + 1] = two[1];
        }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::B_LOADS) : "memory");  // this step's C tile, not the next B tile
    V8 cf[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) cf[j] = c_frag(j);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    load_c(step + kSplitWaves);
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) o[rt][j] = Elem<T>::mfma16(cf[j], pf[rt], o[rt][j]);
  }

  // ---- the eight partial results of a row meet in LDS (no direct load may still be on its way into it)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  wg_sync();
  float* const Om = reinterpret_cast<float*>(smem_sp);          // [wave][16 RT][ORS]
  float* const Ml = Om + kSplitWaves * 16 * RT * ORS;           // [wave][16 RT][reference exponent, sum]
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float* const row = Om + (w * 16 * RT + 16 * rt + c) * ORS + 4 * q;
#pragma unroll
    for (int j = 0; j < CT; ++j) *reinterpret_cast<f32x4*>(row + 16 * j) = o[rt][j];
    if constexpr (kSoftmax) {
      float s = lsum[rt];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (q == 0) {
        Ml[2 * (w * 16 * RT + 16 * rt + c)] = ref[rt];
        Ml[2 * (w * 16 * RT + 16 * rt + c) + 1] = s;
      }
    }
  }
  wg_sync();
  const long long f0 = be.f;
  for (int e = tid; e < 16 * RT * 4 * CT; e += 64 * kSplitWaves) {
    const int row = e / (4 * CT), n0 = 4 * (e - row * 4 * CT);
    float wt[kSplitWaves];
    if constexpr (kSoftmax) {
      float mx = kNoKeyYet, s = 0.f;
#pragma unroll
      for (int i = 0; i < kSplitWaves; ++i) mx = fmaxf(mx, Ml[2 * (i * 16 * RT + row)]);
#pragma unroll
      for (int i = 0; i < kSplitWaves; ++i) {
        wt[i] = __builtin_amdgcn_exp2f(Ml[2 * (i * 16 * RT + row)] - mx);
        s += wt[i] * Ml[2 * (i * 16 * RT + row) + 1];
      }
      const float inv = 1.f / s;
#pragma unroll
      for (int i = 0; i < kSplitWaves; ++i) wt[i] *= inv;
    }
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kSplitWaves; ++i) {
      const f32x4 part = *reinterpret_cast<const f32x4*>(Om + (i * 16 * RT + row) * ORS + n0);
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = kSoftmax ? __builtin_fmaf(wt[i], part[t], x[t]) : x[t] + part[t];
    }
    if (p.relu_out)
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = fmaxf(x[t], 0.f);
    if (m0 + row < M && col0 + n0 < N) {  // N is a multiple of 8
      const long long at = f0 + (long long)(m0 + row) * p.f_rs + col0 + n0;
      if (p.out_f32) {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.f) + at) = x;
      } else {
        const V2 lo = cvt2<T>(x[0], x[1]), hi = cvt2<T>(x[2], x[3]);
        *reinterpret_cast<V4*>(reinterpret_cast<T*>(p.f) + at) = V4{lo[0], lo[1], hi[0], hi[1]};
      }
    }
  }
#else
  (void)p;
#endif
}

template <typename T, int DT, int RT, int INTER, bool B_KL, int CT = DT, typename Args>
hipError_t launch_bmm_chain_split(const Args& args, hipStream_t stream) {
  const int lds = bmm_chain_split_lds(DT, CT, RT, B_KL);
  auto kern = bmm_chain_split_kernel<T, DT, RT, INTER, B_KL, Args, CT>;
  static thread_local int configured_dev = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  const unsigned cols = CT == DT ? 1u : (unsigned)(args.N + 16 * CT - 1) / (16u * CT);
  hipLaunchKernelGGL(kern, dim3((unsigned)args.mblocks * (unsigned)args.batch * cols), dim3(64 * kSplitWaves), lds, stream, args);
  return hipGetLastError();
}

}  // namespace ditto
