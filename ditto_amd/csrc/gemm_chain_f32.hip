// fp32 / fp64 GEMM -> cast|relu|softmax -> GEMM chain  F = inter(A.B).C  for the reference's fp32 configurations
// (python_test/auto_tensorize/test_hyper_fusion.py:16-21: 512x64 . 64x64 . 64x64; the fp32 BMM -> softmax -> BMM of
// benchmark/chimera/cpu/bmm_softmax_bmm.py:64-170) and its ("80", "float64", "float64") row
// (benchmark/chimera/cuda/bmm_bmm_cuda.py:273-288).
//
// fp32: gemm_chain_f32_kernel below, on v_mfma_f32_16x16x4_f32.  fp64: plain FMAs over LDS tiles
// (gemm_chain_f64_kernel), the arithmetic type the matrix cores' fp32 path does not cover.
#include "common.h"
#include "gemm_chain_f32.h"

namespace ditto {

namespace {
constexpr int kMaxD = 128;
constexpr int kWaves = 8;  // waves of an fp32 workgroup: they split the keys
constexpr unsigned kLaunchBlocks = 1u << 22;  // most fp32 workgroups of one launch
}

// ---- fp32 ------------------------------------------------------------------------------------
// A workgroup owns 16 * RT rows of A; its eight waves split L: wave w takes the steps w, w + 8, ... of 16 keys, and the
// eight partial results of a row meet once, in LDS, at the end (with the softmax: each wave has its own reference
// exponent and sum).  Sixteen rows of one head are too little work for eight waves any other way, and at the sizes
// this type is used at (6144 rows in all on 256 compute units) splitting the rows alone leaves most SIMDs idle.
//
// With S^T = B^T.A^T on the 16x16x4 MFMA a lane (c = lane % 16, q = lane / 16)
// ends with keys 4q + r, r = 0..3, of row c, which is operand r of a second contraction over the four keys
// {4q + r : q}: F^T = C^T.P^T takes the probabilities where they are.  The contraction index of either product may run
// in any order both operands agree on, so every operand is loaded as 16-byte pieces of its own rows straight from
// memory: k = 16 s + 4 q + t is k step (s, t) of the first product, and column n = 64 g + 4 c + t is output tile (g, t) of
// the second.  K fragments are fetched during the second product of the step before, V fragments during the first.
//
// Bound: the fp32 matrix pipe (256 flop per cycle and compute unit) from a few rounds of workgroups on, the chain of
// first loads, steps and merge below that.  12 x 512 x 512 x 64 (BERT-base, batch 1), softmax: 13.7 us per launch,
// 59 TFLOP/s: 192 workgroups leave a quarter of the compute units idle, the others' matrix pipes are busy for 6.8 us of the
// 11 beyond the launch, LDS hardly, and the rest goes to waits for loads (56 MB out of L2).  The plain
// fp32 FMAs over LDS tiles that this kernel replaced took 178 us (one row per eight threads, an LDS read per operand of
// every FMA); 64 x 512 x 512 x 64: 49.4 us, 87 TFLOP/s; 4 x 1024 x 1024 x 128: 26.1 us, 82 TFLOP/s.
//
// With few rows the matrix pipes of a few compute units are the bound and the others idle: workgroups then own W = 64, 32 or 16
// of the columns of F as well (0: all), computing the first product once each, 8 DT MFMAs a step down to 4 DT + W / 4: softmax
// 3 x 132 x 756 x 80 13.5 -> 9.8 us, 11 x 79 x 609 x 128 19.5 -> 15.7 (12.5 with the trip through LDS below), 1 x 180 x 387 x 80 8.9 -> 7.0.  As narrow as leaves every
// workgroup a compute unit: beyond that the repeated first products cost what the others save.
// DT: column tiles of 16 that K and N are padded to.  EXACT: K = N = 16 DT and every row starts on a 16-byte boundary;
// otherwise elements are loaded one by one and columns past K or N are zeros.
//
// EXACT, 64 or 128 columns, but for f32_direct: A and, with B stored [L][K], the steps' keys come through LDS.  Fetched the way the MFMA wants them, every
// lane's 16 bytes lie in another row, and the address unit, which takes four lanes at a time and spends a cycle on every line they
// touch, was busy for 14 thousand of the 27 thousand cycles of 12 x 512 x 512 x 64; rows end to end take a quarter of that.  us per
// launch before / here: 12 x 512 x 512 x 64 14.9 / 14.3, 8 x 627 x 61 x 64 5.7 / 5.0, 1 x 729 x 995 x 128 21.2 / 18.2, 5 x 1009 x 341
// x 128 without softmax 23.9 / 19.9 (B [K][L] 24.4 / 21.8), 7 x 337 x 139 x 128 8.7 / 7.4.  At 80 columns the trip through LDS costs what it saves (8.2 / 8.4
// at 5 x 761 x 396, 9.7 / 10.2 at 3 x 132 x 756).  A row is CPR 16-byte chunks in LDS, swizzled by its index so that sixteen rows
// are read without bank conflicts and every four lanes of a load still fetch 64 bytes end to end.  A wave's keys lie in front of
// its partial results (one or the other is there); A is the workgroup's.
template <int DT, int RT, int W>
struct F32Lds {
  static constexpr int CPR = 4 * DT;
  static constexpr int K_LOADS = DT == 5 ? 0 : 16 * CPR / 64, Q_LOADS = RT * K_LOADS;  // of 64 chunks
  static constexpr int ORS = (W ? W : 16 * DT) + 4;  // row stride of a parked partial result, floats
  static constexpr int WAVE = 1024 * K_LOADS > 64 * RT * ORS ? 256 * K_LOADS : 16 * RT * ORS;  // floats of one wave
  static constexpr int SUMS = kWaves * WAVE, AGAIN = SUMS + kWaves * 16 * RT * 2, Q = AGAIN + 4;  // at these floats
  static constexpr int BYTES = 4 * Q + 1024 * Q_LOADS;
  static __device__ int swz(int row) { return row & 15; }
};

// Waves of a SIMD that the compiler is held to where its own choice misses them by a few registers: two workgroups of eight waves to
// a compute unit need 128, and two exact row tiles of 64 columns without softmax, B [L][K], take 130 since their rows come through
// LDS.  us per launch at 130 / 128: 73 x 1022 x 75 40.3 / 30.9, 44 x 1346 x 169 43.9 / 36.7, 52 x 1057 x 599 96.3 / 86.7; on 50 random shapes
// 0.88 in the mean, the worst 1.027 (0.92 and 1.006 of what the kernel took without the trip through LDS).
constexpr int f32_min_waves(int DT, int RT, bool EXACT, bool KL, bool SM) { return DT == 4 && RT == 2 && EXACT && !KL && !SM ? 4 : 1; }
// DIRECT: for chains that f32_direct names, nothing but the merge through LDS.
template <int DT, int RT, bool EXACT, bool KL, bool SM, int W, bool DIRECT>
__global__ __launch_bounds__(64 * kWaves, f32_min_waves(DT, RT, EXACT, KL, SM)) void gemm_chain_f32_kernel(F32ChainArgs p) {
  constexpr int PW = W == 0 || W == 64 ? 4 : W / 16;                   // columns of a lane's piece of a row
  constexpr int G = W == 0 ? DT / 4 : 1, REM = W == 0 ? DT % 4 : 0;  // column groups of 16 PW, column tiles beyond them
  constexpr int NT = PW * G + REM;                                     // column tiles of the workgroup
  typedef F32Lds<DT, RT, W> S;
  constexpr int ORS = S::ORS;
  constexpr bool kStagedA = EXACT && DT != 5 && !DIRECT, kStaged = kStagedA && !KL;
  static_assert(ORS == 16 * NT + 4, "the columns of a workgroup");
  typedef __attribute__((ext_vector_type(PW == 1 ? 2 : PW))) float Piece;
  static_assert(REM <= 1, "columns beyond the groups of 64: at most one tile of 16");
  extern __shared__ __attribute__((aligned(16))) float smem_f32[];
  float* const Om = smem_f32;              // [wave], 16 RT rows of ORS
  float* const Ml = smem_f32 + S::SUMS;    // [wave][16 RT][reference exponent, sum]
  int* const again = reinterpret_cast<int*>(smem_f32 + S::AGAIN);  // a result is not finite
  const int K = p.K, N = p.N, L = p.L, M = p.M;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  // (wave-uniform for the staged loads' sake: the others lose 2 % by what the compiler then makes of their addresses)
  const int wu = __builtin_amdgcn_readfirstlane(tid >> 6), w = kStaged ? wu : tid >> 6;
  unsigned bid = p.block0 + xcd_remap(blockIdx.x, gridDim.x);  // the row blocks of a batch entry read the same B and C
  int col0 = 0;  // the workgroup's first column
  if constexpr (W > 0) {
    const unsigned rows = bid / (unsigned)p.col_blocks;
    col0 = W * (int)(bid - rows * (unsigned)p.col_blocks);
    bid = rows;
  }
  const int bz = bid / (unsigned)p.mblocks, m0 = (bid - bz * (unsigned)p.mblocks) * 16 * RT;
  const float* const Ag = static_cast<const float*>(p.a) + (long long)bz * p.a_bs;
  const float* const Bg = static_cast<const float*>(p.b) + (long long)bz * p.b_bs;
  const float* const Cg = static_cast<const float*>(p.c) + (long long)bz * p.c_bs;
  float* const Fg = static_cast<float*>(p.f) + (long long)bz * p.f_bs;

  // columns k0 .. k0 + 3 of a row, zeros from `n` on
  auto load4 = [](const float* row, int k0, int n) -> f32x4 {
    if constexpr (EXACT) return *reinterpret_cast<const f32x4*>(row + k0);
    f32x4 v;
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = k0 + t < n ? row[k0 + t] : 0.f;
    return v;
  };

  const int nsteps = (L + 15) / 16;
  f32x4 kf[DT], qf[RT][DT], vf[4][G + REM], o[RT][NT];
  const unsigned lds0 = (unsigned)(size_t)(DITTO_LDS char*)smem_f32;
  const float* const own = smem_f32 + w * S::WAVE;  // the wave's keys
  // chunk `ch` of the rows from `first` on (`last` stands for those behind it) to LDS
  auto stage = [&](const float* base, long long rs, int ch, int first, int last, unsigned to) __attribute__((always_inline)) {
    const int row = ch / S::CPR, lc = (ch - row * S::CPR) ^ S::swz(row);
    lds_dma_16_from(base + (long long)min(first + row, last) * rs + 4 * lc, to);
  };
  auto load_k = [&](int step) __attribute__((always_inline)) {
    const int key = min(16 * step + c, L - 1);  // keys past the last are masked below
    if constexpr (kStaged) {
#pragma unroll
      for (int i = 0; i < S::K_LOADS; ++i) stage(Bg, p.b_rs, 64 * i + lane, 16 * step, L - 1, lds0 + 4 * w * S::WAVE + 1024 * i);
      return;
    }
#pragma unroll
    for (int s = 0; s < DT; ++s) {
      if constexpr (KL) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int k = 16 * s + 4 * q + t;
          kf[s][t] = EXACT || k < K ? Bg[(long long)k * p.b_rs + key] : 0.f;
        }
      } else {
        kf[s] = load4(Bg + (long long)key * p.b_rs, 16 * s + 4 * q, K);
      }
    }
  };
  // A step's next keys, once these are in registers.  The wait for the step's rows of C is theirs as well, so they are asked for
  // close to those: in front of them at 128 columns (5 x 1009 x 341 19.9 us, 20.4 behind), behind them at 64 (1 x 512 x 512 7.2, 7.35).
  constexpr bool kNextFirst = DT == 8;
  auto load_next = [&](int step) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (step < nsteps) load_k(step);
  };
  if (!kStaged && w < nsteps) load_k(w);
  if constexpr (kStagedA)
    for (int i = wu; i < S::Q_LOADS; i += kWaves) stage(Ag, p.a_rs, 64 * i + lane, m0, M - 1, lds0 + 4 * S::Q + 1024 * i);
  if (kStaged && w < nsteps) load_k(w);
  if constexpr (kStagedA) {
    if (kStaged && w < nsteps)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::K_LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float* const row = Ag + (long long)min(m0 + 16 * rt + c, M - 1) * p.a_rs;
#pragma unroll
    for (int s = 0; s < DT; ++s) {
      if constexpr (kStagedA)
        qf[rt][s] = *reinterpret_cast<const f32x4*>(smem_f32 + S::Q + 4 * ((16 * rt + c) * S::CPR + ((4 * s + q) ^ S::swz(c))));
      else
        qf[rt][s] = load4(row, 16 * s + 4 * q, K);
    }
  }
  // Softmax in the exp2 domain: a row's reference exponent is its maximum over the wave's first keys, raised only when a
  // later score exceeds it by 2^slack; none yet while the wave's keys all score minus infinity.  Weights of up to 2^20 are
  // no loss but at the end of the range of C: a workgroup with a result that is not finite walks the keys once more with
  // weights of at most one (raising at any excess in the first place waits for the accumulators at every step: 14.4 -> 14.8 us
  // at 12 x 512 x 512 x 64, 4 % at 1000 keys; a reference a few orders above the maximum costs 2 % of the accuracy).
  const float c2 = p.softmax_scale * 1.4426950408889634f;
  float ref[RT], lsum[RT], slack = SM ? 20.f : 0.f;
  if (SM && tid == 0) *again = 0;

  for (;;) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      ref[rt] = kNoKeyYet, lsum[rt] = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) o[rt][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    for (int step = w; step < nsteps; step += kWaves) {
      const int key0 = 16 * step;
      if constexpr (kStaged) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int s = 0; s < DT; ++s) kf[s] = *reinterpret_cast<const f32x4*>(own + 4 * (c * S::CPR + ((4 * s + q) ^ S::swz(c))));
        if (kNextFirst) load_next(step + kWaves);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* const row = Cg + (long long)min(key0 + 4 * q + r, L - 1) * p.c_rs;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int n = col0 + 16 * PW * g + PW * c;
          if constexpr (PW == 4) {
            vf[r][g] = load4(row, n, N);
          } else if constexpr (PW == 2 && EXACT) {
            const Piece two = *reinterpret_cast<const Piece*>(row + n);
            vf[r][g][0] = two[0], vf[r][g][1] = two[1];
          } else {
#pragma unroll
            for (int t = 0; t < PW; ++t) vf[r][g][t] = EXACT || n + t < N ? row[n + t] : 0.f;
          }
        }
        if constexpr (REM > 0) vf[r][G][0] = EXACT || 64 * G + c < N ? row[64 * G + c] : 0.f;
      }
      if (kStaged && !kNextFirst) load_next(step + kWaves);
      f32x4 st[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) st[rt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DT; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            st[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s][t], qf[rt][s][t], st[rt], 0, 0, 0);
      if (!kStaged && step + kWaves < nsteps) load_k(step + kWaves);
      const bool tail = key0 + 16 > L;
      if constexpr (SM) {
        bool raise = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            st[rt][r] *= c2;
            if (tail && key0 + 4 * q + r >= L) st[rt][r] = -INFINITY;
            raise |= st[rt][r] > ref[rt] + slack;
          }
        }
        if (__any(raise)) {
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            float mx = fmaxf(fmaxf(st[rt][0], st[rt][1]), fmaxf(st[rt][2], st[rt][3]));
            mx = quad_max(mx);
            const float up = fmaxf(ref[rt], mx), alpha = exp2f(ref[rt] - up);
            ref[rt] = up;
            lsum[rt] *= alpha;
#pragma unroll
            for (int j = 0; j < NT; ++j) o[rt][j] *= alpha;
          }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            st[rt][r] = __builtin_amdgcn_exp2f(st[rt][r] - ref[rt]);
            lsum[rt] += st[rt][r];
          }
      } else {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (p.relu) st[rt][r] = fmaxf(st[rt][r], 0.f);
            if (tail && key0 + 4 * q + r >= L) st[rt][r] = 0.f;
          }
      }
      if (tail) {  // the clamped rows stand for nothing, whatever the last row holds
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int g = 0; g < G + REM; ++g)
            if (key0 + 4 * q + r >= L) vf[r][g] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            o[rt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][j / PW][j % PW], st[rt][r], o[rt][j], 0, 0, 0);
    }

    // lane (c, q) holds of row c: columns PW (16 g + 4 q + r) + t in register r of tile PW g + t, and 64 G + 4 q + r in the last
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float* const row = Om + w * S::WAVE + (16 * rt + c) * ORS;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if constexpr (PW == 1) {
          *reinterpret_cast<f32x4*>(row + 16 * g + 4 * q) = o[rt][g];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            Piece piece;
#pragma unroll
            for (int t = 0; t < PW; ++t) piece[t] = o[rt][PW * g + t][r];
            *reinterpret_cast<Piece*>(row + PW * (16 * g + 4 * q + r)) = piece;
          }
        }
      }
      if constexpr (REM > 0) *reinterpret_cast<f32x4*>(row + 64 * G + 4 * q) = o[rt][4 * G];
      if constexpr (SM) {
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
    bool bad = false;
    for (int e = tid; e < 16 * RT * 4 * NT; e += 64 * kWaves) {
      const int row = e / (4 * NT), n0 = 4 * (e - row * 4 * NT);
      float wt[kWaves];
      if constexpr (SM) {
        float mx = kNoKeyYet, s = 0.f;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) mx = fmaxf(mx, Ml[2 * (i * 16 * RT + row)]);
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
          wt[i] = exp2f(Ml[2 * (i * 16 * RT + row)] - mx);
          s += wt[i] * Ml[2 * (i * 16 * RT + row) + 1];
        }
        const float inv = 1.f / s;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) wt[i] *= inv;
      } else {
#pragma unroll
        for (int i = 0; i < kWaves; ++i) wt[i] = 1.f;
      }
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kWaves; ++i) {
        const f32x4 part = *reinterpret_cast<const f32x4*>(Om + i * S::WAVE + row * ORS + n0);
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = __builtin_fmaf(wt[i], part[t], x[t]);
      }
      if (p.relu_out)
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = fmaxf(x[t], 0.f);
      if (m0 + row < M) {
        float* const dst = Fg + (long long)(m0 + row) * p.f_rs + col0 + n0;
        if constexpr (EXACT) {
          *reinterpret_cast<f32x4*>(dst) = x;
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (col0 + n0 + t < N) dst[t] = x[t];
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) bad |= (__builtin_bit_cast(int, x[t]) & 0x7f800000) == 0x7f800000;
    }
    if (!SM || slack == 0.f) return;
    if (__any(bad) && lane == 0) *again = 1;
    wg_sync();
    if (*again == 0) return;
    slack = 0.f;
    if (w < nsteps) load_k(w);
  }
}

// ---- fp64 ------------------------------------------------------------------------------------
// A workgroup owns 32 rows of A for one batch entry, walks L in tiles of 32, keeps the 32x32 intermediate tile in LDS and
// its 32xN slice of F in registers.  Sums run over k, then l, in ascending order.  Softmax is the online form over the tiles
// of L: the eight threads of a row share its running maximum (exchanged by lane shuffles), each keeps the sum of its own
// probabilities, and the row's slice of F is rescaled when the maximum rises.
namespace {
constexpr int kBM = 32, kBL = 32;
}

static int f64_chain_lds_bytes(int K, int N) {
  return (kBM * (K + 1) + K * (kBL + 1) + kBL * (N + 1) + kBM * (kBL + 1)) * (int)sizeof(double);
}

__global__ __launch_bounds__(256) void gemm_chain_f64_kernel(F32ChainArgs p) {
  extern __shared__ __attribute__((aligned(16))) double smem_f64[];
  const int K = p.K, N = p.N, L = p.L, M = p.M;
  double* As = smem_f64;             // [32][K+1]
  double* Bs = As + kBM * (K + 1);   // [K][kBL+1]
  double* Cs = Bs + K * (kBL + 1);   // [kBL][N+1]
  double* Ms = Cs + kBL * (N + 1);   // [32][kBL+1]
  const int tid = threadIdx.x;
  const int mb = blockIdx.x % p.mblocks, bz = blockIdx.x / p.mblocks;
  const int m0 = mb * kBM;
  const double* Ag = static_cast<const double*>(p.a) + (long long)bz * p.a_bs;
  const double* Bg = static_cast<const double*>(p.b) + (long long)bz * p.b_bs;
  const double* Cg = static_cast<const double*>(p.c) + (long long)bz * p.c_bs;
  double* Fg = static_cast<double*>(p.f) + (long long)bz * p.f_bs;

  for (int e = tid; e < kBM * K; e += 256) {
    const int r = e / K, k = e % K;
    As[r * (K + 1) + k] = m0 + r < M ? Ag[(long long)(m0 + r) * p.a_rs + k] : 0.0;
  }
  const int r = tid >> 3, c8 = tid & 7;  // this thread's row and its column phase
  double acc[kMaxD / 8];
#pragma unroll
  for (int i = 0; i < kMaxD / 8; ++i) acc[i] = 0.0;

  double mrow = -INFINITY, lsum = 0.0;  // softmax: running maximum (exp2 domain), this thread's share of the row sum
  const double c2 = (double)p.softmax_scale * 1.4426950408889634;

  for (int l0 = 0; l0 < L; l0 += kBL) {
    __syncthreads();
    for (int e = tid; e < K * kBL; e += 256) {
      // consecutive threads read along the contiguous axis of B
      const int k = p.b_lk ? e % K : e / kBL, l = p.b_lk ? e / K : e % kBL;
      double v = 0.0;
      if (l0 + l < L) v = p.b_lk ? Bg[(long long)(l0 + l) * p.b_rs + k] : Bg[(long long)k * p.b_rs + l0 + l];
      Bs[k * (kBL + 1) + l] = v;
    }
    for (int e = tid; e < kBL * N; e += 256) {
      const int l = e / N, n = e % N;
      Cs[l * (N + 1) + n] = l0 + l < L ? Cg[(long long)(l0 + l) * p.c_rs + n] : 0.0;
    }
    __syncthreads();
    double sv[kBL / 8];
#pragma unroll
    for (int j = 0; j < kBL / 8; ++j) {
      const int l = c8 + 8 * j;
      double s = 0.0;
      for (int k = 0; k < K; ++k) s = __builtin_fma(As[r * (K + 1) + k], Bs[k * (kBL + 1) + l], s);
      if (p.relu) s = fmax(s, 0.0);
      sv[j] = s;
    }
    if (p.softmax) {
      double mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < kBL / 8; ++j) {
        sv[j] = l0 + c8 + 8 * j < L ? sv[j] * c2 : (double)-INFINITY;  // keys past L take no part
        mx = fmax(mx, sv[j]);
      }
      // the row's eight threads are eight consecutive lanes
      mx = fmax(mx, __shfl_xor(mx, 1));
      mx = fmax(mx, __shfl_xor(mx, 2));
      mx = fmax(mx, __shfl_xor(mx, 4));
      const double mnew = fmax(mrow, mx);  // finite: every tile holds at least one key
      const double alpha = exp2(mrow - mnew);
      mrow = mnew;
      lsum *= alpha;
#pragma unroll
      for (int i = 0; i < kMaxD / 8; ++i) acc[i] *= alpha;
#pragma unroll
      for (int j = 0; j < kBL / 8; ++j) {
        sv[j] = exp2(sv[j] - mnew);
        lsum += sv[j];
      }
    }
#pragma unroll
    for (int j = 0; j < kBL / 8; ++j) Ms[r * (kBL + 1) + c8 + 8 * j] = sv[j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMaxD / 8; ++i) {
      const int n = c8 + 8 * i;
      if (n < N) {
        double s = acc[i];
        for (int l = 0; l < kBL; ++l) s = __builtin_fma(Ms[r * (kBL + 1) + l], Cs[l * (N + 1) + n], s);
        acc[i] = s;
      }
    }
  }
  double inv = 1.0;
  if (p.softmax) {
    lsum += __shfl_xor(lsum, 1);
    lsum += __shfl_xor(lsum, 2);
    lsum += __shfl_xor(lsum, 4);
    inv = 1.0 / lsum;
  }
  if (m0 + r < M) {
#pragma unroll
    for (int i = 0; i < kMaxD / 8; ++i) {
      const int n = c8 + 8 * i;
      if (n < N) Fg[(long long)(m0 + r) * p.f_rs + n] = p.relu_out ? fmax(acc[i] * inv, 0.0) : acc[i] * inv;
    }
  }
}

// ---- launch ----------------------------------------------------------------------------------
int f32_chain_max_dim() { return kMaxD; }

static int f32_tiles(int K, int N) {  // column tiles of 16 the fp32 kernel is built for
  const int d = K > N ? K : N;
  return d <= 64 ? 4 : d <= 80 ? 5 : 8;
}
template <int DT, int RT>
static int f32_lds_bytes(int width) {
  return width == 16 ? F32Lds<DT, RT, 16>::BYTES : width == 32 ? F32Lds<DT, RT, 32>::BYTES : width == 64 ? F32Lds<DT, RT, 64>::BYTES : F32Lds<DT, RT, 0>::BYTES;
}
int f32_chain_lds_bytes_host(int K, int N, int f64, int rt, int width) {
  if (f64) return f64_chain_lds_bytes(K, N);
  const int dt = f32_tiles(K, N);
  if (rt == 2) return dt == 4 ? f32_lds_bytes<4, 2>(width) : f32_lds_bytes<5, 2>(width);
  return dt == 4 ? f32_lds_bytes<4, 1>(width) : dt == 5 ? f32_lds_bytes<5, 1>(width) : f32_lds_bytes<8, 1>(width);
}
bool f32_chain_exact(int K, int N, long long strides) {
  const int columns = 16 * f32_tiles(K, N);
  return K == columns && N == columns && strides % 4 == 0;
}
// The columns a workgroup owns, 0 for all: the fewest that leave every workgroup a compute unit of its own.
int f32_chain_width(int K, int N, long long row_blocks, int cus) {
  const int dt = f32_tiles(K, N);
  for (int w = 16; w <= 64; w *= 2)
    if (w < 16 * dt && (dt != 5 || w == 16) && row_blocks * ((N + w - 1) / w) <= cus) return w;
  return 0;
}

template <typename Tag, typename Kernel>
static hipError_t launch_with_lds(Kernel kernel, unsigned threads, int lds, const F32ChainArgs& args, hipStream_t stream) {
  static thread_local int configured_dev = -1;  // one per kernel (Tag names it), device and thread
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (configured_dev != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    configured_dev = dev;
  }
  // A launch holds fewer than 2^32 work items, which sixteen rows per 512 threads reach at 134 million rows: such a grid goes
  // out in pieces (the fp64 kernel's 256 threads own 32 rows; it takes what one launch holds).
  const unsigned long long blocks = (unsigned long long)args.mblocks * (unsigned long long)args.batch * (unsigned)(args.f64 ? 1 : args.col_blocks);
  if (blocks > 0x7fffffffull) return hipErrorInvalidConfiguration;
  const unsigned long long most = args.f64 ? blocks : kLaunchBlocks;
  F32ChainArgs piece = args;
  for (unsigned long long at = 0; at < blocks && e == hipSuccess; at += most) {
    piece.block0 = (unsigned)at;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(blocks - at < most ? blocks - at : most)), dim3(threads), lds, stream, piece);
    e = hipGetLastError();
  }
  return e;
}

template <int DT, int RT, bool EXACT, bool KL, bool SM, int W, bool DIRECT>
struct F32Tag {};

// Chains without softmax on up to 24 keys (16 with two row tiles), B [L][K]: one wave or two have a step, too short for the trip through
// LDS to pay.  us per launch through LDS / direct: 24 x 1348 x 8 x 64 10.3 / 8.9, 3 x 74 x 9 x 128 3.38 / 2.98, 31 x 879 x 9 x 128 22.1 /
// 19.9; by columns and keys 1.02 - 1.16 up to 24, 0.96 - 1.01 from 25 to 32.
static bool f32_direct(const F32ChainArgs& a) { return !a.softmax && a.b_lk && a.L <= (a.row_tiles == 1 ? 24 : 16); }

template <int DT, int RT, bool EXACT, int W>
static hipError_t launch_f32(const F32ChainArgs& a, hipStream_t stream) {
  const int lds = f32_chain_lds_bytes_host(a.K, a.N, 0, RT, W), threads = 64 * kWaves;
  if (a.softmax)
    return a.b_lk ? launch_with_lds<F32Tag<DT, RT, EXACT, false, true, W, false>>(gemm_chain_f32_kernel<DT, RT, EXACT, false, true, W, false>, threads, lds, a, stream)
                  : launch_with_lds<F32Tag<DT, RT, EXACT, true, true, W, false>>(gemm_chain_f32_kernel<DT, RT, EXACT, true, true, W, false>, threads, lds, a, stream);
  if constexpr (EXACT && DT != 5)
    if (f32_direct(a))
      return launch_with_lds<F32Tag<DT, RT, true, false, false, W, true>>(gemm_chain_f32_kernel<DT, RT, true, false, false, W, true>, threads, lds, a, stream);
  return a.b_lk ? launch_with_lds<F32Tag<DT, RT, EXACT, false, false, W, false>>(gemm_chain_f32_kernel<DT, RT, EXACT, false, false, W, false>, threads, lds, a, stream)
                : launch_with_lds<F32Tag<DT, RT, EXACT, true, false, W, false>>(gemm_chain_f32_kernel<DT, RT, EXACT, true, false, W, false>, threads, lds, a, stream);
}

template <int DT, bool EXACT>
static hipError_t launch_f32_rows(const F32ChainArgs& a, hipStream_t stream) {
  if constexpr (DT <= 5)
    if (a.row_tiles == 2 && a.width == 0) return launch_f32<DT, 2, EXACT, 0>(a, stream);
  if (a.row_tiles != 1) return hipErrorInvalidValue;
  if (a.width == 0) return launch_f32<DT, 1, EXACT, 0>(a, stream);
  if (a.width == 16) return launch_f32<DT, 1, EXACT, 16>(a, stream);
  if constexpr (DT != 5)
    if (a.width == 32) return launch_f32<DT, 1, EXACT, 32>(a, stream);
  if constexpr (DT == 8)
    if (a.width == 64) return launch_f32<DT, 1, EXACT, 64>(a, stream);
  return hipErrorInvalidValue;
}

template <int DT>
static hipError_t launch_f32_rows(const F32ChainArgs& a, bool exact, hipStream_t stream) {
  return exact ? launch_f32_rows<DT, true>(a, stream) : launch_f32_rows<DT, false>(a, stream);
}

hipError_t launch_gemm_chain_f32(const F32ChainArgs& a, hipStream_t stream) {
  if (a.f64) return launch_with_lds<double>(gemm_chain_f64_kernel, 256, f64_chain_lds_bytes(a.K, a.N), a, stream);
  const int dt = f32_tiles(a.K, a.N);
  // 16-byte pieces of the rows of A, B (stored [L][K]), C and F; a [K][L] B is read one element per lane either way
  long long strides = a.a_bs | a.c_bs | a.f_bs | a.a_rs | a.c_rs | a.f_rs;
  if (a.b_lk) strides |= a.b_bs | a.b_rs;
  const bool exact = f32_chain_exact(a.K, a.N, strides);
  return dt == 4 ? launch_f32_rows<4>(a, exact, stream)
         : dt == 5 ? launch_f32_rows<5>(a, exact, stream)
                   : launch_f32_rows<8>(a, exact, stream);
}

}  // namespace ditto
