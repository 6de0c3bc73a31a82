// C ABI of the chain library: descriptor validation, tile choice, kernel dispatch.
// Declarations and the reference interfaces they replace are in include/ditto_chain.h.
#include "../../include/ditto_chain.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "bmm_chain_fp8.h"
#include "bmm_chain_fp8m16.h"
#include "bmm_chain_fp4m16.h"
#include "bmm_chain_rows.h"
#include "bmm_chain_split.h"
#include "chain_kernels.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

// What one launch holds: fewer than 2^32 work items.  The kernels that give few rows or pixels to many threads reach that
// at sizes the general kernels still take, which keep them.
bool launchable(long long workgroups, int threads) { return workgroups < (1LL << 32) / threads; }

bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// Number of compute units of the current device (cached per thread).
int device_cus() {
  static thread_local int cus = 0;
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      cus = prop.multiProcessorCount;
    if (cus <= 0) cus = 256;
  }
  return cus;
}

struct BmmPlan {
  int family;  // 0: fp16/bf16 register-resident chain, 1: fp32 chain, 2: int8 requant chain
  int d_pad, qt;  // fp chains: head pad and rows-per-wave code; int8 chain: row tiles and ring depth
  // fp chains on few rows: column tiles and row tiles of the key-splitting kernel (0: none), column tiles of a workgroup if not all
  int split_dt = 0, split_rt = 0, split_ct = 0;
  int rows_dt = 0, rows_nw = 0;  // fp chains: column tiles and waves of the kernel of 32 rows per wave and short tiles (0: none)
  int units_rt = 0, slices = 0, slice_blocks = 0;  // int8 chain on few rows: row tiles, slices of the columns, blocks of 64 of each (0: none)
  int f32_width = 0, f32_cols = 1;  // fp32 chain on few rows: columns of a workgroup (0: all), workgroups that share them out
  int nb3 = 0, nb = 0;  // 16x16x32-MFMA kernel: row blocks of 384 rows / row blocks in all, per batch entry
  ditto_tile_param tile;
};

// Row blocks of 384 and of 256 rows for the kernel on the 16x16x32 MFMA.  A 384-row workgroup does half as much
// work again as a 256-row one in about kBig3 of its time, but 384 seldom divides the rows evenly over the compute
// units: every split (a blocks of 384, then blocks of 256 for the rest) is priced by dealing its workgroups out the
// way the hardware does (an XCD takes the large blocks of all of its batch entries first, then the small ones, each
// to the compute unit that is free first) and the shortest finish wins.  Returns a.
constexpr double kBig3 = 1.43;
int plan_rows_384(long long M, long long batch, int cus) {
  thread_local long long last_m = -1, last_batch = -1;
  thread_local int last_cus = -1, last_a = 0;
  if (M == last_m && batch == last_batch && cus == last_cus) return last_a;
  const long long amax = M / 384 + (M % 384 > 256 ? 1 : 0);
  const bool split = batch % 8 == 0 && cus % 8 == 0;
  const long long per = split ? batch / 8 : batch;
  const int cu = split ? cus / 8 : cus;
  int best_a = 0;
  if (amax > 0 && per * (M / 256 + 2) > 4096) {
    best_a = (int)(M / 384);  // so many workgroups that the finish does not matter
  } else if (amax > 0) {
    double best = 0;
    std::vector<double> free_at(cu);
    for (long long a = 0; a <= amax; ++a) {
      if (a > 0 && a < amax - 16) continue;  // the finish is tuned by the last few blocks
      const long long rest = M - 384 * a;
      const long long b = rest > 0 ? (rest + 255) / 256 : 0;
      std::fill(free_at.begin(), free_at.end(), 0.0);
      auto deal = [&](long long n, double cost) {
        for (long long i = 0; i < n; ++i) *std::min_element(free_at.begin(), free_at.end()) += cost;
      };
      deal(per * a, kBig3);
      deal(per * b, 1.0);
      const double finish = *std::max_element(free_at.begin(), free_at.end());
      if (a == 0 || finish < best - 1e-9) best = finish, best_a = (int)a;
    }
  }
  last_m = M, last_batch = batch, last_cus = cus, last_a = best_a;
  return best_a;
}

// What a kernel takes, in us per launch: start + (first + per_key L) for every round of workgroups over the compute units; a
// kernel of several workgroups to a compute unit has a pair for each number of them, the last one for full rounds.
struct BmmPrice {
  int variant, rows, threads, resident;
  float start, first[3], per_key[3];
};
// Least squares over 3300 random shapes (batch 1 - 160, 32 - 4096 rows and keys, fp16 and bf16), those of 2144 and of the 64-row
// kernels with softmax over 3600 others, root mean square error 4 - 12 %; the columns: head sizes up to 64 | 128, without | with softmax, B [L][K] | [K][L].
// (The 20xx, 2148 and 2188 as they were before their rows of A came through LDS, up to 0.2 of a short launch more; few_rows_variant has
// prices of its own for the 20xx.)
constexpr BmmPrice kPrices64[2][2][8] = {
    {{{641, 128, 256, 1, 0.71f, {3.38f}, {.0074f}}, {644, 64, 256, 3, 2.64f, {1.30f, 1.81f, 2.36f}, {.0049f, .0079f, .0121f}},
      {645, 64, 256, 2, 2.98f, {1.34f, 2.09f}, {.0042f, .0070f}}, {649, 256, 512, 1, 0, {5.03f}, {.0118f}},
      {2144, 128, 256, 3, 2.40f, {1.77f, 2.36f, 3.74f}, {.0091f, .0156f, .0208f}}, {2148, 256, 512, 1, 2.23f, {2.31f}, {.0124f}}},
     {{641, 128, 256, 1, 0.68f, {3.38f}, {.0077f}}, {644, 64, 256, 3, 2.75f, {1.33f, 1.93f, 2.79f}, {.0060f, .0092f, .0128f}},
      {645, 64, 256, 2, 3.05f, {1.53f, 2.74f}, {.0049f, .0074f}}, {649, 256, 512, 1, 0, {5.14f}, {.0117f}},
      {2144, 128, 256, 3, 2.11f, {2.30f, 3.42f, 4.75f}, {.0102f, .0154f, .0209f}}, {2148, 256, 512, 1, 1.81f, {3.20f}, {.0116f}},
      {2041, 16, 512, 1, 2.89f, {1.35f}, {.0025f}}, {2042, 32, 512, 1, 2.78f, {2.37f}, {.0027f}}}},
    {{{644, 64, 256, 3, 2.64f, {1.38f, 1.90f, 2.65f}, {.0057f, .0096f, .0132f}}, {645, 64, 256, 2, 3.38f, {1.16f, 2.21f}, {.0054f, .0083f}},
      {646, 256, 512, 1, 0, {6.41f}, {.0170f}}, {649, 256, 512, 1, 0, {5.96f}, {.0159f}},
      {2144, 128, 256, 3, 2.77f, {1.45f, 2.35f, 3.81f}, {.0118f, .0183f, .0242f}}},
     {{644, 64, 256, 3, 2.74f, {1.40f, 2.10f, 3.04f}, {.0062f, .0100f, .0138f}}, {645, 64, 256, 2, 3.54f, {1.34f, 2.81f}, {.0057f, .0085f}},
      {649, 256, 512, 1, 0, {6.02f}, {.0162f}},
      {2144, 128, 256, 3, 2.94f, {1.55f, 2.95f, 4.34f}, {.0119f, .0177f, .0243f}}}}};
constexpr BmmPrice kPrices128[2][2][7] = {
    {{{1281, 128, 256, 1, 0, {5.79f}, {.0113f}}, {1282, 256, 256, 1, 0, {8.95f}, {.0223f}}, {1286, 256, 512, 1, 0, {7.95f}, {.0277f}},
      {1289, 256, 512, 1, 0, {6.92f}, {.0227f}}, {2188, 256, 512, 1, 0, {5.55f}, {.0230f}},
      {2081, 16, 512, 1, 1.70f, {2.93f}, {.0043f}}, {2082, 32, 512, 1, 1.19f, {4.82f}, {.0044f}}},
     {{1281, 128, 256, 1, 0, {5.79f}, {.0116f}}, {1282, 256, 256, 1, 0, {8.58f}, {.0228f}},
      {1289, 256, 512, 1, 0, {7.35f}, {.0245f}}, {2188, 256, 512, 1, 0, {6.83f}, {.0226f}},
      {2081, 16, 512, 1, 1.38f, {3.82f}, {.0059f}}, {2082, 32, 512, 1, 0.64f, {6.61f}, {.0061f}}}},
    {{{1281, 128, 256, 1, 0, {6.58f}, {.0149f}}, {1289, 256, 512, 1, 0, {8.03f}, {.0242f}}, {1286, 256, 512, 1, 0, {8.67f}, {.0244f}},
      {2188, 256, 512, 1, 0, {5.57f}, {.0269f}}, {2081, 16, 512, 1, 1.54f, {3.70f}, {.0043f}},
      {2082, 32, 512, 1, 1.09f, {6.13f}, {.0049f}}},
     {{1281, 128, 256, 1, 0, {6.67f}, {.0154f}}, {1289, 256, 512, 1, 0, {8.50f}, {.0256f}}, {1286, 256, 512, 1, 0, {9.59f}, {.0266f}},
      {2188, 256, 512, 1, 0, {7.13f}, {.0244f}}, {2081, 16, 512, 1, 1.15f, {4.61f}, {.0063f}},
      {2082, 32, 512, 1, 1.43f, {7.09f}, {.0068f}}}}};

long long bmm_workgroups(const BmmPrice& p, const ditto_bmm_chain_desc* d) { return ((d->M + p.rows - 1) / p.rows) * d->batch; }
float bmm_price(const BmmPrice& p, const ditto_bmm_chain_desc* d, int cus) {
  const long long wgs = bmm_workgroups(p, d), full = wgs / (p.resident * cus);  // full rounds
  const int left = (int)((wgs - full * p.resident * cus + cus - 1) / cus), r = p.resident - 1;
  const float L = (float)d->L;
  return p.start + full * (p.first[r] + p.per_key[r] * L) + (left > 0 ? p.first[left - 1] + p.per_key[left - 1] * L : 0.f);
}

// The kernel that is priced at least 7 % below `own`, the one the rules of plan_bmm name, or 0.  The rules draw their lines
// along one size at a time and miss where the rounds of two kernels fall differently: one round of 256-row workgroups against
// two of 128 rows (40 x 809 x 1608 x 128 softmax 59.2 -> 44.2 us), 1.2 rounds of 256 against 2.2 of 128 (30 x 2080 x 2032 x 128
// 122 -> 79), without softmax 50 x 1520 x 576 x 64 24.7 -> 19.1, 5 x 432 x 144 x 128 7.6 -> 6.0.  Softmax chains of up to 64
// columns have one other kernel to go to, 32 rows a wave, from 5 % on (1152 x 512 x 512 122 -> 107 us, 3268 x 197 x 197 110 -> 84;
// long keys on few rows stay: 830 x 192 x 2048 114 against 136).  A price misses a single shape by more than these margins, so
// the pairs of kernels whose shapes went wrong are left out below: of 5000 random shapes whose kernel changes 1 in 1000 takes more
// than 1.03 of its time, the worst 1.04, the mean 0.85 without softmax and at 128 columns and 0.90 with it at 64.
int cheaper_variant(const ditto_bmm_chain_desc* d, int own, int cus) {
  const long long dmax = d->K > d->N ? d->K : d->N;
  const bool sm = d->inter_op == DITTO_INTER_SOFTMAX, kl = d->b_layout == DITTO_B_KL;
  // with softmax the kernels that find a row's first unmasked key wherever it lies (20xx, 21xx, 644, 645) keep what they have
  if (dmax > 64 && (dmax <= 80 || (sm && own >= 2000))) return 0;
  const BmmPrice* const prices = dmax <= 64 ? kPrices64[sm][kl] : kPrices128[sm][kl];
  const BmmPrice* const end = prices + (dmax <= 64 ? 8 : 7);
  auto workgroups = [&](const BmmPrice& p) { return bmm_workgroups(p, d); };
  auto rounds = [&](const BmmPrice& p) { return bmm_workgroups(p, d) / (p.resident * cus); };  // full ones
  auto price = [&](const BmmPrice& p) { return bmm_price(p, d, cus); };
  const BmmPrice* const mine = std::find_if(prices, end, [&](const BmmPrice& p) { return p.variant == own; });
  if (mine == end) return 0;
  // what a kernel's price may be of the rules' kernel's: 2148 is level with the 64-row kernels where it is priced 5 - 10 % below
  // (up to 64 keys 1.05 of the time, 43 x 741 x 34 4.68 -> 5.05 us)
  auto margin = [&](const BmmPrice& p) { return p.variant == 2148 ? 0.90f : sm && dmax <= 64 ? 0.95f : 0.93f; };
  auto taken = [&](const BmmPrice& p) {
    if (!launchable(workgroups(p), p.threads)) return false;
    switch (p.variant) {
      case 2188:  // (beyond these keys its price fits by 4 - 9 %; against 256-row workgroups it takes 0.99 - 1.04 of the time)
        return d->L >= 64 && d->L <= 700 && own != 1282 && own != 1289;
      case 2144:
        // fp16 64-row workgroups scale A beforehand, a fifth of the vector ALU's work in the softmax, which the one price for
        // both types does not show: 1.00 of the time in the mean from 700 keys on, up to 1.05 (252 x 697 x 1083 65.5 -> 68.7 us;
        // [K][L], whose transposing reads weigh more, from 1024 on)
        if (sm && dmax <= 64 && d->in_dtype == DITTO_F16 && (own == 645 || (own == 644 && !kl && d->L > 700))) return false;
        return d->L > (kl && own == 2148 ? 128 : 64) || (sm && rounds(p) > 0);
      case 2081:
      case 2082:
        // (38 x 197 x 2717 without softmax 33.0 -> 34.6 us, 46 x 352 x 4037 48.5 -> 52.8; up to 300 keys 0.92.  With it where B and C
        // pass the L2s several times over: 133 x 61 x 1924 33.9 -> 37.7 [L][K], 69 x 99 x 2768 47.5 -> 50.3 [K][L].)
        return sm ? 2 * d->batch * d->L * (d->K + d->N) <= (kl ? 48 << 20 : 96 << 20) : kl || d->L <= 1024;
      case 644:  // (117 x 1064 x 32 [K][L] 10.8 -> 11.7 us)
        if (kl && own == 2148) return false;
        [[fallthrough]];
      default: return !sm || dmax > 64;
    }
  };
  int best = 0;
  float best_price = 0;
  const float own_price = price(*mine);
  for (const BmmPrice* p = prices; p != end && p->variant != 0; ++p)
    if (p != mine && taken(*p) && price(*p) < margin(*p) * own_price && (best == 0 || price(*p) < best_price))
      best = p->variant, best_price = price(*p);
  return best;
}

// The key-splitting kernel where it is priced well below `own`, a kernel of 64 or 128 rows a workgroup, or 0.  The rules of
// plan_bmm weigh it at what it took before its rows of A came through LDS, and know no shares of the columns.  2.3 us and, for
// every round of workgroups, a start and a share of the keys; fitted to 2200 random shapes (root mean square error 4 % at 64
// columns, 7 at 128).  us per launch: 5 x 256 x 224 x 64 [K][L] 5.05 -> 3.96, 3 x 166 x 166 x 64 4.35 -> 3.76, 1 x 512 x 96 x 64 without
// softmax 3.68 -> 3.22; 3 x 1552 x 272 x 128 [K][L] 10.9 -> 7.9, 13 x 608 x 256 x 128 without softmax 8.2 -> 6.7.  Of 9300 other
// shapes at 128 columns 3 % change, to 0.83 of the time, the worst 0.98; of 8200 at 64 columns 11 %, to 0.88, the worst 1.00.  Up to
// 64 keys, and from 1600 keys on at 128 columns, the price misses by more than there is to gain (1 x 2848 x 64 x 64 1.075, 81 x 64 x 64 x
// 128 0.99, 6 x 1808 x 3888 x 128 1.025).  So it does, for 32 rows a workgroup, up to 128 keys of [K][L] without softmax at 64 columns
// (nine shapes 1.01 - 1.05: 7 x 926 x 112 x 24 3.82 -> 4.00, 2 x 3309 x 120 x 64 4.00 -> 4.12; 5 x 1358 x 136 0.95), and for a second
// round of workgroups at 128 columns where B and C of the batch do not fit the L2s, 32 MB in all (99 x 78 x 1312 [K][L] 22.0 -> 24.6,
// 132 x 63 x 1228 25.5 -> 27.3, eight shapes of 55 MB and more 0.93 - 1.11; below 33 MB 0.89 - 0.98).
int few_rows_variant(const ditto_bmm_chain_desc* d, int own, int cus) {
  const long long dmax = d->K > d->N ? d->K : d->N;
  if (dmax > 64 && dmax <= 80) return 0;
  if (own != 641 && own != 644 && own != 645 && own != 1281) return 0;
  if (d->L <= 64 || (dmax > 64 && d->L > 1600)) return 0;
  const bool sm = d->inter_op == DITTO_INTER_SOFTMAX, kl = d->b_layout == DITTO_B_KL;
  const BmmPrice* const prices = dmax <= 64 ? kPrices64[sm][kl] : kPrices128[sm][kl];
  const BmmPrice* const end = prices + (dmax <= 64 ? 8 : 7);
  const BmmPrice* const mine = std::find_if(prices, end, [&](const BmmPrice& p) { return p.variant == own; });
  if (mine == end) return 0;
  struct Split {
    float first, per_key;
  };
  constexpr Split k64[2][2] = {{{0.94f, .0020f}, {1.40f, .0022f}}, {{1.28f, .0023f}, {1.98f, .0029f}}};   // [softmax][16 | 32 rows]
  constexpr Split k128[2][2] = {{{2.25f, .0038f}, {3.20f, .0042f}}, {{2.72f, .0043f}, {4.12f, .0046f}}};
  const Split* const split = dmax <= 64 ? k64[sm] : k128[sm];
  const float per_kl = !kl ? 1.f : dmax <= 64 ? 1.12f : 1.17f;  // transposing reads of B
  float best = (dmax <= 64 ? 0.84f : 0.90f) * bmm_price(*mine, d, cus);
  int variant = 0;
  for (int rt = 1; rt <= 2; ++rt) {
    const long long wgs = ((d->M + 16 * rt - 1) / (16 * rt)) * d->batch, rounds = (wgs + cus - 1) / cus;
    if (!launchable(wgs, 64 * ditto::kSplitWaves)) continue;
    if (dmax <= 64 ? rt == 2 && kl && !sm && d->L <= 128 : rounds > 1 && 2 * d->batch * d->L * (d->K + d->N) > 32 << 20) continue;
    const float cost = 2.3f + rounds * (split[rt - 1].first + split[rt - 1].per_key * per_kl * (float)d->L);
    if (cost < best) best = cost, variant = (dmax <= 64 ? 2040 : 2080) + rt;
  }
  return variant;
}

int plan_bmm_rules(const ditto_bmm_chain_desc* d, BmmPlan* plan, int cus);

// `few_rows`: few_rows_variant may have its say (not in the plans of chains that share a launch, see plan_sets).
int plan_bmm(const ditto_bmm_chain_desc* d, BmmPlan* plan, bool need_device, bool few_rows = true) {
  // A plan depends on the descriptor and the number of compute units alone: the last few are kept, so that a
  // repeated call pays for a comparison and not for the pricing.
  struct Kept {
    ditto_bmm_chain_desc desc;
    int cus;
    bool few_rows;
    BmmPlan plan;
  };
  constexpr int kKept = 8;
  static thread_local Kept kept[kKept] = {};  // (an all-zero descriptor is refused: abi_version)
  static thread_local int next = 0;
  const int cus = need_device ? device_cus() : 256;
  if (d)
    for (const Kept& k : kept)
      if (k.cus == cus && k.few_rows == few_rows && memcmp(&k.desc, d, sizeof(*d)) == 0) return *plan = k.plan, DITTO_OK;
  int rc = plan_bmm_rules(d, plan, cus);
  if (rc != DITTO_OK) return rc;
  if (plan->family == 0 && d->tile_variant == 0) {
    ditto_bmm_chain_desc forced = *d;
    forced.tile_variant = cheaper_variant(d, plan->tile.variant, cus);
    if (forced.tile_variant != 0) rc = plan_bmm_rules(&forced, plan, cus);
    forced.tile_variant = few_rows && rc == DITTO_OK ? few_rows_variant(d, plan->tile.variant, cus) : 0;
    if (forced.tile_variant != 0) rc = plan_bmm_rules(&forced, plan, cus);
  }
  if (rc == DITTO_OK) {
    kept[next] = {*d, cus, few_rows, *plan};
    next = (next + 1) % kKept;
  }
  return rc;
}

int plan_bmm_rules(const ditto_bmm_chain_desc* d, BmmPlan* plan, int cus) {
  if (!d) return fail(DITTO_EINVAL, "null descriptor");
  if (d->abi_version != DITTO_CHAIN_ABI_VERSION)
    return fail(DITTO_EINVAL, "descriptor abi_version %d, library %d", d->abi_version,
                DITTO_CHAIN_ABI_VERSION);
  if (d->relu_out != 0 && d->relu_out != 1) return fail(DITTO_EINVAL, "relu_out must be 0 or 1");
  if (d->relu_out && (d->in_dtype == DITTO_I8 || d->inter_op == DITTO_INTER_SOFTMAX))
    return fail(DITTO_EUNSUPPORTED, "relu_out is implemented for the cast / relu chains on fp16, bf16 and fp32");
  if (d->tile_variant < 0) return fail(DITTO_EINVAL, "tile_variant must be 0 or a variant id");
  if (d->batch_inner < 0 || (d->batch_inner > 0 && d->batch > 0 && d->batch % d->batch_inner != 0))
    return fail(DITTO_EINVAL, "batch_inner must be 0 or divide batch");
  const bool two_level = d->batch_inner > 0 && d->batch_inner != d->batch;
  if (two_level && d->in_dtype != DITTO_F16 && d->in_dtype != DITTO_BF16)
    return fail(DITTO_EUNSUPPORTED, "two-level batch strides are implemented for the fp16/bf16 chains");
  if (d->batch <= 0 || d->M <= 0 || d->N <= 0 || d->K <= 0 || d->L <= 0)
    return fail(DITTO_EINVAL, "batch, M, N, K, L must be positive (got %lld %lld %lld %lld %lld)",
                (long long)d->batch, (long long)d->M, (long long)d->N, (long long)d->K,
                (long long)d->L);
  if (d->M > 0x7fffffff / 2 || d->L > 0x7fffffff / 2 || d->batch > 0x7fffffff / 2)
    return fail(DITTO_EINVAL, "extent too large");
  if (d->b_layout != DITTO_B_KL && d->b_layout != DITTO_B_LK)
    return fail(DITTO_EINVAL, "unknown b_layout %d", d->b_layout);
  const int in = d->in_dtype;
  memset(plan, 0, sizeof(*plan));

  if (in == DITTO_F16 || in == DITTO_BF16) {
    // (an fp16 accumulator asked for with fp16 operands -- the reference's ("80", "float16", "float16") row -- is
    // served by the MFMA's fp32 accumulator: the precision asked for and more)
    if (d->acc_dtype != DITTO_F32 && !(d->acc_dtype == DITTO_F16 && in == DITTO_F16))
      return fail(DITTO_EUNSUPPORTED, "fp16/bf16 chains accumulate in fp32 (acc_dtype %d)", d->acc_dtype);
    if (d->out_dtype != in && d->out_dtype != DITTO_F32)
      return fail(DITTO_EINVAL, "out_dtype must be in_dtype or fp32");
    if (d->inter_op != DITTO_INTER_CAST && d->inter_op != DITTO_INTER_RELU &&
        d->inter_op != DITTO_INTER_SOFTMAX)
      return fail(DITTO_EINVAL, "inter_op %d not valid for a floating-point chain", d->inter_op);
    if (d->inter_op == DITTO_INTER_SOFTMAX && !(d->softmax_scale > 0.f))
      return fail(DITTO_EINVAL, "softmax_scale must be > 0");
    // 16-byte vector loads: extents and strides in multiples of 8 elements.
    // (The reference builders require multiples of 16: bmm_chain.py:34-38.)
    if (d->K % 8 || d->N % 8) return fail(DITTO_EINVAL, "K and N must be multiples of 8");
    if (d->b_layout == DITTO_B_KL && d->L % 8)
      return fail(DITTO_EINVAL, "L must be a multiple of 8 when B is [K][L]");
    if (d->a_row_stride % 8 || d->b_row_stride % 8 || d->c_row_stride % 8 || d->a_batch_stride % 8 ||
        d->b_batch_stride % 8 || d->c_batch_stride % 8)
      return fail(DITTO_EINVAL, "input strides must be multiples of 8 elements");
    if (two_level && (d->a_batch_stride_outer % 8 || d->b_batch_stride_outer % 8 || d->c_batch_stride_outer % 8 ||
                      d->f_batch_stride_outer % 4))
      return fail(DITTO_EINVAL, "outer batch strides must be multiples of 8 (inputs) / 4 (output) elements");
    const int out_vec = 4;
    if (d->f_row_stride % out_vec || d->f_batch_stride % out_vec)
      return fail(DITTO_EINVAL, "output strides must be multiples of 4 elements");
    if (d->a_row_stride < d->K || d->c_row_stride < d->N || d->f_row_stride < d->N ||
        d->b_row_stride < (d->b_layout == DITTO_B_KL ? d->L : d->K))
      return fail(DITTO_EINVAL, "row stride smaller than row extent");
    if (d->a_row_stride > 0x7fffffff || d->b_row_stride > 0x7fffffff ||
        d->c_row_stride > 0x7fffffff || d->f_row_stride > 0x7fffffff)
      return fail(DITTO_EINVAL, "row stride too large");
    // one batch entry of B and of C is addressed through a 32-bit buffer offset
    {
      const long long b_rows = d->b_layout == DITTO_B_KL ? d->K : d->L;
      if (b_rows * d->b_row_stride * 2 >= 0x7fffffffLL || d->L * d->c_row_stride * 2 >= 0x7fffffffLL)
        return fail(DITTO_EUNSUPPORTED, "a batch entry of B or C exceeds 2 GiB");
    }
    const long long dmax = d->K > d->N ? d->K : d->N;
    if (dmax > 128)
      return fail(DITTO_EUNSUPPORTED, "max(K,N)=%lld: register-resident chain supports up to 128", dmax);
    plan->family = 0;
    plan->d_pad = dmax <= 64 ? 64 : 128;
    // Variant table (measured on MI355X, fp16 and bf16, head_pad 64 and 128).  n8 = number of 256-row
    // workgroups.  Below 3/4 of the CUs the four-wave kernel with 128-row workgroups spreads over more
    // CUs.  From there on eight waves (two per SIMD) win, in their software-pipelined form (9) at every
    // size measured.  Once there are two workgroups per CU the chip runs at its power limit and the
    // kernel on the 16x16x32 MFMA (6), which needs less energy per flop, is ahead
    // (64 x 4096 x 4096 x 128 bf16: 464 vs 484 us with the softmax, 410 vs 443 us without); at
    // head_pad 64 the pipelined kernel stays (32 x 4096 x 4096 x 64 without softmax 127.9 vs 130.0 us).
    // With B stored [K][L] (B fragments through transposing reads on the 16x16x32 kernel) the softmax at
    // head_pad 128 goes the same way (bf16 441 vs 503 us, fp16 482 vs 538), without softmax the four-wave,
    // 256-row kernel stays (431 vs 430 us).
    const long long n8 = ((d->M + 255) / 256) * d->batch;
    const bool sm = d->inter_op == DITTO_INTER_SOFTMAX;
    if (n8 >= 2LL * cus) {
      if (d->b_layout == DITTO_B_LK)
        plan->qt = plan->d_pad == 64 ? 9 : 6;
      else
        plan->qt = sm ? (plan->d_pad == 64 ? 9 : 6) : 2;
    } else if (n8 * 4 >= 3LL * cus) {
      plan->qt = 9;
    } else {
      plan->qt = 1;
    }
    // Head size up to 64: the four-wave kernels with 64-row workgroups (4: a wave owns 16 rows and all keys; 5: 32
    // rows and half the keys of every tile, half the LDS reads per MFMA for a merge at the end, ahead from 1024 keys
    // on).  Measured, fp16 and bf16, us per launch in a graph replay, best other variant -> best of 4 | 5, B stored
    // [L][K]: softmax 96 x 512 x 512 13.2 -> 11.5, 12 x 512 x 512 9.9 -> 6.9, 8 x 1024 x 1024 15.5 -> 9.9,
    // 16 x 512 x 2048 26.3 -> 15.5, 768 x 512 x 512 84.5 -> 78.1, 96 x 2048 x 2048 fp16 119.3 -> 116.7; bf16 at that
    // size and beyond stays on the eight-wave 16x16x32 kernel (115.6 against 120.1; 32 x 4096 x 4096 139.9 against
    // 150.6).  Without the softmax they are ahead below two 256-row workgroups per CU (96 x 512 x 512 11.2 -> 10.7,
    // 16 x 512 x 2048 17.0 -> 14.6) and behind from there on (384 x 512 x 512 38.9 against 39.3); where the 64-row
    // workgroups make one and a half rounds of the CUs and the 128-row ones fit in one, the latter stay
    // (48 x 512 x 512 7.5 against 8.2).  B stored [K][L] (its fragments come out of transposing reads): softmax
    // 96 x 512 x 512 13.1 -> 11.8, 12 x 512 x 512 10.0 -> 7.3, 16 x 512 x 2048 26.9 -> 16.6, 768 x 512 x 512
    // 83.8 -> 81.8, level at 96 x 2048 x 2048 (122.7 / 121.6) and 32 x 4096 x 4096 (153.1 / 154.7: stays); without
    // the softmax only the grids that leave CUs empty gain (12 x 512 x 512 7.5 -> 7.0, 8 x 1024 x 1024 10.9 -> 10.0,
    // 16 x 512 x 2048 17.9 -> 16.0; but 96 x 512 x 512 10.7 against 11.6, 48 x 512 x 512 7.5 against 9.0).
    if (plan->d_pad == 64) {
      const bool lk = d->b_layout == DITTO_B_LK;
      const long long n64 = ((d->M + 63) / 64) * d->batch, n128 = ((d->M + 127) / 128) * d->batch;
      bool rows64;
      if (sm)
        rows64 = !((in == DITTO_BF16 || !lk) && n8 >= 2LL * cus && d->L >= 2048);
      else if (lk)
        rows64 = n8 < 2LL * cus && !(n64 > cus && n128 <= cus);
      else
        rows64 = n64 <= cus;
      if (rows64) plan->qt = d->L >= 1024 ? 5 : 4;
      else if (sm && lk && n8 >= 2LL * cus) plan->qt = 6;
    }
    {
      // Few rows: the kernel whose eight waves split the keys (bmm_chain_split.h), in workgroups of 16 or 32 rows.  (As it was before
      // its rows of A came through LDS: few_rows_variant takes the chains that it has been ahead for since.)  Its cost
      // beyond the launch is a start and a merge plus a share of the keys, `a + b L` us, for every round of workgroups over
      // the compute units; the kernels above walk all keys in one go and their 64 or 128 rows per workgroup need fewer
      // rounds.  Fitted to measurements at head sizes 64, 80 and 128 (us per launch, other kernel -> this one, LK):
      // 16 x 176 x 176 x 80 8.4 -> 4.9, 8 x 461 x 461 x 80 12.7 -> 5.9, 16 x 512 x 512 x 80 12.4 -> 7.3 (32 rows),
      // 2 x 2392 x 2392 x 80 38.5 -> 13.1, 2 x 4096 x 4096 x 128 60.9 -> 28.4, 8 x 512 x 2048 x 64 17.5 -> 8.8; but
      // 40 x 300 x 300 x 80 8.4 against 11.2 and 60 x 58 x 58 x 64 3.7 against 4.1, which stay.
      const int dt = dmax <= 64 ? 4 : dmax <= 80 ? 5 : 8;
      const bool kl_b = d->b_layout == DITTO_B_KL;
      int rt = 0;
      if (d->tile_variant == 0 && (dt == 5 || plan->qt == 1 || plan->qt == 4 || plan->qt == 5)) {
        const double start[2] = {dt == 4 ? 1.2 : dt == 5 ? 2.0 : 3.0, dt == 4 ? 2.7 : dt == 5 ? 2.9 : 4.5};
        const double per_key[2] = {dt == 4 ? 0.0022 : dt == 5 ? 0.0028 : 0.0044, dt == 4 ? 0.0029 : dt == 5 ? 0.0033 : 0.0053};
        const long long n64 = ((d->M + 63) / 64) * d->batch, n128 = ((d->M + 127) / 128) * d->batch;
        double best = dt == 4 ? (0.55 + 0.0065 * d->L) * (n64 <= cus ? 1.0 : 0.8 * ((n64 + cus - 1) / cus))
                              : (sm ? 3.6 + 0.0134 * d->L : 3.2 + 0.0099 * d->L) * ((n128 + cus - 1) / cus);
        best *= 0.95;
        if (dt == 5) {
          // Head sizes 65 to 80: the kernel padded to 80 columns (bmm_chain_rows.h), four waves with 128-row workgroups, two to a
          // compute unit, or eight with 256 rows.  It replaces the kernels padded to 128 but for chains without softmax of one
          // round of 128-row workgroups and more than about 500 keys, where one wave per SIMD of 32x32x16 MFMAs is ahead
          // (12 x 1600 x 1600 20.8 against 22.8).  Fitted like the above, us per launch beyond 2.2, other kernel -> four | eight
          // waves, LK with softmax: 160 x 197 x 197 18.2 -> 9.6 | 9.1, 640 x 49 x 49 22.9 -> 8.8 | 12.0, 80 x 400 x 400
          // 23.2 -> 13.4 | 12.9, 160 x 577 x 577 44.0 -> 33.8 | 34.3, 80 x 1024 x 1024 60.8 -> 41.3 | 50.8,
          // 32 x 4096 x 4096 206 -> 191 | 187; the key-splitting kernel stays at 12 x 400 x 400 (7.1 against 9.9).
          if (sm || plan->qt != 1) best = 1e30;
          const double key = (sm ? 1.0 : 0.9) * (kl_b ? 1.07 : 1.0) * d->L;
          for (int nw = 4; nw <= 8; nw += 4) {
            const long long wgs = ((d->M + 32 * nw - 1) / (32 * nw)) * d->batch, rounds = (wgs + cus - 1) / cus;
            if (!launchable(wgs, 64 * nw)) continue;
            const double cost = nw == 4 ? (rounds == 1 ? 2.3 + 0.0131 * key : 2.1 + rounds * (1.1 + 0.0114 * key))
                                        : (rounds == 1 ? 2.9 + 0.0196 * key : 2.1 + rounds * (2.8 + 0.0226 * key));
            if (cost < best) best = cost, plan->rows_dt = 5, plan->rows_nw = nw;
          }
        }
        for (int r = 1; r <= 2; ++r) {
          const long long wgs = ((d->M + 16 * r - 1) / (16 * r)) * d->batch, rounds = (wgs + cus - 1) / cus;
          if (!launchable(wgs, 64 * ditto::kSplitWaves)) continue;
          const double cost = rounds * (start[r - 1] + per_key[r - 1] * d->L) * (!kl_b ? 1.0 : dt == 8 ? 1.3 : 1.15);
          if (cost < best) best = cost, rt = r;
        }
      }
      for (int id : {2144, 2148, 2154, 2158, 2188})
        if (d->tile_variant == id && 16 * (id / 10 % 10) >= dmax) plan->rows_dt = id / 10 % 10, plan->rows_nw = id % 10;
      if (d->tile_variant == 2001 + 10 * dt || d->tile_variant == 2002 + 10 * dt) rt = d->tile_variant % 10;
      if (rt > 0) {
        plan->split_dt = dt, plan->split_rt = rt;
        plan->nb = (int)((d->M + 16 * rt - 1) / (16 * rt));
        // Half of the columns to a workgroup (32 of 80), or a quarter of 128, where every workgroup still has a compute unit: 0.79 -
        // 0.96 of the time in nine of ten of 24000 random shapes, two workgroups to one 1.1 - 2.2 times as long.  What they pull of B
        // grows with the workgroups, and beyond these lines L2 gives it too slowly: with B as [K][L], whose rows of 32 keys are read
        // in pieces of 64 bytes, three fifths of the compute units past 300 keys (3 x 418 x 976 x 80 7.2 us against 5.9, 2 x 959 x
        // 944 x 64 6.2 / 5.6; at 300 all of them gain, 0.95) and two fifths past 800 (2 x 538 x 2320 x 64 8.7 against 7.7, 19 x 55 x
        // 2528 x 128 18.9 / 17.3); [L][K] at 64 columns four fifths past 1000 (20 x 81 x 3910 x 64 10.8 against 10.1).  Nor where more
        // batch entries than XCDs have so many keys that those an XCD's workgroups belong to pass its L2, 10 MB in all with [K][L]
        // (10 x 72 x 3392 x 128 23.3 / 17.3, 11 x 56 x 3216 x 128 25.5 / 18.4) and 18 MB with [L][K] up to 80 columns (18 x 46 x 3903 x
        // 80 15.3 / 14.0).  Within the lines one of the 24000 takes more than 1.03 (7 x 62 x 3728 x 128 [K][L], 1.04).  With [K][L] a quarter of 128 columns is level with
        // half from 500 keys on (2 x 224 x 1808 x 128 11.0 / 10.2; B [L][K] 21 x 25 x 944 x 128 7.0 / 7.6).
        const long long wgs = plan->nb * d->batch, bytes = 2 * d->batch * d->L * (d->K + d->N);
        auto blocks = [&](int ct) { return (d->N + 16 * ct - 1) / (16 * ct); };
        const int half = dt == 8 ? 4 : 2;
        const int fifths = kl_b ? (d->L <= 300 ? 5 : d->L <= 800 ? 3 : 2) : dt == 4 && d->L > 1000 ? 4 : 5;
        const bool spills = d->batch > 8 && bytes > (kl_b ? 10 << 20 : 18 << 20) && (kl_b || dt != 8);
        auto room = [&](int ct) { return 5 * wgs * blocks(ct) <= (long long)fifths * cus; };
        if (rt == 1 && blocks(half) > 1 && room(half) && !spills)
          plan->split_ct = dt == 8 && blocks(2) > blocks(4) && room(2) && (!kl_b || d->L <= 500) ? 2 : half;
        const int ct = plan->split_ct ? plan->split_ct : dt;
        ditto_tile_param& t = plan->tile;
        t.block_threads = 64 * ditto::kSplitWaves;
        t.block_m = 16 * rt;
        t.block_l = 32 * ditto::kSplitWaves;
        t.block_n = plan->split_ct ? 16 * ct : (int)d->N;
        t.head_pad = 16 * dt;
        t.lds_bytes = ditto::bmm_chain_split_lds(dt, ct, rt, kl_b);
        t.grid_x = (int)(wgs * (plan->split_ct ? blocks(ct) : 1));
        t.grid_y = t.grid_z = 1;
        t.variant = 2000 + 10 * dt + rt;
        return DITTO_OK;
      }
      // The same kernel at 64 and at 128 columns, where its short start and two workgroups on a compute unit tell.
      if (d->tile_variant == 0 && dt == 8 && rt == 0) {
        // Heads of 81 to 128, up to about 500 keys (600 with softmax), eight waves: against the pipelined 256-row kernel (9) at
        // every size measured (128 x 400 x 400 20.8 -> 18.8 us, 320 x 197 x 197 28.9 -> 25.3; 160 x 577 x 577 46.6 -> 45.0, but
        // 80 x 1024 x 1024 65.4 against 68.4), against 128-row workgroups where those take a second round and 256 rows do not
        // (160 x 197 x 197 18.8 -> 12.0, 80 x 400 x 400 25.0 -> 17.5; in one round 80 x 257 x 257 11.1 against 13.9), and against the
        // kernels of large grids unless those cover a head's rows in fewer blocks by taking 384 (512 x 197 x 197 33.2 -> 27.8,
        // 256 x 400 x 400 39.1 -> 35.2; 256 x 257 x 257 25.2 against 28.4, 256 x 577 x 577 61.3 / 66.5).
        const long long rows256 = (d->M + 255) / 256, n128 = ((d->M + 127) / 128) * d->batch;
        bool take = d->L <= (sm ? 600 : 450);
        if (plan->qt == 1) take = take && n128 > cus;
        if (plan->qt == 6 || plan->qt == 2) {
          const long long a384 = plan_rows_384(d->M, d->batch, cus), rest = d->M - 384 * a384;
          take = d->L <= 512 && (plan->qt == 2 || a384 + (rest > 0 ? (rest + 255) / 256 : 0) >= rows256);
        }
        if (take && launchable(n8, 512)) plan->rows_dt = 8, plan->rows_nw = 8;
      }
      if (d->tile_variant == 0 && dt == 4 && rt == 0 && sm && plan->qt != 6) {
        // Heads of up to 64 with softmax where the 64-row kernel, three workgroups to a compute unit, needs a second round and this
        // one in its four-wave form, of 128 rows, does not: on 250 shapes 0.74 - 0.86 of the time at 64 keys,
        // 0.83 - 0.96 at 200, 0.87 - 1.02 at 600 (256 x 197 x 197 10.9 -> 9.0 us, 512 x 100 x 100 9.6 -> 8.2).  Other sizes go by
        // their price.
        const long long n64 = ((d->M + 63) / 64) * d->batch, n128 = ((d->M + 127) / 128) * d->batch;
        if (n64 > 3LL * cus && n128 <= 2LL * cus && d->L <= 600 && launchable(n128, 256)) plan->rows_dt = 4, plan->rows_nw = 4;
      }
      if (d->tile_variant == 0 && dt == 4 && rt == 0 && !sm && n8 >= 2LL * cus && d->L <= 1024) {
        // Heads of up to 64 without softmax from two 256-row workgroups per compute unit on, up to 1024 keys: 512 x 197 x 197 16.8 ->
        // 12.2 us, 256 x 400 x 400 20.0 -> 16.6 (B [K][L] 22.3 -> 18.0), 256 x 577 x 577 35.0 -> 29.9, 128 x 1024 x 1024 35.3 -> 33.8;
        // below that the 64-row kernel's grain is worth more (160 x 400 x 400 13.6 against 15.4), and so it is with softmax
        // (256 x 400 x 400 21.0 against 22.8).
        const int nw = d->M <= 128 ? 4 : 8;
        if (launchable(((d->M + 32 * nw - 1) / (32 * nw)) * d->batch, 64 * nw)) plan->rows_dt = 4, plan->rows_nw = nw;
      }
      if (plan->rows_nw > 0) {
        plan->nb = (int)((d->M + 32 * plan->rows_nw - 1) / (32 * plan->rows_nw));
        ditto_tile_param& t = plan->tile;
        t.block_threads = 64 * plan->rows_nw;
        t.block_m = 32 * plan->rows_nw;
        t.block_l = ditto::kBN;
        t.block_n = (int)d->N;
        t.head_pad = 16 * plan->rows_dt;
        t.lds_bytes = ditto::bmm_chain_rows_lds(plan->rows_dt, plan->rows_nw, kl_b);
        t.grid_x = (int)(plan->nb * d->batch);
        t.grid_y = t.grid_z = 1;
        t.variant = 2100 + 10 * plan->rows_dt + plan->rows_nw;
        return DITTO_OK;
      }
    }
    if (d->tile_variant != 0) {
      const int q = d->tile_variant % 10;
      if (d->tile_variant / 10 != plan->d_pad || (q != 1 && q != 2 && q != 4 && q != 5 && q != 8 && q != 9 && q != 6 && q != 7))
        return fail(DITTO_EINVAL, "tile_variant %d cannot run this shape (head_pad %d; q must be 1, 2, 4, 5, 6, 7, 8 or 9)",
                    d->tile_variant, plan->d_pad);
      if ((q == 4 || q == 5) && plan->d_pad != 64)
        return fail(DITTO_EINVAL, "tile_variant %d: the 64-row kernel serves head_pad 64 only", d->tile_variant);
      plan->qt = q;
    }
    const bool kl = d->b_layout == DITTO_B_KL;
    const bool four16 = plan->qt == 4 || plan->qt == 5;  // four waves, 64-row workgroups
    const bool eight = plan->qt >= 6;  // 6, 8, 9: eight waves owning 32 rows each; 7: 48 rows each in some workgroups
    const bool m16 = plan->qt == 6 || plan->qt == 7;
    if (plan->qt == 6 && d->tile_variant == 0 && plan->d_pad == 128) {
      // the planner's own choice between all-256-row blocks (6) and the mix (7)
      if (plan_rows_384(d->M, d->batch, cus) > 0) plan->qt = 7;
    }
    if (plan->qt == 7) {
      plan->nb3 = plan_rows_384(d->M, d->batch, cus);
      if (plan->nb3 == 0 && d->M > 256) plan->nb3 = 1;  // asked for by tile_variant: at least one large block to show for it
    }
    const int bm = four16 ? 64 : eight ? 256 : 128 * plan->qt;
    ditto_tile_param& t = plan->tile;
    t.block_threads = eight ? 512 : 256;
    t.block_m = bm;
    t.block_l = ditto::kBN;
    t.block_n = (int)d->N;
    t.head_pad = plan->d_pad;
    if (four16)
      t.lds_bytes = ditto::bmm_chain4m16_lds_bytes<64>();
    else if (m16)
      t.lds_bytes = plan->d_pad == 64 ? ditto::bmm_chain8m16_lds_bytes<64>() : ditto::bmm_chain8m16_lds_bytes<128>();
    else if (eight)
      t.lds_bytes = plan->d_pad == 64 ? (kl ? ditto::bmm_chain8_lds_bytes<64, true>() : ditto::bmm_chain8_lds_bytes<64, false>())
                                      : (kl ? ditto::bmm_chain8_lds_bytes<128, true>() : ditto::bmm_chain8_lds_bytes<128, false>());
    else
      t.lds_bytes = plan->d_pad == 64 ? ditto::bmm_chain_lds_bytes<64>() : ditto::bmm_chain_lds_bytes<128>();
    plan->nb = (int)((d->M + bm - 1) / bm);
    if (plan->qt == 7) {
      const long long rest = d->M - 384LL * plan->nb3;
      plan->nb = plan->nb3 + (int)(rest > 0 ? (rest + 255) / 256 : 0);
      if (plan->nb3 > 0) t.block_m = 384;  // the larger of the two block sizes
    }
    t.grid_x = (int)(plan->nb * d->batch);
    t.grid_y = t.grid_z = 1;
    t.variant = plan->d_pad * 10 + plan->qt;
    return DITTO_OK;
  }
  if (in == DITTO_F32 || in == DITTO_F64) {
    if (d->acc_dtype != in || d->out_dtype != in)
      return fail(DITTO_EINVAL, "the fp32 / fp64 chain accumulates and outputs its input type");
    if (d->inter_op != DITTO_INTER_CAST && d->inter_op != DITTO_INTER_RELU && d->inter_op != DITTO_INTER_SOFTMAX)
      return fail(DITTO_EUNSUPPORTED, "the fp32 chain takes inter_op cast, relu or softmax");
    if (d->tile_variant != 0 && d->tile_variant != (in == DITTO_F64 ? 1001 : 1000))  // (the id that select_tile reports)
      return fail(DITTO_EINVAL, "tile_variant %d: the fp32 chain has a single variant, 1000 (fp64: 1001)", d->tile_variant);
    if (d->K > ditto::f32_chain_max_dim() || d->N > ditto::f32_chain_max_dim())
      return fail(DITTO_EUNSUPPORTED, "the fp32 chain supports K, N up to %d", ditto::f32_chain_max_dim());
    if (d->a_row_stride < d->K || d->c_row_stride < d->N || d->f_row_stride < d->N ||
        d->b_row_stride < (d->b_layout == DITTO_B_KL ? d->L : d->K))
      return fail(DITTO_EINVAL, "row stride smaller than row extent");
    if (d->a_row_stride > 0x7fffffff || d->b_row_stride > 0x7fffffff || d->c_row_stride > 0x7fffffff ||
        d->f_row_stride > 0x7fffffff)
      return fail(DITTO_EINVAL, "row stride too large");
    plan->family = 1;
    const bool f64 = in == DITTO_F64;
    // fp32 workgroups of 16 or of 32 rows: a 32-row one does twice the work in 0.9 of the time two 16-row ones take
    // (every B and C fragment fetched from L2 feeds two row tiles), and the fewer rounds over the compute units win.
    // Measured, us per launch, 16 / 32 rows: 12 x 512 x 512 x 64 14.4 / 12.9, 1 x 512 x 512 x 64 7.3 / 13.2,
    // 16 x 700 x 700 x 64 28.3 / 32.2, 64 x 512 x 512 x 64 49.9 / 49.5.  B stored [K][L] does not come through LDS and gains more from
    // feeding two row tiles: from 5 rounds against 3 on (44 x 428 x 112 x 64 19.6 / 16.7, 42 x 431 x 521 x 64 44.5 / 41.5; forty shapes of
    // 64 and 80 columns 0.93 in the mean, the worst 1.02; 8 against 5 0.87 - 1.03).  Rows that are loaded element by element do so with
    // softmax up to 64 columns (27 x 630 x 264, 48 -> 64 51.3 / 45.8; 16 shapes 0.85 - 0.91) and without it beyond (38 x 457 x 246,
    // 80 -> 64 60.4 / 55.0; 15 shapes 0.82 - 0.96); with columns that are no whole tiles from 7 against 4 on (41 x 664 x 462 x 43 85.4 /
    // 73.3, 44 x 575 x 131 x 72 65.0 / 58.6; [L][K] there 1.12 - 1.16).  Without softmax up to 64 columns the loads of one row tile
    // overlap better (42 x 642 x 149 x 32 31.7 / 37.3, 20 x 1292 x 87 x 56 37.2 / 42.4; 16 shapes 1.07 in the mean), and with softmax
    // beyond, where two spill registers, it takes some 200 keys to make up for that (18 x 978 x 125, 80 -> 64 47.3 / 50.8, 41 x 603 x
    // 92, 68 -> 75 47.0 / 50.4; 21 x 1236 x 466 x 72 124 / 113): 9 rounds against 5 there, as with [L][K].  Beyond 80 columns two row
    // tiles do not fit the registers.
    auto rounds = [&](int rows) { return (((d->M + rows - 1) / rows) * d->batch + cus - 1) / cus; };
    const bool wide = d->K > 64 || d->N > 64;
    const bool exact = ditto::f32_chain_exact((int)d->K, (int)d->N, d->a_batch_stride | d->c_batch_stride | d->f_batch_stride |
                                                                        d->a_row_stride | d->c_row_stride | d->f_row_stride);
    const bool gains = exact || (d->inter_op == DITTO_INTER_SOFTMAX ? !wide || d->L > 200 : wide);
    const double worth = d->b_layout != DITTO_B_KL || !gains ? 1.8 : d->K % 16 || d->N % 16 ? 1.7 : 1.65;
    plan->qt = !f64 && (d->K > 80 || d->N > 80 || (double)rounds(16) < worth * (double)rounds(32)) ? 1 : 2;
    plan->f32_width = f64 || plan->qt != 1 ? 0 : ditto::f32_chain_width((int)d->K, (int)d->N, ((d->M + 15) / 16) * d->batch, cus);
    plan->f32_cols = plan->f32_width ? (int)((d->N + plan->f32_width - 1) / plan->f32_width) : 1;
    ditto_tile_param& t = plan->tile;
    t.block_threads = f64 ? 256 : 512;
    t.block_m = 16 * plan->qt;
    t.block_n = plan->f32_width ? plan->f32_width : (int)d->N;
    t.head_pad = 0;
    t.block_l = f64 ? 32 : 128;
    t.lds_bytes = ditto::f32_chain_lds_bytes_host((int)d->K, (int)d->N, f64, plan->qt, plan->f32_width);
    t.grid_x = (int)(((d->M + t.block_m - 1) / t.block_m) * d->batch * plan->f32_cols);
    t.grid_y = t.grid_z = 1;
    t.variant = f64 ? 1001 : 1000;  // fp32 (MFMA) / fp64 (FMA) chain
    return DITTO_OK;
  }
  if (in == DITTO_I8) {
    if (d->acc_dtype != DITTO_I32 || (d->out_dtype != DITTO_I32 && d->out_dtype != DITTO_I8))
      return fail(DITTO_EINVAL, "the int8 chain accumulates in int32 and outputs int32 or (the low byte) int8");
    // requantised middle result, or the reference's wrapping cast (optionally behind a ReLU)
    if (d->inter_op != DITTO_INTER_REQUANT && d->inter_op != DITTO_INTER_CAST && d->inter_op != DITTO_INTER_RELU)
      return fail(DITTO_EUNSUPPORTED, "the int8 chain takes inter_op requant, cast (wrapping) or relu (then wrapping)");
    if (d->b_layout != DITTO_B_KL) return fail(DITTO_EUNSUPPORTED, "the int8 chain takes B as [K][L]");
    if (d->K % 16 || d->L % 16 || d->N % 16)
      return fail(DITTO_EINVAL, "K, L and N must be multiples of 16 for the int8 chain");
    if (d->a_row_stride % 16 || d->b_row_stride % 16 || d->c_row_stride % 16 || d->a_batch_stride % 16 ||
        d->b_batch_stride % 16 || d->c_batch_stride % 16)
      return fail(DITTO_EINVAL, "int8 input strides must be multiples of 16 elements");
    if (d->a_row_stride < d->K || d->b_row_stride < d->L || d->c_row_stride < d->N || d->f_row_stride < d->N)
      return fail(DITTO_EINVAL, "row stride smaller than row extent");
    if (d->a_row_stride > 0x7fffffff || d->b_row_stride > 0x7fffffff || d->c_row_stride > 0x7fffffff ||
        d->f_row_stride > 0x7fffffff || d->K > 0x7fffffff / 2 || d->N > 0x7fffffff / 2)
      return fail(DITTO_EINVAL, "extent or row stride too large");
    const long long Lp = (d->L + 255) / 256 * 256;
    if ((d->M + 64) * d->a_row_stride >= 0x7fffffffLL || d->K * d->b_row_stride >= 0x7fffffffLL ||
        Lp * d->c_row_stride >= 0x7fffffffLL)
      return fail(DITTO_EUNSUPPORTED, "a batch entry of A, B or C exceeds 2 GiB");
    // Compute units that would be idle take a share of the columns of the result, in blocks of 256: their workgroups repeat the
    // first product (2014 x 96 x 192 x 624 7.8 -> 5.9 us with three to a row block, 680 x 736 x 384 x 1024 15.9 -> 12.4).  Beyond a
    // workgroup to a compute unit that costs more than it saves (5020 x 352 x 224 x 448 7.2, 10.7 with two).
    const long long blocks256 = (d->N + 255) / 256;
    const long long rows32 = ((d->M + 31) / 32) * d->batch, most_slices = std::min(blocks256, std::max(1LL, cus / rows32));
    const long long blocks_per_slice = (blocks256 + most_slices - 1) / most_slices;
    // Few rows: the kernel whose waves take units of 64 x 64 weights, with as many workgroups to a row block (slices of its
    // columns) as pay.  Prices in us per launch, least squares over 300 random shapes (64 - 8192 rows, K and N 16 - 1024, L 16 -
    // 512) with 1 - 6 slices, root mean square error 5 %, the other kernel's over 800, 4 %, up to one round of its workgroups.  `pulls`: every
    // workgroup pulls all of B, and past two units of it a wave on all compute units L2 is the bound, 0.4 us a unit (6 x 208 x 992 x
    // 368 x 144 14.9 us where the other kernel takes 11.6, 1 x 3456 x 656 x 432 x 16 12.1 / 10.7).  It has to win by 5 %: of 4300 random
    // shapes that change kernels by that five take more than 1.03 of the other's time, the worst 1.07, the mean 0.78 (224 x 48 x 208 x 928
    // 7.8 -> 4.8 us, 256 x 912 x 96 x 800 10.4 -> 6.2, 1120 x 32 x 48 x 16 4.8 -> 3.8).
    {
      const double nl = (double)((d->L + 63) / 64), units1 = nl * (double)((d->K + 63) / 64) / 8;
      const long long nbt = (d->N + 63) / 64;
      const double chunks1 = (double)(Lp / 256 * ((d->K + 127) / 128)), chunks2 = (double)((d->L + 127) / 128 * blocks_per_slice);
      double best = 0.95 * (3.90 + 0.355 * chunks1 + 0.474 * chunks2 + 0.357e-6 * (double)(d->batch * d->M) * (double)d->N +
                            0.289 * (double)(rows32 * ((blocks256 + blocks_per_slice - 1) / blocks_per_slice)) / cus);
      if (d->tile_variant == 8101 || d->tile_variant == 8102) best = 1e30;
      for (int rt = 1; rt <= 2; ++rt) {
        if (d->tile_variant == 0 ? rows32 > cus : d->tile_variant != 8100 + rt) continue;
        const long long wgs = ((d->M + 16 * rt - 1) / (16 * rt)) * d->batch;
        for (long long s = 1; s <= nbt && s <= 16; ++s) {
          const long long blocks = (nbt + s - 1) / s;
          if ((nbt + blocks - 1) / blocks != s || ditto::i8_units_lds_bytes_host(d->L, rt, (int)std::min(blocks, 1LL << 20)) > 160 * 1024) continue;
          if (!launchable(wgs * s, 512)) break;
          const double rounds = (double)((wgs * s + cus - 1) / cus), units2 = nl * (double)blocks / 8, grid = (double)(wgs * s) / cus;
          const double pulls = 0.4 * std::max(0.0, grid * units1 - 2);
          const double price = pulls + (rt == 1 ? 3.17 + rounds * (0.07 + 0.155 * nl + 0.158 * blocks + 0.417 * units1 + 0.206 * units2 +
                                                           0.056 * ceil(units1) + 0.183 * ceil(units2)) + 0.472 * grid
                                       : 3.5 + rounds * (0.375 * nl + 0.306 * blocks + 0.582 * units1 + 0.474 * units2) + 0.568 * grid);
          if (price < best) best = price, plan->units_rt = rt, plan->slices = (int)s, plan->slice_blocks = (int)blocks;
        }
      }
      if (plan->units_rt > 0) {
        plan->family = 2;
        const int rt = plan->units_rt;
        ditto_tile_param& t = plan->tile;
        t.block_threads = 512;
        t.block_m = 16 * rt;
        t.block_l = 64;
        t.block_n = 64 * plan->slice_blocks;
        t.head_pad = 0;
        t.lds_bytes = (int)ditto::i8_units_lds_bytes_host(d->L, rt, plan->slice_blocks);
        t.grid_x = (int)(((d->M + 16 * rt - 1) / (16 * rt)) * d->batch * plan->slices);
        t.grid_y = t.grid_z = 1;
        t.variant = 8100 + rt;  // units of 64 x 64 weights; row tiles of 16
        return DITTO_OK;
      }
      if (d->tile_variant == 8101 || d->tile_variant == 8102)
        return fail(DITTO_EINVAL, "tile_variant %d cannot run this int8 chain (LDS or grid)", d->tile_variant);
    }
    // 64-row workgroups halve the weight traffic per row but need twice as many rows to fill the
    // chip; the ring of staged chunks is as deep as LDS allows (four or three stages, else two)
    int mt = ((d->M + 63) / 64) * d->batch >= 2LL * cus ? 2 : 1;
    auto fits = [&](int m, int n) { return ditto::i8_chain_lds_bytes_host((int)Lp, m, n) <= 160 * 1024; };
    int nst = mt == 2 ? 3 : 4;
    if (!fits(mt, nst)) nst = 2;
    if (!fits(mt, nst)) mt = 1, nst = 4;
    if (!fits(mt, nst)) nst = 2;
    if (d->tile_variant != 0) {
      // 8000 + 10 * (row tiles of 32) + ring depth, as select_tile reports it
      const int fm = (d->tile_variant - 8000) / 10, fn = d->tile_variant % 10;
      const bool built = (fm == 1 && (fn == 2 || fn == 4)) || (fm == 2 && (fn == 2 || fn == 3));
      if (d->tile_variant < 8000 || !built || !fits(fm, fn))
        return fail(DITTO_EINVAL, "tile_variant %d cannot run this int8 chain (8012, 8014, 8022, 8023, 8101 or 8102, within LDS)",
                    d->tile_variant);
      mt = fm, nst = fn;
    }
    plan->slice_blocks = (int)(mt == 1 ? blocks_per_slice : blocks256);
    plan->slices = (int)((blocks256 + plan->slice_blocks - 1) / plan->slice_blocks);
    const int lds = ditto::i8_chain_lds_bytes_host((int)Lp, mt, nst);
    if (lds > 160 * 1024)
      return fail(DITTO_EUNSUPPORTED, "L=%lld: the requantised row block does not fit in LDS", (long long)d->L);
    plan->family = 2;
    plan->d_pad = mt;
    plan->qt = nst;
    ditto_tile_param& t = plan->tile;
    t.block_threads = ditto::i8_chain_threads();
    t.block_m = 32 * mt;
    t.block_l = (int)Lp;
    t.block_n = 256 * plan->slice_blocks;
    t.head_pad = 0;
    t.lds_bytes = lds;
    t.grid_x = (int)(((d->M + 32 * mt - 1) / (32 * mt)) * d->batch * plan->slices);
    t.grid_y = t.grid_z = 1;
    t.variant = 8000 + 10 * mt + nst;  // int8 chain: 8000 + 10 * (row tiles of 32) + ring depth
    return DITTO_OK;
  }
  return fail(DITTO_EUNSUPPORTED, "no chain kernel for in_dtype %d", in);
}

struct ConvPlan {
  int px2;             // 0: 1x1 second convolution; 1 | 2: larger one, output-pixel tiles per wave
  size_t w2p_bytes;    // size of the repacked W2 (second part of the workspace, px2 > 0)
  int c1_tiles;
  int ch;              // input channels per staged chunk
  size_t w1p_bytes;    // size of the repacked W1 (the workspace)
  ditto::ConvChainArgs args;
  bool dw;             // depthwise first convolution: dwargs / c2_tiles / dw_shared describe the launch
  int c2_tiles;
  int dw_mode;         // 0 | 1: plain kernel (1: multiplier a multiple of 8); 2 | 3: persistent kernel,
                       // depthwise stage on the matrix cores (2) or the vector ALU (3); 4: the row-streaming
                       // kernel (rowargs); 5: the row-streaming kernel for multiplier 16 (row16args)
  ditto::DwConvArgs dwargs;
  ditto::DwRowsArgs rowargs;
  ditto::Dw16RowsArgs row16args;
  bool resident;       // 1x1 -> 3x3 with at most 64 channels: persistent kernel, W2 resident in LDS
  int res_grid;
  ditto::ConvResidentArgs rargs;
  bool rows13;         // 1x1 -> 3x3 with at most 64 channels everywhere: the same pipeline (cvargs.f13), W2 fragments
                       // in the workspace
  bool rows31;         // 3x3 -> 1x1 with at most 64 -> 64 -> 256 channels: the row pipeline (cvargs), W1 fragments
                       // in the workspace
  ditto::ConvRowsArgs cvargs;
  bool tiles;          // dense -> 1x1 on tiles of whole output rows (targs), both weights as fragments in the workspace
  ditto::ConvTilesArgs targs;
  bool tiles13;        // 1x1 -> 3x3 with at most 64 channels on tiles of whole output rows (t13args), weights likewise
  ditto::Conv13TilesArgs t13args;
  ditto::DwTilesArgs dwtargs;
  ditto_tile_param tile;
};

// Depthwise first convolution + 1x1 second (dw_conv_chain.h): everything in one kernel, no workspace.
// dw_mode 2 | 3: the persistent kernel, depthwise stage on the matrix cores (multipliers that are
// multiples of 16) or on the vector ALU (3x3, multiplier 1, 2, 4, 8); dw_mode 0 | 1: the plain
// kernel for what is left (1: multiples of 8, 0: 1, 2, 4).
// dw_mode 4: the row-streaming kernel (dw_rows.h) for multiplier 1, 3x3, pad 1, stride 1, at most 32 input and
// 64 output channels, image rows of whole 16-byte vectors and at most 128 pixels, 16-bit output.
// vec_cap: the widest halo vector (elements) the pointer of this call allows; 8 when planning without one.
// DITTO_DW_ROWS=0 keeps such shapes on the persistent kernel (A/B runs, tests of that kernel).
// dw_mode 5: the row-streaming kernel for multiplier 16 (dw16_rows.h): 3x3, pad 1, stride 1, an even number of at
// most 32 input channels, at most 64 output channels, image rows of whole 16-byte vectors whose ring of row slots
// fits beside the filters in LDS, 16-bit output.  DITTO_DW16_ROWS=0 keeps such shapes on the persistent kernel.
// dw_mode 6: tiles of whole output rows (dwtargs).
// What a forced tile_variant allows (0: everything; see ditto_conv_chain_desc.tile_variant).
struct ConvSteer {
  int tv = 0;
  bool rows = true;      // 3700 / 3800: the row pipelines
  bool resident = true;  // 3600: the persistent kernel with W2 resident in LDS
  bool dw_rows = true;   // 4024
  bool dw16_rows = true; // 4025
  bool tiles = true;     // 3200: tiles of whole output rows
  bool tiles13 = true;   // 3300: tiles of whole output rows, 1x1 -> 3x3
  bool dw_tiles = true;  // 4100: depthwise, tiles of whole output rows
  bool persist = false;  // 3900: the persistent 3x3 -> 1x1 kernel (switched off)
};
int conv_steer(int tv, ConvSteer* st) {
  *st = ConvSteer();
  st->tv = tv;
  if (tv == 0) return DITTO_OK;
  if (tv < 0) return fail(DITTO_EINVAL, "tile_variant must be 0, a variant id or a family id");
  const int fam = tv / 100 * 100;
  st->rows = fam == 3700 || fam == 3800;
  st->resident = fam == 3600;
  st->tiles = fam == 3200;
  st->tiles13 = fam == 3300;
  st->dw_rows = tv == 4024;
  st->dw16_rows = tv == 4025;
  st->dw_tiles = fam == 4100;
  st->persist = fam == 3900;
  if (!(fam == 3000 || fam == 3100 || fam == 3200 || fam == 3300 || fam == 3500 || fam == 3600 || fam == 3700 || fam == 3800 || fam == 3900 || fam == 4000 ||
        fam == 4100))
    return fail(DITTO_EINVAL, "tile_variant %d names no conv chain kernel family", tv);
  return DITTO_OK;
}
// The plan that came out against the variant that was asked for: a family id (a multiple of 100; 3000 also stands
// for the 16-channel-chunk form 31xx, 4000 for every depthwise kernel but the two row-streaming ones) or an exact id.
int conv_steer_check(const ConvSteer& st, int got) {
  if (st.tv == 0 || st.tv == got) return DITTO_OK;
  if (st.tv % 100 == 0) {
    const int fam = got / 100 * 100;
    if (fam == st.tv || (st.tv == 3000 && fam == 3100)) {
      if (st.tv != 4000 || (got != 4024 && got != 4025)) return DITTO_OK;
    }
  }
  return fail(DITTO_EINVAL, "tile_variant %d cannot run this chain (the kernel that fits it under that constraint is %d)",
              st.tv, got);
}

// Depthwise 3x3 on tiles of whole output rows (dw_tiles.h), where it can run the shape at all.
bool plan_dw_tiles(const ditto_conv_chain_desc* d, long long P, long long Q, ConvPlan* plan, int cus) {
  const int mult = (int)(d->C1 / d->C0), slots = 16 * ditto::kDtMaxTiles;
  if (!(mult == 16 || mult == 1) || d->R1 != 3 || d->S1 != 3 || d->pad1 != 1 || d->C2 > 64 || d->W < 8 || Q > slots ||
      (mult == 1 && d->C0 % 8) || d->C0 * d->H * d->W > 0x3fffffff)
    return false;
  auto rows_in = [&](int th) { return (int)((th - 1) * d->stride1 + 3); };
  // A workgroup has eight waves and a tile of 16 pixels needs one: where half or three quarters of them would have none, two or
  // four waves share out the channels of a tile.
  auto groups_of = [&](int th) { return th * Q <= 4 * ditto::kDtWaves ? 4 : th * Q <= 8 * ditto::kDtWaves ? 2 : 1; };
  auto lds_of = [&](int th) {
    return ditto::dw_tiles_lds_bytes(mult, rows_in(th), (int)d->W, d->C2 <= 32 ? 2 : 4, groups_of(th));
  };
  if (lds_of(1) > 160 * 1024) return false;
  // Rows per workgroup.  A workgroup of one pixel tile per wave takes two units alone on a compute unit and three (multiplier
  // 1: 2.6) beside another, one of two tiles 3 and 4.6 (5.2), with two waves to a tile 1.5 and 2.4 (1.9 and 2.3), with four 1.25
  // and 2 (1.65 and 2.1); a compute unit holds two.  The height with the fewest units on the busiest compute unit wins, the smaller
  // one on ties (32 x 64 x 56 x 56 times 16: one row 63 us, two 38, four 29.5; times 1: 22, 16.2, 18.3; 11 x 64 x 28 x 28 times
  // 16: one row 13.1, two 10.6, four 13.7; times 1: 7.2, 6.3, 6.7; 22 x 32 x 23 x 23 times 1: one
  // row 5.8, three 5.2).
  int th = 1;
  double best = 0;
  for (int t = 1; t <= P && t * Q <= slots && lds_of(t) <= 160 * 1024; ++t) {
    const int k = t * Q > 16 * ditto::kDtWaves ? 0 : groups_of(t) == 1 ? 1 : groups_of(t) == 2 ? 2 : 3;
    static constexpr double kAlone[2][4] = {{3, 2, 1.9, 1.65}, {3, 2, 1.5, 1.25}}, kPair[2][4] = {{5.2, 2.6, 2.3, 2.1}, {4.6, 3, 2.4, 2}};
    const double alone = kAlone[mult == 16][k], pair = kPair[mult == 16][k];
    const long long wgs = d->N * ((P + t - 1) / t), per_round = 2LL * lds_of(t) <= 160 * 1024 ? 2 * cus : cus;
    const long long full = wgs / per_round, rest = wgs % per_round;
    const double cost = full * (per_round > cus ? pair : alone) + (rest > cus ? pair : rest > 0 ? alone : 0);
    if (t == 1 || cost < best) best = cost, th = t;
  }
  if (!launchable(d->N * ((P + th - 1) / th), 64 * ditto::kDtWaves)) return false;
  ditto::DwTilesArgs& a = plan->dwtargs;
  a.N = (int)d->N; a.C0 = (int)d->C0; a.H = (int)d->H; a.W = (int)d->W; a.C2 = (int)d->C2;
  a.P = (int)P; a.Q = (int)Q; a.stride = (int)d->stride1;
  a.TH = th;
  a.tiles_h = (int)((P + th - 1) / th);
  a.rows_in = rows_in(th);
  a.groups = groups_of(th);
  a.relu_mid = d->inter_op == DITTO_INTER_RELU;
  a.relu_out = d->relu_out != 0;
  a.out_f32 = d->out_dtype == DITTO_F32;
  a.inv_blocks = 1.f / (float)ditto::dw_tiles_row_blocks((int)d->W);
  a.inv_rows = 1.f / (float)a.rows_in;
  a.inv_group = 1.f / (float)ditto::dw_tiles_group_blocks(a.rows_in, (int)d->W);
  a.inv_q = 1.f / (float)Q;
  plan->dw_mode = 6;
  ditto_tile_param& t = plan->tile;
  t.block_threads = 64 * ditto::kDtWaves;
  t.block_m = th * (int)Q;
  t.block_l = ditto::dw_tiles_chunk(mult) * mult;
  t.block_n = d->C2 <= 32 ? 32 : 64;
  t.head_pad = 0;
  t.lds_bytes = lds_of(th);
  t.grid_x = a.N * a.tiles_h;
  t.grid_y = th;
  t.grid_z = (int)Q;
  t.variant = 4100 + th;
  return true;
}

int plan_dw_conv(const ditto_conv_chain_desc* d, const ConvSteer& steer, long long P, long long Q, ConvPlan* plan,
                 bool need_device, bool allow_dwv = true, int vec_cap = 8, bool allow_rows = true) {
  if (d->C1 % d->C0) return fail(DITTO_EINVAL, "depthwise: C1 must be a multiple of C0");
  const long long mult = d->C1 / d->C0;
  const long long RS = d->R1 * d->S1;
  if (!(d->R2 == 1 && d->S2 == 1 && d->pad2 == 0 && d->stride2 == 1))
    return fail(DITTO_EUNSUPPORTED, "depthwise chain: the second convolution must be 1x1, stride 1, no padding");
  // the persistent kernel: depthwise stage on the matrix cores (multipliers that are multiples of 16)
  // or, for 3x3 filters with multiplier 1, 2, 4, 8 (and whole 16-byte vectors of W1, W2), on the vector ALU
  // (that variant is built with the 16-byte output stores only: output rows of a multiple of 8, not fp32)
  const bool dwv = allow_dwv && d->R1 == 3 && d->S1 == 3 && (mult == 1 || mult == 2 || mult == 4 || mult == 8) &&
                   d->C1 % 8 == 0 && Q % 8 == 0 && d->out_dtype != DITTO_F32;
  const bool mfma = (mult % 16 == 0 && RS <= ditto::kDwMfmaTaps) || dwv;
  if (!mfma && RS > 2 * ditto::kDwPairs - 1)
    return fail(DITTO_EUNSUPPORTED,
                "depthwise chain: filters of at most 9 taps (16 when the channel multiplier is a multiple of 16)");
  if (!(mult == 1 || mult == 2 || mult == 4 || mult % 8 == 0))
    return fail(DITTO_EUNSUPPORTED, "depthwise chain: channel multiplier must be 1, 2, 4 or a multiple of 8");
  if (d->C2 > 256) return fail(DITTO_EUNSUPPORTED, "depthwise chain: at most 256 output channels");
  if (d->C1 > 32768) return fail(DITTO_EUNSUPPORTED, "depthwise chain: at most 32768 intermediate channels");
  memset(plan, 0, sizeof(*plan));
  plan->dw = true;
  if (allow_rows && vec_cap >= 8 && steer.dw_rows && mult == 1 && d->R1 == 3 && d->S1 == 3 && d->pad1 == 1 &&
      d->stride1 == 1 && d->C0 <= ditto::kDwRowsC && d->C2 <= 64 && d->W % 8 == 0 && d->W <= 128 &&
      d->out_dtype != DITTO_F32 && d->H * d->W * 64 < 0x7fffffffLL) {
    // Bands of whole output rows, one workgroup each: all input rows of a band stay in LDS.  Among the
    // band heights that fit, the one with the fewest row steps on the busiest CU (a band costs its rows
    // plus the two halo rows plus about three steps of start-up).
    const int cus = need_device ? device_cus() : 256;
    int band_max = 0;
    while (band_max < d->H && ditto::dw_rows_lds_bytes((int)d->W, band_max + 1) <= 160 * 1024) ++band_max;
    if (band_max >= 1) {
      long long best = -1;
      int best_nb = 0;
      const int nb_min = (int)((d->H + band_max - 1) / band_max);
      for (int nb = nb_min; nb <= d->H && nb < nb_min + 64; ++nb) {
        const int band = (int)((d->H + nb - 1) / nb);
        const long long wgs = d->N * ((d->H + band - 1) / band);
        const long long cost = ((wgs + cus - 1) / cus) * (band + 5);
        if (best < 0 || cost < best) { best = cost; best_nb = nb; }
      }
      ditto::DwRowsArgs& r = plan->rowargs;
      r.N = (int)d->N; r.C0 = (int)d->C0; r.H = (int)d->H; r.W = (int)d->W; r.C2 = (int)d->C2;
      r.band = (int)((d->H + best_nb - 1) / best_nb);
      r.bands = (int)((d->H + r.band - 1) / r.band);
      r.relu_mid = d->inter_op == DITTO_INTER_RELU;
      r.relu_out = d->relu_out != 0;
      plan->dw_mode = 4;
      plan->c2_tiles = 2;
      ditto_tile_param& t = plan->tile;
      t.block_threads = 64 * ditto::kDwRowsWaves;
      t.block_m = r.band * r.W;
      t.block_l = ditto::kDwRowsC;
      t.block_n = 64;
      t.head_pad = 0;
      t.lds_bytes = ditto::dw_rows_lds_bytes(r.W, r.band);
      t.grid_x = r.N * r.bands;
      t.grid_y = r.band;
      t.grid_z = r.W;
      t.variant = 4000 + 20 + 4;
      return DITTO_OK;
    }
  }
  const bool rows16 = mult == 16 && d->R1 == 3 && d->S1 == 3 && d->pad1 == 1 && d->stride1 == 1 && d->C0 <= 32 &&
                      d->C0 % 2 == 0 && d->C2 <= 64 && d->W % 8 == 0 && d->W >= 8 &&
                      ditto::dw16_rows_ni((int)d->C0, (int)d->W) <= 8 &&
                      ditto::dw16_rows_lds_bytes((int)d->C0, (int)d->W) <= 160 * 1024 && d->H * d->W < (1 << 20);
  if (allow_rows && vec_cap >= 8 && steer.dw16_rows && rows16 && d->out_dtype != DITTO_F32) {
    // Bands of whole output rows, one workgroup each, whose pixels eight waves take as one stream of 32-pixel
    // tiles: the band height with the fewest tiles on the busiest SIMD (waves w and w + 4 share one) over
    // the rounds of workgroups, a workgroup's start-up counted as three tiles.
    const int cus = need_device ? device_cus() : 256;
    long long best = -1;
    int best_band = 1;
    for (int nb = 1; nb <= d->H; ++nb) {
      const int band = (int)((d->H + nb - 1) / nb);
      if (nb > 1 && band == (int)((d->H + nb - 2) / (nb - 1))) continue;
      const long long wgs = d->N * ((d->H + band - 1) / band);
      const long long ntiles = (band * d->W + 31) / 32;
      const long long q = ntiles / ditto::kDw16Compute, rem = ntiles % ditto::kDw16Compute;
      const long long busiest = 2 * q + (rem > 0) + (rem > 4);
      const long long cost = ((wgs + cus - 1) / cus) * (busiest + 3);
      if (best < 0 || cost <= best) { best = cost; best_band = band; }
    }
    ditto::Dw16RowsArgs& r = plan->row16args;
    r.N = (int)d->N; r.C0 = (int)d->C0; r.H = (int)d->H; r.W = (int)d->W; r.C2 = (int)d->C2;
    r.band = best_band;
    r.bands = (int)((d->H + r.band - 1) / r.band);
    r.ring = ditto::dw16_rows_ring(r.W);
    r.relu_mid = d->inter_op == DITTO_INTER_RELU;
    r.relu_out = d->relu_out != 0;
    plan->dw_mode = 5;
    plan->c2_tiles = 2;
    ditto_tile_param& t = plan->tile;
    t.block_threads = 64 * ditto::kDw16Waves;
    t.block_m = r.band * r.W;
    t.block_l = (int)d->C1;
    t.block_n = 64;
    t.head_pad = 0;
    t.lds_bytes = ditto::dw16_rows_lds_bytes(r.C0, r.W);
    t.grid_x = r.N * r.bands;
    t.grid_y = r.band;
    t.grid_z = r.W;
    t.variant = 4000 + 20 + 5;
    return DITTO_OK;
  }
  // Tiles of whole output rows: what the two row-streaming kernels do not take (they keep all weights in LDS: 8 x 32 x 56 x
  // 56 times 16 7.6 us against 8.9, 32 x 32 x 56 x 56 times 1 7.8 / 12.5; level or up to 9 % behind on one to four images,
  // whose kernel alone takes less than the host's call), 1.3 to 7 times the kernels below: 32 x 64 x 56 x 56
  // times 16 -> 64 52.5 / 29.5 us, 8 x 32 x 37 x 37 times 16 25.6 / 9.1, 32 x 16 x 147 x 147 times 16 stride 2 127 / 19, 32 x
  // 64 x 112 x 112 times 1 73 / 48.  (The fp32 output of a shape the second one takes stays below, whose order of
  // accumulation is that kernel's.)
  if (steer.dw_tiles && (!rows16 || steer.tv > 0) && plan_dw_tiles(d, P, Q, plan, need_device ? device_cus() : 256)) return DITTO_OK;
  plan->dw_mode = dwv ? 3 : mfma ? 2 : mult % 8 == 0 ? 1 : 0;
  const int c2t = d->C2 <= 32 ? 1 : d->C2 <= 64 ? 2 : d->C2 <= 128 ? 4 : 8;
  const int pxw = mfma ? ditto::dw_mfma_pxw(c2t) : c2t == 8 ? 1 : 2;
  const int groups = mfma ? ditto::dw_mfma_groups(c2t) : 1;
  const int slots = 128 * groups * pxw;  // pixels of a workgroup's tile
  ditto::DwConvArgs& a = plan->dwargs;
  a.N = (int)d->N; a.C0 = (int)d->C0; a.H = (int)d->H; a.W = (int)d->W;
  a.mult = (int)mult; a.C1 = (int)d->C1; a.R = (int)d->R1; a.S = (int)d->S1;
  a.pad = (int)d->pad1; a.stride = (int)d->stride1; a.C2 = (int)d->C2; a.P = (int)P; a.Q = (int)Q;
  // Pixel tile: the split of the output plane into TH x TW pieces of at most `slots` pixels that
  // costs the fewest 32-pixel tile rounds (a round = one tile on each wave; the plain kernel always
  // runs all its rounds); ties go to the wider tile.  Where 16-byte output stores are possible only
  // tile widths that keep them (multiples of 8) are considered.
  const bool want_wide = mfma && d->out_dtype != DITTO_F32 && Q % 8 == 0;
  for (int pass = want_wide ? 0 : 1; pass < 2; ++pass) {  // pass 0: only widths that are multiples of 8
    long long best = -1;
    for (int k = 1; k <= (int)Q; ++k) {
      const int tw = (int)((Q + k - 1) / k);
      if (tw > slots) continue;
      if (tw < 8 && k > 1) break;
      if (pass == 0 && tw % 8) continue;
      int th = slots / tw;
      if (th > P) th = (int)P;
      const long long th_n = (P + th - 1) / th;
      th = (int)((P + th_n - 1) / th_n);
      const long long tw_n = (Q + tw - 1) / tw;
      const long long rounds = mfma ? ((th * tw + 31) / 32 + 4 * groups - 1) / (4 * groups) : pxw;
      const long long cost = th_n * tw_n * rounds;
      if (best < 0 || cost < best) { best = cost; a.TH = th; a.TW = tw; }
    }
    if (best >= 0) break;
  }
  // input channels per chunk: chx * mult a multiple of the MFMA block (32 intermediate channels
  // on the matrix-core path, 16 on the vector path); as many channels as keep two workgroups on a
  // CU, else as many as fit at all, else a smaller pixel tile
  const int cm_unit = mfma ? 32 : 16;
  int step = 1;
  while ((step * mult) % cm_unit) ++step;
  // halo loads: vectors of up to 8 elements that divide W (the run call narrows them if x is less
  // aligned); output through 16-byte stores when rows allow
  const int vec_max = mfma ? (d->W % 8 == 0 && vec_cap >= 8 ? 8 : d->W % 4 == 0 ? 4 : d->W % 2 == 0 ? 2 : 1) : 1;
  a.vec = vec_max;
  a.wide = mfma && d->out_dtype != DITTO_F32 && Q % 8 == 0 && a.TW % 8 == 0;
  auto lds_of = [&](int chx) {
    return mfma ? ditto::dw_conv_mfma_lds_bytes(chx, a.mult, a.rows_in, a.cols_al, 32 * c2t, groups, a.wide != 0)
                : ditto::dw_conv_lds_bytes(chx, a.mult, a.rows_in, a.cols_in, 32 * c2t) + 16;
  };
  // the MFMA kernel keeps a chunk's halo tile in flight in registers (kDwXpf vectors per thread)
  // and addresses it with packed 32-bit offsets
  auto fits_regs = [&](int chx) {
    if (!mfma) return true;
    // a thread owns one (row, vector) position of the halo tile and walks the channels, `cphases`
    // at a time: kDwXpf passes must cover the chunk
    const int nvr = a.cols_al / a.vec;
    const int cphases = (256 * groups / nvr) / a.rows_in;
    const int passes_max = a.vec == 8 ? ditto::kDwXpf / 2 : ditto::kDwXpf;  // a 16-byte vector takes two entries
    return cphases >= 1 && (chx + cphases - 1) / cphases <= passes_max &&
           (long long)(chx + 1) * d->H * d->W < 0x7fffffffLL;
  };
  const int chx_max = (int)((d->C0 + step - 1) / step) * step;
  int lds = 0;
  for (;;) {
    a.rows_in = (a.TH - 1) * a.stride + a.R;
    a.cols_in = (a.TW - 1) * a.stride + a.S;
    a.chx = 0;
    // everything resident (one chunk, filters staged once per workgroup) with the widest loads
    // that leave room for it ...
    for (int vec = vec_max; mfma && vec >= 1 && !a.chx; vec >>= 1) {
      a.vec = vec;
      a.cols_al = (a.cols_in + 2 * vec - 2) / vec * vec;
      a.cols_al += a.cols_al & 1;
      // 16-byte vectors halve the load and LDS-write instructions of the halo staging (5-6 % of the
      // kernel on 16-wide tiles) but pad the halo rows more: not where that is over a third
      if (vec == 8 && 3 * a.cols_al > 4 * ((a.cols_in + 6) / 4 * 4)) continue;
      lds = lds_of(chx_max);
      if (lds <= 160 * 1024 && fits_regs(chx_max)) a.chx = chx_max;
    }
    // ... else chunks: small enough for two workgroups per CU, else whatever fits
    if (!a.chx) {
      a.vec = vec_max;  // 16-byte vectors under the same padding rule as above
      if (a.vec == 8 && 3 * ((a.cols_in + 14) / 8 * 8) > 4 * ((a.cols_in + 6) / 4 * 4)) a.vec = 4;
      a.cols_al = (a.cols_in + 2 * a.vec - 2) / a.vec * a.vec;
      a.cols_al += a.cols_al & 1;
      for (int limit : {78 * 1024, 150 * 1024}) {
        for (int chx = chx_max; chx >= step; chx -= step) {
          lds = lds_of(chx);
          if (lds <= limit && fits_regs(chx)) { a.chx = chx; break; }
        }
        if (a.chx) break;
      }
    }
    if (a.chx) break;
    if (a.TH > 1) a.TH = (a.TH + 1) / 2;
    else if (a.TW > 16) { a.TW = (a.TW + 1) / 2; a.wide = a.wide && a.TW % 8 == 0; }
    else return fail(DITTO_EUNSUPPORTED, "depthwise chain tile does not fit in LDS");
  }
  {  // same number of chunks, evenly sized
    const int chunks = (int)((d->C0 + a.chx - 1) / a.chx);
    const int even = (int)((d->C0 + chunks - 1) / chunks);
    a.chx = (even + step - 1) / step * step;
    lds = lds_of(a.chx);
  }
  a.tiles_h = (int)((P + a.TH - 1) / a.TH);
  a.tiles_w = (int)((Q + a.TW - 1) / a.TW);
  a.relu_mid = d->inter_op == DITTO_INTER_RELU;
  a.relu_out = d->relu_out != 0;
  a.out_f32 = d->out_dtype == DITTO_F32;
  if (dwv && !a.wide) return plan_dw_conv(d, steer, P, Q, plan, need_device, false, vec_cap, false);  // that variant needs the wide stores
  plan->c2_tiles = c2t;
  ditto_tile_param& t = plan->tile;
  t.block_threads = 256 * groups;
  t.block_m = a.TH * a.TW;
  t.block_l = a.chx * a.mult;
  t.block_n = 32 * c2t;
  t.head_pad = 0;
  t.lds_bytes = lds;
  t.grid_x = a.N * a.tiles_h * a.tiles_w;
  if (mfma) {  // persistent workgroups, as many as the CUs hold at this LDS footprint
    // two workgroups per CU where LDS and registers allow: the eight-wave variants use more than
    // 128 registers per lane, so only one of them fits
    const int per_cu = (groups == 1 && 160 * 1024 / lds >= 2) ? 2 : 1;
    const int cap = (need_device ? device_cus() : 256) * per_cu;
    if (t.grid_x > cap) t.grid_x = cap;
    a.grid = t.grid_x;
    a.nt_store = (a.TW * 2) % 128 == 0;
  }
  t.grid_y = a.TH;
  t.grid_z = a.TW;
  t.variant = 4000 + c2t * 10 + plan->dw_mode;
  return DITTO_OK;
}

int plan_conv_steered(const ditto_conv_chain_desc* d, const ConvSteer& steer, ConvPlan* plan, bool need_device,
                      int dw_vec_cap, bool allow_resident, bool allow_dw_rows);

// Dense -> 1x1 on tiles of whole output rows (conv_tiles.h), where that is the kernel for the shape (`forced`: where it can
// run it at all).
bool plan_conv_tiles(const ditto_conv_chain_desc* d, long long P, long long Q, bool forced, ConvPlan* plan, int cus) {
  const int slots = 16 * ditto::kCtMaxTiles;
  if (d->W < 8 || Q > slots) return false;
  const int c0p = (int)((d->C0 + 31) / 32 * 32), c1p = ditto::conv_tiles_c1p((int)d->C1);
  const int cols_in = (int)((Q - 1) * d->stride1 + d->S1);
  auto rows_in = [&](int th) { return (int)((th - 1) * d->stride1 + d->R1); };
  auto lds_of = [&](int th) { return ditto::conv_tiles_lds_bytes(rows_in(th), cols_in, c0p, c1p, slots); };
  if (lds_of(1) > 160 * 1024) return false;
  // The general kernel stays ahead on stride-1 filters over few channels whose image rows are whole 16-byte vectors, with a
  // tile of four rows and more for every compute unit (32 x 64 x 56 x 56 3x3 -> 64 -> 64 15.2 against 15.7 us, 32 x 32 x 56 x 56
  // -> 32 -> 128 11.2 / 15.4, 10 x 64 x 72 x 72 -> 64 -> 256 16.4 / 18.2); with two rows per tile it is behind (8 x 64 x 104 x 104
  // 39.3 / 26.2), and so it is everywhere else: 8 x 32 x 147 x 147 stride 2 -> 64 -> 80 21.5 / 13.3, one image of 128 x 28 x 28 ->
  // 256 -> 128 45.6 / 9.2, 21 x 64 x 106 x 106 stride 2 -> 192 -> 128 109 / 31, 32 x 256 x 56 x 56 1x1 -> 256 -> 64 83 / 31.
  const long long old_rows = d->W > 0 ? 256 / d->W : 0;
  if (!forced && d->W % 8 == 0 && d->stride1 == 1 && d->R1 * d->S1 > 1 && d->C1 <= 64 && old_rows >= 3 &&
      d->N * ((P + old_rows - 1) / old_rows) >= cus)
    return false;
  // Rows per workgroup.  A workgroup streams all of W1 whatever its rows, at 64 bytes per clock - as long as the MFMAs of
  // four pixel tiles take - and fetches its halo rows; the fewest clocks over the rounds of workgroups win, a third more
  // where only one workgroup fits a compute unit (its phases then overlap with nobody's).  Strided filters take few halo
  // rows in common with their neighbours, so their workgroups stay at one output row as soon as that fills three pixel
  // tiles or the grid is small (8 x 16 x 227 x 227 stride 4: one row 7.5 us, two 9.8; 32 x 32 x 112 x 112 stride 2 15.9 / 19.1).
  const long long k_w1 = d->R1 * d->S1 * (c0p / 32) * (c1p / 16);
  int th = 1;
  double best = 0;
  for (int t = 1; t <= P && t * Q <= slots && lds_of(t) <= 160 * 1024; ++t) {
    const long long wgs = d->N * ((P + t - 1) / t), rounds = (wgs + cus - 1) / cus;
    const double work = (double)k_w1 * std::max(16LL, 4 * ((t * Q + 15) / 16)) + rows_in(t) * (double)(d->W * c0p) / 12 + 300;
    const double cost = rounds * work * (rounds > 1 && 2 * lds_of(t) > 160 * 1024 ? 1.35 : 1.0);
    if (t == 1 || cost < best) best = cost, th = t;
    if (d->stride1 > 1 && (t * Q > 32 || wgs <= 2 * cus)) {
      th = t;
      break;
    }
  }
  const ditto::ConvTilesSplit w = ditto::conv_tiles_split((int)d->C1, (int)(d->R1 * d->S1) * c0p / 32);
  if (!launchable(d->N * ((P + th - 1) / th), 64 * w.wc * w.wp)) return false;
  ditto::ConvTilesArgs& a = plan->targs;
  a.N = (int)d->N; a.C0 = (int)d->C0; a.H = (int)d->H; a.W = (int)d->W; a.C1 = (int)d->C1; a.C2 = (int)d->C2;
  a.R = (int)d->R1; a.S = (int)d->S1; a.pad = (int)d->pad1; a.stride = (int)d->stride1;
  a.P = (int)P; a.Q = (int)Q;
  a.TH = th;
  a.tiles_h = (int)((P + th - 1) / th);
  a.rows_in = rows_in(th);
  a.cols_in = cols_in;
  a.c0p = c0p;
  a.relu_mid = d->inter_op == DITTO_INTER_RELU;
  a.relu_out = d->relu_out != 0;
  a.out_f32 = d->out_dtype == DITTO_F32;
  a.inv_cg = 1.f / (float)(c0p / 8), a.inv_ng = 1.f / (float)((d->W + 7) / 8);
  a.inv_q = 1.f / (float)Q;
  plan->tiles = true;
  plan->w1p_bytes = ditto::conv_tiles_w1_bytes((int)d->C1, c0p, (int)(d->R1 * d->S1));
  plan->w2p_bytes = ditto::conv_tiles_w2_bytes((int)d->C2, c1p);
  ditto_tile_param& t = plan->tile;
  t.block_threads = 64 * w.wc * w.wp;
  t.block_m = th * (int)Q;
  t.block_l = c1p;
  t.block_n = (int)d->C2;
  t.head_pad = c0p;
  t.lds_bytes = lds_of(th);
  t.grid_x = a.N * a.tiles_h;
  t.grid_y = th;
  t.grid_z = (int)Q;
  t.variant = 3200 + th;  // tiles of whole output rows; rows per workgroup
  return true;
}

// 1x1 -> 3x3 with at most 64 channels on tiles of whole output rows (conv13_tiles.h), where that is the kernel for the shape
// (`forced`: where it can run it at all).  The row pipeline comes before it: ahead on bands of six rows and more with all
// channels filled (32 x 64 x 56 x 56 12.3 us against 14.1; 16 images, bands of four, 8.4 / 9.1).  On shorter bands and fewer
// channels this kernel can be the faster one (32 x 64 x 40 x 40 10.1 / 8.8, 16 channels of 40 x 40 9.4 / 6.9, one image level):
// such calls are left to tuning, which measures both.  It is ahead of the persistent kernel with W2 in LDS on 16-bit outputs (8 x 64 x 112 x 112 20.3 -> 14.8,
// 32 x 64 x 72 x 72 28.4 -> 21.6, 8 x 64 x 30 x 256 26.8 -> 11.8), which keeps the fp32 ones: here they leave in
// pieces of 16 bytes.
bool plan_conv13_tiles(const ditto_conv_chain_desc* d, bool forced, ConvPlan* plan, int cus) {
  if (d->R1 != 1 || d->S1 != 1 || d->pad1 != 0 || d->stride1 != 1 || d->R2 != 3 || d->S2 != 3 || d->pad2 != 1 || d->stride2 != 1 ||
      d->C0 > 64 || d->C1 > 64 || d->C2 > 64 || d->W < 8)
    return false;
  if (!forced && d->out_dtype == DITTO_F32 && d->C0 % 8 == 0 && d->W % 8 == 0) return false;
  // Rows per workgroup, four waves (up to 128 pixels) or eight (256).  A workgroup alone on its compute unit takes a start, a
  // share per halo pixel and one per pixel tile of a wave; a second and third beside it add two thirds of that with four
  // waves, all of it with eight.  Fitted, us beyond the launch: one row of 56 pixels 3.0, of 112 5.7 (eight waves 5.0), two
  // rows of 56 4.2, of 112 6.2 (eight waves).
  int wp = 0, th = 0;
  double best = 0;
  for (int w = 2; w <= 4; w += 2)
    for (int t = 1; t <= d->H && t * d->W <= ditto::conv13_tiles_slots(w); ++t) {
      if (ditto::conv13_tiles_lds_bytes(t, (int)d->W, w) > 160 * 1024) break;
      const long long wgs = d->N * ((d->H + t - 1) / t);
      if (!launchable(wgs, 128 * w)) continue;
      const long long rounds = (wgs + cus - 1) / cus, tiles = (t * d->W + 16 * w - 1) / (16 * w);
      const double halo = (t + 2.0) * d->W;
      const double one = w == 2 ? 1.7 + 0.3 * tiles + 0.0065 * halo : 2.6 + 0.45 * tiles + 0.004 * halo;
      const double cost = one * (1.0 + (w == 2 ? 0.67 : 1.0) * (rounds - 1));
      if (wp == 0 || cost < best) best = cost, wp = w, th = t;
    }
  if (wp == 0) return false;
  ditto::Conv13TilesArgs& a = plan->t13args;
  a.N = (int)d->N; a.C0 = (int)d->C0; a.H = (int)d->H; a.W = (int)d->W; a.C1 = (int)d->C1; a.C2 = (int)d->C2;
  a.TH = th, a.wp = wp;
  a.tiles_h = (int)((d->H + th - 1) / th);
  a.c0p = d->C0 <= 32 ? 32 : 64;
  a.relu_mid = d->inter_op == DITTO_INTER_RELU;
  a.relu_out = d->relu_out != 0;
  a.out_f32 = d->out_dtype == DITTO_F32;
  a.inv_cg = 8.f / (float)a.c0p, a.inv_ng = 1.f / (float)((d->W + 7) / 8), a.inv_w = 1.f / (float)d->W;
  plan->tiles13 = true;
  plan->w1p_bytes = ditto::kC13W1Bytes;
  plan->w2p_bytes = ditto::kC13W2Bytes;
  ditto_tile_param& t = plan->tile;
  t.block_threads = 128 * wp;
  t.block_m = th * (int)d->W;
  t.block_l = 64;
  t.block_n = (int)d->C2;
  t.head_pad = a.c0p;
  t.lds_bytes = ditto::conv13_tiles_lds_bytes(th, (int)d->W, wp);
  t.grid_x = a.N * a.tiles_h;
  t.grid_y = th;
  t.grid_z = (int)d->W;
  t.variant = 3300 + (wp == 4 ? 50 : 0) + th;  // tiles of whole output rows, 1x1 -> 3x3; 50 more with eight waves; rows per workgroup
  return true;
}

// allow_resident = false: the general kernels only (pointers the specialised ones cannot take);
// allow_dw_rows: y takes 16-byte stores
int plan_conv(const ditto_conv_chain_desc* d, ConvPlan* plan, bool need_device = false, int dw_vec_cap = 8,
              bool allow_resident = true, bool allow_dw_rows = true) {
  if (!d) return fail(DITTO_EINVAL, "null descriptor");
  ConvSteer steer;
  int rc = conv_steer(d->tile_variant, &steer);
  if (rc != DITTO_OK) return rc;
  rc = plan_conv_steered(d, steer, plan, need_device, dw_vec_cap, allow_resident, allow_dw_rows);
  if (rc != DITTO_OK) return rc;
  return conv_steer_check(steer, plan->tile.variant);
}

int plan_conv_steered(const ditto_conv_chain_desc* d, const ConvSteer& steer, ConvPlan* plan, bool need_device,
                      int dw_vec_cap, bool allow_resident, bool allow_dw_rows) {
  if (d->abi_version != DITTO_CHAIN_ABI_VERSION)
    return fail(DITTO_EINVAL, "descriptor abi_version %d, library %d", d->abi_version, DITTO_CHAIN_ABI_VERSION);
  if (d->in_dtype != DITTO_F16 && d->in_dtype != DITTO_BF16)
    return fail(DITTO_EUNSUPPORTED, "conv chains are built for fp16 / bf16 (in_dtype %d)", d->in_dtype);
  if (d->acc_dtype != DITTO_F32) return fail(DITTO_EUNSUPPORTED, "conv chains accumulate in fp32");
  if (d->out_dtype != d->in_dtype && d->out_dtype != DITTO_F32)
    return fail(DITTO_EINVAL, "out_dtype must be in_dtype or fp32");
  if (d->inter_op != DITTO_INTER_CAST && d->inter_op != DITTO_INTER_RELU)
    return fail(DITTO_EINVAL, "inter_op %d not valid for a conv chain", d->inter_op);
  if (d->N <= 0 || d->C0 <= 0 || d->H <= 0 || d->W <= 0 || d->C1 <= 0 || d->C2 <= 0 || d->R1 <= 0 ||
      d->S1 <= 0 || d->R2 <= 0 || d->S2 <= 0 || d->stride1 <= 0 || d->stride2 <= 0 || d->pad1 < 0 || d->pad2 < 0)
    return fail(DITTO_EINVAL, "conv extents must be positive and paddings non-negative");
  const bool dw = d->groups1 != 0 && d->groups1 != 1;
  if (dw && d->groups1 != d->C0) return fail(DITTO_EUNSUPPORTED, "groups1 must be 1 (dense) or C0 (depthwise)");
  const bool second_1x1 = d->R2 == 1 && d->S2 == 1 && d->pad2 == 0;
  // A strided 1x1 second convolution keeps every stride2-th pixel of the intermediate image and nothing else: the
  // chain is the same chain with the first convolution strided by stride1 * stride2 (output p of the second reads
  // intermediate p * stride2, i.e. input rows from p * stride1 * stride2 - pad1 on; the number of outputs agrees,
  // floor(floor(x / s1) / s2) = floor(x / (s1 s2))).  Planned and run that way.
  ditto_conv_chain_desc folded;
  if (second_1x1 && d->stride2 > 1) {
    if (d->stride1 * d->stride2 > 0x7fff) return fail(DITTO_EINVAL, "strides too large");
    folded = *d;
    folded.stride1 = d->stride1 * d->stride2;
    folded.stride2 = 1;
    d = &folded;
  }
  if (dw && d->stride2 != 1) return fail(DITTO_EUNSUPPORTED, "depthwise chain: the second convolution must be 1x1");
  if (!dw) {
    if (!second_1x1 && (d->R2 > 3 || d->S2 > 3))
      return fail(DITTO_EUNSUPPORTED, "a second convolution larger than 1x1 takes filters up to 3x3");
    if (!second_1x1 && d->stride2 > 4) return fail(DITTO_EUNSUPPORTED, "second convolution: strides up to 4");
    if (d->C1 % 8) return fail(DITTO_EINVAL, "C1 must be a multiple of 8");
    if (d->C1 > 256) return fail(DITTO_EUNSUPPORTED, "C1=%lld: at most 256 intermediate channels", (long long)d->C1);
  }
  if (d->R1 > 7 || d->S1 > 7) return fail(DITTO_EUNSUPPORTED, "first filter larger than 7x7");
  const long long P = (d->H + 2 * d->pad1 - d->R1) / d->stride1 + 1;
  const long long Q = (d->W + 2 * d->pad1 - d->S1) / d->stride1 + 1;
  if (d->H + 2 * d->pad1 < d->R1 || d->W + 2 * d->pad1 < d->S1 || P <= 0 || Q <= 0)
    return fail(DITTO_EINVAL, "empty convolution output");
  if (d->N * d->C0 * d->H * d->W > 0x7fffffffLL * 4 || d->N * d->C2 * P * Q > 0x7fffffffLL * 4 ||
      d->H > 65535 || d->W > 65535 || d->N > 65535 || d->C0 > 65535 || d->C2 > 65535)
    return fail(DITTO_EINVAL, "tensor too large");
  // (a y that is not 16-byte aligned rules out both kernels that only store 16-byte vectors)
  if (dw) return plan_dw_conv(d, steer, P, Q, plan, need_device, allow_dw_rows, dw_vec_cap, allow_dw_rows);
  memset(plan, 0, sizeof(*plan));
  const int c1t = d->C1 <= 32 ? 1 : d->C1 <= 64 ? 2 : d->C1 <= 128 ? 4 : 8;
  const int pxw = c1t == 8 ? 1 : 2;
  const int slots = 128 * pxw;
  ditto::ConvChainArgs& a = plan->args;
  a.N = (int)d->N; a.C0 = (int)d->C0; a.H = (int)d->H; a.W = (int)d->W;
  a.C1 = (int)d->C1; a.R = (int)d->R1; a.S = (int)d->S1; a.pad = (int)d->pad1; a.stride = (int)d->stride1;
  a.C2 = (int)d->C2; a.P = (int)P; a.Q = (int)Q;
  if (!second_1x1) {
    // The first convolution produces the output tile grown by the second filter's halo (recomputed
    // per workgroup) into at most `slots` pixel slots; the second reads it from LDS.
    const int s2 = (int)d->stride2;
    if (P + 2 * d->pad2 < d->R2 || Q + 2 * d->pad2 < d->S2) return fail(DITTO_EINVAL, "empty convolution output");
    const long long P2 = (P + 2 * d->pad2 - d->R2) / s2 + 1, Q2 = (Q + 2 * d->pad2 - d->S2) / s2 + 1;
    if (P2 <= 0 || Q2 <= 0) return fail(DITTO_EINVAL, "empty convolution output");
    if (d->N * d->C2 * P2 * Q2 > 0x7fffffffLL * 4) return fail(DITTO_EINVAL, "tensor too large");
    a.R2 = (int)d->R2; a.S2 = (int)d->S2; a.pad2 = (int)d->pad2; a.P2 = (int)P2; a.Q2 = (int)Q2;
    a.stride2 = s2;
    // 1x1 -> 3x3 (pad 1) with at most 64 channels everywhere, 16-bit output and image rows of whole 16-byte
    // vectors up to 64 pixels: the row pipeline with the 1x1 convolution in its transposing stage (conv_rows.h)
    if (allow_resident && steer.rows && s2 == 1 && d->R1 == 1 && d->S1 == 1 && d->pad1 == 0 &&
        d->stride1 == 1 && d->R2 == 3 && d->S2 == 3 && d->pad2 == 1 && d->C0 <= ditto::kCvrC && d->C1 <= ditto::kCvrC &&
        d->C2 <= ditto::kCvrC && d->C0 % 8 == 0 && d->W % 8 == 0 && d->W <= 64 && d->out_dtype != DITTO_F32 &&
        d->C0 * d->H * d->W * 2 < 0x7fffffffLL) {
      const int cus = need_device ? device_cus() : 256;
      int band_max = ditto::conv_rows_band_max((int)d->W);
      if (band_max > d->H) band_max = (int)d->H;
      while (band_max >= 1 && ditto::conv_rows_lds_bytes((int)d->W, band_max, true) > 160 * 1024) --band_max;
      if (band_max >= 1) {
        // fewest steps of two rows on the busiest CU (a band costs its steps plus about three of start-up)
        long long best = -1;
        int best_nb = 0;
        const int nb_min = (int)((d->H + band_max - 1) / band_max);
        for (int nb = nb_min; nb <= d->H && nb < nb_min + 64; ++nb) {
          const int band = (int)((d->H + nb - 1) / nb);
          const long long wgs = d->N * ((d->H + band - 1) / band);
          const long long cost = ((wgs + cus - 1) / cus) * ((band + 1) / 2 + 3);
          if (best < 0 || cost <= best) { best = cost; best_nb = nb; }  // ties: the split that fills more CUs
        }
        ditto::ConvRowsArgs& r = plan->cvargs;
        r.N = (int)d->N; r.C0 = (int)d->C0; r.H = (int)d->H; r.W = (int)d->W;
        r.Cm = (int)d->C1; r.C1 = (int)d->C2; r.C2 = (int)d->C2;
        r.band = (int)((d->H + best_nb - 1) / best_nb);
        r.bands = (int)((d->H + r.band - 1) / r.band);
        r.f13 = 1;
        r.relu_pre = d->inter_op == DITTO_INTER_RELU;
        r.relu_mid = d->relu_out != 0;
        r.relu_out = 0;
        plan->rows13 = true;
        plan->c1_tiles = 2;
        plan->px2 = 1;
        plan->w1p_bytes = 0;
        plan->w2p_bytes = ditto::kCvrW1Bytes;
        ditto_tile_param& t = plan->tile;
        t.block_threads = 64 * ditto::kCvrWaves;
        t.block_m = r.band * r.W;
        t.block_l = ditto::kCvrC;
        t.block_n = (int)d->C2;
        t.head_pad = ditto::kCvrC;
        t.lds_bytes = ditto::conv_rows_lds_bytes(r.W, r.band, true);
        t.grid_x = r.N * r.bands;
        t.grid_y = r.band;
        t.grid_z = r.W;
        t.variant = 3800 + r.band;  // row pipeline, 1x1 first; output rows per workgroup
        return DITTO_OK;
      }
    }
    if (allow_resident && steer.tiles13 && plan_conv13_tiles(d, steer.tv / 100 == 33, plan, need_device ? device_cus() : 256))
      return DITTO_OK;
    // 1x1 -> 3x3 (pad 1) with at most 64 channels everywhere and rows that are whole 16-byte vectors: the
    // persistent kernel that keeps W2 in LDS (conv_chain_resident.h), tiles of whole output rows
    if (allow_resident && steer.resident && s2 == 1 && d->R1 == 1 && d->S1 == 1 && d->pad1 == 0 && d->stride1 == 1 && d->R2 == 3 &&
        d->S2 == 3 && d->pad2 == 1 && d->C0 <= ditto::kCrC && d->C1 <= ditto::kCrC && d->C2 <= ditto::kCrC &&
        d->C0 % 8 == 0 && d->W % 8 == 0 && d->W <= 256 &&
        d->C0 * d->H * d->W * 2 < 0x7fffffffLL) {
      int th2 = (int)(256 / d->W);
      if (th2 > d->H) th2 = (int)d->H;
      while (th2 >= 1 && (ditto::conv_resident_lds_bytes(th2, (int)d->W) > 160 * 1024 ||
                          (th2 + 2) * d->W > 64 * ditto::kCrMaxLoads))
        --th2;
      if (th2 >= 1) {
        const int cus = need_device ? device_cus() : 256;
        ditto::ConvResidentArgs& r = plan->rargs;
        r.N = (int)d->N; r.C0 = (int)d->C0; r.H = (int)d->H; r.W = (int)d->W; r.C1 = (int)d->C1; r.C2 = (int)d->C2;
        r.TH2 = th2;
        r.tiles_h = (int)((d->H + th2 - 1) / th2);
        r.ntiles = r.N * r.tiles_h;
        r.relu_mid = d->inter_op == DITTO_INTER_RELU;
        r.relu_out = d->relu_out != 0;
        r.out_f32 = d->out_dtype == DITTO_F32;
        plan->resident = true;
        plan->res_grid = r.ntiles < cus ? r.ntiles : cus;
        plan->px2 = 1;
        plan->w1p_bytes = 0;
        plan->w2p_bytes = ditto::kCrW2Bytes;
        ditto_tile_param& t = plan->tile;
        t.block_threads = 512;
        t.block_m = th2 * (int)d->W;
        t.block_l = ditto::kCrC;
        t.block_n = (int)d->C2;
        t.head_pad = ditto::kCrC;
        t.lds_bytes = ditto::conv_resident_lds_bytes(th2, (int)d->W);
        t.grid_x = plan->res_grid;
        t.grid_y = th2;
        t.grid_z = (int)d->W;
        t.variant = 3600 + th2;  // persistent, W2 resident in LDS; th2 output rows per tile
        return DITTO_OK;
      }
    }
    // an output tile of TH2 x TW2 pixels needs the intermediate pixels (TH2 - 1) s2 + R2 by (TW2 - 1) s2 + S2
    a.TW2 = (int)Q2;
    while (((a.TW2 - 1) * s2 + a.S2) * a.R2 > slots) a.TW2 = (a.TW2 + 1) / 2;
    a.TW = (a.TW2 - 1) * s2 + a.S2;
    a.TH = slots / a.TW;
    if (a.TH > (P2 - 1) * s2 + a.R2) a.TH = (int)(P2 - 1) * s2 + a.R2;
    a.TH2 = (a.TH - a.R2) / s2 + 1;
    a.TH = (a.TH2 - 1) * s2 + a.R2;
    a.rows_in = (a.TH - 1) * a.stride + a.R;
    a.cols_in = (a.TW - 1) * a.stride + a.S;
    const int RS1 = a.R * a.S;
    int lds = ditto::conv_chain_lds_bytes(a.rows_in, a.cols_in, RS1, 32 * c1t, 32);
    a.wide2 = d->out_dtype != DITTO_F32 && Q2 % 8 == 0 && a.TW2 % 8 == 0;
    const int lds2 = ditto::conv_chain2_lds_bytes(slots, 32 * c1t, a.S2, a.wide2 != 0);
    if (lds2 > lds) lds = lds2;
    if (lds > 160 * 1024) return fail(DITTO_EUNSUPPORTED, "conv chain tile does not fit in LDS");
    a.tiles_h = (int)((P2 + a.TH2 - 1) / a.TH2);
    a.tiles_w = (int)((Q2 + a.TW2 - 1) / a.TW2);
    a.relu_mid = d->inter_op == DITTO_INTER_RELU;
    a.relu_out = d->relu_out != 0;
    a.out_f32 = d->out_dtype == DITTO_F32;
    plan->c1_tiles = c1t;
    plan->ch = 32;
    plan->px2 = a.TH2 * a.TW2 <= 128 ? 1 : 2;
    plan->w1p_bytes = ((size_t)ditto::conv_w1_chunk_bytes(RS1, 32 * c1t, 32) * (size_t)((d->C0 + 31) / 32) + 255) / 256 * 256;
    plan->w2p_bytes = (size_t)ditto::conv_w2_chunk_bytes(a.R2 * a.S2) * (size_t)((d->C2 + 63) / 64) * (size_t)c1t;
    ditto_tile_param& t = plan->tile;
    t.block_threads = 256;
    t.block_m = a.TH2 * a.TW2;
    t.block_l = 32 * c1t;
    t.block_n = (int)d->C2;
    t.head_pad = 32;
    t.lds_bytes = lds;
    t.grid_x = a.N * a.tiles_h * a.tiles_w;
    t.grid_y = a.TH2;
    t.grid_z = a.TW2;
    t.variant = 3500 + c1t * 10 + plan->px2;  // second convolution through LDS
    return DITTO_OK;
  }
  // 3x3 (pad 1, stride 1) -> 1x1 with at most 64 input and intermediate and 256 output channels, image rows of
  // whole 16-byte vectors up to 64 pixels, 16-bit output: the row pipeline (conv_rows.h).  Bands of whole
  // output rows, one workgroup each; a band's rows are all in flight at once, which bounds its height.
  if (allow_resident && steer.rows && !steer.persist && d->R1 == 3 && d->S1 == 3 && d->pad1 == 1 &&
      d->stride1 == 1 && d->C0 <= ditto::kCvrC && d->C1 <= ditto::kCvrC && d->C2 <= 256 && d->W % 8 == 0 && d->W <= 64 &&
      d->out_dtype != DITTO_F32 && d->C0 * d->H * d->W * 2 < 0x7fffffffLL && d->C2 * d->H * d->W * 2 < 0x7fffffffLL &&
      // where it pays (measured against the general kernel): the pipeline pads C0 and C1 to 64, and its gain is the
      // output stream under the compute - wide outputs - or, with few images, more workgroups than the general
      // kernel's tiles of 256 pixels (32 x 32 x 56 x 56 -> 32 -> 128: 16.4 against 12.3 us; 64 -> 64 -> 64: a tie;
      // one image 64 -> 64 -> 256: 8.9 against 15.6 us).  Against the kernel on row tiles it is ahead on wide outputs
      // (16 x 64 x 40 x 40 -> 64 -> 256 10.5 / 12.1) and behind on narrow ones (-> 64 -> 64 9.6 / 7.9), which tuning measures.
      (steer.tv / 100 == 37 ||
       ((d->C0 > 32 || d->C1 > 32) &&
      (d->C2 >= 192 || d->N * ((P + (256 / d->W > 0 ? 256 / d->W : 1) - 1) / (256 / d->W > 0 ? 256 / d->W : 1)) <
                           (need_device ? device_cus() : 256))))) {
    const int cus = need_device ? device_cus() : 256;
    int band_max = ditto::conv_rows_band_max((int)d->W);
    if (band_max > d->H) band_max = (int)d->H;
    while (band_max >= 1 && ditto::conv_rows_lds_bytes((int)d->W, band_max) > 160 * 1024) --band_max;
    if (band_max >= 1) {
      // fewest steps of two rows on the busiest CU (a band costs its steps plus about three of start-up)
      long long best = -1;
      int best_nb = 0;
      const int nb_min = (int)((d->H + band_max - 1) / band_max);
      for (int nb = nb_min; nb <= d->H && nb < nb_min + 64; ++nb) {
        const int band = (int)((d->H + nb - 1) / nb);
        const long long wgs = d->N * ((d->H + band - 1) / band);
        const long long cost = ((wgs + cus - 1) / cus) * ((band + 1) / 2 + 3);
        if (best < 0 || cost <= best) { best = cost; best_nb = nb; }  // ties: the split that fills more CUs
      }
      ditto::ConvRowsArgs& r = plan->cvargs;
      r.N = (int)d->N; r.C0 = (int)d->C0; r.H = (int)d->H; r.W = (int)d->W; r.C1 = (int)d->C1; r.C2 = (int)d->C2;
      r.band = (int)((d->H + best_nb - 1) / best_nb);
      r.bands = (int)((d->H + r.band - 1) / r.band);
      r.relu_mid = d->inter_op == DITTO_INTER_RELU;
      r.relu_out = d->relu_out != 0;
      plan->rows31 = true;
      plan->c1_tiles = 2;
      plan->w1p_bytes = ditto::kCvrW1Bytes;
      plan->w2p_bytes = 0;
      ditto_tile_param& t = plan->tile;
      t.block_threads = 64 * ditto::kCvrWaves;
      t.block_m = r.band * r.W;
      t.block_l = ditto::kCvrC;
      t.block_n = (int)d->C2;
      t.head_pad = ditto::kCvrC;
      t.lds_bytes = ditto::conv_rows_lds_bytes(r.W, r.band);
      t.grid_x = r.N * r.bands;
      t.grid_y = r.band;
      t.grid_z = r.W;
      t.variant = 3700 + r.band;  // row pipeline; output rows per workgroup
      return DITTO_OK;
    }
  }
  if (allow_resident && steer.tiles && plan_conv_tiles(d, P, Q, steer.tv / 100 == 32, plan, need_device ? device_cus() : 256))
    return DITTO_OK;
  // The persistent variant (conv_chain_persist.h: W1 resident in LDS, W2 in registers, one workgroup per
  // CU walking over the tiles) is switched off: it waits for its prefetched halo tile with a hand-counted
  // `s_waitcnt vmcnt` over loads the compiler does not track, and it is slower than the kernel below
  // (33.5 against 30.5 us on 32 x 64 x 56 x 56 -> 64 -> 256).  Asking for it is refused, not ignored.
  if (steer.persist)
    return fail(DITTO_EUNSUPPORTED,
                "tile_variant %d: the persistent conv chain kernel is switched off (untracked prefetch loads; "
                "slower than the default kernel)", steer.tv);
  a.TW = (int)(Q < slots ? Q : slots);
  a.TH = slots / a.TW;
  if (a.TH > P) a.TH = (int)P;
  // Shrink the tile until the halo tile and the weight chunk fit in LDS; prefer 32-channel
  // chunks and a footprint that lets two workgroups share a CU (one stages while the other
  // computes), then 32-channel chunks alone, then 16-channel chunks.
  const int RS = a.R * a.S;
  const int th0 = a.TH, tw0 = a.TW;
  int lds = 0, ch = 32;
  for (int attempt = 0;; ++attempt) {
    ch = attempt < 2 ? 32 : 16;
    const int limit = attempt == 0 ? 78 * 1024 : 150 * 1024;
    a.TH = th0;
    a.TW = tw0;
    bool ok = false;
    for (;;) {
      a.rows_in = (a.TH - 1) * a.stride + a.R;
      a.cols_in = (a.TW - 1) * a.stride + a.S;
      lds = ditto::conv_chain_lds_bytes(a.rows_in, a.cols_in, RS, 32 * c1t, ch);
      if (lds <= limit) { ok = true; break; }
      // the first attempt only gives up rows down to half the slots
      if (a.TH > (attempt == 0 ? (th0 + 1) / 2 : 1)) a.TH = a.TH - 1;
      else if (attempt > 0 && a.TW > 16) a.TW = (a.TW + 1) / 2;
      else break;
    }
    if (ok) break;
    if (attempt == 2) return fail(DITTO_EUNSUPPORTED, "conv chain tile does not fit in LDS");
  }
  plan->ch = ch;
  plan->w1p_bytes = (size_t)ditto::conv_w1_chunk_bytes(RS, 32 * c1t, ch) * (size_t)((d->C0 + ch - 1) / ch);
  a.tiles_h = (int)((P + a.TH - 1) / a.TH);
  a.tiles_w = (int)((Q + a.TW - 1) / a.TW);
  a.relu_mid = d->inter_op == DITTO_INTER_RELU;
  a.relu_out = d->relu_out != 0;
  a.out_f32 = d->out_dtype == DITTO_F32;
  plan->c1_tiles = c1t;
  ditto_tile_param& t = plan->tile;
  t.block_threads = 256;
  t.block_m = a.TH * a.TW;   // output pixels per workgroup
  t.block_l = 32 * c1t;      // intermediate channels held in registers
  t.block_n = (int)d->C2;
  t.head_pad = ch;
  t.lds_bytes = lds;
  t.grid_x = a.N * a.tiles_h * a.tiles_w;
  t.grid_y = a.TH;
  t.grid_z = a.TW;
  t.variant = 3000 + c1t * 10 + pxw + (ch == 16 ? 100 : 0);
  return DITTO_OK;
}

// The kernels that run several chains of one shape in one launch: those of 16 to 64 rows per workgroup or short tiles.  (They
// find a row's first unmasked key wherever it lies, so a chain loses nothing by running with others.)
bool plan_takes_sets(const BmmPlan& plan) { return plan.split_rt > 0 || plan.rows_nw > 0 || plan.qt == 4 || plan.qt == 5; }

// The launch of n chains of one descriptor together, if there is one.
struct SetsPlan {
  ditto_bmm_chain_desc desc;
  BmmPlan plan;
};
bool plan_sets(const ditto_bmm_chain_desc* d, int n, SetsPlan* out) {
  BmmPlan alone;
  if (d->batch <= 0 || d->batch > 0x7fffffff / (2 * ditto::kMaxSets) || plan_bmm(d, &alone, true, false) != DITTO_OK) return false;
  ditto_bmm_chain_desc& all = out->desc;
  all = *d;
  all.batch = d->batch * n;
  if (d->batch_inner == 0 || d->batch_inner == d->batch) {
    all.batch_inner = d->batch;
    all.a_batch_stride_outer = all.b_batch_stride_outer = all.c_batch_stride_outer = all.f_batch_stride_outer = 0;
  }
  if (plan_bmm(&all, &out->plan, true, false) != DITTO_OK) return false;
  // A chain that the rules of plan_bmm have split its keys by itself does so with others too, 16 | 32 rows a workgroup: every part of
  // the keys has its own reference, whose probability is exact, and the kernels with one a row are 0.5 - 12 % further from 64 bits
  // (12 x [8 heads, 172 rows of 64] fp16 2.5e-4 against 2.8e-4).  That costs time, up to 3.5 times theirs (12 x [8 heads, 256 rows of
  // 64] 11.7 us against 6.6, 12 x [16 heads, 197 rows of 80] 33 / 10.6; a launch each 48 and 61), and saves some where they take no
  // sets (12 x [2 heads, 1024 rows of 128] 34 against 51).  Where few_rows_variant has a chain split its keys, the stack stays on the
  // kernels with one reference a row, which were the chain's own before: as exact as then, and 7 - 10 % (fp16 results) to 25 %
  // (fp32 ones) further from 64 bits than the chain by itself now.
  if (alone.split_rt > 0 && out->plan.split_rt == 0) {
    all.tile_variant = alone.tile.variant / 10 * 10 + (d->M <= 16 ? 1 : 2);
    if (plan_bmm(&all, &out->plan, true, false) != DITTO_OK) return false;
  }
  if (!plan_takes_sets(out->plan)) return false;
  // (the plan of the 64-row kernel does not ask: one chain that a launch does not hold has nowhere to go, several have)
  if (!launchable((long long)out->plan.nb * all.batch, out->plan.tile.block_threads)) return false;
  out->plan.split_ct = 0;  // (the key-splitting kernel for several chains has workgroups of all columns only)
  return true;
}

// Calls launch(first chain, plan, where the chains lie) for every launch that `count` chains go out in, until one returns an
// error; the plan is null for a chain by itself.
template <typename Launch>
int for_sets_launches(const ditto_bmm_chain_desc* d, int count, const void* const* a, const void* const* b, const void* const* c,
                      void* const* f, Launch&& launch) {
  const long long elem = 2, out_elem = d->out_dtype == DITTO_F32 ? 4 : 2;
  unsigned refused = 0;  // bit n: no kernel takes n of the chains together
  int alone = 0;         // chains from `at` on that are known to go out by themselves
  for (int at = 0; at < count;) {
    // the chains from `at` on that may share a launch: 16-bit ones whose A, B and C lie equally far from the first one's
    int n = 1;
    ditto::BmmSets sets = {};
    if (alone == 0 && (d->in_dtype == DITTO_F16 || d->in_dtype == DITTO_BF16) && d->inter_op == DITTO_INTER_SOFTMAX &&
        d->b_layout == DITTO_B_LK) {
      auto apart = [](const void* to, const void* from) {
        return (long long)(reinterpret_cast<intptr_t>(to) - reinterpret_cast<intptr_t>(from));
      };
      for (; at + n < count && n < ditto::kMaxSets; ++n) {
        const long long in = apart(a[at + n], a[at]);
        if (!a[at + n] || !b[at + n] || !c[at + n] || !f[at + n] || !aligned(f[at + n], 16) || in % 16 != 0 ||
            apart(b[at + n], b[at]) != in || apart(c[at + n], c[at]) != in)
          break;
        sets.in[n] = in / elem, sets.out[n] = apart(f[at + n], f[at]) / out_elem;
      }
    }
    // as many of them as a kernel takes, by halves: all together may be so large that one is chosen which takes no sets
    SetsPlan together;
    int take = n;
    while (take > 1 && ((refused >> take & 1) != 0 || !plan_sets(d, take, &together))) refused |= 1u << take, take = (take + 1) / 2;
    if (take == 1 && n > 1) alone = n;
    sets.count = take, sets.entries = (int)d->batch;
    const int rc = launch(at, take > 1 ? &together : nullptr, sets);
    if (rc != DITTO_OK) return rc;
    at += take;
    if (alone > 0) --alone;
  }
  return DITTO_OK;
}

// The launch of a planned fp16 / bf16 chain; `sets`: where the tensors of the chains it is one of lie, or null.
int launch_fp_chain(const ditto_bmm_chain_desc* d, const BmmPlan& plan, const void* a, const void* b, const void* c, void* f,
                    const ditto::BmmSets* sets, hipStream_t st) {
  ditto::BmmChainArgs args;
  args.a = a;
  args.b = b;
  args.c = c;
  args.f = f;
  args.a_bs = d->a_batch_stride;
  args.b_bs = d->b_batch_stride;
  args.c_bs = d->c_batch_stride;
  args.f_bs = d->f_batch_stride;
  {
    const bool two = d->batch_inner > 0 && d->batch_inner != d->batch;
    args.batch_inner = two ? (int)d->batch_inner : (int)d->batch;
    args.a_bs2 = two ? d->a_batch_stride_outer : 0;
    args.b_bs2 = two ? d->b_batch_stride_outer : 0;
    args.c_bs2 = two ? d->c_batch_stride_outer : 0;
    args.f_bs2 = two ? d->f_batch_stride_outer : 0;
  }
  args.a_rs = (int)d->a_row_stride;
  args.b_rs = (int)d->b_row_stride;
  args.c_rs = (int)d->c_row_stride;
  args.f_rs = (int)d->f_row_stride;
  args.M = (int)d->M;
  args.N = (int)d->N;
  args.K = (int)d->K;
  args.L = (int)d->L;
  args.batch = (int)d->batch;
  args.mblocks = plan.nb;
  args.mblocks3 = plan.nb3;
  args.scale_log2 = d->softmax_scale * 1.4426950408889634f;
  args.relu = d->inter_op == DITTO_INTER_RELU;
  args.relu_out = d->relu_out;
  args.out_f32 = d->out_dtype == DITTO_F32;
  const bool kl = d->b_layout == DITTO_B_KL;
  const bool sm = d->inter_op == DITTO_INTER_SOFTMAX;
  hipError_t e;
  if (sets) {
    const ditto::BmmSetsKernel k = plan.split_rt > 0 ? ditto::BmmSetsKernel::split
                                   : plan.rows_nw > 0 ? ditto::BmmSetsKernel::rows
                                                      : ditto::BmmSetsKernel::rows64;
    const int dt = plan.split_rt > 0 ? plan.split_dt : plan.rows_dt;
    const int q = plan.split_rt > 0 ? plan.split_rt : plan.rows_nw > 0 ? plan.rows_nw : plan.qt;
    const ditto::BmmSetsArgs all{args, *sets};
    e = d->in_dtype == DITTO_F16 ? ditto::launch_sets_f16(k, dt, q, all, st) : ditto::launch_sets_bf16(k, dt, q, all, st);
  } else if (plan.split_ct > 0)
    e = d->in_dtype == DITTO_F16 ? ditto::launch_split_cols_f16(plan.split_dt, plan.split_ct, sm, kl, args, st)
                                 : ditto::launch_split_cols_bf16(plan.split_dt, plan.split_ct, sm, kl, args, st);
  else if (plan.split_rt > 0)
    e = d->in_dtype == DITTO_F16 ? ditto::launch_split_f16(plan.split_dt, plan.split_rt, sm, kl, args, st)
                                 : ditto::launch_split_bf16(plan.split_dt, plan.split_rt, sm, kl, args, st);
  else if (plan.rows_nw > 0)
    e = d->in_dtype == DITTO_F16 ? ditto::launch_rows_f16(plan.rows_dt, plan.rows_nw, sm, kl, args, st)
                                 : ditto::launch_rows_bf16(plan.rows_dt, plan.rows_nw, sm, kl, args, st);
  else if (d->in_dtype == DITTO_F16)
    e = sm ? ditto::launch_f16_softmax(plan.d_pad, plan.qt, kl, args, st)
           : ditto::launch_f16_cast(plan.d_pad, plan.qt, kl, args, st);
  else
    e = sm ? ditto::launch_bf16_softmax(plan.d_pad, plan.qt, kl, args, st)
           : ditto::launch_bf16_cast(plan.d_pad, plan.qt, kl, args, st);
  if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
  return DITTO_OK;
}

}  // namespace

extern "C" {

int ditto_chain_abi_version(void) { return DITTO_CHAIN_ABI_VERSION; }

const char* ditto_last_error(void) { return g_err; }

int ditto_bmm_chain_select_tile(const ditto_bmm_chain_desc* desc, ditto_tile_param* out) {
  BmmPlan plan;
  int rc = plan_bmm(desc, &plan, true);  // the current device's compute-unit count (256 where there is none)
  if (rc != DITTO_OK) return rc;
  if (!out) return fail(DITTO_EINVAL, "null output");
  *out = plan.tile;
  return DITTO_OK;
}

size_t ditto_bmm_chain_workspace_bytes(const ditto_bmm_chain_desc* desc) {
  (void)desc;
  return 0;
}

int ditto_bmm_chain_run(const ditto_bmm_chain_desc* d, const void* a, const void* b, const void* c,
                        const void* aux, void* f, void* workspace, size_t workspace_bytes,
                        void* stream) {
  (void)workspace;
  (void)workspace_bytes;
  (void)aux;
  BmmPlan plan;
  int rc = plan_bmm(d, &plan, true);
  if (rc != DITTO_OK) return rc;
  if (!a || !b || !c || !f) return fail(DITTO_EINVAL, "null data pointer");
  if (!aligned(a, 16) || !aligned(b, 16) || !aligned(c, 16) || !aligned(f, 16))
    return fail(DITTO_EINVAL, "data pointers must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);

  if (plan.family == 0) return launch_fp_chain(d, plan, a, b, c, f, nullptr, st);
  if (plan.family == 1) {
    ditto::F32ChainArgs args;
    args.a = a;
    args.b = b;
    args.c = c;
    args.f = f;
    args.f64 = d->in_dtype == DITTO_F64;
    args.a_bs = d->a_batch_stride;
    args.b_bs = d->b_batch_stride;
    args.c_bs = d->c_batch_stride;
    args.f_bs = d->f_batch_stride;
    args.a_rs = (int)d->a_row_stride;
    args.b_rs = (int)d->b_row_stride;
    args.c_rs = (int)d->c_row_stride;
    args.f_rs = (int)d->f_row_stride;
    args.M = (int)d->M;
    args.N = (int)d->N;
    args.K = (int)d->K;
    args.L = (int)d->L;
    args.batch = (int)d->batch;
    args.mblocks = (int)((d->M + plan.tile.block_m - 1) / plan.tile.block_m);
    args.row_tiles = plan.qt;
    args.width = plan.f32_width;
    args.col_blocks = plan.f32_cols;
    args.b_lk = d->b_layout == DITTO_B_LK;
    args.relu = d->inter_op == DITTO_INTER_RELU;
    args.relu_out = d->relu_out;
    args.softmax = d->inter_op == DITTO_INTER_SOFTMAX;
    args.softmax_scale = d->softmax_scale;
    hipError_t e = ditto::launch_gemm_chain_f32(args, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.family == 2) {
    if (aux && !aligned(aux, 4)) return fail(DITTO_EINVAL, "aux (scale vector) must be 4-byte aligned");
    ditto::I8ChainArgs args;
    args.a = static_cast<const int8_t*>(a);
    args.b = static_cast<const int8_t*>(b);
    args.d = static_cast<const int8_t*>(c);
    args.scale = static_cast<const float*>(aux);
    args.scale_uniform = d->requant_scale;
    args.wrap = d->inter_op != DITTO_INTER_REQUANT;
    args.relu = d->inter_op == DITTO_INTER_RELU;
    args.out_i8 = d->out_dtype == DITTO_I8;
    args.e = static_cast<int32_t*>(f);
    args.a_bs = d->a_batch_stride;
    args.b_bs = d->b_batch_stride;
    args.d_bs = d->c_batch_stride;
    args.e_bs = d->f_batch_stride;
    args.a_rs = (int)d->a_row_stride;
    args.b_rs = (int)d->b_row_stride;
    args.d_rs = (int)d->c_row_stride;
    args.e_rs = (int)d->f_row_stride;
    args.M = (int)d->M;
    args.N = (int)d->N;
    args.K = (int)d->K;
    args.L = (int)d->L;
    args.batch = (int)d->batch;
    args.mblocks = (int)((d->M + plan.tile.block_m - 1) / plan.tile.block_m);
    args.Lp = plan.tile.block_l;
    args.slices = plan.slices;
    args.slice_blocks = plan.slice_blocks;
    hipError_t e = plan.units_rt > 0 ? ditto::launch_gemm_chain_i8_units(args, plan.units_rt, st)
                                     : ditto::launch_gemm_chain_i8(args, plan.d_pad, plan.qt, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  return fail(DITTO_EUNSUPPORTED, "no kernel family %d", plan.family);
}

int ditto_bmm_chain_run_sets(const ditto_bmm_chain_desc* d, int count, const void* const* a, const void* const* b,
                             const void* const* c, void* const* f, void* stream) {
  if (!d || count < 0 || (count > 0 && (!a || !b || !c || !f))) return fail(DITTO_EINVAL, "null argument or negative count");
  return for_sets_launches(d, count, a, b, c, f, [&](int at, const SetsPlan* together, const ditto::BmmSets& sets) {
    if (!together) return ditto_bmm_chain_run(d, a[at], b[at], c[at], nullptr, f[at], nullptr, 0, stream);
    if (!a[at] || !b[at] || !c[at] || !f[at]) return fail(DITTO_EINVAL, "null data pointer");
    if (!aligned(a[at], 16) || !aligned(b[at], 16) || !aligned(c[at], 16) || !aligned(f[at], 16))
      return fail(DITTO_EINVAL, "data pointers must be 16-byte aligned");
    return launch_fp_chain(&together->desc, together->plan, a[at], b[at], c[at], f[at], &sets, reinterpret_cast<hipStream_t>(stream));
  });
}

int ditto_bmm_chain_sets_launches(const ditto_bmm_chain_desc* d, int count, const void* const* a, const void* const* b,
                                  const void* const* c, void* const* f) {
  if (!d || count < 0 || (count > 0 && (!a || !b || !c || !f))) return fail(DITTO_EINVAL, "null argument or negative count");
  int launches = 0;
  for_sets_launches(d, count, a, b, c, f, [&](int, const SetsPlan*, const ditto::BmmSets&) { return ++launches, (int)DITTO_OK; });
  return launches;
}

int ditto_conv_chain_select_tile(const ditto_conv_chain_desc* desc, ditto_tile_param* out) {
  ConvPlan plan;
  int rc = plan_conv(desc, &plan, true);  // the current device's compute-unit count (256 where there is none)
  if (rc != DITTO_OK) return rc;
  if (!out) return fail(DITTO_EINVAL, "null output");
  *out = plan.tile;
  return DITTO_OK;
}

size_t ditto_conv_chain_workspace_bytes(const ditto_conv_chain_desc* desc) {
  ConvPlan plan;
  if (plan_conv(desc, &plan, true) != DITTO_OK) return 0;
  size_t need = plan.w1p_bytes + plan.w2p_bytes;
  if (plan.resident || plan.rows31 || plan.rows13 || plan.tiles || plan.tiles13) {
    // a call with pointers these kernels cannot take falls back to the general one (tile_variant 0 only): the
    // larger of the two figures, whatever the device's compute-unit count makes of the choice
    ConvPlan general;
    if (desc->tile_variant == 0 && plan_conv(desc, &general, true, 8, false) == DITTO_OK &&
        general.w1p_bytes + general.w2p_bytes > need)
      need = general.w1p_bytes + general.w2p_bytes;
  }
  return need;
}

}  // extern "C"

namespace {
// what a conv chain call does: repack the weights into the workspace, run the fused kernel, or both
enum ConvPhase { kConvPrepare = 1, kConvCompute = 2, kConvBoth = 3 };

// The row pipeline of either element type; few rows of 56 or 64 pixels have kernels of their own (see conv_rows_wide).
hipError_t launch_conv_rows(const ditto::ConvRowsArgs& r, bool f16, hipStream_t st) {
  if (!r.f13 && ditto::conv_rows_wide(r)) return f16 ? ditto::launch_conv_rows_few_f16(r, st) : ditto::launch_conv_rows_few_bf16(r, st);
  return f16 ? ditto::launch_conv_rows_f16(r, st) : ditto::launch_conv_rows_bf16(r, st);
}

int conv_chain_call(int phase, const ditto_conv_chain_desc* d, const void* x, const void* w1, const void* w2,
                    void* y, void* workspace, size_t workspace_bytes, void* stream) {
  ConvPlan plan;
  // (depthwise chains: 16-byte halo vectors only for a 16-byte aligned x; the tile query assumes one)
  // (the row-streaming depthwise kernel moves 16-byte vectors of x and y)
  int rc = plan_conv(d, &plan, true, x && aligned(x, 16) ? 8 : 4, true, !y || aligned(y, 16));
  if (rc != DITTO_OK) return rc;
  if (((phase & kConvCompute) && (!x || !y)) || !w1 || !w2) return fail(DITTO_EINVAL, "null data pointer");
  if (plan.resident) {
    // 16-byte direct loads of X and W1 fragments, stores of 4 pixels
    const bool ok = aligned(w1, 16) && (!(phase & kConvCompute) || (aligned(x, 16) && aligned(y, 16)));
    if (!ok && phase == kConvBoth) {
      rc = plan_conv(d, &plan, true, 4, false);  // the general kernel takes any element-aligned pointer
      if (rc != DITTO_OK) return rc;
    } else if (!ok) {
      return fail(DITTO_EINVAL, "misaligned data pointer: this shape runs with x, w1 and y 16-byte aligned "
                                "(its prepared weights are in the resident kernel's layout)");
    }
  }
  if (plan.rows13) {
    // 16-byte direct loads of X, W1 fragments and output stores; W2 as MFMA fragments in the workspace
    const bool ok = aligned(w1, 16) && workspace && workspace_bytes >= plan.w2p_bytes && aligned(workspace, 16) &&
                    (!(phase & kConvCompute) || (aligned(x, 16) && aligned(y, 16)));
    if (!ok && phase == kConvBoth) {
      rc = plan_conv(d, &plan, true, 4, false);  // the general kernel: any element-aligned pointer, workspace optional
      if (rc != DITTO_OK) return rc;
    } else if (!ok) {
      if (!workspace || workspace_bytes < plan.w2p_bytes)
        return fail(DITTO_EWORKSPACE, "prepared weights live in the workspace: need %zu bytes", plan.w2p_bytes);
      return fail(DITTO_EINVAL, "misaligned data pointer: this shape runs with x, w1, y and the workspace 16-byte "
                                "aligned (its prepared weights are in the row pipeline's layout)");
    }
  }
  if (plan.rows13) {
    ditto::ConvRowsArgs r = plan.cvargs;
    r.x = x;
    r.w1x = w1;
    r.w1f = workspace;
    r.w2 = nullptr;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = d->in_dtype == DITTO_F16;
    hipError_t e = hipSuccess;
    if (phase & kConvPrepare)  // W2 [C2][C1][3][3] into fragments
      e = f16 ? ditto::pack_conv_w2_resident_f16(w2, workspace, r.Cm, r.C2, st)
              : ditto::pack_conv_w2_resident_bf16(w2, workspace, r.Cm, r.C2, st);
    if (e == hipSuccess && (phase & kConvCompute)) e = launch_conv_rows(r, f16, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.rows31) {
    // 16-byte direct loads of X, W2 fragments and output stores; W1 as MFMA fragments in the workspace
    const bool ok = aligned(w2, 16) && workspace && workspace_bytes >= plan.w1p_bytes && aligned(workspace, 16) &&
                    (!(phase & kConvCompute) || (aligned(x, 16) && aligned(y, 16)));
    if (!ok && phase == kConvBoth) {
      rc = plan_conv(d, &plan, true, 4, false);  // the general kernel: any element-aligned pointer, workspace optional
      if (rc != DITTO_OK) return rc;
    } else if (!ok) {
      if (!workspace || workspace_bytes < plan.w1p_bytes)
        return fail(DITTO_EWORKSPACE, "prepared weights live in the workspace: need %zu bytes", plan.w1p_bytes);
      return fail(DITTO_EINVAL, "misaligned data pointer: this shape runs with x, w2, y and the workspace 16-byte "
                                "aligned (its prepared weights are in the row pipeline's layout)");
    }
  }
  if (plan.rows31) {
    ditto::ConvRowsArgs r = plan.cvargs;
    r.x = x;
    r.w1f = workspace;
    r.w2 = w2;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = d->in_dtype == DITTO_F16;
    hipError_t e = hipSuccess;
    if (phase & kConvPrepare)  // W1 [C1][C0][3][3] into fragments: the same layout as the resident kernel's W2
      e = f16 ? ditto::pack_conv_w2_resident_f16(w1, workspace, r.C0, r.C1, st)
              : ditto::pack_conv_w2_resident_bf16(w1, workspace, r.C0, r.C1, st);
    if (e == hipSuccess && (phase & kConvCompute)) e = launch_conv_rows(r, f16, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.tiles || plan.tiles13) {
    // both weights as MFMA fragments in the workspace; x and y at any element
    const size_t need = plan.w1p_bytes + plan.w2p_bytes;
    const bool ok = workspace && workspace_bytes >= need && aligned(workspace, 16);
    if (!ok && phase == kConvBoth && d->tile_variant == 0) {
      rc = plan_conv(d, &plan, true, 4, false);  // the general kernel: workspace optional
      if (rc != DITTO_OK) return rc;
    } else if (!workspace || workspace_bytes < need) {
      return fail(DITTO_EWORKSPACE, "prepared weights live in the workspace: need %zu bytes", need);
    } else if (!ok) {
      return fail(DITTO_EINVAL, "workspace must be 16-byte aligned");
    }
  }
  if (plan.tiles) {
    ditto::ConvTilesArgs r = plan.targs;
    if (!aligned(x, 2) || !aligned(y, r.out_f32 ? 4 : 2) || !aligned(w1, 2) || !aligned(w2, 2))
      return fail(DITTO_EINVAL, "misaligned data pointer");
    r.x = x;
    r.w1f = workspace;
    r.w2f = static_cast<char*>(workspace) + plan.w1p_bytes;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = d->in_dtype == DITTO_F16;
    hipError_t e = hipSuccess;
    if (phase & kConvPrepare)
      e = f16 ? ditto::pack_conv_tiles_f16(r, w1, w2, const_cast<void*>(r.w1f), const_cast<void*>(r.w2f), st)
              : ditto::pack_conv_tiles_bf16(r, w1, w2, const_cast<void*>(r.w1f), const_cast<void*>(r.w2f), st);
    if (e == hipSuccess && (phase & kConvCompute))
      e = f16 ? ditto::launch_conv_tiles_f16(r, st) : ditto::launch_conv_tiles_bf16(r, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.tiles13) {
    ditto::Conv13TilesArgs r = plan.t13args;
    if (!aligned(x, 2) || !aligned(y, r.out_f32 ? 4 : 2) || !aligned(w1, 2) || !aligned(w2, 2)) return fail(DITTO_EINVAL, "misaligned data pointer");
    r.x = x;
    r.w1f = workspace;
    r.w2f = static_cast<char*>(workspace) + plan.w1p_bytes;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = d->in_dtype == DITTO_F16;
    hipError_t e = hipSuccess;
    if (phase & kConvPrepare)
      e = f16 ? ditto::pack_conv13_tiles_f16(r, w1, w2, const_cast<void*>(r.w1f), const_cast<void*>(r.w2f), st)
              : ditto::pack_conv13_tiles_bf16(r, w1, w2, const_cast<void*>(r.w1f), const_cast<void*>(r.w2f), st);
    if (e == hipSuccess && (phase & kConvCompute))
      e = f16 ? ditto::launch_conv13_tiles_f16(r, st) : ditto::launch_conv13_tiles_bf16(r, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.resident) {
    if (!workspace) return fail(DITTO_EWORKSPACE, "this conv chain needs the workspace (%zu bytes)", plan.w2p_bytes);
    if (workspace_bytes < plan.w2p_bytes)
      return fail(DITTO_EWORKSPACE, "workspace of %zu bytes, need %zu", workspace_bytes, plan.w2p_bytes);
    if (!aligned(workspace, 16)) return fail(DITTO_EINVAL, "workspace must be 16-byte aligned");
    ditto::ConvResidentArgs r = plan.rargs;
    r.x = x;
    r.w1 = w1;
    r.w2f = workspace;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = d->in_dtype == DITTO_F16;
    hipError_t e = hipSuccess;
    if (phase & kConvPrepare)
      e = f16 ? ditto::pack_conv_w2_resident_f16(w2, workspace, r.C1, r.C2, st)
              : ditto::pack_conv_w2_resident_bf16(w2, workspace, r.C1, r.C2, st);
    if (e == hipSuccess && (phase & kConvCompute))
      e = f16 ? ditto::launch_conv_resident_f16(r, plan.res_grid, st) : ditto::launch_conv_resident_bf16(r, plan.res_grid, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (plan.dw && plan.dw_mode == 6) {  // x, weights and y at any element
    if (!(phase & kConvCompute)) return DITTO_OK;
    ditto::DwTilesArgs r = plan.dwtargs;
    if (!aligned(x, 2) || !aligned(w1, 2) || !aligned(w2, 2) || !aligned(y, r.out_f32 ? 4 : 2))
      return fail(DITTO_EINVAL, "misaligned data pointer");
    r.x = x;
    r.w1 = w1;
    r.w2 = w2;
    r.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int mult = (int)(d->C1 / d->C0);
    hipError_t e = d->in_dtype == DITTO_F16 ? ditto::launch_dw_tiles_f16(mult, r, st) : ditto::launch_dw_tiles_bf16(mult, r, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  if (!aligned(x, 2) || !aligned(w1, 2) || !aligned(w2, 8) || !aligned(y, 4))
    return fail(DITTO_EINVAL, "misaligned data pointer");
  if (phase != kConvBoth && !plan.dw && !workspace)
    return fail(DITTO_EWORKSPACE, "prepared weights live in the workspace: none given");
  if (plan.dw) {
    if (!(phase & kConvCompute)) return DITTO_OK;  // nothing to prepare: the kernel stages the filters itself
    if (plan.dw_mode == 4) {
      ditto::DwRowsArgs r = plan.rowargs;
      r.x = x;
      r.w1 = w1;
      r.w2 = w2;
      r.y = y;
      hipStream_t st = reinterpret_cast<hipStream_t>(stream);
      hipError_t e = d->in_dtype == DITTO_F16 ? ditto::launch_dw_rows_f16(r, st) : ditto::launch_dw_rows_bf16(r, st);
      if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
      return DITTO_OK;
    }
    if (plan.dw_mode == 5) {
      ditto::Dw16RowsArgs r = plan.row16args;
      r.x = x;
      r.w1 = w1;
      r.w2 = w2;
      r.y = y;
      hipStream_t st = reinterpret_cast<hipStream_t>(stream);
      hipError_t e = d->in_dtype == DITTO_F16 ? ditto::launch_dw16_rows_f16(r, st) : ditto::launch_dw16_rows_bf16(r, st);
      if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
      return DITTO_OK;
    }
    if (!aligned(w2, 16)) return fail(DITTO_EINVAL, "misaligned data pointer");
    ditto::DwConvArgs a = plan.dwargs;
    // less aligned pointers: narrower halo loads (the LDS layout stays valid) while the chunk still
    // fits the registers that keep it in flight; plain 2-byte output stores
    while (a.vec > 1 && !aligned(x, 2 * (size_t)a.vec)) a.vec >>= 1;
    if (plan.dw_mode >= 2) {
      const int nvr = a.cols_al / a.vec;
      const int cphases = (256 * ditto::dw_mfma_groups(plan.c2_tiles) / nvr) / a.rows_in;
      if (cphases < 1 || (a.chx + cphases - 1) / cphases > (a.vec == 8 ? ditto::kDwXpf / 2 : ditto::kDwXpf))
        return fail(DITTO_EINVAL, "misaligned data pointer: x must be aligned to %d bytes for this shape",
                    2 * plan.dwargs.vec);
      if (!aligned(w1, 16)) return fail(DITTO_EINVAL, "misaligned data pointer");
    }
    if (a.wide && !aligned(y, 16)) {
      if (plan.dw_mode == 3) return fail(DITTO_EINVAL, "misaligned data pointer: y must be 16-byte aligned for this shape");
      a.wide = 0;
    }
    a.x = x;
    a.w1 = w1;
    a.w2 = w2;
    a.y = y;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipError_t e = d->in_dtype == DITTO_F16 ? ditto::launch_dw_conv_f16(plan.c2_tiles, plan.dw_mode, a, st)
                                            : ditto::launch_dw_conv_bf16(plan.c2_tiles, plan.dw_mode, a, st);
    if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
    return DITTO_OK;
  }
  const size_t need = plan.w1p_bytes + plan.w2p_bytes;
  if (plan.w1p_bytes >= (1ull << 31) || plan.w2p_bytes >= (1ull << 31))  // the repack kernels index with 32 bits
    return fail(DITTO_EUNSUPPORTED, "conv chain weights too large to repack");
  if (plan.px2 > 0 && !workspace)
    return fail(DITTO_EWORKSPACE, "a second convolution larger than 1x1 needs the workspace (%zu bytes)", need);
  if (workspace && workspace_bytes < need)
    return fail(DITTO_EWORKSPACE, "workspace of %zu bytes, need %zu", workspace_bytes, need);
  if (workspace && !aligned(workspace, 16)) return fail(DITTO_EINVAL, "workspace must be 16-byte aligned");
  ditto::ConvChainArgs a = plan.args;
  a.x = x;
  a.w1 = w1;
  a.w2 = w2;
  a.w1p = workspace;
  a.y = y;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool f16 = d->in_dtype == DITTO_F16;
  hipError_t e = hipSuccess;
  const bool prepare = (phase & kConvPrepare) != 0, compute = (phase & kConvCompute) != 0;
  if (workspace && plan.px2 == 0 && prepare)  // W1 into the chunked layout the chain kernel copies straight into LDS
    e = f16 ? ditto::pack_conv_w1_f16(plan.c1_tiles, plan.ch, a, workspace, st)
            : ditto::pack_conv_w1_bf16(plan.c1_tiles, plan.ch, a, workspace, st);
  if (plan.px2 > 0) {
    void* w2p = static_cast<char*>(workspace) + plan.w1p_bytes;
    a.w2p = w2p;
    if (a.wide2 && !aligned(y, 16)) a.wide2 = 0;  // plain 2-byte stores (the LDS size follows the flag)
    // both weight tensors into their chunked layouts, one launch
    if (prepare)
      e = f16 ? ditto::pack_conv_w2_f16(plan.c1_tiles, a, workspace, w2p, st)
              : ditto::pack_conv_w2_bf16(plan.c1_tiles, a, workspace, w2p, st);
    if (e == hipSuccess && compute)
      e = f16 ? ditto::launch_conv2_f16(plan.c1_tiles, plan.px2, a, st) : ditto::launch_conv2_bf16(plan.c1_tiles, plan.px2, a, st);
  } else if (e == hipSuccess && compute) {
    e = f16 ? ditto::launch_conv_f16(plan.c1_tiles, plan.ch, a, st) : ditto::launch_conv_bf16(plan.c1_tiles, plan.ch, a, st);
  }
  if (e != hipSuccess) return fail(DITTO_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
  return DITTO_OK;
}

}  // namespace

extern "C" {

int ditto_conv_chain_run(const ditto_conv_chain_desc* d, const void* x, const void* w1, const void* w2,
                         void* y, void* workspace, size_t workspace_bytes, void* stream) {
  return conv_chain_call(kConvBoth, d, x, w1, w2, y, workspace, workspace_bytes, stream);
}

int ditto_conv_chain_prepare(const ditto_conv_chain_desc* d, const void* w1, const void* w2, void* workspace,
                             size_t workspace_bytes, void* stream) {
  return conv_chain_call(kConvPrepare, d, nullptr, w1, w2, nullptr, workspace, workspace_bytes, stream);
}

int ditto_conv_chain_run_prepared(const ditto_conv_chain_desc* d, const void* x, const void* w1, const void* w2,
                                  void* y, void* workspace, size_t workspace_bytes, void* stream) {
  return conv_chain_call(kConvCompute, d, x, w1, w2, y, workspace, workspace_bytes, stream);
}

}  // extern "C"

// ---- the entry point that allocates nothing -------------------------------------------------
// Its workspace (the repacked weights of a conv chain) is a file-scope device array instead of
// caller memory.  Every device the library runs on holds its own copy of the array at its own
// address until the process ends; host code reaches it only through the address taken with
// hipGetSymbolAddress on that device (the array's name is a host-side stand-in, not a device
// address).
static __device__ __align__(256) unsigned char scratch[DITTO_STATIC_WORKSPACE_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];  // per device, filled at the first call on that device

// Device address of `scratch` on the current device.
int static_workspace(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(DITTO_EHIP, "hipGetDevice failed: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(DITTO_EUNSUPPORTED, "device ordinal %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(DITTO_EHIP, "hipGetSymbolAddress(static workspace) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return DITTO_OK;
}
}  // namespace

extern "C" int ditto_conv_chain_run_static(const ditto_conv_chain_desc* d, const void* x, const void* w1,
                                           const void* w2, void* y, void* stream) {
  ConvPlan plan;
  int rc = plan_conv(d, &plan, true);
  if (rc != DITTO_OK) return rc;
  size_t need = plan.w1p_bytes + plan.w2p_bytes;
  if (need > (size_t)DITTO_STATIC_WORKSPACE_BYTES && (plan.tiles || plan.tiles13) && d->tile_variant == 0) {
    // the kernels on row tiles repack both weights, the general one (which the call then runs) W1 alone
    rc = plan_conv(d, &plan, true, 4, false);
    if (rc != DITTO_OK) return rc;
    need = plan.w1p_bytes + plan.w2p_bytes;
  }
  if (need > (size_t)DITTO_STATIC_WORKSPACE_BYTES)
    return fail(DITTO_EWORKSPACE, "the repacked weights take %zu bytes, the static workspace holds %zu", need,
                (size_t)DITTO_STATIC_WORKSPACE_BYTES);
  void* ws = nullptr;
  if (need > 0) {  // (depthwise chains stage their filters themselves and take no workspace)
    rc = static_workspace(&ws);
    if (rc != DITTO_OK) return rc;
  }
  // every byte of the workspace that the fused kernel reads is written by the repacking kernel of the
  // same call, ahead of it on `stream`: nothing has to be cleared between calls
  return conv_chain_call(kConvBoth, d, x, w1, w2, y, ws, ws ? (size_t)DITTO_STATIC_WORKSPACE_BYTES : 0, stream);
}
