// C ABI of libfrisk_hip.so: descriptor validation, the planner (tile / wave
// grid / LDS layout choice) and kernel dispatch.  Host code only.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "frisk_hip.h"
#include "gemm_internal.h"
#include "lds_model.h"
#include "tile_ops.h"
#include "attention.h"

// Scratch memory of frisk_hip_gemm_static_ws: the split-K / tail-split partial sums of callers that cannot allocate.
// Every GPU the library runs on holds its own copy of this array, at its own address, until the process ends.  In host
// code the name below is only a handle for hipGetSymbolAddress; kernels and copies get the device address it returns.
static __device__ __align__(256) unsigned char scratch[FRISK_HIP_STATIC_WS_BYTES];

namespace frisk {

static thread_local std::string g_last_error;

// device address of `scratch` on each device, resolved once per device with that device current
static constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];

static hipError_t scratch_of_current_device(void** out) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)); e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev].store(p, std::memory_order_release);  // racing threads resolve the same address
  }
  *out = p;
  return hipSuccess;
}

static int fail(int status, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return status;
}

static const std::vector<const KernelEntry*>& kernels() {
  static const std::vector<const KernelEntry*> all = [] {
    std::vector<const KernelEntry*> v;
    auto add = [&](const KernelEntry* table, int n) { for (int i = 0; i < n; ++i) v.push_back(&table[i]); };
    add(kKernelsF16, kNumKernelsF16);
    add(kKernelsF16_2, kNumKernelsF16_2);
    add(kKernelsF16_3, kNumKernelsF16_3);
    add(kKernelsF16_4, kNumKernelsF16_4);
    add(kKernelsBF16, kNumKernelsBF16);
    add(kKernelsBF16_2, kNumKernelsBF16_2);
    add(kKernelsBF16_3, kNumKernelsBF16_3);
    add(kKernelsBF16_4, kNumKernelsBF16_4);
    add(kKernelsI8, kNumKernelsI8);
    add(kKernelsI8_2, kNumKernelsI8_2);
    add(kKernelsI8_3, kNumKernelsI8_3);
    add(kKernelsI8_4, kNumKernelsI8_4);
    add(kKernelsE4M3, kNumKernelsE4M3);
    add(kKernelsE4M3_2, kNumKernelsE4M3_2);
    add(kKernelsE4M3_3, kNumKernelsE4M3_3);
    add(kKernelsE4M3_4, kNumKernelsE4M3_4);
    add(kKernelsF32, kNumKernelsF32);
    add(kKernelsF32_2, kNumKernelsF32_2);
    return v;
  }();
  return all;
}

static int elem_size(int dt) {
  switch (dt) {
    case FRISK_F32: case FRISK_I32: return 4;
    case FRISK_F16: case FRISK_BF16: return 2;
    case FRISK_I8: case FRISK_E4M3: return 1;
    default: return 0;
  }
}
static int frag_bytes(int dt) { return dt == FRISK_E4M3 ? 32 : 16; }
static int mfma_k(int dt) { return dt == FRISK_F32 ? 2 : (2 * frag_bytes(dt)) / elem_size(dt); }

// Wave partition of a block tile: the reference's computeWarpPartition
// (lib/Dialect/Frisk/IR/FriskOps.cpp:825-888) with waves of 64 lanes and
// per-wave granularity kM x kN (32 x 32 for the MFMA atoms used here).
static void wave_partition(int policy, int64_t M, int64_t N, int num_waves, int kM, int kN, int* wm, int* wn) {
  int64_t m_w = 1, n_w = num_waves;
  if (M == 0 || N == 0 || num_waves == 0) { *wm = 1; *wn = 1; return; }
  if (policy == FRISK_POLICY_FULL_ROW) {
    m_w = num_waves;
    if (M % (m_w * kM) != 0) {
      int64_t max_m = std::max<int64_t>(1, M / kM);
      m_w = std::max<int64_t>(1, std::min<int64_t>(num_waves, max_m));
    }
    n_w = std::max<int64_t>(1, num_waves / m_w);
  } else if (policy == FRISK_POLICY_FULL_COL) {
    n_w = num_waves;
    if (N % (n_w * kN) != 0) {
      int64_t max_n = std::max<int64_t>(1, N / kN);
      n_w = std::max<int64_t>(1, std::min<int64_t>(num_waves, max_n));
    }
    m_w = std::max<int64_t>(1, num_waves / n_w);
  } else {
    float ideal = (float)M / (float)N;
    float best = INFINITY;
    for (int64_t m = 1; m <= num_waves; ++m) {
      if (num_waves % m) continue;
      int64_t n = num_waves / m;
      float mp = (float)M / (float)(m * kM), np = (float)N / (float)(n * kN);
      if (mp < 1 || np < 1) continue;
      float score = std::fabs(mp / np - ideal);
      if (score < best) { best = score; m_w = m; n_w = n; }
    }
  }
  *wm = (int)std::max<int64_t>(1, m_w);
  *wn = (int)std::max<int64_t>(1, n_w);
}

// Kernels that the search over the variants leaves out, and no descriptor can name: the planner goes over to them from the kernel that the search has
// found (`follow_up` and `other_tile`).
static bool is_follow_up(const KernelEntry* k) {
  if (k->dtype == FRISK_F32) return k->bm == 32 && k->bn == 32 && !k->splitk;
  return (k->bm == 64 && k->bn == 64) || k->bm == 160 || k->bm == 224 || (k->bm == 128 && k->bn == 128 && k->edge && k->stages == 3);
}

// The compiled variants of one element type and pair of layouts, in table order, with what the planner would otherwise work out
// for each of them on every call: which wave policies their wave grid satisfies (computeWarpPartition gives it for their tile and
// wave count).  A launch of a 128x128x128 product spent 0.75 of its 3.9 us of host time walking the whole table.
struct Variant { const KernelEntry* k; int id; bool policy[3]; bool follow_up; };
static const std::vector<Variant>& variants(int dtype, bool transA, bool transB) {
  static const std::vector<std::vector<Variant>> all = [] {
    std::vector<std::vector<Variant>> v(6 * 4);
    const auto& ks = kernels();
    for (size_t i = 0; i < ks.size(); ++i) {
      Variant x{ks[i], (int)i, {}, is_follow_up(ks[i])};
      for (int policy = 0; policy < 3; ++policy) {
        int wm = 0, wn = 0;
        wave_partition(policy, x.k->bm, x.k->bn, x.k->wm * x.k->wn, x.k->atom, x.k->atom, &wm, &wn);
        x.policy[policy] = wm == x.k->wm && wn == x.k->wn;
      }
      v[(size_t)(x.k->dtype * 4 + x.k->transA * 2 + x.k->transB)].push_back(x);
    }
    return v;
  }();
  return all[(size_t)(dtype * 4 + (transA ? 2 : 0) + (transB ? 1 : 0))];
}

static int validate(const frisk_gemm_desc* d) {
  if (!d) return fail(FRISK_ERR_NULL, "descriptor is null");
  if (d->abi_version != FRISK_HIP_ABI_VERSION)
    return fail(FRISK_ERR_ABI, "descriptor abi_version %d, library %d", d->abi_version, FRISK_HIP_ABI_VERSION);
  const int ab = d->dtype_ab, acc = d->dtype_acc, out = d->dtype_out;
  bool ok = false;
  switch (ab) {
    case FRISK_F32: ok = acc == FRISK_F32 && out == FRISK_F32; break;
    case FRISK_F16: ok = acc == FRISK_F32 && (out == FRISK_F16 || out == FRISK_F32); break;
    case FRISK_BF16: ok = acc == FRISK_F32 && (out == FRISK_BF16 || out == FRISK_F32); break;
    case FRISK_I8: ok = acc == FRISK_I32 && (out == FRISK_I32 || out == FRISK_F16 || out == FRISK_F32); break;
    case FRISK_E4M3: ok = acc == FRISK_F32 && (out == FRISK_BF16 || out == FRISK_F16 || out == FRISK_F32); break;
    default: ok = false;
  }
  if (!ok) return fail(FRISK_ERR_DTYPE, "unsupported element types: ab=%d acc=%d out=%d", ab, acc, out);
  if (d->epilogue < FRISK_EPI_NONE || d->epilogue > FRISK_EPI_TENSOR_SCALE)
    return fail(FRISK_ERR_EPILOGUE, "unknown epilogue %d", d->epilogue);
  if (out == FRISK_I32 && d->epilogue != FRISK_EPI_NONE)
    return fail(FRISK_ERR_EPILOGUE, "int32 output carries the raw accumulators; scales need a floating output type");
  if (d->policy < FRISK_POLICY_SQUARE || d->policy > FRISK_POLICY_FULL_COL)
    return fail(FRISK_ERR_TILE, "unknown wave policy %d", d->policy);
  if (d->atom != 0 && d->atom != 16 && d->atom != 32) return fail(FRISK_ERR_TILE, "MFMA atoms have 32 or 16 rows, not %d", d->atom);
  if (d->M < 0 || d->N < 0 || d->K < 0) return fail(FRISK_ERR_SHAPE, "negative extent M=%lld N=%lld K=%lld", (long long)d->M, (long long)d->N, (long long)d->K);
  if (d->M > INT32_MAX || d->N > INT32_MAX || d->K > INT32_MAX) return fail(FRISK_ERR_SHAPE, "extent exceeds 2^31-1");
  const int64_t a_cols = d->transA ? d->M : d->K, b_cols = d->transB ? d->K : d->N;
  if (d->lda < std::max<int64_t>(1, a_cols)) return fail(FRISK_ERR_SHAPE, "lda=%lld smaller than the stored row length %lld", (long long)d->lda, (long long)a_cols);
  if (d->ldb < std::max<int64_t>(1, b_cols)) return fail(FRISK_ERR_SHAPE, "ldb=%lld smaller than the stored row length %lld", (long long)d->ldb, (long long)b_cols);
  if (d->ldc < std::max<int64_t>(1, d->N)) return fail(FRISK_ERR_SHAPE, "ldc=%lld smaller than N=%lld", (long long)d->ldc, (long long)d->N);
  return FRISK_OK;
}

static void fill_layout(frisk_lds_layout* L, bool kcontig, int es, int fragb, int mn, int bk, int nw, int atom) {
  TileShape t{kcontig ? mn : bk, (kcontig ? bk : mn) * es, kcontig, es, fragb, mn, bk, atom};
  Swizzle s = default_swizzle(kcontig, es, t.rowb, atom);
  L->rows = t.rows;
  L->row_bytes = t.rowb;
  L->k_contiguous = kcontig;
  L->row_shift = s.sh;
  L->row_mask = s.mk;
  L->chunk_shift = s.cs;
  L->row_shift2 = s.sh2;
  L->row_mask2 = s.mk2;
  L->chunk_shift2 = s.cs2;
  L->read_instr = kcontig ? 0 : (es == 4 ? 3 : (es == 2 ? 1 : 2));
  int atoms = mn / atom < 4 ? mn / atom : 4;
  int n_access = atoms * ((bk * es) / frag_kstep_bytes(fragb, atom)) * frag_instr_count(kcontig, es, fragb);
  // evaluating the bank model costs ~0.1 ms of host time
  L->read_cycles = n_access ? (float)swizzle_read_cycles(t, s) / (float)n_access : 0.f;
  // the direct-to-LDS transfer writes 64 consecutive 16-byte slots: no conflicts by construction
  L->write_cycles = 16.f;
  (void)nw;
}

// Workspace a plan may use: any (what frisk_hip_plan reports), a limit (splits of K of as many slices as fit; a tail split fits or is dropped), or
// none.
static constexpr size_t kAnyWorkspace = ~(size_t)0;

// Tail split: a grid of a little more than a whole number of rounds of 256 tiles leaves most CUs idle in its last round.
// The last tiles % 256 tiles (at most half a round) are then computed by several work-groups each: with a kernel that has the split-K store path by 2, 4
// or 8 with an equal share of the K tiles apiece, with a large edge kernel by any 2 to 8, whose last share may be shorter.  Returns that count, 1 for no
// split.
static int tail_split_of(const KernelEntry* k, int64_t tiles, int64_t kt, bool whole_k_tiles, size_t workspace) {
  // the edge kernels deal any number of K tiles: their last slice may be shorter (us unsplit / split: bf16 3000x11008x4096 NT, 516
  // tiles, 248 / 212; fp16 4097x4097x4096 NT, 289 tiles, 161 / 126; 4095x4097x4001 NN with its copy to aligned rows 204 / 150)
  const bool edge = k->edge && !k->splitk && (int64_t)k->bm * k->bn >= 192 * 256;
  if (!edge && (!k->splitk || k->bm < 128 || k->wk > 1 || !whole_k_tiles)) return 1;
  if (tiles <= 256 || workspace == 0) return 1;
  const int64_t rest = tiles % 256;
  if (rest == 0 || rest > 128) return 1;
  // shallower slices do not repay the second launch (measured); the 8-bit kernels run a K tile of twice the depth in the same
  // time, so the summing pass weighs twice as much against their slices (fp8 5120x4096x4096: 64 tiles in 4 slices of 8 K tiles
  // 92.4 us, unsplit 84, 256x128 tiles 81.4)
  const int min_slice = elem_size(k->dtype) == 1 ? 16 : 8;
  for (int s = 8; s >= 2; s = edge ? s - 1 : s / 2) {
    const int64_t per = (kt + s - 1) / s;
    if (rest * s <= 256 && (edge ? (s - 1) * per < kt : kt % s == 0) && per >= min_slice) return (size_t)(s * rest) * k->bm * k->bn * 4 <= workspace ? s : 1;
  }
  return 1;
}

// The same for edge kernels on grids of at most half a round, whose tiles are then all split: the most slices that leave one work-group
// per CU and enough K tiles to each (any K, unequal slices: what the split-K kernels do for whole tiles).  us unsplit / split:
// fp16 1589x3072x9600 NN 114 / 91, 2100x2100x8000 TN 130 / 103, 1500x2816x11008 NN 131 / 90, 1001x1003x4001 NN 56.5 / 31.3, 1000x1000x4000 NT
// 45.0 / 24.9, 600x4100x4100 TN 59.9 / 54.4, bf16 704x960x4032 TN 39.6 / 20.8, 17x4096x4096 TN 52.7 / 18.9, int8 576x1088x8064 TN 46.1 / 25.2,
// e4m3 704x512x5760 TT 32.8 / 23.5
static bool edge_slices_ok(const KernelEntry* k, const frisk_gemm_desc* d, int slices) {
  const int64_t kt = (d->K + k->bk - 1) / k->bk, per = (kt + slices - 1) / slices;
  return per >= (elem_size(k->dtype) == 1 ? 16 : 8) && (slices - 1) * per < kt;
}
static int edge_split_of(const KernelEntry* k, const frisk_gemm_desc* d, size_t workspace) {
  if (!k->edge || k->splitk || k->wk > 1 || k->bm < 128 || k->dtype == FRISK_F32) return 1;
  const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn);
  if (tiles > 128 || tiles == 0) return 1;
  for (int s = (int)std::min<int64_t>(8, 256 / tiles); s >= 2; --s)
    if (edge_slices_ok(k, d, s) && (size_t)(s * tiles) * k->bm * k->bn * 4 <= workspace) return s;
  return 1;
}

// Slices of K are whole K tiles, of unequal length where their number does not divide the K tiles: all as long as the first but the last, which gets
// what is left, at least what the kernel's loop is written for.  (Divisors alone left a
// prime number of K tiles, or twice one, in few slices or one: us so / now, fp16 4x576x6784 NN 17.4 / 9.6, 21x5952x7808 32.8 / 21.4, bf16 3x6848x6016 25.3 / 18.7,
// 198x896x7552 22.0 / 15.5, int8 3x2240x6784 16.5 / 10.3, e4m3 58x2240x7552 19.2 / 11.9.)
static bool slices_ok(const KernelEntry* k, int64_t kt, int slices) {
  const int64_t per = (kt + slices - 1) / slices, last = kt - (slices - 1) * per;
  return last >= std::max(1, slices > 1 ? k->min_k_tiles : 1);
}

// the split the planner gives a grid below one round of a variant with the split-K store path: up to one work-group per CU,
// at least 4 K tiles per slice
static int sub_round_split(const KernelEntry* k, const frisk_gemm_desc* d, int64_t tiles, int64_t kt, size_t workspace) {
  int split = 1;
  for (int c = 2; c <= 64 && tiles * c <= 256; ++c)
    if (slices_ok(k, kt, c) && (kt + c - 1) / c >= std::max(4, k->min_k_tiles) && (size_t)c * (size_t)d->M * (size_t)d->N * 4 <= workspace) split = c;
  return split;
}

// K tile of the kernel that stages through registers against the one of the same tile that transfers straight to LDS (fp16 NN, us,
// registers against copy + LDS transfers on 128x128 tiles: 4095x4097x4001 304 / 227, 1999x4099x3001 154 / 100, 1001x999x1003 31 / 21)
static constexpr double kStagedFactor = 1.6;

// Relative time of a problem on a kernel variant, used only to rank the variants.  One wave of work-groups = one per CU
// (256); a K tile of a 256x256 tile costs 1.5 units when every CU runs one, and less when the chip is partly idle
// (less contention in the L2 and a higher clock): factor 0.6 + 0.4 * fill.  The constants are measured on fp16 problems
// between 1024^3 and 8192^3 and carry over to the 8-bit types, whose K tiles hold the same number of bytes.
static double estimated_cost(const KernelEntry* k, const frisk_gemm_desc* d, bool may_split, bool split_edges, size_t workspace) {
  const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn);
  const double kt = (double)((d->K + k->bk - 1) / k->bk);
  double c;  // cost of one K tile with the chip full
  const int64_t area = (int64_t)k->bm * k->bn;
  if (k->dtype == FRISK_F32) {
    // Measured with 16-byte fragments (K-contiguous tiles read by ds_read_b128), us, NN: 1024^3 64x64x32 18.8, x64 19.4, x128 on 8 waves
    // 19.5; 1536^3 69.4 / 73.8 / 78.6; 2048^3 128x128x32 120.8, x16 in a ring of 4 124.1, 64x64x32 123.3; 4096^3 928 / 941 / 962.
    const double c128 = k->bk <= 16 ? ((!k->transA && k->transB) ? 1.0 : 0.91) : 1.74;
    // 64x64x32 per round and K tile of 32: 0.497 us over 9, 25 and 43 rounds (3072^3 429, 5120^3 1987, 4096x11008x4096 2779 us) against
    // 1.81 us for a round of 128x128x32 (4096^3 926, 4096x11008x4096 2549): a quarter of the tile at 0.27 of the cost
    c = area >= 128 * 128 ? c128 : (k->wk > 1 ? (tiles <= 256 ? 1.8 : 2.3) : (k->bk >= 64 ? 1.0 : (tiles <= 256 ? 0.44 : 0.465)));
  } else if (k->bm == 32) {
    // 32x32 with a 4x deeper K tile; 32x128 (8-bit: 60.1 us for 256 tiles x 64 K tiles, the rate of the 32x32 kernel per K tile)
    c = k->wk > 1 ? 0.8 : (elem_size(k->dtype) == 1 ? 0.85 : 0.25);
  } else if (area >= 256 * 256) {
    c = k->wm * k->wn > 4 ? 1.56 : (k->stages_b > k->stages ? 1.5 : 1.55);  // 2 + 3 ring < 2 + 2 < 8 waves
    // 16x16 atoms: the same cycles at a higher clock when most CUs are busy (fp16 4096^3 NT 100 against 112 us); with an operand
    // read by transpose reads (twice the LDS instructions) less of it is left (NN 104 against 108).  How full the round is decides:
    // 192 or 196 tiles, NN 78 against 82 us (3584^3) and 164 against 172 (4096x3072x8192), TN 79 against 85 and 169 against 182;
    // 144 tiles (3072^3): NN 61 against 59 and TN even while the loop held several LDS reads per MFMA slot, NN 51.3 against 53.7
    // (fp16), 50.4 against 51.3 (bf16), 30.6 against 31.2 (int8) since it holds one
    // 8-bit floats on the 16x16x128 atom (NT only), us against the 32x32x64 atoms: 8192^3 331 / 351, 4096^3 45.1 / 48.8, 4096x4096x512
    // 11.8 / 12.9, 4096x11008x4096 128 / 133, 6144^3 176 / 183; 3072^3 (144 tiles) 29.6 / 28.6
    if (k->atom == 16) c *= k->dtype == FRISK_E4M3 ? (tiles >= 176 ? 0.94 : 1.04) : (!k->transA && k->transB) ? 0.93 : (tiles >= 176 ? 0.96 : 0.98);
  } else if (k->bm == 192) {
    // three quarters of a 256x256 tile at 0.78 to 0.80 of its time.  us on 256x256 / 192x256 tiles: bf16 3000x4096x11008 NN (192 / 256
    // tiles) 202.8 / 178.6, fp16 1999x4099x3001 NN 77.2 / 64.8, 2880x3840x2048 NT 47.8 / 38.3, 6720x5760x1024 NN 101 / 92, int8
    // 3000x4096x4096 NN 54.8 / 43.1, 7296x4992x4096 NT 148 / 122, e4m3 the same two NT 52.3 / 42.8 and 142 / 124; where 256x256 tiles
    // fill their rounds: fp16 3840x4096x8192 172 / 195, int8 89 / 117
    c = k->dtype == FRISK_E4M3 ? 1.2 : 1.12;
  } else if (area >= 256 * 128) {
    c = 0.93;
  } else {
    // 3 + 3 tiles when the grid is one wave, 2 + 2 (two work-groups per CU) beyond
    c = k->stages >= 3 ? (tiles <= 256 ? 0.46 : 0.55) : (tiles <= 256 ? 0.55 : 0.52);
    // 128x64 tiles with a K tile twice as deep: as many MFMAs a K tile as 128x128, 1.5 times its transfers.  us on 128x64 / what it runs on instead: fp16
    // 3072x1792x1536 NT 32.8 / 21.9, 3200x1920x4352 85.9 / 53.5, 896x6592x6016 117 / 81
    if (k->bm == 128 && k->bn == 64) c *= 1.5;
  }
  if (k->guard && !k->edge && k->dtype == FRISK_F32) c *= kStagedFactor;  // (the other types: make_plan, at its search)
  if (k->bm == 32 && k->wk > 1) {
    // The 32x32 kernel streams B.  With a ring of 4 tiles one work-group fills a CU: whole rounds of 256, each paying its
    // own start (measured 14.8 us for 256 tiles, 35.8 for 512).  With a ring of 2 two work-groups share a CU: slower alone
    // (17.5 us for 256 tiles), but beyond 256 tiles the rounds overlap (29.3 us for 512, 46.6 for 896).
    if (k->stages >= 3) return (double)((tiles + 255) / 256) * kt * c * (tiles > 256 ? 1.2 : 1.0) / (tiles < 256 ? std::max((double)tiles / 256.0, 0.25) : 1.0);
    return tiles <= 256 ? kt * c * 1.19 / std::max((double)tiles / 256.0, 0.25) : (double)tiles / 256.0 * kt * c;
  }
  const int64_t full = tiles / 256, rest = tiles % 256;
  const double rest_fill = (double)rest / 256.0;
  if (may_split && k->splitk && k->bm >= 128 && tiles < 256 && d->K % k->bk == 0) {
    // below one round with a deep K the planner splits K over the idle CUs (2048x4096x16384 fp16: 128 tiles of 256x256 in 2
    // slices 209.5 us, 256 tiles of 256x128 unsplit 243.6): the slices' K tiles at the fill they reach, plus the summing pass
    const int cs = sub_round_split(k, d, tiles, (int64_t)kt, workspace);
    // (measured: the slices' loops 8 % above the per-K-tile rate of a long loop, the pass at 256 KiB per tile and slice in 0.07 us;
    // 1024x8192x8192 comes out even with 256x128 tiles unsplit, 123.7 against 123.9 us, and stays unsplit)
    if (cs > 1) return (double)(((int64_t)kt + cs - 1) / cs) * c * (0.6 + 0.4 * rest_fill * cs) * 1.08 + 5.0 + 0.07 * (double)(tiles * cs);
  }
  double cost = (double)full * kt * c;
  if (rest) {
    if (k->bm == 32)  // the skinny kernels are bound by streaming B and need the parallelism: idle CUs are lost bandwidth
      cost += full ? kt * c : kt * c / std::max(rest_fill, 0.25);
    else
      cost += kt * c * (0.6 + 0.4 * rest_fill);
  }
  // the last `rest` tiles as ts work-groups each, a ts-th of the K tiles apiece, plus the pass that sums them
  // (a dependent launch, and rest * ts tiles of 32-bit partial sums to read)
  auto tail_cost = [&](int ts) { return (double)full * kt * c + kt / ts * c * (0.6 + 0.4 * rest_fill * ts) + 5.0 + 0.04 * (double)(rest * ts); };
  if (k->edge && !k->splitk) {
    if (!may_split || !split_edges) return cost;
    // at most what one pass costs; but rows that end off a K tile slow a pass of many K tiles more than this knows (bf16 4099x3857x1976 TN, us in
    // one pass / split: 88.8 / 74.9; at K = 1984 89.6 / 77.3)
    const double one_pass = d->K % k->bk == 0 ? cost : INFINITY;
    if (const int cs = tiles <= 128 ? edge_split_of(k, d, workspace) : 1; cs > 1)
      return std::min(one_pass, kt / cs * c * (0.6 + 0.4 * rest_fill * cs) * 1.08 + 5.0 + 0.07 * (double)(tiles * cs) * (double)area / (256 * 256));
    const int ts = tail_split_of(k, tiles, (int64_t)kt, false, workspace);
    return ts > 1 ? std::min(one_pass, tail_cost(ts)) : cost;
  }
  if (const int ts = tail_split_of(k, tiles, (int64_t)kt, d->K % k->bk == 0, workspace ? workspace : kAnyWorkspace); ts > 1) return tail_cost(ts);
  return cost;
}

// Grids of at most 256 tiles of 128 x 128 (a few hundred rows, or a small square): no variant fills the chip with one
// work-group per tile, so the choice is a (variant, split of K) pair.  Measured per element type over 81 skinny shapes (M 32 ..
// 2048, N and K 1024 .. 28672) and 90 squarish ones (sides 768 .. 2048, K 1024 .. 8192), both layouts of B, every variant at
// every split 1 .. 32, B taken in turn from as many copies as fill 400 MiB so that it streams from HBM as the weights of a model
// do (with one B of at most 128 MiB the last-level cache serves it: 26.5 instead of 38 us at fp16 64x8192x8192).  The sweep's splits of a
// variant were the powers of two that keep tiles x split within `w` work-groups and `kmin` K tiles per slice (small_grid_split goes beyond them); variants and splits are compared by a time model fitted to the sweep, in microseconds:
//   launch + whole rounds x (K tiles x tk + ps) + a last round at K tiles x tk x (a + (1 - a) x fill) + the summing pass
//   (r0 + r1 x megabytes of partial sums) when split;
// variants of which a CU holds two work-groups (`cap` 512) pay tk2 per K tile more once any CU holds its second one:
// K tiles x tk2 x (a2 + (1 - a2) x fill of the second half).  The pair chosen this way is 2 % slower on average than the
// best pair of the sweep (more than 1.2x in 24 of 966 cases); the one-size rule used before lost 35-40 % on
// average on the skinny shapes.
struct SmallGridModel { int cap, w, kmin; float launch, tk, a, r0, r1, ps, tk2, a2; };
static const SmallGridModel kSmallGrid[3][14] = {
    {  // 16-bit
        {512, 0, 0, 0.57f, 0.783f, 0.77f, 5.00f, 0.200f, 1.00f, 0.300f, 0.50f},  // 128x128 s2
        {256, 256, 16, 2.32f, 0.551f, 0.73f, 5.64f, 0.300f, 4.27f, 0.000f, 0.00f},  // 128x128 s3
        {256, 0, 0, 3.66f, 0.879f, 0.76f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 128x256 s3
        {256, 0, 0, 4.17f, 0.833f, 0.74f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x128 s3
        {256, 256, 16, 9.37f, 1.496f, 0.52f, 0.00f, 0.300f, 8.37f, 0.000f, 0.00f},  // 256x256 s2
        {256, 256, 16, 5.82f, 1.307f, 0.66f, 2.98f, 0.300f, 8.84f, 0.000f, 0.00f},  // 256x256 s2 a16
        {256, 0, 0, 0.83f, 2.046f, 0.53f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x256 s2 w8
        {512, 128, 16, 0.36f, 0.456f, 0.74f, 6.46f, 0.300f, 0.00f, 0.211f, 0.88f},  // 32x128 s3 n
        {512, 128, 16, 0.12f, 0.465f, 0.76f, 6.43f, 0.300f, 0.00f, 0.170f, 1.00f},  // 32x128 s3 t
        {512, 256, 16, 2.40f, 0.744f, 0.68f, 7.68f, 0.000f, 0.00f, 0.222f, 0.72f},  // 32x32 s2 t
        {256, 128, 16, 2.88f, 0.580f, 0.65f, 6.64f, 0.000f, 0.03f, 0.000f, 0.00f},  // 32x32 s4 t
        {512, 256, 16, 1.56f, 0.436f, 0.69f, 7.25f, 0.300f, 2.21f, 0.315f, 0.41f},  // 64x128 s3
        {256, 256, 16, 3.28f, 0.638f, 0.82f, 6.76f, 0.000f, 1.01f, 0.000f, 0.00f},  // 64x32 s3
        {256, 256, 16, 2.59f, 0.851f, 0.83f, 5.42f, 0.065f, 0.79f, 0.000f, 0.00f},  // 128x64 s3
    },
    {  // int8
        {512, 0, 0, 2.56f, 0.726f, 0.76f, 5.00f, 0.200f, 1.00f, 0.300f, 0.50f},  // 128x128 s2
        {256, 256, 16, 3.38f, 0.558f, 0.65f, 5.70f, 0.300f, 4.52f, 0.000f, 0.00f},  // 128x128 s3
        {256, 0, 0, 4.88f, 0.908f, 0.71f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 128x256 s3
        {256, 0, 0, 4.92f, 0.827f, 0.76f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x128 s3
        {256, 256, 16, 8.27f, 1.618f, 0.56f, 0.00f, 0.300f, 7.84f, 0.000f, 0.00f},  // 256x256 s2
        {256, 256, 16, 6.65f, 1.471f, 0.60f, 2.63f, 0.300f, 5.73f, 0.000f, 0.00f},  // 256x256 s2 a16
        {256, 0, 0, 4.80f, 1.741f, 0.61f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x256 s2 w8
        {512, 128, 16, 2.00f, 0.461f, 0.65f, 4.98f, 0.300f, 0.00f, 0.222f, 0.70f},  // 32x128 s3 n
        {512, 128, 16, 1.96f, 0.436f, 0.69f, 5.27f, 0.300f, 0.00f, 0.188f, 0.88f},  // 32x128 s3 t
        {512, 256, 16, 3.09f, 0.678f, 0.71f, 4.29f, 0.300f, 0.59f, 0.199f, 1.00f},  // 32x32 s2 t
        {256, 128, 16, 3.29f, 0.532f, 0.66f, 4.15f, 0.000f, 0.53f, 0.000f, 0.00f},  // 32x32 s4 t
        {512, 256, 16, 2.72f, 0.443f, 0.65f, 6.47f, 0.300f, 1.56f, 0.377f, 0.36f},  // 64x128 s3
        {256, 256, 16, 3.47f, 0.646f, 0.87f, 4.48f, 0.300f, 1.19f, 0.000f, 0.00f},  // 64x32 s3
        {256, 256, 16, 3.04f, 0.844f, 0.83f, 4.14f, 0.300f, 0.89f, 0.000f, 0.00f},  // 128x64 s3
    },
    {  // 8-bit float
        {512, 0, 0, 2.63f, 0.708f, 0.74f, 5.00f, 0.200f, 1.00f, 0.300f, 0.50f},  // 128x128 s2
        {256, 256, 16, 3.32f, 0.485f, 0.67f, 4.85f, 0.300f, 2.07f, 0.000f, 0.00f},  // 128x128 s3
        {256, 0, 0, 4.85f, 0.854f, 0.62f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 128x256 s3
        {256, 0, 0, 4.62f, 0.802f, 0.67f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x128 s3
        {256, 256, 16, 7.47f, 1.283f, 0.68f, 0.41f, 0.300f, 7.22f, 0.000f, 0.00f},  // 256x256 s2
        {256, 256, 16, 6.48f, 1.195f, 0.74f, 1.99f, 0.300f, 6.48f, 0.000f, 0.00f},  // 256x256 s2 a16
        {256, 0, 0, 4.17f, 1.217f, 1.00f, 5.00f, 0.200f, 1.00f, 0.000f, 0.00f},  // 256x256 s2 w8
        {512, 128, 16, 1.98f, 0.421f, 0.67f, 5.23f, 0.300f, 0.00f, 0.148f, 1.00f},  // 32x128 s3 n
        {512, 128, 16, 1.98f, 0.421f, 0.67f, 5.23f, 0.300f, 0.00f, 0.148f, 1.00f},  // 32x128 s3 t
        {512, 256, 16, 2.79f, 0.698f, 0.71f, 4.93f, 0.000f, 0.57f, 0.225f, 1.00f},  // 32x32 s2 t
        {256, 128, 16, 2.98f, 0.514f, 0.73f, 4.23f, 0.000f, 0.67f, 0.000f, 0.00f},  // 32x32 s4 t
        {512, 256, 16, 2.79f, 0.386f, 0.74f, 5.38f, 0.300f, 0.88f, 0.302f, 0.44f},  // 64x128 s3
        {256, 256, 16, 3.53f, 0.630f, 0.89f, 4.81f, 0.291f, 1.23f, 0.000f, 0.00f},  // 64x32 s3
        {256, 256, 16, 3.26f, 0.649f, 0.80f, 5.42f, 0.095f, 1.14f, 0.000f, 0.00f},  // 128x64 s3
    },
};
// fp32: one 64x64 work-group of four waves already keeps a CU's matrix pipe busy (a 32x32x2 MFMA is 64 cycles), so time follows
// the work of the busiest CU and idle CUs are lost outright: 256x256x8192 runs 127 us on its 16 tiles and 23 us with K split 16
// ways.  Fitted to 70 skinny and 50 squarish shapes, both layouts of B, B from HBM.
static const SmallGridModel kSmallGridF32[11] = {
    {512, 0, 0, 4.84f, 1.832f, 0.94f, 0.00f, 0.000f, 1.00f, 0.300f, 0.50f},  // 128x128x32 s2
    {512, 0, 0, 4.95f, 0.944f, 0.91f, 0.00f, 0.000f, 1.00f, 0.300f, 0.50f},  // 128x128x16 s4
    {512, 0, 0, 2.36f, 0.612f, 0.73f, 0.00f, 0.000f, 0.00f, 0.398f, 0.87f},  // 64x64x32 s2
    {512, 4096, 8, 3.95f, 0.536f, 0.72f, 5.54f, 0.071f, 1.66f, 0.443f, 0.83f},  // 64x64x32 s3
    {512, 0, 0, 2.38f, 1.208f, 0.82f, 0.00f, 0.000f, 0.00f, 0.905f, 0.87f},  // 64x64x64 s2
    {256, 0, 0, 4.18f, 2.138f, 0.87f, 0.00f, 0.000f, 1.27f, 0.000f, 0.00f},  // 64x64x128 s2, 8 waves
    {512, 512, 8, 3.12f, 0.630f, 0.76f, 4.56f, 0.817f, 0.00f, 0.635f, 0.48f},  // 32x128x32 s3 n
    {512, 512, 8, 2.58f, 0.639f, 0.72f, 5.36f, 0.534f, 0.36f, 0.594f, 0.53f},  // 32x128x32 s3 t
    {512, 512, 4, 2.35f, 0.857f, 0.78f, 4.01f, 0.947f, 0.00f, 0.573f, 0.50f},  // 32x32x128 s2 t
    {256, 256, 4, 3.06f, 0.735f, 0.89f, 3.36f, 1.485f, 1.05f, 0.000f, 0.00f},  // 32x32x128 s4 t
    {256, 256, 4, 3.32f, 1.127f, 0.98f, 4.25f, 0.048f, 2.24f, 0.000f, 0.00f},  // 64x32x128 s3 t
};
static int small_grid_class_f32(const KernelEntry* k) {
  if (k->bm == 32) return k->bn == 32 ? (k->stages >= 3 ? 9 : 8) : (k->transB ? 7 : 6);
  if (k->bn == 32) return 10;
  if (k->bm == 128) return k->bk <= 16 ? 1 : 0;
  if (k->bk >= 128) return 5;
  if (k->bk >= 64) return 4;
  return k->stages >= 3 ? 3 : 2;
}
static int small_grid_class(const KernelEntry* k) {
  if (k->bm == 32) return k->bn == 32 ? (k->stages >= 3 ? 10 : 9) : (k->transB ? 8 : 7);
  if (k->bm == 64) return k->wk > 1 ? 12 : 11;
  if (k->bm == 128 && k->bn == 64) return 13;
  if ((int64_t)k->bm * k->bn >= 256 * 256) return k->wm * k->wn > 4 ? 6 : (k->atom == 16 ? 5 : 4);
  if (k->bm == 256) return 3;
  if (k->bn == 256) return 2;
  return k->stages >= 3 ? 1 : 0;
}
static bool small_grid(const frisk_gemm_desc* d) {
  return d->split_k <= 1 && ((d->M + 127) / 128) * ((d->N + 127) / 128) <= 256;
}
static const SmallGridModel& small_grid_model(const KernelEntry* k) {
  if (k->dtype == FRISK_F32) return kSmallGridF32[small_grid_class_f32(k)];
  return kSmallGrid[k->dtype == FRISK_I8 ? 1 : (k->dtype == FRISK_E4M3 ? 2 : 0)][small_grid_class(k)];
}
static double small_grid_time(const SmallGridModel& m, const KernelEntry* k, const frisk_gemm_desc* d, int split) {
  const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn);
  const double kt = (double)(((d->K + k->bk - 1) / k->bk + split - 1) / split);  // of the longest slice
  const int64_t wgs = tiles * split, full = wgs / m.cap, rest = wgs % m.cap;
  // One row of 64x128 tiles against a B stored [N][K] streams it 128 bytes of a row at a time, which is slow where its rows are a multiple of 16 KiB
  // apart and little slower elsewhere.  us on them / on 64x32 tiles, whose K tiles are four times as deep: fp16 48x8192x8192 37.0 / 28.7,
  // 48x16384x8192 64.3 / 54.8; but 49x10368x3712 18.6 / 23.8, 51x10112x2688 14.2 / 19.4, 35x14400x3968 26 / 32 (B from the last-level cache)
  const bool one_row = k->bm == 64 && k->bn == 128 && k->transB && tiles * k->bn < d->N + k->bn;
  const bool far_rows = d->K * elem_size(k->dtype) % 16384 == 0;
  const double tk = m.tk * (!one_row ? 1.0 : far_rows ? 1.4 : split == 1 ? 1.05 : 1.0);
  double t = m.launch, whole = kt * tk + m.ps, last = 0.0;
  if (m.cap == 512) {  // two work-groups per CU: the second one of any CU sets the pace of the round
    whole += kt * m.tk2;
    const double f1 = (double)std::min<int64_t>(rest, 256) / 256.0, f2 = (double)std::max<int64_t>(rest - 256, 0) / 256.0;
    last = kt * (tk * (m.a + (1.0 - m.a) * f1) + (rest > 256 ? m.tk2 * (m.a2 + (1.0 - m.a2) * f2) : 0.0));
  } else {
    last = kt * tk * (m.a + (1.0 - m.a) * (double)rest / m.cap);
  }
  t += (double)full * whole + (rest ? last : 0.0);
  // (64x32 tiles beyond one round, which the sweep behind the table held few of, take 10 % longer than their rounds add up to: with both rules 12 of 1048
  // drawn problems of 1 to 64 rows are more than 8 % slower than on 64x128 and 32x128 tiles, 134 before)
  if (k->bm == 64 && k->wk > 1 && k->dtype != FRISK_F32 && wgs > 256 && !far_rows) t *= 1.1;
  if (split > 1) t += m.r0 + m.r1 * ((double)d->M * (double)d->N * split * 4.0 / 1e6);
  return k->guard && !k->edge ? kStagedFactor * t : t;
}
// the split of a variant: among those the rule admits, the one the model makes fastest; *cost receives its time.  `edges`: edge kernels may
// be split too.  `table_range`: only splits of the range that the table was fitted over; *range_cost receives the time of the best of those
static bool in_table_range(const KernelEntry* k, const frisk_gemm_desc* d, int split) {
  const SmallGridModel& m = small_grid_model(k);
  const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn);
  return split == 1 || (!(split & (split - 1)) && d->K / k->bk % split == 0 && d->K / k->bk / split >= m.kmin && tiles * split <= m.w);
}
static int small_grid_split(const KernelEntry* k, const frisk_gemm_desc* d, size_t workspace, bool edges, bool table_range, double* cost = nullptr, double* range_cost = nullptr) {
  const SmallGridModel& m = small_grid_model(k);
  int best = 1;
  double best_t = small_grid_time(m, k, d, 1), range_t = best_t;
  if (k->splitk && workspace && d->split_k != 1 && m.w != 0 && d->K % k->bk == 0) {
    const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn), kt = d->K / k->bk;
    // any divisor of the K tiles (K = 5760 is 45 tiles of 128: the powers of two left it unsplit); the sweeps behind the tables: up to 64
    // slices, fp32 32
    // At least 4 K tiles a slice and up to 256 work-groups, whatever range of splits a class was fitted over (`kmin`, `w`; B stored [N][K]
    // keeps its `w`: there the unsplit tiles that stream B are as good): the model holds beyond it.  us at 16 K tiles and 128 or 256 work-groups / now: int8
    // 40x2880x7040 NN 29.5 / 12.8, e4m3 59x7104x4608 21.7 / 14.2, fp16 37x6720x3328 23.7 / 14.5, 16x2496x4224 14.7 / 11.3, 276x1280x3520 17.5 / 12.4;
    // 70 drawn sizes whose split changed 1.27 times faster, the worst 0.94 (3x9536x5760).  512 work-groups: 0.96 on 45.
    // A descriptor that names a tile stays within the fitted range: the unsplit and the split kernel of one tile are different kernels, and
    // which of the two a tile names is not to move with the model (e4m3 512x512x2048 on 256x256 tiles of the 16x16x128 atom: unsplit).
    const bool named = d->tile_m || d->tile_n || d->tile_k;
    const int64_t wgs = k->transB || named ? m.w : std::max(m.w, 256);
    const int kmin = std::max(named ? m.kmin : std::min(m.kmin, 4), k->min_k_tiles);
    const int64_t most = std::min<int64_t>({k->dtype == FRISK_F32 ? 32 : 64, tiles > 0 ? wgs / tiles : 0, kt / kmin});
    // fp32: a split within the range that the table was fitted over (powers of two) gives way to one of more slices of at most 10 K tiles for 12 % of modelled
    // time: the bare model takes some to shorter slices that are slower.  us in 4 slices / in what it takes: 60x2752x1152 NT 12.2 / 13.3 (9), 88x1536x1152
    // 11.5 / 12.7 (9), 107x1408x2176 15.9 / 17.4 (17), 411x384x2944 18.3 / 20.2 (23), 456x448x1280 12.8 / 13.9 (8); longer slices gain as modelled:
    // 592x1280x7296 NT 114.9 in 2, 99.9 in 6, 975x384x8064 67.5 in 4, 60.3 in 21
    int fitted = 1, uneven = 1;
    double fitted_t = INFINITY, uneven_t = INFINITY;
    for (int c = 2; c <= most; ++c)
      if (slices_ok(k, kt, c) && (kt % c == 0 || (k->dtype != FRISK_F32 && !named)) && (size_t)c * (size_t)d->M * (size_t)d->N * 4 <= workspace && (!table_range || in_table_range(k, d, c))) {
        const double t = small_grid_time(m, k, d, c);
        if (kt % c) {
          if (t < uneven_t) { uneven = c; uneven_t = t; }
          continue;
        }
        if (t < best_t) { best = c; best_t = t; }
        if (range_cost && t < range_t && in_table_range(k, d, c)) range_t = t;
        if (k->dtype == FRISK_F32 && in_table_range(k, d, c) && t < fitted_t) { fitted = c; fitted_t = t; }
      }
    // slices of unequal length for 10 % of modelled time and what the model leaves out, 0.15 us a slice and 1 us for a second launch where there was
    // none: us without / with them, fp16 96x768x6528 NN 11.1 in 6 slices, 11.8 in 13, e4m3 6x576x3712 8.8 in one, 9.9 in 6
    if (uneven_t + 0.15 * (uneven - best) + (best == 1 ? 1.0 : 0.0) < 0.9 * best_t) { best = uneven; best_t = uneven_t; }
    if (best > fitted && fitted > 1 && kt / best <= 10 && fitted_t < 1.12 * best_t) { best = fitted; best_t = fitted_t; }
  }
  // the edge kernels: slices of unequal length, whole tiles of partial sums
  if (const int most = edges ? edge_split_of(k, d, workspace) : 1; most > 1)
    for (int c = 2; c <= most; ++c)
      if (edge_slices_ok(k, d, c)) {
        const double t = small_grid_time(m, k, d, c);
        if (t < best_t) { best = c; best_t = t; }
      }
  if (cost) *cost = best_t;
  if (range_cost) *range_cost = range_t;
  return best;
}

// Beyond the range of the table (other splits than those of its sweep, kernels that the sweep did not hold) its times are off by a factor of each variant's
// own, and a split costs more by the slice than it knows, since the summing pass waits for its slices.  This is the time with both put right, for the choice
// between a route beyond the range and the best one within it; 16- and 8-bit types.  Over 64 rows whole x the table's in one pass, scale x the table's
// + split + slice x (slices - 1) in slices, fitted to 4600 problems of M and N from 128 and 512, K 1024 to 16384, operands in rotation (deviation of a variant's times 4 to 9 %, 5 to
// 14 without).
static double refined_time(const KernelEntry* k, const frisk_gemm_desc* d, int split) {
  struct Fit { float whole, scale, split, slice; };
  static const Fit fits[2][14] = {  // in the order of kSmallGrid
      {{1.02f, 1.0f, 0.0f, 0.0f}, {1.1f, 1.035f, -2.6f, 0.155f}, {1.0f, 1.0f, 0.0f, 0.0f}, {1.0f, 1.0f, 0.0f, 0.0f}, {1.0f, 1.15f, -3.7f, 0.04f}, {1.0f, 1.15f, -3.7f, 0.04f},  // 16-bit
       {1.0f, 1.0f, 0.0f, 0.0f}, {0.94f, 0.754f, 0.25f, 0.18f}, {0.94f, 0.754f, 0.25f, 0.18f}, {0.85f, 0.85f, 0.0f, 0.18f}, {0.85f, 0.85f, 0.0f, 0.18f},
       {0.92f, 0.897f, -2.54f, 0.199f}, {0.97f, 0.943f, -0.69f, 0.086f}, {1.02f, 1.061f, -2.07f, 0.188f}},
      {{1.17f, 1.0f, 0.0f, 0.0f}, {0.99f, 0.97f, -1.79f, 0.161f}, {1.0f, 1.0f, 0.0f, 0.0f}, {1.0f, 1.0f, 0.0f, 0.0f}, {1.0f, 1.0f, 0.0f, 0.1f}, {1.0f, 1.0f, 0.0f, 0.1f},  // 8-bit
       {1.0f, 1.0f, 0.0f, 0.0f}, {0.85f, 0.829f, -0.53f, 0.183f}, {0.85f, 0.829f, -0.53f, 0.183f}, {0.888f, 0.888f, 0.0f, 0.18f}, {0.888f, 0.888f, 0.0f, 0.18f},
       {0.95f, 0.924f, -1.89f, 0.189f}, {0.99f, 0.95f, 0.0f, 0.1f}, {1.01f, 1.0f, -1.17f, 0.153f}},
  };
  const int es = elem_size(k->dtype);
  double t = small_grid_time(small_grid_model(k), k, d, split);
  if (d->M > 64) {
    const Fit& f = fits[es == 1][small_grid_class(k)];
    return split > 1 ? f.scale * t + f.split + f.slice * (split - 1) : f.whole * t;
  }
  const int64_t wgs = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn) * split, kt = (d->K + k->bk - 1) / k->bk;
  if (es == 2 && k->bm == 64) {
    // fp16 62x4672x7424 NT 26.1 us on 64x32 tiles, 23.6 on 64x128 tiles in 4 slices; bf16 49x3648x5888 NN 18.1 on 32x128 tiles, 14.2 on 64x128 ones
    if (k->wk > 1 && d->K > 4096 && d->K * es % 16384) t *= 1.15;
    if (k->bn == 128 && !k->transB && split > 1 && split < 8) t *= 0.93;
  } else if (es == 1 && k->bm == 32) {
    // 32x32 tiles beyond one round, a K tile of 512, where K ends inside one of a few: int8 32x9216x2688 NT 9.1 us, on 32x128 tiles 8.1; 5x14528x2688
    // 9.6 / 8.8; but e4m3 7x13504x3712 12.0 / 14.2, 2x15808x3200 11.5 / 13.3
    if (k->bn == 32 && wgs > 256 && d->K % k->bk && kt <= 6) t *= 1.17;
  }
  return t;
}

// Edge kernels without a plain twin of the same tile: 192x256, and the tiles that stream B [N][K] for up to 64 rows, any number of rows
// and any K.  Before those, rows off a multiple of 32 and K off 4 K tiles ran on 32x128 and 64x128 tiles, which fetch 128 bytes of a row of B
// at a time, split along K.  us before / now, B from HBM: 17x8192x8192 fp16 45.9 / 24.6, int8 21.1 / 14.2, e4m3 20.5 / 13.8;
// 48x8192x8192 37.4 / 29.5, 19.8 / 18.2, 19.4 / 17.7; 5x14336x4096 (448 tiles, ring of 2) 30.6 / 20.7, 18.5 / 13.0, 18.0 / 12.7; 24x16384x4224
// (K a half K tile over) 33.6 / 27.8, 19.6 / 17.0, 19.1 / 16.9; 33x4096x2048 15.5 / 7.1, 7.2 / 6.8, 6.6 / 5.2; 40x11008x4096 fp16 28.5 / 28.7
static bool planners_own(const KernelEntry* k) { return k->edge && !k->splitk && (k->bm == 192 || k->wk > 1); }

// What rounds of large tiles take, in microseconds: start + whole rounds of `cap` work-groups x (round + K tiles x tk) + a last one at round + K tiles x
// tk x (part + (1 - part) x fill).  `round` is what a round costs beside its K loop (first transfers, stores): 3 us for two 128x128 tiles a CU, 9 for
// a 256x256 one, which is why the larger tiles need a deep K.  Fitted to 1100 problems of 257 to 2200 tiles of 128x128, K 256 to 8192, operands in
// rotation (standard deviation 3 to 8 %).
struct RoundModel { int cap; float start, round, tk, part; };
static const RoundModel* round_model(const KernelEntry* k) {
  static const RoundModel edge[2][3] = {{{512, 2.8f, 2.8f, 0.95f, 0.38f}, {256, 0.8f, 7.3f, 1.00f, 0.64f}, {256, 1.1f, 8.7f, 1.33f, 0.61f}},    // 16-bit: 128x128, 192x256, 256x256
                                        {{512, 3.1f, 3.25f, 1.00f, 0.46f}, {256, 1.5f, 9.0f, 1.00f, 0.63f}, {256, 1.7f, 11.6f, 1.31f, 0.59f}}};  // 8-bit
  static const RoundModel plain[2][3] = {{{512, 1.3f, 2.3f, 1.02f, 0.33f}, {256, 1.8f, 1.7f, 0.53f, 0.60f}, {256, 2.2f, 2.6f, 0.91f, 0.56f}},   // 128x128 in rings of 2 and 3, 256x128 and 128x256
                                         {{512, 1.7f, 1.1f, 1.04f, 0.46f}, {256, 1.8f, 1.7f, 0.53f, 0.62f}, {256, 2.4f, 2.4f, 0.85f, 0.50f}}};
  const int es = elem_size(k->dtype), area = k->bm * k->bn;
  if (es == 4 || k->bm < 128 || k->bn < 128 || k->wk > 1 || k->wm * k->wn != 4) return nullptr;
  if (k->edge && !k->splitk) return &edge[es == 1][area == 128 * 128 ? 0 : k->bm == 192 ? 1 : 2];
  if (k->edge || k->guard || area == 256 * 256) return nullptr;
  return &plain[es == 1][area == 128 * 128 ? (k->stages >= 3 ? 1 : 0) : 2];
}
// The same for the tiles that only `other_tile` takes, and for 256x256 in whole tiles.
static const RoundModel* tile_model(const KernelEntry* k) {
  static const RoundModel more[2][3] = {{{256, 1.0f, 6.0f, 0.875f, 0.66f}, {256, 1.0f, 8.0f, 1.165f, 0.62f}, {256, 1.1f, 8.2f, 1.33f, 0.61f}},    // 16-bit: 160x256, 224x256, 256x256
                                        {{256, 1.5f, 7.5f, 0.875f, 0.66f}, {256, 1.6f, 10.3f, 1.15f, 0.61f}, {256, 1.7f, 11.1f, 1.31f, 0.59f}}};  // 8-bit
  const int es = elem_size(k->dtype);
  if (es == 4 || k->wm * k->wn * k->wk != 4 || k->bn != 256) return round_model(k);
  if (k->edge && (k->bm == 160 || k->bm == 224)) return &more[es == 1][k->bm == 224];
  return !k->edge && !k->guard && k->bm == 256 ? &more[es == 1][2] : round_model(k);
}
// `slices` > 1: every tile (up to half a round of them) or those behind the whole rounds split along K, and the pass that sums them
static double round_time(RoundModel m, const KernelEntry* k, const frisk_gemm_desc* d, int slices) {
  const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn), kt = (d->K + k->bk - 1) / k->bk;
  const int64_t split = slices <= 1 ? 0 : tiles <= 128 ? tiles : tiles % 256, plain = tiles - split, full = plain / m.cap, last = plain % m.cap + split * slices;
  const double k_last = split ? (double)((kt + slices - 1) / slices) : (double)kt;
  double t = m.start + (double)full * (m.round + (double)kt * m.tk);
  if (last) t += m.round + k_last * m.tk * (m.part + (1.0 - m.part) * (double)last / m.cap);
  if (split) t += 3.5 + 0.25 * (double)(split * slices) * k->bm * k->bn * 4.0 / 1e6;
  return t;
}

// What a launch knows beyond the descriptor: pointers off 16-byte boundaries (C: or a column-scale pointer off its vector), and
// how much workspace there is to use.
struct PlanContext { bool a_off = false, b_off = false, c_off = false; size_t workspace = kAnyWorkspace; };
// Operands that are copied to aligned rows in the workspace before the product runs, and where they go.
struct Repack { bool a = false, b = false; int64_t lda = 0, ldb = 0; size_t b_offset = 0, bytes = 0; };
// What a launch needs of a plan beyond the public structure: the copies, and the tail split of an edge kernel (whose slices may
// differ in length), its partial sums behind the copies in the workspace.
struct LaunchExtras { Repack repack; int tail_split = 1, tail_tiles = 0; size_t partial_offset = 0; };

static Repack repack_of(const frisk_gemm_desc* d, bool a, bool b) {
  Repack r;
  const int es = elem_size(d->dtype_ab), per16 = 16 / es;
  r.a = a; r.b = b;
  const int64_t a_rows = d->transA ? d->K : d->M, a_cols = d->transA ? d->M : d->K, b_rows = d->transB ? d->N : d->K, b_cols = d->transB ? d->K : d->N;
  r.lda = (a_cols + per16 - 1) / per16 * per16;
  r.ldb = (b_cols + per16 - 1) / per16 * per16;
  if (a) r.b_offset = ((size_t)a_rows * (size_t)r.lda * es + 255) & ~(size_t)255;
  r.bytes = r.b_offset + (b ? (size_t)b_rows * (size_t)r.ldb * es : 0);
  return r;
}

// The 128x128 edge tile with 3 + 3 tiles of LDS, which takes over the launch of the one with 2 + 2 as it is, slices included.
static bool same_edge_tile(const KernelEntry* k) { return k->bm == 128 && k->bn == 128 && k->edge && k->stages == 3; }

// The kernel (its index) that runs a problem in place of `k`, which the search has found with `split` slices of K or `slices` of its edge tiles: -1, that
// one stays.  Where every CU has one work-group at most, the bytes that it fetches, (rows + columns) x K, are a first measure of the time: fp16 tiles of one round reach, in bytes a
// nanosecond and CU from the last-level cache / from memory, 85 / 55 (64x64 NT), 74 / 46 (NN), 80 / 53 (64x128 NT), 67 / 61 (128x128 in a ring of 3) and 51 / 49 (256x256, bound by its
// MFMAs).  No more than that: where each rule below ends is the edge of a sweep over drawn problems, timed on both sides, not a consequence of these rates.
static int follow_up(const std::vector<Variant>& list, const KernelEntry* k, const frisk_gemm_desc* d, bool rows_aligned, int split, int slices, const Repack& packed) {
  const int es = elem_size(k->dtype);
  const bool staged = k->guard && !k->edge;  // through registers
  if (staged || (split > 1 && k->dtype == FRISK_F32)) return -1;
  auto tiles_of = [&](int bm, int bn) { return ((d->M + bm - 1) / bm) * ((d->N + bn - 1) / bn); };
  // the variant of a tile for this problem: the plain kernel where it fits, else the edge kernel, named for what it takes (an incumbent that
  // works on copies of its operands hands them on)
  auto variant = [&](int bm, int bn, int stages) {
    const KernelEntry *plain = nullptr, *edge[3] = {};
    int id = -1, edge_id[3] = {-1, -1, -1};
    for (const Variant& v : list)
      if ((v.follow_up || (bm == 128 && !v.k->edge && !v.k->guard && !v.k->splitk)) && v.k->bm == bm && v.k->bn == bn && v.k->stages == stages) {
        if (v.k->edge) { edge[v.k->guard] = v.k; edge_id[v.k->guard] = v.id; }
        else { plain = v.k; id = v.id; }
      }
    const KernelEntry* x = edge[0] ? edge[0] : plain;
    if (!x) return -1;
    const double span_a = (double)(packed.a ? packed.lda : d->lda) * es * (d->transA ? x->bk : x->bm), span_b = (double)(packed.b ? packed.ldb : d->ldb) * es * (d->transB ? x->bn : x->bk);
    if (span_a >= 4294967296.0 || span_b >= 4294967296.0) return -1;
    const bool whole_k = d->K % x->bk == 0;
    if (rows_aligned && whole_k && d->M % bm == 0 && d->N % bn == 0) return id;
    if (!edge[0]) return -1;
    return rows_aligned && whole_k ? edge_id[0] : rows_aligned && d->K % (16 / es) == 0 ? edge_id[1] : k->guard == 2 ? edge_id[2] : -1;
  };
  if (k->dtype == FRISK_F32) {
    // 32x32 tiles, the four waves splitting K, on up to 512 work-groups (two a CU): a 64x64 tile keeps its CU's matrix pipe busy and a quarter of
    // as many leave most CUs without one.  us, operands in the last-level cache and no workspace (with one these are split along K), on 64x64 or 32x128 tiles / so: 128x1280x1024 NN 18.9 / 9.1,
    // 896x256x1792 30.8 / 14.1, 128x384x896 16.3 / 7.6, 256x2048x1408 (512) 24.9 / 17.8; off the tiles 323x130x437 NT 13.8 / 10.0, 8-row problems of 4000 to
    // 9000 columns half the time; but 512x1152x512 (576) 11.2 / 12.4, 1280x640x768 (800) 16.2 / 19.7, and in a second round on fewer than two K
    // tiles of 128 296x856x160 (270) 6.2 / 7.2; whole tiles under A [K][M] 256x256x512 TN 10.5 / 6.0, 512x512x512 TT 11.4 / 6.7, 1024x512x256 7.6 / 6.6
    return k->wk == 1 && d->K >= (tiles_of(32, 32) <= 256 ? 128 : 256) && tiles_of(32, 32) <= 512 ? variant(32, 32, 2) : -1;
  }
  const int64_t k_bytes = d->K * es;
  if (d->M <= 64) {
    // 64x64 tiles for up to 64 rows where they are one round that fills half the CUs and more, with 256 bytes of a row of B at a time and three tiles under way on
    // each.  In place of unsplit 32x128 and 64x128 tiles; of 32x128 ones in 2 slices on B [K][N], for the second launch that goes; and below 32 rows on B [N][K] of
    // two 32x32 work-groups a CU (16-bit from 9 rows on and not where rows of B are a multiple of 4 KiB apart, 8-bit up to 6000 of K: elsewhere as many are slower).  us, B from memory, before / so: bf16 5x11584x2304
    // NN 17.9 / 12.3, 58x9536x3584 NN 22.1 / 15.9, 12x15296x6400 NN 41 / 32, fp16 13x10432x3456 NT 19.5 / 17.4, e4m3 1x9856x2944 NT 12.2 / 9.6; but fp16
    // 6x14016x7808 NT 40.0 / 45, 24x15552x8192 NT (rows 16 KiB apart) 35 / 44, bf16 19x15424x4096 NT (8 KiB) 20 % slower, 21x12736x6144 (12 KiB) 12 %, 10752x6144 NN in 3 slices 29.7 / 37.  Of 280 drawn problems 93 change over,
    // 13 % faster, none of them slower by 3 % and more.
    const int64_t wgs = tiles_of(64, 64);
    if (wgs <= 128 || wgs > 256 || (d->transB && d->M >= 32) || k_bytes < 2048) return -1;  // (measured from 2 KiB of K on)
    const bool two_a_cu = k->bm == 32 && k->bn == 32 && k->stages == 2;
    const bool so = k->bn == 128 ? split == 1 || (split == 2 && !d->transB && k->bm == 32 && wgs > 170)
                                 : two_a_cu && split == 1 && (es == 2 ? d->M > 8 && d->ldb * es % 4096 : d->K < 6000 && d->K % 4096);
    return so ? variant(64, 64, 3) : -1;
  }
  const bool edge128 = k->edge && !k->splitk && k->bm == 128 && k->bn == 128;
  // 64x64 tiles in a single round, in place of 128x128 edge tiles, split or not, and of unsplit 64x128 tiles.  us, operands in the last-level cache:
  // fp16 525x1136x1480 NT 19.1 / 9.6, 558x296x1200 16.1 / 7.1, 852x824x1840 NN 19.8 / 11.8, 1229x608x3960 22.9 / 18.7, 768x1152x2048 12.0 / 9.3,
  // e4m3 1408x576x2208 NT 18.7 / 8.2; in place of 64x128 tiles not for less than 1 KiB of K, 906x312x320 NT 5.0 / 5.2; with more than 7.5 KiB the slices have caught up, B [K][N] more than 7: from
  // memory 239x183x3823 NN 21.3 in 8 slices / 25.1, 107x688x3480 19.8 / 22.7 (6 to 7 KiB 4 % faster, and NT 9 %)
  // ... and of 64x128 tiles whatever the K where they are unsplit, and where they are split into 2 slices (B [K][N]: up to 12 KiB of K) or 16-bit ones into
  // 3 (up to 7 KiB), for the second launch that goes: fp16 832x1216x6144 NN 29.6 / 22.2, 1088x832x4864 NT 19.5 / 17.7, 876x1088x5120 NN 22.0 / 19.7; in 2 slices
  // 928x896x4480 NT 23 % faster, e4m3 332x1920x6656 NT 16 %; but fp16 68x6656x8576 NN in 2 slices 17 % slower, 416x1408x8064 NN in 3 12 %.  Of 120 drawn problems
  // 67 change over, 13 % faster, one of them slower, by 3 %.
  const bool tall = k->bm == 64 && k->bn == 128;
  const bool sliced = tiles_of(64, 64) > 128 && (split == 2 ? d->transB || k_bytes <= 12288 : split == 3 && es == 2 && k_bytes <= 7168);
  if (tiles_of(64, 64) < 256 && ((edge128 && k_bytes <= (d->transB ? 7680 : 7168)) || (tall && (split == 1 ? k_bytes >= 1024 : sliced))))
    if (const int id = variant(64, 64, 3); id >= 0) return id;
  if (split > 1) return -1;
  // 128x128 tiles with 3 + 3 tiles of LDS in a single round, one on each CU, in place of unsplit 64x128 ones of which some CUs hold two: a third less to transfer.  us
  // on 64x128 / so: fp16 363x8512x2176 NT 25.2 / 20.8, 1206x3072x1280 NN 17.6 / 15.9, bf16 1108x3008x1792 NT 20.2 / 18.1, 5952x640x7296 NN 82.5 / 73.1.  Of 79 drawn 16-bit
  // problems all are faster, by 18 %, and all of 48 8-bit ones of 2 KiB of K and more, by 20 % (of 37 with less 14 are slower, int8 1856x1152x1024 NT by 17 %).  Of 243 more,
  // from memory, 11 are slower, by 3 to 7 % (bf16 2752x1024x896 NT 11.5 / 12.4)
  if (k->bm == 64 && k->bn == 128 && (es == 2 || k_bytes >= 2048) && tiles_of(64, 128) > 256 && tiles_of(128, 128) <= 256)
    if (const int id = variant(128, 128, 3); id >= 0) return id;
  // 128x128 edge tiles with 3 + 3 tiles of LDS where no CU has two work-groups.  us with 2 + 2 / 3 + 3: fp16 3916x632x2592 NT 32.4 / 24.4, 512x1392x1368 TN
  // 18.3 / 13.5, 558x296x1200 16.1 / 12.2, e4m3 2304x1664x4048 NN 28.1 / 21.9; under 12 K tiles the longer prologue costs up to 4 %
  if (edge128 && tiles_of(128, 128) * (tiles_of(128, 128) <= 128 ? slices : 1) <= 256 && (d->K + k->bk - 1) / k->bk >= 12 && !(tiles_of(128, 128) > 128 && slices > 1))
    return variant(128, 128, 3);
  return -1;
}

// 256x256 edge tiles in slices of K (their index), for 16- and 8-bit problems of a quarter of a round to two of 128x128 tiles whose K is deep and whose tiles are not split otherwise; -1 elsewhere.
// Up to 256 tiles of 128x128, on those, one a CU, or on 64x128 tiles: such a CU takes 192 or 256 rows and columns a K tile, 0.5 us at the 60 to 70 bytes a nanosecond that it
// pulls from the last-level cache, however many others are idle; a 256x256 tile takes half of that for the same work, and its slices fill the grid.  They cost 40 to 66 MB of
// partial sums: the pass that adds them takes 9 to 13 us, and with the writing and what a slice pays beside its K tiles a call spends 25 to 30 us that do not grow with K (19 of 144 work-groups).
// Beyond 256 of them, on edge tiles in one pass, which are a round that is not full or two: 2 or 3 slices of up to 112 tiles (above, where smaller tiles nearly fill their
// round, 7 % on average are left).  us before / so, from memory: bf16 2043x1144x9024 NN 90.6 / 58.9, fp16 2114x1152x10752 NT 95.6 / 69.7, 1777x1024x13376 NT (64x128) 90.4 / 60.5, 1137x2880x11968 NT (4
// slices) 110.7 / 87.3, bf16 454x4951x16128 NT 137.2 / 81.2, e4m3 1883x720x17920 NN 77.4 / 43.2, fp16 1019x5408x6912 NT 117.3 / 84.9, bf16 995x5616x8192 NN 140.4 / 98.5, 1012x4640x5248 NT (3) 86.3 / 60.2,
// int8 1921x2848x12800 NN 109.3 / 85.4.
// Problems whose M and N are multiples of 256 are not here: they have split-K kernels of their own (2048x1280x8192 runs in 4 slices).
// Error against 64 bits, fp32 C of fp16 1137x2880x11968: 6.9e-7 in one chain, 3.5e-7 in four.
//
// The least K of 16- and 8-bit types: where operands from memory, or the weights alone, gain (0.92 to 1.00 in a few of 300 measured at a line: fp16 2043x1144x7488 NN with the weights alone 46.7 / 50.9).  With both operands in the last-level cache, as in a
// call repeated on the same buffers, a product at its line runs at 0.82 to 1.35 times its former speed, at 1.3 times that K at 0.92 to 1.42.  At the lines (and beyond), all from memory / the weights alone / all
// from the cache, three to seven shapes in two layouts:
struct DeepLine { int64_t k16, k8, k8_nk; };  // k8_nk: of 8-bit types against B [N][K]
static constexpr DeepLine kDeepLines[] = {
    {7488, 14592, 14592},   // five slices and more in place of 128x128 tiles: 16-bit 1.16 to 1.31, cache 0.93 to 1.09, then 0.98 to 1.15; 8-bit 1.17 to 1.38, cache 0.87 to 1.08, 0.94 to 1.13
    {8192, 16384, 18432},   // four: 16-bit 1.01 to 1.20 / 0.98 to 1.12 / 0.89 to 1.04, at 9472 1.07 to 1.29 / 1.06 to 1.21 / 0.94 to 1.09; 8-bit NN 1.23 to 1.35 / 1.21 to 1.28 / 0.94 to 1.09; e4m3 NT at 16384
                            // 0.97 to 1.08 / 0.96 to 1.03 / 0.84 to 0.89 (944x3472 62.5 us before, 65.1 so), at 18432 1.07 to 1.20 / 1.08 to 1.18 / 0.87 to 0.92
    {10496, 16512, 16512},  // four and more in place of 64x128 tiles, two of which on a CU hide more: 16-bit 1.20 to 1.62 / 1.18 to 1.29 / 0.92 to 1.24; 8-bit 1.10 to 1.67 / 0.97 to 1.50 / 0.82 to 1.35
    {4352, 8576, 8576},     // three beyond 256 tiles: 16-bit 1.03 to 1.32 / 1.03 to 1.11 / 0.92 to 0.98, at 4992 1.12 to 1.38 / 1.12 to 1.15 / 1.00 to 1.02; 8-bit 1.09 to 1.38, cache 0.92 to 1.11
    {6144, 12032, 12032},   // two: 16-bit 1.02 to 1.35, cache 0.98 to 1.05; 8-bit 1.05 to 1.44, cache 0.93 to 1.17
};
static int deep_tile(const std::vector<Variant>& list, const KernelEntry* k, const frisk_gemm_desc* d, bool rows_aligned, size_t workspace) {
  const int64_t tiles = ((d->M + 127) / 128) * ((d->N + 127) / 128);
  const int64_t tiles256 = ((d->M + 255) / 256) * ((d->N + 255) / 256);
  const int es = elem_size(k->dtype);
  if (es == 4 || k->guard || !rows_aligned || k->wk > 1 || tiles < 64 || tiles > 512 || d->M <= 256 || d->N <= 256) return -1;
  if (tiles > 256 ? !k->edge || k->splitk || tiles256 > 112 : k->bn != 128 || k->stages != 3) return -1;
  auto deep = [&](int slices) {
    if (slices < (tiles > 256 ? 2 : 4)) return false;
    const DeepLine& line = kDeepLines[tiles > 256 ? (slices == 2 ? 4 : 3) : k->bm == 64 ? 2 : slices == 4 ? 1 : 0];
    return d->K >= (es == 2 ? line.k16 : d->transB ? line.k8_nk : line.k8);
  };
  for (const Variant& v : list) {
    const KernelEntry* x = v.k;
    if (!x->edge || x->guard || x->splitk || x->bm != 256 || x->bn != 256 || (d->M % 256 == 0 && d->N % 256 == 0) || d->K % x->bk) continue;
    if ((double)d->lda * es * (d->transA ? x->bk : x->bm) >= 4294967296.0 || (double)d->ldb * es * (d->transB ? x->bn : x->bk) >= 4294967296.0) continue;
    if (deep(edge_split_of(x, d, workspace))) return v.id;
  }
  return -1;
}

// The edge tile (its index) that takes a problem of more than 256 tiles of 128x128 over from `k`, which the search has found and
// which runs it in one pass: the one whose rounds the model sees through 3 % sooner, -1 where there is none.  The search's costs know nothing of what a round pays beside
// its K loop, nor of bytes of C: a 256x256 tile of 4-byte C with old values is 512 KiB, 19 us of a round whatever the K.  us before / now, operands
// from memory: fp16 1596x3540x778 NN 24.4 on 192x256 / 18.8 on 128x128, 6656x1664x361 TN into fp32 sums 34.8 on 256x256 / 26.6 on 128x128; 3325x2420x2483 NT 56.6 on
// 128x128 / 49.1 on 160x256, 2368x5376x5376 NT 111.6 on 256x256 / 105.1 on 224x256.  Of 600 problems drawn
// over the four types 150 or so change over, 15 % faster, one of them slower (int8 4288x7424x640 NT, 38.1 / 39.7).  The 160- and 224-row tiles from 12 K tiles on (their longer
// prologue; with fewer the smaller tiles are as good).
// Where the 128x128 tiles are one round, two a CU, which hides a wait for memory that one 160x256 tile cannot, what is gained hangs on where the operands come from: of 99 drawn 16-bit
// problems 160x256 tiles are 10 % faster with both in the last-level cache (2156x3328x6528 NN 102.2 / 89.9), 5 % with A there and B from memory (101.2 / 94.8) and 3 % slower, NN 6 %, with both from
// memory (101.1 / 108.2).  int8, of 87, 3, 2 and -6 % (960x6144x4096
// NT 29.4 / 31.0, 34.4 / 34.8, 35.7 / 39.3) and e4m3, on 192x256 tiles 5 to 11 % slower wherever they come from, stay on 128x128.
static int other_tile(const std::vector<Variant>& list, const KernelEntry* k, const frisk_gemm_desc* d, bool rows_aligned, const Repack& packed) {
  const int es = elem_size(k->dtype), os = elem_size(d->dtype_out);
  const bool whole_k = d->K % k->bk == 0;
  const double more_bytes = os - 2 + (d->clear_accum ? 0 : os);  // of C, by the element, beyond those of the models' fits
  auto time = [&](const KernelEntry* x, const RoundModel* m) {
    RoundModel with_c = *m;
    with_c.round += (float)(more_bytes * (m->cap == 512 ? 0.92 : 3.2 * x->bm * x->bn / 65536.0));
    return round_time(with_c, x, d, 1);
  };
  const RoundModel* now = k->guard && !k->edge ? nullptr : tile_model(k);
  if (!now || d->K <= k->bk) return -1;  // (a single K tile has no loop to model)
  const bool two_a_cu = now->cap == 512 && ((d->M + 127) / 128) * ((d->N + 127) / 128) <= 512;  // a single round of 128x128 tiles
  double best_time = 0.97 * time(k, now);
  int best = -1;
  for (const Variant& v : list) {
    const KernelEntry* x = v.k;
    const RoundModel* m = x != k && x->edge && !x->splitk && x->stages == 2 ? tile_model(x) : nullptr;
    if (!m || x->guard != (rows_aligned && whole_k ? 0 : rows_aligned && d->K % (16 / es) == 0 ? 1 : 2) || (x->guard == 2 && k->guard != 2)) continue;
    if ((x->bm == 128 || x->bm == 256) && x->guard == 0 && d->M % x->bm == 0 && d->N % x->bn == 0) continue;  // the plain twin was there to be found
    if (es == 1 && two_a_cu && x->bm != 128) continue;
    if ((x->bm == 160 || x->bm == 224) && (d->K + x->bk - 1) / x->bk < 12) continue;
    if ((d->K + x->bk - 1) / x->bk < x->min_k_tiles) continue;
    const double span_a = (double)(packed.a ? packed.lda : d->lda) * es * (d->transA ? x->bk : x->bm), span_b = (double)(packed.b ? packed.ldb : d->ldb) * es * (d->transB ? x->bn : x->bk);
    if (span_a >= 4294967296.0 || span_b >= 4294967296.0) continue;
    if (const double t = time(x, m); t < best_time) { best = v.id; best_time = t; }
  }
  return best;
}

static int make_plan(const frisk_gemm_desc* d, frisk_gemm_plan* plan, bool with_model, const PlanContext& ctx = {}, LaunchExtras* extras = nullptr) {
  const bool no_split = ctx.workspace == 0;
  int st = validate(d);
  if (st != FRISK_OK) return st;
  if (!plan) return fail(FRISK_ERR_NULL, "plan is null");
  std::memset(plan, 0, sizeof *plan);
  if (extras) *extras = LaunchExtras{};  // (a call that plans once more for the workspace it has hands in those of its first plan)
  plan->kernel_id = -1;
  const int es = elem_size(d->dtype_ab), os = elem_size(d->dtype_out);
  plan->flops = 2.0 * (double)d->M * (double)d->N * (double)d->K;
  plan->bytes = (double)d->M * d->K * es + (double)d->K * d->N * es + (double)d->M * d->N * os;
  if (d->epilogue == FRISK_EPI_ROW_COL_SCALE) plan->bytes += 4.0 * ((double)d->M + (double)d->N);
  if (d->epilogue == FRISK_EPI_TENSOR_SCALE) plan->bytes += 8.0;
  plan->split_k = 1;

  const bool a_aligned = (d->lda * es) % 16 == 0 && !ctx.a_off, b_aligned = (d->ldb * es) % 16 == 0 && !ctx.b_off;
  const bool rows_aligned = a_aligned && b_aligned && (d->ldc * os) % 16 == 0 && !ctx.c_off;
  // what it would take to put the operands' rows on 16-byte boundaries, in bytes and in microseconds: a dependent launch, and every
  // byte read and written once
  const Repack packed = repack_of(d, !a_aligned, !b_aligned);
  const double repack_cost = packed.bytes ? 4.0 + (double)packed.bytes / 2.2e6 : 0.0;
  const auto& ks = kernels();
  const auto& list = variants(d->dtype_ab, d->transA != 0, d->transB != 0);
  int best = -1;
  double best_cost = 0.0;
  const bool tile_requested = d->tile_m || d->tile_n || d->tile_k || d->waves_m || d->waves_n || d->stages || d->atom;
  // The kernels staged through registers take any rows in one launch, 1.4 us per K tile of 128 bytes behind those that work on copies (TT 1.25, 8-bit 2.2, fp32 0.7), so
  // with few K tiles the launch that makes the copies costs more than it saves.  us staged / on copies: fp32 28x24x26 NN 4.8 / 7.5, 69x16x17 4.9 / 7.2,
  // 78x18x35 TN 5.9 / 7.0, bf16 16x25x21 NT 6.9 / 7.6; but int8 24x884x344 TN 10.6 / 8.4,
  // fp32 123x9x168 NN 9.7 / 7.7
  const int64_t k_tiles = ((int64_t)d->K * es + 127) / 128, tiles128 = ((d->M + 127) / 128) * ((d->N + 127) / 128), tiles64 = ((d->M + 63) / 64) * ((d->N + 63) / 64);
  const double staged_rounds = std::max(1.0, (double)tiles128 / 512.0);
  // Two more cases of grids of at most 256 tiles of 128x128.  8-bit problems of two K tiles (all layouts but TN, where A comes in rows of M and B in rows of N and both are turned on the way to
  // LDS; us staged / on copies: int8 76x529x162 NN 9.3 / 10.7, e4m3 158x1761x133 NN 9.4 / 10.7, 73x294x179 TT 9.3 / 10.4, NN 6 % and TT 9 % on average, TN 6 % faster on copies; three K
  // tiles NN 9.3 / 8.5).  Operands stored along K, which staging through registers costs least, beyond the 64x64 tiles and short of the ring of 3 that `follow_up` has for copies: 4
  // to 11 K tiles 5 % on average, e4m3 525x3807x542 13.2 / 14.5, int8 1482x2240x730 14.1 / 15.9, bf16 943x2739x586 17.4 / 18.8; with 12 and more, or in 64x64 tiles, copies gain 4 to 50 %.
  const bool staged_ahead = es < 4 && tiles128 <= 256 && (!d->transA && d->transB ? k_tiles < 12 && tiles64 >= 256 : es == 1 && k_tiles <= 2 && !(d->transA && !d->transB));
  const bool copies_lose = packed.bytes && !tile_requested && d->policy == FRISK_POLICY_SQUARE &&
                           (staged_ahead || staged_rounds * (double)k_tiles * (es == 4 ? 0.72 : es == 1 ? 2.2 : d->transA && d->transB ? 1.25 : 1.4) < 3.5 + (double)packed.bytes / 2.2e6);
  bool policy_excluded = false;
  const bool any_layout = !list.empty();
  const bool small = small_grid(d);
  bool split_edges = false, settled = false;  // settled: without the 192x256 tile and without splits of edge tiles
  // small grids: the best of the kernels and splits that their table was fitted over, found beside the best of all
  const bool want_range = small && es < 4 && rows_aligned && !tile_requested && d->split_k <= 1;
  int best_in = -1;
  double best_in_cost = 0.0;
  bool table_range = false;  // that one is taken
  // what the partial sums of a kernel may take of the workspace: all of it, or what lies behind the copies it works on
  auto left_for_sums = [&](const KernelEntry* k) {
    const size_t copies = k->guard == 2 && packed.bytes ? (packed.bytes + 255) & ~(size_t)255 : 0;
    return ctx.workspace == kAnyWorkspace ? kAnyWorkspace : ctx.workspace > copies ? ctx.workspace - copies : 0;
  };
  auto search = [&](bool want_split) {
    for (const Variant& v : list) {
      const KernelEntry* k = v.k;
      if (v.follow_up) continue;
      if (d->tile_m && d->tile_m != k->bm) continue;
      if (d->tile_n && d->tile_n != k->bn) continue;
      if (d->tile_k && d->tile_k != k->bk) continue;
      if (d->waves_m && d->waves_m != k->wm) continue;
      if (d->waves_n && d->waves_n != k->wn) continue;
      if (d->stages && d->stages != k->stages_b) continue;  // the deeper ring names the variant
      if (d->atom && d->atom != k->atom) continue;
      // frisk.gemm's wave policy (FriskOps.td:248-289) decides the wave grid unless the descriptor names one: only variants
      // whose compiled grid is what computeWarpPartition gives for their tile and wave count under that policy qualify
      if (!d->waves_m && !d->waves_n && !v.policy[d->policy]) { policy_excluded = true; continue; }
      if (want_split && !k->splitk) continue;
      // a kernel whose loop needs a minimum of K tiles: per slice when the descriptor asks for a split
      if (k->min_k_tiles > 1 && (d->K + k->bk - 1) / k->bk / (want_split && d->split_k > 1 ? d->split_k : 1) < k->min_k_tiles) continue;
      // the fast kernels need whole tiles and rows that start on 16-byte boundaries; their edge variants take any M and N (and
      // are left out where the plain twin fits)
      const bool whole_mn = d->M % k->bm == 0 && d->N % k->bn == 0;
      if (!k->guard && (!rows_aligned || d->K % k->bk || (k->edge ? whole_mn : !whole_mn))) continue;
      // the 192x256 tile and the unsplit tiles that stream B (edge kernels without a plain twin) are the planner's own: a tile, wave grid,
      // ring or atom that is asked for names the other variants
      // (whole 256x256 tiles keep the default kernel: which one the square sizes run on is part of the planner's interface.  That costs time where they
      // leave CUs idle -- fp16 3072x3072x4096 NN, 144 of them, 70.6 us, 62.4 on 192x256 tiles -- and holds for every multiple of 256)
      const bool whole_256 = rows_aligned && d->M % 256 == 0 && d->N % 256 == 0 && d->K % k->bk == 0;
      if (planners_own(k) && (tile_requested || d->split_k > 1 || (k->bm == 192 ? small || whole_256 || settled : d->M > 64))) continue;
      // the edge kernels once more under their guarded names: K off the K tile (a whole number of chunks), and anything at all,
      // with A and B copied to aligned rows where theirs are not
      if (k->guard == 1 && k->edge && (!rows_aligned || d->K % (16 / es))) continue;
      if (k->guard == 2 && packed.bytes && (packed.bytes > ctx.workspace || d->split_k != 0 || copies_lose)) continue;
      // ... and address a tile's chunks by 32-bit lane offsets from its first row: the stored rows of one tile must span
      // less than 4 GiB
      const double span_a = (double)(packed.a ? packed.lda : d->lda) * es * (d->transA ? k->bk : k->bm),
                   span_b = (double)(packed.b ? packed.ldb : d->ldb) * es * (d->transB ? k->bn : k->bk);
      if ((!k->guard || k->edge) && (span_a >= 4294967296.0 || span_b >= 4294967296.0)) continue;
      // never a guarded kernel when a fast one fits -- except those, which run at their full rate whatever their name
      if (k->guard && !planners_own(k) && best >= 0 && !ks[best]->guard) continue;
      const size_t left = left_for_sums(k);
      double cost = 0.0, range_cost = 0.0;
      if (small && !want_split) small_grid_split(k, d, left, split_edges, false, &cost, want_range ? &range_cost : nullptr);
      else cost = estimated_cost(k, d, !want_split && left > 0 && d->split_k == 0, !settled, left);
      // (a 32-row edge tile above 64 rows streams B once per 32 rows where the 64-row tile wastes at most as much: 130x11008x4096
      // NT 64.5 against 53.5 us)
      if (k->edge && k->bm == 32 && d->M > 64 && !d->tile_m) continue;
      if (k->edge || k->guard) {
        // (the kernels staged through registers too: one row on a 128-row tile is not a 128th of its price)
        // the models see whole tiles; rows and columns beyond M and N are work all the same (a 64-row tile on 32 rows is no
        // better than the 32-row tile that fits): the square root of the covered area over M x N, as a penalty
        const double covered = (double)((d->M + k->bm - 1) / k->bm * k->bm) * (double)((d->N + k->bn - 1) / k->bn * k->bn);
        const double waste = std::sqrt(covered / ((double)d->M * (double)d->N));
        cost *= waste;
        range_cost *= waste;
      }
      if (k->guard == 2) cost += repack_cost;
      // What staging through registers costs beyond the model of its tile, a K tile of 128 bytes: on small grids 0.3 us where both operands are stored along K,
      // else 1.0 (8-bit 0.75); on larger ones, whose CUs hold two, 0.55, 1.0, 1.2 (int8) and 1.9 (8-bit float).  Fitted to 330 and 75 problems.  (As a factor of
      // 1.6 alone it kept problems of many K tiles from the copies.  Of 400 drawn problems with rows off 16 bytes 248 change over, 25 % faster.  The few that were slower, by
      // 3 to 25 %, `staged_ahead` leaves as they were.  us staged / on copies: e4m3 2410x865x1222 TN 24.8 / 18.1, 2511x2241x536 TT 26.7 / 17.2, fp16 1524x1901x861 NN 29.7 / 21.3,
      // 6720x832x1337 NN 44.0 / 30.8, bf16 2321x2172x1978 NT 50.7 / 38.4; but int8 445x2933x150 NN 10.3 / 11.6, 464x2236x198 NT 8.8 / 11.7, which stay staged)
      if (k->guard == 1 && !k->edge && es < 4) {
        const bool along_k = !d->transA && d->transB;
        const double rate = along_k ? (small ? 0.32 : 0.55) : es == 2 ? 1.0 : small ? 0.75 : k->dtype == FRISK_I8 ? 1.2 : 1.9;
        cost += staged_rounds * (double)k_tiles * rate;
      }
      // ties: the first listed variant is the tuned default
      if (best < 0 || (ks[best]->guard && !k->guard && !planners_own(ks[best])) || cost < best_cost) { best = v.id; best_cost = cost; }
      if (want_range && !k->guard && !planners_own(k) && (best_in < 0 || range_cost < best_in_cost)) { best_in = v.id; best_in_cost = range_cost; }
    }
  };
  // an explicit split_k looks among the variants with the split-K store path first; if none of them fits, the choice among
  // all variants reports below that it cannot split
  const bool explicit_split = d->split_k > 1 && !no_split;
  search(explicit_split);
  if (best < 0 && explicit_split) search(false);
  // A small grid that falls to a kernel without the split-K store path looks at split edge kernels as well, where K is deep enough to split at
  // all and the kernel is not one of those that stream B for up to 64 rows.  (The sweeps behind the tables held none, and beside the split-K kernels the tables flatter them: fp16 100x4096x4096 NN 20.6 us so, 16.8 on
  // 64x128 tiles in 4 slices.)
  if (small && best >= 0 && !planners_own(ks[best]) && !no_split && d->split_k == 0 && es < 4 && d->K > (es == 1 ? 16 * 128 : 8 * 64) && !ks[best]->splitk && small_grid_split(ks[best], d, left_for_sums(ks[best]), false, false) == 1) {
    split_edges = true;
    search(false);
  }
  // slices of the chosen kernel where it is an edge kernel: of its tiles on grids of up to half a round, of the last ones beyond
  auto edge_slices = [&]() {
    const KernelEntry* k = ks[best];
    if (!k->edge || k->splitk || no_split || d->split_k != 0 || settled) return 1;
    const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn);
    const size_t left = left_for_sums(k);
    return tiles > 128 ? tail_split_of(k, tiles, (d->K + k->bk - 1) / k->bk, false, left) : small ? small_grid_split(k, d, left, split_edges, false) : edge_split_of(k, d, left);
  };
  // A small grid whose route lies beyond the range of its table keeps it unless the refined times see the best route within the range ahead, over 64 rows by
  // 3 %.  The routes that this changes are 5 % faster up to 64 rows (165 drawn problems, 4 of them slower by 3 % or more); over 64 rows, of 127, 8 % faster
  // with operands that the last-level cache holds and 2 % slower with operands from memory.  us within / beyond: fp16 1024x1024x6272 NT 23.0 in 2
  // slices of 64x128 tiles, 31.0 in 7 of 256x256 (and 25.6 in 3 of 128x128 where slices of unequal length did not have to gain a fifth); 384x256x5888 NT 11.1 / 14.4, 128x1024x4864 NN 11.7 / 14.9, int8 640x128x14848 NT 13.0 / 16.6,
  // 32x9216x2688 NT 8.1 / 9.1.
  if (best >= 0 && best_in >= 0) {
    const KernelEntry *k = ks[best], *in = ks[best_in];
    const int split = k->splitk && d->K % k->bk == 0 ? small_grid_split(k, d, left_for_sums(k), false, false) : 1;
    if ((planners_own(k) ? edge_slices() == 1 : k->splitk && !in_table_range(k, d, split)) &&
        refined_time(k, d, split) * (d->K / k->bk % split ? 1.2 : d->M > 64 ? 0.97 : 1.0) >= refined_time(in, d, small_grid_split(in, d, left_for_sums(in), false, true))) {
      best = best_in;
      table_range = true;
      split_edges = false;
    }
  }
  // The 192x256 tile and split edge tiles against what a problem of whole K tiles and aligned rows runs on otherwise, 128x128 and 256x256 tiles in one
  // pass at their full rate: the costs above come out a few per cent apart there, closer than they are accurate, so the model of rounds must see a
  // gain too, of 4 % where the tile is another one.  us in one pass / so: bf16 2496x1664x3584 NN (260 tiles of 128x128) 39.8 / 44.1,
  // fp16 1500x2816x3008 NN 34.3 / 39.9, int8 1728x4480x640 NN 13.0 / 15.5, 6464x960x2560 NN 24.2 / 28.0.  Of 301 other
  // problems of 257 to 2200 tiles 144 were slower by 3 % and more on the route of the costs alone and 1 (int8 5952x1024x8192 NT, 59.2 / 61.9) with this
  // rule, which keeps 111 of 135 gains beyond 3 % (of those it leaves, f16 1856x4288x4736 NT, 82 / 69, is the largest).
  if (best >= 0 && rows_aligned && d->K % ks[best]->bk == 0 && round_model(ks[best])) {
    const int fresh = best, slices = edge_slices();
    if (slices > 1 || ks[fresh]->bm == 192) {
      const bool edges_were_split = split_edges;
      const double fresh_time = round_time(*round_model(ks[fresh]), ks[fresh], d, slices);
      best = -1;
      settled = true;
      split_edges = false;
      search(false);
      const KernelEntry* k = best >= 0 ? ks[best] : nullptr;
      const RoundModel* m = k ? round_model(k) : nullptr;
      const bool own_split = k && k->splitk && (small ? small_grid_split(k, d, left_for_sums(k), false, table_range) : 1) > 1;
      const bool same_tile = k && k->bm == ks[fresh]->bm && k->bn == ks[fresh]->bn;
      // one round of two 128x128 tiles a CU beats a partial one of unsplit 192x256 tiles, which has more to do on each CU than the model knows (us: bf16
      // 2624x3008x7680 NN 119.9 / 140.3, 1536x5312x7424 116.5 / 133.1, fp16 1920x4224x5120 87.6 / 93.7; 11 of 11 drawn problems slower by 3 to 15 %)
      const bool one_round = m && m->cap == 512 && slices == 1 && (((d->M + 127) / 128) * ((d->N + 127) / 128) <= 512);
      if (!m || own_split || (!one_round && fresh_time < (same_tile ? 0.99 : 0.96) * round_time(*m, k, d, 1))) {
        best = fresh;
        settled = false;
        split_edges = edges_were_split;
      }
    }
  }
  // Slices of the edge kernel that the search has found, and of K on a small grid; then the kernels that only follow up on one of the search.
  int found_slices = best >= 0 ? edge_slices() : 1;
  int found_split = 1;
  if (best >= 0 && small && ks[best]->splitk && !no_split && d->K % ks[best]->bk == 0) found_split = small_grid_split(ks[best], d, ctx.workspace, false, table_range);
  const bool follows = best >= 0 && !tile_requested && d->split_k <= 1 && d->policy == FRISK_POLICY_SQUARE;
  int next = follows ? follow_up(list, ks[best], d, rows_aligned, found_split, found_slices, packed) : -1;
  if (follows && next < 0 && !small && es < 4 && !(rows_aligned && d->M % 256 == 0 && d->N % 256 == 0 && d->K % ks[best]->bk == 0)) {
    // (what is split along K stays as it is: the models of split and unsplit grids are not close enough, fp16 1563x3054x3567 NT 51.0 us on 192x256 tiles in
    // 2 slices, 59.0 on 128x128 ones)
    const KernelEntry* k = ks[best];
    const int64_t tiles = ((d->M + k->bm - 1) / k->bm) * ((d->N + k->bn - 1) / k->bn), kt = d->K / k->bk;
    const bool splits = k->splitk && !no_split && d->split_k == 0 && d->K % k->bk == 0;
    if (found_slices == 1 && (!splits || (tiles < 256 ? sub_round_split(k, d, tiles, kt, ctx.workspace) : tail_split_of(k, tiles, kt, true, ctx.workspace)) == 1))
      next = other_tile(list, k, d, rows_aligned, packed);
  }
  if (follows && d->split_k == 0 && !no_split && found_slices == 1 && found_split == 1)
    if (const int id = deep_tile(list, ks[next >= 0 ? next : best], d, rows_aligned, left_for_sums(ks[best])); id >= 0) {
      best = id;
      next = -1;
      found_slices = edge_split_of(ks[id], d, left_for_sums(ks[id]));
    }
  if (next >= 0) best = next;
  const bool one_pass = next >= 0 && !same_edge_tile(ks[best]);
  if (d->M == 0 || d->N == 0) {  // nothing to compute
    plan->grid_x = plan->grid_y = 0;
    return FRISK_OK;
  }
  if (best < 0) {
    if (!any_layout) return fail(FRISK_ERR_DTYPE, "no kernel compiled for dtype %d transA=%d transB=%d", d->dtype_ab, d->transA, d->transB);
    if (policy_excluded && d->policy != FRISK_POLICY_SQUARE)
      return fail(FRISK_ERR_TILE, "wave policy %s: no compiled kernel for M=%lld N=%lld K=%lld has the wave grid that policy gives (compiled grids: 2x2, 1x4, 2x4, 1x1)",
                  d->policy == FRISK_POLICY_FULL_ROW ? "FullRow" : "FullCol", (long long)d->M, (long long)d->N, (long long)d->K);
    if (tile_requested)
      return fail(FRISK_ERR_TILE, "no compiled kernel with tile %dx%dx%d waves %dx%d atom %d divides M=%lld N=%lld K=%lld", d->tile_m, d->tile_n,
                  d->tile_k, d->waves_m, d->waves_n, d->atom, (long long)d->M, (long long)d->N, (long long)d->K);
    return fail(FRISK_ERR_SHAPE, "M=%lld N=%lld K=%lld is not a multiple of any compiled tile", (long long)d->M, (long long)d->N, (long long)d->K);
  }
  const KernelEntry* k = ks[best];
  if (k->lds_bytes > 160 * 1024) return fail(FRISK_ERR_LDS, "tile needs %d bytes of LDS", k->lds_bytes);
  plan->kernel_id = best;
  plan->tile_m = k->bm; plan->tile_n = k->bn; plan->tile_k = k->bk;
  plan->waves_m = k->wm; plan->waves_n = k->wn; plan->waves_k = k->wk; plan->threads = k->wm * k->wn * k->wk * 64;
  plan->mfma_m = k->atom; plan->mfma_n = k->atom; plan->mfma_k = mfma_k(d->dtype_ab) * (32 / k->atom);
  plan->lds_bytes = k->lds_bytes;
  plan->stages = k->stages;
  plan->stages_b = k->stages_b;
  plan->grid_x = (int)((d->N + k->bn - 1) / k->bn);
  plan->grid_y = (int)((d->M + k->bm - 1) / k->bm);
  plan->guarded = k->guard != 0;
  // (grids that are no multiple of 8 too, their last few ids staying in place; us in launch order / regrouped: bf16 3000x11008x4096 NT,
  // 516 tiles, 208.5 / 198.2; bf16 7168x6912x4096 TN, 756 tiles, 274.5 / 264.5; single rounds even)
  // One row of tiles against B [K][N] whose rows lie a multiple of 2 KiB apart stays in launch order: its tiles share A alone, which every L2 gets either way, and neighbouring
  // columns on one XCD are the same few of its L2's channels in every row.  us regrouped / in launch order, B from memory: fp16 48x8192x8192 32.8 / 31.4, 1x8192x8192 30.8 / 29.2, bf16 16x8192x5120
  // 22.4 / 20.8, 48x12288x8192 45.7 / 44.7, int8 16x8192x2048 7.9 / 7.4, e4m3 8x12288x2048 10.1 / 9.6; 100 problems with N a multiple of 1024 or 2048 1.02 times as fast, none slower by 3 %.
  // Elsewhere 8-bit rows end inside lines that neighbouring tiles share (e4m3 5x5184x4096 10.2 / 11.1); B [N][K] 16x8192x2048 8.7 / 11.0.
  const bool columns = plan->grid_y == 1 && !d->transB && d->ldb * es % 2048 == 0;
  plan->xcd_remap = (int64_t)plan->grid_x * plan->grid_y >= 8 && !columns;
  if (with_model) {  // for the caller of frisk_hip_plan: no launch looks at the LDS layouts
    fill_layout(&plan->lds_a, !d->transA, es, frag_bytes(d->dtype_ab), k->bm, k->bk, k->wm * k->wn * k->wk, k->atom);
    fill_layout(&plan->lds_b, d->transB != 0, es, frag_bytes(d->dtype_ab), k->bn, k->bk, k->wm * k->wn * k->wk, k->atom);
  }
  plan->workspace_bytes = 0;
  if (k->guard == 2 && packed.bytes) {
    plan->workspace_bytes = packed.bytes;
    if (extras) extras->repack = packed;
  }
  if (const int ts = one_pass ? 1 : found_slices; ts > 1) {
    const int64_t edge_tiles = (int64_t)plan->grid_x * plan->grid_y, split_tiles = edge_tiles <= 128 ? edge_tiles : edge_tiles % 256;
    const size_t offset = (plan->workspace_bytes + 255) & ~(size_t)255;
    plan->workspace_bytes = offset + (size_t)ts * (size_t)split_tiles * (size_t)k->bm * (size_t)k->bn * 4;
    if (extras) { extras->tail_split = ts; extras->tail_tiles = (int)split_tiles; extras->partial_offset = offset; }
  }
  // Split K over the grid's y dimension when the tile grid alone leaves most CUs idle (skinny problems are
  // bound by streaming the large operand, which needs many work-groups in flight).  Slices hold whole K tiles.
  const int64_t kt = d->K / k->bk, tiles = (int64_t)plan->grid_x * plan->grid_y;
  int split = 1;
  if (k->splitk && !no_split && d->K % k->bk == 0) {
    if (d->split_k > 1) {
      if (kt % d->split_k) return fail(FRISK_ERR_TILE, "split_k=%d does not divide the %lld K tiles", d->split_k, (long long)kt);
      if (kt / d->split_k < k->min_k_tiles)
        return fail(FRISK_ERR_TILE, "split_k=%d leaves %lld K tiles per slice, the chosen kernel %s needs %d", d->split_k, (long long)(kt / d->split_k), k->name, k->min_k_tiles);
      split = d->split_k;
    } else if (small) {
      split = found_split;
    } else if (d->split_k == 0 && tiles < 256) {
      split = sub_round_split(k, d, tiles, kt, ctx.workspace);
    } else if (d->split_k == 0) {
      const int ts = tail_split_of(k, tiles, kt, true, ctx.workspace);
      if (ts > 1) {
        plan->tail_split = ts;
        plan->tail_tiles = (int)(tiles % 256);
        plan->workspace_bytes = (size_t)ts * (size_t)plan->tail_tiles * (size_t)k->bm * (size_t)k->bn * 4;
      }
    }
  } else if (d->split_k > 1 && !no_split) {
    return fail(FRISK_ERR_TILE, "split_k=%d: the chosen kernel %s has no split-K path", d->split_k, k->name);
  }
  plan->split_k = split;
  if (split > 1) plan->workspace_bytes = (size_t)split * (size_t)d->M * (size_t)d->N * 4;
  if (plan->tail_split <= 1) { plan->tail_split = 1; plan->tail_tiles = 0; }
  return FRISK_OK;
}

// make_plan without the model of the LDS layouts, for the calls that launch.  A program's few descriptors come round again and again, and walking the
// variants takes 0.9 us (128x128x128) to 4 (a few rows against a large B, with all their splits) of a call that takes 7 to 8 through Python; a plan
// depends on nothing but the descriptor's values and the context, so each thread keeps those of the last descriptors that it has met: kept by value, in
// kKeptPlans places of 0.5 KiB, refused descriptors not at all.  us a call through Python before / now:
// 128x128x128 fp16 8.0 / 7.5 in a row, 18.7 / 18.0 waited for.
constexpr unsigned kKeptPlans = 64;  // a power of two
static int planned(const frisk_gemm_desc* d, frisk_gemm_plan* plan, const PlanContext& ctx, LaunchExtras* extras) {
  struct Kept { frisk_gemm_desc desc; PlanContext ctx; frisk_gemm_plan plan; LaunchExtras extras; bool used = false; };
  static thread_local std::unique_ptr<Kept[]> kept(new (std::nothrow) Kept[kKeptPlans]);
  if (!d || !kept) return make_plan(d, plan, false, ctx, extras);
  // (one shape on two leading dimensions, output types or pointer alignments in turn are two places)
  uint64_t h = (uint64_t)d->M * 0x9e3779b97f4a7c15ull ^ (uint64_t)d->N * 0xc2b2ae3d27d4eb4full ^ (uint64_t)d->K * 0x165667b19e3779f9ull;
  h ^= (uint64_t)ctx.workspace * 0xd6e8feb86659fd93ull + (uint64_t)((d->dtype_ab * 4 + d->transA * 2 + d->transB) * 16 + d->epilogue * 4 + (d->clear_accum ? 1 : 0));
  h += (uint64_t)d->lda * 0xa0761d6478bd642full ^ (uint64_t)d->ldb * 0xe7037ed1a0b428dbull ^ (uint64_t)d->ldc * 0x8ebc6af09c88c6e3ull;
  h += (uint64_t)(d->dtype_out * 8 + ctx.a_off * 4 + ctx.b_off * 2 + ctx.c_off) * 0x589965cc75374cc3ull;
  Kept& k = kept[(h * 0x9e3779b97f4a7c15ull) >> 58];
  static_assert(kKeptPlans == 64, "the place is the top six bits of the product");
  const bool same = k.used && std::memcmp(&k.desc, d, sizeof *d) == 0 && k.ctx.a_off == ctx.a_off && k.ctx.b_off == ctx.b_off && k.ctx.c_off == ctx.c_off && k.ctx.workspace == ctx.workspace;
  if (!same) {
    LaunchExtras fresh;
    frisk_gemm_plan p;
    if (int st = make_plan(d, &p, false, ctx, &fresh); st != FRISK_OK) return st;  // (p may not have been written)
    k = Kept{*d, ctx, p, fresh, true};
  }
  *plan = k.plan;
  if (extras) *extras = k.extras;
  return FRISK_OK;
}

// rows of tiles walked together so that the work-groups resident on one XCD form a compact block
static int group_rows(int tiles_m, int tiles_n) {
  int64_t total = (int64_t)tiles_m * tiles_n;
  int64_t per_xcd = std::max<int64_t>(1, std::min<int64_t>(total / 8, 32));
  int g = 1;
  while ((int64_t)(2 * g) * (2 * g) <= per_xcd) g *= 2;
  return std::max(1, std::min(g, tiles_m));
}

static int device_ok() {
  static std::atomic<int> cached{-1};  // the answer for the process's GPU; racing threads compute the same value
  int c = cached.load(std::memory_order_relaxed);
  if (c >= 0) return c;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
  c = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
  cached.store(c, std::memory_order_relaxed);
  return c;
}

// a rank-2 view handed to the tile ops: element type, extents, leading dimension, pointer
static int check_view(const char* what, int dtype, const void* p, int64_t rows, int64_t cols, int64_t ld) {
  if (dtype != FRISK_F32 && dtype != FRISK_F16 && dtype != FRISK_BF16) return fail(FRISK_ERR_DTYPE, "%s: element type %d is not f32, f16 or bf16", what, dtype);
  if (rows < 0 || cols < 0) return fail(FRISK_ERR_SHAPE, "%s: negative extent %lld x %lld", what, (long long)rows, (long long)cols);
  if (rows > INT32_MAX || cols > INT32_MAX) return fail(FRISK_ERR_SHAPE, "%s: extent exceeds 2^31-1", what);
  if (ld < cols) return fail(FRISK_ERR_SHAPE, "%s: leading dimension %lld smaller than the row length %lld", what, (long long)ld, (long long)cols);
  if (rows * cols > 0 && !p) return fail(FRISK_ERR_NULL, "%s: pointer is null", what);
  if ((uintptr_t)p & (uintptr_t)(elem_size(dtype) - 1)) return fail(FRISK_ERR_ALIGNMENT, "%s: pointer is not aligned to its element size", what);
  return FRISK_OK;
}

}  // namespace frisk

using namespace frisk;

extern "C" {

int frisk_hip_abi_version(void) { return FRISK_HIP_ABI_VERSION; }

const char* frisk_hip_last_error(void) { return g_last_error.c_str(); }

int frisk_hip_init(void) {
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  for (const KernelEntry* k : kernels())
    for (auto prepare : {k->prepare, k->prepare_old_c})
      if (hipError_t e = prepare ? prepare() : hipSuccess; e != hipSuccess) return fail(FRISK_ERR_DEVICE, "preparing %s failed: %s", k->name, hipGetErrorString(e));
  if (hipError_t e = prepare_attention(); e != hipSuccess) return fail(FRISK_ERR_DEVICE, "preparing the attention kernels failed: %s", hipGetErrorString(e));
  void* ws = nullptr;
  if (hipError_t e = scratch_of_current_device(&ws); e != hipSuccess) return fail(FRISK_ERR_DEVICE, "resolving the static workspace failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_plan(const frisk_gemm_desc* desc, frisk_gemm_plan* plan) { return make_plan(desc, plan, true); }

size_t frisk_hip_workspace_bytes(const frisk_gemm_desc* desc) {
  frisk_gemm_plan plan;
  if (planned(desc, &plan, {}, nullptr) != FRISK_OK) return 0;
  return plan.workspace_bytes;
}

int frisk_hip_gemm(const frisk_gemm_desc* desc, const void* A, const void* B, void* C, const float* scaleA,
                   const float* scaleB, void* workspace, size_t workspace_bytes, void* stream) {
  frisk_gemm_plan plan;
  LaunchExtras extras;
  PlanContext ctx;
  ctx.a_off = (uintptr_t)A & 15;
  ctx.b_off = (uintptr_t)B & 15;
  ctx.c_off = ((uintptr_t)C & 15) || (desc && desc->epilogue == FRISK_EPI_ROW_COL_SCALE && ((uintptr_t)scaleB & 15));
  int st = planned(desc, &plan, ctx, &extras);
  if (st != FRISK_OK) return st;
  if (desc->M == 0 || desc->N == 0) return FRISK_OK;
  if (!A || !B || !C) return fail(FRISK_ERR_NULL, "A, B and C must be device pointers");
  if (desc->epilogue != FRISK_EPI_NONE && (!scaleA || !scaleB)) return fail(FRISK_ERR_EPILOGUE, "epilogue %d needs scaleA and scaleB", desc->epilogue);
  const uintptr_t es = (uintptr_t)elem_size(desc->dtype_ab), os = (uintptr_t)elem_size(desc->dtype_out);
  if (((uintptr_t)A | (uintptr_t)B) & (es - 1) || (uintptr_t)C & (os - 1) || (((uintptr_t)scaleA | (uintptr_t)scaleB) & 3))
    return fail(FRISK_ERR_ALIGNMENT, "pointers must be aligned to their element size");
  const bool ws_aligned = ((uintptr_t)workspace & 15) == 0;
  if (plan.workspace_bytes > 0 && (!workspace || workspace_bytes < plan.workspace_bytes || (!ws_aligned && desc->split_k <= 1))) {
    // an explicit split_k needs its workspace; the planner's own choice takes the splits that fit the one there is, and one pass without one it can
    // use, be it missing or off 16-byte boundaries: a caller cannot know which sizes the planner splits
    if (desc->split_k > 1) return fail(FRISK_ERR_WORKSPACE, "split_k=%d needs %zu bytes of workspace", desc->split_k, plan.workspace_bytes);
    const size_t wanted = plan.workspace_bytes;
    ctx.workspace = workspace && ws_aligned ? workspace_bytes : 0;
    st = planned(desc, &plan, ctx, &extras);
    // a tile or wave policy that the caller named and that only kernels without staging through registers have: they want the copies
    if (st != FRISK_OK)
      return fail(FRISK_ERR_WORKSPACE, "rows or pointers off 16-byte boundaries: the tile or wave policy asked for runs on aligned copies of A or B, which need %zu bytes of 16-byte aligned workspace", wanted);
  }
  if (plan.workspace_bytes > 0 && !ws_aligned) return fail(FRISK_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");

  GemmParams p;
  p.A = A; p.B = B; p.C = C; p.scaleA = scaleA; p.scaleB = scaleB;
  p.lda = desc->lda; p.ldb = desc->ldb; p.ldc = desc->ldc;
  p.M = (int)desc->M; p.N = (int)desc->N; p.K = (int)desc->K;
  p.tiles_m = plan.grid_y; p.tiles_n = plan.grid_x;
  p.group_m = group_rows(p.tiles_m, p.tiles_n);
  p.xcd_remap = plan.xcd_remap;
  p.epilogue = desc->epilogue; p.dtype_out = desc->dtype_out; p.accumulate = desc->clear_accum ? 0 : 1;
  const KernelEntry* k = kernels()[plan.kernel_id];
  p.split_k = plan.split_k;
  p.kt_per_slice = (int)(((desc->K + k->bk - 1) / k->bk + p.split_k - 1) / p.split_k);
  const Repack& repack = extras.repack;
  const int tail_split = std::max(plan.tail_split, extras.tail_split);
  p.partial = p.split_k > 1 || tail_split > 1 ? (char*)workspace + extras.partial_offset : nullptr;
  p.tail_split = tail_split;
  p.tail_tiles = extras.tail_split > 1 ? extras.tail_tiles : plan.tail_tiles;
  p.tail_from = p.tiles_m * p.tiles_n - p.tail_tiles;
  p.tail_kt = tail_split > 1 ? (p.kt_per_slice + tail_split - 1) / tail_split : 0;
  p.tile_m = k->bm; p.tile_n = k->bn;
  // 64x32 tiles in more than one row share their rows of A and B through the L2, which work-groups at different K tiles do not: us rotated / not, 400 problems
  // of 65 to 2048 rows, operands in the last-level cache: 8.6 % slower on average, 1024x512x6400 fp16 28.2 / 17.0; from memory 2.8 % faster.  The fp32 tiles of
  // 32x32 that follow up on larger ones likewise (94 problems, 3.5 % slower rotated, 710x693x3944 73 / 61)
  p.k_rotate = (k->bm == 32 && !is_follow_up(k)) || p.tiles_m == 1;
  hipError_t e = hipSuccess;
  if (repack.bytes) {
    RepackParams r;
    auto side = [&](RepackParams::Side& s, bool on, const void* src, void* dst, int64_t rows, int64_t cols, int64_t ld, int64_t dst_ld) {
      if (on) s = {src, dst, ld * (int64_t)es, dst_ld * (int64_t)es, rows, cols * (int64_t)es};
    };
    side(r.a, repack.a, A, workspace, desc->transA ? desc->K : desc->M, desc->transA ? desc->M : desc->K, desc->lda, repack.lda);
    side(r.b, repack.b, B, (char*)workspace + repack.b_offset, desc->transB ? desc->N : desc->K, desc->transB ? desc->K : desc->N, desc->ldb, repack.ldb);
    if (repack.a) { p.A = r.a.dst; p.lda = repack.lda; }
    if (repack.b) { p.B = r.b.dst; p.ldb = repack.ldb; }
    e = launch_repack(r, (hipStream_t)stream);
    if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "launch of the copy to aligned rows failed: %s", hipGetErrorString(e));
  }
  const bool old_c = k->launch_old_c && p.accumulate && p.dtype_out == FRISK_F32 && p.epilogue == FRISK_EPI_NONE;
  e = (old_c ? k->launch_old_c : k->launch)(p, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "launch of %s failed: %s", k->name, hipGetErrorString(e));
  if (p.split_k > 1) {
    e = launch_splitk_reduce(p, desc->dtype_acc == FRISK_I32, (hipStream_t)stream);
    if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "launch of the split-K reduction failed: %s", hipGetErrorString(e));
  }
  if (tail_split > 1) {
    e = launch_tail_reduce(p, desc->dtype_acc == FRISK_I32, (hipStream_t)stream);
    if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "launch of the tail reduction failed: %s", hipGetErrorString(e));
  }
  return FRISK_OK;
}

size_t frisk_hip_static_workspace_bytes(void) { return (size_t)FRISK_HIP_STATIC_WS_BYTES; }

int frisk_hip_gemm_static_ws(const frisk_gemm_desc* desc, const void* A, const void* B, void* C, const float* scaleA, const float* scaleB,
                             void* stream) {
  frisk_gemm_plan plan;
  int st = planned(desc, &plan, {}, nullptr);
  if (st != FRISK_OK) return st;
  // What does not fit the array: an explicit split_k is refused (the caller asked for exactly that split), and so is a named tile that runs on copies
  // larger than it; of the splits the planner chooses by itself it takes those that fit (a split of K of fewer slices; no tail split: those of
  // large grids reach 64 MiB).
  if (plan.workspace_bytes > (size_t)FRISK_HIP_STATIC_WS_BYTES) {
    if (desc->split_k > 1)
      return fail(FRISK_ERR_WORKSPACE, "split_k=%d needs %zu bytes of partial sums, the static workspace holds %zu: pass a smaller split_k, or use frisk_hip_gemm with a workspace",
                  desc->split_k, plan.workspace_bytes, (size_t)FRISK_HIP_STATIC_WS_BYTES);
    PlanContext limited;
    limited.workspace = FRISK_HIP_STATIC_WS_BYTES;
    st = planned(desc, &plan, limited, nullptr);
    if (st != FRISK_OK || plan.workspace_bytes == 0) return frisk_hip_gemm(desc, A, B, C, scaleA, scaleB, nullptr, 0, stream);
  }
  void* ws = nullptr;
  if (plan.workspace_bytes > 0) {
    if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
    if (hipError_t e = scratch_of_current_device(&ws); e != hipSuccess) return fail(FRISK_ERR_DEVICE, "resolving the static workspace failed: %s", hipGetErrorString(e));
  }
  // every slice of a split stores its whole share of the partial sums before the reduction reads it: nothing to clear
  return frisk_hip_gemm(desc, A, B, C, scaleA, scaleB, ws, ws ? (size_t)FRISK_HIP_STATIC_WS_BYTES : 0, stream);
}

float frisk_hip_lds_access_cycles(int instr, const int32_t* lane_byte_addr) {
  if (!lane_byte_addr) return -1.f;
  int addr[64];
  for (int i = 0; i < 64; ++i) addr[i] = lane_byte_addr[i];
  return (float)lds_access_cycles(instr == 2 ? 1 : instr, addr);
}

int frisk_hip_lds_search(const frisk_lds_layout* shape, int elem_bytes, int frag_bytes, int tile_mn, int tile_k, int waves,
                         frisk_lds_layout* best, float* unswizzled_cycles) {
  return frisk_hip_lds_search_atom(shape, elem_bytes, frag_bytes, tile_mn, tile_k, waves, 32, best, unswizzled_cycles);
}

int frisk_hip_lds_search_atom(const frisk_lds_layout* shape, int elem_bytes, int frag_bytes, int tile_mn, int tile_k, int waves, int atom,
                              frisk_lds_layout* best, float* unswizzled_cycles) {
  if (atom != 32 && atom != 16) return fail(FRISK_ERR_TILE, "MFMA atoms have 32 or 16 rows, not %d", atom);
  if (atom == 16 && elem_bytes == 4) return fail(FRISK_ERR_TILE, "the 32-bit operands have no 16-row atom here");
  if (!shape || !best) return fail(FRISK_ERR_NULL, "shape and best must be given");
  if (shape->rows <= 0 || shape->row_bytes < 16 || shape->row_bytes % 16 || shape->row_bytes > 1024 || 1024 % shape->row_bytes)
    return fail(FRISK_ERR_TILE, "tile rows must be 16..1024 bytes and divide 1024");
  if ((elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4) || frag_bytes < elem_bytes || waves <= 0 || tile_mn < 32 || tile_k <= 0)
    return fail(FRISK_ERR_TILE, "unsupported operand description");
  const bool kc = shape->k_contiguous != 0;
  TileShape t{shape->rows, shape->row_bytes, kc, elem_bytes, frag_bytes, tile_mn, tile_k, atom};
  const Swizzle s = choose_swizzle(t, waves);
  const int atoms = tile_mn / atom < 4 ? tile_mn / atom : 4;
  const int n_access = atoms * ((tile_k * elem_bytes) / frag_kstep_bytes(frag_bytes, atom)) * frag_instr_count(kc, elem_bytes, frag_bytes);
  if (n_access <= 0) return fail(FRISK_ERR_TILE, "tile holds no whole MFMA step");
  *best = *shape;
  best->row_shift = s.sh; best->row_mask = s.mk; best->chunk_shift = s.cs;
  best->row_shift2 = s.sh2; best->row_mask2 = s.mk2; best->chunk_shift2 = s.cs2;
  best->read_instr = elem_bytes == 4 ? (kc && frag_bytes >= 16 ? 0 : 3) : (kc ? 0 : (elem_bytes == 2 ? 1 : 2));
  best->read_cycles = (float)swizzle_read_cycles(t, s) / (float)n_access;
  best->write_cycles = 16.f;
  if (unswizzled_cycles) *unswizzled_cycles = (float)swizzle_read_cycles(t, Swizzle{0, 0, 0}) / (float)n_access;
  return FRISK_OK;
}

int32_t frisk_hip_lds_offset(const frisk_lds_layout* L, int32_t row, int32_t col_byte) {
  if (!L) return -1;
  return lds_offset(L->row_bytes, Swizzle{L->row_shift, L->row_mask, L->chunk_shift, L->row_shift2, L->row_mask2, L->chunk_shift2}, row, col_byte);
}

int frisk_hip_wave_partition(int policy, int tile_m, int tile_n, int num_waves, int* waves_m, int* waves_n) {
  if (!waves_m || !waves_n) return fail(FRISK_ERR_NULL, "output pointers are null");
  if (policy < FRISK_POLICY_SQUARE || policy > FRISK_POLICY_FULL_COL) return fail(FRISK_ERR_TILE, "unknown wave policy %d", policy);
  wave_partition(policy, tile_m, tile_n, num_waves, 32, 32, waves_m, waves_n);
  return FRISK_OK;
}

int frisk_hip_fill(int dtype, void* dst, int64_t rows, int64_t cols, int64_t ld, double value, void* stream) {
  if (int st = check_view("fill destination", dtype, dst, rows, cols, ld)) return st;
  if (rows == 0 || cols == 0) return FRISK_OK;
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  if (ld == cols) { cols *= rows; rows = 1; ld = cols; }  // a dense view is one long row
  hipError_t e = launch_fill(dtype, dst, rows, cols, ld, value, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "fill launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_copy(int src_dtype, const void* src, int64_t src_ld, int dst_dtype, void* dst, int64_t dst_ld, int64_t rows, int64_t cols,
                   void* stream) {
  if (int st = check_view("copy source", src_dtype, src, rows, cols, src_ld)) return st;
  if (int st = check_view("copy destination", dst_dtype, dst, rows, cols, dst_ld)) return st;
  if (rows == 0 || cols == 0) return FRISK_OK;
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  if (src_ld == cols && dst_ld == cols) { cols *= rows; rows = 1; src_ld = dst_ld = cols; }
  hipError_t e = launch_copy(src_dtype, src, src_ld, dst_dtype, dst, dst_ld, rows, cols, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "copy launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_copy_tiles(int src_dtype, const void* src, int64_t src_ld, int dst_dtype, void* dst, int64_t dst_ld, int64_t tile_rows, int64_t tile_cols,
                         int64_t n0, int64_t src_step0, int64_t dst_step0, int64_t n1, int64_t src_step1, int64_t dst_step1, void* stream) {
  const int64_t view_rows = (n0 == 0 || n1 == 0) ? 0 : tile_rows;  // no tile: no pointer is looked at
  if (int st = check_view("tiled copy source", src_dtype, src, view_rows, tile_cols, src_ld)) return st;
  if (int st = check_view("tiled copy destination", dst_dtype, dst, view_rows, tile_cols, dst_ld)) return st;
  if (n0 < 0 || n1 < 0 || src_step0 < 0 || src_step1 < 0 || dst_step0 < 0 || dst_step1 < 0) return fail(FRISK_ERR_SHAPE, "tiled copy: negative tile count or step");
  if (n0 > INT32_MAX || n1 > INT32_MAX || n0 * n1 > INT32_MAX) return fail(FRISK_ERR_SHAPE, "tiled copy: more than 2^31-1 tiles");
  if (tile_rows == 0 || tile_cols == 0 || n0 == 0 || n1 == 0) return FRISK_OK;
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  TilePlacement t;
  t.n0 = n0; t.n1 = n1; t.src_step0 = src_step0; t.src_step1 = src_step1; t.dst_step0 = dst_step0; t.dst_step1 = dst_step1;
  hipError_t e = launch_copy_tiles(src_dtype, src, src_ld, dst_dtype, dst, dst_ld, tile_rows, tile_cols, t, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "tiled copy launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_elementwise(const frisk_elementwise_desc* d, const void* const* inputs, void* out, void* stream) {
  if (!d) return fail(FRISK_ERR_NULL, "elementwise descriptor is null");
  if (d->abi_version != FRISK_HIP_ABI_VERSION) return fail(FRISK_ERR_ABI, "descriptor abi_version %d, library %d", d->abi_version, FRISK_HIP_ABI_VERSION);
  if (d->n_inputs < 0 || d->n_inputs > FRISK_EW_MAX_INPUTS) return fail(FRISK_ERR_ARGUMENT, "elementwise: %d operands, at most %d", d->n_inputs, FRISK_EW_MAX_INPUTS);
  if (d->n_ops < 1 || d->n_ops > FRISK_EW_MAX_OPS) return fail(FRISK_ERR_ARGUMENT, "elementwise: a program of %d steps, 1 to %d allowed", d->n_ops, FRISK_EW_MAX_OPS);
  if (int st = check_view("elementwise output", d->out_dtype, out, d->rows, d->cols, d->out_ld)) return st;
  if (d->n_inputs > 0 && !inputs) return fail(FRISK_ERR_NULL, "elementwise: the operand pointer array is null");
  // the program on a counting stack: never empty when it pops, never deeper than the interpreter's registers, one value left
  int depth = 0;
  for (int i = 0; i < d->n_ops; ++i) {
    const int op = d->op[i];
    if (op < FRISK_EW_INPUT || op > FRISK_EW_LOG2) return fail(FRISK_ERR_ARGUMENT, "elementwise: unknown opcode %d at step %d", op, i);
    if (op == FRISK_EW_INPUT && (d->arg[i] < 0 || d->arg[i] >= d->n_inputs)) return fail(FRISK_ERR_ARGUMENT, "elementwise: step %d reads operand %d of %d", i, d->arg[i], d->n_inputs);
    const int pops = op <= FRISK_EW_CONST ? 0 : (op >= FRISK_EW_NEG ? 1 : 2);
    if (depth < pops) return fail(FRISK_ERR_ARGUMENT, "elementwise: step %d pops an empty stack", i);
    depth += 1 - pops;
    if (depth > FRISK_EW_MAX_STACK) return fail(FRISK_ERR_ARGUMENT, "elementwise: the program needs a stack deeper than %d", FRISK_EW_MAX_STACK);
  }
  if (depth != 1) return fail(FRISK_ERR_ARGUMENT, "elementwise: the program leaves %d values, not one", depth);
  if (d->rows == 0 || d->cols == 0) return FRISK_OK;
  EwParams p{};
  // a dense problem (every operand walked, every row following the one before) is one long row
  bool dense = d->out_ld == d->cols;
  for (int k = 0; k < d->n_inputs; ++k) dense = dense && d->in_col_stride[k] == 1 && d->in_row_stride[k] == d->cols;
  p.rows = dense ? 1 : d->rows;
  p.cols = dense ? d->rows * d->cols : d->cols;
  for (int k = 0; k < d->n_inputs; ++k) {
    const int dt = d->in_dtype[k];
    if (dt != FRISK_F32 && dt != FRISK_F16 && dt != FRISK_BF16) return fail(FRISK_ERR_DTYPE, "elementwise operand %d: element type %d is not f32, f16 or bf16", k, dt);
    if (d->in_col_stride[k] != 0 && d->in_col_stride[k] != 1) return fail(FRISK_ERR_SHAPE, "elementwise operand %d: column stride %d is not 0 or 1", k, d->in_col_stride[k]);
    if (d->in_row_stride[k] < 0) return fail(FRISK_ERR_SHAPE, "elementwise operand %d: negative row stride", k);
    if (!inputs[k]) return fail(FRISK_ERR_NULL, "elementwise operand %d: pointer is null", k);
    if ((uintptr_t)inputs[k] & (uintptr_t)(elem_size(dt) - 1)) return fail(FRISK_ERR_ALIGNMENT, "elementwise operand %d: pointer is not aligned to its element size", k);
    p.in[k] = inputs[k]; p.in_row_stride[k] = d->in_row_stride[k]; p.in_dtype[k] = dt; p.in_col_stride[k] = d->in_col_stride[k];
  }
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  p.out = out; p.out_ld = d->out_ld; p.out_dtype = d->out_dtype; p.n_ops = d->n_ops;
  for (int i = 0; i < d->n_ops; ++i) { p.op[i] = d->op[i]; p.arg[i] = d->arg[i]; p.imm[i] = d->imm[i]; }
  hipError_t e = launch_elementwise(p, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "elementwise launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

size_t frisk_hip_reduce_workspace_bytes(int dtype, int64_t rows, int64_t cols, int dim) {
  if ((dtype != FRISK_F32 && dtype != FRISK_F16 && dtype != FRISK_BF16) || rows <= 0 || cols <= 0 || (dim != 0 && dim != 1)) return 0;
  const int slices = reduce_slices(dtype, rows, cols, dim);
  return slices > 1 ? (size_t)slices * (size_t)(dim == 1 ? rows : cols) * 4 : 0;
}

int frisk_hip_reduce(int dtype, const void* src, int64_t rows, int64_t cols, int64_t ld, int dim, int kind, int clear, void* dst, void* workspace,
                     size_t workspace_bytes, void* stream) {
  if (int st = check_view("reduce source", dtype, src, rows, cols, ld)) return st;
  if (dim != 0 && dim != 1) return fail(FRISK_ERR_ARGUMENT, "reduce dim %d is out of range for a source of rank 2", dim);
  if (kind < FRISK_REDUCE_ADD || kind > FRISK_REDUCE_MAX) return fail(FRISK_ERR_ARGUMENT, "unsupported reduce kind %d (add, mul, min, max)", kind);
  const int64_t kept = dim == 1 ? rows : cols;
  if (kept == 0) return FRISK_OK;
  if (!dst) return fail(FRISK_ERR_NULL, "reduce destination: pointer is null");
  if ((uintptr_t)dst & (uintptr_t)(elem_size(dtype) - 1)) return fail(FRISK_ERR_ALIGNMENT, "reduce destination: pointer is not aligned to its element size");
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  int slices = (rows > 0 && cols > 0) ? reduce_slices(dtype, rows, cols, dim) : 1;
  // without a (large enough, 4-byte aligned) workspace the reduction runs unsplit: same result, fewer work-groups
  if (slices > 1 && (!workspace || workspace_bytes < (size_t)slices * (size_t)kept * 4 || ((uintptr_t)workspace & 3))) slices = 1;
  hipError_t e = launch_reduce(dtype, src, rows, cols, ld, dim, kind, clear ? 1 : 0, dst, (float*)workspace, slices, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "reduce launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

size_t frisk_hip_softmax_workspace_bytes(int dtype, int64_t rows, int64_t cols) {
  if ((dtype != FRISK_F32 && dtype != FRISK_F16 && dtype != FRISK_BF16) || rows <= 0 || cols <= 0) return 0;
  const int slices = softmax_slices(dtype, rows, cols);
  return slices > 1 ? (size_t)rows * (size_t)slices * 8 : 0;
}

int frisk_hip_softmax(int dtype, const void* src, int64_t src_ld, void* dst, int64_t dst_ld, int64_t rows, int64_t cols, float scale_log2, float* lse,
                      void* workspace, size_t workspace_bytes, void* stream) {
  if (int st = check_view("softmax source", dtype, src, rows, cols, src_ld)) return st;
  if (int st = check_view("softmax destination", dtype, dst, rows, cols, dst_ld)) return st;
  if (!std::isfinite(scale_log2)) return fail(FRISK_ERR_ARGUMENT, "softmax scale %g is not finite", (double)scale_log2);
  if ((uintptr_t)lse & 3) return fail(FRISK_ERR_ALIGNMENT, "lse must be 4-byte aligned");
  if (rows == 0 || cols == 0) return FRISK_OK;
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  int slices = softmax_slices(dtype, rows, cols);
  // without a (large enough, 4-byte aligned) workspace the rows are not split: same result, fewer work-groups
  if (slices > 1 && (!workspace || workspace_bytes < (size_t)rows * (size_t)slices * 8 || ((uintptr_t)workspace & 3))) slices = 1;
  hipError_t e = launch_softmax_rows(dtype, src, src_ld, dst, dst_ld, rows, cols, scale_log2, lse, (float*)workspace, slices, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "softmax launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_attention(const frisk_attention_desc* d, const void* Q, const void* K, const void* V, void* O, float* lse, void* stream) {
  if (!d) return fail(FRISK_ERR_NULL, "attention descriptor is null");
  if (d->abi_version != FRISK_HIP_ABI_VERSION) return fail(FRISK_ERR_ABI, "descriptor abi_version %d, library %d", d->abi_version, FRISK_HIP_ABI_VERSION);
  if (d->dtype != FRISK_F16 && d->dtype != FRISK_BF16) return fail(FRISK_ERR_DTYPE, "attention element type %d is not f16 or bf16", d->dtype);
  if (d->batch < 0 || d->heads < 0 || d->seq_q < 0 || d->seq_k < 0) return fail(FRISK_ERR_SHAPE, "negative extent");
  if (d->head_dim != kAttnHeadDim) return fail(FRISK_ERR_SHAPE, "head_dim %lld: the attention kernel is built for %d", (long long)d->head_dim, kAttnHeadDim);
  if (d->seq_q % kAttnQueriesPerGroup) return fail(FRISK_ERR_SHAPE, "seq_q %lld is not a multiple of %d", (long long)d->seq_q, kAttnQueriesPerGroup);
  if (d->seq_k % kAttnKeysPerTile || d->seq_k == 0) return fail(FRISK_ERR_SHAPE, "seq_k %lld is not a positive multiple of %d", (long long)d->seq_k, kAttnKeysPerTile);
  if (!(d->scale > 0.f) || !std::isfinite(d->scale)) return fail(FRISK_ERR_ARGUMENT, "softmax scale %g is not a positive finite number", (double)d->scale);
  const int64_t bh = d->batch * d->heads, groups = bh * (d->seq_q / kAttnQueriesPerGroup);
  if (d->seq_q > INT32_MAX || d->seq_k > INT32_MAX || bh > INT32_MAX || groups > INT32_MAX) return fail(FRISK_ERR_SHAPE, "extent exceeds 2^31-1");
  if (groups == 0) return FRISK_OK;
  if (!Q || !K || !V || !O) return fail(FRISK_ERR_NULL, "attention operand pointer is null");
  if (((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)O) & 15) return fail(FRISK_ERR_ALIGNMENT, "attention operands must be 16-byte aligned");
  if ((uintptr_t)lse & 3) return fail(FRISK_ERR_ALIGNMENT, "lse must be 4-byte aligned");
  if (!device_ok()) return fail(FRISK_ERR_DEVICE, "no gfx950 device is current");
  AttentionParams p;
  p.Q = Q; p.K = K; p.V = V; p.O = O; p.lse = lse;
  p.batch_heads = (int32_t)bh; p.seq_q = (int32_t)d->seq_q; p.seq_k = (int32_t)d->seq_k;
  p.scale_log2 = d->scale * 1.4426950408889634f;
  hipError_t e = launch_attention(d->dtype, d->k_transposed ? 1 : 0, p, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FRISK_ERR_DEVICE, "attention launch failed: %s", hipGetErrorString(e));
  return FRISK_OK;
}

int frisk_hip_kernel_count(void) { return (int)kernels().size(); }
const char* frisk_hip_kernel_name(int id) {
  if (id < 0 || id >= (int)kernels().size()) return nullptr;
  return kernels()[id]->name;
}

}  // extern "C"
