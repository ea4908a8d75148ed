// frisk.fill, frisk.copy and frisk.reduce on rank-2 views of device memory.  All three are bound by
// HBM traffic: a lane moves 16 bytes at a time, wherever the rows start (only a row's last group, when it is not whole, goes element
// by element), and a launch covers the view with many more work-groups than the 256 CUs.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "tile_ops.h"

namespace frisk {
namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// streaming reads: every byte is read once, so the caches are told not to keep it; on stores the hint pays in copy
// between equally wide types (6.3 against 5.9 TB/s) and changes nothing in fill, so only copy uses it
// (16 bytes that start on any element: loads and stores of this type are one instruction at any address)
typedef unsigned v4u_any __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ v4u load16(const void* p) { return __builtin_nontemporal_load((const v4u_any*)p); }
__device__ __forceinline__ void store16(void* p, v4u v) { *(v4u_any*)p = v; }
__device__ __forceinline__ void store16_stream(void* p, v4u v) { __builtin_nontemporal_store(v, (v4u_any*)p); }

template <int DT> struct Elem;
template <> struct Elem<FRISK_F32> { typedef float T; static __device__ float load(const T& x) { return x; } static __device__ T store(float x) { return x; } };
template <> struct Elem<FRISK_F16> { typedef _Float16 T; static __device__ float load(const T& x) { return (float)x; } static __device__ T store(float x) { return (_Float16)x; } };
template <> struct Elem<FRISK_BF16> { typedef __bf16 T; static __device__ float load(const T& x) { return (float)x; } static __device__ T store(float x) { return (__bf16)x; } };

// A rows x cols view is cut into groups of G columns (16 bytes of the narrower type) and walked without any division:
// 2^lanes_log2 lanes of a work-group lie along a row, the remaining 256 >> lanes_log2 across rows, work-groups step
// along the row in x and down the rows in y.  Every lane handles several groups per step: ALONG (1, 2 or 4) neighbours along the row
// (4 KiB apart) where the row is long enough to give them work, or (ALONG 0) the same columns of eight rows.

template <int ALONG> struct Walk {
  static constexpr int PER = ALONG ? ALONG : kPerLaneAcross;
  int64_t slabs, row_blocks, rows, groups_per_row;
  int lanes, lane_group, lane_row, row_step;
  __device__ Walk(int64_t rows_, int64_t groups_per_row_, int lanes_log2) : rows(rows_), groups_per_row(groups_per_row_) {
    lanes = 1 << lanes_log2;
    row_step = 256 >> lanes_log2;
    lane_group = threadIdx.x & (lanes - 1);
    lane_row = threadIdx.x >> lanes_log2;
    // groups of a slab and rows of a row block are powers of two: shifts (a 64-bit division is 150 instructions, and most work-groups
    // take a single step)
    constexpr int kPerLog2 = PER == 8 ? 3 : PER == 4 ? 2 : PER == 2 ? 1 : 0;
    static_assert(PER == 1 << kPerLog2, "groups per lane and step");
    const int x_log2 = lanes_log2 + (ALONG ? kPerLog2 : 0), y_log2 = 8 - lanes_log2 + (ALONG ? 0 : kPerLog2);
    slabs = (groups_per_row + ((int64_t)1 << x_log2) - 1) >> x_log2;
    row_blocks = (rows + ((int64_t)1 << y_log2) - 1) >> y_log2;
  }
  // the u-th group of this lane in step (slab, rb); false when it lies outside the view
  __device__ bool at(int64_t slab, int64_t rb, int u, int64_t& row, int64_t& group) const {
    group = (ALONG ? slab * PER + u : slab) * lanes + lane_group;
    row = (ALONG ? rb : rb * PER + u) * row_step + lane_row;
    return group < groups_per_row && row < rows;
  }
  // every group of the step (slab, rb) lies inside the view and is whole (wave-uniform)
  __device__ bool inside(int64_t slab, int64_t rb, int64_t cols, int G) const {
    return (slab + 1) * (ALONG ? PER : 1) * lanes * G <= cols && (rb + 1) * row_step * (ALONG ? 1 : PER) <= rows;
  }
};

template <int DT, int ALONG> __global__ void __launch_bounds__(256)
fill_kernel(typename Elem<DT>::T* dst, int64_t rows, int64_t cols, int64_t ld, float value, int lanes_log2) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T);
  const Walk<ALONG> w(rows, (cols + G - 1) / G, lanes_log2);
  constexpr int PER = Walk<ALONG>::PER;
  const T v = Elem<DT>::store(value);
  T tmp[G];
#pragma unroll
  for (int e = 0; e < G; ++e) tmp[e] = v;
  for (int64_t rb = blockIdx.y; rb < w.row_blocks; rb += gridDim.y)
    for (int64_t slab = blockIdx.x; slab < w.slabs; slab += gridDim.x) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        int64_t r, g;
        if (!w.at(slab, rb, u, r, g)) continue;
        const int64_t c0 = g * G;
        T* p = dst + r * ld + c0;
        if (c0 + G <= cols) store16(p, *(const v4u*)tmp);
        else for (int e = 0; e < G && c0 + e < cols; ++e) p[e] = v;
      }
    }
}

template <int SDT, int DDT, int ALONG> __device__ __forceinline__ void
copy_window(const typename Elem<SDT>::T* src, int64_t sld, typename Elem<DDT>::T* dst, int64_t dld, int64_t rows, int64_t cols, int lanes_log2) {
  typedef typename Elem<SDT>::T S;
  typedef typename Elem<DDT>::T D;
  constexpr int G = 16 / (sizeof(S) < sizeof(D) ? sizeof(S) : sizeof(D));  // 16 bytes of the narrower side, 32 of the wider
  const Walk<ALONG> w(rows, (cols + G - 1) / G, lanes_log2);
  constexpr int PER = Walk<ALONG>::PER;
  for (int64_t rb = blockIdx.y; rb < w.row_blocks; rb += gridDim.y)
    for (int64_t slab = blockIdx.x; slab < w.slabs; slab += gridDim.x) {
      S in[PER][G];
      // one group converted and stored
      auto put = [&](D* dp, const S (&x)[G]) {
        D out[G];
#pragma unroll
        for (int e = 0; e < G; ++e) {
          if constexpr (SDT == DDT) out[e] = x[e]; else out[e] = Elem<DDT>::store(Elem<SDT>::load(x[e]));
        }
#pragma unroll
        for (int q = 0; q < (int)(G * sizeof(D) / 16); ++q) {
          // a lane's two stores of a widening copy each cover half of its 32 bytes: the cache has to merge them
          if constexpr (sizeof(D) > sizeof(S)) store16((v4u*)dp + q, ((const v4u*)out)[q]); else store16_stream((v4u*)dp + q, ((const v4u*)out)[q]);
        }
      };
      if (w.inside(slab, rb, cols, G)) {  // nothing to check
        const S* sp[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          int64_t r, g;
          w.at(slab, rb, u, r, g);
          sp[u] = src + r * sld + g * G;
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          // The groups along a row are fetched one after the other, each waited for before the next is requested, and all stored at the
          // end: reads and writes then reach memory in longer runs (512 MiB + 512 MiB f32: 6.0 TB/s with both requests in flight
          // together, 7.4 one after the other).
          if (ALONG > 1 && u > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
          for (int q = 0; q < (int)(G * sizeof(S) / 16); ++q) ((v4u*)in[u])[q] = load16((const v4u*)sp[u] + q);
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          int64_t r, g;
          w.at(slab, rb, u, r, g);
          put(dst + r * dld + g * G, in[u]);
        }
        continue;
      }
      bool whole[PER];
      // every load of the step is issued before the first store
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        int64_t r, g;
        whole[u] = w.at(slab, rb, u, r, g) && g * G + G <= cols;
        if (whole[u]) {
#pragma unroll
          for (int q = 0; q < (int)(G * sizeof(S) / 16); ++q) ((v4u*)in[u])[q] = load16((const v4u*)(src + r * sld + g * G) + q);
        }
      }
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        int64_t r, g;
        if (!w.at(slab, rb, u, r, g)) continue;
        const int64_t c0 = g * G;
        D* dp = dst + r * dld + c0;
        if (whole[u]) {
          put(dp, in[u]);
        } else {
          const S* sp = src + r * sld + c0;
          for (int e = 0; e < G && c0 + e < cols; ++e) {
            if constexpr (SDT == DDT) dp[e] = sp[e]; else dp[e] = Elem<DDT>::store(Elem<SDT>::load(sp[e]));
          }
        }
      }
    }
}

template <int SDT, int DDT, int ALONG> __global__ void __launch_bounds__(256)
copy_kernel(const typename Elem<SDT>::T* src, int64_t sld, typename Elem<DDT>::T* dst, int64_t dld, int64_t rows, int64_t cols, int lanes_log2) {
  copy_window<SDT, DDT, ALONG>(src, sld, dst, dld, rows, cols, lanes_log2);
}

// the same window copied once per tile of a placement: z walks the n0 x n1 tiles, each displacing both sides by its steps
template <int SDT, int DDT, int ALONG> __global__ void __launch_bounds__(256)
copy_tiles_kernel(const typename Elem<SDT>::T* src, int64_t sld, typename Elem<DDT>::T* dst, int64_t dld, int64_t rows, int64_t cols, TilePlacement t, int lanes_log2) {
  const int64_t tiles = t.n0 * t.n1;
  for (int64_t z = blockIdx.z; z < tiles; z += gridDim.z) {
    const int64_t a = z / t.n1, b = z - a * t.n1;
    copy_window<SDT, DDT, ALONG>(src + a * t.src_step0 + b * t.src_step1, sld, dst + a * t.dst_step0 + b * t.dst_step1, dld, rows, cols, lanes_log2);
  }
}

// ------------------------------------------------------------------ reduce
template <int KIND> struct Op;
template <> struct Op<FRISK_REDUCE_ADD> { static __device__ float id() { return 0.f; } static __device__ float f(float a, float b) { return a + b; } };
template <> struct Op<FRISK_REDUCE_MUL> { static __device__ float id() { return 1.f; } static __device__ float f(float a, float b) { return a * b; } };
template <> struct Op<FRISK_REDUCE_MIN> { static __device__ float id() { return __builtin_inff(); } static __device__ float f(float a, float b) { return __builtin_fminf(a, b); } };
template <> struct Op<FRISK_REDUCE_MAX> { static __device__ float id() { return -__builtin_inff(); } static __device__ float f(float a, float b) { return __builtin_fmaxf(a, b); } };

template <int KIND> __device__ __forceinline__ float wave_reduce(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = Op<KIND>::f(v, __shfl_xor(v, off, 64));
  return v;
}

// along dim 1: work-group (x = row, y = column slice) reduces every gridDim.y-th run of THREADS 16-byte groups of one row, so that
// the slices of a row read neighbouring memory at any time.
// With gridDim.y == 1 the result goes to dst (combined with the old value unless clear), else to partial[y][row].
// A row's last group, where it is not whole, is fetched first, with the elements before it that fill it up, which are left out: every load is 16 bytes of the row, those of a lane are under way
// together, and the loop over the whole groups knows nothing of it.  us element by element behind the loop / as a group of the loop / so, from memory: f16 3000 x 4095 9.7 / 7.3 / 7.3, 2490 x 2453
// 7.0 / 5.4 / 5.1, 10069 x 4946 20.2 / 18.4 / 16.1, f32 5531 x 1315 10.0 / 7.8 / 7.6; rows of whole groups, f16 2177 x 8944 8.4 / 9.8 / 8.7, 1024 x 16384 7.2 / 8.4 / 7.3.
// LOADS: views of up to 64 MiB are read through the caches, where the call behind often finds them: cast, row sums, (x - s c) g + b and softmax in a row of 4096 x 8192 f16 93.6 us so, 96.8 with sums
// past the caches, f32 3029 x 3796 60.8 / 64.5, 131 drawn views 1.003 times as fast.  (On their own, rows on 16-byte boundaries would be read sooner past them: out of the last-level cache f16 4096 x 8192 9.4 us,
// 11.2 so, from memory 11.6 / 12.3; off them, groups that straddle 128-byte lines are fetched twice there, 2490 x 4453 5.14 us, 4.96 so.)  Beyond, past them, with the groups starting at a row's first
// boundary where rows start off one, what lies before it being a group that overlaps like the last (bf16 6199 x 10825 27.4 at the rows' starts, 21.3 so).
// A group's elements are added in pairs, then to what the lane has: the sums of 256 lanes are no further from the exact ones than those of 512 that add one element after the other (f32
// 2000 x 6144, 2-norm of the error over that of the sums: 1.21e-7 one after the other, 1.06e-7 on 512 lanes, 0.99e-7 so; times even, 9.83 / 9.85 us from memory, f16 8192 x 8192 20.9 / 20.9).
enum RowLoads { LOADS_CACHED, LOADS_PAST, LOADS_FROM_BOUNDARY };
template <int DT, int KIND, int THREADS, int LOADS> __global__ void __launch_bounds__(THREADS)
reduce_rows_kernel(const typename Elem<DT>::T* src, int64_t rows, int64_t cols, int64_t ld, int clear, typename Elem<DT>::T* dst, float* partial) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T), FLIGHT = 4;
  const int64_t step = (int64_t)gridDim.y * THREADS, me = (int64_t)blockIdx.y * THREADS + threadIdx.x;
  auto load = [](const T* at) {
    if constexpr (LOADS == LOADS_CACHED) return *(const v4u_any*)at;
    else return load16(at);
  };
  __shared__ float wsum[THREADS / 64];
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    float acc = Op<KIND>::id();
    const T* row = src + r * ld;
    // groups 0 .. full - 1 from element `head` on, then the one that ends with the row, then the one it starts with: the last ones of their lanes (slices are a power of two)
    const int64_t head = LOADS == LOADS_FROM_BOUNDARY ? ((0 - (uintptr_t)row) & 15) / sizeof(T) : 0, full = (cols - head) / G, tail = cols - head - full * G;
    const bool ends = tail > 0 && (full & (step - 1)) == me, starts = head > 0 && ((full + (tail > 0)) & (step - 1)) == me;
    T edge[G];
    if (ends || starts) *(v4u*)edge = load(row + (ends ? cols - G : 0));
    // four groups of a lane under way together, combined in their order (one after the other 98 x 12807 bf16 took 6.2 us, 8192 x 8192 f16 22.9)
    for (int64_t g = me; g < full; g += FLIGHT * step) {
      T in[FLIGHT][G];
#pragma unroll
      for (int u = 0; u < FLIGHT; ++u)
        if (g + u * step < full) *(v4u*)in[u] = load(row + head + (g + u * step) * G);
#pragma unroll
      for (int u = 0; u < FLIGHT; ++u) {
        if (g + u * step >= full) continue;
        float t[G];
#pragma unroll
        for (int e = 0; e < G; ++e) t[e] = Elem<DT>::load(in[u][e]);
#pragma unroll
        for (int half = G / 2; half >= 1; half >>= 1)
#pragma unroll
          for (int e = 0; e < half; ++e) t[e] = Op<KIND>::f(t[e], t[e + half]);
        acc = Op<KIND>::f(acc, t[0]);
      }
    }
    if (ends || starts) {
      const int lo = ends ? G - (int)tail : 0, hi = ends ? G : (int)head;  // its own elements
#pragma unroll
      for (int e = 0; e < G; ++e)
        if (e >= lo && e < hi) acc = Op<KIND>::f(acc, Elem<DT>::load(edge[e]));
    }
    acc = wave_reduce<KIND>(acc);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      float v = Op<KIND>::f(Op<KIND>::f(wsum[0], wsum[1]), Op<KIND>::f(wsum[2], wsum[3]));
      if constexpr (THREADS == 512) v = Op<KIND>::f(v, Op<KIND>::f(Op<KIND>::f(wsum[4], wsum[5]), Op<KIND>::f(wsum[6], wsum[7])));
      if (gridDim.y > 1) partial[(int64_t)blockIdx.y * rows + r] = v;
      else dst[r] = Elem<DT>::store(clear ? v : Op<KIND>::f(Elem<DT>::load(dst[r]), v));
    }
    __syncthreads();
  }
}

// along dim 1, rows of at most 256 groups of 16 bytes: 2^lanes_log2 <= 64 lanes of one wave share a row, each taking up to
// NPT groups, and combine by shuffles; a work-group holds 256 >> lanes_log2 rows and takes 4 / NPT such sets of rows per
// step, so that every lane has four loads in flight before the first is used.
// TAIL: rows of whole groups (with the code for another last group f16 20000 x 1000 10.5 us out of the last-level cache, 9.2 so, bf16 5878 x 864 5.8 from memory, 5.4 so); with a last group that is
// fetched with the elements before it that fill it up, which count as nothing (element by element behind the others / behind a branch / so, from memory: bf16 14242 x 790 10.0 / 10.3 / 7.2, f16 20000 x 1003
// 15.5 / 12.2 / 11.7, 16384 x 2047 20.5 / 16.9 / 15.2, 100000 x 27 7.0 / 5.7 / 5.4); of less than a group, element by element.
enum RowTail { TAIL_WHOLE, TAIL_PART, TAIL_NARROW };
template <int DT, int KIND, int NPT, int TAIL> __global__ void __launch_bounds__(256)
reduce_short_rows_kernel(const typename Elem<DT>::T* src, int64_t rows, int64_t cols, int64_t ld, int clear, typename Elem<DT>::T* dst, int lanes_log2) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T), SETS = 4 / NPT;
  const int lanes = 1 << lanes_log2, lane = threadIdx.x & (lanes - 1), rows_per_set = 256 >> lanes_log2;
  const int64_t blocks = (rows + rows_per_set * SETS - 1) / (rows_per_set * SETS);
  for (int64_t rb = blockIdx.x; rb < blocks; rb += gridDim.x) {
    T in[SETS][NPT][G];
    bool inside[SETS][NPT];
#pragma unroll
    for (int t = 0; t < SETS; ++t) {
      const int64_t r = (rb * SETS + t) * rows_per_set + (threadIdx.x >> lanes_log2);
#pragma unroll
      for (int q = 0; q < NPT; ++q) {
        const int c0 = (q * lanes + lane) * G;
        inside[t][q] = r < rows && c0 < (int)cols;
        if (!inside[t][q]) continue;
        const T* at = src + r * ld;
        if constexpr (TAIL == TAIL_NARROW) {
#pragma unroll
          for (int e = 0; e < G; ++e) in[t][q][e] = at[e < (int)cols ? e : 0];
        } else *(v4u*)in[t][q] = load16(at + (TAIL == TAIL_WHOLE || c0 + G <= (int)cols ? c0 : (int)cols - G));
      }
    }
#pragma unroll
    for (int t = 0; t < SETS; ++t) {
      const int64_t r = (rb * SETS + t) * rows_per_set + (threadIdx.x >> lanes_log2);
      const bool live = r < rows;  // lanes of rows past the end still take part in the shuffles
      float acc = Op<KIND>::id();
#pragma unroll
      for (int q = 0; q < NPT; ++q) {
        if (!inside[t][q]) continue;
        const int past = (q * lanes + lane + 1) * G - (int)cols;
        const int lo = TAIL == TAIL_PART && past > 0 ? past : 0, hi = TAIL == TAIL_NARROW ? (int)cols : G;
#pragma unroll
        for (int e = 0; e < G; ++e) acc = Op<KIND>::f(acc, TAIL == TAIL_WHOLE || (e >= lo && e < hi) ? Elem<DT>::load(in[t][q][e]) : Op<KIND>::id());
      }
      for (int off = lanes >> 1; off >= 1; off >>= 1) acc = Op<KIND>::f(acc, __shfl_xor(acc, off, 64));
      if (live && lane == 0) dst[r] = Elem<DT>::store(clear ? acc : Op<KIND>::f(Elem<DT>::load(dst[r]), acc));
    }
  }
}

// along dim 0: a work-group owns a strip of 2^lanes_log2 x G columns and every gridDim.y-th chunk of rows; 2^lanes_log2 column
// lanes x (256 >> lanes_log2) row lanes, kStripFlight rows in flight per lane.  The strip is kStripLanes x 16 bytes of every
// row, or the power of two that covers a narrower view (of a dense one a wave then reads consecutive memory), or wider
// when the view has too few rows to give every row lane a full set of loads.  Four rows in flight (2 to 16 measure within
// 4 % of each other) when the view has many strips; a single strip gives one work-group per slice, 256 at most, and takes
// 16 (5.5 against 4.2 TB/s on a 1M x 128 f16 view).  The row lanes combine by halving in LDS.
constexpr int kStripLanes = 32;  // 16 and 64 lanes measured 9 % and 15 % slower on wide views

template <int DT, int KIND, int kStripFlight> __global__ void __launch_bounds__(256)
reduce_cols_kernel(const typename Elem<DT>::T* src, int64_t rows, int64_t cols, int64_t ld, int clear, typename Elem<DT>::T* dst, float* partial, int lanes_log2) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T);
  const int cl = threadIdx.x & ((1 << lanes_log2) - 1), rl = threadIdx.x >> lanes_log2, row_lanes = 256 >> lanes_log2;
  const int64_t c0 = (((int64_t)blockIdx.x << lanes_log2) + cl) * G;
  const int64_t chunk = (int64_t)kStripFlight * row_lanes;
  float acc[G];
#pragma unroll
  for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::id();
  if (c0 < cols) {
    const bool whole = c0 + G <= cols;
    for (int64_t base = (int64_t)blockIdx.y * chunk; base < rows; base += (int64_t)gridDim.y * chunk) {
      if (whole && base + chunk <= rows) {
        T in[kStripFlight][G];
#pragma unroll
        for (int u = 0; u < kStripFlight; ++u) *(v4u*)in[u] = load16(src + (base + rl + (int64_t)row_lanes * u) * ld + c0);
#pragma unroll
        for (int u = 0; u < kStripFlight; ++u)
#pragma unroll
          for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::f(acc[e], Elem<DT>::load(in[u][e]));
      } else {
        for (int64_t r = base + rl; r < rows && r < base + chunk; r += row_lanes) {
          const T* p = src + r * ld + c0;
          if (whole) {
            T in[G];
            *(v4u*)in = load16(p);
#pragma unroll
            for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::f(acc[e], Elem<DT>::load(in[e]));
          } else {
            for (int e = 0; e < G && c0 + e < cols; ++e) acc[e] = Op<KIND>::f(acc[e], Elem<DT>::load(p[e]));
          }
        }
      }
    }
  }
  __shared__ float red[256][G + 1];  // [row lane * column lanes + column lane]
#pragma unroll
  for (int e = 0; e < G; ++e) red[threadIdx.x][e] = acc[e];
  __syncthreads();
  for (int half = row_lanes >> 1; half >= 1; half >>= 1) {
    if (rl < half) {
#pragma unroll
      for (int e = 0; e < G; ++e) red[threadIdx.x][e] = Op<KIND>::f(red[threadIdx.x][e], red[threadIdx.x + (half << lanes_log2)][e]);
    }
    __syncthreads();
  }
  if (rl == 0 && c0 < cols) {
    for (int e = 0; e < G && c0 + e < cols; ++e) {
      const float v = red[cl][e];
      if (gridDim.y > 1) partial[(int64_t)blockIdx.y * cols + c0 + e] = v;
      else dst[c0 + e] = Elem<DT>::store(clear ? v : Op<KIND>::f(Elem<DT>::load(dst[c0 + e]), v));
    }
  }
}

// along dim 0 in one launch, for views that would otherwise be split down the rows but have few enough of them (cols_in_one_launch): 1024 lanes on
// a strip of 8 x 16 bytes (or fewer, of a narrower view), eight rows under way per lane.  The row lanes of a wave combine by shuffles, the waves in
// LDS.  What it saves is the launch that combines the slices: us in two launches / so, f16 309 x 3904 6.9 / 4.1, 256 x 1024 7.0 / 4.1, 1259 x 1728 7.6 /
// 6.3, f32 309 x 3904 7.4 / 4.3.  A work-group walks its strip at some 40 bytes a nanosecond (1024 lanes, of which all wait, then all add), so from
// 2000 rows on the slices are ahead again (f16 2000 x 1984 7.9 / 8.3, 3000 x 1024 8.6 / 13.3), and so they are where there is more than one strip for
// every CU (1000 x 65536 25.2 / 27.7).  Rows that do not start on 128-byte lines, of which a strip takes two each, leave the range from 1152 on unless they are short (f32 1452 x
// 460 7.1 / 9.2, f16 1379 x 2120 7.9 / 9.7, 1228 x 1544 11 % slower; but 970 x 8671 12.3 / 8.9, 1354 x 56 10.6 / 5.4, and on lines 1434 x 7414 13.4 / 8.1).
template <int DT, int KIND> __global__ void __launch_bounds__(1024)
reduce_tall_kernel(const typename Elem<DT>::T* src, int64_t rows, int64_t cols, int64_t ld, int clear, typename Elem<DT>::T* dst, int lanes_log2) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T), FLIGHT = 8;
  const int lanes = 1 << lanes_log2, cl = threadIdx.x & (lanes - 1), rl = threadIdx.x >> lanes_log2, row_lanes = 1024 >> lanes_log2;
  // A row's last group, where it is not whole, is read with the columns before it that fill it up, which are another lane's: every load is 16 bytes of the
  // row and eight are under way.  (Element by element, a row after the other, it held up the call: f16 1435 x 1495 25.0 us, 10.5 so,
  // 970 x 8671 19.0 and 8.9.)
  const int64_t first = (((int64_t)blockIdx.x << lanes_log2) + cl) * G;
  const int before = first < cols && first + G > cols && cols >= G ? (int)(first + G - cols) : 0;
  const int64_t c0 = first - before;
  float acc[G];
#pragma unroll
  for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::id();
  if (c0 + G <= cols) {
    for (int64_t r = rl; r < rows; r += FLIGHT * row_lanes) {
      T in[FLIGHT][G];
#pragma unroll
      for (int u = 0; u < FLIGHT; ++u)
        if (r + u * row_lanes < rows) *(v4u*)in[u] = load16(src + (r + u * row_lanes) * ld + c0);
#pragma unroll
      for (int u = 0; u < FLIGHT; ++u) {
        if (r + u * row_lanes >= rows) continue;
#pragma unroll
        for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::f(acc[e], Elem<DT>::load(in[u][e]));
      }
    }
  } else if (c0 < cols) {  // the only group of a row that has no more
    for (int64_t r = rl; r < rows; r += row_lanes) {
#pragma unroll
      for (int e = 0; e < G; ++e)
        if (c0 + e < cols) acc[e] = Op<KIND>::f(acc[e], Elem<DT>::load(src[r * ld + c0 + e]));
    }
  }
  for (int off = 32; off >= lanes; off >>= 1) {
#pragma unroll
    for (int e = 0; e < G; ++e) acc[e] = Op<KIND>::f(acc[e], __shfl_xor(acc[e], off, 64));
  }
  __shared__ float red[16][8 * G];  // [wave][column of the strip]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane < lanes) {
#pragma unroll
    for (int e = 0; e < G; ++e)
      if (e >= before) red[wave][lane * G + e - before] = acc[e];
  }
  __syncthreads();
  const int64_t c = ((int64_t)blockIdx.x << lanes_log2) * G + threadIdx.x;
  if ((int)threadIdx.x >= lanes * G || c >= cols) return;
  float part[16];  // in pairs: in a row the 16 came out 1.2 times as far from the exact sum as the slices did
#pragma unroll
  for (int w = 0; w < 16; ++w) part[w] = red[w][threadIdx.x];
#pragma unroll
  for (int half = 8; half >= 1; half >>= 1)
#pragma unroll
    for (int w = 0; w < half; ++w) part[w] = Op<KIND>::f(part[w], part[w + half]);
  const float v = part[0];
  dst[c] = Elem<DT>::store(clear ? v : Op<KIND>::f(Elem<DT>::load(dst[c]), v));
}

// second pass of a split reduction: out[i] = kind over s of partial[s][i] (combined with dst unless clear).  64 outputs x 4
// slice lanes per work-group: a lane combines every fourth slice with four loads in flight, so that 256 slices cost 16
// memory round trips instead of 256.
template <int DT, int KIND> __global__ void __launch_bounds__(256)
reduce_finish_kernel(const float* partial, int slices, int64_t n, int clear, typename Elem<DT>::T* dst) {
  const int ol = threadIdx.x & 63, sl = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + ol;
  float v = Op<KIND>::id();
  if (i < n) {
    int s = sl;
    for (; s + 12 < slices; s += 16) {
      float t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) t[u] = partial[(int64_t)(s + 4 * u) * n + i];
#pragma unroll
      for (int u = 0; u < 4; ++u) v = Op<KIND>::f(v, t[u]);
    }
    for (; s < slices; s += 4) v = Op<KIND>::f(v, partial[(int64_t)s * n + i]);
  }
  __shared__ float red[4][64];
  red[sl][ol] = v;
  __syncthreads();
  if (sl == 0 && i < n) {
    v = Op<KIND>::f(Op<KIND>::f(red[0][ol], red[1][ol]), Op<KIND>::f(red[2][ol], red[3][ol]));
    dst[i] = Elem<DT>::store(clear ? v : Op<KIND>::f(Elem<DT>::load(dst[i]), v));
  }
}

template <int DT> hipError_t fill_t(void* dst, int64_t rows, int64_t cols, int64_t ld, double value, hipStream_t s) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T);
  const WalkGrid w = walk_grid(rows, (cols + G - 1) / G);
  const dim3 grid(w.x, w.y);
  if (w.along) hipLaunchKernelGGL((fill_kernel<DT, 2>), grid, dim3(256), 0, s, (T*)dst, rows, cols, ld, (float)value, w.lanes_log2);
  else hipLaunchKernelGGL((fill_kernel<DT, 0>), grid, dim3(256), 0, s, (T*)dst, rows, cols, ld, (float)value, w.lanes_log2);
  return hipGetLastError();
}

template <int SDT, int DDT> hipError_t copy_t(const void* src, int64_t sld, void* dst, int64_t dld, int64_t rows, int64_t cols, hipStream_t s) {
  typedef typename Elem<SDT>::T S;
  typedef typename Elem<DDT>::T D;
  constexpr int G = 16 / (sizeof(S) < sizeof(D) ? sizeof(S) : sizeof(D));
  const WalkGrid w = walk_grid(rows, (cols + G - 1) / G, copy_groups_per_lane(rows, (cols + G - 1) / G));
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(w.x, w.y), dim3(256), 0, s, (const S*)src, sld, (D*)dst, dld, rows, cols, w.lanes_log2); };
  switch (w.along) {
    case 1: launch(copy_kernel<SDT, DDT, 1>); break;
    case 2: launch(copy_kernel<SDT, DDT, 2>); break;
    case 4: launch(copy_kernel<SDT, DDT, 4>); break;
    default: launch(copy_kernel<SDT, DDT, 0>); break;
  }
  return hipGetLastError();
}

template <int SDT, int DDT> hipError_t copy_tiles_t(const void* src, int64_t sld, void* dst, int64_t dld, int64_t rows, int64_t cols, const TilePlacement& t, hipStream_t s) {
  typedef typename Elem<SDT>::T S;
  typedef typename Elem<DDT>::T D;
  constexpr int G = 16 / (sizeof(S) < sizeof(D) ? sizeof(S) : sizeof(D));
  const WalkGrid w = walk_grid(rows, (cols + G - 1) / G);
  const int64_t tiles = t.n0 * t.n1;
  const dim3 grid(w.x, w.y, (unsigned)(tiles > 65535 ? 65535 : tiles));
  if (w.along) hipLaunchKernelGGL((copy_tiles_kernel<SDT, DDT, 2>), grid, dim3(256), 0, s, (const S*)src, sld, (D*)dst, dld, rows, cols, t, w.lanes_log2);
  else hipLaunchKernelGGL((copy_tiles_kernel<SDT, DDT, 0>), grid, dim3(256), 0, s, (const S*)src, sld, (D*)dst, dld, rows, cols, t, w.lanes_log2);
  return hipGetLastError();
}

// a launch may hold fewer than 2^32 lanes: grids are capped and work-groups loop
constexpr int64_t kMaxGrid = 1 << 22;

// `on_lines`: every row starts on a 128-byte boundary.  Where they don't, a strip of 128 bytes takes two lines of every row, and the slices are ahead sooner (lines
// at reduce_tall_kernel).
// Long rows on lines, which give most CUs a strip, stay in it longer: us in slices / in one launch, bf16 2000 x 7168 10.8 / 10.7, 2000 x 8192 11.4 / 10.8, 2500 x 8192
// 12.5 / 13.3, 2500 x 11008 15.2 / 13.7, 3000 x 11008 17.9 / 15.6, 3000 x 16384 21.1 / 20.2, f32 3000 x 7168 18.3 / 17.5; 4096 x 12288 bf16 20.6 / 21.6.
bool cols_in_one_launch(int64_t rows, int64_t row_bytes, bool on_lines) {
  const int64_t most = !on_lines && row_bytes > 256 ? 1152 : !on_lines || row_bytes < 14 << 10 ? 1536 : row_bytes < 20 << 10 ? 2048 : 3072;
  return rows <= most && row_bytes <= 256 * 128;
}

// slices of the reduced extent that give the launch enough work-groups
int split_of(int dtype, int64_t rows, int64_t cols, int dim) {
  // Split the reduced extent so that about 1024 work-groups exist, each still reducing at least 16 KiB.  Rows of up to 64 KiB stay whole, however few (us in slices and a second launch / in
  // one, f32 394 x 9229 7.4 / 4.8, 64 x 16000 7.8 / 4.6).
  const int es = dtype == FRISK_F32 ? 4 : 2;
  if (dim == 1 && cols * es <= 65536) return 1;
  const int G = 16 / es;
  const int64_t groups = dim == 1 ? rows : (cols + kStripLanes * G - 1) / (kStripLanes * G);
  const int64_t strip_bytes = cols * es < kStripLanes * 16 ? cols * es : kStripLanes * 16;
  const int64_t extent_bytes = dim == 1 ? cols * es : rows * strip_bytes;  // bytes one work-group would walk unsplit
  int slices = 1;
  while (groups * slices < 1024 && extent_bytes / (slices * 2) >= 16384 && slices < 256) slices *= 2;
  return slices;
}

template <int DT, int KIND> hipError_t reduce_t(const void* src, int64_t rows, int64_t cols, int64_t ld, int dim, int clear, void* dst, float* partial,
                                                int slices, hipStream_t s) {
  typedef typename Elem<DT>::T T;
  constexpr int G = 16 / sizeof(T);
  const int64_t gpr = (cols + G - 1) / G;
  // (without slices the one launch takes every view of its range)
  const bool tall = dim == 0 && split_of(DT, rows, cols, dim) > 1 &&
                    cols_in_one_launch(rows, cols * (int64_t)sizeof(T), slices == 1 || ((uintptr_t)src % 128 == 0 && ld * sizeof(T) % 128 == 0));
  if (tall) slices = 1;
  if (dim == 1) {
    if (gpr <= 256 && slices == 1) {
      int lanes_log2 = 0;
      while (lanes_log2 < 6 && (int64_t(1) << lanes_log2) < gpr) ++lanes_log2;
      const int64_t rows_per_step = (256 >> lanes_log2) * (gpr <= 64 ? 4 : (gpr <= 128 ? 2 : 1)), blocks = (rows + rows_per_step - 1) / rows_per_step;
      const dim3 grid((unsigned)(blocks < kMaxGrid ? blocks : kMaxGrid));
      auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, (const T*)src, rows, cols, ld, clear, (T*)dst, lanes_log2); };
      const bool whole = cols % G == 0;
#define FRISK_REDUCE_SHORT(NPT) { if (whole) launch(reduce_short_rows_kernel<DT, KIND, NPT, TAIL_WHOLE>); else launch(reduce_short_rows_kernel<DT, KIND, NPT, TAIL_PART>); }
      if (cols < G) launch(reduce_short_rows_kernel<DT, KIND, 1, TAIL_NARROW>);
      else if (gpr <= 64) FRISK_REDUCE_SHORT(1)
      else if (gpr <= 128) FRISK_REDUCE_SHORT(2)
      else FRISK_REDUCE_SHORT(4)
#undef FRISK_REDUCE_SHORT
    } else {
      const dim3 grid((unsigned)(rows < kMaxGrid ? rows : kMaxGrid), (unsigned)slices);
      const bool aligned = (((uintptr_t)src | ld * sizeof(T)) & 15) == 0, large = rows * cols * (int64_t)sizeof(T) > (int64_t)64 << 20;
      // 512 lanes where they have three groups each or the rows are few (us 256 / 512 lanes: f32 4000 x 8192 18.9 / 18.0, f16 2048 x 16384 11.7 / 11.5, bf16 1000 x 9000 5.6 / 5.2; but 1126 and
      // 1354 groups of more rows, f32 4111 x 4501 10.8 / 11.9, bf16 6199 x 10825 21.3 / 22.1)
      const bool wide = gpr > 1536 || (gpr > 1024 && rows <= 1024);
      auto launch = [&](auto kernel, int threads) { hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, (const T*)src, rows, cols, ld, clear, (T*)dst, partial); };
#define FRISK_REDUCE_ROWS(LOADS) { if (wide) launch(reduce_rows_kernel<DT, KIND, 512, LOADS>, 512); else launch(reduce_rows_kernel<DT, KIND, 256, LOADS>, 256); }
      if (!large) FRISK_REDUCE_ROWS(LOADS_CACHED)
      else if (aligned) FRISK_REDUCE_ROWS(LOADS_PAST)
      else FRISK_REDUCE_ROWS(LOADS_FROM_BOUNDARY)
#undef FRISK_REDUCE_ROWS
    }
  } else if (tall) {
    int lanes_log2 = 0;
    while (lanes_log2 < 3 && (int64_t(1) << lanes_log2) < gpr) ++lanes_log2;
    hipLaunchKernelGGL((reduce_tall_kernel<DT, KIND>), dim3((unsigned)((gpr + (1 << lanes_log2) - 1) >> lanes_log2)), dim3(1024), 0, s, (const T*)src, rows, cols, ld, clear,
                       (T*)dst, lanes_log2);
  } else {
    int lanes_log2 = 0;
    while ((1 << lanes_log2) < kStripLanes && (int64_t(1) << lanes_log2) < gpr) ++lanes_log2;
    while (lanes_log2 < 8 && (int64_t(1) << lanes_log2) < gpr && (256 >> lanes_log2) * 4 > rows) ++lanes_log2;  // few rows: wider strips
    const unsigned strips = (unsigned)((gpr + (1 << lanes_log2) - 1) >> lanes_log2);
    // a view of one strip gives at most one work-group per slice: its lanes keep more rows in flight instead
    if (strips == 1) hipLaunchKernelGGL((reduce_cols_kernel<DT, KIND, 16>), dim3(strips, (unsigned)slices), dim3(256), 0, s, (const T*)src, rows, cols, ld, clear, (T*)dst,
                                        partial, lanes_log2);
    else hipLaunchKernelGGL((reduce_cols_kernel<DT, KIND, 4>), dim3(strips, (unsigned)slices), dim3(256), 0, s, (const T*)src, rows, cols, ld, clear, (T*)dst, partial,
                            lanes_log2);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || slices == 1) return e;
  const int64_t n = dim == 1 ? rows : cols;
  hipLaunchKernelGGL((reduce_finish_kernel<DT, KIND>), dim3((unsigned)((n + 63) / 64)), dim3(256), 0, s, partial, slices, n, clear, (T*)dst);
  return hipGetLastError();
}

template <int DT> hipError_t reduce_k(int kind, const void* src, int64_t rows, int64_t cols, int64_t ld, int dim, int clear, void* dst, float* partial, int slices,
                                      hipStream_t s) {
  switch (kind) {
    case FRISK_REDUCE_ADD: return reduce_t<DT, FRISK_REDUCE_ADD>(src, rows, cols, ld, dim, clear, dst, partial, slices, s);
    case FRISK_REDUCE_MUL: return reduce_t<DT, FRISK_REDUCE_MUL>(src, rows, cols, ld, dim, clear, dst, partial, slices, s);
    case FRISK_REDUCE_MIN: return reduce_t<DT, FRISK_REDUCE_MIN>(src, rows, cols, ld, dim, clear, dst, partial, slices, s);
    default: return reduce_t<DT, FRISK_REDUCE_MAX>(src, rows, cols, ld, dim, clear, dst, partial, slices, s);
  }
}

}  // namespace

// (where the one launch depends on the rows' pitch, the slices' sums have their place all the same)
int reduce_slices(int dtype, int64_t rows, int64_t cols, int dim) {
  return dim == 0 && cols_in_one_launch(rows, cols * (dtype == FRISK_F32 ? 4 : 2), false) ? 1 : split_of(dtype, rows, cols, dim);
}

hipError_t launch_fill(int dtype, void* dst, int64_t rows, int64_t cols, int64_t ld, double value, hipStream_t s) {
  switch (dtype) {
    case FRISK_F32: return fill_t<FRISK_F32>(dst, rows, cols, ld, value, s);
    case FRISK_F16: return fill_t<FRISK_F16>(dst, rows, cols, ld, value, s);
    default: return fill_t<FRISK_BF16>(dst, rows, cols, ld, value, s);
  }
}

hipError_t launch_copy_tiles(int sdt, const void* src, int64_t sld, int ddt, void* dst, int64_t dld, int64_t rows, int64_t cols, const TilePlacement& t, hipStream_t s) {
#define FRISK_COPY_CASE(S, D) if (sdt == S && ddt == D) return copy_tiles_t<S, D>(src, sld, dst, dld, rows, cols, t, s);
  FRISK_COPY_CASE(FRISK_F32, FRISK_F32) FRISK_COPY_CASE(FRISK_F32, FRISK_F16) FRISK_COPY_CASE(FRISK_F32, FRISK_BF16)
  FRISK_COPY_CASE(FRISK_F16, FRISK_F32) FRISK_COPY_CASE(FRISK_F16, FRISK_F16) FRISK_COPY_CASE(FRISK_F16, FRISK_BF16)
  FRISK_COPY_CASE(FRISK_BF16, FRISK_F32) FRISK_COPY_CASE(FRISK_BF16, FRISK_F16) FRISK_COPY_CASE(FRISK_BF16, FRISK_BF16)
#undef FRISK_COPY_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_copy(int sdt, const void* src, int64_t sld, int ddt, void* dst, int64_t dld, int64_t rows, int64_t cols, hipStream_t s) {
#define FRISK_COPY_CASE(S, D) if (sdt == S && ddt == D) return copy_t<S, D>(src, sld, dst, dld, rows, cols, s);
  FRISK_COPY_CASE(FRISK_F32, FRISK_F32) FRISK_COPY_CASE(FRISK_F32, FRISK_F16) FRISK_COPY_CASE(FRISK_F32, FRISK_BF16)
  FRISK_COPY_CASE(FRISK_F16, FRISK_F32) FRISK_COPY_CASE(FRISK_F16, FRISK_F16) FRISK_COPY_CASE(FRISK_F16, FRISK_BF16)
  FRISK_COPY_CASE(FRISK_BF16, FRISK_F32) FRISK_COPY_CASE(FRISK_BF16, FRISK_F16) FRISK_COPY_CASE(FRISK_BF16, FRISK_BF16)
#undef FRISK_COPY_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_reduce(int dtype, const void* src, int64_t rows, int64_t cols, int64_t ld, int dim, int kind, int clear, void* dst, float* partial, int slices,
                         hipStream_t s) {
  switch (dtype) {
    case FRISK_F32: return reduce_k<FRISK_F32>(kind, src, rows, cols, ld, dim, clear, dst, partial, slices, s);
    case FRISK_F16: return reduce_k<FRISK_F16>(kind, src, rows, cols, ld, dim, clear, dst, partial, slices, s);
    default: return reduce_k<FRISK_BF16>(kind, src, rows, cols, ld, dim, clear, dst, partial, slices, s);
  }
}

}  // namespace frisk
