// Row softmax in base 2: y[r][j] = 2^(c x[r][j]) / sum_j 2^(c x[r][j]), the kernel the reference sketches as
// @online_softmax (tmp/ir.mlir:21-66): per row, chunks of 1024 go through frisk.copy, frisk.reduce max, a frisk.block
// of exp2(x * cst - max * cst), frisk.reduce sum and a running log-sum (:33-57), then a second sweep writes
// exp2(x * cst - lse) (:58-68).  Here rows of up to 256 groups of 16 bytes (2048 f16) are shared by 1 to 64 lanes of one
// wave and combined by shuffles; longer rows get a work-group of 256 or 512 lanes each.  Rows of up to 4096 groups (32768 f16, 16384 f32) are
// read once and held in registers (maximum, exponentials, sum, scaling: one read and one write of HBM per element);
// longer rows take the sketch's two sweeps with a running maximum and sum per lane, the second sweep re-reading x.
// A lane moves 16 bytes at a time, wherever the rows start.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "tile_ops.h"

namespace frisk {
namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));
// 16 bytes that start on any element: loads and stores of this type are one instruction at any address
typedef unsigned v4u_any __attribute__((ext_vector_type(4), aligned(2)));

template <int DT> struct SElem;
template <> struct SElem<FRISK_F32> { typedef float T; static __device__ float load(const T& x) { return x; } static __device__ T store(float x) { return x; } };
template <> struct SElem<FRISK_F16> { typedef _Float16 T; static __device__ float load(const T& x) { return (float)x; } static __device__ T store(float x) { return (_Float16)x; } };
template <> struct SElem<FRISK_BF16> { typedef __bf16 T; static __device__ float load(const T& x) { return (float)x; } static __device__ T store(float x) { return (__bf16)x; } };

// group g (G elements, 16 bytes) of a row of cols elements as floats times c; -inf beyond the row
template <int DT, bool STREAMED> __device__ __forceinline__ void load_group(const typename SElem<DT>::T* x, int64_t g, int64_t cols, float c, float (&v)[16 / sizeof(typename SElem<DT>::T)]) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  const int64_t left = cols - g * G;
  T in[G];
  if (left >= G) {
    if constexpr (STREAMED) *(v4u*)in = __builtin_nontemporal_load((const v4u_any*)(x + g * G));
    else *(v4u*)in = *(const v4u_any*)(x + g * G);
#pragma unroll
    for (int e = 0; e < G; ++e) v[e] = SElem<DT>::load(in[e]) * c;
  } else {
#pragma unroll
    for (int e = 0; e < G; ++e) v[e] = e < left ? SElem<DT>::load(x[g * G + e]) * c : -INFINITY;
  }
}
template <int DT> __device__ __forceinline__ void store_group(typename SElem<DT>::T* y, int64_t g, int64_t cols, const float (&v)[16 / sizeof(typename SElem<DT>::T)]) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  const int64_t left = cols - g * G;
  T out[G];
#pragma unroll
  for (int e = 0; e < G; ++e) out[e] = SElem<DT>::store(v[e]);
  if (left >= G) __builtin_nontemporal_store(*(const v4u*)out, (v4u_any*)(y + g * G));
  else {
#pragma unroll
    for (int e = 0; e < G; ++e)
      if (e < left) y[g * G + e] = out[e];
  }
}

// (maximum, sum of 2^(v - maximum)) pairs combine associatively
struct MaxSum {
  float m, l;
  __device__ void add(float v) {
    // a masked element (-inf) adds nothing; without the test an all-masked prefix would compute 2^(-inf - -inf)
    if (v == -INFINITY) return;
    if (v > m) { l = l * __builtin_amdgcn_exp2f(m - v) + 1.f; m = v; }
    else l += __builtin_amdgcn_exp2f(v - m);
  }
  __device__ void merge(const MaxSum& o) {
    const float nm = fmaxf(m, o.m);
    // an empty partner has m = -inf, l = 0: its term must not become 0 * 2^(-inf - -inf)
    const float a = m == nm ? l : l * __builtin_amdgcn_exp2f(m - nm), b = o.m == nm ? o.l : o.l * __builtin_amdgcn_exp2f(o.m - nm);
    m = nm;
    l = a + b;
  }
};

__device__ __forceinline__ MaxSum block_merge(MaxSum v, float* lds) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    MaxSum o;
    o.m = __shfl_xor(v.m, off);
    o.l = __shfl_xor(v.l, off);
    v.merge(o);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { lds[2 * wave] = v.m; lds[2 * wave + 1] = v.l; }
  __syncthreads();
  MaxSum r = {lds[0], lds[1]};
#pragma unroll
  for (int w = 1; w < 4; ++w) r.merge(MaxSum{lds[2 * w], lds[2 * w + 1]});
  __syncthreads();
  return r;
}

// the maximum (SUM false) or the sum of a value of every lane of the work-group; `lds`: a float per wave that nothing else has touched since the last barrier
template <bool SUM, int THREADS> __device__ __forceinline__ float block_all(float v, float* lds) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float o = __shfl_xor(v, off);
    v = SUM ? v + o : fmaxf(v, o);
  }
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = lds[0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; ++w) r = SUM ? r + lds[w] : fmaxf(r, lds[w]);
  return r;
}

// Rows of 257 to 4096 groups, a work-group each, NPT groups a lane in registers.  A row's last group, where it is not whole, is read and written together with the
// elements before it that fill it up (which enter the sum as their own lane's): every access is 16 bytes of the row and all loads of a row are under way
// together.  Fetched element by element behind the others, that group held up every row by a memory latency: us before / now, f16 10069 x 4946 49.5 / 33.7,
// 2490 x 2453 11.8 / 6.9, 870 x 16370 20.0 / 10.4 (with 512 lanes: 12.5 with 256), f32 5531 x 1315 17.6 / 10.6, 394 x 9229 (two launches before) 11.9 / 6.9;
// rows that are whole groups gain by the shorter reductions, f16 8192 x 8192 47.3 / 43.0, which a plain copy takes 39 for.
// HELD: rows of whole groups on 16-byte boundaries know of no other group.  On 128-byte lines and up to 56 MiB they are read past the caches (f16 4096 x 4096 out of the last-level cache 10.6 us through
// the caches, 9.0 past them, f32 3000 x 4096 15.5 / 13.4), beyond through them (4096 x 8192 20.6 us, 23.2 past them), and past them again where the last-level cache does not hold the view beside its result (8192 x 8192
// behind the pass that wrote it 43.9 through them, 43.0 past them).  Others are read through the caches (870 x 16370 10.4,
// 11.9 past them), and past them in views that the last-level cache does not hold beside their result; there, where rows start off 16-byte boundaries, the groups start at the first boundary, what lies
// before it being a group that overlaps like the last one: stores that cross lines half way cost memory traffic (4426 x 15161 f16 54.9 at the rows' starts, 47.5 so; out of the cache 7.1 either way, 545 x 12163).
enum HeldRows { HELD_WHOLE_PAST, HELD_WHOLE, HELD_CACHED, HELD_FROM_BOUNDARY };
template <int DT, int NPT, int THREADS, int HELD>
__global__ void __launch_bounds__(THREADS) softmax_held_rows_kernel(const typename SElem<DT>::T* src, int64_t sld, typename SElem<DT>::T* dst, int64_t dld, int64_t rows,
                                                                    int cols, float c, float* lse) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  __shared__ float lds[2][THREADS / 64];  // one row's sum is read before the next row's maximum has passed its barrier
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const T* x = src + r * sld;
    T* y = dst + r * dld;
    // groups 0 .. full - 1 from element `head` on, then the one that ends with the row, then the one it starts with
    const int head = HELD == HELD_FROM_BOUNDARY ? (int)((0 - (uintptr_t)y) & 15) / (int)sizeof(T) : 0;
    const int full = (cols - head) / G, body = head + full * G, tail = HELD <= HELD_WHOLE ? 0 : cols - body, groups = full + (tail > 0) + (head > 0);
    T in[NPT][G];
    int at[NPT];
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
      const int g = q * THREADS + (int)threadIdx.x;
      at[q] = g < full ? head + g * G : (tail > 0 && g == full ? cols - G : 0);
      if (g < groups) {
        if constexpr (HELD == HELD_CACHED || HELD == HELD_WHOLE) *(v4u*)in[q] = *(const v4u_any*)(x + at[q]);
        else *(v4u*)in[q] = __builtin_nontemporal_load((const v4u_any*)(x + at[q]));
      }
    }
    float v[NPT][G], mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NPT; ++q)
#pragma unroll
      for (int e = 0; e < G; ++e) {
        v[q][e] = q * THREADS + (int)threadIdx.x < groups ? SElem<DT>::load(in[q][e]) * c : -INFINITY;
        mx = fmaxf(mx, v[q][e]);
      }
    const float top = block_all<false, THREADS>(mx, lds[0]);
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
      const int g = q * THREADS + (int)threadIdx.x;
      // which elements of the group are its own
      const bool last = tail > 0 && g == full;
      const int lo = last ? G - tail : 0, hi = g < full || last ? G : head;
#pragma unroll
      for (int e = 0; e < G; ++e) {
        v[q][e] = __builtin_amdgcn_exp2f(v[q][e] - top);
        sum += g < groups && e >= lo && e < hi ? v[q][e] : 0.f;
      }
    }
    const float all = block_all<true, THREADS>(sum, lds[1]);
    const float inv = 1.f / all;
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
      T out[G];
#pragma unroll
      for (int e = 0; e < G; ++e) out[e] = SElem<DT>::store(v[q][e] * inv);
      if (q * THREADS + (int)threadIdx.x < groups) __builtin_nontemporal_store(*(const v4u*)out, (v4u_any*)(y + at[q]));
    }
    if (lse && threadIdx.x == 0) lse[r] = top + __builtin_amdgcn_logf(all);
  }
}

// Rows beyond that, a work-group each: two sweeps.
template <int DT>
__global__ void __launch_bounds__(256) softmax_rows_kernel(const typename SElem<DT>::T* src, int64_t sld, typename SElem<DT>::T* dst, int64_t dld, int64_t rows,
                                                           int64_t cols, float c, float* lse) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  const int64_t groups = (cols + G - 1) / G;
  __shared__ float lds[8];
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const T* x = src + r * sld;
    T* y = dst + r * dld;
    MaxSum acc = {-INFINITY, 0.f};
    for (int64_t g = threadIdx.x; g < groups; g += 256) {
      float v[G];
      load_group<DT, false>(x, g, cols, c, v);
#pragma unroll
      for (int e = 0; e < G; ++e) acc.add(v[e]);
    }
    const MaxSum all = block_merge(acc, lds);
    const float ref = all.m + __builtin_amdgcn_logf(all.l);  // log2 of the denominator
    for (int64_t g = threadIdx.x; g < groups; g += 256) {
      float v[G];
      load_group<DT, false>(x, g, cols, c, v);
#pragma unroll
      for (int e = 0; e < G; ++e) v[e] = __builtin_amdgcn_exp2f(v[e] - ref);
      store_group<DT>(y, g, cols, v);
    }
    if (lse && threadIdx.x == 0) lse[r] = ref;
  }
}

// Rows of at most 256 groups of 16 bytes: 2^lanes_log2 <= 64 lanes of one wave share a row, each holding up to NPT groups in
// registers, and combine maximum and sum by shuffles (no LDS, no barrier); a work-group holds 256 >> lanes_log2 rows.
// TAIL: rows of whole groups (with the code for another last group, of any length, f16 32768 x 512 17.7 us, 14.4 so, 100000 x 64 from memory 8.2 / 7.1, 8192 x 1024 8.0 / 6.5); with a last
// group that is read and written with the elements before it, which are another lane's (bf16 14242 x 790 beside the code for less than one 11.9 us, 10.5 so); of less than a group, element by element.
enum RowTail { TAIL_WHOLE, TAIL_PART, TAIL_NARROW };
template <int DT, int NPT, int TAIL>
__global__ void __launch_bounds__(256) softmax_short_rows_kernel(const typename SElem<DT>::T* src, int64_t sld, typename SElem<DT>::T* dst, int64_t dld, int64_t rows,
                                                                 int cols, float c, float* lse, int lanes_log2) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  const int lanes = 1 << lanes_log2, lane = threadIdx.x & (lanes - 1), rows_per_group = 256 >> lanes_log2;
  const int64_t blocks = (rows + rows_per_group - 1) / rows_per_group;
  for (int64_t rb = blockIdx.x; rb < blocks; rb += gridDim.x) {
    const int64_t r = rb * rows_per_group + (threadIdx.x >> lanes_log2);
    const bool live = r < rows;  // lanes of rows past the end still take part in the shuffles
    const T* x = src + r * sld;
    T* y = dst + r * dld;
    float v[NPT][G];
    T in[NPT][G];
    int at[NPT], twice[NPT];  // where a group starts, and how many of its elements are another lane's
    bool inside[NPT];
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
      const int c0 = (q * lanes + lane) * G;
      inside[q] = live && c0 < cols;
      twice[q] = TAIL == TAIL_PART && c0 + G > cols ? c0 + G - cols : 0;
      at[q] = c0 - twice[q];
      if (!inside[q]) continue;
      if constexpr (TAIL == TAIL_NARROW) {
#pragma unroll
        for (int e = 0; e < G; ++e) in[q][e] = x[e < cols ? e : 0];
      } else *(v4u*)in[q] = __builtin_nontemporal_load((const v4u_any*)(x + at[q]));
    }
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NPT; ++q)
#pragma unroll
      for (int e = 0; e < G; ++e) {
        v[q][e] = inside[q] && (TAIL != TAIL_NARROW || e < cols) ? SElem<DT>::load(in[q][e]) * c : -INFINITY;
        mx = fmaxf(mx, v[q][e]);
      }
    for (int off = lanes >> 1; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < NPT; ++q)
#pragma unroll
      for (int e = 0; e < G; ++e) {
        v[q][e] = __builtin_amdgcn_exp2f(v[q][e] - mx);
        sum += TAIL != TAIL_PART || e >= twice[q] ? v[q][e] : 0.f;
      }
    for (int off = lanes >> 1; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
    const float inv = 1.f / sum;
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
      if (!inside[q]) continue;
      T out[G];
#pragma unroll
      for (int e = 0; e < G; ++e) out[e] = SElem<DT>::store(v[q][e] * inv);
      if constexpr (TAIL == TAIL_NARROW) {
#pragma unroll
        for (int e = 0; e < G; ++e)
          if (e < cols) y[e] = out[e];
      } else __builtin_nontemporal_store(*(const v4u*)out, (v4u_any*)(y + at[q]));
    }
    if (lse && live && lane == 0) lse[r] = mx + __builtin_amdgcn_logf(sum);
  }
}

// A few very long rows: a row is dealt to gridDim.y work-groups in runs of 256 groups (neighbouring work-groups read
// neighbouring memory).  First launch: every work-group leaves the (maximum, sum) of its share in partial[row][slice];
// second launch: every work-group merges the row's pairs and writes its share of exp2(x * c - log-sum).  Two reads and
// one write per element, as in the two sweeps above, but on rows x slices work-groups instead of rows.
template <int DT>
__global__ void __launch_bounds__(256) softmax_split_stats_kernel(const typename SElem<DT>::T* src, int64_t sld, int64_t cols, float c, float* partial) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  __shared__ float lds[8];
  const T* x = src + (int64_t)blockIdx.x * sld;
  MaxSum acc = {-INFINITY, 0.f};
  for (int64_t g = (int64_t)blockIdx.y * 256 + threadIdx.x; g * G < cols; g += (int64_t)gridDim.y * 256) {
    float v[G];
    load_group<DT, false>(x, g, cols, c, v);
#pragma unroll
    for (int e = 0; e < G; ++e) acc.add(v[e]);
  }
  const MaxSum all = block_merge(acc, lds);
  if (threadIdx.x == 0) {
    float* out = partial + ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * 2;
    out[0] = all.m;
    out[1] = all.l;
  }
}

template <int DT>
__global__ void __launch_bounds__(256) softmax_split_write_kernel(const typename SElem<DT>::T* src, int64_t sld, typename SElem<DT>::T* dst, int64_t dld, int64_t cols,
                                                                  float c, float* lse, const float* partial) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  __shared__ float lds[8];
  const T* x = src + (int64_t)blockIdx.x * sld;
  T* y = dst + (int64_t)blockIdx.x * dld;
  MaxSum acc = {-INFINITY, 0.f};
  for (int k = threadIdx.x; k < (int)gridDim.y; k += 256) {
    const float* in = partial + ((int64_t)blockIdx.x * gridDim.y + k) * 2;
    acc.merge(MaxSum{in[0], in[1]});
  }
  const MaxSum all = block_merge(acc, lds);
  const float ref = all.m + __builtin_amdgcn_logf(all.l);  // log2 of the denominator
  for (int64_t g = (int64_t)blockIdx.y * 256 + threadIdx.x; g * G < cols; g += (int64_t)gridDim.y * 256) {
    float v[G];
    load_group<DT, true>(x, g, cols, c, v);
#pragma unroll
    for (int e = 0; e < G; ++e) v[e] = __builtin_amdgcn_exp2f(v[e] - ref);
    store_group<DT>(y, g, cols, v);
  }
  if (lse && blockIdx.y == 0 && threadIdx.x == 0) lse[blockIdx.x] = ref;
}

// groups of a row that a work-group holds, bytes of a view from which on its rows stream past the caches (with the result they are most of the 256 MiB of
// the last-level cache), and bytes up to which rows of whole groups on lines do too
constexpr int64_t kHeldGroups = 4096, kStreamedBytes = (int64_t)112 << 20, kPastBytes = (int64_t)56 << 20;

template <int DT> hipError_t launch_typed(const void* src, int64_t sld, void* dst, int64_t dld, int64_t rows, int64_t cols, float c, float* lse, float* partial,
                                          int slices, hipStream_t s) {
  typedef typename SElem<DT>::T T;
  constexpr int G = 16 / (int)sizeof(T);
  const unsigned grid = (unsigned)(rows < 256 * 64 ? rows : 256 * 64);
  const T* x = (const T*)src;
  T* y = (T*)dst;
  const int64_t groups = (cols + G - 1) / G;
  if (slices > 1) {
    const dim3 sgrid((unsigned)rows, (unsigned)slices);
    hipLaunchKernelGGL((softmax_split_stats_kernel<DT>), sgrid, dim3(256), 0, s, x, sld, cols, c, partial);
    hipLaunchKernelGGL((softmax_split_write_kernel<DT>), sgrid, dim3(256), 0, s, x, sld, y, dld, cols, c, lse, (const float*)partial);
    return hipGetLastError();
  }
  if (groups <= 256) {
    int lanes_log2 = 0;
    while (lanes_log2 < 6 && (int64_t(1) << lanes_log2) < groups) ++lanes_log2;
    const int64_t rows_per_group = 256 >> lanes_log2, blocks = (rows + rows_per_group - 1) / rows_per_group;
    const dim3 sgrid((unsigned)(blocks < (1 << 22) ? blocks : (1 << 22)));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, sgrid, dim3(256), 0, s, x, sld, y, dld, rows, (int)cols, c, lse, lanes_log2); };
    const bool whole = cols % G == 0;
#define FRISK_SOFTMAX_SHORT(NPT) { if (whole) launch(softmax_short_rows_kernel<DT, NPT, TAIL_WHOLE>); else launch(softmax_short_rows_kernel<DT, NPT, TAIL_PART>); }
    if (cols < G) launch(softmax_short_rows_kernel<DT, 1, TAIL_NARROW>);
    else if (groups <= 64) FRISK_SOFTMAX_SHORT(1)
    else if (groups <= 128) FRISK_SOFTMAX_SHORT(2)
    else FRISK_SOFTMAX_SHORT(4)
#undef FRISK_SOFTMAX_SHORT
    return hipGetLastError();
  }
  if (groups <= kHeldGroups) {
    const int64_t bytes = rows * cols * (int64_t)sizeof(T);
    const uintptr_t starts = (uintptr_t)x | (uintptr_t)y | sld * sizeof(T) | dld * sizeof(T);
    const bool whole = cols % G == 0 && starts % 16 == 0, past = whole && (bytes > kStreamedBytes || (starts % 128 == 0 && bytes <= kPastBytes)), large = !whole && bytes > kStreamedBytes;
    const int64_t most = groups + (large ? 1 : 0);  // a row that starts off a boundary may have a group more
    auto launch = [&](auto kernel, int threads) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, s, x, sld, y, dld, rows, (int)cols, c, lse); };
#define FRISK_SOFTMAX_HELD(NPT, THREADS) \
  if (most <= NPT * THREADS) {                                                                          \
    if (past) launch(softmax_held_rows_kernel<DT, NPT, THREADS, HELD_WHOLE_PAST>, THREADS);             \
    else if (whole) launch(softmax_held_rows_kernel<DT, NPT, THREADS, HELD_WHOLE>, THREADS);            \
    else if (large) launch(softmax_held_rows_kernel<DT, NPT, THREADS, HELD_FROM_BOUNDARY>, THREADS);    \
    else launch(softmax_held_rows_kernel<DT, NPT, THREADS, HELD_CACHED>, THREADS);                      \
  }
    FRISK_SOFTMAX_HELD(2, 256)
    else FRISK_SOFTMAX_HELD(3, 256)
    else FRISK_SOFTMAX_HELD(2, 512)
    else FRISK_SOFTMAX_HELD(3, 512)
    else FRISK_SOFTMAX_HELD(4, 512)
    else FRISK_SOFTMAX_HELD(6, 512)
    else FRISK_SOFTMAX_HELD(9, 512)
#undef FRISK_SOFTMAX_HELD
  } else hipLaunchKernelGGL((softmax_rows_kernel<DT>), dim3(grid), dim3(256), 0, s, x, sld, y, dld, rows, cols, c, lse);
  return hipGetLastError();
}

}  // namespace

int softmax_slices(int dtype, int64_t rows, int64_t cols) {
  // Fewer than 1024 rows that a work-group cannot hold: split each so that about 1024 work-groups exist, each with at least 16 KiB.  (The others stay whole, in one launch, however few
  // they are: f32 64 x 16000 10.6 us in slices, 5.5 whole.)
  const int64_t row_bytes = cols * (dtype == FRISK_F32 ? 4 : 2);
  if (row_bytes <= kHeldGroups * 16) return 1;
  int slices = 1;
  while (rows * slices < 1024 && row_bytes / (slices * 2) >= 16384 && slices < 256) slices *= 2;
  return slices;
}

hipError_t launch_softmax_rows(int dtype, const void* src, int64_t sld, void* dst, int64_t dld, int64_t rows, int64_t cols, float scale_log2, float* lse,
                               float* partial, int slices, hipStream_t s) {
  switch (dtype) {
    case FRISK_F32: return launch_typed<FRISK_F32>(src, sld, dst, dld, rows, cols, scale_log2, lse, partial, slices, s);
    case FRISK_F16: return launch_typed<FRISK_F16>(src, sld, dst, dld, rows, cols, scale_log2, lse, partial, slices, s);
    default: return launch_typed<FRISK_BF16>(src, sld, dst, dld, rows, cols, scale_log2, lse, partial, slices, s);
  }
}

}  // namespace frisk
