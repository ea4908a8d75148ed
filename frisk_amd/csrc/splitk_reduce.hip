// Second pass of a split-K GEMM: sums the raw 32-bit accumulators the K slices
// left in the workspace ([slice][M][N], row length N) and applies what the
// single-pass epilogue applies: integer output as is, otherwise (x * scaleA) *
// scaleB with two separately rounded multiplies, then accumulate-into-C, then
// the conversion to the output type.  A thread owns 4 consecutive columns.
//
// What bounds it is latency: a launch, a trip to memory for the slices and one for the stores.  So every lane has one quad, its place in C takes
// 32-bit divisions, up to eight slices are under way together with the scales and the old C, and a quad leaves in one store.
#include <hip/hip_runtime.h>
#include "gemm_internal.h"

namespace frisk {

// four columns of the partial sums, of 32-bit and of 16-bit C: one instruction wherever their row starts
typedef int r_v4i __attribute__((ext_vector_type(4)));
typedef int r_v4i_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t r_v4h __attribute__((ext_vector_type(4)));
typedef uint16_t r_v4h_any __attribute__((ext_vector_type(4), aligned(2)));

// What a quad of C at row m, columns n .. n + valid - 1 (valid <= 4) needs beside its sums, fetched ahead of them.
struct Beside {
  float sa, sb[4];
  r_v4i old;  // old C as it is stored: 32-bit values, or 16-bit ones in the low halves

  __device__ __forceinline__ void fetch(const GemmParams& p, int64_t m, int64_t n, int valid) {
    sa = 1.f;
    if (p.epilogue == FRISK_EPI_TENSOR_SCALE) {
      sa = p.scaleA[0];
      sb[0] = sb[1] = sb[2] = sb[3] = p.scaleB[0];
    } else if (p.epilogue == FRISK_EPI_ROW_COL_SCALE) {
      sa = p.scaleA[m];
#pragma unroll
      for (int e = 0; e < 4; ++e) sb[e] = p.scaleB[n + (e < valid ? e : 0)];
    }
    old = r_v4i{0, 0, 0, 0};
    if (!p.accumulate) return;
    const int64_t at = m * p.ldc + n;
    if (p.dtype_out == FRISK_F16 || p.dtype_out == FRISK_BF16) {
      const uint16_t* q = (const uint16_t*)p.C + at;
      if (valid == 4) {
        const r_v4h v = *(const r_v4h_any*)q;
        old = r_v4i{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e) if (e < valid) old[e] = q[e];
      }
    } else {
      const int* q = (const int*)p.C + at;
      if (valid == 4) old = *(const r_v4i_any*)q;
      else {
#pragma unroll
        for (int e = 0; e < 3; ++e) if (e < valid) old[e] = q[e];
      }
    }
  }
};

// scales, accumulation, conversion and the store of a quad whose slices sum to `sum` (integers, or the bits of floats)
template <bool INT_ACC> __device__ __forceinline__ void finish_quad(const GemmParams& p, const Beside& b, const r_v4i& sum, int64_t m, int64_t n, int valid) {
  const int64_t at = m * p.ldc + n;
  r_v4i out;
  if (INT_ACC && p.dtype_out == FRISK_I32) {
    out = sum + b.old;
  } else {
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = sum[e];  // copy first: bit_cast applied to a vector element reads element 0
      x[e] = INT_ACC ? (float)t : __builtin_bit_cast(float, t);
    }
    if (p.epilogue != FRISK_EPI_NONE) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = (x[e] * b.sa) * b.sb[e];
        asm volatile("" : "+v"(x[e]));  // rounded to fp32 before what follows
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int o = b.old[e];
      if (p.dtype_out == FRISK_F16) {
        if (p.accumulate) x[e] += (float)__builtin_bit_cast(_Float16, (uint16_t)o);
        out[e] = __builtin_bit_cast(uint16_t, (_Float16)x[e]);
      } else if (p.dtype_out == FRISK_BF16) {
        if (p.accumulate) x[e] += (float)__builtin_bit_cast(__bf16, (uint16_t)o);
        out[e] = __builtin_bit_cast(uint16_t, (__bf16)x[e]);
      } else {
        if (p.accumulate) x[e] += __builtin_bit_cast(float, o);
        out[e] = __builtin_bit_cast(int, x[e]);
      }
    }
  }
  if (p.dtype_out == FRISK_F16 || p.dtype_out == FRISK_BF16) {
    uint16_t* q = (uint16_t*)p.C + at;
    if (valid == 4) *(r_v4h_any*)q = r_v4h{(uint16_t)out[0], (uint16_t)out[1], (uint16_t)out[2], (uint16_t)out[3]};
    else {
#pragma unroll
      for (int e = 0; e < 3; ++e) if (e < valid) q[e] = (uint16_t)out[e];
    }
  } else {
    int* q = (int*)p.C + at;
    if (valid == 4) *(r_v4i_any*)q = out;
    else {
#pragma unroll
      for (int e = 0; e < 3; ++e) if (e < valid) q[e] = out[e];
    }
  }
}

template <bool INT_ACC> __device__ __forceinline__ void add_quad(r_v4i& sum, const r_v4i& t) {
  if (INT_ACC) sum += t;
  else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int a = sum[e], b = t[e];
      sum[e] = __builtin_bit_cast(int, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b));
    }
  }
}

// a quad of COUNT slices, added in slice order
template <bool INT_ACC, int COUNT> __device__ __forceinline__ void sum_slices(r_v4i& sum, const int* src, size_t slice) {
  r_v4i t[COUNT];
#pragma unroll
  for (int i = 0; i < COUNT; ++i) t[i] = *(const r_v4i_any*)(src + i * slice);
#pragma unroll
  for (int i = 0; i < COUNT; ++i) add_quad<INT_ACC>(sum, t[i]);
}

// WIDE: more quads than 32-bit ids count
template <bool INT_ACC, bool WIDE> __global__ void __launch_bounds__(256) splitk_reduce_kernel(GemmParams p) {
  const unsigned quads_per_row = ((unsigned)p.N + 3) / 4;
  int64_t m, n;
  if constexpr (WIDE) {
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    m = id / quads_per_row;
    n = (id - m * quads_per_row) * 4;
  } else {
    const unsigned id = blockIdx.x * 256 + threadIdx.x, row = id / quads_per_row;
    m = row;
    n = (id - row * quads_per_row) * 4;
  }
  if (m >= p.M) return;
  const int valid = p.N - n < 4 ? (int)(p.N - n) : 4;
  Beside beside;
  beside.fetch(p, m, n, valid);
  const size_t slice = (size_t)p.M * (size_t)p.N;
  r_v4i sum = {0, 0, 0, 0};
  const int* src = (const int*)p.partial + (size_t)m * p.N + n;
  if (valid == 4) {
    // the slices' quads are fetched eight at a time and then added in slice order: one memory latency per eight slices instead
    // of one per slice (16 slices of a 256 x 256 result: 9.9 -> 4.4 us in a kernel trace), the same sum
    int left = p.split_k;
    for (; left >= 8; left -= 8) { sum_slices<INT_ACC, 8>(sum, src, slice); src += 8 * slice; }
    switch (left) {
      case 7: sum_slices<INT_ACC, 7>(sum, src, slice); break;
      case 6: sum_slices<INT_ACC, 6>(sum, src, slice); break;
      case 5: sum_slices<INT_ACC, 5>(sum, src, slice); break;
      case 4: sum_slices<INT_ACC, 4>(sum, src, slice); break;
      case 3: sum_slices<INT_ACC, 3>(sum, src, slice); break;
      case 2: sum_slices<INT_ACC, 2>(sum, src, slice); break;
      case 1: sum_slices<INT_ACC, 1>(sum, src, slice); break;
    }
  } else {
    for (int z = 0; z < p.split_k; ++z, src += slice) {
      r_v4i t = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 3; ++e) if (e < valid) t[e] = src[e];
      add_quad<INT_ACC>(sum, t);
    }
  }
  finish_quad<INT_ACC>(p, beside, sum, m, n, valid);
}

// The tiles of a tail split in SLICES slices: partial[slice][tail tile][BM][BN], the tile's place in C from the same id mapping as the GEMM
// kernel's.  A quad a lane: with four one after the other, on a quarter of the work-groups, 4 tiles of 256 x 256 in 8 slices took 9.6 us in a kernel
// trace.
template <bool INT_ACC, int SLICES> __global__ void __launch_bounds__(256) tail_reduce_kernel(GemmParams p) {
  const unsigned BM = (unsigned)p.tile_m, BN = (unsigned)p.tile_n, quads_per_row = BN / 4;
  const int t = blockIdx.y;
  int tm, tn;
  tile_of_workgroup(p.tail_from + t, p.tiles_m, p.tiles_n, p.group_m, p.xcd_remap, tm, tn);
  const size_t tile_elems = (size_t)BM * BN;
  const unsigned id = blockIdx.x * 256 + threadIdx.x, r = id / quads_per_row, c = (id - r * quads_per_row) * 4;
  const int64_t m = (int64_t)tm * BM + r, n = (int64_t)tn * BN + c;
  if (r >= BM || m >= p.M || n >= p.N) return;
  const int valid = p.N - n < 4 ? (int)(p.N - n) : 4;
  r_v4i v[SLICES], sum = {0, 0, 0, 0};  // all fetched before the first addition, added in slice order
  const int* src = (const int*)p.partial + (size_t)t * tile_elems + (size_t)r * BN + c;
#pragma unroll
  for (int z = 0; z < SLICES; ++z) v[z] = *(const r_v4i*)(src + (size_t)z * p.tail_tiles * tile_elems);
  Beside beside;
  beside.fetch(p, m, n, valid);
#pragma unroll
  for (int z = 0; z < SLICES; ++z) add_quad<INT_ACC>(sum, v[z]);
  finish_quad<INT_ACC>(p, beside, sum, m, n, valid);
}

template <bool INT_ACC> hipError_t launch_tail(const GemmParams& p, hipStream_t stream) {
  const int quads = p.tile_m * p.tile_n / 4;
  const dim3 grid((unsigned)((quads + 255) / 256), (unsigned)p.tail_tiles);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, p); return hipGetLastError(); };
  switch (p.tail_split) {
    case 2: return launch(tail_reduce_kernel<INT_ACC, 2>);
    case 3: return launch(tail_reduce_kernel<INT_ACC, 3>);
    case 4: return launch(tail_reduce_kernel<INT_ACC, 4>);
    case 5: return launch(tail_reduce_kernel<INT_ACC, 5>);
    case 6: return launch(tail_reduce_kernel<INT_ACC, 6>);
    case 7: return launch(tail_reduce_kernel<INT_ACC, 7>);
    case 8: return launch(tail_reduce_kernel<INT_ACC, 8>);
    default: return hipErrorInvalidValue;
  }
}
hipError_t launch_tail_reduce(const GemmParams& p, int acc_is_int, hipStream_t stream) { return acc_is_int ? launch_tail<true>(p, stream) : launch_tail<false>(p, stream); }

hipError_t launch_splitk_reduce(const GemmParams& p, int acc_is_int, hipStream_t stream) {
  const int64_t quads = (((int64_t)p.N + 3) / 4) * p.M;
  const unsigned blocks = (unsigned)((quads + 255) / 256);
  const bool wide = quads + 255 > UINT32_MAX;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, p); };
  if (acc_is_int) wide ? launch(splitk_reduce_kernel<true, true>) : launch(splitk_reduce_kernel<true, false>);
  else wide ? launch(splitk_reduce_kernel<false, true>) : launch(splitk_reduce_kernel<false, false>);
  return hipGetLastError();
}

}  // namespace frisk
