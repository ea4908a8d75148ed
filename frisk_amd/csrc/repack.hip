// Copies an operand whose rows do not start on 16-byte boundaries (an odd leading dimension, a pointer inside a row) to a workspace
// where they do, so that the product can run on the kernels that move operands straight into LDS in 16-byte chunks.  Bound by
// memory traffic: every byte is read once and written once, 16 at a time on both sides; the loads need no alignment
// (global_load_dwordx4 takes any address), a row's last chunk is loaded so that it ends with the row and shifted into place.
// fp16 1999x4099x3001 NN, both operands copied (37 MB): 465 us without it on element-wise loads, 154 us staged through registers,
// 74.8 us with the copy.
#include <hip/hip_runtime.h>
#include "gemm_internal.h"

namespace frisk {
namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));
constexpr int kRowsPerLane = 4;  // loads in flight per lane

// 2^lanes_log2 lanes walk a row, 256 >> lanes_log2 rows side by side, kRowsPerLane of such sets per work-group
__global__ void __launch_bounds__(256) repack_kernel(RepackParams p, unsigned blocks_a, int lanes_log2_a, int lanes_log2_b) {
  const bool is_b = blockIdx.x >= blocks_a;
  const RepackParams::Side s = is_b ? p.b : p.a;
  const int lanes_log2 = is_b ? lanes_log2_b : lanes_log2_a, lanes = 1 << lanes_log2, rows_per_set = 256 >> lanes_log2;
  const int64_t row0 = (int64_t)(is_b ? blockIdx.x - blocks_a : blockIdx.x) * rows_per_set * kRowsPerLane + (threadIdx.x >> lanes_log2);
  const int64_t chunks = s.dst_ld / 16;
  for (int64_t c = threadIdx.x & (lanes - 1); c < chunks; c += lanes) {
    const int64_t left = s.row_bytes - c * 16;
    const int over = left >= 16 ? 0 : 16 - (int)left;
    v4u v[kRowsPerLane];
    if (s.row_bytes >= 16) {
#pragma unroll
      for (int u = 0; u < kRowsPerLane; ++u) {
        const int64_t r = row0 + u * rows_per_set;
        if (r < s.rows) __builtin_memcpy(&v[u], (const char*)s.src + r * s.src_ld + c * 16 - over, 16);
      }
    } else {  // rows shorter than a chunk: bytes
#pragma unroll
      for (int u = 0; u < kRowsPerLane; ++u) {
        const int64_t r = row0 + u * rows_per_set;
        v[u] = v4u{0, 0, 0, 0};
        if (r < s.rows)
          for (int e = 0; e < (int)s.row_bytes; ++e) v[u][e >> 2] |= (unsigned)((const unsigned char*)s.src)[r * s.src_ld + e] << (8 * (e & 3));
      }
    }
#pragma unroll
    for (int u = 0; u < kRowsPerLane; ++u) {
      const int64_t r = row0 + u * rows_per_set;
      if (over > 0 && s.row_bytes >= 16) v[u] = __builtin_bit_cast(v4u, __builtin_bit_cast(unsigned __int128, v[u]) >> (over * 8));
      if (r < s.rows) *(v4u*)((char*)s.dst + r * s.dst_ld + c * 16) = v[u];
    }
  }
}

}  // namespace

hipError_t launch_repack(const RepackParams& p, hipStream_t stream) {
  auto lanes_of = [](const RepackParams::Side& s) {
    int l = 0;
    while (l < 8 && ((int64_t)1 << l) < s.dst_ld / 16) ++l;
    return l;
  };
  const int la = lanes_of(p.a), lb = lanes_of(p.b);
  auto blocks_of = [](const RepackParams::Side& s, int l) { const int64_t per = (int64_t)(256 >> l) * kRowsPerLane; return (s.rows + per - 1) / per; };
  const int64_t ba = blocks_of(p.a, la), bb = blocks_of(p.b, lb);
  hipLaunchKernelGGL(repack_kernel, dim3((unsigned)(ba + bb)), dim3(256), 0, stream, p, (unsigned)ba, la, lb);
  return hipGetLastError();
}

}  // namespace frisk
