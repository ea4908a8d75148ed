// What the library would launch, on a machine without a GPU: the calls of the HIP runtime that the library makes are defined here, in the executable, where the
// loader finds them first, and print what they are asked for instead.  Pointers are made up; nothing reads them.
//
//   launch_recorder gemm keep|nokeep <dtype> <M> <N> <K> <transA> <transB> <workspace bytes>
//   launch_recorder kept
//   launch_recorder block <dtype> <rows> <cols> <operands: m = rows x cols, r = one value a row, s = that times a constant, c = one a column>
//   launch_recorder reduce <dtype> <rows> <cols> <leading dimension> <dim> <bytes from the source to a 256-byte boundary> <workspace: 1 what the library asks for, 0 none>
//   launch_recorder softmax <dtype> <rows> <cols> <leading dimension> <bytes from either matrix to a 256-byte boundary>
#include <hip/hip_runtime_api.h>
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include "frisk_hip.h"

static bool g_keep = true, g_quiet = false;

static std::map<const void*, std::string>& kernel_names() {
  static auto* names = new std::map<const void*, std::string>;
  return *names;
}

extern "C" {
static struct { dim3 grid, block; size_t lds; hipStream_t stream; } g_pushed;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) { g_pushed = {grid, block, lds, stream}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
  *grid = g_pushed.grid; *block = g_pushed.block; *lds = g_pushed.lds; *stream = g_pushed.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  if (g_quiet) return hipSuccess;
  const auto name = kernel_names().find(kernel);
  std::printf("launch %s %u %u %u %u\n", name != kernel_names().end() ? name->second.c_str() : "?", grid.x, grid.y, grid.z, block.x);
  return hipSuccess;
}
// (called as the library is loaded: kernels of anonymous namespaces have no name that dladdr finds)
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) { kernel_names()[host] = name; }
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) { std::memset(p, 0, sizeof *p); std::strcpy(p->gcnArchName, "gfx950"); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
}
// the storage of the plans that a thread keeps
void* operator new[](size_t n, const std::nothrow_t&) noexcept { return g_keep ? std::malloc(n) : nullptr; }
void operator delete[](void* p) noexcept { std::free(p); }

static void* at(int i) { return (void*)((size_t)1 << (32 + i)); }

static int gemm(char** arg) {
  g_keep = !std::strcmp(arg[0], "keep");
  frisk_gemm_desc d{};
  d.abi_version = FRISK_HIP_ABI_VERSION;
  d.dtype_ab = std::atoi(arg[1]);
  d.dtype_acc = d.dtype_ab == FRISK_I8 ? FRISK_I32 : FRISK_F32;
  d.dtype_out = d.dtype_ab == FRISK_I8 ? FRISK_I32 : d.dtype_ab == FRISK_E4M3 ? FRISK_BF16 : d.dtype_ab;
  d.M = std::atoll(arg[2]); d.N = std::atoll(arg[3]); d.K = std::atoll(arg[4]);
  d.transA = std::atoi(arg[5]); d.transB = std::atoi(arg[6]);
  d.lda = d.transA ? d.M : d.K; d.ldb = d.transB ? d.K : d.N; d.ldc = d.N;
  d.clear_accum = 1;
  const size_t bytes = (size_t)std::atoll(arg[7]);
  const int st = frisk_hip_gemm(&d, at(0), at(1), at(2), nullptr, nullptr, bytes ? at(3) : nullptr, bytes, nullptr);
  std::printf("status %d\n", st);
  return 0;
}

// nanoseconds of a call, the least of many rounds: one call over and over; the same shape in turn on two leading dimensions, output types and pointer alignments,
// the median of seven shapes (two plans in 64 places may still meet); a shape that comes round too late to be kept
static int kept() {
  g_quiet = true;
  frisk_gemm_desc base{};
  base.abi_version = FRISK_HIP_ABI_VERSION;
  base.dtype_ab = FRISK_F16; base.dtype_acc = FRISK_F32; base.dtype_out = FRISK_F16;
  base.M = 48; base.N = 4096; base.K = 4096;
  base.lda = base.K; base.ldb = base.ldc = base.N;
  base.clear_accum = 1;
  auto least = [](auto call) {
    double best = 1e9;
    for (int round = 0; round < 40; ++round) {
      const auto t0 = std::chrono::steady_clock::now();
      for (int i = 0; i < 200; ++i) call(i);
      best = std::min(best, std::chrono::duration<double, std::nano>(std::chrono::steady_clock::now() - t0).count() / 200);
    }
    return best;
  };
  auto pair = [&](const char* what, auto change, size_t off) {
    double ns[7];
    for (int k = 0; k < 7; ++k) {
      frisk_gemm_desc one = base, other = base;
      one.M = other.M = 41 + k;
      change(other);
      ns[k] = least([&](int i) { frisk_hip_gemm(i & 1 ? &other : &one, (char*)at(0) + (i & 1 ? off : 0), at(1), at(2), nullptr, nullptr, nullptr, 0, nullptr); });
    }
    std::sort(ns, ns + 7);
    std::printf("%s %.1f\n", what, ns[3]);
  };
  pair("again", [](frisk_gemm_desc&) {}, 0);
  pair("lda", [](frisk_gemm_desc& d) { d.lda += 8; }, 0);
  pair("ldb", [](frisk_gemm_desc& d) { d.ldb += 8; }, 0);
  pair("ldc", [](frisk_gemm_desc& d) { d.ldc += 8; }, 0);
  pair("dtype_out", [](frisk_gemm_desc& d) { d.dtype_out = FRISK_F32; }, 0);
  pair("alignment", [](frisk_gemm_desc&) {}, 2);
  int n = 0;
  std::printf("new %.1f\n", least([&](int) { frisk_gemm_desc d = base; d.M = 33 + n++ % 32; d.N += 64 * (n % 97); d.ldb = d.ldc = d.N; frisk_hip_gemm(&d, at(0), at(1), at(2), nullptr, nullptr, nullptr, 0, nullptr); }));
  return 0;
}

static int block(char** arg) {
  frisk_elementwise_desc d{};
  const std::string operands = arg[3];
  d.abi_version = FRISK_HIP_ABI_VERSION;
  d.out_dtype = std::atoi(arg[0]);
  d.rows = std::atoll(arg[1]); d.cols = d.out_ld = std::atoll(arg[2]);
  d.n_inputs = (int)operands.size();
  const void* in[FRISK_EW_MAX_INPUTS] = {};
  for (int k = 0; k < d.n_inputs; ++k) {  // x, then + or * the next operand
    in[k] = at(k);
    d.in_dtype[k] = d.out_dtype;
    const bool of_row = operands[k] == 'r' || operands[k] == 's';
    d.in_row_stride[k] = operands[k] == 'm' ? d.cols : of_row;
    d.in_col_stride[k] = !of_row;
    d.op[d.n_ops] = FRISK_EW_INPUT;
    d.arg[d.n_ops++] = k;
    if (operands[k] == 's') {
      d.op[d.n_ops] = FRISK_EW_CONST;
      d.imm[d.n_ops++] = 0.5f;
      d.op[d.n_ops++] = FRISK_EW_MUL;
    }
    if (k) d.op[d.n_ops++] = k & 1 ? FRISK_EW_ADD : FRISK_EW_MUL;
  }
  std::printf("status %d\n", frisk_hip_elementwise(&d, in, at(8), nullptr));
  return 0;
}

static int reduce(char** arg) {
  const int dtype = std::atoi(arg[0]), dim = std::atoi(arg[4]);
  const int64_t rows = std::atoll(arg[1]), cols = std::atoll(arg[2]);
  const size_t bytes = std::atoi(arg[6]) ? frisk_hip_reduce_workspace_bytes(dtype, rows, cols, dim) : 0;
  std::printf("status %d\n", frisk_hip_reduce(dtype, (char*)at(0) + std::atoi(arg[5]), rows, cols, std::atoll(arg[3]), dim, FRISK_REDUCE_ADD, 1, at(1), bytes ? at(3) : nullptr, bytes, nullptr));
  return 0;
}

static int softmax(char** arg) {
  const int dtype = std::atoi(arg[0]);
  const int64_t rows = std::atoll(arg[1]), cols = std::atoll(arg[2]), ld = std::atoll(arg[3]);
  std::printf("status %d\n", frisk_hip_softmax(dtype, (char*)at(0) + std::atoi(arg[4]), ld, (char*)at(1) + std::atoi(arg[4]), ld, rows, cols, 1.f, nullptr, nullptr, 0, nullptr));
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "gemm" && argc == 10) return gemm(argv + 2);
  if (what == "kept") return kept();
  if (what == "reduce" && argc == 9) return reduce(argv + 2);
  if (what == "softmax" && argc == 7) return softmax(argv + 2);
  if (what == "block" && argc == 6) return block(argv + 2);
  return 2;
}
