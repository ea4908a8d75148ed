// The body of a frisk.block (include/Dialect/Frisk/IR/FriskOps.td:143-190; built by ffi/ir.cpp:383-394) run over a
// rank-2 iteration space: for every (row, col) evaluate an expression of loads, constants and arith / math ops and store
// the value.  The reference defines the op and lowers it nowhere.  Here the expression arrives as a postfix program (at
// most FRISK_EW_MAX_OPS steps over FRISK_EW_MAX_INPUTS operands) and ONE kernel interprets it: no run-time compilation.
//
// What bounds it is the vector pipe and the dispatch of a step, not memory, so the host first turns the postfix steps into steps of a
// machine with a top value: a binary operation whose right operand is an input or a constant takes it directly, and only a value
// that must survive goes below the top.  A lane evaluates 8 consecutive columns at a time.  The loop over the steps is written as inline
// assembly over fixed registers: a step is two lane reads of the program, a jump to its handler and 8 vector instructions in
// place, the operand picked by the register index mode.  (As a C++ switch the compiler joins the values of all cases after every
// step by register moves: 327 vector, 300 scalar and 120 branch instructions per group of 8 columns for (x - s * c) * g + b; here
// 109, 125 and 34.)  That body on 8192 x 8192 f16: 137 us before, 42.5 now on the same buffers, 49.4 with operands from memory (a plain copy: 38.8, 41.7); log2(max(x, c) / (x + c)), bound by
// the vector pipe in its division, 123 -> 69.5; x + y 80 -> 58; rows off 16-byte boundaries (4095 x 8191) 369 -> 29.
// Operands that are the same for every row stay in registers while the lane's columns do, values of one per row stay one
// register, and what the next groups need from memory is fetched while the current one is evaluated.  All arithmetic is
// fp32; the result is rounded once to the output type.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "tile_ops.h"

namespace frisk {
namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));
// 16 bytes that start on any element: loads and stores of this type are one instruction at any address
typedef unsigned v4u_any __attribute__((ext_vector_type(4), aligned(2)));
constexpr int V = 8;  // columns per lane and step

// The machine.  Registers of a lane, 8 columns each: top v[16:23] and the slots v[24 + 8 j : 31 + 8 j], which a step names by 8 j:
// below the top S0 (j = 0) and, in deep programs, S1 .. S4 (j = 5 .. 8); X (1) what a step fetched or a quotient's divisor; COL0, COL1
// (2, 3) operands that are the same for every row; WALK2 (4) the second operand that walks the rows.  v14, v15: values of one per row.
// A step is (handler << 24) | (input of STEP_FETCH << 8) | register index; constants lie beside it.  Suffix V: operand in a slot, S: constant,
// R: value of the row.  STEP_END .. STEP_DIV* leave the assembly; the quotient and the fetch are C++.
enum Step {
  STEP_END = 0, STEP_MORE, STEP_FETCH, STEP_DIVV, STEP_RDIVV, STEP_DIVS, STEP_DIVR,  // leave the assembly
  STEP_SAVE, STEP_LOADV, STEP_LOADS, STEP_LOADR, STEP_ADDV, STEP_ADDS, STEP_ADDR, STEP_SUBV, STEP_RSUBV, STEP_SUBR, STEP_MULV, STEP_MULS, STEP_MULR,
  STEP_MAXV, STEP_MAXS, STEP_MAXR, STEP_MINV, STEP_MINS, STEP_MINR, STEP_NEG, STEP_EXP2, STEP_LOG2
};
constexpr int kSlotS0 = 0, kSlotX = 8, kSlotCol0 = 16, kSlotCol1 = 24, kSlotWalk2 = 32, kSlotS1 = 40;
constexpr int kChunk = 64;  // steps in one register of a wave, one per lane; STEP_MORE goes on to the second register
// What an operand of one value per row goes through before the steps see it: value * mul + add, one operation with a constant (or none) whose other part changes
// nothing, so that it rounds once as that operation does.  Done on a row's value it is one instruction a group; as steps on eight columns a lane, with the value
// below the top kept meanwhile, it was four steps in place of one: (x - s c) g + b as steps / so, from memory, 8192 x 8192 f16 51.1 us / 49.4, bf16
// 3077 x 3724 12.4 / 11.5, 12208 x 658 12.4 / 10.9, 6199 x 10825 even (on the same buffers 49.6 / 44.5); f32, which memory bounds, even.  Programs without such a constant run on kernels without the multiply-add
// (HELD_ALL): under it they were 1 to 2 % slower, f16 100000 x 24 x g + y 6.9 us, 6.2 without, x s 6.0 / 5.6, 3168 x 2891 (x - s) g + b 13.65 / 13.3, x g + b 12.93 / 12.69, 4096 x 4096 15.15 / 14.95.
struct RowScale { float mul = 1.f, add = -0.f; };
struct EwSteps {
  int code[2 * kChunk];
  float imm[2 * kChunk];
  int n;                  // steps
  int depth;              // most values below the top at any time
  int head, walk2;        // operands fetched a group ahead: the one the program starts with, and another that walks the rows (-1: none)
  int col0, col1;         // operands that are the same for every row, kept in registers while the columns stay
  int row0, row1;         // operands of one value per row, fetched a group ahead
  RowScale scale0, scale1;
  bool scaled;            // either of them meets a constant
};
// An operand as the kernel addresses it, resolved on the host (an operand looked up by its number is a chain of dependent scalar loads).
struct EwOperand {
  const char* at;     // nullptr: none
  int64_t row_bytes;  // to the next row
  int dt, walks;      // walks: one element per column
};
struct EwArgs {
  int64_t rows, cols, out_row_bytes;
  char* out;
  int out_dt, n_steps;
  EwOperand head, walk2, row0, row1, col0, col1;
  EwOperand in[FRISK_EW_MAX_INPUTS];  // for STEP_FETCH, by number
  int code[2 * kChunk];
  float imm[2 * kChunk];
  RowScale scale0, scale1;  // HELD_SCALED
  int past;                 // halves: stores pass the caches
};

// ---- the interpreter loop.  EACH: one instruction per column.  Handlers lie 256 bytes apart, in the order of Step; NEXT fetches
// the step s51 counts and jumps to its handler.  s50 holds the step being run, s56 its constant.  (A lane select written by a scalar
// instruction, the index mode and a jump need no wait states; a vector instruction that reads an exponential or a logarithm needs one.)
#define EW_EACH(I) ".irp e,0,1,2,3,4,5,6,7\n" I "\n.endr\n"
#define EW_NEXT                                                                                                              \
  "v_readlane_b32 s50, v12, s51\nv_readlane_b32 s56, v13, s51\ns_addk_i32 s51, 1\ns_lshr_b32 s52, s50, 16\n"              \
  "s_add_u32 s54, s48, s52\ns_addc_u32 s55, s49, 0\ns_setpc_b64 s[54:55]\n"
#define EW_HANDLER(BODY) ".p2align 8\n" BODY EW_NEXT
#define EW_LEAVE(BODY) ".p2align 8\n" BODY "s_branch .Lew_out%=\n"
#define EW_INDEXED(I) "s_set_gpr_idx_on s50, gpr_idx(SRC0)\n" EW_EACH(I) "s_set_gpr_idx_off\n"
#define EW_V(OP) EW_HANDLER(EW_INDEXED(OP " v[16+\\e], v[24+\\e], v[16+\\e]"))
#define EW_S(OP) EW_HANDLER(EW_EACH(OP " v[16+\\e], s56, v[16+\\e]"))
#define EW_R(OP) EW_HANDLER(EW_INDEXED(OP " v[16+\\e], v14, v[16+\\e]"))
// maximum and minimum ignore a NaN operand, a signalling one too: both sides go through X and a maximum with themselves first
#define EW_QUIET_TOP EW_EACH("v_max_f32 v[16+\\e], v[16+\\e], v[16+\\e]")
#define EW_MV(OP)                                                                                                            \
  EW_HANDLER("s_set_gpr_idx_on s50, gpr_idx(SRC0,SRC1)\n" EW_EACH("v_max_f32 v[32+\\e], v[24+\\e], v[24+\\e]")       \
             "s_set_gpr_idx_off\n" EW_QUIET_TOP EW_EACH(OP " v[16+\\e], v[32+\\e], v[16+\\e]"))
#define EW_MS(OP) EW_HANDLER(EW_QUIET_TOP EW_EACH(OP " v[16+\\e], s56, v[16+\\e]"))
#define EW_MR(OP)                                                                                                            \
  EW_HANDLER("s_set_gpr_idx_on s50, gpr_idx(SRC0,SRC1)\nv_max_f32 v32, v14, v14\ns_set_gpr_idx_off\n" EW_QUIET_TOP          \
             EW_EACH(OP " v[16+\\e], v32, v[16+\\e]"))
#define EW_INTERPRETER                                                                                                       \
  "s_getpc_b64 s[48:49]\n.Lew_here%=:\ns_add_u32 s48, s48, (.Lew_handlers%=-.Lew_here%=)&4294967295\n"                     \
  "s_addc_u32 s49, s49, (.Lew_handlers%=-.Lew_here%=)>>32\n" EW_NEXT ".p2align 8\n.Lew_handlers%=:\n"                       \
  EW_LEAVE("") EW_LEAVE("") EW_LEAVE("")                                                                   /* END MORE FETCH */ \
  EW_LEAVE(EW_INDEXED("v_mov_b32 v[32+\\e], v[24+\\e]"))                                                        /* DIVV */  \
  EW_LEAVE(EW_EACH("v_mov_b32 v[32+\\e], v[16+\\e]") EW_INDEXED("v_mov_b32 v[16+\\e], v[24+\\e]"))            /* RDIVV */ \
  EW_LEAVE(EW_EACH("v_mov_b32 v[32+\\e], s56")) EW_LEAVE(EW_INDEXED("v_mov_b32 v[32+\\e], v14"))          /* DIVS DIVR */ \
  EW_HANDLER("s_set_gpr_idx_on s50, gpr_idx(DST)\n" EW_EACH("v_mov_b32 v[24+\\e], v[16+\\e]") "s_set_gpr_idx_off\n") /* SAVE */ \
  EW_HANDLER(EW_INDEXED("v_mov_b32 v[16+\\e], v[24+\\e]")) EW_HANDLER(EW_EACH("v_mov_b32 v[16+\\e], s56"))           \
  EW_HANDLER(EW_INDEXED("v_mov_b32 v[16+\\e], v14"))                                               /* LOADV LOADS LOADR */ \
  EW_V("v_add_f32") EW_S("v_add_f32") EW_R("v_add_f32")                                                                      \
  EW_V("v_subrev_f32") EW_V("v_sub_f32") EW_R("v_subrev_f32")                                             /* SUBV RSUBV SUBR */ \
  EW_V("v_mul_f32") EW_S("v_mul_f32") EW_R("v_mul_f32")                                                                      \
  EW_MV("v_max_f32") EW_MS("v_max_f32") EW_MR("v_max_f32") EW_MV("v_min_f32") EW_MS("v_min_f32") EW_MR("v_min_f32")          \
  EW_HANDLER(EW_EACH("v_xor_b32 v[16+\\e], 0x80000000, v[16+\\e]"))                                               /* NEG */  \
  EW_HANDLER(EW_EACH("v_exp_f32 v[16+\\e], v[16+\\e]") "s_nop 0\n")                                                     \
  EW_HANDLER(EW_EACH("v_log_f32 v[16+\\e], v[16+\\e]") "s_nop 0\n")                                                     \
  ".Lew_out%=:\n"
// (M0, which the index mode writes, is a reserved register that the compiler refuses among the clobbers: these kernels must have no other use of it,
// as tests/test_asm_hazards.py checks in their listing)
#define EW_CLOBBERS "s48", "s49", "s52", "s54", "s55", "s56", "scc"

typedef float v8f __attribute__((ext_vector_type(8)));

struct Raw { v4u a, b; };  // 8 elements of a 32-bit operand, or (a) of a 16-bit one

__device__ __forceinline__ Raw load_raw(const char* at, int dt, bool streamed) {
  Raw r;
  if (streamed) {
    r.a = __builtin_nontemporal_load((const v4u_any*)at);
    if (dt == FRISK_F32) r.b = __builtin_nontemporal_load((const v4u_any*)at + 1);
  } else {
    r.a = *(const v4u_any*)at;
    if (dt == FRISK_F32) r.b = *((const v4u_any*)at + 1);
  }
  return r;
}
// the same of two halves of 4 columns, the second one `apart` columns behind the first
__device__ __forceinline__ Raw load_halves(const char* at, int dt, int64_t apart, bool streamed) {
  typedef unsigned v2u_any __attribute__((ext_vector_type(2), aligned(2)));
  Raw r;
  if (dt == FRISK_F32) {
    r.a = streamed ? __builtin_nontemporal_load((const v4u_any*)at) : *(const v4u_any*)at;
    r.b = streamed ? __builtin_nontemporal_load((const v4u_any*)(at + apart * 4)) : *(const v4u_any*)(at + apart * 4);
  } else {
    const v2u_any lo = *(const v2u_any*)at, hi = *(const v2u_any*)(at + apart * 2);
    r.a = v4u{lo[0], lo[1], hi[0], hi[1]};
  }
  return r;
}
// The first `valid` (1 to 7) of 8 elements, of a row that has no more: without branches, the last one again in place of those beyond it, so that all
// are under way together
__device__ __forceinline__ Raw load_raw_narrow(const char* at, int dt, int valid) {
  unsigned w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (dt == FRISK_F32) {
#pragma unroll
    for (int e = 0; e < V; ++e) w[e] = ((const unsigned*)at)[e < valid ? e : valid - 1];
  } else {
    unsigned h[V];
#pragma unroll
    for (int e = 0; e < V; ++e) h[e] = ((const uint16_t*)at)[e < valid ? e : valid - 1];
#pragma unroll
    for (int e = 0; e < V; ++e) w[e / 2] |= h[e] << (16 * (e & 1));
  }
  return Raw{v4u{w[0], w[1], w[2], w[3]}, v4u{w[4], w[5], w[6], w[7]}};
}
template <class F> __device__ __forceinline__ void to_float(const Raw& r, int dt, F& out) {
  if (dt == FRISK_F32) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned lo = r.a[e], hi = r.b[e];  // copy first: bit_cast applied to a vector element reads element 0
      out[e] = __builtin_bit_cast(float, lo);
      out[4 + e] = __builtin_bit_cast(float, hi);
    }
  } else if (dt == FRISK_F16) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const h8 h = __builtin_bit_cast(h8, r.a);
#pragma unroll
    for (int e = 0; e < V; ++e) out[e] = (float)h[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) { out[2 * e] = __builtin_bit_cast(float, r.a[e] << 16); out[2 * e + 1] = __builtin_bit_cast(float, r.a[e] & 0xffff0000u); }
  }
}
__device__ __forceinline__ float load_one(const char* at, int dt) {
  if (dt == FRISK_F32) return *(const float*)at;
  if (dt == FRISK_F16) return (float)*(const _Float16*)at;
  return (float)*(const __bf16*)at;
}
// columns first .. last - 1 of a group that starts at `at`
__device__ __forceinline__ void store_group(char* at, int dt, const v8f& r, int first, int last) {
  if (first == 0 && last == V) {
    if (dt == FRISK_F32) {
      v4u a, b;
#pragma unroll
      for (int e = 0; e < 4; ++e) { const float lo = r[e], hi = r[4 + e]; a[e] = __builtin_bit_cast(unsigned, lo); b[e] = __builtin_bit_cast(unsigned, hi); }
      *(v4u_any*)at = a;
      *((v4u_any*)at + 1) = b;
    } else if (dt == FRISK_F16) {
      typedef _Float16 h8 __attribute__((ext_vector_type(8)));
      h8 h;
#pragma unroll
      for (int e = 0; e < V; ++e) h[e] = (_Float16)r[e];
      __builtin_nontemporal_store(__builtin_bit_cast(v4u, h), (v4u_any*)at);
    } else {
      typedef __bf16 b8 __attribute__((ext_vector_type(8)));
      b8 h;
#pragma unroll
      for (int e = 0; e < V; ++e) h[e] = (__bf16)r[e];
      __builtin_nontemporal_store(__builtin_bit_cast(v4u, h), (v4u_any*)at);
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < V; ++e) {
    if (e < first || e >= last) continue;
    if (dt == FRISK_F32) ((float*)at)[e] = r[e];
    else if (dt == FRISK_F16) ((_Float16*)at)[e] = (_Float16)r[e];
    else ((__bf16*)at)[e] = (__bf16)r[e];
  }
}

template <bool V> struct StreamedTag { static constexpr bool value = V; };
// half a group of 32-bit columns from `first` (0 to 4) on
template <bool STREAMED> __device__ __forceinline__ void store_half(char* at, const v8f& r, int half, int first) {
  v4u w;
#pragma unroll
  for (int e = 0; e < 4; ++e) { const float x = r[4 * half + e]; w[e] = __builtin_bit_cast(unsigned, x); }
  if (first == 0) {
    if constexpr (STREAMED) __builtin_nontemporal_store(w, (v4u_any*)at); else *(v4u_any*)at = w;
    return;
  }
#pragma unroll
  for (int e = 1; e < 4; ++e)
    if (e >= first) ((unsigned*)at)[e] = w[e];
}

// DT: element type of the operands that walk the rows and of the output (-1: mixed, read from the arguments).  HELD: which operands beside
// `head` are held or fetched ahead: none; the second one that walks the rows; that one and the broadcast ones, whose values of the row may meet constants first (HELD_SCALED) (44 more registers for 32-bit
// operands, 32 for 16-bit ones, and 1500 instructions in front of the first step instead of 650: x + y of 1024 x 4096 f16 7.4 us with them,
// 6.5 without, f32 11.3 and 9.9, 100000 x 24 f16 5.6 and 4.5, 8192 x 8192 f16 74.4 and 71).  DEPTH: values below the top the program needs.
// ROWS: a wave's lanes lie in several rows, in one (rows of at least 64 groups), or in one each, of less than a group (as a case of the first, its loads
// cost that one 0.4 us in 4.8 of 6304 x 136 f16).
enum Rows { ROWS_SHARED, ROWS_UNIFORM, ROWS_NARROW };
enum Held { HELD_NONE, HELD_WALK, HELD_ALL, HELD_SCALED };
// Kernels that hold all of them run four waves a SIMD where their registers allow it ((x - s c) g + b of 100000 x 24 f16: 136 registers and three
// waves 8.6 us, 7.4 with four).
constexpr bool four_waves(int dt, int held, int depth, bool uniform_row) { return held >= HELD_ALL && depth == 1 && !(dt == FRISK_F32 && !uniform_row); }
template <int DT, int HELD, int DEPTH, int ROWS> __global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(four_waves(DT, HELD, DEPTH, ROWS == ROWS_UNIFORM) ? 4 : 1, four_waves(DT, HELD, DEPTH, ROWS == ROWS_UNIFORM) ? 4 : 8))) elementwise_kernel(EwArgs p, int lanes_log2) {
  const int lanes = 1 << lanes_log2, row_step = 256 >> lanes_log2;
  const int lane_group = threadIdx.x & (lanes - 1);
  int lane_row = threadIdx.x >> lanes_log2;
  if constexpr (ROWS == ROWS_UNIFORM) lane_row = __builtin_amdgcn_readfirstlane(lane_row);
  const int64_t groups = (p.cols + V - 1) / V, slabs = (groups + lanes - 1) >> lanes_log2, row_blocks = (p.rows + row_step - 1) / row_step;
  constexpr bool narrow = ROWS == ROWS_NARROW;
  // HALVES: a lane's 8 columns of 32-bit operands are 4 and 4, a slab's lanes side by side in either half, so that every access of a wave is one run of memory.  (With a
  // lane's two accesses side by side each takes half of every line, and stores past the caches, which halves allow, would write lines twice.  us side by side / so, f32 from memory: (x - s c) g + b of
  // 4096 x 4096 28.9 / 27.7, 2000 x 2500 15.7 / 13.2, 4111 x 4501 37.6 / 33.3, 8192 x 8192 102.4 / 96.8, exp2(x) c of 4111 x 4501 29.6 / 25.7, x + y of 1500 x 2000 9.9 / 9.0; halves with stores through
  // the caches 27.2, 14.5, 35.4, 98.4, 27.7, 9.6.)
  constexpr bool HALVES = DT == FRISK_F32 && !narrow;
  // step i of a chunk of the program in lane i: a lane read instead of a dependent scalar load
  int code_reg[2] = {p.code[threadIdx.x & 63], 0}, imm_reg[2] = {__builtin_bit_cast(int, p.imm[threadIdx.x & 63]), 0};
  if (p.n_steps > kChunk) {
    code_reg[1] = p.code[kChunk + (threadIdx.x & 63)];
    imm_reg[1] = __builtin_bit_cast(int, p.imm[kChunk + (threadIdx.x & 63)]);
  }
  auto type_of = [&](const EwOperand& k) { return DT >= 0 ? DT : k.dt; };
  auto row_value = [&](int dt, unsigned bits) {
    if (dt == FRISK_F32) return __builtin_bit_cast(float, bits);
    if (dt == FRISK_F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
    return __builtin_bit_cast(float, bits << 16);
  };
  const int64_t rb0 = blockIdx.y, row_stride = (int64_t)gridDim.y * row_step;  // rows between this lane's groups
  if (rb0 >= row_blocks) return;
  // A lane keeps its columns and walks down the rows, every operand's address moving on by one stride: worked out anew for every
  // group, place and addresses made the counts above 136, 171 and 35 (203.8 us instead of 195.2 for cast, mean, that body and softmax; a SIMD issues one scalar instruction in
  // four cycles, so they weigh as much as the vector ones).
  for (int64_t slab = blockIdx.x; slab < slabs; slab += gridDim.x) {
    // lanes beyond the view repeat its last row or group and store nothing
    const int64_t left = groups - (slab << lanes_log2);
    const int off = lane_group < left ? lane_group : (int)left - 1;
    // A row's last group, where it is not whole, is evaluated together with the columns before it that fill it up: every load is then 16 bytes of
    // the row.  The lane stores columns `mine` and up of its 8, the others being the neighbour's (whose store may have come first where the
    // output is an operand too).  Fetched element by element behind branches, that group held up every row: (x - s c) g + b of 4095 x 8191 bf16 47.6 us, 32.3 so,
    // 16000 x 3999 f16 99.0 and 61.0, 6330 x 669 17.7 and 11.9.
    const int64_t past = ((slab << lanes_log2) + off + 1) * V - p.cols;
    const int mine = past > 0 && !narrow ? (int)past : 0, last = narrow ? (int)p.cols : V;
    // HALVES: columns that the slab has, where the lane's halves start, and the columns of either that are another lane's (4: all)
    const int64_t rest = p.cols - (slab << lanes_log2) * V;
    const int col_a = lane_group * 4, col_b = (lanes + lane_group) * 4;
    if constexpr (ROWS == ROWS_UNIFORM) {  // a wave beyond the row's end (repeating its last group it cost (x - s c) g + b of 2490 x 4453 f16 0.6 us of 12.4, 3168 x 2891 0.4 of 11.0)
      const int wave = __builtin_amdgcn_readfirstlane(lane_group);
      if (HALVES ? wave * 4 >= rest : wave >= left) continue;
    }
    const int64_t at_a = col_a + 4 <= rest ? col_a : rest - 4, at_b = col_b + 4 <= rest ? col_b : rest - 4, apart = at_b - at_a;
    const int mine_a = col_a - at_a < 4 ? (int)(col_a - at_a) : 4, mine_b = col_b - at_b < 4 ? (int)(col_b - at_b) : 4;
    // (32 bits but for halves: as 64 it was 20 more instructions in front of a 16-bit body's first step, (x - s c) g + b of 1925 x 1826 f16 7.36 us, 7.15 so, 3168 x 2891 13.65 / 13.42)
    std::conditional_t<HALVES, int64_t, int> lane_col;
    if constexpr (HALVES) lane_col = at_a; else lane_col = off * V - mine;
    int64_t row = rb0 * row_step + lane_row;
    const int64_t row_in = row < p.rows ? row : p.rows - 1;
    // element (r, first column of the group) of an operand whose elements are of type dt
    auto operand_at = [&](const EwOperand& k, int dt, bool walks, int64_t r) {
      const int es = dt == FRISK_F32 ? 4 : 2;
      const char* base = k.at + r * k.row_bytes;
      return walks ? base + (slab << lanes_log2) * (V * es) + lane_col * es : base;
    };
    auto fetch_at = [&](const char* at, int dt, bool streamed) {
      if constexpr (narrow) return load_raw_narrow(at, dt, last);
      else if constexpr (HALVES) return load_halves(at, dt, apart, streamed);
      else return load_raw(at, dt, streamed);
    };
    auto fetch_row_at = [&](const char* at, int dt) { return dt == FRISK_F32 ? *(const unsigned*)at : (unsigned)*(const uint16_t*)at; };
    const char *head_at = nullptr, *walk2_at = nullptr, *row0_at = nullptr, *row1_at = nullptr;
    int64_t head_step = 0, walk2_step = 0, row0_step = 0, row1_step = 0;
    if (p.head.at) { head_at = operand_at(p.head, type_of(p.head), true, row_in); head_step = row_stride * p.head.row_bytes; }
    if constexpr (HELD >= HELD_WALK) {
      if (p.walk2.at) { walk2_at = operand_at(p.walk2, type_of(p.walk2), true, row_in); walk2_step = row_stride * p.walk2.row_bytes; }
    }
    if constexpr (HELD >= HELD_ALL) {
      if (p.row0.at) { row0_at = operand_at(p.row0, p.row0.dt, false, row_in); row0_step = row_stride * p.row0.row_bytes; }
      if (p.row1.at) { row1_at = operand_at(p.row1, p.row1.dt, false, row_in); row1_step = row_stride * p.row1.row_bytes; }
    }
    const int out_dt = DT >= 0 ? DT : p.out_dt, out_es = out_dt == FRISK_F32 ? 4 : 2;
    char* out_at = p.out + row_in * p.out_row_bytes + (slab << lanes_log2) * (V * out_es) + lane_col * out_es;
    const int64_t out_step = row_stride * p.out_row_bytes;

    // what is under way from memory: the next group of 32-bit operands, the next two of 16-bit ones (16 bytes a lane and four waves a SIMD
    // are a third of what the memory's latency asks for: one group ahead 195.2 us for the four calls of cast, mean, scale and shift, softmax on 8192 x 8192 f16, two 191.8)
    constexpr int SETS = (DT == FRISK_F16 || DT == FRISK_BF16) && DEPTH == 1 && ROWS == ROWS_UNIFORM ? 2 : 1;
    struct Ahead { Raw head, walk2; unsigned row0, row1; } held0{}, held1{};
    v8f col0{}, col1{};
    auto fetch_ahead = [&](Ahead& h) __attribute__((always_inline)) {
      if (p.head.at) h.head = fetch_at(head_at, type_of(p.head), true);
      if constexpr (HELD >= HELD_WALK) {
        if (p.walk2.at) h.walk2 = fetch_at(walk2_at, type_of(p.walk2), true);
      }
      if constexpr (HELD >= HELD_ALL) {
        if (p.row0.at) h.row0 = fetch_row_at(row0_at, p.row0.dt);
        if (p.row1.at) h.row1 = fetch_row_at(row1_at, p.row1.dt);
      }
    };
    int64_t fetched = row;  // row of the last fetch
    auto next_row = [&]() __attribute__((always_inline)) {
      fetched += row_stride;
      if (fetched < p.rows) {  // (a lane whose next row lies beyond the view fetches the present one again)
        head_at += head_step;
        if constexpr (HELD >= HELD_WALK) walk2_at += walk2_step;
        if constexpr (HELD >= HELD_ALL) { row0_at += row0_step; row1_at += row1_step; }
      }
    };
    fetch_ahead(held0);
    if constexpr (SETS == 2) {
      if (rb0 + gridDim.y < row_blocks) {
        next_row();
        fetch_ahead(held1);
      }
    }
    if constexpr (HELD >= HELD_ALL) {
      if (p.col0.at) to_float(fetch_at(operand_at(p.col0, p.col0.dt, true, 0), p.col0.dt, false), p.col0.dt, col0);
      if (p.col1.at) to_float(fetch_at(operand_at(p.col1, p.col1.dt, true, 0), p.col1.dt, false), p.col1.dt, col1);
    }
    int64_t rb = rb0;
    // one group, whose operands are in h; true: it was the last one
    auto group = [&](Ahead& h) __attribute__((always_inline)) {
      const bool live = row < p.rows && lane_group < left;
      v8f top, s0, s1, s2, s3, s4, x, walk2;
      asm volatile("" : "=v"(top), "=v"(s0), "=v"(x), "=v"(walk2));  // written by the program before it reads them
      if constexpr (DEPTH > 1) asm volatile("" : "=v"(s1), "=v"(s2), "=v"(s3), "=v"(s4));
      float row_a = 0.f, row_b = 0.f;
      if (p.head.at) to_float(h.head, type_of(p.head), top);
      if constexpr (HELD >= HELD_WALK) {
        if (p.walk2.at) to_float(h.walk2, type_of(p.walk2), walk2);
      }
      if constexpr (HELD >= HELD_ALL) {
        if (p.row0.at) row_a = row_value(p.row0.dt, h.row0);
        if (p.row1.at) row_b = row_value(p.row1.dt, h.row1);
      }
      if constexpr (HELD == HELD_SCALED) {
        row_a = __builtin_fmaf(row_a, p.scale0.mul, p.scale0.add);
        row_b = __builtin_fmaf(row_b, p.scale1.mul, p.scale1.add);
      }
      const int64_t here = row < p.rows ? row : p.rows - 1;
      if (rb + SETS * (int64_t)gridDim.y < row_blocks) {
        next_row();
        fetch_ahead(h);
      }
      int pc = 0, code = code_reg[0], imm = imm_reg[0];
      for (;;) {
        int step;
#define EW_RUN(MORE_OUT, IN)                                                                                                                   \
  asm volatile(EW_INTERPRETER : "={s50}"(step), "+{s51}"(pc), "+{v[16:23]}"(top), "+{v[24:31]}"(s0), "+{v[32:39]}"(x) MORE_OUT                 \
               : "{v12}"(code), "{v13}"(imm) IN : EW_CLOBBERS)
#define EW_DEEP , "+{v[64:71]}"(s1), "+{v[72:79]}"(s2), "+{v[80:87]}"(s3), "+{v[88:95]}"(s4)
#define EW_WALK2 , "{v[56:63]}"(walk2)
#define EW_BROADCAST , "{v14}"(row_a), "{v15}"(row_b), "{v[40:47]}"(col0), "{v[48:55]}"(col1)
        if constexpr (HELD >= HELD_ALL && DEPTH > 1) EW_RUN(EW_DEEP, EW_BROADCAST EW_WALK2);
        else if constexpr (HELD >= HELD_ALL) EW_RUN(, EW_BROADCAST EW_WALK2);
        else if constexpr (HELD == HELD_WALK && DEPTH > 1) EW_RUN(EW_DEEP, EW_WALK2);
        else if constexpr (HELD == HELD_WALK) EW_RUN(, EW_WALK2);
        else if constexpr (DEPTH > 1) EW_RUN(EW_DEEP, );
        else EW_RUN(, );
#undef EW_RUN
#undef EW_DEEP
#undef EW_WALK2
#undef EW_BROADCAST
        const int what = step >> 24;
        if (what == STEP_END) break;
        if (what == STEP_FETCH) {
          const EwOperand& k = p.in[(step >> 8) & 15];
          if (k.walks) to_float(fetch_at(operand_at(k, k.dt, true, here), k.dt, false), k.dt, x);
          else x = v8f{} + row_value(k.dt, fetch_row_at(operand_at(k, k.dt, false, here), k.dt));
        } else if (what == STEP_MORE) {
          code = code_reg[1];
          imm = imm_reg[1];
          pc = 0;
        } else {
  #pragma unroll
          for (int e = 0; e < V; ++e) top[e] = top[e] / x[e];
        }
      }
      if constexpr (HALVES) {
        auto store = [&](auto streamed) __attribute__((always_inline)) {
          if (mine_a < 4) store_half<decltype(streamed)::value>(out_at, top, 0, mine_a);
          if (mine_b < 4) store_half<decltype(streamed)::value>(out_at + apart * 4, top, 1, mine_b);
        };
        if (row < p.rows) {
          if (p.past) {
            asm volatile("");  // (these keep the compiler from making one store of the two, which is then not streamed)
            store(StreamedTag<true>{});
          } else {
            store(StreamedTag<false>{});
            asm volatile("");
          }
        }
      } else if (live) store_group(out_at, out_dt, top, mine, last);
      out_at += out_step;
      row += row_stride;
      rb += gridDim.y;
      return rb >= row_blocks;
    };
    for (;;) {
      if (group(held0)) break;
      if constexpr (SETS == 2) { if (group(held1)) break; }
    }
  }
}

// The postfix program as steps.  `held`: which inputs may be held in slots (each mention of the others is fetched where it stands).
EwSteps steps_of(const EwParams& p, int held) {
  EwSteps s{};
  s.head = s.walk2 = s.col0 = s.col1 = s.row0 = s.row1 = -1;
  int n = 0, below = -1;  // steps so far, values below the top
  auto emit = [&](int what, int index = 0, float imm = 0.f, int input = 0) {
    if (n == kChunk - 1) s.code[n++] = STEP_MORE << 24;
    s.code[n] = what << 24 | input << 8 | index;
    s.imm[n++] = imm;
  };
  auto slot_below = [](int depth) { return depth == 1 ? kSlotS0 : kSlotS1 + 8 * (depth - 2); };  // of the depth-th value below the top
  const int by_slot[6] = {STEP_ADDV, STEP_SUBV, STEP_MULV, STEP_DIVV, STEP_MAXV, STEP_MINV};
  const int by_const[6] = {STEP_ADDS, STEP_ADDS, STEP_MULS, STEP_DIVS, STEP_MAXS, STEP_MINS};  // x - c is x + (-c)
  const int by_row[6] = {STEP_ADDR, STEP_SUBR, STEP_MULR, STEP_DIVR, STEP_MAXR, STEP_MINR};
  const int from_below[6] = {STEP_ADDV, STEP_RSUBV, STEP_MULV, STEP_RDIVV, STEP_MAXV, STEP_MINV};  // the value below is the left operand
  bool seen[FRISK_EW_MAX_INPUTS] = {};
  // with no second operand that moves with the rows, the place of one serves an operand that is the same for every row
  bool col_as_walk2 = held == HELD_WALK;
  for (int i = 1; i < p.n_ops; ++i)
    if (p.op[i] == FRISK_EW_INPUT && p.in_col_stride[p.arg[i]] && (p.in_row_stride[p.arg[i]] || p.in_dtype[p.arg[i]] != p.out_dtype) && p.arg[i] != (p.op[0] == FRISK_EW_INPUT ? p.arg[0] : -1))
      col_as_walk2 = false;
  int mentions[FRISK_EW_MAX_INPUTS] = {};
  for (int i = 0; i < p.n_ops; ++i)
    if (p.op[i] == FRISK_EW_INPUT) ++mentions[p.arg[i]];
  // steps i, i + 1 and i + 2 combine the only mention of an operand of one value per row, which a slot can hold, with a constant
  auto scaled_row = [&](int i, RowScale& scale) {
    if (held != HELD_ALL || i + 2 >= p.n_ops || (s.row0 >= 0 && s.row1 >= 0)) return -1;
    const bool value_first = p.op[i] == FRISK_EW_INPUT;
    if (p.op[value_first ? i : i + 1] != FRISK_EW_INPUT || p.op[value_first ? i + 1 : i] != FRISK_EW_CONST) return -1;
    const int k = p.arg[value_first ? i : i + 1];
    const float c = p.imm[value_first ? i + 1 : i];
    if (p.in_col_stride[k] != 0 || mentions[k] != 1) return -1;
    switch (p.op[i + 2]) {
      case FRISK_EW_ADD: scale.add = c; return k;
      case FRISK_EW_SUB: scale.mul = value_first ? 1.f : -1.f; scale.add = value_first ? -c : c; return k;
      case FRISK_EW_MUL: scale.mul = c; return k;
      default: return -1;
    }
  };
  for (int i = 0; i < p.n_ops; ++i) {
    const int op = p.op[i];
    RowScale scale;
    if (const int k = scaled_row(i, scale); k >= 0) {
      const bool first = s.row0 < 0;
      (first ? s.row0 : s.row1) = k;
      (first ? s.scale0 : s.scale1) = scale;
      s.scaled = true;
      const int next = i + 3 < p.n_ops ? p.op[i + 3] : -1;
      const bool fused = next >= FRISK_EW_ADD && next <= FRISK_EW_MIN;
      if (!fused && ++below > 0) emit(STEP_SAVE, slot_below(below));
      if (below > s.depth) s.depth = below;
      emit(fused ? by_row[next - FRISK_EW_ADD] : STEP_LOADR, !first);
      i += 2 + fused;
      continue;
    }
    if (op == FRISK_EW_INPUT || op == FRISK_EW_CONST) {
      const int k = op == FRISK_EW_INPUT ? p.arg[i] : 0, next = i + 1 < p.n_ops ? p.op[i + 1] : -1;
      const bool walks = p.in_col_stride[k] != 0;
      if (op == FRISK_EW_INPUT && !seen[k]) {
        seen[k] = true;
        const bool same_every_row = p.in_row_stride[k] == 0 && p.rows > 1;
        if (i == 0 && walks) s.head = k;
        else if (held == HELD_ALL && !walks) { if (s.row0 < 0) s.row0 = k; else if (s.row1 < 0) s.row1 = k; }
        else if (held == HELD_ALL && same_every_row) { if (s.col0 < 0) s.col0 = k; else if (s.col1 < 0) s.col1 = k; }
        else if (held != HELD_NONE && walks && s.walk2 < 0 && (!same_every_row || col_as_walk2)) s.walk2 = k;
      }
      const bool fused = next >= FRISK_EW_ADD && next <= FRISK_EW_MIN;  // pushed only to be the right operand of the next step
      if (!fused && ++below > 0) emit(STEP_SAVE, slot_below(below));
      if (below > s.depth) s.depth = below;
      const int which = fused ? next - FRISK_EW_ADD : 0;
      if (op == FRISK_EW_CONST) emit(fused ? by_const[which] : STEP_LOADS, 0, fused && next == FRISK_EW_SUB ? -p.imm[i] : p.imm[i]);
      else if (k == s.row0 || k == s.row1) emit(fused ? by_row[which] : STEP_LOADR, k == s.row1);
      else if (i == 0 && k == s.head) {}  // the top starts with it
      else {
        const int slot = k == s.walk2 ? kSlotWalk2 : k == s.col0 ? kSlotCol0 : k == s.col1 ? kSlotCol1 : kSlotX;
        if (slot == kSlotX) emit(STEP_FETCH, 0, 0.f, k);
        emit(fused ? by_slot[which] : STEP_LOADV, slot);
      }
      i += fused;
    } else if (op <= FRISK_EW_MIN) {
      emit(from_below[op - FRISK_EW_ADD], slot_below(below));
      --below;
    } else {
      emit(op == FRISK_EW_NEG ? STEP_NEG : op == FRISK_EW_EXP2 ? STEP_EXP2 : STEP_LOG2);
    }
  }
  emit(STEP_END);
  s.n = n;
  return s;
}
// two postfix steps make at most four steps (a value saved, fetched, loaded and combined from below)
static_assert(2 * FRISK_EW_MAX_OPS + 2 <= 2 * kChunk, "a program fits into two chunks");

template <int DT, int HELD> void launch_typed(const dim3& grid, const EwArgs& a, int depth, int lanes_log2, hipStream_t s) {
#define FRISK_EW_LAUNCH(DEPTH)                                                                                                                   \
  if (a.cols < V) hipLaunchKernelGGL((elementwise_kernel<DT, HELD, DEPTH, ROWS_NARROW>), grid, dim3(256), 0, s, a, lanes_log2);                 \
  else if (lanes_log2 >= 6) hipLaunchKernelGGL((elementwise_kernel<DT, HELD, DEPTH, ROWS_UNIFORM>), grid, dim3(256), 0, s, a, lanes_log2);      \
  else hipLaunchKernelGGL((elementwise_kernel<DT, HELD, DEPTH, ROWS_SHARED>), grid, dim3(256), 0, s, a, lanes_log2);
  if (depth <= 1) { FRISK_EW_LAUNCH(1) } else { FRISK_EW_LAUNCH(5) }
#undef FRISK_EW_LAUNCH
}
template <int DT> void launch_held(int held, bool scaled, const dim3& grid, const EwArgs& a, int depth, int lanes_log2, hipStream_t s) {
  if (held == HELD_ALL && scaled) launch_typed<DT, HELD_SCALED>(grid, a, depth, lanes_log2, s);
  else if (held == HELD_ALL) launch_typed<DT, HELD_ALL>(grid, a, depth, lanes_log2, s);
  else if (held == HELD_WALK) launch_typed<DT, HELD_WALK>(grid, a, depth, lanes_log2, s);
  else launch_typed<DT, HELD_NONE>(grid, a, depth, lanes_log2, s);
}

}  // namespace

// 32-bit bodies store past the caches, but for those of one operand that walks the rows and of values of the row, which as a rule have just been reduced from it, in views of more than kPastUpTo bytes and up to
// kPastFrom, the size of the last-level cache: between the reduction that has read the operand and a softmax that reads the result, stores through the caches leave more to be found there.  us past / through, cast, row
// sums, (x - s c) g + b and softmax together: 8192 x 8192 324 / 319 (319 before stores passed the caches; the body alone in that row 98.5 / 88.3), 16384 x 4096 314 / 307, 6000 x 8000 237 / 231, 4096 x 8192 171 / 163, 4111 x 4501
// 109 / 106, 50000 x 400 113 / 109, 100000 x 600 294 / 284; 4096 x 4096 and 3029 x 3796 even; 16384 x 16384 1294 / 1313.  On their own, operands from memory, bodies are 1 to 4 % faster past the caches ((x - s c) g + b of
// 8192 x 8192 96.8 / 98.4, exp2(x) c 94.7 / 98.4, x + y 137.3 / 138.6).  Rows of up to 32 columns, whose halves are parts of lines, never pass them.
constexpr int64_t kPastUpTo = (int64_t)64 << 20, kPastFrom = (int64_t)256 << 20;

hipError_t launch_elementwise(const EwParams& given, hipStream_t s) {
  EwParams p = given;
  // A dense view is one row, down which no lane walks and fetches ahead.  A 16-bit one that gives every lane more than one group is folded to
  // rows of one group a lane (8192 x 8192 f16: log2(max(x, c) / (x + c)) 73.6 -> 69.5 us, x * y + z 95.7 -> 95.4; f32, of which one group less
  // is under way, lost: 117 -> 119).
  constexpr int64_t kFold = 256 * V, kCap = 256 * 16, kHeldCap = 256 * 4;
  bool half = p.out_dtype != FRISK_F32;
  for (int k = 0; k < FRISK_EW_MAX_INPUTS; ++k) half = half && (p.in_col_stride[k] == 0 || p.in_dtype[k] == p.out_dtype);
  if (p.rows == 1 && half && p.cols % kFold == 0 && p.cols / kFold > kCap) {
    p.rows = p.cols / kFold;
    p.cols = p.out_ld = kFold;
    for (int k = 0; k < FRISK_EW_MAX_INPUTS; ++k) p.in_row_stride[k] = p.in_col_stride[k] ? kFold : 0;
  }
  const int64_t groups = (p.cols + V - 1) / V;
  int lanes_log2 = 0;
  while (lanes_log2 < 8 && ((int64_t)1 << lanes_log2) < groups) ++lanes_log2;
  const int64_t lanes = (int64_t)1 << lanes_log2, row_step = 256 >> lanes_log2;
  // Enough work-groups to fill the chip several times over, every lane walking its row / column strides beyond that: 16 per CU; of the kernels that
  // hold more than the first operand 4 per CU, a single round of those with broadcast operands (four waves a SIMD), so that what stands in front of the
  // first group (up to 1000 instructions) is paid once per lane.  us with 16 / 4 per CU: (x - s c) g + b of 8192 x 8192 f16 54.8 / 51.6, 3000 x 4096 16.7 /
  // 11.5, 6330 x 669 11.9 / 8.8, 4095 x 8191 bf16 32.3 / 28.5, 4000 x 4096 f32 28.1 / 26.0; x + y of 8192 x 8192 f16 69 / 64; but exp2(x) c of 16000 x
  // 3999, which holds no more than the first operand, 44.7 / 48.1.  f32, of which a lane has one group under way, goes back to 16 per CU where the set-up weighs little:
  // from 12 groups a lane (on 4 per CU) with operands of one value a column held, from 7 with those of one value a row alone, from 5 with a second operand
  // that walks the rows.  us with 16 / 4 per CU: (x - s c) g + b of 4096 x 4096 26.5 / 25.5, 4000 x 3000 30.3 / 27.9, but 4095 x 8191 60.4 / 60.9, 20000 x 2048
  // 65.3 / 67.0, 10000 x 5000 85.4 / 88.1, 1000000 x 24 49.0 / 51.0; x s 2000 x 5000 16.9 / 15.3, 4000 x 3000 25.8 / 27.2; x g + y 2048 x 4096 21.8 / 20.1, 20000 x 300
  // 20.4 / 18.4, but 3000 x 4096 30.1 / 31.0, 20000 x 2048 90.7 / 93.4; x + y 2048 x 4096 20.3 / 20.6, 4096 x 4096 38.4 / 39.2.  Never more than the cap, where a row's slabs do not divide it: the few above a single round ran as a second one
  // (1026 instead of 1020, x + b of 3000 x 11008 f16 29.3 us, 23.3 so, (x - s c) g + b 35.2 and 25.9, f32 66.4 and 59.1; 10000 x 5000 f16 54.7 and 40.1).
  const int64_t row_blocks = (p.rows + row_step - 1) / row_step;
  int64_t gx = 0, gy = 0;
  auto set_grid = [&](int64_t cap) {
    gx = (groups + lanes - 1) / lanes;
    gy = row_blocks;
    if (gx > cap) gx = cap;
    if (gx * gy > cap) gy = cap / gx;
    if (gy > 65535) gy = 65535;
  };
  // Holding the broadcast operands pays where a lane walks down two rows or more, not where its one group waits for them to be set up, and the kernels that hold none fit
  // five work-groups on a CU: up to 5 / 4 of the smaller grid is a round of one group a lane.  us on 4 per CU, held / one group a lane, 1.004, 1.1, 1.25 and 1.5 times that grid: f16 x + b
  // of 2048 columns 4.9 / 4.0, 5.0 / 4.2, 5.0 / 4.3, 5.1 / 5.3, (x - s c) g + b 5.7 / 5.6, 5.8 / 5.8, 5.9 / 5.9, 5.9 / 7.7, x y + z 5.9 / 5.2, 6.1 / 5.3, 6.4 / 5.6, 7.6 / 8.3, f32 x g + b
  // 6.8 / 6.4, 7.4 / 7.0, 7.9 / 7.7, 8.8 / 9.3; Alone, without a second operand that walks the rows, 6 / 4 for one operand of one value a row (x s 4.8 / 4.2, 4.8 / 4.3, 4.9 / 4.5, 5.0 / 4.8, twice the grid 5.5 / 6.2), twice the grid for one of one value a column
  // in f32 or in rows shorter than a wave (x + b f16 of 24 columns 5.2 / 4.9, f32 of 4096 9.3 / 9.5, 1.75 times 9.0 / 8.9).  f32 with operands of one value a row in longer rows holds them at once (x s 6.1 / 6.3).
  // f32 in rows shorter than a wave, whose lanes each look for a column's value, holds none up to 5 times the grid beside a second operand that walks the rows, up to 12 times where there are one or two and
  // up to twice with more: us held on 4 per CU / not held on 16, 2, 4 and 8 times, 24 columns: x + b 9.9 / 8.1, 16.6 / 14.9, 28.0 / 23.3, x s 9.8 / 8.9, 16.3 / 15.3, 27.9 / 26.0, x g + b 10.7 / 9.3,
  // 17.5 / 16.9, 28.4 / 27.2, x g + y 11.6 / 11.3, 20.1 / 19.1, 34.7 / 33.7 (held on 16 33.7), (x - s c) g + b 11.5 / 10.7, 18.6 / 19.8, 30.2 / 32.7; 12 times, held on 16 / not, x g + b 39.0 / 37.8, 16 times 46.8 / 47.3.
  const EwSteps all = steps_of(p, HELD_ALL);
  const bool f32 = p.out_dtype == FRISK_F32, short_rows = lanes_log2 < 6;
  const int columns = (all.col0 >= 0) + (all.col1 >= 0), per_row = (all.row0 >= 0) + (all.row1 >= 0);
  int quarters = 5;  // of kHeldCap work-groups
  if (f32 && short_rows && columns + per_row) quarters = all.walk2 >= 0 ? 20 : columns + per_row <= 2 ? 48 : 8;
  else if (f32 && per_row) quarters = 4;
  else if (all.walk2 < 0 && columns == 1 && !per_row && (f32 || short_rows)) quarters = 8;
  else if (all.walk2 < 0 && per_row == 1 && !columns) quarters = 6;
  const int64_t steps = ((groups + lanes - 1) / lanes) * row_blocks;  // work-groups of one group a lane
  const bool few = 4 * steps <= quarters * kHeldCap;
  // one type for everything that moves with the rows: the kernels for it; mixed types: the one that looks at each operand's type,
  // which holds nothing ahead but the first operand
  EwSteps prog = few ? steps_of(p, HELD_WALK) : all;
  int dt = p.out_dtype;
  int held = prog.col0 >= 0 || prog.row0 >= 0 ? HELD_ALL : prog.walk2 >= 0 ? HELD_WALK : HELD_NONE;
// (16-bit ones too, beside a second operand that walks long rows and from 28 groups a lane on: x g + y of 8192 x 8192 f16 59.9 with 16 per CU, 63.8 with 4; 24 groups, 6144 x 8192, 58.7 / 56.0)
  const bool deep = f32 ? steps > (prog.walk2 >= 0 ? 5 : prog.col0 < 0 ? 7 : 12) * kHeldCap : prog.walk2 >= 0 && held == HELD_ALL && lanes_log2 == 8 && steps > 28 * kHeldCap;
  // (f32 with two operands that walk long rows on 64 per CU: us on 16 / 64, x + y of 8192 x 8192 143.6 / 139.8, x g + y 145.2 / 141.2, 10000 x 5000 115.6 / 106.8, 4096 x 8192 70.4 / 67.9, 3000 x 8192 52.1 / 51.4, even below;
  // rows of 24 columns 60.3 / 69.7)
  set_grid(held == HELD_NONE || few || deep ? (f32 && prog.walk2 >= 0 && !short_rows && 2 * steps > 5 * kCap ? kCap * 4 : kCap) : kHeldCap);
  if ((prog.head >= 0 && p.in_dtype[prog.head] != dt) || (prog.walk2 >= 0 && p.in_dtype[prog.walk2] != dt)) {
    dt = -1;
    held = HELD_NONE;
    prog = steps_of(p, HELD_NONE);
    set_grid(kCap);
  }
  EwArgs a{};
  a.rows = p.rows; a.cols = p.cols;
  a.out = (char*)p.out; a.out_dt = p.out_dtype; a.out_row_bytes = p.out_ld * (p.out_dtype == FRISK_F32 ? 4 : 2);
  auto operand = [&](int k) {
    if (k < 0) return EwOperand{};
    return EwOperand{(const char*)p.in[k], p.in_row_stride[k] * (p.in_dtype[k] == FRISK_F32 ? 4 : 2), p.in_dtype[k], p.in_col_stride[k]};
  };
  for (int k = 0; k < FRISK_EW_MAX_INPUTS; ++k) a.in[k] = operand(k);
  a.head = operand(prog.head); a.walk2 = operand(prog.walk2);
  a.row0 = operand(prog.row0); a.row1 = operand(prog.row1); a.col0 = operand(prog.col0); a.col1 = operand(prog.col1);
  a.scale0 = prog.scale0; a.scale1 = prog.scale1;
  const int64_t bytes = p.rows * p.cols * 4;
  a.past = lanes_log2 >= 3 && (prog.walk2 >= 0 || !per_row || bytes <= kPastUpTo || bytes > kPastFrom);
  a.n_steps = prog.n;
  __builtin_memcpy(a.code, prog.code, sizeof a.code);
  __builtin_memcpy(a.imm, prog.imm, sizeof a.imm);
  const dim3 grid((unsigned)gx, (unsigned)gy);
  switch (dt) {
    case FRISK_F32: launch_held<FRISK_F32>(held, prog.scaled, grid, a, prog.depth, lanes_log2, s); break;
    case FRISK_F16: launch_held<FRISK_F16>(held, prog.scaled, grid, a, prog.depth, lanes_log2, s); break;
    case FRISK_BF16: launch_held<FRISK_BF16>(held, prog.scaled, grid, a, prog.depth, lanes_log2, s); break;
    default: launch_typed<-1, HELD_NONE>(grid, a, prog.depth, lanes_log2, s); break;
  }
  return hipGetLastError();
}

}  // namespace frisk
