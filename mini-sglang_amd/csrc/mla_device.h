// Device helpers shared by the gfx950 MLA decode kernels.
#pragma once

#include <type_traits>

#include "mla_common.h"

namespace mla {

// Row swizzle of the LDS tiles: 16-byte chunk c of token t is stored at chunk
// position c ^ swz(t & 7).
__device__ __forceinline__ int swz(int t7) { return ((t7 & 3) << 1) | ((t7 >> 2) & 1); }

// Decode LDS tile of the streaming kernels: nine 128-byte column blocks, [block][32 tokens][128 B]; 16-byte chunk
// ch of a block is stored at slot ch ^ tswz(token). Both operand reads are then bank-conflict free. A ds_read_b128
// serves 16 lanes of 16 different tokens at a time, 8 of a 16-lane group and 8 of its neighbour; the groups read
// chunks that differ by 2 (half 0 or 1 of a block: group g its chunk tperm(g); the same order for K and Q, so it only
// permutes the dims of an MFMA k-step). A transposing read serves the chunk pairs of 8 tokens, which lie in different
// slot pairs. Loads stay whole lines: a 1 KB DMA load is 8 tokens of a block, 128 bytes each, and a wave that loads
// token octet o of every block needs one source offset per lane, plus 128 bytes a block.
// (Rows of 1152 bytes with XOR-swizzled chunks left the K reads 2-way conflicted.)
constexpr int kTileBlocks = kRowBytes / 128;
constexpr int kTileBlockBytes = kTile * 128;
__device__ __forceinline__ int tswz(int t) { return (((t >> 1) & 3) << 1) | ((t >> 3) & 1); }
__device__ __forceinline__ int tperm(int g) { return ((g & 1) << 1) | (g >> 1); }
// lane's token of octet o, and its source offset in the token's row (first block)
__device__ __forceinline__ int octet_token(int o, int lane) { return 8 * o + (lane >> 3); }
__device__ __forceinline__ uint32_t octet_chunk(int lane, int token) { return ((lane & 7) ^ tswz(token)) << 4; }

// Combines a lane's value with lanes l ^ 16, l ^ 32 and l ^ 48 (the four lane groups; every lane gets the
// result) by v_permlane16_swap / v_permlane32_swap: no LDS traffic and no LDS latency.
template <typename F>
__device__ __forceinline__ float group_reduce(float v, F&& f) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float wave_max_g(float v) {
  return group_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum_g(float v) {
  return group_reduce(v, [](float a, float b) { return a + b; });
}

// A lane's value combined over the whole wave (every lane gets the result): four row rotations by DPP, then
// the group swaps: a dozen vector instructions, where six ds_bpermute steps wait out the LDS latency each.
template <typename F>
__device__ __forceinline__ float wave_reduce(float v, F&& f) {
  auto ror = [&](auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value,
                                                                  0xf, 0xf, false));
  };
  v = f(v, ror(std::integral_constant<int, 0x128>{}));  // row_ror:8
  v = f(v, ror(std::integral_constant<int, 0x124>{}));
  v = f(v, ror(std::integral_constant<int, 0x122>{}));
  v = f(v, ror(std::integral_constant<int, 0x121>{}));
  return group_reduce(v, f);
}
__device__ __forceinline__ float wave_max64(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum64(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

// Wait until at most N vector-memory operations of this wave are outstanding.
// The counter saturates at 63; a smaller count only waits longer, so N is clamped.
template <int N0>
__device__ __forceinline__ void wait_vmcnt() {
  constexpr int N = N0 > 63 ? 63 : N0;
  static_assert(N >= 0, "vmcnt range");
  // gfx9 encoding: vmcnt[3:0] | expcnt[6:4]=7 | lgkmcnt[11:8]=15 | vmcnt[5:4] at [15:14]
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x70 | 0xF00 | ((N >> 4) << 14));
}

// 16-byte global -> LDS DMA; lane i's data lands at LDS byte address
// lds_base + 16*i. Issued as inline asm so that the compiler's wait-count
// pass does not serialise later LDS reads of other stages behind it: every
// read of a staged tile is preceded by wait_vmcnt + a workgroup barrier.
// The compiler's hazard recognizer does not look inside inline asm, so the
// wait states it would add are written here: one between a scalar write of
// M0 (the compiler writes it just before the statement) and an LDS DMA. The
// base's scalar registers need five after a vector-ALU write: uniform_ptr
// waits them out, and the build checks the assembly for any other write (a
// spilled base's v_readlane), which this statement could not survive (waits of
// its own here cost a prefill step 1.3 %).
__device__ __forceinline__ void dma16_saddr(const char* base, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "{m0}"(lds_base) : "memory");
}
// All column blocks of a token octet, one wave's 9 loads of a tile, as one statement that waits for its own base: a
// base restored from a spill by a v_readlane right before the loads is then safe (with one statement per load, such a
// restore loaded from a wild address). Block i lies 128 i bytes into the row and 4096 i bytes into the tile; the
// immediate offset is added to the source and to the LDS address, so M0 steps by the difference. kNt: the
// non-temporal hint, for data read once (streamed KV rows), so the caches keep the lines that are reused.
#define MLA_DMA_BLOCK(offset, hint) \
  "s_add_u32 m0, m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:" #offset hint "\n\t"
#define MLA_DMA_OCTET(hint)                                                                                       \
  asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" hint "\n\t" MLA_DMA_BLOCK(128, hint)               \
               MLA_DMA_BLOCK(256, hint) MLA_DMA_BLOCK(384, hint) MLA_DMA_BLOCK(512, hint) MLA_DMA_BLOCK(640, hint) \
               MLA_DMA_BLOCK(768, hint) MLA_DMA_BLOCK(896, hint) MLA_DMA_BLOCK(1024, hint)                         \
               : "+{m0}"(lds_base) : "v"(voff), "s"(base), "n"(kTileBlockBytes - 128) : "scc", "memory")
template <bool kNt>
__device__ __forceinline__ void dma16_octet(const char* base, uint32_t voff, uint32_t lds_base) {
  static_assert(kTileBlocks == 9, "one load per column block");
  if constexpr (kNt) MLA_DMA_OCTET(" nt");
  else MLA_DMA_OCTET("");
}
#undef MLA_DMA_OCTET
#undef MLA_DMA_BLOCK
__device__ __forceinline__ void dma16_vaddr(const char* addr, uint32_t lds_base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(addr), "{m0}"(lds_base) : "memory");
}
// A 64-bit scalar base from a uniform vector value, for a DMA's address. A lane read needs a wait state
// after the vector-ALU write of its register (the compiler does not add it inside asm: without it the
// low half was read before a v_lshl_add_u64 wrote it), and a vector-ALU write of an SGPR needs 5 before a
// memory instruction reads it; readfirstlane and the nops are volatile asm, so they stay in order with the
// DMA asm statements that follow.
__device__ __forceinline__ const char* uniform_ptr(uint32_t lo, uint32_t hi) {
  uint32_t slo, shi;
  asm volatile("s_nop 0\n\tv_readfirstlane_b32 %0, %2\n\tv_readfirstlane_b32 %1, %3\n\ts_nop 4"
               : "=s"(slo), "=s"(shi) : "v"(lo), "v"(hi));
  return reinterpret_cast<const char*>(((uint64_t)shi << 32) | slo);
}

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  // round-to-nearest-even, matching torch's float->bfloat16 conversion; one v_cvt_pk_bf16_f32
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
}


// Workgroup barrier that orders LDS only: waits for this wave's LDS ops, then
// s_barrier. Unlike __syncthreads() it never waits on vector-memory counters,
// so in-flight DMA loads and output stores stay in flight.
__device__ __forceinline__ void barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Scalar (wave-uniform) 32-bit load, waited for before returning.
__device__ __forceinline__ int sload_i32(const int32_t* ptr) {
  int v;
  asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(ptr) : "memory");
  return v;
}

// Scalar load of four consecutive 32-bit values (16-byte aligned), waited for.
__device__ __forceinline__ void sload_i32x4(const int32_t* ptr, int& a, int& b, int& c, int& d) {
  typedef int i32x4_t __attribute__((__vector_size__(16)));
  i32x4_t v;
  asm volatile("s_load_dwordx4 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(ptr) : "memory");
  a = v[0];
  b = v[1];
  c = v[2];
  d = v[3];
}

// Binary tree of scalar branches over wait counts 8 Lo, 8 (Lo + 1), ... 8 Hi.
template <int Lo, int Hi>
__device__ __forceinline__ void wait_vmcnt_tree(int n) {
  if constexpr (Lo == Hi) {
    wait_vmcnt<8 * Lo>();
  } else {
    constexpr int Mid = (Lo + Hi) / 2;
    if (n < 8 * (Mid + 1)) wait_vmcnt_tree<Lo, Mid>(n);
    else wait_vmcnt_tree<Mid + 1, Hi>(n);
  }
}

// wait_vmcnt with a run-time count (clamped to the counter range, made wave-uniform so that the selection
// compiles to scalar branches). kUsual, the count of a loop's steady state, is tested first, and other counts
// (after a piece's stores, at the stream's end) wait for a multiple of 8, at most 7 operations more than they need:
// a tree of all 64 counts took about 550 cycles of a decode step's 3200 (split step of 64 requests of 1k to 8k
// tokens, 8 heads: 62.2 -> 58.9 us; 64 heads, with its marks and page ids kept a step ahead: 73.7 -> 71.1 us;
// 8 requests of 32k to 128k tokens, 64 heads: 158.5 -> 147.5 us).
template <int kUsual>
__device__ __forceinline__ void wait_vmcnt_dyn(int n) {
  n = __builtin_amdgcn_readfirstlane(n);
  if (n == kUsual) {
    wait_vmcnt<kUsual>();
    return;
  }
  wait_vmcnt_tree<0, 7>(n > 63 ? 63 : (n < 0 ? 0 : n));
}

}  // namespace mla
