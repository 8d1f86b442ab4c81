// Chunked MLA prefill (non-absorbed form), causal and bottom-right aligned over
// a paged prefix: query i of a request with prefix P attends keys j <= P + i.
// Per head: q [192] (128 nope + 64 rope), K [192], V [128]. A K row is read from two places: its
// 128 nope dims and, a per-head byte offset after them, its 64 rope dims (the per-head page layout
// [.., H, 192] has them adjacent; the latent-decompression scratch keeps one rope copy per token,
// shared by all heads, after the heads' [k_nope | v] blocks).
//
// One CTA per (request, 32 NW query rows, head), NW waves x 32 query rows, two waves per SIMD: NW = 8 (one CTA
// per compute unit) or NW = 4 (two; the launcher chooses by the requests' size).
//  * Keys stream in stages of 32 tokens (K 12 KB + V 8 KB) through a K ring and a V ring in LDS filled by
//    16-byte DMA loads (PShape). K rows (384 B) are stored with the
//    16-byte chunk index XOR ((token >> 1) & 7) inside each 8-chunk group, V rows
//    (256 B) with XOR 4 * (token & 3): the K operand reads (ds_read_b128) and the
//    transposing V reads (ds_read_b64_tr_b16) are then bank-conflict free, as
//    rocprof's SQ_LDS_BANK_CONFLICT reads them on this part (XOR (token & 7) and
//    XOR 2 * (token & 3) leave both 2-way conflicted).
//  * S^T[32 keys x 32 queries] = K . Q^T and O^T[128 dims x 32 queries] +=
//    V^T . P^T on 32x32x16 bf16 MFMA; queries (the B operand) and O stay in
//    registers for the whole head.
//  * Software pipeline over the stages: step j issues the value MFMAs of stage
//    j-1 and the score MFMAs of stage j+1 while the vector ALU runs the online
//    softmax of stage j, the two instruction streams interleaved slot by slot
//    (one MFMA per slot). Every step of a wave runs this same body: a diagonal
//    step first masks its stage's scores, the first step sets the reference,
//    and the last step's score pass works on a fully masked stage.
//  * Online softmax in the log2 domain against a lazy row reference: the exact
//    max of the wave's first stage, moved (with O and l rescaled, and the
//    stage redone) only when a stage's numerators sum past 2^32.
//  * The heads of one (request, query block) are consecutive CTAs, so the query blocks of one head are H
//    CTAs apart and, with that a multiple of 8, land on the same XCD and share its L2 for K/V.
// Bound: with whole 256-row blocks the step's chain of MFMAs, LDS operand reads and softmax; with many short
// requests the memory round trips of a CTA's start (requests, page table, queries, first stage), which the
// second CTA of a compute unit fills.
// Measured: four chunks of 2048 rows on prefixes of 4969 to 7961 keys, 64 heads, 2278 us (1159 TFLOP/s); 2293 us
// with K and V stages in one ring (the V reads' addresses then pass the 64 KB offset field, 8 more vector
// instructions per step) and two heads run by a CTA one after the other.
#include <type_traits>

#include "mla_common.h"
#include "mla_device.h"

namespace mla {
namespace {

typedef float f32x16_t __attribute__((__vector_size__(64)));

constexpr int kPStage = 32;                             // keys per stage
constexpr int kPKRowBytes = kPrefillQkDim * 2;          // 384
constexpr int kPVRowBytes = kPrefillVDim * 2;           // 256
constexpr int kPKBytes = kPStage * kPKRowBytes;         // 12288
constexpr int kPVBytes = kPStage * kPVRowBytes;         // 8192
// Shape of a CTA with NW waves of 32 query rows. K and V stages have rings of their own in LDS. DMA group n is K
// stage n and V stage n - kVLag; step j issues group j + kDist, scores stage j + 1 and adds the values of stage
// j - 1. Every kSync steps a barrier makes K stages up to j + kSync and V stages up to j + kSync - 1 visible to
// every wave; the rings are as long as that needs, so that no wave refills a stage another still reads.
//  NW = 8 (256 rows, one CTA per compute unit): barriers every two steps, loads four stages ahead.
//  NW = 4 (128 rows, two CTAs per compute unit): half the LDS, so V follows one group behind K (its stage is
//  needed two steps after K's), three stages ahead, a barrier per step; the other CTA fills the waits.
template <int NW>
struct PShape;
template <>
struct PShape<8> {
  static constexpr int kSync = 2, kDist = 4, kVLag = 0, kKRing = 7, kVRing = 7;
  static constexpr int kUnroll = 14;  // steps unrolled: whole rounds of the rings, and an even count (the score
                                      // and numerator registers alternate by step parity)
  static constexpr int kWindow = 1024;  // stage sources held in LDS at a time
};
template <>
struct PShape<4> {
  static constexpr int kSync = 1, kDist = 3, kVLag = 1, kKRing = 3, kVRing = 4;
  static constexpr int kUnroll = 12;
  static constexpr int kWindow = 512;
};
template <int NW>
constexpr bool shape_ok() {
  using S = PShape<NW>;
  // K live: stages j + 1 .. j + kDist and, until the next barrier, kSync - 1 older ones (read at step j: j + 1);
  // V live: j - 1 .. j + kDist - kVLag likewise
  return S::kKRing >= S::kDist + S::kSync - 1 && S::kVRing >= S::kDist - S::kVLag + 1 + S::kSync &&
         S::kUnroll % S::kKRing == 0 && S::kUnroll % S::kVRing == 0 && S::kUnroll % 2 == 0 &&
         S::kWindow > S::kUnroll + S::kVLag;  // a window holds the groups of kUnroll steps
}
static_assert(shape_ok<8>() && shape_ok<4>(), "ring lengths");
// Wave-wide 1 KiB DMA loads of a stage: 12 of the K tile and 8 of the V tile; load i of a tile lands at i KiB.
// With 4 waves wave w issues K loads w + 4k (k < 3) and V loads w + 4k (k < 2); with 8 waves, waves 0-3 issue
// the K loads (w + 4k, k < 3) and waves 4-7 the V loads ((w - 4) + 4k, k < 2).
constexpr int kPKDma = 3;  // K loads of a wave that issues K loads
constexpr int kPVDma = 2;  // V loads of a wave that issues V loads

// ---- the softmax of one stage as a list of micro-operations, spread over the MFMA slots of a
// pipelined step in proportion to their cost (~4-cycle units; next to running MFMAs a vector
// instruction costs ~8 cycles and exp2 ~11). A step has 8 value MFMAs + 12 score MFMAs (its slots)
// and 24 softmax micro-ops: for u = 3 k + r (pair k of a lane's 16 scores), r < 2 is the exp2 of
// score 2k + r against the row reference, r == 2 adds the pair to the row sum and packs it to bf16.
// No exp2 result is used by the next instruction (that would cost a wait state).
constexpr int kSlots = 20;
// LDS operand reads run ahead of their MFMAs: K operand ks + kAK is read in the slot of K operand
// ks, V^T operand st + kAV in the slot of V^T operand st (the first kAV by the step before)
constexpr int kAK = 4, kAV = 3;
static_assert(kAK >= 3 && kAK <= 8 && kAV >= 1 && kAV <= 12, "read-ahead outside the step's slots");
constexpr int kUops = 24;
constexpr int uop_weight(int u) { return u % 3 < 2 ? 5 : 6; }
constexpr int uop_total() {
  int t = 0;
  for (int u = 0; u < kUops; ++u) t += uop_weight(u);
  return t;
}
constexpr int uop_slot(int u) {
  int t = 0;
  for (int v = 0; v < u; ++v) t += uop_weight(v);
  return t * kSlots / uop_total();
}
// The row reference m (log2 domain) is the exact max of the wave's first stage and moves only when
// a stage's numerators sum past 2^32 (a score 32 above m, in log2 units) or overflow: then that
// stage is redone against its exact max. fp32 keeps its relative precision at any scale, so the
// lagging reference costs no accuracy.
constexpr float kPLazyMax = 4294967296.0f;

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ int kswz(int c, int t) { return (c & ~7) | ((c & 7) ^ ((t >> 1) & 7)); }
__device__ __forceinline__ int vswz(int c, int t) { return c ^ (4 * (t & 3)); }
// max / sum of a lane's value with lane ^ 32 (v_permlane32_swap, no LDS traffic)
__device__ __forceinline__ float max_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// S^T += K . Q^T and O^T += V^T . P^T: builtins, so that the compiler places the MFMAs' wait states.
__device__ __forceinline__ void mfma_qk(f32x16_t& d, const bf16x8& k, const bf16x8& q) {
  d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, q, d, 0, 0, 0);
}
__device__ __forceinline__ void mfma_pv(f32x16_t& o, const bf16x8& v, const u32x4& p) {
  o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, __builtin_bit_cast(bf16x8, p), o, 0, 0, 0);
}
// keeps an output block in the vector registers and its MFMA in its slot
__device__ __forceinline__ void pin_o(f32x16_t& o) { asm volatile("" : "+v"(o)); }

// Pin a vector-ALU result to its slot of the instruction stream: volatile asm statements keep their order, and the
// slots' scheduling barriers keep each on its side.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(uint32_t& x) { asm volatile("" : "+v"(x)); }

template <int N>
using ic = std::integral_constant<int, N>;
// f(ic<0>{}), ..., f(ic<N-1>{}): a loop whose index is a compile-time constant in the body
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(ic<I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int NW>  // waves
__global__ __launch_bounds__(NW * 64, 2) void mla_prefill_kernel(const PrefillParams p) {
  using S = PShape<NW>;
  constexpr bool kBoth = NW == 4;  // every wave issues K and V loads
  constexpr int kRows = 32 * NW;   // query rows of the CTA
  constexpr int kKRingBytes = S::kKRing * kPKBytes;
  // the K ring, the V ring, then 1 KB that the loads of dummy DMA groups land in
  __shared__ __attribute__((aligned(1024))) char smem[kKRingBytes + S::kVRing * kPVBytes + 1024];
  __shared__ __attribute__((aligned(16))) uint32_t s_src[S::kWindow][4];  // K and V source of a window's stages

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = p.heads;

  // ---- work item: request b, query block qb, head h (heads fastest). A request's last items (the latest query blocks,
  // which see the most keys) are dispatched first, and of up to 64 requests the one with the most keys first: the long
  // CTAs then do not run alone at the end (chunks of 531, 354 and 604 rows on prefixes of 2666, 197 and 296 keys, 64
  // heads: 119.3 us, 123.7 us in reverse request order)
  int b = -1, local = 0, q0 = 0, E = 0, L = 0;
  int item = (int)blockIdx.x;
  if (p.batch <= 64) {
    const bool in = lane < p.batch;
    const int lo = in ? p.cu_seqlens_q[lane] : 0, hi = in ? p.cu_seqlens_q[lane + 1] : 0, lk = in ? p.seq_lens_k[lane] : 0;
    const int n = in ? ((hi - lo + kRows - 1) / kRows) * H : 0;
    int excl = 0;  // items of the requests before this lane's: longer ones, and as long ones of a lower index
    for (int i = 0; i < p.batch; ++i) {
      const int ni = __builtin_amdgcn_readlane(n, i), li = __builtin_amdgcn_readlane(lk, i);
      if (li > lk || (li == lk && i < lane)) excl += ni;
    }
    const uint64_t hit = __ballot(in && item >= excl && item < excl + n);
    if (hit != 0) {
      const int fl = __builtin_ctzll(hit);
      b = fl;
      local = __builtin_amdgcn_readlane(n, fl) - 1 - (item - __builtin_amdgcn_readlane(excl, fl));
      q0 = __builtin_amdgcn_readlane(lo, fl);
      E = __builtin_amdgcn_readlane(hi, fl) - q0;
      L = __builtin_amdgcn_readlane(lk, fl);
    }
  } else {
    auto items_of = [&](int r) __attribute__((always_inline)) {
      return r < p.batch ? ((p.cu_seqlens_q[r + 1] - p.cu_seqlens_q[r] + kRows - 1) / kRows) * H : 0;
    };
    int total = 0;
    for (int c0 = 0; c0 < p.batch; c0 += 64) total += wave_sum(items_of(c0 + lane));
    total = __builtin_amdgcn_readfirstlane(total);
    item = total - 1 - item;
    int acc = 0;
    for (int c0 = 0; item >= 0 && c0 < p.batch && b < 0; c0 += 64) {
      const int r = c0 + lane;
      const bool in = r < p.batch;
      // the request's query range and key count come with the scan (no second memory round trip)
      const int lo = in ? p.cu_seqlens_q[r] : 0, hi = in ? p.cu_seqlens_q[r + 1] : 0, lk = in ? p.seq_lens_k[r] : 0;
      const int n = in ? ((hi - lo + kRows - 1) / kRows) * H : 0;
      int incl = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
      }
      const int excl = incl - n;
      const uint64_t hit = __ballot(r < p.batch && item >= acc + excl && item < acc + incl);
      if (hit != 0) {
        const int fl = __builtin_ctzll(hit);
        b = c0 + fl;
        local = item - acc - __shfl(excl, fl);
        q0 = __shfl(lo, fl);
        E = __shfl(hi, fl) - q0;
        L = __shfl(lk, fl);
      }
      acc += __shfl(incl, 63);
    }
  }
  b = __builtin_amdgcn_readfirstlane(b);
  if (b < 0) return;  // uniform: beyond the last item
  local = __builtin_amdgcn_readfirstlane(local);
  q0 = __builtin_amdgcn_readfirstlane(q0);
  E = __builtin_amdgcn_readfirstlane(E);
  L = __builtin_amdgcn_readfirstlane(L);
  const int h = local % H;
  const int qb = local / H;
  const int P = L - E;  // prefix length
  const int row0 = qb * kRows + 32 * wave;  // this wave's first query row in the request
  const int cta_rows_end = min(E, (qb + 1) * kRows);
  const int nkeys = P + cta_rows_end;  // keys the CTA needs
  const int nst = __builtin_amdgcn_readfirstlane((nkeys + kPStage - 1) / kPStage);
  const int wave_rows = max(0, min(E - row0, 32));
  const int W =  // stages this wave needs
      __builtin_amdgcn_readfirstlane(wave_rows > 0 ? (P + row0 + wave_rows + kPStage - 1) / kPStage : 0);

  const int g32 = lane >> 5;  // half of the wave
  const int c32 = lane & 31;
  const int ps_mask = (1 << p.log2_ps) - 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MLA_LDS char*)smem;

  // queries of head h: qf[ks] = row row0 + c32, dims 16ks + 8g32 .. +8 (a column past the
  // extend loads the first row: finite scores in a column whose output is not written; no select,
  // so that nothing waits for these loads before the first ring loads are issued)
  bf16x8 qf[12];
  auto load_q = [&]() __attribute__((always_inline)) {
    const int row = row0 + c32;
    const bool ok = row < E;
    const __bf16* qrow = p.q + (int64_t)(q0 + (ok ? row : 0)) * p.q_stride_t + (int64_t)h * p.q_stride_h + 8 * g32;
#pragma unroll
    for (int ks = 0; ks < 12; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(qrow + 16 * ks);
  };

  // a K row is 128 nope dims at kbase (+ token row) and 64 rope dims rope_delta bytes after them
  // (the host checks 0 <= rope_delta < 2^31 for every head)
  const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)h * p.k_head_stride * 2;
  const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)h * p.v_head_stride * 2;
  const uint32_t rope_delta = (uint32_t)(p.k_rope_delta0 + (int64_t)h * p.k_rope_delta_h);
  const int krow_bytes = (int)(p.k_row_stride * 2), vrow_bytes = (int)(p.v_row_stride * 2);
  // source byte offset of logical K chunk c (16 bytes; 0..15 nope, 16..23 rope) of a row
  auto kchunk_src = [&](int c) __attribute__((always_inline)) {
    return c < 16 ? (uint32_t)(c * 16) : rope_delta + (uint32_t)((c - 16) * 16);
  };
  // bytes of one page of K / V rows (< 4 GiB, checked by the host)
  const uint32_t kpage_bytes = (uint32_t)krow_bytes << p.log2_ps, vpage_bytes = (uint32_t)vrow_bytes << p.log2_ps;
  // first source row of the stage that starts at token t0, on page pid
  auto stage_src = [&](const char* base, uint32_t pid, int t0, uint32_t page_bytes, int row_bytes)
                       __attribute__((always_inline)) {
    return base + ((uint64_t)pid * page_bytes + (uint32_t)((t0 & ps_mask) * row_bytes));
  };

  // ---- source addresses of the CTA's full stages, a window of them at a time: s_src[i] is stage w0 + i's; stage
  // n_defer's is the first stage's, the source of dummy groups. The step loop fills the next window when its next
  // kUnroll steps would pass this one (every 500 steps and more: one drain of the loads). With a single window, CTAs
  // of more keys than it holds loaded each stage at once after a page-table read, with no loads ahead; single -> next
  // windows: 2048 rows on 20,000 keys, 8 heads 628 -> 366 us; 40 rows on 30,000, 64 heads 909 -> 480; four of 512
  // rows on 16,000 1662 -> 1196; 2048 rows on 40,000 (256-row CTAs) 3293 -> 2860.
  const int n_defer = min(nst, L >> 5);  // stages the pipelined step may load itself
  int w0 = 0;
  auto stage_window = [&](auto&& between) __attribute__((always_inline)) {
    constexpr int kPer = S::kWindow / (NW * 64);  // entries per thread
    static_assert(kPer * NW * 64 == S::kWindow, "every thread fills as many entries");
    int pid_u[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int g = w0 + threadIdx.x + NW * 64 * u;
      const int t0 = g < n_defer ? g * kPStage : 0;  // (an unconditional read: the first page's entry)
      pid_u[u] = p.page_table[(int64_t)b * p.pt_stride + (t0 >> p.log2_ps)];
    }
    between();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = threadIdx.x + NW * 64 * u, g = w0 + i;
      if (g > n_defer) continue;
      const int t0 = g < n_defer ? g * kPStage : 0;
      const uint32_t pid = (uint32_t)min(max(pid_u[u], 0), p.num_pages - 1);
      const uint64_t ka = (uint64_t)stage_src(kbase, pid, t0, kpage_bytes, krow_bytes);
      const uint64_t va = (uint64_t)stage_src(vbase, pid, t0, vpage_bytes, vrow_bytes);
      *reinterpret_cast<MLA_LDS u32x4*>((MLA_LDS char*)s_src + 16 * i) =
          u32x4{(uint32_t)ka, (uint32_t)(ka >> 32), (uint32_t)va, (uint32_t)(va >> 32)};
    }
  };
  // the page-table reads, then the queries, then the table writes: the writes wait
  // for the page-table reads alone, and the queries stay in flight behind the first ring loads
  stage_window([&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    load_q();
    __builtin_amdgcn_sched_barrier(0);
  });
  barrier_lds();  // the source table is written (the queries may still be in flight)

  // ---- DMA of stage n (32 tokens of one page: page_size >= 64); rows past the last key load the
  // last key. LDS position s (16 bytes each) of the K tile holds token s / 24, chunk kswz(s % 24);
  // of the V tile token s / 16, chunk vswz(s % 16).
  const int wq = wave & 3;
  const bool k_wave = kBoth || wave < 4;  // this wave issues K loads wq + 4k
  const bool v_wave = kBoth || wave >= 4;  // this wave issues V loads wq + 4k
  constexpr int kPDmaMax = kBoth ? kPKDma + kPVDma : kPKDma;  // loads per wave and group, at most
  uint32_t koff[kPKDma], voff[kPVDma];
#pragma unroll
  for (int k = 0; k < kPKDma; ++k) {
    const int s = (wq + 4 * k) * 64 + lane, t = s / 24;
    koff[k] = (uint32_t)(t * krow_bytes) + kchunk_src(kswz(s - 24 * t, t));
  }
#pragma unroll
  for (int k = 0; k < kPVDma; ++k) {
    const int s = (wq + 4 * k) * 64 + lane, t = s >> 4;
    voff[k] = (uint32_t)(t * vrow_bytes + vswz(s & 15, t) * 16);
  }
  // DMA groups (a wave's loads of one K stage and one V stage: 5 loads with 4 waves; 3 or 2 with 8) are issued
  // in order, stage n into ring slot n % ring. Every step issues exactly one group, one load at a time in its
  // slots: stages that are full, otherwise dummy loads (the first stage again, every
  // load into one 1 KB area past the rings, which nothing reads), so that the slots carry no branches; a tail
  // stage is loaded at once, ahead of those dummies.
  // With 8 waves a wave's loads are all K or all V, so its slot work is one list: per-lane source offsets
  // doff, the source from entry half src_sel of the stage's s_src row, the LDS destination from ring_lds
  // (the V-only waves' third load is absent).
  const uint32_t lds_v = lds0 + kKRingBytes, lds_dummy = lds_v + S::kVRing * kPVBytes;
  const uint32_t ring_lds = (k_wave ? lds0 : lds_v) + wq * 1024, ring_stage = k_wave ? kPKBytes : kPVBytes;
  const int src_sel = k_wave ? 0 : 8;
  uint32_t doff[kPKDma];
#pragma unroll
  for (int d = 0; d < kPKDma; ++d) doff[d] = k_wave ? koff[d] : voff[d < kPVDma ? d : kPVDma - 1];
  int n_groups = 0;
  // the step's group: s_src entry, LDS destination of this wave's first load and distance of its successive
  // loads (0 for dummies); [0] K (with 8 waves: the wave's tile), [1] V
  int dma_idx[2] = {0, 0};
  uint32_t dma_m0w[2] = {0, 0}, dma_pst[2] = {0, 0};
  auto load_now = [&](int n, bool do_k, bool do_v) __attribute__((always_inline)) {  // stage n < nst, all loads now
    const int t0 = n * kPStage;
    const int tlim = L - 1 - t0;
    const uint32_t pid = (uint32_t)min(
        max(sload_i32(p.page_table + (int64_t)b * p.pt_stride + (t0 >> p.log2_ps)), 0), p.num_pages - 1);
    // (the sources through readfirstlane: under register pressure the compiler may keep these
    // uniform values in vector registers, which the DMA's scalar base operand cannot take)
    const uint64_t ka = (uint64_t)stage_src(kbase, pid, t0, kpage_bytes, krow_bytes);
    const uint64_t va = (uint64_t)stage_src(vbase, pid, t0, vpage_bytes, vrow_bytes);
    const char* ksrc = uniform_ptr((uint32_t)ka, (uint32_t)(ka >> 32));
    const char* vsrc = uniform_ptr((uint32_t)va, (uint32_t)(va >> 32));
    // rows past the last key reload the last key (the lane index from a volatile asm, so that these
    // offsets are computed here and not kept in registers across the loop)
    int ln;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
    if (do_k) {
      const uint32_t st = lds0 + (uint32_t)(n % S::kKRing) * kPKBytes;
#pragma unroll
      for (int k = 0; k < kPKDma; ++k) {
        const int s = (wq + 4 * k) * 64 + ln, t = s / 24;
        const uint32_t o = (uint32_t)(min(t, tlim) * krow_bytes) + kchunk_src(kswz(s - 24 * t, t));
        dma16_saddr(ksrc, o, st + (wq + 4 * k) * 1024);
      }
    }
    if (do_v) {
      const uint32_t st = lds_v + (uint32_t)(n % S::kVRing) * kPVBytes;
#pragma unroll
      for (int k = 0; k < kPVDma; ++k) {
        const int s = (wq + 4 * k) * 64 + ln, t = s >> 4;
        const uint32_t o = (uint32_t)(min(t, tlim) * vrow_bytes + vswz(s & 15, t) * 16);
        dma16_saddr(vsrc, o, st + (wq + 4 * k) * 1024);
      }
    }
  };
  // the group of a step; uk, uv: the ring slots of its K and V stage (the unrolled loop knows them), or -1 to
  // compute them
  auto group_setup = [&](auto uk_c, auto uv_c) __attribute__((always_inline)) {
    constexpr int UK = decltype(uk_c)::value, UV = decltype(uv_c)::value;
    if constexpr (!kBoth) {
      const bool real = n_groups < n_defer;
      dma_idx[0] = min(n_groups, n_defer) - w0;
      dma_m0w[0] = real ? ring_lds + (UK >= 0 ? UK : n_groups % S::kKRing) * ring_stage : lds_dummy;
      dma_pst[0] = real ? 4 * 1024 : 0;
      if (__builtin_expect(!real && n_groups < nst, 0)) load_now(n_groups, k_wave, v_wave);
    } else {
      const int nv = n_groups - S::kVLag;
      const bool real_k = n_groups < n_defer, real_v = nv >= 0 && nv < n_defer;
      dma_idx[0] = min(n_groups, n_defer) - w0;
      dma_m0w[0] = real_k ? lds0 + wq * 1024 + (UK >= 0 ? UK : n_groups % S::kKRing) * kPKBytes : lds_dummy;
      dma_pst[0] = real_k ? 4 * 1024 : 0;
      dma_idx[1] = min(max(nv, 0), n_defer) - w0;
      dma_m0w[1] = real_v ? lds_v + wq * 1024 + (UV >= 0 ? UV : nv % S::kVRing) * kPVBytes : lds_dummy;
      dma_pst[1] = real_v ? 4 * 1024 : 0;
      if (__builtin_expect(!real_k && n_groups < nst, 0)) load_now(n_groups, true, false);
      if (__builtin_expect(!real_v && nv >= 0 && nv < nst, 0)) load_now(nv, false, true);
    }
    ++n_groups;
  };
  // slot work of the step's group: part 0 reads its sources (in the step, so the compiler waits
  // for that LDS read alone), parts 1..kPDmaMax issue the loads (a V-only wave has no part 3)
  u32x2 dma_ek, dma_ev;
  const char* dma_k = kbase;
  const char* dma_v = vbase;
  auto dma_part = [&](int k) __attribute__((always_inline)) {
    if (k == 0) {
      dma_ek = *reinterpret_cast<const MLA_LDS u32x2*>((const MLA_LDS char*)s_src + 16 * dma_idx[0] + (kBoth ? 0 : src_sel));
      if constexpr (kBoth)
        dma_ev = *reinterpret_cast<const MLA_LDS u32x2*>((const MLA_LDS char*)s_src + 16 * dma_idx[1] + 8);
      return;
    }
    const int d = k - 1;
    if (d == 0) dma_k = uniform_ptr(dma_ek[0], dma_ek[1]);
    if constexpr (kBoth) {
      if (d == kPKDma) dma_v = uniform_ptr(dma_ev[0], dma_ev[1]);
      if (d < kPKDma) dma16_saddr(dma_k, koff[d], dma_m0w[0] + d * dma_pst[0]);
      else dma16_saddr(dma_v, voff[d - kPKDma], dma_m0w[1] + (d - kPKDma) * dma_pst[1]);
    } else {
      if (d < kPVDma || k_wave) dma16_saddr(dma_k, doff[d], dma_m0w[0] + d * dma_pst[0]);
    }
  };
  // all loads of the step's group at once (a wave without work in the step, and the groups before
  // the first step)
  auto group_now = [&](auto uk_c, auto uv_c) __attribute__((always_inline)) {
    group_setup(uk_c, uv_c);
#pragma unroll
    for (int k = 0; k <= kPDmaMax; ++k) dma_part(k);
  };
  // the stages before the last NG groups a wave issued have landed for every wave, and every wave
  // is done with the steps before (so the stages they finished with may be refilled). Every step
  // issues exactly one group (a step that loads a tail stage at once issues one more, which only
  // makes the wait stricter), so at most (loads per group) NG loads may still be in flight.
  auto sync_groups = [&](auto ng_c) __attribute__((always_inline)) {
    constexpr int NG = decltype(ng_c)::value;
    if (kBoth) wait_vmcnt<(kPKDma + kPVDma) * NG>();
    else if (k_wave) wait_vmcnt<kPKDma * NG>();
    else wait_vmcnt<kPVDma * NG>();
    __builtin_amdgcn_s_barrier();
  };
  // a barrier step n: groups up to n + kSync landed; steps n .. n + kSync - 1 read K stages up to n + kSync and V
  // stages up to n + kSync - 1
  auto step_sync = [&]() __attribute__((always_inline)) { sync_groups(ic<S::kDist - 1 - S::kSync>{}); };

  for (int g = 0; g < S::kDist - 1; ++g) group_now(ic<-1>{}, ic<-1>{});
  // the queries stay in registers and have landed here, with the first loads of the ring issued behind
  // them. The wait is explicit and full: the compiler does not count the DMA loads (inline assembly).
  wait_vmcnt<0>();
#pragma unroll
  for (int ks = 0; ks < 12; ++ks) asm volatile("" : "+v"(qf[ks]));

  // ---- per-lane LDS read offsets
  // K operand of k-step ks = 4m + r: chunk 8m + 2r + g32 of key c32 at k_off[r] + 128m
  int k_off[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) k_off[r] = c32 * kPKRowBytes + kswz(2 * r + g32, c32) * 16;
  // V^T operand: 16-lane group gq = lane / 16 covers dims 16(gq & 1) .. +16 of a 32-dim block and
  // the key quarter vh = gq >> 1; lane a16 reads token 4vh + (a16 >> 2) (+ 16 ksp + 8 second), dims
  // 4(a16 & 3) .. +4; chunk 4db + y (y < 4) of token t is stored at 4(db ^ (t & 3)) + y
  const int gq = lane >> 4, a16 = lane & 15, vh = gq >> 1, vt = a16 >> 2;
  int v_off[4];
  {
    const int y = 2 * (gq & 1) + ((a16 & 3) >> 1);
#pragma unroll
    for (int db = 0; db < 4; ++db) v_off[db] = kKRingBytes + (4 * vh + vt) * kPVRowBytes + (4 * (db ^ vt) + y) * 16 + (a16 & 1) * 8;
  }
  // K operand ks of the stage at byte offset `kt` of the K ring
  auto kread = [&](int kt, int ks) __attribute__((always_inline)) {
    return *reinterpret_cast<const MLA_LDS bf16x8*>((const MLA_LDS char*)smem + kt + k_off[ks & 3] +
                                                   128 * (ks >> 2));
  };
  // V^T operand st = (32-dim block db = st / 2, 16-key step ksp = st % 2) of the stage at byte offset
  // `vt_` of the V ring; its
  // k order (keys 16ksp + 8e + 4g32 + (0..3), e = 0, 1) matches the lanes' P^T values
  auto vop = [&](int vt_, int st) __attribute__((always_inline)) {
    const int db = st >> 1, ksp = st & 1;
    const MLA_LDS char* base = (const MLA_LDS char*)smem + vt_ + v_off[db] + 16 * ksp * kPVRowBytes;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((MLA_LDS bf16x4*)base);
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((MLA_LDS bf16x4*)(base + 8 * kPVRowBytes));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  f32x16_t O[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) O[db] = f32x16_t{};
  float m_ref = -INFINITY, l_run = 0.f;
  f32x16_t sc[2];  // [parity]: scores of the stage being softmaxed / being computed
  u32x4 pb[2][2];  // [parity][ksp]: bf16 numerators P^T
  bf16x8 vb[kAV + 1];  // V^T operands in flight (the first kAV of a step are read by the step before)
  bf16x8 kb[kAK + 1];  // K operands in flight

  // ---- scores of stage 0 (before the first pipelined step)
  auto qk_plain = [&](f32x16_t& dst, int kt) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) kb[r] = kread(kt, r);
#pragma unroll
    for (int ks = 0; ks < 12; ++ks) {
      const bf16x8 a = kb[ks & 3];
      if (ks + 4 < 12) kb[ks & 3] = kread(kt, ks + 4);
      if (ks == 0) dst = f32x16_t{};
      mfma_qk(dst, a, qf[ks]);
    }
  };
  // causal mask of stage j's scores (stages that reach past the wave's first query); all == true
  // masks every score
  auto mask_scores = [&](f32x16_t& sv, int j, bool all) __attribute__((always_inline)) {
    // key kfirst + 8(i/4) + 4 g32 + i%4 follows query P + row0 + c32 when
    // 8(i/4) + i%4 > lim, lim = P + row0 + c32 - kfirst - 4 g32
    const int lim = all ? -1 : P + row0 + c32 - j * kPStage - 4 * g32;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (8 * (i >> 2) + (i & 3) > lim) sv[i] = -INFINITY;
  };
  float negm = 0.f;  // -reference (log2 domain)
  // reference of the wave's first stage: its exact row max
  auto init_ref = [&](f32x16_t& sv) __attribute__((always_inline)) {
    float m = sv[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) m = fmaxf(m, sv[i]);
    m_ref = max_halves(m) * p.scale_log2;
    negm = -m_ref;
  };
  // stage j again, its reference raised to its exact max (rare): from its raw (masked) scores,
  // which the pipelined step keeps; O and l (which hold the stages before it) rescaled; numerators
  // and their sum redone
  auto redo_stage = [&](f32x16_t& sv, u32x4 (&dst)[2], float& l_step) __attribute__((always_inline)) {
    float m = sv[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) m = fmaxf(m, sv[i]);
    const float m_new = fmaxf(max_halves(m) * p.scale_log2, m_ref);
    const float fr = __builtin_amdgcn_exp2f(m_ref - m_new);
    m_ref = m_new;
    negm = -m_new;
    l_run *= fr;
    float l = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float e0 = __builtin_amdgcn_exp2f(fmaf(sv[2 * k], p.scale_log2, negm));
      const float e1 = __builtin_amdgcn_exp2f(fmaf(sv[2 * k + 1], p.scale_log2, negm));
      l += e0 + e1;
      dst[k >> 2][k & 3] = pack_bf16x2(e0, e1);
    }
    l_step = l;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      O[db] *= fr;
      pin_o(O[db]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- pipelined step j: value MFMAs of stage j - 1 (slots 0 .. 7), score MFMAs of stage
  // j + 1 (the next 12 slots), softmax of stage j spread over all slots; one MFMA per slot, the
  // order pinned by scheduling barriers; LDS operand reads kAK / kAV operands ahead.
  // step j = j0 + U with j0 a multiple of both rings: the slots of V stages j - 1 and j and of K stage j + 1
  // are compile-time constants
  auto step_fast = [&](auto par_c, auto u_c) __attribute__((always_inline)) {
    constexpr int U = decltype(u_c)::value;
    constexpr int v_prev = (U + S::kVRing - 1) % S::kVRing * kPVBytes;
    constexpr int v_cur = U % S::kVRing * kPVBytes;
    constexpr int k_next = (U + 1) % S::kKRing * kPKBytes;
    constexpr int par = decltype(par_c)::value;
    constexpr int NS = kSlots;
    constexpr int kDmaPeriod = NS / kPDmaMax;  // DMA part p (1..) goes to slot kDmaPeriod (p - 1) + 3
    f32x16_t& scs = sc[par];
    f32x16_t& scn = sc[par ^ 1];
    u32x4(&pbw)[2] = pb[par];
    const u32x4(&pbr)[2] = pb[par ^ 1];
    const int kt = k_next, vtile = v_prev;
    float l_step, ev[2];  // ev: the numerators of the pair being packed (raw scores stay)
    float l_step_max;
    auto uop = [&](auto u_c) __attribute__((always_inline)) {
      constexpr int u = decltype(u_c)::value;
      constexpr int k = u / 3, r = u % 3;
      if constexpr (r < 2) {
        ev[r] = __builtin_amdgcn_exp2f(fmaf(scs[2 * k + r], p.scale_log2, negm));
        pin(ev[r]);
      } else {
        l_step = k == 0 ? ev[0] + ev[1] : l_step + ev[0] + ev[1];
        uint32_t w = pack_bf16x2(ev[0], ev[1]);
        pin(l_step);
        pin(w);
        pbw[k >> 2][k & 3] = w;
      }
    };
    static_for<NS>([&](auto s_c) __attribute__((always_inline)) {
      constexpr int s = decltype(s_c)::value;
      if constexpr (s < 8) {
        constexpr int st = s;
        mfma_pv(O[st >> 1], vb[st % (kAV + 1)], pbr[st & 1]);
        pin_o(O[st >> 1]);
      } else {
        constexpr int ks = s - 8;
        if constexpr (ks == 0) scn = f32x16_t{};
        mfma_qk(scn, kb[ks % (kAK + 1)], qf[ks]);
      }
      if constexpr (s == 0) dma_part(0);  // the stage refill, spread over the step
      if constexpr (s % kDmaPeriod == 3 && s / kDmaPeriod < kPDmaMax) dma_part(s / kDmaPeriod + 1);
      {  // operand reads
        constexpr int st = s + kAV, stn = s + kAV - 20, ks = s - 8 + kAK;
        if constexpr (st < 8) vb[st % (kAV + 1)] = vop(vtile, st);
        if constexpr (stn >= 0 && stn < kAV) vb[stn % (kAV + 1)] = vop(v_cur, stn);  // the next step's
        if constexpr (ks >= 0 && ks < 12) kb[ks % (kAK + 1)] = kread(kt, ks);
      }
      static_for<kUops>([&](auto u_c) __attribute__((always_inline)) {
        if constexpr (uop_slot(decltype(u_c)::value) == s) uop(u_c);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    // any lane's sum at 2^32 or more, or infinite: one compare into a lane mask, no reduction
    uint64_t big;
    asm volatile("v_max_f32 %1, %2, %3\n\tv_cmp_le_f32_e64 %0, %4, %1"
                 : "=s"(big), "=&v"(l_step_max) : "v"(l_step), "v"(l_step), "v"(kPLazyMax));
    if (big != 0) redo_stage(scs, pbw, l_step);
    l_run += l_step;
  };

  // step j <= W of a wave: the pipelined step. At j = 0 the value pass has no stage to add and is
  // undone; at j = W - 1 the scores of stage W are computed, and at
  // j = W fully masked, so that step W only adds the values of stage W - 1.
  const int j_diag = (P + row0 + 1) >> 5;  // first stage that reaches past the wave's first query
  auto step = [&](auto u_c, int j) __attribute__((always_inline)) {
    constexpr int U = decltype(u_c)::value;
    constexpr int par = U & 1;
    using uk_c = ic<(U + S::kDist) % S::kKRing>;
    using uv_c = ic<(U + S::kDist - S::kVLag) % S::kVRing>;
    if (j > nst) return;  // uniform over the CTA: past the last stage
    if constexpr (U % S::kSync == 0) step_sync();
    if (__builtin_expect(j <= W && W > 0, 1)) {
      group_setup(uk_c{}, uv_c{});
      if (__builtin_expect(j >= j_diag, 0)) mask_scores(sc[par], j, j == W);
      if constexpr (U == 0) if (__builtin_expect(j == 0, 0)) init_ref(sc[par]);
      step_fast(ic<par>{}, u_c);
      if constexpr (U == 0) if (__builtin_expect(j == 0, 0)) {
        // step 0 has no stage before it: its value pass multiplied zero numerators with whatever the V ring's
        // last slot held (NaN, if the LDS was left so), which must not count
#pragma unroll
        for (int db = 0; db < 4; ++db) O[db] = f32x16_t{};
      }
    } else {
      group_now(uk_c{}, uv_c{});
    }
  };

  // step -1: scores of stage 0; then steps 0..nst (every wave takes every barrier; the unrolled
  // steps past nst are skipped). A wave without rows has W = 0 and only takes the barriers and
  // loads its groups.
  pb[1][0] = pb[1][1] = u32x4{};
  sync_groups(ic<S::kDist - 2>{});  // K and V stage 0 landed (every wave has waited for all its loads above)
  group_now(ic<-1>{}, ic<-1>{});
  if (W > 0) {
    qk_plain(sc[0], 0);
#pragma unroll
    for (int st = 0; st < kAV; ++st) vb[st] = vop(0, st);
  }
  for (int j0 = 0; j0 <= nst; j0 += S::kUnroll) {
    // the next kUnroll steps issue K stages j0 + kDist .. + kUnroll - 1 and V stages kVLag behind them
    if (__builtin_expect(w0 + S::kWindow <= min(j0 + S::kDist + S::kUnroll - 1, n_defer), 0)) {
      barrier_lds();  // every wave is done with the window's entries
      w0 = j0 + S::kDist - S::kVLag;
      // (a wait of its own: page-table reads that a path leaves open make every step wait for all its loads)
      stage_window([] { wait_vmcnt<0>(); });
      barrier_lds();
    }
    static_for<S::kUnroll>([&](auto u_c) __attribute__((always_inline)) { step(u_c, j0 + decltype(u_c)::value); });
  }
  wait_vmcnt<0>();  // the last groups' loads into LDS have landed before the CTA ends

  // ---- finalise: lane holds query column c32 and dims 32db + 8(i/4) + 4*g32 + i%4
  const int row = row0 + c32;
  const float l_tot = sum_halves(l_run);
  if (row >= E || wave_rows == 0) return;
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  __bf16* orow = p.out + (int64_t)(q0 + row) * p.out_stride_t + (int64_t)h * p.out_stride_h;
  auto packed = [&](int db, int i4) {  // dims 32db + 8i4 + 4g32 .. +4 of this lane's row
    u32x2 v;
    v[0] = pack_bf16x2(O[db][4 * i4 + 0] * inv, O[db][4 * i4 + 1] * inv);
    v[1] = pack_bf16x2(O[db][4 * i4 + 2] * inv, O[db][4 * i4 + 3] * inv);
    return v;
  };
  if (p.out_16b) {
    // 16-byte stores (half the store instructions): the lanes of a row (c32, g32 = 0, 1) swap
    // one 8-byte part of each 16 dims, so that lane g32 holds dims 32db + 16m + 8g32 .. +8
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const u32x2 va = packed(db, 2 * m), vb = packed(db, 2 * m + 1);
        const u32x2 x = g32 == 0 ? vb : va;
        const uint32_t y0 = (uint32_t)__shfl_xor((int)x[0], 32), y1 = (uint32_t)__shfl_xor((int)x[1], 32);
        const u32x4 v = g32 == 0 ? u32x4{va[0], va[1], y0, y1} : u32x4{y0, y1, vb[0], vb[1]};
        *reinterpret_cast<u32x4*>(orow + 32 * db + 16 * m + 8 * g32) = v;
      }
  } else {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) *reinterpret_cast<u32x2*>(orow + 32 * db + 8 * i4 + 4 * g32) = packed(db, i4);
  }
  if (p.lse != nullptr && g32 == 0)
    p.lse[(int64_t)(q0 + row) * p.lse_stride_t + h] =
        l_tot > 0.f ? (m_ref + log2f(l_tot)) * 0.69314718055994531f : -INFINITY;
}

}  // namespace

template <int NW>
static void launch_shape(const PrefillParams& p, int32_t total_q, hipStream_t stream) {
  // upper bound on sum_b ceil(E_b / rows) over the batch
  const int64_t blocks = (int64_t)(total_q + 32 * NW - 1) / (32 * NW) + p.batch;
  hipLaunchKernelGGL(mla_prefill_kernel<NW>, dim3((unsigned)(blocks * p.heads)), dim3(NW * 64), 0, stream, p);
}

// CTAs of 128 query rows, two on a compute unit, when the requests average at most kPrefillSmallRows rows (the
// requests' lengths are on the device), where half-empty last blocks cost more than reading the keys once per 128
// rows, or when CTAs of 256 would leave compute units idle; CTAs of 256 rows otherwise. Measured (64 heads
// unless said), 256 rows / 128 rows: two requests of 600 rows on 600 keys 73.8 / 65.1 us; 16 of 384 on 1000
// 402 / 380; six of 1 to 294 rows 55.7 / 52.3; 4 of 700 on 1000 188 / 191; one of 1500 60.7 / 65.5; four of 2048
// on 4969 to 7961 keys 2278 / 2412; two of 1024 on 1000, 16 heads (128 CTAs of 256 rows) 56.9 / 46.1.
// Requests of whole 256-row blocks (an average that is a multiple of 256: a scheduler's chunks) have no half-empty
// ones: from kPrefillLongKeys keys on they take CTAs of 256 rows where these keep more than half of the compute units
// busy (fewer run faster as twice as many CTAs). The keys are on the device too; the page table's row stride stands for
// them (it chooses the launch, no more). 256 / 128 rows, 64 heads: eight of 512 rows on 1000 keys 240 / 238 us, on 2000
// 380 / 385; four of 512 on 8000 612 / 645, on 30,000 2172 / 2297; four of 256 on 8000 (256 CTAs of 256 rows) 337 / 356;
// one of 512 on 8000 (128) 232 / 187. With other requests 128 rows stay the better choice at any prefix: 700
// batches of up to 640 rows a request on 3000 to 16,000 keys took 8 % less in the geometric mean than in CTAs of 256,
// and the worst class, requests of up to 256 rows whose 256-row CTAs just fill the chip, up to 1.33 times as long.
constexpr int kPrefillSmallRows = 640;
constexpr int kPrefillLongKeys = 2048;

hipError_t launch_prefill(const PrefillParams& p, int32_t total_q, hipStream_t stream) {
  if (total_q <= 0 || p.heads <= 0 || p.batch <= 0) return hipSuccess;
  const int64_t rows = ((int64_t)total_q + p.batch - 1) / p.batch;  // of an average request
  const int64_t ctas = (rows + 255) / 256 * p.batch * p.heads, cus = current_device_cus();
  const bool whole = (int64_t)total_q % (256 * (int64_t)p.batch) == 0;
  const bool small = whole && p.pt_stride > (kPrefillLongKeys - 1) >> p.log2_ps ? 2 * ctas <= cus
                                                                                : rows <= kPrefillSmallRows || ctas <= cus;
  if (small) launch_shape<4>(p, total_q, stream);
  else launch_shape<8>(p, total_q, stream);
  return hipGetLastError();
}

}  // namespace mla
