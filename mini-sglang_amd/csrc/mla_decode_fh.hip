// Absorbed-MLA decode for up to 16 query heads (a tensor-parallel rank), any page size. Same plan,
// workspace and outputs as mla_decode_kernel.
//
// Bound: HBM. A 32-token tile (36 KB) is 68 MFMAs here and takes a compute unit about 1.3 us to stream, so
// the kernel is laid out to keep three tiles of loads in flight all the time and to make a tile's work short:
//  * the CTA's whole (request, token) range is one stream of 32-row tiles through a 4-stage LDS ring
//    filled by global->LDS DMA: per piece one tile of queries (a query row has the latent row's 576 dims)
//    and then the piece's KV tiles. Nothing drains between pieces.
//  * four waves share every tile. Scores: wave (th, kh) multiplies tokens 16 th .. +16 with dims 288 kh ..
//    +288 (9 K reads, 9 MFMAs); the partial scores meet in LDS (one LDS-only barrier), and every wave adds
//    the two halves and takes the softmax of the whole tile itself (8 exponentials per lane, the same bits
//    in every wave, so references and rescales need no agreement). Values: wave d accumulates dims
//    128 d .. +128 (16 transposing reads, 8 MFMAs).
//  * the exponent reference is the piece's first-tile max and moves (O and l rescaled) only when a later
//    score passes it by 2^64.
//  * tiles are column blocks (mla_device.h), with no bank conflicts and one source offset per lane for a
//    wave's 9 loads of a tile: 67.7 -> 62.6 us against rows of 1152 bytes (page size 1: 64.1 -> 61.0; one
//    request of 1,500 tokens: 7.1 -> 6.5 us), sizes as below.
// Measured (split step, 64 requests of 1k to 8k tokens, 363 MB, 8 heads): 58.7 us at page size 64 (6.2
// TB/s) and 60.4 us at page size 1, against 86.6 and 210.9 us of the general kernel, whose one wave runs a
// tile's MFMAs and 100 LDS reads as one serial chain and drains its ring at every piece. 17 heads and more
// go to the warp-specialized kernel, padded to 64: a second head block here (eight waves) measured 72.0 us
// against its 67.9 us at 32 heads (both before the tile layout changed).
#include "mla_common.h"
#include "mla_decode_stage.h"
#include "mla_device.h"

namespace mla {
namespace {

constexpr int kFWaves = 4;  // waves that load and compute; wave w issues a tile's loads of token octet w
constexpr int kFParts = kTileBlocks;  // loads of a KV tile per wave, one per column block
static_assert(kFWaves * kFParts == kTileDma, "every load of a tile is issued once");
constexpr int kFAhead = 3;  // stream tiles in flight beyond the one being worked on
constexpr int kFKPrefetch = 6;  // K operands in flight
constexpr int kFVPrefetch = 4;  // V operand pairs in flight
constexpr int kFMaxTiles = 2 * kMaxCtaBlocks;
constexpr float kFRescaleLog2 = 64.0f;
// The lowest maximum of a tile: where all scores of a first tile are -inf its numerators are then zero, and the first
// finite score moves the reference (against -inf the numerators, and with them the whole piece, would be NaN).
constexpr float kFLowest = -3.402823466e38f;
static_assert(kFAhead == kStages - 1 && kFAhead == 3, "a tile is issued into the stage of the tile just finished");

struct FCursor {
  int r, t, t0, t1, q;  // request rb + r, piece [t0, t1); q == 0: query tile, q == 1: KV tile at token t
};

// kSmall: pages of fewer than 32 tokens; a tile's rows lie on
// several pages, and the loads take one 32-bit row offset (from the pool base) per token. One more wave,
// which issues no DMA (its page-table loads are the only vector-memory operations it waits for), loads the
// page-table entries of stream tile n at step n - 5 and writes the tile's 32 row offsets to slot n % 4 of a
// ring in LDS at step n - 4; the other waves read them at step n - 3, when they issue the tile. (With the
// page-table entries loaded by DMA and the offsets made by wave 0 between its own loads and scores, every
// step waits for wave 0: 74 us against 64 us at 8 heads, page size 1, 64 requests of 1k to 8k tokens.) The
// launcher takes this path only when every row offset of the pool fits in 32 bits.
template <bool kSmall>
__global__ __launch_bounds__((kFWaves + (kSmall ? 1 : 0)) * 64, 1) void mla_decode_fh_kernel(const DecodeParams p) {
  constexpr int kThreads = (kFWaves + (kSmall ? 1 : 0)) * 64;
  __shared__ __attribute__((aligned(1024))) char smem[kStages * kTileBytes];
  // partial scores of the tile: [dim half][token half][lane]
  __shared__ __attribute__((aligned(16))) f32x4 s_s[2][2][64];
  __shared__ int s_t0[kMaxCtaRequests], s_t1[kMaxCtaRequests], s_tbase[kMaxCtaRequests + 1];
  __shared__ int s_np[kMaxCtaRequests], s_slot0[kMaxCtaRequests];
  __shared__ int s_pid[kSmall ? 4 * kTile : kFMaxTiles];  // page id per KV tile; kSmall: the row-offset ring

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = p.heads;
  const int ps_mask = (1 << p.log2_ps) - 1;
  const int row_bytes = (int)(p.kv_row_stride * 2);
  const uint32_t qrow_bytes = (uint32_t)(p.q_stride_h * 2);
  const char* kv = reinterpret_cast<const char*>(p.kv);
  const uint32_t lds_ring = (uint32_t)(uintptr_t)(MLA_LDS char*)smem;

  // A plan range of this CTA; false for a padding range (all later ranges are padding too).
  auto range = [&](const int w) -> bool {
    int rb, kb, re, ke;
    sload_i32x4(p.plan + 4 * w, rb, kb, re, ke);
    if (rb >= p.batch) return false;
    const int rlast = min(ke == 0 ? re - 1 : re, p.batch - 1);
    const int nreq = min(rlast - rb + 1, kMaxCtaRequests);
    if (nreq <= 0) return true;  // uniform: an empty range

    auto fresh_lane = [&]() {  // the lane index from a volatile asm: offsets made from it are computed in place
      int ln;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
      return ln;
    };
    const int lane = fresh_lane();
    const int g = lane >> 4, c = lane & 15;
    // the 16 query rows are octets 0 and 1 of a tile: waves 0 and 1 load them
    const int nq = wave < 2 ? kFParts : 0;
    auto issue_query = [&](int b, uint32_t stage) {  // rows past the last head load the last head
      if (wave >= 2) return;
      const char* src = reinterpret_cast<const char*>(p.q) + (int64_t)b * p.q_stride_b * 2;
      const int ln = fresh_lane(), t = octet_token(wave, ln);
      dma16_octet<false>(src, min(t, H - 1) * qrow_bytes + octet_chunk(ln, t), stage + wave * 1024);
    };
    // The first piece is request rb's unless its part of the range is empty (only for an empty request): its
    // queries land in ring stage 0 while the range is staged (the staging's barriers wait on LDS only).
    issue_query(rb, lds_ring);

    stage_range<kThreads, !kSmall, kFMaxTiles>(p, rb, kb, re, ke, nreq, lane, wave,
                                               RangeTables{s_t0, s_t1, s_tbase, s_np, s_slot0, s_pid});

    // ---- stream cursors over (request, tile); all values wave-uniform
    auto seek = [&](FCursor& cur, int r) -> bool {  // first non-empty piece at or after request rb + r
      for (; r < nreq; ++r) {
        const int t0 = __builtin_amdgcn_readfirstlane(s_t0[r]);
        const int t1 = __builtin_amdgcn_readfirstlane(s_t1[r]);
        if (t1 > t0) {
          cur = FCursor{r, t0, t0, t1, 0};
          return true;
        }
      }
      return false;
    };
    auto advance = [&](FCursor& cur) -> bool {
      if (cur.q == 0) {
        cur.q = 1;
        return true;
      }
      cur.t += kTile;
      return cur.t < cur.t1 ? true : seek(cur, cur.r + 1);
    };
    FCursor cs;  // the tile of this step
    if (!seek(cs, 0)) {  // uniform: every piece of the range is empty (no barrier follows)
      wait_vmcnt<0>();   // the early query loads land before the CTA can end
      return true;
    }

    if (kSmall && wave == kFWaves) {
      // ---- row-offset producer: lane l (< 32) holds token t + l of a tile, clamped to the piece
      auto load = [&](const FCursor& cur, bool valid, int& tok, int& page) -> bool {
        if (!valid || cur.q == 0) return false;
        tok = min(cur.t + (lane & 31), cur.t1 - 1);
        page = p.page_table[(int64_t)(rb + cur.r) * p.pt_stride + (tok >> p.log2_ps)];
        return true;
      };
      auto store = [&](int n, int tok, int page) {
        const uint32_t pg = (uint32_t)min(max(page, 0), p.num_pages - 1);
        if (lane < kTile)
          s_pid[(n & 3) * kTile + lane] = (int)(((pg << p.log2_ps) | (uint32_t)(tok & ps_mask)) * (uint32_t)row_bytes);
      };
      FCursor la = cs;
      bool la_valid = true;
      int tok[kFAhead + 1], page[kFAhead + 1];
      bool kvt[kFAhead + 1];
#pragma unroll
      for (int n = 0; n <= kFAhead; ++n) {  // the first tiles' page-table loads back to back
        tok[n] = page[n] = 0;
        kvt[n] = load(la, la_valid, tok[n], page[n]);
        if (la_valid) la_valid = advance(la);
      }
#pragma unroll
      for (int n = 0; n <= kFAhead; ++n)
        if (kvt[n]) store(n, tok[n], page[n]);
      int la_tok = 0, la_page = 0;
      bool la_kv = load(la, la_valid, la_tok, la_page);
      barrier_lds();  // the first tiles' offsets are written
      for (int j = 0;; ++j) {
        barrier_lds();
        if (la_kv) store(j + kFAhead + 1, la_tok, la_page);
        if (la_valid) la_valid = advance(la);
        la_kv = load(la, la_valid, la_tok, la_page);
        if (cs.q != 0) barrier_lds();  // the score exchange
        if (!advance(cs)) break;
      }
      return true;
    }

    // ---- per-lane LDS read offsets (bytes within a tile)
    const int th = wave & 1, kh = wave >> 1;
    const int xk = tswz(c);  // token 16 tb + c has the swizzle of token c
    const int k_lo = c * 128 + ((tperm(g) ^ xk) << 4), k_hi = c * 128 + (((4 + tperm(g)) ^ xk) << 4);
    // operand i of this wave's dim half is k-step 9 kh + i (half a column block each)
    const int k_a = kh ? k_hi + 4 * kTileBlockBytes : k_lo, k_b = kh ? k_lo + 5 * kTileBlockBytes : k_hi;
    int v_off[4];  // value dims 128 wave .. +128 are column blocks 2 wave, 2 wave + 1
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int t = 4 * g + (c >> 2);
      v_off[q4] = 2 * wave * kTileBlockBytes + t * 128 + (((2 * q4 + ((c & 3) >> 1)) ^ tswz(t)) << 4) + ((c & 1) << 3);
    }
    const int dma_t = octet_token(wave, lane);  // this lane's token of a tile, and its source offset there
    const uint32_t dma_ch = octet_chunk(lane, dma_t);
    int iss_kv = 0;  // KV tiles issued (index into s_pid)
    // vector-memory operations this wave issued, and the count right after its loads of the stream tiles of this
    // step and the next three: a tile has landed once at most (ops - mark) operations are outstanding
    int ops = nq, mark0 = nq, mark1 = 0, mark2 = 0, mark3 = 0;
    int pid_v = kSmall ? 0 : s_pid[0];  // page id of KV tile iss_kv, read a step ahead of its use
    auto issue = [&](const FCursor& cur, int n) {  // this wave's loads of stream tile n (at cur)
      const uint32_t stage = lds_ring + (n % kStages) * kTileBytes;
      if (cur.q == 0) {
        issue_query(rb + cur.r, stage);
        ops += nq;
      } else {
        if constexpr (kSmall) {  // the token's row from the offset ring (clamped rows included)
          dma16_octet<true>(kv, (uint32_t)s_pid[(n & 3) * kTile + dma_t] + dma_ch, stage + wave * 1024);
        } else {
          const int pid = __builtin_amdgcn_readfirstlane(pid_v);
          pid_v = s_pid[min(++iss_kv, kFMaxTiles - 1)];
          const char* src = kv + ((int64_t)pid * (ps_mask + 1) + (cur.t & ps_mask)) * row_bytes;
          const int tlim = cur.t1 - 1 - cur.t;  // loads clamp to the piece's last token
          dma16_octet<true>(src, min(dma_t, tlim) * row_bytes + dma_ch, stage + wave * 1024);
        }
        ops += kFParts;
      }
    };

    if constexpr (kSmall) barrier_lds();  // the first tiles' row offsets are written
    FCursor iss = cs;
    int n_issued = 0;
    bool iss_valid = true;
    if (cs.r == 0) {  // the early query loads are stream tile 0
      n_issued = 1;
      iss_valid = advance(iss);
    } else {  // request rb is empty: its query loads land before the stream reuses their stage
      wait_vmcnt<0>();
    }
    while (n_issued < kFAhead && iss_valid) {
      issue(iss, n_issued);
      (n_issued == 0 ? mark0 : n_issued == 1 ? mark1 : mark2) = ops;
      ++n_issued;
      iss_valid = advance(iss);
    }

    bf16x8 qf[9];
    f32x4 O[8];
    float m_ref = 0.f, l_run = 0.f;
#pragma unroll
    for (int db = 0; db < 8; ++db) O[db] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int j = 0;; ++j) {
      // tile j lands: wait for this wave's loads of it, then the whole CTA's; stage (j - 1) % 4 is free
      wait_vmcnt_dyn<(kFAhead - 1) * kFParts>(ops - mark0);
      barrier_lds();
      if (iss_valid) {
        issue(iss, n_issued++);
        mark3 = ops;
        iss_valid = advance(iss);
      }
      const MLA_LDS char* T = (const MLA_LDS char*)smem + (j % kStages) * kTileBytes;
      if (cs.q == 0) {  // a piece starts: this wave's dim half of the query rows
#pragma unroll
        for (int i = 0; i < 9; ++i)
          qf[i] = *reinterpret_cast<const MLA_LDS bf16x8*>(T + ((i & 1) ? k_b : k_a) + kTileBlockBytes * (i >> 1));
      } else {
        // ---- partial S^T[16 tokens (half th) x 16 heads] over dims 288 kh .. +288
        const MLA_LDS char* K = T + th * (16 * 128);
        auto kread = [&](int i) {
          return *reinterpret_cast<const MLA_LDS bf16x8*>(K + ((i & 1) ? k_b : k_a) + kTileBlockBytes * (i >> 1));
        };
        f32x4 sacc[2];
        sacc[0] = sacc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        bf16x8 kbuf[kFKPrefetch];
#pragma unroll
        for (int i = 0; i < kFKPrefetch; ++i) kbuf[i] = kread(i);
#pragma unroll
        for (int i = 0; i < 9; ++i) {
          const bf16x8 a = kbuf[i % kFKPrefetch];
          if (i + kFKPrefetch < 9) kbuf[i % kFKPrefetch] = kread(i + kFKPrefetch);
          sacc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[i], sacc[i & 1], 0, 0, 0);
        }
        s_s[kh][th][lane] = sacc[0] + sacc[1];
        barrier_lds();
        // ---- scores of the tile: lane (g, c) holds head c, tokens 4g + i and 16 + 4g + i
        f32x4 sv[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) sv[t] = s_s[0][t][lane] + s_s[1][t][lane];
        // the V^T operands do not depend on the softmax: read the first ones now
        auto vread = [&](int db, int half) {
          const int off = v_off[db & 3] + kTileBlockBytes * (db >> 2) + half * 16 * 128;
          return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((MLA_LDS bf16x4*)(T + off));
        };
        bf16x4 vlo[kFVPrefetch], vhi[kFVPrefetch];
#pragma unroll
        for (int db = 0; db < kFVPrefetch; ++db) {
          vlo[db] = vread(db, 0);
          vhi[db] = vread(db, 1);
        }
        const int valid = cs.t1 - cs.t;
        float x[8], mt = kFLowest;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          x[i] = sv[i >> 2][i & 3] * p.scale_log2;
          if (valid < kTile && 16 * (i >> 2) + 4 * g + (i & 3) >= valid) x[i] = -INFINITY;
          mt = fmaxf(mt, x[i]);
        }
        if (cs.t == cs.t0) {
          m_ref = wave_max_g(mt);
        } else if (__ballot(mt > m_ref + kFRescaleLog2) != 0) {  // rare, and the same in every wave
          const float m_new = fmaxf(wave_max_g(mt), m_ref);
          const float f = __builtin_amdgcn_exp2f(m_ref - m_new);
          m_ref = m_new;
          l_run *= f;
#pragma unroll
          for (int db = 0; db < 8; ++db) O[db] *= f;
        }
        float pr[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          pr[i] = __builtin_amdgcn_exp2f(x[i] - m_ref);
          l_run += pr[i];
        }
        u32x4 pw;
#pragma unroll
        for (int i = 0; i < 4; ++i) pw[i] = pack_bf16x2(pr[2 * i], pr[2 * i + 1]);
        const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
        // ---- O^T[16 dims x 16 heads] += V^T . P^T over this wave's 8 dim blocks
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          const bf16x8 a =
              __builtin_shufflevector(vlo[db % kFVPrefetch], vhi[db % kFVPrefetch], 0, 1, 2, 3, 4, 5, 6, 7);
          if (db + kFVPrefetch < 8) {
            vlo[db % kFVPrefetch] = vread(db + kFVPrefetch, 0);
            vhi[db % kFVPrefetch] = vread(db + kFVPrefetch, 1);
          }
          O[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb, O[db], 0, 0, 0);
        }
        if (cs.t + kTile >= cs.t1) {
          // ---- the piece ends: normalise and write this wave's dims (lanes c == 0 always hold a head, so
          // each store below is one counted vector-memory operation)
          const int b = rb + cs.r;
          const int npieces = __builtin_amdgcn_readfirstlane(s_np[cs.r]);
          const int slot = __builtin_amdgcn_readfirstlane(s_slot0[cs.r]) + w;
          const bool to_ws = npieces != 1;
          const float l = wave_sum_g(l_run);
          // no score above -inf: nothing to the merge, and no result (NaN) for a whole request
          const float inv = to_ws && !(l > 0.f) ? 0.f : 1.f / l;
          const float lse_nat = l > 0.f ? (m_ref + log2f(l)) * 0.69314718055994531f : -INFINITY;
          if (to_ws) {
            if (slot >= 0 && slot < p.ws_slots) {
              // bf16 partial for the merge, one 16-byte chunk per dim-block pair: chunk 16 wave + 4 pp + g of
              // the row (the chunk order of mla_amd.h)
              if (c < H) {
                __bf16* orow = p.ws_o + ((int64_t)slot * H + c) * kVDim + 128 * wave + 8 * g;
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                  u32x4 v;
                  v[0] = pack_bf16x2(O[2 * pp][0] * inv, O[2 * pp][1] * inv);
                  v[1] = pack_bf16x2(O[2 * pp][2] * inv, O[2 * pp][3] * inv);
                  v[2] = pack_bf16x2(O[2 * pp + 1][0] * inv, O[2 * pp + 1][1] * inv);
                  v[3] = pack_bf16x2(O[2 * pp + 1][2] * inv, O[2 * pp + 1][3] * inv);
                  *reinterpret_cast<u32x4*>(orow + 32 * pp) = v;
                }
              }
              ops += 4;
              if (wave == 0) {
                if (g == 0 && c < H) p.ws_lse[(int64_t)slot * H + c] = lse_nat;
                ops += 1;
              }
            }
          } else {
            if (c < H) {
              __bf16* orow = p.out + (int64_t)b * p.out_stride_b + (int64_t)c * p.out_stride_h + 128 * wave + 4 * g;
#pragma unroll
              for (int db = 0; db < 8; ++db) {
                u32x2 v;
                v[0] = pack_bf16x2(O[db][0] * inv, O[db][1] * inv);
                v[1] = pack_bf16x2(O[db][2] * inv, O[db][3] * inv);
                *reinterpret_cast<u32x2*>(orow + 16 * db) = v;
              }
            }
            ops += 8;
            if (wave == 0 && p.lse != nullptr) {
              if (g == 0 && c < H) p.lse[(int64_t)b * p.lse_stride_b + c] = lse_nat;
              ops += 1;
            }
          }
          l_run = 0.f;
#pragma unroll
          for (int db = 0; db < 8; ++db) O[db] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
      mark0 = mark1;
      mark1 = mark2;
      mark2 = mark3;
      if (!advance(cs)) break;
    }
    return true;
  };

  for (int w = blockIdx.x; w < p.num_ctas; w += gridDim.x) {
    if (w != (int)blockIdx.x) {  // the previous range's waves are done with the LDS tables and ring
      wait_vmcnt<0>();
      __syncthreads();
    }
    if (!range(w)) break;
  }
}

}  // namespace

bool decode_fh_takes(const DecodeParams& p) { return p.heads >= 1 && p.heads <= 16 && row_offsets_fit(p, 16); }

hipError_t launch_decode_fh(const DecodeParams& p, hipStream_t stream) {
  const int cus = current_device_cus();
  const int grid = p.num_ctas < cus ? p.num_ctas : cus;
  if (p.log2_ps >= 5)
    hipLaunchKernelGGL(mla_decode_fh_kernel<false>, dim3(grid), dim3(kFWaves * 64), 0, stream, p);
  else
    hipLaunchKernelGGL(mla_decode_fh_kernel<true>, dim3(grid), dim3((kFWaves + 1) * 64), 0, stream, p);
  return hipGetLastError();
}

}  // namespace mla
