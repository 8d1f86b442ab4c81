// Warp-specialized absorbed-MLA decode for 17 heads and more (the Kimi-K2 / DeepSeek-V3 decode shapes), in
// groups of 64, any page size. Same plan, workspace and outputs as mla_decode_kernel.
//
//  * The CTA's whole (request, token) range is one stream of 32-row tiles: per piece, two tiles of
//    queries (heads 0..31, 32..63; a query row has the latent row's 576 dims, so it is staged like
//    a KV row) and then the piece's 32-token KV tiles, through a 4-stage LDS ring filled by
//    global->LDS DMA (non-temporal for the KV rows, which are read once). The page id of every KV
//    tile and the bounds of every request of the range are staged in LDS once, at CTA start.
//  * 8 waves, two per SIMD, in two roles that run one tile apart:
//      score waves (hg, th) = (s & 1, s >> 1), s = 0..3 (heads 32hg .. 32hg+31, tokens 16th .. +16
//      of a tile):
//        S^T[16 tokens x 32 heads] = K . Q^T                  36 MFMAs, 18 K reads
//        softmax numerators against the piece's reference (its first tile's max over both halves,
//        agreed by the pair (hg, 0) / (hg, 1) at the piece's first KV tile), written as bf16 to a
//        double-buffered P block in LDS
//      output waves o = 0..3 (value dims 128o .. 128o+127, all 64 heads), one tile behind:
//        O^T[128 dims x 64 heads] += V^T . P^T                 32 MFMAs, 16 transposing V reads
//    Every K row is read from LDS by two waves, every V row by one. Tiles are column blocks (mla_device.h):
//    rows of 1152 bytes left the K reads 2-way bank conflicted, 12 of the 29 % of cycles the LDS was busy, and
//    needed 9 source offsets per lane. Split step before -> after: 128 heads, 32 requests of 1k to 8k tokens
//    79.6 -> 77.1 us (page size 1: 80.6 -> 76.3); 64 heads, 64 requests 74.3 -> 73.4 us (page size 1:
//    78.0 -> 75.2); 8 requests of 1k to 8k tokens 18.6 -> 18.1; one of 1,500 tokens 11.35 -> 10.8 us.
//    A SIMD holds one wave of each
//    role, so one role's LDS and barrier waits are covered by the other's MFMAs. One barrier per step
//    (two at a piece's first KV tile): step j scores tile j and accumulates tile j - 1; the output
//    waves normalise and store a piece (bf16 output, or the bf16 partial of a split request) and
//    write its LSE.
//  * No accumulator rescaling: exponents are taken against the piece's first-tile max; a piece whose
//    later scores exceed it by 2^64 is rerun with its exact max (the vote is taken at the step after
//    the piece's last tile, before any wave touches the next tile).
//  * Barriers wait on LDS only; each wave counts its own DMA loads and output stores and waits for
//    a tile's loads by that count (wait_vmcnt_dyn).
// Bound: the output waves' chain (about 2,800 cycles a tile: 1,000 to issue their nine loads, 1,330 of operand
// reads and MFMAs), just above the tile's HBM time (2,700 cycles).
#include <type_traits>

#include "mla_common.h"
#include "mla_decode_stage.h"
#include "mla_device.h"

namespace mla {
namespace {

constexpr int kWWaves = 8;
constexpr int kWAhead = 2;         // stream tiles in flight beyond the one being scored
static_assert(kWAhead == 2, "two marks beyond the step's own");
// Output wave r issues a tile's 9 loads of token octet r (one per column block) at the step's start.
// (Any of them on the score waves, at the step's start or after their work, measured 4 to 10 us more a launch: a
// blocked issue stalls the score work, which is nearly critical too.)
constexpr int kWParts = kTileBlocks;
static_assert(4 * kWParts == kTileDma, "every load of a tile is issued once");
constexpr int kWKPrefetch = 6;     // K operands in flight
constexpr int kWVPrefetch = 4;     // V operand pairs in flight
constexpr int kWMaxTiles = 2 * kMaxCtaBlocks;
constexpr float kWOverflowLog2 = 64.0f;

struct WCursor {
  int r, t, t0, t1, q;  // request rb + r, piece [t0, t1); q < 2: query tile q, q == 2: KV tile at token t
};

// kSmall: pages of fewer than 32 tokens. A tile's rows then lie on several pages, so instead of one
// page id per tile the DMA takes one 32-bit row offset (from the pool base) per token: score wave 0
// loads the page-table entries of stream tile n at step n - 4, writes the tile's 32 row offsets to
// slot n % 4 of a ring in LDS at step n - 3, and the output waves read them at step n - 2, after that
// step's barrier, when they issue the tile. The launcher takes this path only when every row offset
// of the pool fits in 32 bits.
//
// kLoop: the plan has more than two ranges per compute unit (one laid out for a larger grid, as a captured decode
// step's is); the launch has one CTA per compute unit (and group), which runs its range and every n-th after it in
// turn and stops at the first padding range. Without it each CTA runs one range and the body has no loop around it
// (the loop makes the compiler keep values across both roles' step loops and spill). A padding range then costs a
// CTA that takes a compute unit's LDS to find it has nothing to do. Split step, loop-free / loop: 128 heads, 32
// requests of 1k to 8k tokens in 256 ranges of a plan for 512: 65.7 / 66.5 us, for 2048: 70.7-74.6 / 66.5; 32
// heads, 64 requests, for 2048: 66.0 / 64.0; one request of 1,500 tokens, 64 heads, for 512: 9.4 / 10.0; 40 requests
// of 960 to 1,120 tokens in 341 ranges, 24 heads 23.9 / 24.6, 64 heads 26.7 / 27.0, 128 heads 40.1 / 41.3.
// kMode kPadded: 17 to 63 heads; query rows past the last head load the last head again and their outputs are
// not written (the padding costs MFMAs, which the KV stream hides: 32 heads, 64 requests of 1k to 8k tokens,
// 67.9 us against 78.1 us on the general kernel; 48 heads 70.7 against 82.5 us).
// kMode kGroups: more than 64 heads, in groups of 64 (the last one padded): a CTA runs one group of one range, and
// the groups of a range are CTAs 8 apart, which the dispatcher puts on the same XCD at about the same time: the
// range's KV tiles come from HBM once and from that XCD's L2 for the other groups (so they are loaded without the
// non-temporal hint). One launch per group, each streaming the KV from HBM, took 80.8 us for 128 heads, 32 requests
// of 1k to 8k tokens, where this took 77.2 us (and 66 us with the tile layout and waits of today; HBM no longer
// bounds it).
enum WMode { kExact, kPadded, kGroups };

template <bool kSmall, bool kLoop, WMode kMode>
__global__ __launch_bounds__(kWWaves * 64, 1) void mla_decode_ws_kernel(const DecodeParams p0) {
  DecodeParams p = p0;
  int w_first = blockIdx.x;
  if constexpr (kMode == kGroups) {
    const int groups = (p0.heads + 63) >> 6;
    const int i = (int)blockIdx.x >> 3, grp = i % groups;
    w_first = (i / groups) * 8 + ((int)blockIdx.x & 7);
    if (w_first >= p0.num_ctas) return;
    const int h0 = 64 * grp;
    p.heads = min(64, p0.heads - h0);
    p.q = p0.q + (int64_t)h0 * p0.q_stride_h;
    p.ws_o = p0.ws_o + (int64_t)p0.ws_slots * h0 * kVDim;  // the group's own [ws_slots, group heads] block
    p.ws_lse = p0.ws_lse + (int64_t)p0.ws_slots * h0;
    p.out = p0.out + (int64_t)h0 * p0.out_stride_h;
    if (p0.lse != nullptr) p.lse = p0.lse + h0;
  }
  constexpr bool kNt = kMode != kGroups;  // KV loads are non-temporal where the rows are read once
  // first query row of query tile qt, and row t of it from there (rows past the last head: the last head)
  auto q_tile_row = [&](int qt) __attribute__((always_inline)) {
    return kMode == kExact ? 32 * qt : min(32 * qt, p.heads - 1);
  };
  auto q_row = [&](int t, int qt) __attribute__((always_inline)) {
    return kMode == kExact ? t : min(t, p.heads - 1 - q_tile_row(qt));
  };
  // head blocks of 16 with a head in them: the stores of an output wave are counted for these
  const int hblocks = kMode == kExact ? 4 : (p.heads + 15) >> 4;
  __shared__ __attribute__((aligned(1024))) char smem[kStages * kTileBytes];
  // softmax numerators of the last two scored tiles: [tile parity][head block][lane], 16 B per lane
  __shared__ __attribute__((aligned(16))) u32x4 s_p[2][4][64];
  __shared__ float s_l[2][64];   // per token half and head: row sums of the piece that just ended
  __shared__ float s_mref[64];   // per head: that piece's exponent reference
  __shared__ float s_mx[2][64];  // per token half and head: a max (piece start: first tile; end: piece)
  __shared__ int s_flag[4];      // per score wave: that piece overflowed its exponent reference
  __shared__ int s_t0[kMaxCtaRequests], s_t1[kMaxCtaRequests], s_tbase[kMaxCtaRequests + 1];
  __shared__ int s_np[kMaxCtaRequests], s_slot0[kMaxCtaRequests];
  __shared__ int s_pid[kWMaxTiles];  // page id per KV tile; kSmall: the row-offset ring [4][32]

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool scorer = wave < 4;
  const int role = wave & 3;  // score wave: head block; output wave: value-dim quarter

  // Plan range w; false for a padding range (all later ranges are padding too).
  auto range = [&](const int w) -> bool {
    // the lane index from a volatile asm: what derives from it is computed per range, not hoisted
    // out of a loop over ranges
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    const int g = lane >> 4;
    const int c = lane & 15;
    int rb, kb, re, ke;
    sload_i32x4(p.plan + 4 * w, rb, kb, re, ke);
    if (rb >= p.batch) return false;
    const int ps_mask = (1 << p.log2_ps) - 1;
    const int row_bytes = (int)(p.kv_row_stride * 2);
    const char* kv = reinterpret_cast<const char*>(p.kv);
    const uint32_t lds_ring = (uint32_t)(uintptr_t)(MLA_LDS char*)smem;

    // ---- per-lane LDS read offsets (bytes within a tile)
    const int xk = tswz(c);  // token 16 tb + c has the swizzle of token c
    const int k_off_even = c * 128 + ((tperm(g) ^ xk) << 4);
    const int k_off_odd = c * 128 + (((4 + tperm(g)) ^ xk) << 4);
    int v_off[4];  // output wave `role`: value dims 128 role .. +128 are column blocks 2 role, 2 role + 1
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int t = 4 * g + (c >> 2);
      v_off[q4] = 2 * role * kTileBlockBytes + t * 128 + (((2 * q4 + ((c & 3) >> 1)) ^ tswz(t)) << 4) + ((c & 1) << 3);
    }

    // ---- stage the range: request bounds, then one page id per 32-token tile
    int rlast = (ke == 0 ? re - 1 : re);
    rlast = min(rlast, p.batch - 1);
    const int nreq = min(rlast - rb + 1, kMaxCtaRequests);
    if (nreq <= 0) return true;  // uniform: an empty range
    // The first piece is request rb's in all but rare cases (rb's part of the range is empty only for
    // an empty request): the output waves load its two query tiles into ring stages 0 and 1 now, so
    // that they land while the range is staged (the staging's barriers wait on LDS only). If the
    // first piece turns out to be another request's, the stream issues its query tiles into the same
    // stages after these loads, and loads of one wave complete in order.
    const uint32_t qrow_bytes = (uint32_t)(p.q_stride_h * 2);
    auto issue_query = [&](int b, int qt, uint32_t stage) {  // this output wave's octet of query tile qt of request b
      const char* qsrc = reinterpret_cast<const char*>(p.q) +
                         ((int64_t)b * p.q_stride_b + (int64_t)q_tile_row(qt) * p.q_stride_h) * 2;
      int ln;  // lane index from a volatile asm, so these offsets are computed here
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
      const int t = octet_token(role, ln);
      dma16_octet<false>(qsrc, q_row(t, qt) * qrow_bytes + octet_chunk(ln, t), stage + role * 1024);
    };
    if (!scorer) {
      issue_query(rb, 0, lds_ring);
      issue_query(rb, 1, lds_ring + kTileBytes);
    }
    stage_range<kWWaves * 64, !kSmall, kWMaxTiles>(p, rb, kb, re, ke, nreq, lane, wave,
                                                   RangeTables{s_t0, s_t1, s_tbase, s_np, s_slot0, s_pid});

    // ---- stream cursors over (request, tile); all values wave-uniform
    auto seek = [&](WCursor& cur, int r) -> bool {  // first non-empty piece at or after request rb + r
      for (; r < nreq; ++r) {
        const int t0 = __builtin_amdgcn_readfirstlane(s_t0[r]);
        const int t1 = __builtin_amdgcn_readfirstlane(s_t1[r]);
        if (t1 > t0) {
          cur = WCursor{r, t0, t0, t1, 0};
          return true;
        }
      }
      return false;
    };
    auto advance = [&](WCursor& cur) -> bool {
      if (cur.q < 2) {
        ++cur.q;
        return true;
      }
      cur.t += kTile;
      return cur.t < cur.t1 ? true : seek(cur, cur.r + 1);
    };
    // Each role runs its own copy of the step loop (the same stream, the same barriers), so that only
    // that role's state is live in its registers.
    auto run = [&](auto role_tag) {
    constexpr bool kScore = decltype(role_tag)::value;
    constexpr int nparts = kScore ? 0 : kWParts;
    const int dma_t = octet_token(role, lane);  // this lane's token of a tile, and its source offset there
    const uint32_t dma_ch = octet_chunk(lane, dma_t);
    int iss_kv = 0;  // KV tiles issued (index into s_pid)
    // vector-memory operations this wave issued, and the count right after its loads of the stream tiles of this
    // step and the next two: a tile has landed once at most (ops - mark) operations are outstanding
    int ops = 2 * nparts, mark0 = nparts, mark1 = ops, mark2 = 0;
    int pid_v = 0;  // !kSmall: page id of KV tile iss_kv, read a step ahead of its use
    auto fetch_pid = [&]() {
      if constexpr (!kSmall) pid_v = s_pid[min(iss_kv, kWMaxTiles - 1)];
    };
    auto issue = [&](const WCursor& cur, int n) {  // this wave's DMA parts of stream tile n (at cur)
      const uint32_t stage = lds_ring + (n % kStages) * kTileBytes;
      if (cur.q < 2) {
        issue_query(rb + cur.r, cur.q, stage);
      } else if constexpr (kSmall) {  // the token's row from the offset ring (clamped rows included)
        dma16_octet<kNt>(kv, (uint32_t)s_pid[(n & 3) * 32 + dma_t] + dma_ch, stage + role * 1024);
      } else {
        const int pid = __builtin_amdgcn_readfirstlane(pid_v);
        ++iss_kv;
        const char* tsrc = kv + ((int64_t)pid * (ps_mask + 1) + (cur.t & ps_mask)) * row_bytes;
        const int tlim = cur.t1 - 1 - cur.t;  // loads clamp to the piece's last token
        dma16_octet<kNt>(tsrc, min(dma_t, tlim) * row_bytes + dma_ch, stage + role * 1024);
      }
      ops += nparts;
      fetch_pid();
    };

    WCursor cs;  // the tile scored at this step
    if (!seek(cs, 0)) {  // uniform: every piece of the range is empty (no barrier follows)
      wait_vmcnt<0>();   // the early query loads land before the CTA can end
      return;
    }
    WCursor iss = cs;
    int n_issued = 0;
    bool iss_valid = true;
    if constexpr (nparts > 0) {
      if (cs.r == 0) {  // the early query loads are stream tiles 0 and 1 (a piece starts at q = 0)
        for (int s = 0; s < 2 && iss_valid; ++s) {
          ++n_issued;
          iss_valid = advance(iss);
        }
      } else {  // request rb is empty: its query loads land before the stream reuses their stages
        wait_vmcnt<0>();
        ops = mark0 = mark1 = 0;
      }
    }
    auto prologue = [&](const int from) {
      if constexpr (nparts == 0) return;  // a role without DMA parts keeps no issue cursor
      fetch_pid();
      for (int s = from; s < kWAhead && iss_valid; ++s) {
        issue(iss, n_issued++);
        (s == 0 ? mark0 : mark1) = ops;
        iss_valid = advance(iss);
      }
    };
    // kSmall: score wave 0's row-offset producer. la is the stream tile (index la_n) whose
    // page-table entries are in flight; lane l (< 32) holds its token t + l, clamped to the piece.
    WCursor la = cs;
    int la_n = 0, la_tok = 0, la_page = 0;
    bool la_valid = false, la_kv = false;
    auto la_load = [&]() {
      la_kv = la_valid && la.q == 2;
      if (la_kv) {
        la_tok = min(la.t + (lane & 31), la.t1 - 1);
        la_page = p.page_table[(int64_t)(rb + la.r) * p.pt_stride + (la_tok >> p.log2_ps)];
      }
    };
    auto la_store = [&]() {  // waits for la_page (this wave issues no other vector-memory loads)
      if (la_kv && lane < 32) {
        const uint32_t page = (uint32_t)min(max(la_page, 0), p.num_pages - 1);
        s_pid[(la_n & 3) * 32 + lane] = (int)(((page << p.log2_ps) | (uint32_t)(la_tok & ps_mask)) * (uint32_t)row_bytes);
      }
    };
    auto la_step = [&]() {  // store the in-flight tile's offsets, then load the next tile's entries
      la_store();
      if (la_valid) la_valid = advance(la);
      ++la_n;
      la_load();
    };
    auto seed = [&](const WCursor& from, int n0) {  // offsets of tiles n0 .. n0 + 2; n0 + 3 in flight
      la = from;
      la_valid = true;
      int tok[3], pg[3];
      bool kv3[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {  // the three tiles' page-table loads back to back
        kv3[i] = la_valid && la.q == 2;
        tok[i] = min(la.t + (lane & 31), la.t1 - 1);
        pg[i] = kv3[i] ? p.page_table[(int64_t)(rb + la.r) * p.pt_stride + (tok[i] >> p.log2_ps)] : 0;
        if (la_valid) la_valid = advance(la);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (kv3[i] && lane < 32) {
          const uint32_t page = (uint32_t)min(max(pg[i], 0), p.num_pages - 1);
          s_pid[((n0 + i) & 3) * 32 + lane] =
              (int)(((page << p.log2_ps) | (uint32_t)(tok[i] & ps_mask)) * (uint32_t)row_bytes);
        }
      }
      la_n = n0 + 3;
      la_load();
    };
    if constexpr (kSmall) {  // every wave: the first tiles' offsets before the first DMA
      if constexpr (kScore) if (role == 0) seed(cs, 0);
      barrier_lds();
    }
    prologue(n_issued);

    // score-wave state: queries of head blocks 2 hg, 2 hg + 1; per head block (lane: head c of it)
    // the piece's reference, max and this half's row sum
    const int hg = role & 1, th = role >> 1;
    bf16x8 qf[2][18];
    float m_ref[2] = {0.f, 0.f}, m_max[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
    bool overflow = false, first_kv = true;
    // output-wave state
    f32x4 O[4][8];
#pragma unroll
    for (int hq = 0; hq < 4; ++hq)
#pragma unroll
      for (int db = 0; db < 8; ++db) O[hq][db] = f32x4{0.f, 0.f, 0.f, 0.f};

    int attempt = 0;
    bool s_valid = true;                          // cs is a tile
    bool prev_kv = false, prev_end = false;       // the tile scored at the previous step
    int prev_r = 0;
    WCursor piece_cur = cs;                       // first KV tile of the current piece
    int piece_j = 0, piece_kv = 0, comp_kv = 0;   // its stream / KV indices; KV tiles scored

    for (int j = 0;;) {
      // ---- step j: tile j (cs) lands; wait for this wave's DMA parts of it, then the whole CTA's
      if (nparts > 0 && s_valid) wait_vmcnt_dyn<(kWAhead - 1) * kWParts>(ops - mark0);
      barrier_lds();

      if (prev_kv && prev_end && attempt == 0 && (s_flag[0] | s_flag[1] | s_flag[2] | s_flag[3]) != 0) {
        // rare: the piece that just ended overflowed its exponent reference somewhere. Drain, rewind
        // the stream to its first KV tile and rerun it with each head's exact max (queries are still
        // in registers: no wave has touched tile j yet).
        wait_vmcnt<0>();
        barrier_lds();
        if constexpr (kScore) {
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) {  // the piece's exact max over both token halves
            const int h = 32 * hg + 16 * hb + c;
            m_ref[hb] = fmaxf(s_mx[0][h], s_mx[1][h]);
            m_max[hb] = -INFINITY;
            l_run[hb] = 0.f;
          }
          overflow = false;
        } else {
#pragma unroll
          for (int hq = 0; hq < 4; ++hq)
#pragma unroll
            for (int db = 0; db < 8; ++db) O[hq][db] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        attempt = 1;
        first_kv = true;
        cs = piece_cur;
        iss = piece_cur;
        j = piece_j;
        n_issued = nparts > 0 ? piece_j : 0;
        iss_kv = piece_kv;
        comp_kv = piece_kv;
        iss_valid = true;
        s_valid = true;
        prev_kv = false;
        ops = 0;
        if constexpr (kSmall) {  // the rewound tiles' offsets again (their ring slots were reused)
          if constexpr (kScore) if (role == 0) seed(piece_cur, piece_j);
          barrier_lds();
        }
        prologue(0);
        continue;
      }
      if (prev_kv && prev_end) attempt = 0;

      auto issue_next = [&]() __attribute__((always_inline)) {
        if (nparts > 0 && iss_valid) {
          issue(iss, n_issued++);
          mark2 = ops;
          iss_valid = advance(iss);
        }
      };
      // An output step requests its first LDS operands before it issues, so that they arrive meanwhile (split step,
      // 8 requests of 32k to 128k tokens: 147.3 -> 144.7 us; 64 of 1k to 8k: 69.7 -> 69.2). With small pages the
      // issue itself begins with an LDS read, and comes first (1.5 % slower after the operands).
      if (kSmall || !prev_kv) issue_next();

      const bool cur_kv = s_valid && cs.q == 2;
      const bool cur_end = cur_kv && cs.t + kTile >= cs.t1;
      if (cur_kv && first_kv) {
        piece_cur = cs;
        piece_j = j;
        piece_kv = comp_kv;
      }

      if constexpr (kScore) {
        const MLA_LDS char* T = (const MLA_LDS char*)smem + (j % kStages) * kTileBytes;
        if (s_valid && cs.q < 2) {
          // a piece starts: head group hg reads its 32 query rows (two head blocks) from query tile hg
          if (hg == cs.q) {
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
              for (int ks = 0; ks < 18; ++ks) {
                const int off = ((ks & 1) ? k_off_odd : k_off_even) + (ks >> 1) * kTileBlockBytes + 16 * hb * 128;
                qf[hb][ks] = *reinterpret_cast<const MLA_LDS bf16x8*>(T + off);
              }
          }
        } else if (cur_kv) {
          // ---- S^T[16 tokens (half th) x 16 heads] for head blocks hb = 0, 1; two chains each
          auto kread = [&](int ks) {
            const int off = ((ks & 1) ? k_off_odd : k_off_even) + (ks >> 1) * kTileBlockBytes + 16 * th * 128;
            return *reinterpret_cast<const MLA_LDS bf16x8*>(T + off);
          };
          f32x4 sacc[2][2];
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) sacc[hb][0] = sacc[hb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
          bf16x8 kbuf[kWKPrefetch];
#pragma unroll
          for (int r = 0; r < kWKPrefetch; ++r) kbuf[r] = kread(r);
#pragma unroll
          for (int ks = 0; ks < 18; ++ks) {
            const bf16x8 a = kbuf[ks % kWKPrefetch];
            if (ks + kWKPrefetch < 18) kbuf[ks % kWKPrefetch] = kread(ks + kWKPrefetch);
            sacc[0][ks & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[0][ks], sacc[0][ks & 1], 0, 0, 0);
            sacc[1][ks & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[1][ks], sacc[1][ks & 1], 0, 0, 0);
          }
          // ---- softmax numerators: lane (g, c) holds head 32 hg + 16 hb + c, tokens 16 th + 4 g + i
          const int valid = cs.t1 - cs.t;
          float x[2][4], mt[2];
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) {
            const f32x4 sv = sacc[hb][0] + sacc[hb][1];
            mt[hb] = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              x[hb][i] = sv[i] * p.scale_log2;
              if (valid < kTile && 16 * th + 4 * g + i >= valid) x[hb][i] = -INFINITY;
              mt[hb] = fmaxf(mt[hb], x[hb][i]);
            }
          }
          if (first_kv && attempt == 0) {
            mt[0] = wave_max_g(mt[0]);  // each head's max over this half of the tile
            mt[1] = wave_max_g(mt[1]);
            // the piece's reference: the first tile's max over both halves, agreed with the wave that
            // holds the other half (an extra barrier, which every wave takes at this step; the output
            // waves are idle here, the previous tile being a query tile)
            if (g == 0) {
              s_mx[th][32 * hg + c] = mt[0];
              s_mx[th][32 * hg + 16 + c] = mt[1];
            }
            barrier_lds();
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
              const int h = 32 * hg + 16 * hb + c;
              m_ref[hb] = fmaxf(s_mx[0][h], s_mx[1][h]);
            }
          }
          u32x2 pown[2];
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) {
            m_max[hb] = fmaxf(m_max[hb], mt[hb]);  // (over this lane's tokens; reduced when the piece ends)
            overflow |= mt[hb] > m_ref[hb] + kWOverflowLog2;
            float pr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              pr[i] = __builtin_amdgcn_exp2f(x[hb][i] - m_ref[hb]);
              l_run[hb] += pr[i];
            }
            pown[hb][0] = pack_bf16x2(pr[0], pr[1]);
            pown[hb][1] = pack_bf16x2(pr[2], pr[3]);
          }
          // the P^T B operand of head block 2 hg + hb, lane (g, c): k = 8g + i is token 4g + i (i < 4,
          // written by half 0) or 16 + 4g + i - 4 (half 1)
#pragma unroll
          for (int hb = 0; hb < 2; ++hb)
            reinterpret_cast<u32x2*>(&s_p[j & 1][2 * hg + hb][lane])[th] = pown[hb];
          if (cur_end) {
            // publish this half's row sums, the reference, the max and the overflow; reset
            const bool wave_overflow = __ballot(overflow) != 0;
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
              const float l_half = wave_sum_g(l_run[hb]);
              const float m_half = wave_max_g(m_max[hb]);
              const int h = 32 * hg + 16 * hb + c;
              if (g == 0) {
                s_l[th][h] = l_half;
                s_mx[th][h] = m_half;
                if (th == 0) s_mref[h] = m_ref[hb];
              }
              m_max[hb] = -INFINITY;
              l_run[hb] = 0.f;
            }
            if (lane == 0) s_flag[role] = wave_overflow ? 1 : 0;
            overflow = false;
          }
        }
      } else {
        // the score waves' reference exchange at a piece's first KV tile takes a barrier: take it too
        // (the previous tile is the piece's second query tile, so there is no output work here)
        if (cur_kv && first_kv && attempt == 0) barrier_lds();
      }
      if constexpr (!kScore) if (prev_kv) {
        // ---- output wave: O^T[16 dims x 16 heads] += V^T . P^T for tile j - 1, this wave's 8 dim
        // blocks and all 4 head blocks
        const MLA_LDS char* T = (const MLA_LDS char*)smem + ((j - 1) % kStages) * kTileBytes;
        auto vread = [&](int db, int half) {
          const int off = v_off[db & 3] + (db >> 2) * kTileBlockBytes + half * 16 * 128;
          return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((MLA_LDS bf16x4*)(T + off));
        };
        bf16x4 vlo[kWVPrefetch], vhi[kWVPrefetch];
#pragma unroll
        for (int r = 0; r < kWVPrefetch; ++r) {
          vlo[r] = vread(r, 0);
          vhi[r] = vread(r, 1);
        }
        bf16x8 pb[4];
#pragma unroll
        for (int hq = 0; hq < 4; ++hq) pb[hq] = __builtin_bit_cast(bf16x8, s_p[(j - 1) & 1][hq][lane]);
        if constexpr (!kSmall) issue_next();
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          const bf16x8 a =
              __builtin_shufflevector(vlo[db % kWVPrefetch], vhi[db % kWVPrefetch], 0, 1, 2, 3, 4, 5, 6, 7);
          if (db + kWVPrefetch < 8) {
            vlo[db % kWVPrefetch] = vread(db + kWVPrefetch, 0);
            vhi[db % kWVPrefetch] = vread(db + kWVPrefetch, 1);
          }
#pragma unroll
          for (int hq = 0; hq < 4; ++hq)
            O[hq][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[hq], O[hq][db], 0, 0, 0);
        }
        if (prev_end && (s_flag[0] | s_flag[1] | s_flag[2] | s_flag[3]) == 0) {
          // ---- the piece ended at tile j - 1: normalise and write this wave's dims of all 64 heads.
          // (An overflowed first attempt writes nothing; the vote at the next step reruns it.)
          const int b = rb + prev_r;
          const int npieces = __builtin_amdgcn_readfirstlane(s_np[prev_r]);
          const int slot = __builtin_amdgcn_readfirstlane(s_slot0[prev_r]) + w;
          const bool to_ws = npieces != 1;
          if (!to_ws || (slot >= 0 && slot < p.ws_slots)) {
#pragma unroll
            for (int hq = 0; hq < 4; ++hq) {
              const int h = 16 * hq + c;
              if (kMode != kExact && h >= p.heads) continue;
              const float l = s_l[0][h] + s_l[1][h];
              const float inv = l > 0.f ? 1.f / l : 0.f;
              if (to_ws) {
                // bf16 partial for the merge, one 16-byte chunk per dim-block pair (2 pp, 2 pp + 1): chunk
                // 16 role + 4 pp + g of the row (the chunk order of mla_amd.h)
                __bf16* orow = p.ws_o + ((int64_t)slot * p.heads + h) * kVDim + 128 * role + 8 * g;
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) {
                  u32x4 v;
                  v[0] = pack_bf16x2(O[hq][2 * pp][0] * inv, O[hq][2 * pp][1] * inv);
                  v[1] = pack_bf16x2(O[hq][2 * pp][2] * inv, O[hq][2 * pp][3] * inv);
                  v[2] = pack_bf16x2(O[hq][2 * pp + 1][0] * inv, O[hq][2 * pp + 1][1] * inv);
                  v[3] = pack_bf16x2(O[hq][2 * pp + 1][2] * inv, O[hq][2 * pp + 1][3] * inv);
                  *reinterpret_cast<u32x4*>(orow + 32 * pp) = v;
                }
              } else {
                __bf16* orow = p.out + (int64_t)b * p.out_stride_b + (int64_t)h * p.out_stride_h + 128 * role + 4 * g;
#pragma unroll
                for (int db = 0; db < 8; ++db) {
                  u32x2 v;
                  v[0] = pack_bf16x2(O[hq][db][0] * inv, O[hq][db][1] * inv);
                  v[1] = pack_bf16x2(O[hq][db][2] * inv, O[hq][db][3] * inv);
                  *reinterpret_cast<u32x2*>(orow + 16 * db) = v;
                }
              }
            }
            ops += (to_ws ? 4 : 8) * hblocks;
            // the LSE of head block `role`
            const int h = 16 * role + c;
            const float l = s_l[0][h] + s_l[1][h];
            const float lse_nat = l > 0.f ? (s_mref[h] + log2f(l)) * 0.69314718055994531f : -INFINITY;
            if (role < hblocks) {
              const bool h_ok = kMode == kExact || h < p.heads;
              if (!to_ws) {
                if (p.lse != nullptr) {
                  if (g == 0 && h_ok) p.lse[(int64_t)b * p.lse_stride_b + h] = lse_nat;
                  ops += 1;
                }
              } else {
                if (g == 0 && h_ok) p.ws_lse[(int64_t)slot * p.heads + h] = lse_nat;
                ops += 1;
              }
            }
          }
#pragma unroll
          for (int hq = 0; hq < 4; ++hq)
#pragma unroll
            for (int db = 0; db < 8; ++db) O[hq][db] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }

      if constexpr (kSmall && kScore) if (role == 0) la_step();  // tile j + 3's offsets, tile j + 4 in flight
      // ---- advance: tile j becomes the previous tile
      prev_kv = cur_kv;
      prev_end = cur_end;
      prev_r = cs.r;
      if (cur_kv) {
        ++comp_kv;
        first_kv = cur_end;  // the next KV tile starts a piece
      }
      if (s_valid) s_valid = advance(cs);
      mark0 = mark1;
      mark1 = mark2;
      ++j;
      if (!s_valid && !prev_kv) break;
    }
    };
    if (scorer) run(std::true_type{});
    else run(std::false_type{});
    return true;
  };

  if constexpr (kLoop) {
    const int step = kMode == kGroups ? (int)gridDim.x / ((p0.heads + 63) >> 6) : (int)gridDim.x;
    for (int w = w_first; w < p.num_ctas; w += step) {
      if (w != w_first) {  // the previous range's waves are done with the LDS tables and ring
        wait_vmcnt<0>();
        __syncthreads();
      }
      if (!range(w)) break;
    }
  } else {
    range(w_first);
  }
}

}  // namespace

bool decode_ws_takes(const DecodeParams& p) { return p.heads > 16 && row_offsets_fit(p, 32); }

template <bool kSmall, WMode kMode>
static void launch_mode(const DecodeParams& p, int groups, hipStream_t stream) {
  const int cus = current_device_cus();
  const bool loop = p.num_ctas > 2 * cus;  // measured at kLoop
  int ctas = loop ? cus : p.num_ctas;
  if (kMode == kGroups) ctas = (ctas + 7) / 8 * 8;  // ranges in eights (one per XCD)
  const dim3 grid(ctas * groups), threads(kWWaves * 64);
  if (loop) hipLaunchKernelGGL((mla_decode_ws_kernel<kSmall, true, kMode>), grid, threads, 0, stream, p);
  else hipLaunchKernelGGL((mla_decode_ws_kernel<kSmall, false, kMode>), grid, threads, 0, stream, p);
}

template <bool kSmall>
static void launch_ws(const DecodeParams& p, hipStream_t stream) {
  if (p.heads > 64) launch_mode<kSmall, kGroups>(p, (p.heads + 63) / 64, stream);
  else if (p.heads < 64) launch_mode<kSmall, kPadded>(p, 1, stream);
  else launch_mode<kSmall, kExact>(p, 1, stream);
}

hipError_t launch_decode_ws(const DecodeParams& p, hipStream_t stream) {
  if (p.log2_ps >= 5) launch_ws<false>(p, stream);
  else launch_ws<true>(p, stream);
  return hipGetLastError();
}

}  // namespace mla
