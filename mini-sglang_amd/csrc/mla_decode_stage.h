// Staging of a decode CTA's plan range in LDS, shared by the streaming decode kernels.
#pragma once

#include "mla_common.h"
#include "mla_device.h"

namespace mla {

// A request's length and plan entry {first CTA, pieces, slot base} by scalar loads, waited for together.
__device__ __forceinline__ void sload_request(const int32_t* seq_len, const int32_t* info, int& len, int& first,
                                              int& pieces, int& slot) {
  typedef int i32x2_t __attribute__((__vector_size__(8)));
  int l, s;
  i32x2_t v;
  asm volatile("s_load_dword %0, %3, 0x0\n\ts_load_dwordx2 %1, %4, 0x0\n\ts_load_dword %2, %4, 0x8\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&s"(l), "=&s"(v), "=&s"(s) : "s"(seq_len), "s"(info) : "memory");
  len = l;
  first = v[0];
  pieces = v[1];
  slot = s;
}

// LDS tables of a decode CTA's plan range [(rb, kb), (re, ke)): per request its token bounds, pieces and slot
// base, and (kPages) one clamped page id per 32-token tile of the range, page_cap at most.
struct RangeTables {
  int* t0;     // [kMaxCtaRequests]
  int* t1;     // [kMaxCtaRequests]
  int* tbase;  // [kMaxCtaRequests + 1] scratch: first tile of each request
  int* np;     // [kMaxCtaRequests]
  int* slot0;  // [kMaxCtaRequests]
  int* pid;
};

// Fills the tables for the nreq (1..kMaxCtaRequests) requests of the range; every thread of the CTA calls it, and
// it ends with a barrier (LDS only). A range inside one request, the usual case of a batch smaller than the
// grid, needs no scan and one barrier where the general case takes three. The page ids are read once the
// request's length is known: what bounds the columns of a row that exist is its length alone, not the plan
// (made for another step's lengths, perhaps) nor the table's row stride (1 for a one-row table's transpose).
template <int kThreads, bool kPages, int kPageCap>
__device__ __forceinline__ void stage_range(const DecodeParams& p, int rb, int kb, int re, int ke, int nreq, int lane,
                                            int wave, const RangeTables& s) {
  const int32_t* req_info = p.plan + 4 * (int64_t)p.num_ctas;
  const int tid = threadIdx.x;
  constexpr int kPer = (kPageCap + kThreads - 1) / kThreads;
  int pid[kPer];
  auto load_pages = [&](int t0, int t1) {
    const int32_t* row = p.page_table + (int64_t)rb * p.pt_stride;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int t = t0 + kTile * (tid + kThreads * u);
      pid[u] = t < t1 ? row[t >> p.log2_ps] : 0;
    }
  };
  if (nreq == 1) {
    const int t0 = kb * kPlanBlock;
    int L, first, pieces, slot;
    sload_request(p.seq_lens + rb, req_info + 3 * (int64_t)rb, L, first, pieces, slot);
    const int t1 = max(t0, re == rb ? min(ke * kPlanBlock, L) : L);
    if (tid == 0) {
      s.t0[0] = t0;
      s.t1[0] = t1;
      s.np[0] = pieces;
      s.slot0[0] = slot - first;
    }
    if constexpr (kPages) {
      load_pages(t0, t1);
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int k = tid + kThreads * u;
        if (k < kPageCap && t0 + kTile * k < t1) s.pid[k] = min(max(pid[u], 0), p.num_pages - 1);
      }
    }
    barrier_lds();
    return;
  }
  for (int r = tid; r < nreq; r += kThreads) {
    const int b = rb + r;
    const int L = p.seq_lens[b];
    const int t0 = (r == 0) ? kb * kPlanBlock : 0;
    const int t1 = max(t0, (b == re) ? min(ke * kPlanBlock, L) : L);
    s.t0[r] = t0;
    s.t1[r] = t1;
    s.tbase[r + 1] = (t1 - t0 + kTile - 1) / kTile;
    const int first = req_info[3 * b + 0];
    s.np[r] = req_info[3 * b + 1];
    s.slot0[r] = req_info[3 * b + 2] - first;
  }
  barrier_lds();
  if constexpr (kPages) {
    if (wave == 0) {  // exclusive prefix of tile counts (64-wide scans)
      int carry = 0;
      for (int c0 = 0; c0 < nreq; c0 += 64) {
        const int r = c0 + lane;
        int v = r < nreq ? s.tbase[r + 1] : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int u = __shfl_up(v, o);
          if (lane >= o) v += u;
        }
        if (r < nreq) s.tbase[r + 1] = carry + v;
        carry += __shfl(v, 63);
      }
      if (lane == 0) s.tbase[0] = 0;
    }
    barrier_lds();
    const int ntiles = min(s.tbase[nreq], kPageCap);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = tid + kThreads * u;
      pid[u] = 0;
      if (k < ntiles) {
        int lo = 0, hi = nreq - 1;  // last request whose first tile is <= k
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (s.tbase[mid] <= k) lo = mid;
          else hi = mid - 1;
        }
        const int t = s.t0[lo] + kTile * (k - s.tbase[lo]);
        pid[u] = p.page_table[(int64_t)(rb + lo) * p.pt_stride + (t >> p.log2_ps)];
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = tid + kThreads * u;
      if (k < ntiles) s.pid[k] = min(max(pid[u], 0), p.num_pages - 1);
    }
    barrier_lds();
  }
}

}  // namespace mla
