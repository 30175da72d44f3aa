// Shared pieces of the gfx950 absorbed-MLA decode kernels (mla_coop.hip: up
// to 16 query rows per CTA; mla_rows64.hip: 64 or 32): the fused fp8 row format,
// launch parameters, exact fp8 -> bf16 widening, and the device-side split
// plans the kernels deal their units from.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "mm_common.hpp"

namespace mm {
namespace mla {

constexpr int kLat = 512;
constexpr int kRope = 64;
constexpr int kQK = kLat + kRope;              // 576 bytes per fp8 row
constexpr int kPage = 64;                      // tokens per page of a block table
constexpr int kTileTok = 64;                   // tokens per tile; parts are whole tiles
constexpr int kMaxQLen = 8;
constexpr int kMaxHeads = 128;
// A row's running max is fixed at its first non-empty tile; later tiles may
// exceed it by up to 2^64 (p <= 2^64, no fp32 overflow of O or l). Beyond that
// the CTA falls back to an exact-max second pass.
constexpr float kGrowLimit = 64.f;
constexpr float kGrowSum = 18446744073709551616.f;  // 2^kGrowLimit, for tests on sums of p
constexpr int kRows64 = 64;  // query rows per CTA of the 64-row kernel
// Split partial records. Workspace: the O records (one per (b, part): rec_rows
// rows of 512 fp32, row-major), then
// the (m, l) pair of every (b, part, query row), then an 8-byte (parts, first
// record) entry per request. kMaxRecords caps the O rows of a workspace.
constexpr size_t kMaxRecords = 65536;

struct Params {
  const uint16_t* q_lat;  // [B, q_len, H, 512] bf16 (q_len 1: [B, H, 512])
  const uint16_t* q_pe;   // [B, q_len, H, 64]
  const uint8_t* kv;      // paged: [slots, 576] fp8; contiguous: [B, S, 576]
  uint16_t* o_lat;        // like q_lat
  float* ws;              // split partials (parts > 1)
  const int* seq_lens;    // [B] (paged)
  const int* rows;        // [B] q/out row per request, or null
  const int* kv_indices;  // flat per-token slots (paged)
  const int* kv_indptr;   // [B+1] (paged)
  const int* table;       // [B, max_blocks] 64-token pages (paged, instead of kv_indices / kv_indptr), or null
  int max_blocks, num_blocks;
  int B, H, q_len, S_fixed, parts, ngroups, paged;
  int unit_cap;           // units one round of CTAs over the CUs holds
  int min_chunk;          // tokens of the shortest part (equal parts)
  int workers;            // > 0: balanced split over this many units (see plan_work), 0: equal parts
  int qrows;              // H * q_len
  int rec_rows;           // O rows per split record (>= qrows)
  int q_plain;            // the query rows are off a 16-byte boundary: plain loads instead of gathers
  float score_c;          // scale * kv_scale * log2(e), fp32
  float kv_scale;
};

// Request b's context length and its place in the index array: its first flat
// slot, or its row of the block table. With a table no length reaches past the
// row and no page id (page_slot: the slot of its first token) past the pool.
__device__ __forceinline__ int req_len(const Params& p, int b) {
  const int len = p.seq_lens[b];
  if (!p.table) return len;
  const long long most = (long long)p.max_blocks * kPage;
  return len < 0 ? 0 : (len < most ? len : (int)most);
}
__device__ __forceinline__ int req_slot0(const Params& p, int b) {
  return p.table ? b * p.max_blocks : p.kv_indptr[b];
}
__device__ __forceinline__ int page_slot(const Params& p, int page) {
  return (page < 0 ? 0 : (page < p.num_blocks ? page : p.num_blocks - 1)) * kPage;
}

// Split workspace regions (see kMaxRecords).
__device__ __forceinline__ float* ws_rec_o(const Params& p, size_t rec) { return p.ws + rec * p.rec_rows * kLat; }
__device__ __forceinline__ float* ws_ml(const Params& p) { return p.ws + (size_t)p.B * p.parts * p.rec_rows * kLat; }
__device__ __forceinline__ int* ws_tbl(const Params& p) {
  return reinterpret_cast<int*>(ws_ml(p) + (size_t)p.B * p.parts * p.qrows * 2);
}

typedef int i32x2 __attribute__((ext_vector_type(2)));

// Two fp8 of a dword (lo or hi half) -> two bf16, exact (scale 1).
template <bool HI>
__device__ __forceinline__ uint32_t fp8x2_bf16(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, HI));
}
__device__ __forceinline__ bf16x8 fp8x8_bf16(uint32_t lo, uint32_t hi) {
  u32x4 o = {fp8x2_bf16<false>(lo), fp8x2_bf16<true>(lo), fp8x2_bf16<false>(hi), fp8x2_bf16<true>(hi)};
  return __builtin_bit_cast(bf16x8, o);
}

// Field `k` (16 bits) of a packed pair, extracted where it is used (volatile:
// not hoisted, so the packed pairs are what stays live).
__device__ __forceinline__ uint32_t u16_field(uint32_t w, int k) {
  uint32_t r;
  asm volatile("v_bfe_u32 %0, %1, %2, 16" : "=v"(r) : "v"(w), "i"(16 * k));
  return r;
}

// ---- split plan ------------------------------------------------------------------------
// The caller's `parts` P and the launch's unit cap (the CTAs of one round of
// the grid over the CUs, divided by the CTAs per unit) set a budget of
//   U = max(B, min(B * P, cap))
// units (request parts). Every request is cut into chunks of C tokens, request
// b getting nparts_b = max(1, ceil(L_b / C)) parts of equal size (rounded up to
// a tile; the last part takes the remainder), with C the smallest multiple of
// the tile, at least min_chunk, for which sum_b nparts_b <= U -- found by bisection,
// since the count only falls as C grows and C = max_b L_b gives B units. So the
// partial records always fit the B * P * qrows workspace, one round of CTAs
// covers the batch, and the longest part (the CTA that ends last) is as short
// as the budget allows.
// The paged plan keeps three B-entry tables (12 * B bytes) in LDS scratch.
constexpr int kMaxPagedB = 3072;  // 12 B per request: 36 KB of plan scratch

// ceil(a / d) for 0 <= a, 1 <= d, a + d < 2^32.
__host__ __device__ __forceinline__ int ceil_div_u(int a, int d) {
  return (int)(((unsigned)a + (unsigned)d - 1u) / (unsigned)d);
}
__device__ __forceinline__ int nparts_of(int L, int C) { return L <= C ? 1 : ceil_div_u(L, C); }
// Tokens per part of a request of L tokens in np parts: equal shares rounded up
// to whole tiles (the last part takes the remainder).
__device__ __forceinline__ int part_tokens(int L, int np) {
  return (ceil_div_u(L, np) + kTileTok - 1) & ~(kTileTok - 1);
}
__device__ __forceinline__ int unit_budget(int B, int P, int cap) {
  const long long bp = (long long)B * (P < 1 ? 1 : P);
  const long long m = bp < cap ? bp : cap;
  return (int)(m > B ? m : B);
}
// Smallest chunk C (a multiple of the tile, >= min_chunk) with units(C) <= budget,
// for a units(C) that is non-increasing in C with units(max L) = B <= budget.
// Wave-uniform.
template <class UnitsFn>
__device__ int search_chunk(long long sumL, int maxL, int B, int budget, int min_chunk, UnitsFn units) {
  int hi = maxL < min_chunk ? min_chunk : ((maxL + kTileTok - 1) & ~(kTileTok - 1));
  if (budget <= B) return hi;  // one part per request
  // ceil(L / C) < L / C + 1, so C >= sumL / (budget - B) is feasible too.
  auto ceil_div_ll = [](long long a, int d) -> long long {  // 32-bit division whenever it suffices
    return a < 0x7FFFFFFF ? (long long)ceil_div_u((int)a, d) : (a + d - 1) / d;
  };
  const long long ok = ceil_div_ll(sumL, budget - B);
  if (ok < hi) hi = ok < min_chunk ? min_chunk : (int)((ok + kTileTok - 1) & ~(long long)(kTileTok - 1));
  // units(C) >= sumL / C, so C >= sumL / budget.
  const long long need = ceil_div_ll(sumL, budget);
  int lo = need > hi ? hi : (int)need;
  lo = (lo + kTileTok - 1) & ~(kTileTok - 1);
  lo = lo < min_chunk ? min_chunk : (lo > hi ? hi : lo);
  while (lo < hi) {
    const int mid = lo + ((hi - lo) / (2 * kTileTok)) * kTileTok;
    if (units(mid) <= budget) {
      hi = mid;
    } else {
      lo = mid + kTileTok;
    }
  }
  return hi;
}

// Wave64 reductions on DPP row shifts / broadcasts (no LDS); wave_incl_scan is
// in mm_common.hpp.
__device__ __forceinline__ int wave_sum_i(int v) { return __builtin_amdgcn_readlane(wave_incl_scan(v), 63); }
__device__ __forceinline__ int wave_max_i(int v) {
  // Invalid DPP sources return `old` = the lane's own value (neutral for max).
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

struct Unit {
  int b;       // request
  int part;    // part within the request
  int nparts;  // parts of the request
  int rec0;    // record part index of the request's part 0 (request-index order)
  int ptok;    // tokens per part of this request
  int units;   // total units (request parts) in the batch
  int len;     // context length of request b
  int slot0;   // first flat slot index of request b (paged: kv_indptr[b])
};

// Unit `u` of the batch. When the units fit one round of CTAs they run in
// request order; otherwise in longest-first order: requests sorted into 16
// linear buckets of their part size (largest first, request index inside a
// bucket), each request's parts consecutive. Wave-uniform, computed by one wave
// in `scratch` (12 * B bytes of LDS that no other wave touches meanwhile). The
// first 64 lengths and kv_indptr entries are loaded in one round of latency, so
// the unit's length and slot offset cost no further round trip for b < 64.
__device__ Unit plan_unit_paged(const Params& p, int u, int lane, int* scratch) {
  const int B = p.B, P = p.parts, cap = p.unit_cap;
  int* lens = scratch;            // [B] lengths
  int* req_at = scratch + B;      // [B] request at each position
  int* np_at = scratch + 2 * B;   // [B] parts of the request at each position
  const int ip0 = lane < B ? req_slot0(p, lane) : 0;
  const int l0 = lane < B ? req_len(p, lane) : 0;  // the first 64 lengths stay in a register
  long long suml = 0;
  int maxl = 0;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const int l = c0 == 0 ? l0 : ((c0 + lane < B) ? req_len(p, c0 + lane) : 0);
    if (c0 + lane < B) lens[c0 + lane] = l;
    suml += wave_sum_i(l);  // per-chunk sums stay below 2^31 for lengths < 2^25
    maxl = max(maxl, wave_max_i(l));
  }
  auto len_at = [&](int c0) { return c0 == 0 ? l0 : ((c0 + lane < B) ? lens[c0 + lane] : 0); };
  const int budget = unit_budget(B, P, cap);
  const int C = search_chunk(suml, maxl, B, budget, p.min_chunk, [&](int c) {
    int n = 0;
    for (int c0 = 0; c0 < B; c0 += 64) n += wave_sum_i(c0 + lane < B ? nparts_of(len_at(c0), c) : 0);
    return n;
  });
  if (budget <= cap) {
    // Every unit gets a CTA of the first round, so their order does not matter:
    // units in request order, which is also the record order (unit u of request
    // b is record rec0(b) + part).
    Unit r{0, 0, 1, 0, kTileTok, 0, 0, 0};
    int run = 0;  // units of the requests before this chunk
    bool found = false;
    for (int c0 = 0; c0 < B; c0 += 64) {
      const bool valid = c0 + lane < B;
      const int l = len_at(c0);
      const int np = valid ? nparts_of(l, C) : 0;
      const int inc = wave_incl_scan(np);
      const int excl = run + inc - np;
      const unsigned long long hit = __builtin_amdgcn_ballot_w64(valid && u >= excl && u < excl + np);
      if (!found && hit) {
        const int hl = (int)__builtin_ctzll(hit);
        r.b = c0 + hl;
        r.rec0 = __builtin_amdgcn_readlane(excl, hl);
        r.part = u - r.rec0;
        r.nparts = __builtin_amdgcn_readlane(np, hl);
        r.len = __builtin_amdgcn_readlane(l, hl);
        found = true;
      }
      run += __builtin_amdgcn_readlane(inc, 63);
    }
    r.units = run;
    r.ptok = part_tokens(r.len, r.nparts);
    r.slot0 = r.b < 64 ? __builtin_amdgcn_readlane(ip0, r.b) : req_slot0(p, r.b);
    return r;
  }
  // More requests than the cap (several rounds of CTAs): longest parts first.
  int maxp = 0;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const bool valid = c0 + lane < B;
    const int l = valid ? lens[c0 + lane] : 0;
    const int pt = valid ? part_tokens(l, nparts_of(l, C)) : 0;
    maxp = max(maxp, wave_max_i(pt));
  }
  maxp = __builtin_amdgcn_readfirstlane(maxp);
  auto bucket_of = [&](int pt) {  // 0 = largest parts; pt <= maxp < 2^27
    const unsigned q = (unsigned)pt * 16u / ((unsigned)maxp + 1u);
    return 15 - (int)q;
  };
  int start[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) start[k] = 0;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const bool valid = c0 + lane < B;
    const int l = valid ? lens[c0 + lane] : 0;
    const int bk = valid ? bucket_of(part_tokens(l, nparts_of(l, C))) : -1;
#pragma unroll
    for (int k = 0; k < 16; ++k) start[k] += __builtin_popcountll(__builtin_amdgcn_ballot_w64(bk == k));
  }
  int acc = 0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int c = start[k];
    start[k] = acc;
    acc += c;
  }
  const unsigned long long lt = (1ull << lane) - 1ull;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const bool valid = c0 + lane < B;
    const int l = valid ? lens[c0 + lane] : 0;
    const int np = nparts_of(l, C);
    const int bk = valid ? bucket_of(part_tokens(l, np)) : -1;
    int pos = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const unsigned long long m = __builtin_amdgcn_ballot_w64(bk == k);
      if (bk == k) pos = start[k] + __builtin_popcountll(m & lt);
      start[k] += __builtin_popcountll(m);
    }
    if (valid) {
      req_at[pos] = c0 + lane;
      np_at[pos] = np;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  Unit r{0, 0, 1, 0, kTileTok, 0, 0, 0};
  int run = 0;  // units before this chunk of positions
  bool found = false;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const bool valid = c0 + lane < B;
    const int np = valid ? np_at[c0 + lane] : 0;
    const int inc = wave_incl_scan(np);
    const int excl = run + inc - np;
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(valid && u >= excl && u < excl + np);
    if (!found && hit) {
      const int hl = (int)__builtin_ctzll(hit);
      r.b = __builtin_amdgcn_readlane(req_at[c0 + lane], hl);
      r.part = u - __builtin_amdgcn_readlane(excl, hl);
      r.nparts = __builtin_amdgcn_readlane(np, hl);
      found = true;
    }
    run += __builtin_amdgcn_readlane(inc, 63);
  }
  r.units = run;
  r.len = lens[r.b];
  r.ptok = part_tokens(r.len, r.nparts);
  r.slot0 = r.b < 64 ? __builtin_amdgcn_readlane(ip0, r.b) : req_slot0(p, r.b);
  // Record offset: parts of the requests before b, in request-index order.
  int rec0 = 0;
  for (int c0 = 0; c0 < B; c0 += 64) {
    const int idx = c0 + lane;
    rec0 += wave_sum_i(idx < B && idx < r.b ? nparts_of(lens[idx], C) : 0);
  }
  r.rec0 = rec0;
  return r;
}

// Unit `u` of a contiguous batch (every request S tokens): the same chunking,
// units in request order.
__device__ __forceinline__ Unit plan_unit_contig(int S, int B, int P, int cap, int min_chunk, int u) {
  const int C =
      search_chunk((long long)B * S, S, B, unit_budget(B, P, cap), min_chunk, [&](int c) { return B * nparts_of(S, c); });
  const int np = nparts_of(S, C);
  return Unit{u / np, u % np, np, (u / np) * np, part_tokens(S, np), B * np, S, 0};
}

// ---- balanced split --------------------------------------------------------------------
// With records for it (W + B - 1 <= B * P) a round of W units shares the
// batch's tiles evenly, whatever its lengths: the requests' 64-token tiles are
// laid end to end, kSegCost places before each request standing for what
// starting one costs a unit (2 .. 8 measured: 64 requests of 1024 .. 8192
// tokens, 16 heads 39.2 us with 3, 38.3 with 4 and 5; 128 heads 103.3 us with 2,
// 101.0 with 4, 101.6 with 8), and unit u walks places [u * tw, (u + 1) * tw), one
// segment per request it meets there. Equal parts per request leave the longest
// part 14% (256 units) to 80% (64 units) above the mean on lengths of
// U[1024, 8192]. A request's segments are consecutive units, so its records
// are consecutive too: segment (u, b) takes record u + b.
constexpr int kSegCost = 4;
constexpr int kMinWork = 4;    // places per unit at least

// A part of a request: what a CTA works on at a time.
struct Seg {
  int b;               // request, -1: none
  int part, nparts;    // part within the request
  int rec0;            // record index of the request's part 0
  int kv_lo, kv_hi;    // tokens of the part
  int len;             // context length of the request
  int slot0;           // its first flat slot index (paged)
  int pos;             // place of the request's first tile (balanced split)
  int tw;              // places per unit (0: equal parts, one segment per unit)
};
__host__ __device__ __forceinline__ int work_tiles(int len) { return len > kTileTok ? (len - 1) / kTileTok + 1 : 1; }

// Places per unit when `total` of them share `workers` units.
__host__ __device__ __forceinline__ int work_share(int total, int workers) {
  const int tw = ceil_div_u(total, workers);
  return tw > kMinWork ? tw : kMinWork;
}

// Unit u's segment of a request whose first tile is at `pos`.
__host__ __device__ __forceinline__ Seg work_seg(int u, int tw, int b, int pos, int len, int slot0) {
  const int nt = work_tiles(len);
  const int u0 = pos / tw;
  const int lo = u * tw > pos ? u * tw - pos : 0;
  const int hi = (u + 1) * tw - pos < nt ? (u + 1) * tw - pos : nt;
  const int end = len > 0 ? len : 0;
  Seg r{b, u - u0, (pos + nt - 1) / tw - u0 + 1, u0 + b, lo * kTileTok, end, len, slot0, pos, tw};
  if (hi < nt) r.kv_hi = hi * kTileTok;
  if (hi <= 0) r.b = -1;  // the unit's places end before the tiles begin
  return r;
}

// The first segment of unit u, by one wave (`scratch`: as plan_unit_paged).
template <bool PAGED>
__device__ Seg plan_work(const Params& p, int u, int lane, int* scratch) {
  if (p.workers == 0) {
    const Unit un = PAGED ? plan_unit_paged(p, u, lane, scratch)
                          : plan_unit_contig(p.S_fixed, p.B, p.parts, p.unit_cap, p.min_chunk, u);
    const long long lo = (long long)un.part * un.ptok;
    const int kv_lo = lo < un.len ? (int)lo : un.len;
    const int kv_hi = lo + un.ptok < un.len ? (int)(lo + un.ptok) : un.len;
    return Seg{u < un.units ? un.b : -1, un.part, un.nparts, un.rec0, kv_lo, kv_hi, un.len, un.slot0, 0, 0};
  }
  const Seg none{-1, 0, 1, 0, 0, 0, 0, 0, 0, 1};
  if (u >= p.workers) return none;
  if constexpr (!PAGED) {
    const int per = work_tiles(p.S_fixed) + kSegCost;
    const int tw = work_share(p.B * per, p.workers);
    const int b = u * tw / per;
    return b < p.B ? work_seg(u, tw, b, b * per + kSegCost, p.S_fixed, 0) : none;
  }
  const int l0 = lane < p.B ? req_len(p, lane) : 0;  // the first 64 requests cost one round trip
  const int s0 = lane < p.B ? req_slot0(p, lane) : 0;
  auto len_at = [&](int c0) { return c0 == 0 ? l0 : (c0 + lane < p.B ? req_len(p, c0 + lane) : 0); };
  auto places = [&](int c0, int l) { return c0 + lane < p.B ? work_tiles(l) + kSegCost : 0; };
  int total = 0;
  for (int c0 = 0; c0 < p.B; c0 += 64) total += wave_sum_i(places(c0, len_at(c0)));
  const int tw = work_share(total, p.workers);
  int run = 0;
  for (int c0 = 0; c0 < p.B; c0 += 64) {
    const int l = len_at(c0);
    const int inc = run + wave_incl_scan(places(c0, l));  // end of the request's places
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(c0 + lane < p.B && inc > u * tw);
    if (hit) {
      const int h = (int)__builtin_ctzll(hit);
      const int len = __builtin_amdgcn_readlane(l, h);
      const int pos = __builtin_amdgcn_readlane(inc, h) - work_tiles(len);
      const int slot0 = c0 == 0 ? __builtin_amdgcn_readlane(s0, h) : req_slot0(p, c0 + h);
      return work_seg(u, tw, c0 + h, pos, len, slot0);
    }
    run = __builtin_amdgcn_readlane(inc, 63);
  }
  return none;
}

// Unit u's segment after `sg`, or b = -1. `len`, `slot0`: of request sg.b + 1.
__host__ __device__ __forceinline__ Seg next_work(int B, const Seg& sg, int u, int len, int slot0) {
  Seg r = sg;
  r.b = -1;
  if (sg.tw == 0 || sg.b + 1 >= B) return r;
  const int pos = sg.pos + work_tiles(sg.len) + kSegCost;
  return pos < (u + 1) * sg.tw ? work_seg(u, sg.tw, sg.b + 1, pos, len, slot0) : r;
}

// One wave's segment to all: posted in `misc` (10 ints), read after a barrier.
__device__ __forceinline__ void post_seg(int* misc, const Seg& s) {
  const int v[10] = {s.b, s.part, s.nparts, s.rec0, s.kv_lo, s.kv_hi, s.len, s.slot0, s.pos, s.tw};
#pragma unroll
  for (int i = 0; i < 10; ++i) misc[i] = v[i];
}
__device__ __forceinline__ Seg read_seg(const int* misc) {
  auto at = [&](int i) { return __builtin_amdgcn_readfirstlane(misc[i]); };
  return Seg{at(0), at(1), at(2), at(3), at(4), at(5), at(6), at(7), at(8), at(9)};
}

// 4-byte global -> LDS DMA (lane l's dword lands at lds_dst + 4*l), counted by
// the kernel itself like dma16_opaque.
__device__ __forceinline__ void dma4_opaque(const void* gsrc, const char* lds_dst) {
  const uint32_t m0v = (uint32_t)(uintptr_t)(MM_LDS const char*)lds_dst;
  asm volatile("global_load_lds_dword %0, off" ::"v"(gsrc), "{m0}"(m0v) : "memory");
}

// 16 bytes from any address to LDS (`lds_dst`: this lane's), by plain loads.
__device__ __forceinline__ void copy16_plain(const void* gsrc, char* lds_dst) {
  u32x4 v;
  __builtin_memcpy(&v, gsrc, 16);
  *reinterpret_cast<u32x4*>(lds_dst) = v;
}

// Staging layout of one tile: token t's 576-byte row at t*576, its 16-byte
// piece c stored at piece slot c ^ swz(t) (a permutation inside each aligned
// group of 4 pieces) so the 32 lanes of a K read and the 8-token groups of a
// V^T transpose read hit distinct LDS banks.
__device__ __forceinline__ int swz(int t) { return (t >> 2) & 3; }

// Host launchers of the 16-row kernel (mla_coop.hip) and the 64-row kernel
// (mla_rows64.hip); grid = CTAs.
int launch_coop_kernel(const Params& p, long long grid, hipStream_t st);
int launch_rows64_kernel(const Params& p, long long grid, hipStream_t st);

}  // namespace mla
}  // namespace mm
