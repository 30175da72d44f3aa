// Absorbed-MLA decode for query blocks of more than 16 rows (H * q_len > 16) on
// MI355X (gfx950). Same contract, split plan and numerics as the 16-row kernel
// (reference csrc/mla_decode_a16w8.hip:183-754, csrc/mla_decode_a16w8_multiq.hip
// :282-856), cut for two waves per SIMD:
//
//  * One CTA = 64 query rows (two row tiles of 32; one in calls of 17..32 rows
//    and in small ones of 33..64, see cta_rows_for) of one request part, 8
//    waves. The part's fp8 rows are gathered in 64-token tiles into a shared
//    3-slot LDS ring, wave w gathering tokens 8w .. 8w+7 of every tile.
//  * S^T = K Q^T on v_mfma_f32_32x32x16_bf16: wave (rt, tt, kh) scores row tile
//    rt against token half tt over dims 288 kh .. 288 kh + 287, so a wave holds
//    half of its rows' Q (72 VGPRs) and widens half of a 32-token tile. The two
//    dim halves are summed through LDS: each wave of a pair hands the other 8
//    of its 16 accumulators and finishes 16 tokens itself. (The dim-half 1
//    wave reads its K rows with bit 4 of the token flipped, so that in both
//    waves registers 0..7 are the ones to keep.)
//  * Softmax in base 2 on the integer grid: each row's max m is fixed for the
//    whole CTA at the part's first tile, p = exp2(s c - m) (<= 2^64 later, else
//    the exact-max fallback). A wave's 8 p per lane are exactly one B operand
//    of PV, published in LDS as one 1 KB fragment.
//  * O^T = V^T P^T is split by output dims: wave w accumulates latent dims
//    64w .. 64w+63 of all 64 rows (2 d-tiles x 2 row tiles, 64 VGPRs) over all
//    64 tokens: each V^T fragment is widened once per CTA and feeds two MFMAs,
//    and no output crosses waves at the end.
//  * Two barriers per tile. Between them (phase B) a wave finishes its 16
//    tokens' softmax under the second half of the previous tile's PV MFMAs,
//    whose operands are in registers by the first barrier; that barrier also
//    frees the previous tile's slot, into which the tile two ahead is gathered.
//
// What bounds it (128 heads, 128 x 4096 tokens): a tile takes 1.87 us on every
// CU = 1.22 PFLOP/s, the rate of a large bf16 library GEMM here, with the clock
// held at 1.95 GHz by the power limit. Copies of the kernel without the exchange
// barrier, without the exchange or without the converts are 0..4% faster, one
// without the gathers 27% (the clock rises to 2.35 GHz): energy, not issue.
// Against the kernels it replaced (128 rows per CTA with one wave per SIMD, and
// 32 rows with a 4-wave merge), with the balanced split: 64 requests of
// 1024..8192 tokens, 128 heads 104.9 -> 98.4 us, with 2 drafts 184.8 -> 174.6;
// 32 requests, 16 heads, 4 drafts 44.1 -> 40.8; 3 requests of 2..8K tokens, 16
// heads, 8 drafts 53 -> 30.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <type_traits>

#include "mla_common.hpp"

namespace mm {
namespace mla {

constexpr int kRRows = kRows64;                         // query rows per CTA
constexpr int kRWaves = 8;
constexpr int kRThreads = 64 * kRWaves;
constexpr int kRTileTok = 64;                           // tokens per tile
constexpr int kRSubTok = kRTileTok / kRWaves;           // tokens a wave gathers per tile
constexpr int kRTileBytes = kRTileTok * kQK;            // 36864
constexpr int kRSubBytes = kRSubTok * kQK;              // 4608: four and a half 1 KB DMAs
constexpr int kRDma = 5;                                // DMA instructions per wave and tile
constexpr int kRDmaB = 2;                               // of them issued in phase B, the rest in the next phase A
constexpr int kRSlots = 3;
static_assert(kRRows * kQK * 2 <= 2 * kRTileBytes, "the query rows fit two ring slots");
constexpr int kRPairs = kQK / 64;                       // 32-dim pairs of one dim half

// LDS map (bytes). Ring slot 2 receives its first tile only after the first
// tile's first barrier; before that it holds the plan scratch (wave 0). The
// epilogue stages the 64 output rows over the ring, P and X.
constexpr int kRRingBytes = kRSlots * kRTileBytes;                // 110592
constexpr int kRScratchOff = 2 * kRTileBytes;
constexpr int kRPOff = kRRingBytes;                               // P^T fragments [token quarter][row tile] x 1 KB
constexpr int kRPBytes = 8 * 1024;                                // double-buffered by tile parity
constexpr int kRXOff = kRPOff + 2 * kRPBytes;                     // exchanged scores [receiving wave] x 2 KB
constexpr int kRIdxOff = kRXOff + kRWaves * 2048;                 // slot indices [wave][2 batches of 8 tiles][8 tokens]
constexpr int kRIdxBytes = 2 * 64 * 4;                            // per wave
constexpr int kRMaxOff = kRIdxOff + kRWaves * kRIdxBytes;         // [token quarter][64 rows] row max
constexpr int kRLOff = kRMaxOff + 4 * kRRows * 4;                 // [token quarter][64 rows] row l
constexpr int kRMiscOff = kRLOff + 4 * kRRows * 4;                // unit broadcast, fallback flags
constexpr int kRLdsBytes = kRMiscOff + 64;
static_assert(12 * kMaxPagedB <= kRTileBytes, "plan scratch fits ring slot 2");
static_assert(kRRows * kLat * 4 <= kRIdxOff, "the staged output rows leave the rest alone");
static_assert(kRLdsBytes <= 160 * 1024, "LDS budget");

// NRT: row tiles of a CTA (1: at most 32 rows in the call, or groups of 32). NT:
// non-temporal gathers, for calls whose tokens one CTA reads once (one row
// group).
template <bool PAGED, int NRT, bool NT>
__global__ __launch_bounds__(kRThreads, 1) void mla_rows64_kernel(Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kRLdsBytes];
  const int tid = threadIdx.x;
  const int lane0 = tid & 63;
  const int wave0 = __builtin_amdgcn_readfirstlane(tid >> 6);
  int* misc = reinterpret_cast<int*>(lds + kRMiscOff);

  // ---- work item: units dealt over the XCDs in snake order, the ngroups CTAs
  // of a unit consecutive on one XCD (they read the same tokens) ------------------
  const int xcd = blockIdx.x % kNumXcds;
  const int k_in_xcd = blockIdx.x / kNumXcds;
  const int uslot = k_in_xcd / p.ngroups;
  const int grp = k_in_xcd % p.ngroups;
  const int u = 16 * (uslot >> 1) + ((uslot & 1) ? 15 - xcd : xcd);
  Seg sg;
  if constexpr (PAGED) {
    // Wave 0 plans in ring slot 2 and broadcasts the segment.
    if (wave0 == 0) {
      const Seg s0 = plan_work<true>(p, u, lane0, reinterpret_cast<int*>(lds + kRScratchOff));
      if (lane0 == 0) post_seg(misc, s0);
    }
    lds_reads_done_barrier();
    sg = read_seg(misc);
  } else {
    sg = plan_work<false>(p, u, lane0, nullptr);
  }
  if (sg.b < 0) return;  // nothing for this unit: every wave leaves together

  // One part after the other (the balanced split gives a unit several).
  for (;;) {
    // Opaque per part: what follows from the lane and wave ids is worked out
    // again for each part instead of being carried (and spilled) across them.
    int lane = lane0, wave = wave0;
    asm volatile("" : "+v"(lane), "+s"(wave));
    const int n = lane & 31;  // MFMA column (query row) / row of A (token for QK, dim for PV)
    const int g = lane >> 5;  // lane half
    // Roles in QK and softmax. Waves w and w + 4 share a SIMD: with one row tile
    // (NRT 1) every SIMD has one scoring wave.
    const int rt = wave >> 2;
    const int tt = (wave >> 1) & 1;
    const int kh = wave & 1;
    const int quarter = 2 * tt + kh;  // the 16 tokens of a tile this wave finishes
    const bool scores = NRT == 2 || rt < NRT;
    char* idx = lds + kRIdxOff + wave * kRIdxBytes;  // this wave's slot indices
    float* red_m = reinterpret_cast<float*>(lds + kRMaxOff);
    float* red_l = reinterpret_cast<float*>(lds + kRLOff);

    const int b = __builtin_amdgcn_readfirstlane(sg.b);
    const int part = sg.part;
    // The next request's length and first slot, loaded early.
    const int bn = b + 1 < p.B ? b + 1 : b;
    const int next_len = PAGED ? req_len(p, bn) : p.S_fixed;
    const int next_slot0 = PAGED ? req_slot0(p, bn) : 0;
    int qb = b;
    if (p.rows) {
      qb = p.rows[b];
      qb = qb < 0 ? 0 : (qb >= p.B ? p.B - 1 : qb);
    }
    const int S = sg.len;
    const int slot0 = sg.slot0;
    const int kv_lo = __builtin_amdgcn_readfirstlane(sg.kv_lo);
    const int kv_hi = __builtin_amdgcn_readfirstlane(sg.kv_hi);

    // ---- the query row of this lane's MFMA column --------------------------------------
    const int row0 = grp * 32 * NRT;
    const int qrow = row0 + 32 * rt + n;
    const int qr = qrow < p.qrows ? qrow : p.qrows - 1;  // padding columns repeat the last row
    const int lim = S - (p.q_len - 1 - qr / p.H);          // tokens >= lim are masked for this row
    const int lim_min = S - (p.q_len - 1 - row0 / p.H);    // no row of the CTA has a smaller one

    const int ntiles = (kv_hi - kv_lo + kRTileTok - 1) / kRTileTok;

    // ---- per-lane constant offsets inside a staged tile ---------------------------------
    // Token t's 576-byte row at t*576, its 16-byte piece c at piece slot c ^ swz(t).
    // K read of pair s: token 32 tt + (n ^ 16 kh), piece 18 kh + 2s + g. The piece
    // is 0 or 2 (mod 4) plus g: even pairs from koff_e, odd ones from koff_o.
    const int ktok = 32 * tt + (n ^ (16 * kh));
    const int kA = ktok * kQK + 16 * (g ^ swz(ktok));
    const int kB = ktok * kQK + 16 * ((2 + g) ^ swz(ktok));
    const int koff_e = kh ? kB + 256 : kA;
    const int koff_o = kh ? kA + 320 : kB;
    // V^T transpose read (16-lane group 2g + mh, member j): member j supplies 8
    // bytes of token T = 8(e/4) + 4g + e%4 (e = j/2, +16 per k-step), dims
    // 64w + 32dt + 16mh + 8(j&1) .. +8; swz(T) = 2(e/4) + g for every k-step.
    const int vj = lane & 15, vmh = (lane >> 4) & 1, ve = vj >> 1;
    const int vT = 8 * (ve >> 2) + 4 * g + (ve & 3);
    const int vsw = 2 * (ve >> 2) + g;
    const int voff0 = vT * kQK + 16 * (vmh ^ vsw) + 8 * (vj & 1) + 64 * wave;
    const int voff1 = vT * kQK + 16 * ((2 + vmh) ^ vsw) + 8 * (vj & 1) + 64 * wave;
    // DMA: instruction k moves LDS pieces 64k .. 64k+63 of this wave's 8 rows (36
    // pieces per row; the fifth is half an instruction): lane l fills piece slot
    // pc = 64k + l, i.e. token tg = pc / 36, slot cs = pc % 36, with global piece
    // cs ^ swz(8w + tg). Offsets < 2^13, two per VGPR.
    uint32_t dma_pk[3];
#pragma unroll
    for (int k = 0; k < kRDma; ++k) {
      const int pc = 64 * k + lane;
      const int tg = pc / 36, cs = pc % 36;
      const uint32_t off = tg * kQK + 16 * (cs ^ swz(kRSubTok * wave + tg));
      dma_pk[k / 2] = (k & 1) ? (dma_pk[k / 2] | (off << 16)) : off;
    }
    // The same for the slow paths, worked out again from a lane id the compiler
    // cannot hoist, so that nothing of it stays live through the tile loop.
    auto dma_place = [&](int k, int& tg, int& off) {
      int l = lane;
      asm volatile("" : "+v"(l));
      const int pc = 64 * k + l;
      tg = pc / 36;
      off = 16 * ((pc - 36 * tg) ^ swz(kRSubTok * wave + tg));
    };
    auto dma_offv = [&](int k) { return u16_field(dma_pk[k / 2], k & 1); };
    auto dma_row = [&](const void* src, const char* dst) {
      if constexpr (NT) {
        dma16_opaque_nt(src, dst);
      } else {
        dma16_opaque(src, dst);
      }
    };

    // Slot indices of this wave's 8 tokens of tiles 8q .. 8q + 7 (lane 8j + i: tile
    // 8q + j, token i), into half q & 1 of its index ring: per-token slots, or with
    // a block table the tile's page. Tokens past the part re-read its last index.
    auto load_idx = [&](int q) {
      int tok = kv_lo + kRTileTok * (8 * q + (lane >> 3)) + kRSubTok * wave + (lane & 7);
      tok = tok < kv_hi ? tok : kv_hi - 1;
      dma4_opaque(p.table ? p.table + slot0 + tok / kPage : p.kv_indices + slot0 + tok, idx + 256 * (q & 1));
    };
    // Slot of token lane % 8 of this wave's share of tile j; past the part's end
    // that of its last token (a page's rows beyond it may hold anything, and 0 x
    // NaN in PV is not 0).
    auto idx_at = [&](int j) -> int {
      if constexpr (PAGED) {
        const int v = *reinterpret_cast<const int*>(idx + 32 * (j & 15) + 4 * (lane & 7));
        const int last = kv_hi - 1 - (kv_lo + kRTileTok * j), tok = kRSubTok * wave + (lane & 7);
        return p.table ? page_slot(p, v) + (tok < last ? tok : last) : v;
      } else {
        return 0;
      }
    };

    // This wave's share of the gather of tile j (slots `v`: idx_at(j)) into ring
    // slot `slot`. Fast path: 8 consecutive slots, left pending (pend_base,
    // pend_dst) with `defer`, to go out one DMA at a time under MFMAs. Partial:
    // rows past the valid ones re-read the last valid row. Slow: row by row from
    // the slots. The indices of the batch after next take the half that tile j's
    // batch has just followed.
    const uint8_t* pend_base = nullptr;
    const char* pend_dst = nullptr;
    int pend = 0;
    auto issue_tile = [&](int j, int slot, int v, bool defer) -> bool {
      const char* dst = lds + slot * kRTileBytes + wave * kRSubBytes;
      const int tok0 = kv_lo + j * kRTileTok + kRSubTok * wave;
      const int nvalid = kv_hi - tok0;  // <= 0: every row re-reads the segment's last token
      const uint8_t* base;
      bool fast = true;
      if constexpr (PAGED) {
        if ((j & 7) == 0 && j > 0 && j + 8 < ntiles) load_idx(j / 8 + 1);
        const int s0 = __builtin_amdgcn_readfirstlane(v);
        base = p.kv + (long long)s0 * kQK;
        fast = __builtin_amdgcn_ballot_w64(tok0 + (lane & 7) < kv_hi && v != s0 + (lane & 7)) == 0;
      } else {
        base = p.kv + ((long long)b * p.S_fixed + (nvalid > 0 ? tok0 : kv_hi - 1)) * kQK;
      }
      if (fast && nvalid >= kRSubTok) {
        if (defer) {
          pend_base = base;
          pend_dst = dst;
          return true;
        }
#pragma unroll
        for (int k = 0; k < kRDma; ++k) {
          if (k < kRDma - 1 || lane < 32) dma_row(base + dma_offv(k), dst + 1024 * k);
        }
      } else if (fast) {
        const int nv = nvalid > 0 ? nvalid : 1;
#pragma unroll 1
        for (int k = 0; k < kRDma; ++k) {
          int tg, off;
          dma_place(k, tg, off);
          const int t = tg < nv ? tg : nv - 1;
          if (k < kRDma - 1 || lane < 32) dma_row(base + t * kQK + off, dst + 1024 * k);
        }
      } else {
#pragma unroll 1
        for (int k = 0; k < kRDma; ++k) {
          int tg, off;
          dma_place(k, tg, off);
          const int row = __shfl(v, tg & 7);
          if (k < kRDma - 1 || lane < 32) dma_row(p.kv + (long long)row * kQK + off, dst + 1024 * k);
        }
      }
      return false;
    };
    bool primed = false;  // tile 0 is on its way
    auto prime = [&]() {
      if constexpr (PAGED) {
        load_idx(0);
        if (ntiles > 8) load_idx(1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      issue_tile(0, 0, idx_at(0), false);
      primed = true;
    };
    if (ntiles > 0) prime();
    // The CTA's query rows, 1152 bytes each (512 latent dims, 64 rope dims), into
    // ring slots 1 and 2 by whole-row DMAs while tile 0 is on its way (fragment
    // loads straight from memory touch 32 rows each and took 2 us to issue), row
    // rr's 16-byte chunk c at rr * 1152 + 16 * (c ^ ((rr / 2) & 7)): the fragment
    // reads are conflict-free. Wave w fetches rows 8w .. 8w+7.
    char* qstage = lds + kRTileBytes;
    auto q_src = [&](int k) {
      const int pc = 64 * k + lane;
      const int rl = pc / 72, cs = pc - 72 * rl;
      const int rr = 8 * wave + rl;
      const int ch = cs ^ ((rr >> 1) & 7);
      const int row = row0 + rr < p.qrows ? row0 + rr : p.qrows - 1;
      const long long qoff = (long long)qb * p.qrows + row;
      return ch < 64 ? p.q_lat + qoff * kLat + 8 * ch : p.q_pe + qoff * kRope + 8 * (ch - 64);
    };
    if (wave < 4 * NRT) {
      if (p.q_plain) {
#pragma unroll 1
        for (int k = 0; k < 9; ++k) copy16_plain(q_src(k), qstage + 9216 * wave + 1024 * k + 16 * lane);
      } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) dma16_opaque(q_src(k), qstage + 9216 * wave + 1024 * k);
      }
    }
    lds_reads_done_barrier_vm0();
    // Q, the B operand of S^T = K Q^T: pair s of this dim half covers dims
    // 288 kh + 32 s + 16 g .. +16 of lane half g, the first 8 for k-step 2s and the
    // next 8 for k-step 2s + 1 (the K fragment holds the same dims).
    bf16x8 qf[2 * kRPairs];
    if (scores) {
      const int rr = 32 * rt + n;
#pragma unroll
      for (int s = 0; s < 2 * kRPairs; ++s) {
        const int ch = 36 * kh + 4 * (s >> 1) + 2 * g + (s & 1);
        qf[s] = *reinterpret_cast<const bf16x8*>(qstage + rr * 1152 + 16 * (ch ^ ((rr >> 1) & 7)));
      }
    } else {
#pragma unroll
      for (int s = 0; s < 2 * kRPairs; ++s) qf[s] = bf16x8{};
    }
    lds_reads_done_barrier();  // the slots are free again

    f32x16 oacc[2][NRT];  // O^T: d-tile dt, row tile; lane (n, g) register 4j + e = dim 64w + 32dt + 8j + 4g + e
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < NRT; ++r) oacc[dt][r] = f32x16{};
    float row_m = -__builtin_inff();  // CTA-wide max of this lane's row (integer grid) once fixed
    float row_l = 0.f;                // this lane's share of the row's sum
    bool m_fixed = false;
    bool grew = false;                // some later p exceeded 2^kGrowLimit
    const float c = p.score_c;

    // One pass over the part. Accumulate mode: softmax + PV with each row's max
    // fixed at the part's first tile (or before the pass). Max-only mode: QK and
    // this lane's largest masked score (row_m).
    auto sweep = [&](auto max_only_tag) {
      constexpr bool kMaxOnly = decltype(max_only_tag)::value;
      if (ntiles > 0) {
        // A second pass: every wave is done with the ring. (The first tile of the
        // first one was gathered before Q, into slot 0.)
        if (!primed) {
          lds_reads_done_barrier();
          prime();
        }
        primed = false;
        const int eff = lim < kv_hi ? lim : kv_hi;              // this row's token limit in the part
        const int eff_min = lim_min < kv_hi ? lim_min : kv_hi;  // tiles below it need no mask

        // DMA k of a pending gather, skipped inside the asm when nothing is pending
        // (no branch for the compiler to split the step sequence at). The fifth
        // moves 512 bytes: its upper lanes are switched off around it.
        auto dma_if = [&](int pending, int k) {
          const uint32_t m0v = (uint32_t)(uintptr_t)(MM_LDS const char*)(pend_dst + 1024 * k);
          const int pu = __builtin_amdgcn_readfirstlane(pending);
          if (k < kRDma - 1) {
            if constexpr (NT) {
              asm volatile("s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 1f\n\tglobal_load_lds_dwordx4 %0, %1 nt\n1:" ::"v"(
                               dma_offv(k)),
                           "s"(pend_base), "{m0}"(m0v), "s"(pu)
                           : "memory", "scc");
            } else {
              asm volatile("s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 1f\n\tglobal_load_lds_dwordx4 %0, %1\n1:" ::"v"(
                               dma_offv(k)),
                           "s"(pend_base), "{m0}"(m0v), "s"(pu)
                           : "memory", "scc");
            }
          } else {
            if constexpr (NT) {
              asm volatile(
                  "s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 1f\n\ts_mov_b32 exec_hi, 0\n\t"
                  "global_load_lds_dwordx4 %0, %1 nt\n\ts_mov_b32 exec_hi, -1\n1:" ::"v"(dma_offv(k)),
                  "s"(pend_base), "{m0}"(m0v), "s"(pu)
                  : "memory", "scc");
            } else {
              asm volatile(
                  "s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 1f\n\ts_mov_b32 exec_hi, 0\n\t"
                  "global_load_lds_dwordx4 %0, %1\n\ts_mov_b32 exec_hi, -1\n1:" ::"v"(dma_offv(k)),
                  "s"(pend_base), "{m0}"(m0v), "s"(pu)
                  : "memory", "scc");
            }
          }
        };
        auto vfrag = [&](const char* sv, int kk, int dt) {
          return __builtin_amdgcn_ds_read_tr8_b64_v2i32((MM_LDS i32x2*)(sv + (dt ? voff1 : voff0) + kk * 16 * kQK));
        };
        auto pfrag = [&](const char* pb, int kk, int r) {
          return *reinterpret_cast<const bf16x8*>(pb + (kk * NRT + r) * 1024 + lane * 16);
        };

        // One tile. Phase A: the 18 QK MFMAs of tile t with the first half (token
        // quarters 0 and 1) of tile t-1's PV MFMAs; the other half's operands are
        // read meanwhile. Phase B, after the exchange barrier: the second half of
        // PV(t-1) over this wave's softmax of 16 tokens and the DMAs of tile t+2.
        // sc: ring slot of tile t; sp: of tile t-1, which takes tile t+2.
        auto tile = [&](int t, int sc, int sp, auto with_pv) {
          constexpr bool kPV = decltype(with_pv)::value;
          const char* sk = lds + sc * kRTileBytes;
          const char* sv = lds + sp * kRTileBytes;
          const char* pb = lds + kRPOff + ((t - 1) & 1) * kRPBytes;
          const bool more = t + 2 < ntiles;
          const int idx_next = more ? idx_at(t + 2) : 0;
          f32x16 sacc = f32x16{};
          i32x2 v0[4], v1[4];            // V^T fragments 2 * (kk % 2) + dt of quarters 0..1, 2..3
          bf16x8 p0[2][NRT], p1[2][NRT];  // P^T fragments
          if constexpr (kPV) {
            v0[0] = vfrag(sv, 0, 0);
            v0[1] = vfrag(sv, 0, 1);
#pragma unroll
            for (int r = 0; r < NRT; ++r) p0[0][r] = pfrag(pb, 0, r);
          }
          // PV operand reads of step s: quarter 1 by step 2 NRT, quarters 2 and 3
          // into the registers that quarters 0 and 1 leave.
          auto pv_reads = [&](int s) {
            if (s == 0) {
              v0[2] = vfrag(sv, 1, 0);
              p0[1][0] = pfrag(pb, 1, 0);
            }
            if (s == 1) {
              v0[3] = vfrag(sv, 1, 1);
              if constexpr (NRT == 2) p0[1][NRT - 1] = pfrag(pb, 1, NRT - 1);
            }
            if (s >= 4 && s < 8) {
              const int f = s - 4;
              v1[f] = vfrag(sv, 2 + (f >> 1), f & 1);
              if (f >= 2 && f - 2 < NRT) p1[0][f - 2] = pfrag(pb, 2, f - 2);
            }
          };
          bf16x8 vw;
          auto pv = [&](int m, const i32x2 (&v)[4], const bf16x8 (&pp)[2][NRT]) {  // m = NRT * fragment + row tile
            const int f = m / NRT, r = m % NRT;
            if (r == 0) vw = fp8x8_bf16((uint32_t)v[f][0], (uint32_t)v[f][1]);
            oacc[f & 1][r] = mfma32(vw, pp[f >> 1][r], oacc[f & 1][r]);
          };
          constexpr int kAhead = 3;
          u32x4 kr[kAhead];
          auto kaddr = [&](int s) { return sk + ((s & 1) ? koff_o : koff_e) + 64 * (s >> 1); };
          if (scores) {
#pragma unroll
            for (int s = 0; s < kAhead; ++s) kr[s] = *reinterpret_cast<const u32x4*>(kaddr(s));
#pragma unroll
            for (int s = 0; s < kRPairs; ++s) {
              const u32x4 raw = kr[s % kAhead];
              if (s + kAhead < kRPairs) kr[s % kAhead] = *reinterpret_cast<const u32x4*>(kaddr(s + kAhead));
              const bf16x8 ka = fp8x8_bf16(raw[0], raw[1]);
              const bf16x8 kb = fp8x8_bf16(raw[2], raw[3]);
              sacc = mfma32(ka, qf[2 * s], sacc);
              if ((s & 1) == 0 && kRDmaB + s / 2 < kRDma) dma_if(pend, kRDmaB + s / 2);
              if constexpr (kPV) {
                if (s < 4 * NRT) pv(s, v0, p0);
                pv_reads(s);
              }
              sacc = mfma32(kb, qf[2 * s + 1], sacc);
              sched_fence();
            }
            // Registers 8..15 are the partner's tokens.
            char* xo = lds + kRXOff + (wave ^ 1) * 2048 + lane * 16;
            *reinterpret_cast<f32x4*>(xo) = f32x4{sacc[8], sacc[9], sacc[10], sacc[11]};
            *reinterpret_cast<f32x4*>(xo + 1024) = f32x4{sacc[12], sacc[13], sacc[14], sacc[15]};
          } else {
#pragma unroll
            for (int k = kRDmaB; k < kRDma; ++k) dma_if(pend, k);
          }
          if constexpr (NRT == 1 && kPV) {
            if (!scores) {
#pragma unroll
              for (int s = 0; s < 8; ++s) {
                if (s < 4 * NRT) pv(s, v0, p0);
                pv_reads(s);
              }
            }
          }
          // ---- exchange barrier: partial scores published, every read of tile
          // t-1 and its P^T done: its slot takes tile t+2 ----
          lds_reads_done_barrier();
          pend = (more && issue_tile(t + 2, sp, idx_next, true)) ? 1 : 0;
          if (scores) {
            const char* xi = lds + kRXOff + wave * 2048 + lane * 16;
            const f32x4 xa = *reinterpret_cast<const f32x4*>(xi);
            const f32x4 xb = *reinterpret_cast<const f32x4*>(xi + 1024);
            if constexpr (kPV) {
#pragma unroll
              for (int r = 0; r < NRT; ++r) p1[1][r] = pfrag(pb, 3, r);
            }
            sched_fence();
            if constexpr (kPV) {
#pragma unroll
              for (int m = 0; m < 2 * NRT; ++m) {
                pv(m, v1, p1);
                if (m < kRDmaB) dma_if(pend, m);
                sched_fence();
              }
            } else {
#pragma unroll
              for (int k = 0; k < kRDmaB; ++k) dma_if(pend, k);
            }
            // Lane (n, g), element i: token 16 * quarter + 8(i/4) + 4g + i%4 of row n.
            float s[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              s[i] = sacc[i] + xa[i];
              s[4 + i] = sacc[4 + i] + xb[i];
            }
            const int tok0 = kv_lo + t * kRTileTok;
            if (tok0 + kRTileTok > eff_min) {
              const int rel = eff - tok0 - 16 * quarter - 4 * g;
#pragma unroll
              for (int i = 0; i < 8; ++i) s[i] = (8 * (i >> 2) + (i & 3)) < rel ? s[i] : -__builtin_inff();
            }
            float bm = 0.f;
            if (kMaxOnly || !m_fixed) {
              bm = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
            }
            if constexpr (kMaxOnly) {
              row_m = fmaxf(row_m, bm);
            } else {
              if (!m_fixed) {
                // The part's first tile fixes each row's max for the whole CTA.
                bm = xor32_max(bm);
                if (g == 0) red_m[quarter * kRRows + 32 * rt + n] = bm;
                lds_reads_done_barrier();
                const float* rm = red_m + 32 * rt + n;
                const float M = fmaxf(fmaxf(rm[0], rm[kRRows]), fmaxf(rm[2 * kRRows], rm[3 * kRRows]));
                row_m = (M == -__builtin_inff()) ? M : __builtin_ceilf(M * c);
              }
              // No finite score in the first tile (nor a token, where the window ends
              // before it): a later one gives p = inf, which asks for the exact max.
              const float neg_m = (row_m == -__builtin_inff()) ? -kNegFltMax : -row_m;
              float pe[8];
              if constexpr (kPV) {
#pragma unroll
                for (int m = 0; m < 2 * NRT; ++m) {
                  pv(2 * NRT + m, v1, p1);
#pragma unroll
                  for (int e = 0; e < 4 / NRT; ++e) {
                    const int i = (4 / NRT) * m + e;
                    pe[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c, neg_m));
                  }
                  sched_fence();
                }
              } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) pe[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c, neg_m));
              }
              const float lsum = ((pe[0] + pe[1]) + (pe[2] + pe[3])) + ((pe[4] + pe[5]) + (pe[6] + pe[7]));
              row_l += lsum;
              grew = grew || lsum > kGrowSum;
              const u32x4 w = {pack2_bf16<kRTNE>(pe[0], pe[1]), pack2_bf16<kRTNE>(pe[2], pe[3]),
                               pack2_bf16<kRTNE>(pe[4], pe[5]), pack2_bf16<kRTNE>(pe[6], pe[7])};
              *reinterpret_cast<u32x4*>(lds + kRPOff + (t & 1) * kRPBytes + (quarter * NRT + rt) * 1024 + lane * 16) = w;
            }
          } else {
            if constexpr (kPV) {
#pragma unroll
              for (int r = 0; r < NRT; ++r) p1[1][r] = pfrag(pb, 3, r);
#pragma unroll
              for (int m = 0; m < 4 * NRT; ++m) pv(m, v1, p1);
            }
#pragma unroll
            for (int k = 0; k < kRDmaB; ++k) dma_if(pend, k);
            if constexpr (!kMaxOnly) {
              if (!m_fixed) lds_reads_done_barrier();
            }
          }
          if constexpr (!kMaxOnly) m_fixed = true;
          // ---- tile barrier: P^T(t) published, tile t+1 landed (only tile t+2's
          // first DMAs may be out) ----
          if (more) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kRDmaB) : "memory");
          } else {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
          }
        };

        if (ntiles > 1) issue_tile(1, 1, idx_at(1), false);
        if (ntiles > 1) {
          asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        // Tile 0 has no PV before it.
        tile(0, 0, 2, std::false_type{});
        int sc = 1, sp = 0;
        for (int t = 1; t < ntiles; ++t) {
          if constexpr (kMaxOnly) {
            tile(t, sc, sp, std::false_type{});
          } else {
            tile(t, sc, sp, std::true_type{});
          }
          sp = sc;
          sc = sc == 2 ? 0 : sc + 1;
        }
        if constexpr (!kMaxOnly) {  // PV of the last tile (in slot sp)
          const char* sv = lds + sp * kRTileBytes;
          const char* pb = lds + kRPOff + ((ntiles - 1) & 1) * kRPBytes;
#pragma unroll
          for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) {
              const i32x2 v = vfrag(sv, kk, dt);
              const bf16x8 a = fp8x8_bf16((uint32_t)v[0], (uint32_t)v[1]);
#pragma unroll
              for (int r = 0; r < NRT; ++r) oacc[dt][r] = mfma32(a, pfrag(pb, kk, r), oacc[dt][r]);
            }
        }
      }
    };

    // Each scoring wave posts its rows' l sums, each wave its fallback flag, then
    // one barrier.
    auto post_l = [&]() {
      const float l = xor32_sum(row_l);
      if (scores && g == 0) red_l[quarter * kRRows + 32 * rt + n] = l;
      const bool any = __builtin_amdgcn_ballot_w64(grew) != 0;
      if (lane == 0) misc[wave] = any;
      lds_reads_done_barrier_vm0();
    };
    auto any_grew = [&]() {
      int f = 0;
#pragma unroll
      for (int w = 0; w < kRWaves; ++w) f |= misc[w];
      return __builtin_amdgcn_readfirstlane(f) != 0;
    };
    sweep(std::false_type{});
    post_l();
    // Fallback (only when some row's scores rise more than 2^64 above the part's
    // first tile): redo the part with the exact row max. CTA-uniform: the flags
    // are read after a barrier.
    if (any_grew()) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has read the flags
      row_m = -__builtin_inff();
      sweep(std::true_type{});
      const float wm = xor32_max(row_m);
      if (scores && g == 0) red_m[quarter * kRRows + 32 * rt + n] = wm;
      lds_reads_done_barrier();
      const float* rm = red_m + 32 * rt + n;
      const float M = fmaxf(fmaxf(rm[0], rm[kRRows]), fmaxf(rm[2 * kRRows], rm[3 * kRRows]));
      row_m = (M == -__builtin_inff()) ? M : __builtin_ceilf(M * c);
      m_fixed = true;
      row_l = 0.f;
      grew = false;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < NRT; ++r) oacc[dt][r] = f32x16{};
      sweep(std::false_type{});
      post_l();
    }

    // ---- epilogue -----------------------------------------------------------------------
    // The rows go through LDS (over the ring, P and X, all idle now) so that every
    // store instruction writes whole rows: row rr's 16-byte chunk cc (4 dims) at
    // rr * 2048 + 16 * (cc ^ (rr & 31)), conflict-free both ways.
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < NRT; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int cc = 16 * wave + 8 * dt + 2 * j + g;
          *reinterpret_cast<f32x4*>(lds + (32 * r + n) * 2048 + 16 * (cc ^ n)) =
              f32x4{oacc[dt][r][4 * j], oacc[dt][r][4 * j + 1], oacc[dt][r][4 * j + 2], oacc[dt][r][4 * j + 3]};
        }
    const bool split = sg.nparts > 1;
    const size_t rec = (size_t)sg.rec0 + part;
    if (split && scores && quarter == 0 && g == 0 && qrow < p.qrows) {
      const float* rl = red_l + 32 * rt + n;
      float* pml = ws_ml(p) + (rec * p.qrows + qrow) * 2;
      pml[0] = row_m;
      pml[1] = (rl[0] + rl[kRRows]) + (rl[2 * kRRows] + rl[3 * kRRows]);
    }
    lds_reads_done_barrier();
    constexpr int kWaveRows = 32 * NRT / kRWaves;  // rows each wave stores
#pragma unroll
    for (int k = 0; k < kWaveRows; ++k) {
      const int rr = kWaveRows * wave + k;
      const int orow = row0 + rr;
      if (orow >= p.qrows) break;
      const char* src = lds + rr * 2048;
      if (split) {
        // Unnormalised fp32 O of this part.
        float* dst = ws_rec_o(p, rec) + (size_t)orow * kLat;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int cc = 64 * h + lane;
          *reinterpret_cast<f32x4*>(dst + 4 * cc) = *reinterpret_cast<const f32x4*>(src + 16 * (cc ^ (rr & 31)));
        }
      } else {
        const float L = (red_l[rr] + red_l[kRRows + rr]) + (red_l[2 * kRRows + rr] + red_l[3 * kRRows + rr]);
        const float inv = (L == 0.f) ? 0.f : p.kv_scale * __builtin_amdgcn_rcpf(L);
        const f32x4 a = *reinterpret_cast<const f32x4*>(src + 16 * ((2 * lane) ^ (rr & 31)));
        const f32x4 d = *reinterpret_cast<const f32x4*>(src + 16 * ((2 * lane + 1) ^ (rr & 31)));
        const u32x4 o = {pack2_bf16_canon<kRTNE>(a[0] * inv, a[1] * inv), pack2_bf16_canon<kRTNE>(a[2] * inv, a[3] * inv),
                         pack2_bf16_canon<kRTNE>(d[0] * inv, d[1] * inv), pack2_bf16_canon<kRTNE>(d[2] * inv, d[3] * inv)};
        *reinterpret_cast<u32x4*>(p.o_lat + ((long long)qb * p.qrows + orow) * kLat + 8 * lane) = o;
      }
    }
    if (p.parts > 1 && part == 0 && grp == 0 && tid == 0) {
      // Per-request (parts, first record) table for the merge kernel.
      int* tbl = ws_tbl(p);
      tbl[2 * b] = sg.nparts;
      tbl[2 * b + 1] = sg.rec0;
    }
    sg = next_work(p.B, sg, u, next_len, next_slot0);
    if (sg.b < 0) break;
    lds_reads_done_barrier();  // every wave is done with this part's LDS
  }
}

template <bool PAGED>
static void launch_rows64(const Params& p, dim3 grid, hipStream_t st) {
  if (p.qrows <= 32)
    hipLaunchKernelGGL((mla_rows64_kernel<PAGED, 1, true>), grid, dim3(kRThreads), 0, st, p);
  else if (p.qrows <= kRows64 && p.ngroups == 2)
    hipLaunchKernelGGL((mla_rows64_kernel<PAGED, 1, false>), grid, dim3(kRThreads), 0, st, p);
  else if (p.ngroups == 1)
    hipLaunchKernelGGL((mla_rows64_kernel<PAGED, 2, true>), grid, dim3(kRThreads), 0, st, p);
  else
    hipLaunchKernelGGL((mla_rows64_kernel<PAGED, 2, false>), grid, dim3(kRThreads), 0, st, p);
}

int launch_rows64_kernel(const Params& p, long long grid, hipStream_t st) {
  if (p.paged)
    launch_rows64<true>(p, dim3((unsigned)grid), st);
  else
    launch_rows64<false>(p, dim3((unsigned)grid), st);
  return 0;
}

}  // namespace mla
}  // namespace mm
