// Absorbed-MLA decode for MI355X (gfx950): bf16 queries against an fp8 (OCP
// e4m3fn) latent KV cache, 576-wide fused rows ([0:512] latent = K and V,
// [512:576] rope = K only) at one per-tensor kv_scale.
//
//   score[r, j] = (q_lat[r] . c[j, 0:512] + q_pe[r] . c[j, 512:576]) * scale * kv_scale
//   o_lat[r]    = sum_j softmax_j(score[r, :]) * c[j, 0:512] * kv_scale
//
// Replaces the reference's gfx942 single-q and multi-q kernels (moonmath
// reference csrc/mla_decode_a16w8.hip:183-754, csrc/mla_decode_a16w8_multiq.hip
// :282-856). A query row r is (draft position t, head h) = (r / H, r % H); draft
// position t attends tokens [0, S - (q_len - 1 - t)) (end-aligned causal window,
// reference mla_decode_a16w8.hip:213-217). Two decode kernels share the row
// format, the work split, the split records and the numerics (mla_common.hpp):
// mla_coop.hip for up to 16 query rows, mla_rows64.hip for more (64 or 32 rows
// per CTA). This file holds what surrounds them: the merge of split requests, the
// planners and the C ABI.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "mla_common.hpp"

namespace mm {
namespace mla {

// Merge of one query row over its request's parts: M = max_p m_p, w_p = 2^(m_p - M)
// (exact, m_p integer-valued), out = sum w_p O_p * kv_scale / sum w_p l_p.
__device__ __forceinline__ float part_weight(float m_p, float M) {
  const float diff = m_p - M;  // integer-valued or -inf, <= 0
  return (m_p == -__builtin_inff()) ? 0.f : ((diff >= -126.f) ? __builtin_ldexpf(1.0f, (int)diff) : 0.f);
}
__device__ __forceinline__ u32x2 merge_finish(f32x4 acc, float L, float kv_scale) {
  const float inv = (L == 0.f) ? 0.f : kv_scale * __builtin_amdgcn_rcpf(L);
  return u32x2{pack2_bf16_canon<kRTNE>(acc[0] * inv, acc[1] * inv), pack2_bf16_canon<kRTNE>(acc[2] * inv, acc[3] * inv)};
}
// Parts j0, j0 + step, ... (up to kMergeBatch of them below nparts) added to
// (acc, L) under the max M: their (m, l) pairs and O slices are loaded together,
// one round of memory latency.
constexpr int kMergeBatch = 8;
template <class OAt, class MlAt>
__device__ __forceinline__ void merge_batch(int j0, int step, int nparts, OAt o_at, MlAt ml_at, bool own_max, float& M,
                                            f32x4& acc, float& L) {
  float mb[kMergeBatch], lb[kMergeBatch];
  f32x4 ob[kMergeBatch];
#pragma unroll
  for (int k = 0; k < kMergeBatch; ++k) {
    const int j = j0 + k * step;
    mb[k] = -__builtin_inff();
    lb[k] = 0.f;
    ob[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (j < nparts) {
      const float2 m_l = *reinterpret_cast<const float2*>(ml_at(j));
      mb[k] = m_l.x;
      lb[k] = m_l.y;
      ob[k] = *reinterpret_cast<const f32x4*>(o_at(j));
    }
  }
  if (own_max) {
#pragma unroll
    for (int k = 0; k < kMergeBatch; ++k) M = fmaxf(M, mb[k]);
  }
#pragma unroll
  for (int k = 0; k < kMergeBatch; ++k) {
    if (j0 + k * step < nparts) {
      const float wt = part_weight(mb[k], M);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(wt, ob[k][e], acc[e]);
      L = __builtin_fmaf(wt, lb[k], L);
    }
  }
}

__device__ __forceinline__ int merge_out_row(const Params& p, int b) {
  int qb = b;
  if (p.rows) {
    qb = p.rows[b];
    qb = qb < 0 ? 0 : (qb >= p.B ? p.B - 1 : qb);
  }
  return qb;
}

// Merge of the split requests' records, 128 threads (4 output dims each) times
// GROUPS per query row; group g adds parts g, g + GROUPS, ... and the groups'
// sums meet in LDS, each under the max its group has seen. A thread's parts cost
// a round of memory latency per batch of 8: eight groups for many parts, as long
// as the rows are few (with many, latency is covered and the threads only cost).
// Whole calls, one -> four -> eight groups: 16 rows in 33 parts 15.1 -> 12.5 ->
// 11.6 us, 128 rows in 17 parts 16.1 with four and eight; one -> four: 1024 rows
// in 17 parts 26.9 -> 31.8, 2048 rows in 9 parts 41.1 -> 45.5, 1024 rows in 5
// parts 38.3 -> 41.6.
constexpr int kMergeWideParts = 8;
constexpr int kMergeWideRows = 256;
template <int GROUPS>
__global__ __launch_bounds__(GROUPS == 1 ? 256 : 128 * GROUPS) void mla_merge_kernel(Params p) {
  constexpr int kRowsPerCta = GROUPS == 1 ? 2 : 1;
  const int tid = threadIdx.x;
  const int cell = tid & 127;
  const int grp = GROUPS == 1 ? 0 : tid >> 7;
  const long long row = (long long)blockIdx.x * kRowsPerCta + (GROUPS == 1 ? tid >> 7 : 0);
  if (row >= (long long)p.B * p.qrows) return;  // GROUPS > 1: the grid is exact
  const int b = (int)(row / p.qrows);
  const int qrow = (int)(row % p.qrows);
  const int d = cell * 4;
  const float* ml = ws_ml(p);
  const int* tbl = ws_tbl(p);
  const int nparts = tbl[2 * b];
  const int rec0 = tbl[2 * b + 1];
  if (nparts <= 1) return;  // the decode kernel wrote this request's output
  auto o_at = [&](int j) { return ws_rec_o(p, (size_t)rec0 + j) + (size_t)qrow * kLat + d; };
  auto ml_at = [&](int j) { return ml + (((size_t)rec0 + j) * p.qrows + qrow) * 2; };
  float M = -__builtin_inff(), L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (nparts <= kMergeBatch * GROUPS) {
    merge_batch(grp, GROUPS, nparts, o_at, ml_at, true, M, acc, L);  // under the group's own max
  } else {
    // The row's max by the wave: lane l looks at parts l, l + 64, ...
    for (int j = tid & 63; j < nparts; j += 64) M = fmaxf(M, ml_at(j)[0]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) M = fmaxf(M, __shfl_xor(M, off));
    for (int j0 = grp; j0 < nparts; j0 += kMergeBatch * GROUPS)
      merge_batch(j0, GROUPS, nparts, o_at, ml_at, false, M, acc, L);
  }
  if constexpr (GROUPS > 1) {
    __shared__ f32x4 part_o[GROUPS][128];
    __shared__ float part_m[GROUPS], part_l[GROUPS];
    part_o[grp][cell] = acc;
    if (cell == 0) {
      part_m[grp] = M;
      part_l[grp] = L;
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int k = 1; k < GROUPS; ++k) M = fmaxf(M, part_m[k]);
    L = 0.f;
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < GROUPS; ++k) {
      const float wt = part_weight(part_m[k], M);
      const f32x4 o = part_o[k][cell];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(wt, o[e], acc[e]);
      L = __builtin_fmaf(wt, part_l[k], L);
    }
  }
  // Non-temporal: written once, read by no later kernel of the call (H=16:
  // 45.8 -> 44.4 us per call; the same in the decode kernels measured neutral
  // or slower).
  __builtin_nontemporal_store(merge_finish(acc, L, p.kv_scale),
                              reinterpret_cast<u32x2*>(p.o_lat + ((long long)merge_out_row(p, b) * p.qrows + qrow) * kLat + d));
}

// Test hook: decode fp8 bytes with the same hardware convert the kernel uses.
__global__ void fp8_to_bf16_kernel(const uint8_t* in, uint16_t* out, int n) {
  const int i = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  uint32_t v = 0;
  for (int k = 0; k < 4; ++k) v |= (uint32_t)(i + k < n ? in[i + k] : 0) << (8 * k);
  const uint32_t lo = fp8x2_bf16<false>(v);
  const uint32_t hi = fp8x2_bf16<true>(v);
  const uint16_t r[4] = {(uint16_t)(lo & 0xFFFF), (uint16_t)(lo >> 16), (uint16_t)(hi & 0xFFFF), (uint16_t)(hi >> 16)};
  for (int k = 0; k < 4; ++k)
    if (i + k < n) out[i + k] = r[k];
}

}  // namespace mla
}  // namespace mm

// ===========================================================================
// Host side: planners + C ABI
// ===========================================================================
namespace {
using namespace mm::mla;

constexpr int kNumCUs = 256;
constexpr int kMaxParts = 256;
constexpr int kScratchParts = 64;          // parts that the allocation-free entry's size limit counts
constexpr size_t kScratchRecords = 32768;  // record rows of the allocation-free entry's array

// Query rows of a CTA. Requests of at most 16 rows run mla_coop_kernel, larger ones
// mla_rows64_kernel in groups of 64 rows (at 32 rows and 256 requests of 2048
// tokens it is bound by HBM, 54 us; the 16-row kernel would read every token
// twice). Calls of 33..64 rows that one round of 32-row groups holds run those
// instead, two to a token read, while the batch is small: half the round's units,
// so half the records, and half of Q and O per CTA, against a second reading of
// the tokens from L2. 64 -> 32 rows, us: one request of 550 tokens 16.1 -> 13.0; 10
// of 9028 35.1 -> 29.1; 123 of 599 32.6 -> 21.4; 128 of 2048 (4096 tiles) 58.5 ->
// 49.3; 60 of 6147 (5820) 77.7 -> 74.1; over the line 32 of 7041..16338 (5850) 74.2
// -> 76.0, 65 of 7245 (7410) 90.6 -> 99.9, 216 of 1303 54.5 -> 63.6. `tokens`: of the
// whole call or a bound on them, 0 if unknown.
constexpr int kCoopMaxRows = 16;
constexpr int kRows32MaxTiles = 5120;
bool use_coop(int H, int q_len) { return H * q_len <= kCoopMaxRows; }
int cta_rows_for(int B, int H, int q_len, long long tokens) {
  if (use_coop(H, q_len)) return kCoopMaxRows;
  const bool small = tokens > 0 && tokens <= (long long)kRows32MaxTiles * kTileTok;
  return small && H * q_len > 32 && H * q_len <= kRows64 && B <= kNumCUs / 2 ? 32 : kRows64;
}
int ngroups_for(int H, int q_len, int cta_rows) { return (H * q_len + cta_rows - 1) / cta_rows; }

// O rows of one split record in the workspace: whole 32-row tiles for 96..128
// query rows (the size its callers have), otherwise the query rows.
int rec_rows_for(int H, int q_len) {
  const int qrows = H * q_len;
  return qrows >= 96 && qrows <= 128 ? 32 * ((qrows + 31) / 32) : qrows;
}

// Split workspace bytes: O records, (m, l) pairs, the per-request table.
size_t split_ws_bytes(int B, int H, int parts, int q_len) {
  return (size_t)B * parts * ((size_t)rec_rows_for(H, q_len) * kLat + (size_t)H * q_len * 2) * sizeof(float) +
         (size_t)B * 8;
}

// Largest parts the fixed record workspace allows for (B, H, q_len).
int max_parts_for(int B, int H, int q_len) {
  const long long per_part = (long long)B * rec_rows_for(H, q_len);
  long long m = per_part > 0 ? (long long)kMaxRecords / per_part : 1;
  if (m > kMaxParts) m = kMaxParts;
  return m < 1 ? 1 : (int)m;
}

// Units one round of CTAs over the CUs holds (one CTA per CU fits in LDS). A unit's
// ngroups CTAs share an XCD, so it is what one XCD's CUs hold, times the XCDs: with
// 3 groups 85 units are 33 CTAs on some XCDs, and one CTA's second round doubles
// the longest path: 32 requests of 1024..8192 tokens, 64 heads, 3 drafts 123 us with
// 85 units, 78 with 80; 12 of 5580, 128 heads, 3 drafts 100 with 42, 66 with 40.
// Per-CTA set-up dominates short CTAs, so a second round costs more than longer
// parts.
int unit_cap_for(int H, int q_len, int cta_rows) {
  const int per_xcd = kNumCUs / mm::kNumXcds / ngroups_for(H, q_len, cta_rows);
  return mm::kNumXcds * (per_xcd < 1 ? 1 : per_xcd);
}

// Tokens of the shortest part worth a CTA. One request of 4097 tokens: 16 heads
// 12.9 us with 64, 12.5 with 128, 12.9 with 192, 13.5 with 256, 17.0 with 512; 128
// heads 27.7, 20.8, 19.7, 19.7, 23.9 (64-row CTAs: more set-up and larger records).
int min_chunk_for(int H, int q_len) { return use_coop(H, q_len) ? 128 : 256; }

// Split planner: parts whose records let the balanced split fill the unit cap
// (see workers_for), within the record workspace and the allocation-free
// entry's array, or one where the tiles saved on the longest path (the batch's
// mean length taken as 0.6 of the longest) are worth less than the merge launch:
// 100 requests of 300 tokens, 16 heads: 17.7 us split, 12.9 whole.
constexpr int kMergeCostTiles = 5;
int plan_parts(int B, int H, int max_seq_len, int q_len) {
  if (B < 1) B = 1;
  if (q_len < 1) q_len = 1;
  const int units = unit_cap_for(H, q_len, cta_rows_for(B, H, q_len, 0));
  const int min_chunk = min_chunk_for(H, q_len);
  const long long tiles = (long long)max_seq_len / kTileTok + 1;
  const long long whole = tiles * ((B + units - 1) / units);
  const long long shared = tiles * B * 3 / (5LL * units);
  if (whole - (shared > min_chunk / kTileTok ? shared : min_chunk / kTileTok) < kMergeCostTiles) return 1;
  int p = 1 + (units + B - 2) / B;
  const int by_len = 1 + max_seq_len / min_chunk;
  if (p > by_len) p = by_len;
  const int cap = max_parts_for(B, H, q_len);
  if (p > cap) p = cap;
  const long long rows = (long long)B * rec_rows_for(H, q_len);
  if (p * rows > (long long)kScratchRecords) p = (int)(kScratchRecords / rows);
  return p < 1 ? 1 : p;
}

// Units of the balanced split: a full round, where its records fit (unit u's
// segment of request b is record u + b, so W units need W + B - 1 of the B *
// parts); otherwise 0, equal parts per request.
int workers_for(int B, int H, int parts, int q_len, int cta_rows) {
  const int cap = unit_cap_for(H, q_len, cta_rows);
  return parts > 1 && (long long)B * (parts - 1) + 1 >= cap ? cap : 0;
}

// Parts of a contiguous batch: every length is S, so where whole requests fill most
// of a round (more than half of its W units) they are weighed against the balanced
// split as it would run, in tiles of the longest unit. A record (a CTA's rows
// written and read back) is rows / 9 tiles of traffic, and a border every tw tiles
// of a request leaves one on both sides of it; whole requests on B of W units take
// kIdle + (1 - kIdle) B / W of a tile's time on all of them (128 units against 256:
// 1.21 of 1.56 us with 16 rows, 1.72 of 1.87 with 64). Split -> whole, us: 230
// requests of 1000 tokens, 16 heads 34.9 -> 25.8; 190 of 2000 49.3 -> 40.7; 230 of
// 2000, 32 heads 70.9 -> 52.5; 128 of 1500, 128 heads 58.1 -> 54.7; the other way
// 150 of 2000, 16 heads 39.1 -> 40.8, 80 of 3000, 128 heads 78.9 -> 82.2.
constexpr double kIdleCoop = 0.56, kIdleRows64 = 0.86;
constexpr double kSlabMergeTiles = 1.0;
int slab_parts(int B, int H, int S, int q_len) {
  const int parts = plan_parts(B, H, S, q_len);
  const int cta_rows = cta_rows_for(B, H, q_len, (long long)B * S);
  const int units = unit_cap_for(H, q_len, cta_rows);
  if (parts <= 1 || B > units || 2 * B <= units) return parts;
  const int tiles = work_tiles(S);
  const double idle = use_coop(H, q_len) ? kIdleCoop : kIdleRows64;
  const double whole = tiles * (idle + (1.0 - idle) * B / units);
  const int tw = work_share(B * (tiles + kSegCost), units);
  const double borders = (double)B * (tiles - 1) / tw;
  const double records = borders + (borders < B ? borders : B);
  const int rows = H * q_len < cta_rows ? H * q_len : cta_rows;
  return whole <= tw + records * rows / (9.0 * units) + kSlabMergeTiles ? 1 : parts;
}

int clamp_parts(int parts, int B, int H, int q_len, bool have_ws) {
  int p = parts < 1 ? 1 : parts;
  const int cap = max_parts_for(B, H, q_len);
  if (p > cap) p = cap;
  if (!have_ws) p = 1;
  return p;
}

// Tokens of `kv_bytes` fused rows, at least.
long long tokens_of(size_t kv_bytes) { return (long long)(kv_bytes / kQK); }

// Argument codes shared by every decode launcher (0 = arguments usable).
int check_launch_args(const void* q_lat, const void* q_pe, const void* kv, const void* o_lat, const void* seq_lens,
                      const void* kv_indices, const void* kv_indptr, int B, int H, int S_fixed, int q_len,
                      int lat_dim, int rope_dim, bool paged) {
  if (lat_dim != kLat || rope_dim != kRope) return -2;
  if (H < 1 || H > kMaxHeads) return -3;
  if (q_len < 1 || q_len > kMaxQLen || B < 1) return -4;
  if (paged && B > kMaxPagedB) return -4;
  if (!q_lat || !q_pe || !kv || !o_lat) return -6;
  if (paged && (!seq_lens || !kv_indices || !kv_indptr)) return -6;
  if (!paged && S_fixed < 1) return -7;
  return 0;
}

int launch(const void* q_lat, const void* q_pe, const void* kv, void* o_lat, const void* seq_lens,
           const void* rows, const void* kv_indices, const void* kv_indptr, int B, int H, int S_fixed, int parts,
           int q_len, int lat_dim, int rope_dim, float scale, float kv_scale, void* workspace, void* stream,
           bool paged, long long tokens, const void* table = nullptr, int max_blocks = 0, int num_blocks = 0) {
  const int arg_rc = check_launch_args(q_lat, q_pe, kv, o_lat, seq_lens, kv_indices, kv_indptr, B, H, S_fixed, q_len,
                                       lat_dim, rope_dim, paged);
  if (arg_rc != 0) return arg_rc;
  Params p{};
  p.q_lat = static_cast<const uint16_t*>(q_lat);
  p.q_pe = static_cast<const uint16_t*>(q_pe);
  p.kv = static_cast<const uint8_t*>(kv);
  p.o_lat = static_cast<uint16_t*>(o_lat);
  p.ws = static_cast<float*>(workspace);
  p.seq_lens = static_cast<const int*>(seq_lens);
  p.rows = static_cast<const int*>(rows);
  p.kv_indices = static_cast<const int*>(kv_indices);
  p.kv_indptr = static_cast<const int*>(kv_indptr);
  p.table = static_cast<const int*>(table);
  p.max_blocks = max_blocks;
  p.num_blocks = num_blocks;
  p.B = B;
  p.H = H;
  p.q_len = q_len;
  p.S_fixed = S_fixed;
  p.parts = clamp_parts(parts, B, H, q_len, workspace != nullptr);
  const int cta_rows = cta_rows_for(B, H, q_len, tokens);
  p.ngroups = ngroups_for(H, q_len, cta_rows);
  p.unit_cap = unit_cap_for(H, q_len, cta_rows);
  p.workers = workers_for(B, H, p.parts, q_len, cta_rows);
  p.min_chunk = min_chunk_for(H, q_len);
  p.paged = paged ? 1 : 0;
  p.qrows = H * q_len;
  p.rec_rows = rec_rows_for(H, q_len);
  p.score_c = (float)((double)scale * (double)kv_scale * 1.4426950408889634);
  p.kv_scale = kv_scale;
  p.q_plain = ((reinterpret_cast<uintptr_t>(q_lat) | reinterpret_cast<uintptr_t>(q_pe)) & 15) != 0;
  // Unit slots per XCD for the snake deal of units 0..U-1, U <= B * parts (the
  // kernel's split plan never exceeds that bound; CTAs past the real count exit).
  const long long umax = p.workers > 0 ? p.workers : (long long)B * p.parts;
  const long long slots_per_xcd = 2 * ((umax - 1) / 16) + (((umax - 1) % 16) >= 8 ? 2 : 1);
  const long long grid = (long long)mm::kNumXcds * slots_per_xcd * p.ngroups;
  if (grid > 0x7FFFFFFFLL) return -8;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (use_coop(H, q_len))
    launch_coop_kernel(p, grid, st);
  else
    launch_rows64_kernel(p, grid, st);
  if (p.parts > 1) {
    const long long rows_all = (long long)B * p.qrows;
    if (p.parts > kMergeWideParts && rows_all <= kMergeWideRows)
      hipLaunchKernelGGL(mla_merge_kernel<8>, dim3((unsigned)rows_all), dim3(1024), 0, st, p);
    else
      hipLaunchKernelGGL(mla_merge_kernel<1>, dim3((unsigned)((rows_all + 1) / 2)), dim3(256), 0, st, p);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

// ---------------------------------------------------------------------------
// Allocation-free launches: the split records and merge table of one launch
// live in a file-scope device array (64.3 MiB, zero-filled at load, held on
// every GPU the library runs on until the process ends). Its device address
// is looked up once per device with hipGetSymbolAddress and kept; host code
// never hands the array's name itself to a kernel (on the host that name is a
// stand-in, not a device address). The decode writes every record and table
// entry the merge reads, so nothing needs clearing between calls; calls that
// overlap on one GPU share the array and race.
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = kScratchRecords * (kLat + 2) * sizeof(float) + (size_t)kMaxPagedB * 8;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (0 or a HIP error code).
int scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return -10;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!ptr) return -10;
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return 0;
}

}  // namespace

extern "C" {

// Records (O [512] + (m, l) per query row and part) plus an 8-byte
// (parts, first record) entry per request.
size_t mla_decode_a16w8_workspace_bytes(void) { return kMaxRecords * (kLat + 2) * sizeof(float) + kMaxRecords * 8; }

size_t mla_decode_a16w8_multiq_workspace_for(int B, int H, int parts, int q_len) {
  if (B < 1 || H < 1 || q_len < 1) return 0;
  return split_ws_bytes(B, H, clamp_parts(parts, B, H, q_len, true), q_len);
}

int launch_mla_decode_a16w8(const void* q_lat, const void* q_pe, const void* c_kv, const void* k_pe, void* o_lat,
                            int B, int H, int S, int lat_dim, int rope_dim, float scale, float kv_scale,
                            float scale_p, void* workspace, void* stream) {
  (void)k_pe;
  (void)scale_p;
  const int parts = workspace ? slab_parts(B, H, S, 1) : 1;
  return launch(q_lat, q_pe, c_kv, o_lat, nullptr, nullptr, nullptr, nullptr, B, H, S, parts, 1, lat_dim, rope_dim,
                scale, kv_scale, workspace, stream, false, (long long)B * S);
}

int launch_mla_decode_a16w8_paged_dev(const void* q_lat, const void* q_pe, const void* kv_pool, void* o_lat,
                                      const void* seq_lens, const void* rows, const void* kv_indices,
                                      const void* kv_indptr, int B, int H, int parts, int lat_dim, int rope_dim,
                                      float scale, float kv_scale, float scale_p, void* workspace, void* stream,
                                      size_t kv_bytes, int q_len) {
  (void)scale_p;
  return launch(q_lat, q_pe, kv_pool, o_lat, seq_lens, rows, kv_indices, kv_indptr, B, H, 0, parts, q_len, lat_dim,
                rope_dim, scale, kv_scale, workspace, stream, true, tokens_of(kv_bytes));
}

int launch_mla_decode_a16w8_paged_dev_noalloc(const void* q_lat, const void* q_pe, const void* kv_pool, void* o_lat,
                                              const void* seq_lens, const void* rows, const void* kv_indices,
                                              const void* kv_indptr, int B, int H, int parts, int lat_dim,
                                              int rope_dim, float scale, float kv_scale, float scale_p, void* stream,
                                              size_t kv_bytes, int q_len) {
  (void)scale_p;
  // The workspace launcher's argument codes first, then the scratch limit.
  const int arg_rc = check_launch_args(q_lat, q_pe, kv_pool, o_lat, seq_lens, kv_indices, kv_indptr, B, H, 0, q_len,
                                       lat_dim, rope_dim, true);
  if (arg_rc != 0) return arg_rc;
  int eff = clamp_parts(parts, B, H, q_len, true);
  void* ws = nullptr;
  if (eff > 1) {
    // The limit is on up to 64 parts; more of them share what fits.
    const size_t rows_b = (size_t)B * rec_rows_for(H, q_len);
    if (rows_b * (eff < kScratchParts ? eff : kScratchParts) > kScratchRecords) return -9;
    if (rows_b * eff > kScratchRecords) eff = (int)(kScratchRecords / rows_b);
    const int rc = scratch_ptr(&ws);
    if (rc != 0) return rc;
  }
  return launch(q_lat, q_pe, kv_pool, o_lat, seq_lens, rows, kv_indices, kv_indptr, B, H, 0, eff, q_len, lat_dim,
                rope_dim, scale, kv_scale, ws, stream, true, tokens_of(kv_bytes));
}

size_t mla_decode_a16w8_blocks_index_bytes(int B, int max_blocks) {
  if (B < 1 || max_blocks < 1) return 0;
  return ((size_t)B * max_blocks * 64 + 2 * (size_t)B + 1) * sizeof(int);
}

int launch_mla_decode_a16w8_paged_blocks_dev(const void* q_lat, const void* q_pe, const void* kv_pool, void* o_lat,
                                             const void* seq_lens, const void* rows, const void* block_table,
                                             int max_blocks, int num_blocks, int B, int H, int parts, int q_len,
                                             int lat_dim, int rope_dim, float scale, float kv_scale, float scale_p,
                                             void* workspace, void* index_workspace, void* stream) {
  (void)scale_p;
  if (!seq_lens || !block_table || !index_workspace) return -6;
  if (B < 1 || B > kMaxPagedB) return -4;
  if (max_blocks < 1 || num_blocks < 1) return -11;
  const long long words = (long long)B * max_blocks * 64 + 2LL * B + 1;
  if (words > 0x7FFFFFFFLL || (long long)num_blocks * 64 > 0x7FFFFFFFLL) return -11;
  // The kernels read the table themselves (a page is a tile): no per-token slots
  // are written, and the index workspace, sized for them, stays untouched.
  return launch(q_lat, q_pe, kv_pool, o_lat, seq_lens, rows, block_table, block_table, B, H, 0, parts, q_len, lat_dim,
                rope_dim, scale, kv_scale, workspace, stream, true, (long long)B * max_blocks * kPage, block_table,
                max_blocks, num_blocks);
}

int launch_mla_decode_a16w8_multiq(const void* q_lat, const void* q_pe, const void* kv, void* o_lat, int B, int H,
                                   int S, int q_len, int lat_dim, int rope_dim, float scale, float kv_scale,
                                   void* workspace, void* stream) {
  const int parts = workspace ? slab_parts(B, H, S, q_len) : 1;
  return launch(q_lat, q_pe, kv, o_lat, nullptr, nullptr, nullptr, nullptr, B, H, S, parts, q_len, lat_dim,
                rope_dim, scale, kv_scale, workspace, stream, false, (long long)B * S);
}

int launch_mla_decode_a16w8_multiq_paged_dev(const void* q_lat, const void* q_pe, const void* kv_pool, void* o_lat,
                                             const void* seq_lens, const void* rows, const void* kv_indices,
                                             const void* kv_indptr, int B, int H, int parts, int q_len,
                                             int lat_dim, int rope_dim, float scale, float kv_scale,
                                             void* workspace, void* stream, size_t kv_bytes) {
  return launch(q_lat, q_pe, kv_pool, o_lat, seq_lens, rows, kv_indices, kv_indptr, B, H, 0, parts, q_len, lat_dim,
                rope_dim, scale, kv_scale, workspace, stream, true, tokens_of(kv_bytes));
}

int mla_decode_a16w8_plan_parts(int B, int H, int max_seq_len, int lat_dim) {
  (void)lat_dim;
  return plan_parts(B, H, max_seq_len, 1);
}

int mla_decode_a16w8_plan_parts_q(int B, int max_seq_len, int q_len, int H) {
  if (q_len > kMaxQLen) return -4;
  return plan_parts(B, H, max_seq_len, q_len < 1 ? 1 : q_len);
}

int mla_decode_a16w8_plan_parts_capped(int B, int H, int max_seq_len, int lat_dim) {
  (void)lat_dim;
  return plan_parts(B, H, max_seq_len, 1);
}

int mla_decode_a16w8_multiq_plan_parts_q(int B, int max_seq_len, int q_len, int H) {
  if (q_len > kMaxQLen) return -4;
  return plan_parts(B, H, max_seq_len, q_len < 1 ? 1 : q_len);
}

int mla_decode_a16w8_max_ctas(void) { return (int)(kMaxRecords / 32); }

int moonmath_mla_effective_parts(int B, int H, int parts, int q_len, int have_workspace) {
  if (B < 1 || H < 1 || q_len < 1) return 1;
  return clamp_parts(parts, B, H, q_len, have_workspace != 0);
}

int moonmath_mla_slab_parts(int B, int H, int S, int q_len) {
  if (q_len > kMaxQLen) return -4;
  return slab_parts(B, H, S, q_len < 1 ? 1 : q_len);
}

int moonmath_mla_split(int B, const int* lens, int H, int q_len, int parts, long long tokens, int* segments,
                       int max_segments) {
  if (B < 1 || H < 1 || q_len < 1 || !lens || !segments) return -6;
  const int workers =
      workers_for(B, H, clamp_parts(parts, B, H, q_len, true), q_len, cta_rows_for(B, H, q_len, tokens));
  if (workers == 0) return 0;
  int total = 0, count = 0;
  for (int b = 0; b < B; ++b) total += work_tiles(lens[b]) + kSegCost;
  const int tw = work_share(total, workers);
  int b0 = 0, end = work_tiles(lens[0]) + kSegCost;  // the first request that ends past the unit's places
  for (int u = 0; u < workers; ++u) {
    while (end <= u * tw && ++b0 < B) end += work_tiles(lens[b0]) + kSegCost;
    if (b0 == B) break;
    Seg s = work_seg(u, tw, b0, end - work_tiles(lens[b0]), lens[b0], 0);
    for (; s.b >= 0; ++count) {
      if (count < max_segments) {
        const int v[7] = {u, s.b, s.part, s.nparts, s.rec0 + s.part, s.kv_lo, s.kv_hi};
        for (int i = 0; i < 7; ++i) segments[7 * (size_t)count + i] = v[i];
      }
      s = next_work(B, s, u, s.b + 1 < B ? lens[s.b + 1] : 0, 0);
    }
  }
  return count;
}

int moonmath_fp8e4m3_to_bf16(const void* in, void* out, int n, void* stream) {
  if (!in || !out || n < 0) return -6;
  if (n == 0) return 0;
  const int threads = 256;
  const int blocks = ((n + 3) / 4 + threads - 1) / threads;
  hipLaunchKernelGGL(fp8_to_bf16_kernel, dim3(blocks), dim3(threads), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint8_t*>(in), static_cast<uint16_t*>(out), n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

}  // extern "C"
