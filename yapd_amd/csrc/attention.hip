// (a) Paged-KV block attention for the block-diffusion step.
//
// Every query of a row's current block attends to all kv_len = cache_start +
// bl keys of that row: the committed prefix plus the whole block,
// bidirectionally (engines/flashinfer.py:884-886 plans causal=False;
// engines/torch_sdpa.py:299-307 uses a zero mask).  The block's own K/V are
// already in the pool (written by the QKV epilogue or yapd_kv_write).
//
// Work decomposition (attn_paged_kernel; few rows: attn_ring_kernel): a workgroup of four waves serves one (row, key range)
// work item for four heads, one head per wave, so a workgroup streams
// 4 heads x (2 KiB K + 2 KiB V) contiguous bytes per page.  The H / 4
// workgroups of one item are consecutive in the 1-D grid: they are dispatched
// together and read the neighbouring 8 KiB runs of the same pages at about
// the same time (measured 170 -> 164 us per layer at 512 rows x 32 against a
// 2-D grid whose head groups of one item were a whole grid row apart).  Per 32-key chunk a
// wave computes S^T = K Q^T (v_mfma_f32_16x16x32_bf16, M = keys, N = 16
// queries) and O^T += V^T P^T (M = head dim, N = queries): with the
// transposed products every lane owns one query, so the online-softmax
// statistics and the O^T accumulator need no lane shuffles except the
// 4-lane-group row max/sum.  Key rows inside the S^T tiles are permuted so
// that a lane's P^T operand covers 8 consecutive keys, which are 8 consecutive
// bf16 of one V^T row in the pool (kv_layout.h).
//
// Long rows may be split over several work items (split-KV); their partial
// (O, max, sum) go to a workspace and a merge kernel combines them.  The host
// planner orders work items longest first.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

#include "attention.h"
#include "common.h"
#include "kv_layout.h"
#include "lds_dma.h"

namespace yapd {
namespace {

constexpr int kWaves = 4;
constexpr int kChunk = 32;  // keys per inner step (two pages)

struct AttnParams {
  const uint16_t* q;     // [rows, bl, H, 64]
  const uint16_t* pool;  // [n_pages, 2, H, 1024]
  int64_t n_pages;
  const int32_t* table;
  int table_stride, table_cols;
  const int32_t* kv_len;
  int rows, bl, H;
  const int32_t* work;  // [n_work][4]: row, key_begin, key_end, slot (-1: final output)
  const int32_t* counts;  // optional device {n_work, n_merge}: grids sized by upper bounds (graph replay)
  float* part_o;        // [slots, bl, H, 64]
  float* part_ml;       // [slots, bl, H, 2]
  int n_slots;          // partials exist for slots [0, n_slots); an item naming another slot writes nothing
  float scale_log2;     // softmax scale * log2(e)
  int causal;           // 1: query i of the block sees keys < kv_len - n_q(row) + i + 1 (prefix prefill)
  uint16_t* out;        // [rows, bl, H, 64] (packed: [n_q, H, 64])
  // Packed queries (NULL: row r's bl queries are rows r*bl ..): row r's queries
  // are q / out rows [q_start[r], q_start[r+1]) of n_q, at most bl of them.
  const int32_t* q_start;
  int n_q;
};

// First query row of row r in q / out and its query count.
__device__ __forceinline__ int2 row_queries(const int32_t* q_start, int n_q, int r, int bl) {
  if (q_start == nullptr) return make_int2(r * bl, bl);
  const int qs = min(max(q_start[r], 0), n_q);
  return make_int2(qs, min(max(q_start[r + 1] - qs, 0), min(bl, n_q - qs)));
}

__device__ __forceinline__ u32x4_t load16(const uint16_t* p) {
  return *reinterpret_cast<const u32x4_t*>(p);
}

// K/V pages are streamed once per step: non-temporal loads keep them from
// evicting the q / K / V lines the QKV GEMM has just written, whose
// write-back would otherwise land in the middle of this stream (measured
// 195 -> 179 us per layer right after the QKV GEMM).
__device__ __forceinline__ u32x4_t load16_stream(const uint16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
}

// Lane l combined with lane l ^ 16 (l ^ 32): v_permlane16_swap (32_swap) of a
// value with itself returns the two halves of every exchanged pair, so the
// max or sum of its two results is the pair's in both lanes -- a VALU
// exchange instead of an LDS permute.
__device__ __forceinline__ float2 swap16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float2 swap32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor16_32(float v) {
  const float2 a = swap16(v);
  const float2 b = swap32(fmaxf(a.x, a.y));
  return fmaxf(b.x, b.y);
}
__device__ __forceinline__ float sum_xor16_32(float v) {
  const float2 a = swap16(v);
  const float2 b = swap32(a.x + a.y);
  return b.x + b.y;
}

// One 32-key chunk of a 16-query tile: S^T = K Q^T, the online-softmax step, O^T += V^T P^T.  A lane
// serves query n = lane & 15 with keys k0 + 8g .. + 7; with mask, keys from klim on are left out.
__device__ __forceinline__ void attn_chunk(const bf16x8_t (&qf)[2], const u32x4_t (&kf)[2][2], const u32x4_t (&vf)[4],
                                           float scale_log2, bool mask, int key0, int klim, float& m, float& l,
                                           f32x4_t (&o)[4]) {
  f32x4_t s[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[t][0]), qf[0], f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
  for (int t = 0; t < 2; ++t)
    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[t][1]), qf[1], s[t], 0, 0, 0);
  // s[t][j] = S[q = n][key 8g + 4t + j]
  float sv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) sv[i] = s[i >> 2][i & 3] * scale_log2;
  if (mask) {  // uniform
#pragma unroll
    for (int i = 0; i < 8; ++i) sv[i] = key0 + i >= klim ? -INFINITY : sv[i];
  }
  float cm = sv[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) cm = fmaxf(cm, sv[i]);
  cm = max_xor16_32(cm);
  const float mn = fmaxf(m, cm);
  // A query that has seen no key yet (every score so far -inf: a split
  // item past the query's causal limit, or a plan longer than the device
  // kv_len) keeps m = -inf; exponents taken against 0 then give alpha = 0
  // and p = 0 instead of exp2(-inf - -inf) = NaN, so its l and O stay 0.
  const float mref = mn == -INFINITY ? 0.f : mn;
  const float alpha = __builtin_amdgcn_exp2f(m - mref);
  float p[8];
  float ps = 0.f;  // in key order
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    p[i] = __builtin_amdgcn_exp2f(sv[i] - mref);
    ps += p[i];
  }
  l = l * alpha + ps;
  m = mn;
  u32x4_t pw;
#pragma unroll
  for (int w = 0; w < 4; ++w) pw[w] = pack_bf16x2(p[2 * w], p[2 * w + 1]);
  const bf16x8_t pf = as_bf16x8(pw);
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    o[mt] *= alpha;
    o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vf[mt]), pf, o[mt], 0, 0, 0);
  }
}

// Keys past kv_len contribute P = 0; clear their V too (a lane's keys key0 .. key0 + 7) so stale or
// uninitialised pool memory can never turn 0 * V into NaN.
__device__ __forceinline__ void clear_tail(u32x4_t (&vf)[4], int key0, int kvl) {
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int key = key0 + 2 * w;
      uint32_t x = vf[mt][w];
      if (key >= kvl) x &= 0xffff0000u;
      if (key + 1 >= kvl) x &= 0x0000ffffu;
      vf[mt][w] = x;
    }
  }
}

// Q^T fragments (B operand) of tile qt: lane holds Q[q = qt*16 + n][hd = ks*32 + 8g .. +7].
__device__ __forceinline__ void load_q(const AttnParams& P, int qs, int qc, int qt, int h, int g, int n,
                                       bf16x8_t (&qf)[2]) {
  const int q = qt * 16 + n;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    u32x4_t v = {0u, 0u, 0u, 0u};
    if (q < qc) v = load16(P.q + ((static_cast<int64_t>(qs) + q) * P.H + h) * kHeadDim + ks * 32 + 8 * g);
    qf[ks] = as_bf16x8(v);
  }
}

// o[mt][j] = O^T[hd = 16mt + 4g + j][q = qt*16 + n] to the output or, for a split item, to its slot.
__device__ __forceinline__ void store_tile(const AttnParams& P, int qs, int qc, int qt, int h, int g, int n, int slot,
                                           float m, float l, const f32x4_t (&o)[4]) {
  const float L = sum_xor16_32(l);
  const int q = qt * 16 + n;
  if (q >= qc) return;
  const int64_t row_q = (static_cast<int64_t>(qs) + q) * P.H + h;
  if (slot < 0) {
    // L = 0 only for a query that sees no key at all (an empty row): zeros, not NaN
    const float inv = L > 0.f ? 1.f / L : 0.f;
    uint16_t* op = P.out + row_q * kHeadDim + 4 * g;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      u32x2_t w2;
      w2[0] = pack_bf16x2(o[mt][0] * inv, o[mt][1] * inv);
      w2[1] = pack_bf16x2(o[mt][2] * inv, o[mt][3] * inv);
      *reinterpret_cast<u32x2_t*>(op + 16 * mt) = w2;
    }
  } else if (slot < P.n_slots) {
    const int64_t prow = (static_cast<int64_t>(slot) * P.bl + q) * P.H + h;
    float* pp = P.part_o + prow * kHeadDim + 4 * g;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) *reinterpret_cast<f32x4_t*>(pp + 16 * mt) = o[mt];
    if (g == 0) {
      P.part_ml[prow * 2] = m;
      P.part_ml[prow * 2 + 1] = L;
    }
  }
}

// The row's page ids, 64 at a time: lane i holds the page of table column
// base + i (clamped), and a chunk picks its two with readlane, so the
// K/V loads never wait on a page-table load inside the loop.
struct PageRow {
  const int32_t* tab;
  int last_page, max_page, lane, base, v;
  __device__ __forceinline__ PageRow(const AttnParams& P, int r, int kvl, int kb, int lane_)
      : tab(P.table + static_cast<int64_t>(r) * P.table_stride),
        // reads stay inside the row even if kv_len exceeds what the table maps or is 0 (an empty row's page
        // is masked or never fetched)
        last_page(max(min((kvl + kPageSize - 1) / kPageSize, P.table_cols) - 1, 0)),
        max_page(static_cast<int>(min(P.n_pages - 1, int64_t{0x7fffffff}))), lane(lane_) {
    load(min(kb / kPageSize, last_page));
  }
  __device__ __forceinline__ void load(int b) {
    base = b;
    v = tab[min(base + lane, last_page)];
    asm volatile("" ::"v"(v));  // complete here: later uses wait on no load
  }
  __device__ __forceinline__ int operator()(int pi) {
    pi = min(pi, last_page);
    if (pi - base >= 64) load(pi);  // uniform: pi is the same for the wave
    return min(max(__builtin_amdgcn_readlane(v, pi - base), 0), max_page);  // a bad table entry cannot fault
  }
};

// Registers, measured: three and four tiles (blocks of 33-64 queries, the 64-token
// prefill chunks) are held to two waves per SIMD -- without the bound the compiler
// takes 222 VGPRs + 64 AGPRs for four tiles, one wave per SIMD (prefill 294 -> 280
// ms).  One and two tiles are left at the compiler's choice: with the bound and two
// chunks a turn a wave needs fewer instructions, but its page streams come faster
// than HBM serves them in order (512 rows x 32: 149 -> 157 us).
template <int NQT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(NQT >= 3 ? 2 : 1))) void
attn_paged_kernel(const AttnParams P) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int hgroups = P.H / kWaves;
  const int item = static_cast<int>(blockIdx.x) / hgroups;
  const int h = (static_cast<int>(blockIdx.x) - item * hgroups) * kWaves + wave;
  if (P.counts != nullptr && item >= P.counts[0]) return;
  const int4 it = reinterpret_cast<const int4*>(P.work)[item];
  const int r = it.x, kb = it.y, ke = it.z, slot = it.w;
  const int kvl = P.kv_len[r];
  const int g = lane >> 4;   // lane group: key group / head-dim group
  const int n = lane & 15;   // query within a 16-query tile / row within an M tile
  const int H = P.H, bl = P.bl;
  const int2 rq = row_queries(P.q_start, P.n_q, r, bl);
  const int qs = rq.x, qc = rq.y;  // the row's first query row and query count

  bf16x8_t qf[NQT][2];
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) load_q(P, qs, qc, qt, h, g, n, qf[qt]);

  f32x4_t o[NQT][4];
  float m[NQT], l[NQT];
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) {
    m[qt] = -INFINITY;
    l[qt] = 0.f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) o[qt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  PageRow page_of(P, r, kvl, kb, lane);
  // Key served by row n of S^T tile t: 8*(n/4) + 4t + n%4, so that lane group g
  // ends up holding keys 8g .. 8g+7 of the chunk.
  const int key_t0 = 8 * (n >> 2) + (n & 3);

  // K fragments (A operand of S^T): tile t row n -> key key_t0 + 4t.
  // V^T fragments (A operand of O^T): row hd = 16mt + n, keys 8g .. 8g+7.
  auto load_chunk = [&](int k0, u32x4_t (&kf)[2][2], u32x4_t (&vf)[4]) {
    const int pi0 = k0 / kPageSize;
    const int64_t p0 = page_of(pi0), p1 = page_of(pi0 + 1);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = key_t0 + 4 * t;
      const int64_t pg = key < kPageSize ? p0 : p1;
      const uint16_t* kp = P.pool + k_offset(pg, h, H, key & (kPageSize - 1), 8 * g);
      kf[t][0] = load16_stream(kp);
      kf[t][1] = load16_stream(kp + 32);
    }
    const int64_t pg = g < 2 ? p0 : p1;
    const uint16_t* vp = P.pool + v_offset(pg, h, H, 8 * (g & 1), n);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) vf[mt] = load16_stream(vp + 16 * mt * kPageSize);
  };

  // Chunk k0 + 32 is loaded while chunk k0 is multiplied.
  u32x4_t kf[2][2], vf[4], kn[2][2], vn[4];
  if (kb < ke) load_chunk(kb, kf, vf);
  // The first chunk (and q) complete here, before the loop: with a load still
  // pending on entry the compiler's wait at the loop's first MFMA is vmcnt(0),
  // which would also wait for the next chunk's loads issued just before it.
#pragma unroll
  for (int t = 0; t < 2; ++t) asm volatile("" ::"v"(kf[t][0]), "v"(kf[t][1]));
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) asm volatile("" ::"v"(vf[mt]));
  const int diag0 = kvl - qc;  // causal: query q may see keys <= diag0 + q
  for (int k0 = kb; k0 < ke; k0 += kChunk) {
    if (k0 + kChunk < ke) load_chunk(k0 + kChunk, kn, vn);
    const bool tail = k0 + kChunk > kvl;
    const bool mask_chunk = tail || (P.causal && k0 + kChunk > diag0 + 1);
    if (tail) clear_tail(vf, k0 + 8 * g, kvl);
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
      const int klim = P.causal ? min(kvl, diag0 + qt * 16 + n + 1) : kvl;
      attn_chunk(qf[qt], kf, vf, P.scale_log2, mask_chunk, k0 + 8 * g, klim, m[qt], l[qt], o[qt]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      kf[t][0] = kn[t][0];
      kf[t][1] = kn[t][1];
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) vf[mt] = vn[mt];
  }
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) store_tile(P, qs, qc, qt, h, g, n, slot, m[qt], l[qt], o[qt]);
}

// Wait until at most `later` (<= MAX) chunks of 8 loads are in flight, then the workgroup barrier.
template <int MAX>
__device__ __forceinline__ void ring_wait(int later) {
  if constexpr (MAX > 0) {
    if (later < MAX) {
      ring_wait<MAX - 1>(later);
      return;
    }
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(MAX * 8) : "memory");
}

// Few rows: a workgroup serves one head of an item, one wave per 16-query tile,
// and one more wave brings the K/V chunks into an LDS ring (8 KB each) by direct
// loads, so a row's chunks do not wait a memory latency each and the tiles of a
// block run side by side.  What bounds it is one wave's issue of a chunk's ~150
// instructions; with the loads among them, on the same wave, ~200: 2 rows x 32
// queries 10.0 us against 8.6, 8 rows x 16 on 64-2048 keys 21.3 against 17.6.
// Every query takes its keys in the order and with the operations of
// attn_paged_kernel: its result does not depend on which kernel runs it.
// (Splitting a head's keys over eight waves that merge in LDS measured 8.7 us
// against 8.6 at 2 rows x 32 queries, and its sums depend on the split.)
//
// LDS: K rows of 128 bytes, 16-byte chunk c of key k in slot c ^ (2 (k / 8) + (k / 2 & 1)); V^T pages of
// 64 x 32 bytes, the halves swapped where hd & 8: the 16 lanes of a fragment read fill 16 distinct slots.
constexpr int kRing = 3;  // chunks; 4 and 8 measured the same for few rows, slower for many (fewer workgroups per CU)
constexpr int kRingStage = 2 * kChunk * kHeadDim * 2;

template <int NQT>
__global__ __launch_bounds__(64 * (NQT + 1)) __attribute__((amdgpu_waves_per_eu(2))) void  // 2: MFMAs on VGPRs
attn_ring_kernel(const AttnParams P) {
  constexpr int NS = kRing, kStage = kRingStage;
  extern __shared__ __attribute__((aligned(16))) char ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int item = static_cast<int>(blockIdx.x) / P.H;
  const int h = static_cast<int>(blockIdx.x) - item * P.H;
  if (P.counts != nullptr && item >= P.counts[0]) return;
  const int4 it = reinterpret_cast<const int4*>(P.work)[item];
  const int r = it.x, kb = it.y, ke = it.z, slot = it.w;
  const int kvl = P.kv_len[r];
  const int g = lane >> 4, n = lane & 15;
  const int2 rq = row_queries(P.q_start, P.n_q, r, P.bl);
  const int qs = rq.x, qc = rq.y;
  const int n_ch = (ke - kb + kChunk - 1) / kChunk;

  if (wave == NQT) {
    // load j of a chunk (j = 0 .. 3: K keys 8j .. 8j+7; 4 .. 7: half of a V^T page), 1 KB each
    PageRow page_of(P, r, kvl, kb, lane);
    uint32_t ofs[5];  // K rows j, then V^T
#pragma unroll
    for (int j = 0; j < 4; ++j) ofs[j] = (lane >> 3) * 128 + 16 * ((lane & 7) ^ (2 * j + (lane >> 4 & 1)));
    ofs[4] = (lane >> 1) * 32 + 16 * ((lane & 1) ^ (lane >> 4 & 1));
    const uint32_t k_plane = static_cast<uint32_t>(kv_plane_offset(0, 0, h, P.H) * 2);
    const uint32_t v_plane = static_cast<uint32_t>(kv_plane_offset(0, 1, h, P.H) * 2);
    auto issue = [&](int c, int st) {
      const int pi = (kb + c * kChunk) / kPageSize;
      const __amdgpu_buffer_rsrc_t r0 = buffer_from(P.pool + kv_plane_offset(page_of(pi), 0, 0, P.H));
      const __amdgpu_buffer_rsrc_t r1 = buffer_from(P.pool + kv_plane_offset(page_of(pi + 1), 0, 0, P.H));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        load_lds16<true>((j & 2) ? r1 : r0, ofs[j < 4 ? j : 4], (j < 4 ? k_plane : v_plane) + (j & 1) * 1024,
                         ring + st * kStage + j * 1024);
    };
    for (int c = 0; c < NS && c < n_ch; ++c) issue(c, c);
    if (n_ch > 0) ring_wait<NS - 1>(min(NS - 1, n_ch - 1));
    int st = 0;
    for (int c = 0; c + 1 < n_ch; ++c) {
      // chunk c + 1 has landed and every wave has read chunk c: its slot takes chunk c + NS
      ring_wait<NS - 2>(min(NS - 2, n_ch - 2 - c));
      if (c + NS < n_ch) issue(c + NS, st);
      st = st + 1 == NS ? 0 : st + 1;
    }
    return;
  }
  bf16x8_t qf[2];
  load_q(P, qs, qc, wave, h, g, n, qf);
  // this wave's LDS reads are done; the loader's chunk has landed
  auto hand_over = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  const int key_t0 = 8 * (n >> 2) + (n & 3);
  const int k_sw = 2 * (n >> 2) + ((n >> 1) & 1);
  auto read = [&](int st, u32x4_t (&kf)[2][2], u32x4_t (&vf)[4]) {
    const char* s = ring + st * kStage;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        kf[t][ks] = *reinterpret_cast<const u32x4_t*>(s + (key_t0 + 4 * t) * 128 + ((4 * ks + g) ^ k_sw) * 16);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
      vf[mt] = *reinterpret_cast<const u32x4_t*>(s + 4096 + (g >> 1) * 2048 + (16 * mt + n) * 32 + ((g & 1) ^ (n >> 3)) * 16);
  };

  f32x4_t o[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) o[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  u32x4_t kf[2][2], vf[4], kn[2][2], vn[4];
  if (n_ch > 0) {
    hand_over();
    read(0, kf, vf);
  }
  const int diag0 = kvl - qc;  // causal: query q may see keys <= diag0 + q
  const int klim = P.causal ? min(kvl, diag0 + wave * 16 + n + 1) : kvl;
  int st = 0;
  auto step = [&](int c, bool more, u32x4_t (&kf)[2][2], u32x4_t (&vf)[4], u32x4_t (&kn)[2][2], u32x4_t (&vn)[4]) {
    const int k0 = kb + c * kChunk;
    const int nst = st + 1 == NS ? 0 : st + 1;
    if (more) {
      hand_over();
      read(nst, kn, vn);
    }
    const bool tail = k0 + kChunk > kvl;
    if (tail) clear_tail(vf, k0 + 8 * g, kvl);
    attn_chunk(qf, kf, vf, P.scale_log2, tail || (P.causal && k0 + kChunk > diag0 + 1), k0 + 8 * g, klim, m, l, o);
    st = nst;
  };
  // Two chunks a turn: the fragment sets swap without copies.  Nothing in the loop
  // is conditional: past a conditional read the compiler's waits would cover the
  // chunk just requested.
  int c = 0;
  for (; c + 2 < n_ch; c += 2) {
    step(c, true, kf, vf, kn, vn);
    step(c + 1, true, kn, vn, kf, vf);
  }
  if (c + 1 < n_ch) {
    step(c, true, kf, vf, kn, vn);
    step(c + 1, false, kn, vn, kf, vf);
  } else if (c < n_ch) {
    step(c, false, kf, vf, kn, vn);
  }
  store_tile(P, qs, qc, wave, h, g, n, slot, m, l, o);
}

struct MergeParams {
  const int32_t* merge;  // [n_merge][3]: row, first slot, n slots
  const int32_t* counts;
  const float* part_o;
  const float* part_ml;
  int bl, H;
  int n_slots;  // parts outside [0, n_slots) are skipped
  uint16_t* out;
  const int32_t* q_start;  // packed queries, as in AttnParams
  int n_q;
};

__device__ __forceinline__ void merge_one(const MergeParams& P, int3 mi, int q) {
  const int2 rq = row_queries(P.q_start, P.n_q, mi.x, P.bl);
  if (q >= rq.y) return;
  mi.y = max(mi.y, 0);
  mi.z = max(min(mi.z, P.n_slots - mi.y), 0);  // a merge record past the partials reads nothing
  for (int t = threadIdx.x; t < P.H * 16; t += blockDim.x) {
    const int h = t >> 4;
    const int d0 = (t & 15) * 4;
    float M = -INFINITY;
    for (int s = 0; s < mi.z; ++s) {
      const int64_t prow = (static_cast<int64_t>(mi.y + s) * P.bl + q) * P.H + h;
      M = fmaxf(M, P.part_ml[prow * 2]);
    }
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
    for (int s = 0; s < mi.z; ++s) {
      const int64_t prow = (static_cast<int64_t>(mi.y + s) * P.bl + q) * P.H + h;
      const float ls = P.part_ml[prow * 2 + 1];
      if (!(ls > 0.f)) continue;  // a part in which this query saw no key
      const float w = __builtin_amdgcn_exp2f(P.part_ml[prow * 2] - M);
      L += w * ls;
      acc += w * *reinterpret_cast<const f32x4_t*>(P.part_o + prow * kHeadDim + d0);
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    u32x2_t w2;
    w2[0] = pack_bf16x2(acc[0] * inv, acc[1] * inv);
    w2[1] = pack_bf16x2(acc[2] * inv, acc[3] * inv);
    *reinterpret_cast<u32x2_t*>(P.out + ((static_cast<int64_t>(rq.x) + q) * P.H + h) * kHeadDim + d0) = w2;
  }
}

// A grid-stride loop over (split row, query) pairs, at most kMergeGrid
// workgroups: with no live split row (the device count of a graph-replayed
// plan is often 0) the launch is a handful of empty workgroups rather than
// one per planned slot.  A thread owns 4 head-dim values of one head.
constexpr int kMergeGrid = 1024;

__global__ __launch_bounds__(256) void attn_merge_kernel(const MergeParams P, int n_merge) {
  const int live = P.counts != nullptr ? min(P.counts[1], n_merge) : n_merge;
  for (int it = blockIdx.x; it < live * P.bl; it += gridDim.x) {
    const int mrow = it / P.bl, q = it - mrow * P.bl;
    const int3 mi = make_int3(P.merge[mrow * 3], P.merge[mrow * 3 + 1], P.merge[mrow * 3 + 2]);
    merge_one(P, mi, q);
  }
}

struct KvWriteParams {
  const uint16_t* k;
  const uint16_t* v;
  int64_t k_tok_stride, v_tok_stride;  // elements between consecutive tokens
  uint16_t* pool;
  int64_t n_pages;
  const int32_t* table;
  int table_stride, table_cols;
  const int32_t* pos0;  // [rows] first position of the block
  int rows, bl, H;
};

// Thread per (token, head, 8 head-dim values).
__global__ __launch_bounds__(256) void kv_write_kernel(const KvWriteParams P) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(P.rows) * P.bl * P.H * 8;
  if (idx >= total) return;
  const int d0 = static_cast<int>(idx & 7) * 8;
  const int h = static_cast<int>((idx >> 3) % P.H);
  const int64_t tok = (idx >> 3) / P.H;
  const int r = static_cast<int>(tok / P.bl);
  const int pos = P.pos0[r] + static_cast<int>(tok - static_cast<int64_t>(r) * P.bl);
  const int pi = min(max(pos, 0) / kPageSize, P.table_cols - 1);
  int64_t page = P.table[static_cast<int64_t>(r) * P.table_stride + pi];
  page = min(max(page, int64_t{0}), P.n_pages - 1);
  const int s = pos & (kPageSize - 1);
  const u32x4_t kx = load16(P.k + tok * P.k_tok_stride + h * kHeadDim + d0);
  *reinterpret_cast<u32x4_t*>(P.pool + k_offset(page, h, P.H, s, d0)) = kx;
  const u32x4_t vx = load16(P.v + tok * P.v_tok_stride + h * kHeadDim + d0);
  uint16_t* vp = P.pool + v_offset(page, h, P.H, s, d0);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    vp[(2 * w) * kPageSize] = static_cast<uint16_t>(vx[w] & 0xffffu);
    vp[(2 * w + 1) * kPageSize] = static_cast<uint16_t>(vx[w] >> 16);
  }
}

struct KvGatherParams {
  const uint16_t* pool;
  int64_t n_pages;
  const int32_t* table_row;
  int table_len, kv_len, H;
  uint16_t* k_out;  // [kv_len, H, 64]
  uint16_t* v_out;
};

__global__ __launch_bounds__(256) void kv_gather_kernel(const KvGatherParams P) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(P.kv_len) * P.H * kHeadDim;
  if (idx >= total) return;
  const int d = static_cast<int>(idx % kHeadDim);
  const int h = static_cast<int>((idx / kHeadDim) % P.H);
  const int pos = static_cast<int>(idx / (kHeadDim * P.H));
  int64_t page = P.table_row[min(pos / kPageSize, P.table_len - 1)];
  page = min(max(page, int64_t{0}), P.n_pages - 1);
  const int s = pos & (kPageSize - 1);
  P.k_out[idx] = P.pool[k_offset(page, h, P.H, s, d)];
  P.v_out[idx] = P.pool[v_offset(page, h, P.H, s, d)];
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace yapd

extern "C" int yapd_attn_plan(const int32_t* kv_len, int rows, int target_items, int min_split_keys,
                              int32_t* work, int work_cap, int32_t* merge, int merge_cap, int* n_work, int* n_merge,
                              int* n_slots) {
  YAPD_REQUIRE(kv_len && work && merge && n_work && n_merge && n_slots, "attn_plan: NULL pointer");
  YAPD_REQUIRE(rows >= 1 && target_items >= 1 && min_split_keys >= yapd::kChunk,
               "attn_plan: need rows >= 1, target_items >= 1, min_split_keys >= 32");
  const int unit = yapd::kChunk;
  int64_t total_units = 0;
  for (int r = 0; r < rows; ++r) {
    YAPD_REQUIRE(kv_len[r] >= 1, "attn_plan: kv_len[%d] = %d < 1", r, kv_len[r]);
    total_units += (kv_len[r] + unit - 1) / unit;
  }
  const int64_t min_units = min_split_keys / unit;
  const int64_t per_item = std::max<int64_t>(min_units, (total_units + target_items - 1) / target_items);
  struct Item {
    int row, kb, ke, slot;
  };
  std::vector<Item> items;
  std::vector<int32_t> mrg;
  int slots = 0;
  for (int r = 0; r < rows; ++r) {
    const int units = (kv_len[r] + unit - 1) / unit;
    const int splits = static_cast<int>(std::min<int64_t>(units, (units + per_item - 1) / per_item));
    if (splits <= 1) {
      items.push_back({r, 0, kv_len[r], -1});
      continue;
    }
    const int base = units / splits, extra = units % splits;
    int u = 0;
    for (int s = 0; s < splits; ++s) {
      const int take = base + (s < extra ? 1 : 0);
      items.push_back({r, u * unit, std::min(kv_len[r], (u + take) * unit), slots + s});
      u += take;
    }
    mrg.insert(mrg.end(), {r, slots, splits});
    slots += splits;
  }
  // Longest first, so short items fill the tail of the launch.
  std::stable_sort(items.begin(), items.end(),
                   [](const Item& a, const Item& b) { return (a.ke - a.kb) > (b.ke - b.kb); });
  YAPD_REQUIRE(static_cast<int>(items.size()) <= work_cap, "attn_plan: work_cap %d < %zu", work_cap, items.size());
  YAPD_REQUIRE(static_cast<int>(mrg.size() / 3) <= merge_cap, "attn_plan: merge_cap %d < %zu", merge_cap,
               mrg.size() / 3);
  for (size_t i = 0; i < items.size(); ++i) {
    work[4 * i] = items[i].row;
    work[4 * i + 1] = items[i].kb;
    work[4 * i + 2] = items[i].ke;
    work[4 * i + 3] = items[i].slot;
  }
  std::copy(mrg.begin(), mrg.end(), merge);
  *n_work = static_cast<int>(items.size());
  *n_merge = static_cast<int>(mrg.size() / 3);
  *n_slots = slots;
  return YAPD_OK;
}

namespace yapd {
namespace {

// Workgroups of at most 320 threads that a launch of fewer than 2^32 threads holds, with room.
constexpr int64_t kRingGrid = 1 << 22;

// The ring kernel while its head-wide workgroups and their waves leave room on
// the chip: 96 rows of 16 heads, 64 with three tiles, with four, whose workgroups
// are five waves, 24 rows or 48 work items (three workgroups per CU); more rows keep
// enough page streams in flight with four heads to a workgroup.  Up to 64 rows it asks for LDS that holds it to four
// workgroups per CU, as many as unsplit rows need: on long rows six are more
// scattered page streams at once (64 rows x 16 on 2000-2048 keys 98.8 against 94.6
// us).  Measured (us per launch, paged -> ring; bit-identical): blocks of 32 on
// 182-632 keys, 2 rows 18.6 -> 8.0, 32 26.1 -> 13.5, 64 28.1 -> 21.4, 96 39.7 ->
// 30.4, on 2000-2048 keys 32 51.4 -> 51.1, 64 97.6 -> 97.1, 96 165.9 -> 150.3;
// blocks of 16 on 64-2048 keys, 64 65.6 -> 56.2, 96 87.2 -> 72.4; causal segments of
// 64 on <= 300 keys, 2 20.0 -> 7.5, 32 22.2 -> 10.3, 48 22.5 -> 15.1, blocks of 64 on
// 2000-2048 keys, 24 62.5 -> 49.2, 28 56.4 -> 62.5 (not taken).  The kernel reads K/V
// with non-temporal loads as the paged one does: without, 64 rows x 32 on 2000-2048
// keys take 115 us and 32 rows 56.  A captured launch gives the capacity of its work
// list for n_work, the same on every replay.
template <int NQT>
void launch_paged(const AttnParams& P, int n_work, hipStream_t st) {
  const int64_t row_heads = static_cast<int64_t>(P.rows) * P.H, wgs = static_cast<int64_t>(n_work) * P.H;
  if ((row_heads <= (NQT == 4 ? 384 : NQT == 3 ? 1024 : 1536) || (NQT == 4 && wgs <= 768)) && wgs <= kRingGrid) {
    const int lds = row_heads <= 1024 ? 40 * 1024 : kRing * kRingStage;
    hipLaunchKernelGGL(attn_ring_kernel<NQT>, dim3(n_work * P.H), dim3(64 * (NQT + 1)), lds, st, P);
  } else {
    hipLaunchKernelGGL(attn_paged_kernel<NQT>, dim3(n_work * (P.H / kWaves)), dim3(64 * kWaves), 0, st, P);
  }
}

}  // namespace

int attn_checks(const void* q, const void* kv_pool, int64_t n_pages, const int32_t* page_table, int table_stride,
                int table_cols, const int32_t* kv_len, int rows, int bl, int n_heads, const int32_t* work, int n_work,
                void* out) {
  YAPD_REQUIRE(q && kv_pool && page_table && kv_len && work && out, "attn: NULL pointer");
  YAPD_REQUIRE(yapd::aligned16(q) && yapd::aligned16(kv_pool) && yapd::aligned16(out) && yapd::aligned16(work),
               "attn: q, kv_pool, out and work must be 16-byte aligned");
  YAPD_REQUIRE(rows >= 1 && bl >= 1 && bl <= 64, "attn: need rows >= 1 and 1 <= bl <= 64 (got %d, %d)", rows, bl);
  YAPD_REQUIRE(n_heads >= yapd::kWaves && n_heads % yapd::kWaves == 0, "attn: n_heads must be a multiple of %d",
               yapd::kWaves);
  YAPD_REQUIRE(n_pages >= 1 && table_cols >= 1 && table_stride >= table_cols, "attn: empty pool or table");
  YAPD_REQUIRE(n_work >= 1 && n_work < (1 << 30), "attn: n_work = %d", n_work);
  return YAPD_OK;
}

int attn_launch(const void* q, const void* kv_pool, int64_t n_pages, const int32_t* page_table, int table_stride,
                int table_cols, const int32_t* kv_len, int rows, int bl, int n_heads, const int32_t* work, int n_work,
                const int32_t* merge, int n_merge, const int32_t* counts, float* part_o, float* part_ml, int n_slots,
                float scale, int causal, void* out, void* stream, const int32_t* q_start, int n_q) {
  yapd::AttnParams P;
  P.q = static_cast<const uint16_t*>(q);
  P.pool = static_cast<const uint16_t*>(kv_pool);
  P.n_pages = n_pages;
  P.table = page_table;
  P.table_stride = table_stride;
  P.table_cols = table_cols;
  P.kv_len = kv_len;
  P.rows = rows;
  P.bl = bl;
  P.H = n_heads;
  P.work = work;
  P.counts = counts;
  P.part_o = part_o;
  P.part_ml = part_ml;
  P.n_slots = (part_o != nullptr && part_ml != nullptr) ? n_slots : 0;
  P.scale_log2 = scale * 1.4426950408889634f;
  P.causal = causal != 0;
  P.out = static_cast<uint16_t*>(out);
  P.q_start = q_start;
  P.n_q = n_q;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  switch ((bl + 15) / 16) {
    case 1: yapd::launch_paged<1>(P, n_work, st); break;
    case 2: yapd::launch_paged<2>(P, n_work, st); break;
    case 3: yapd::launch_paged<3>(P, n_work, st); break;
    default: yapd::launch_paged<4>(P, n_work, st); break;
  }
  YAPD_LAUNCH_CHECK("attn_paged_kernel launch");
  if (n_merge > 0) {
    yapd::MergeParams M{merge, counts, part_o, part_ml, bl, n_heads, P.n_slots, static_cast<uint16_t*>(out), q_start,
                        n_q};
    const int64_t pairs = static_cast<int64_t>(n_merge) * bl;
    const dim3 mgrid(static_cast<unsigned>(pairs < yapd::kMergeGrid ? pairs : yapd::kMergeGrid));
    hipLaunchKernelGGL(yapd::attn_merge_kernel, mgrid, dim3(256), 0, st, M, n_merge);
    YAPD_LAUNCH_CHECK("attn_merge_kernel launch");
  }
  return YAPD_OK;
}

}  // namespace yapd

extern "C" int yapd_attn_paged_block(const void* q, const void* kv_pool, int64_t n_pages, const int32_t* page_table,
                                     int table_stride, int table_cols, const int32_t* kv_len, int rows, int bl, int n_heads,
                                     const int32_t* work, int n_work, const int32_t* merge, int n_merge,
                                     const int32_t* counts, float* part_o, float* part_ml, int n_slots,
                                     float scale, int causal, void* out, void* stream) {
  const int rc = yapd::attn_checks(q, kv_pool, n_pages, page_table, table_stride, table_cols, kv_len, rows, bl, n_heads,
                             work, n_work, out);
  if (rc != YAPD_OK) return rc;
  YAPD_REQUIRE(n_merge == 0 || (merge && part_o && part_ml && n_slots >= 1), "attn: split items need a workspace");
  YAPD_REQUIRE(n_merge == 0 || (yapd::aligned16(part_o)), "attn: part_o must be 16-byte aligned");
  return yapd::attn_launch(q, kv_pool, n_pages, page_table, table_stride, table_cols, kv_len, rows, bl, n_heads, work,
                           n_work, merge, n_merge, counts, part_o, part_ml, n_slots, scale, causal, out, stream);
}

extern "C" int yapd_kv_write(const void* k, const void* v, int64_t k_tok_stride, int64_t v_tok_stride, void* kv_pool,
                             int64_t n_pages, const int32_t* page_table, int table_stride, int table_cols,
                             const int32_t* pos0, int rows, int bl, int n_heads, void* stream) {
  YAPD_REQUIRE(k && v && kv_pool && page_table && pos0, "kv_write: NULL pointer");
  YAPD_REQUIRE(yapd::aligned16(k) && yapd::aligned16(v) && yapd::aligned16(kv_pool),
               "kv_write: k, v, kv_pool must be 16-byte aligned");
  YAPD_REQUIRE(k_tok_stride % 8 == 0 && v_tok_stride % 8 == 0, "kv_write: token strides must be multiples of 8");
  YAPD_REQUIRE(rows >= 1 && bl >= 1 && n_heads >= 1 && n_pages >= 1, "kv_write: empty shape");
  YAPD_REQUIRE(table_cols >= 1 && table_stride >= table_cols, "kv_write: bad table shape");
  const int64_t total = static_cast<int64_t>(rows) * bl * n_heads * 8;
  yapd::KvWriteParams P{static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), k_tok_stride, v_tok_stride,
                        static_cast<uint16_t*>(kv_pool), n_pages, page_table, table_stride, table_cols, pos0, rows, bl,
                        n_heads};
  hipLaunchKernelGGL(yapd::kv_write_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), P);
  YAPD_LAUNCH_CHECK("kv_write_kernel launch");
  return YAPD_OK;
}

extern "C" int yapd_kv_gather(const void* kv_pool, int64_t n_pages, const int32_t* table_row, int table_len,
                              int kv_len, int n_heads, void* k_out, void* v_out, void* stream) {
  YAPD_REQUIRE(kv_pool && table_row && k_out && v_out, "kv_gather: NULL pointer");
  YAPD_REQUIRE(kv_len >= 1 && n_heads >= 1 && n_pages >= 1 && table_len >= 1, "kv_gather: empty shape");
  const int64_t total = static_cast<int64_t>(kv_len) * n_heads * yapd::kHeadDim;
  yapd::KvGatherParams P{static_cast<const uint16_t*>(kv_pool), n_pages, table_row, table_len, kv_len, n_heads,
                         static_cast<uint16_t*>(k_out), static_cast<uint16_t*>(v_out)};
  hipLaunchKernelGGL(yapd::kv_gather_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), P);
  YAPD_LAUNCH_CHECK("kv_gather_kernel launch");
  return YAPD_OK;
}
