// Routed GQA decode for gfx950: one new query token per sequence attends its
// KV cache, either fully (causal over the whole cache) or over the last
// `window` keys -- the routing rule of the prefill path applied to its last
// row (F:145-155: query position p = len - 1 sees keys [0, p] when full and
// [p - window + 1, p] when local).  The reference has no decode path.
//
// HBM-bound: every cached key and value of the routed range is read once per
// KV head.  Split-K: the routed keys of all (sequence, KV head) pairs, pair
// after pair, form one line, and every workgroup streams an equal share of it
// with an online softmax, so that one long sequence, many short ones and any
// mix of full and local sequences load the chip evenly in a single round of
// workgroups.  Which keys are routed is known only on the device: up to
// kInlineSeqs sequences every workgroup finds its share by itself
// (plan_inline); beyond that a one-workgroup kernel writes the sequences'
// places on the line first.  A last kernel merges the fp32 partials in the
// log2 domain (LSE as V:236-241).
//
// Layout: q [B, Hq, 128], caches [B, L, Hkv, 128] bf16; out [B, Hq, 128] bf16,
// lse [B, Hq] fp32.  Group size G = Hq / Hkv <= 8.

#include <math.h>

#include <mutex>
#include <string>

#include "common.h"

namespace swattn {
namespace {

constexpr int kD = 128;
constexpr int kDecWaves = 4;         // waves per workgroup
constexpr int kMaxG = 8;
constexpr int kMaxSplitsDev = 256;   // partials per (sequence, KV head), at most
constexpr int kMinShare = 128;       // line positions per workgroup, at least (64 and 256: up to
                                     // 7 % and 10 % slower on single short caches)
constexpr uint32_t kPairPad = 192;   // a pair's start, in keys
constexpr uint32_t kLongShare = 2048;   // shares from this length on are halved
constexpr uint32_t kAlignSlack = 80;
constexpr int kInlinePer = 4;        // sequences per thread that a split workgroup plans itself
constexpr int kInlineSeqs = 256 * kInlinePer;

struct DecodeParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const int32_t* lens;
  const uint8_t* full;
  float* part_o;     // [slot][G][128] unnormalised sum of p * v, per workgroup and pair
  float* part_ml;    // [slot][G][2]   maximum (exp2 domain) and sum of p
  int32_t* list;     // sequences with keys, in order                      (plan kernel)
  uint4* plan;       // [0] {positions per workgroup, positions of the line (low, high)}; [1 + b]
                     // plan_entry of sequence b
  uint16_t* out;
  float* lse;
  int cache_len;     // L
  int batch, hq, hkv, group, window;
  uint32_t target;   // workgroups that are resident at once
  uint32_t pad;      // line positions a pair takes beside its keys (shared layout)
  float c;           // sm_scale * log2(e)
};

__device__ __forceinline__ float bf(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

// Sum over each row of 16 lanes, every lane getting the row's sum, with DPP
// moves only (no LDS round trip): swap neighbours, swap pairs, then add the
// mirror image within 8 and within 16 lanes.
__device__ __forceinline__ float row16_sum(float x) {
  constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kMirror = 0x140;
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kXor1, 0xf, 0xf, false));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kXor2, 0xf, 0xf, false));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kHalfMirror, 0xf, 0xf, false));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kMirror, 0xf, 0xf, false));
  return x;
}

// Key range of sequence b: first key and number of keys.
__device__ __forceinline__ void key_range(const DecodeParams& p, int b, int& lo, int& n) {
  const int len = min(max(p.lens[b], 0), p.cache_len);
  lo = p.full[b] ? 0 : max(len - p.window, 0);
  n = len - lo;
}

// The line's layout, chosen from the total of routed keys and the number of
// pairs that have any (both over all KV heads).  Positions are 32-bit where the
// workgroups plan for themselves, which they do for caches of fewer than 2^31
// rows (512 GiB), and 64-bit in the plan kernel; a share and a pair's keys fit 32
// bits in both (the host sees to it).
//
// * Shared: every pair takes its keys plus p.pad positions (what starting a
//   pair costs, in keys), and the line is cut into p.target equal shares,
//   twice as many when a share is long (kLongShare: two rounds then even out
//   the CUs' speeds).  B64 L4096-8192 Hq32/Hkv8 p_full 0.25: 144.5 us without
//   padding, 142.3 with 64 positions, 139.1 with 192, 139.9 with 256; B40
//   L2500-5000 Hq64/Hkv8 W512: 78.7 with 64, 72.5 with 192; all full, B64:
//   321 us with shares of 6144 keys left whole, 310 halved.
// * Aligned, for few pairs: every pair takes a whole number of shares, so that
//   no workgroup takes pieces of two pairs one after the other (about 4 us).
//   p.target shares then hold every pair if each is total / (p.target - pairs)
//   keys long; taken while that is at most kAlignSlack keys more than the
//   shared layout's, less time than the second piece's start.  One cache of
//   about 3300 keys, Hq32/Hkv8: 14.6 us, shared 18.9; B8 L2048-4096 p_full
//   0.5: 28.6 against 31.5.
//
// A share is at least kMinShare keys and at least ceil(L / 255), so that a
// pair is spread over at most 256 workgroups, rounded up to 16.
template <typename Pos>
struct Line {
  uint32_t share, aligned;
  Pos total;   // positions of the line
  __device__ __forceinline__ uint32_t length(uint32_t n, uint32_t pad) const {
    return n == 0 ? 0u : aligned ? (n + share - 1u) / share * share : n + pad;
  }
};
template <typename Pos>
__device__ __forceinline__ Line<Pos> plan_line(const DecodeParams& p, Pos keys, uint32_t pairs) {
  const uint32_t target = p.target;
  const uint32_t by_len = (static_cast<uint32_t>(p.cache_len) + kMaxSplitsDev - 2u) / (kMaxSplitsDev - 1u);
  const uint32_t least = max(by_len, static_cast<uint32_t>(kMinShare));
  Line<Pos> L;
  L.total = keys + pairs * p.pad;
  L.share = static_cast<uint32_t>((L.total + target - 1u) / target);
  L.aligned = 0u;
  if (pairs < target) {
    const Pos a = max((keys + target - pairs - 1u) / (target - pairs), static_cast<Pos>(least));
    if (a <= max(L.share, least) + kAlignSlack) {
      L.aligned = 1u;
      L.share = static_cast<uint32_t>(a);
    }
  }
  if (L.aligned == 0u && L.share >= kLongShare) L.share = (L.share + 1u) / 2u;
  L.share = (max(L.share, least) + 15u) & ~15u;
  return L;
}

// Exclusive prefix sums over the workgroup's threads of (keys, cnt), and both
// totals; one barrier.  (kUse: calls of one kernel use separate LDS words.)
template <int kWaves, int kUse, typename Pos>
__device__ __forceinline__ void scan_keys(Pos keys, uint32_t cnt, Pos& keys_before,
                                          uint32_t& cnt_before, Pos& keys_total,
                                          uint32_t& cnt_total) {
  __shared__ Pos s_keys[kWaves];
  __shared__ uint32_t s_cnt[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  Pos ik = keys;
  uint32_t ic = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const Pos uk = __shfl_up(ik, off);
    const uint32_t uc = __shfl_up(ic, off);
    ik += lane >= off ? uk : Pos{0};
    ic += lane >= off ? uc : 0u;
  }
  if (lane == 63) {
    s_keys[wave] = ik;
    s_cnt[wave] = ic;
  }
  __syncthreads();
  keys_before = ik - keys;
  cnt_before = ic - cnt;
  keys_total = Pos{0};
  cnt_total = 0u;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    keys_before += w < wave ? s_keys[w] : Pos{0};
    cnt_before += w < wave ? s_cnt[w] : 0u;
    keys_total += s_keys[w];
    cnt_total += s_cnt[w];
  }
}

// Sequence b's place on the line as the merge (and the listed plan) reads it:
// position of its first key, its keys, its rank among those with keys, positions
// per pair.  Ranks are below 65536, so the position has 48 bits.
struct SeqPlace {
  uint64_t off;
  uint32_t n, rank, len;
};
__device__ __forceinline__ uint4 plan_entry(uint64_t off, uint32_t n, uint32_t rank, uint32_t len) {
  return make_uint4(static_cast<uint32_t>(off), n, rank | static_cast<uint32_t>(off >> 32) << 16, len);
}
__device__ __forceinline__ SeqPlace seq_place(const uint4& e) {
  return SeqPlace{e.x | static_cast<uint64_t>(e.z >> 16) << 32, e.y, e.z & 0xffffu, e.w};
}

// a / b where the quotient fits 32 bits.
__device__ __forceinline__ uint32_t quotient(uint64_t a, uint32_t b) {
  return (a >> 32) == 0 ? static_cast<uint32_t>(a) / b : static_cast<uint32_t>(a / b);
}

// A sequence with keys: its index, first key, number of keys, and the
// positions each of its pairs takes on the line.
struct SeqEntry {
  int b, lo, n;
  uint32_t len;
};

// Where a split workgroup starts on the line: position `key` of pair (entry r,
// KV head kvh), and how many positions it takes.
struct SplitStart {
  uint32_t r, kvh, key, take;
};

// Start inside the sequence of rank r, from_off positions after its first; its
// pairs take len positions each.
__device__ __forceinline__ void split_start(SplitStart& st, uint32_t r, uint64_t from_off,
                                            uint32_t len) {
  st.r = r;
  st.kvh = quotient(from_off, len);
  st.key = static_cast<uint32_t>(from_off - static_cast<uint64_t>(st.kvh) * len);
}

// The start of this workgroup, found by itself: thread t holds sequences
// per*t .. per*t + per - 1 (per = ceil(batch / 256), at most kInlinePer), the
// workgroup scans their routed keys, keeps the sequences that have any in LDS
// and the one thread whose sequences hold line position blockIdx.x * share
// publishes it.  The lengths and routes are L2-resident after the first
// workgroups; against a list planned by a kernel of its own this costs about
// the same dependent latency and saves the launch (5-7 us of a 24-150 us
// call).  Workgroup 0 leaves every sequence's place on the line for the merge.
// Returns false past the end of the line.
__device__ __forceinline__ bool plan_inline(const DecodeParams& p, SeqEntry* s_ent, SplitStart& st) {
  __shared__ SplitStart s_start;
  const int tid = threadIdx.x;
  const int per = (p.batch + 255) >> 8;
  int lo[kInlinePer], n[kInlinePer];
  uint32_t keys = 0, cnt = 0;
#pragma unroll
  for (int j = 0; j < kInlinePer; ++j) {
    const int b = tid * per + j;
    lo[j] = n[j] = 0;
    if (j < per && b < p.batch) key_range(p, b, lo[j], n[j]);
    keys += n[j];
    cnt += n[j] > 0 ? 1 : 0;
  }
  uint32_t before, rank, all_keys, all_cnt;
  scan_keys<4, 0, uint32_t>(keys, cnt, before, rank, all_keys, all_cnt);
  Line<uint32_t> L = plan_line<uint32_t>(p, all_keys * p.hkv, all_cnt * p.hkv);
  before += rank * p.pad;
  if (L.aligned) {
    uint32_t len = 0, none;
#pragma unroll
    for (int j = 0; j < kInlinePer; ++j) len += L.length(n[j], 0);
    scan_keys<4, 1, uint32_t>(len, 0, before, none, L.total, none);
    L.total *= p.hkv;
  }
  const uint64_t pos64 = static_cast<uint64_t>(blockIdx.x) * L.share;
  const uint32_t pos = static_cast<uint32_t>(min(pos64, static_cast<uint64_t>(L.total)));
#pragma unroll
  for (int j = 0; j < kInlinePer; ++j) {
    const int b = tid * per + j;
    const uint32_t off = before * p.hkv, len = L.length(n[j], p.pad);
    if (blockIdx.x == 0 && j < per && b < p.batch) p.plan[1 + b] = plan_entry(off, n[j], rank, len);
    if (n[j] > 0) {
      s_ent[rank] = SeqEntry{b, lo[j], n[j], len};
      if (pos >= off && pos - off < len * p.hkv) split_start(s_start, rank, pos - off, len);
      ++rank;
    }
    before += len;
  }
  if (blockIdx.x == 0 && tid == 0) p.plan[0] = make_uint4(L.share, L.total, 0u, 0u);
  if (pos >= L.total) return false;   // uniform
  __syncthreads();
  st = s_start;
  st.take = min(L.total - pos, L.share);
  return true;
}

// The sequences' places on the line for more of them than that: one workgroup
// of 1024 threads.
constexpr int kPlanThreads = 1024;
__global__ __launch_bounds__(kPlanThreads) void decode_plan_kernel(const DecodeParams p) {
  const int tid = threadIdx.x;
  const int per = (p.batch + kPlanThreads - 1) / kPlanThreads;
  const int b0 = min(tid * per, p.batch), b1 = min(b0 + per, p.batch);
  uint64_t keys = 0;
  uint32_t cnt = 0;
  for (int b = b0; b < b1; ++b) {
    int lo, n;
    key_range(p, b, lo, n);
    keys += n;
    cnt += n > 0 ? 1 : 0;
  }
  uint64_t before, all_keys;
  uint32_t rank, all_cnt;
  scan_keys<kPlanThreads / 64, 0, uint64_t>(keys, cnt, before, rank, all_keys, all_cnt);
  Line<uint64_t> L = plan_line<uint64_t>(p, all_keys * p.hkv, all_cnt * p.hkv);
  before += static_cast<uint64_t>(rank) * p.pad;
  if (L.aligned) {   // few of the sequences hold keys
    uint64_t len = 0;
    uint32_t none;
    for (int b = b0; b < b1; ++b) {
      int lo, n;
      key_range(p, b, lo, n);
      len += L.length(n, 0);
    }
    scan_keys<kPlanThreads / 64, 1, uint64_t>(len, 0, before, none, L.total, none);
    L.total *= p.hkv;
  }
  for (int b = b0; b < b1; ++b) {
    int lo, n;
    key_range(p, b, lo, n);
    const uint32_t len = L.length(n, p.pad);
    p.plan[1 + b] = plan_entry(before * p.hkv, n, rank, len);
    if (n > 0) p.list[rank++] = b;
    before += len;
  }
  if (tid == 0) p.plan[0] = make_uint4(L.share, static_cast<uint32_t>(L.total), static_cast<uint32_t>(L.total >> 32), 0u);
}

// The start of this workgroup from the plan kernel's table: a search for the
// last sequence whose line position is at or before the workgroup's (one with
// keys: the sequences after it start later, and one without keys shares its
// position with the next).  Every thread runs the same search.
__device__ __forceinline__ bool plan_listed(const DecodeParams& p, SplitStart& st) {
  const uint4 line = p.plan[0];
  const uint32_t share = line.x;
  const uint64_t total = line.y | static_cast<uint64_t>(line.z) << 32;
  const uint64_t pos = static_cast<uint64_t>(blockIdx.x) * share;
  if (pos >= total) return false;
  int lo = 0, hi = p.batch - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (seq_place(p.plan[1 + mid]).off <= pos) lo = mid; else hi = mid - 1;
  }
  const SeqPlace q = seq_place(p.plan[1 + lo]);
  split_start(st, q.rank, pos - q.off, q.len);
  st.take = static_cast<uint32_t>(min(total - pos, static_cast<uint64_t>(share)));
  return true;
}

// Streams K and V at 5.2 TB/s where sequences are long (B64 L4096-8192 all
// full, whole call 345 -> 310 us against chunks planned by a kernel of their
// own with up to three uneven rounds of workgroups); B64 p_full 0.25 152 ->
// 139 us, B24 L1500-3000 p_full 0.5 60 -> 44 us, B1 L2048-4096 22.8 -> 14.6 us.
// Short calls are bound by their dependent latencies: plan, Q and first keys,
// the combine, and the merge kernel's launch.
//
// One workgroup per share of the line; it takes its pairs one after the other,
// a piece of each.  Lane l works on the keys of key group kg = l / 16 and on
// dims 8*(l%16) .. +7: wave w takes the keys 16*i + 4*w + kg of its piece, so
// the four waves sweep the piece together, four keys per wave per step.
// Each key group keeps its own online-softmax state (running max m, sum l,
// unnormalised sum acc of p * v) for every head of the group; the max moves
// only when a score exceeds it by more than 8 in the exp2 domain, so the
// state is rarely rescaled (the prefill kernel's rule).  The groups and
// waves are combined at the end into one partial per piece, in slot
// blockIdx.x + (pair's rank): both only grow along the line, one of them at
// every step from piece to piece, so that no two pieces share a slot and a
// pair's slots are consecutive.
template <int G, bool kInline>
__global__ __launch_bounds__(256) void decode_split_kernel(const DecodeParams p) {
  __shared__ float s_m[kDecWaves][G], s_l[kDecWaves][G];
  __shared__ float s_acc[kDecWaves][G][kD];
  __shared__ SeqEntry s_ent[kInline ? kInlineSeqs : 1];
  SplitStart st;
  if constexpr (kInline) {
    if (!plan_inline(p, s_ent, st)) return;
  } else {
    if (!plan_listed(p, st)) return;
  }
  // Workgroup-uniform walk over the pieces, in scalar registers.
  auto uniform = [](uint32_t x) { return static_cast<int>(__builtin_amdgcn_readfirstlane(static_cast<int>(x))); };
  int r = uniform(st.r), kvh = uniform(st.kvh);
  uint32_t key = uniform(st.key);
  uint32_t left = uniform(st.take);   // positions of the line this workgroup still has to take
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int kg = lane >> 4, ds = lane & 15;
  const int64_t row_stride = static_cast<int64_t>(p.hkv) * kD;   // elements per cache row
  for (;;) {
    SeqEntry e;
    if constexpr (kInline) {
      e = s_ent[r];
    } else {
      e.b = p.list[r];
      key_range(p, e.b, e.lo, e.n);
      e.len = p.plan[1 + e.b].w;
    }
    const int b = uniform(e.b);
    const uint32_t n = uniform(e.n), len = uniform(e.len);
    const uint32_t took = min(left, len - key);
    left -= took;
    if (key < n) {   // else this share starts in the pair's padding
    const int64_t slot = static_cast<int64_t>(blockIdx.x) + static_cast<int64_t>(r) * p.hkv + kvh;
    // Piece [k0, k1) of the pair's keys.
    const int k0 = uniform(e.lo) + static_cast<int>(key), k1 = k0 + static_cast<int>(min(took, n - key));
    // Q rows of the group: dims 8*ds .. +7 of each head, in fp32, pre-scaled
    // by c so that a dot product is already the exp2-domain score.
    float qv[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const uint4 u = *reinterpret_cast<const uint4*>(
          p.q + (static_cast<int64_t>(b) * p.hq + kvh * G + h) * kD + 8 * ds);
      const uint32_t x[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        qv[h][2 * i] = bf(x[i] & 0xffffu) * p.c;
        qv[h][2 * i + 1] = bf(x[i] >> 16) * p.c;
      }
    }
    const uint16_t* kb = p.k + static_cast<int64_t>(b) * p.cache_len * row_stride + kvh * kD + 8 * ds;
    const uint16_t* vb = p.v + static_cast<int64_t>(b) * p.cache_len * row_stride + kvh * kD + 8 * ds;
    // Keys of this lane: first = k0 aligned down to 16, then every 16.
    const int base = (k0 & ~15) + 4 * wave + kg;
    const int steps = (k1 - (k0 & ~15) + 15) >> 4;
    // Loads run kPf steps ahead of the compute (a ring of registers, the loop
    // unrolled by kPf so that every slot is static): one step alone is four
    // keys per wave, far too little to cover HBM latency.
    constexpr int kPf = G <= 4 ? 8 : 4;
    uint4 kr[kPf], vr[kPf];
    auto load = [&](int i, uint4& kv, uint4& vv) {
      const int kk = min(max(base + 16 * i, k0), k1 - 1);   // in bounds; masked below
      kv = *reinterpret_cast<const uint4*>(kb + kk * row_stride);
      vv = *reinterpret_cast<const uint4*>(vb + kk * row_stride);
    };
#pragma unroll
    for (int j = 0; j < kPf; ++j) load(j, kr[j], vr[j]);
    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
      m[h] = -INFINITY;
      l[h] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[h][i] = 0.f;
    }
    for (int i0 = 0; i0 < steps; i0 += kPf) {
#pragma unroll
      for (int j = 0; j < kPf; ++j) {
        const int i = i0 + j;
        if (i >= steps) break;
        const int kk = base + 16 * i;
        const bool live = kk >= k0 && kk < k1;
        const uint32_t kx[4] = {kr[j].x, kr[j].y, kr[j].z, kr[j].w};
        float s[G];
#pragma unroll
        for (int h = 0; h < G; ++h) s[h] = 0.f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const float a0 = bf(kx[d] & 0xffffu), a1 = bf(kx[d] >> 16);
#pragma unroll
          for (int h = 0; h < G; ++h)
            s[h] = __builtin_fmaf(a1, qv[h][2 * d + 1], __builtin_fmaf(a0, qv[h][2 * d], s[h]));
        }
        bool moved = false;
#pragma unroll
        for (int h = 0; h < G; ++h) {
          s[h] = row16_sum(s[h]);
          if (!live) s[h] = -INFINITY;
          moved = moved || (s[h] - m[h] > 8.0f);
        }
        if (__builtin_amdgcn_ballot_w64(moved)) {   // rare: move the maxima, rescale
#pragma unroll
          for (int h = 0; h < G; ++h) {
            const float mn = s[h] - m[h] > 8.0f ? s[h] : m[h];
            const float a = mn == m[h] ? 1.0f : __builtin_amdgcn_exp2f(m[h] - mn);
            m[h] = mn;
            l[h] *= a;
#pragma unroll
            for (int d = 0; d < 8; ++d) acc[h][d] *= a;
          }
        }
        const uint32_t vx[4] = {vr[j].x, vr[j].y, vr[j].z, vr[j].w};
#pragma unroll
        for (int h = 0; h < G; ++h) {
          const float pr = live ? __builtin_amdgcn_exp2f(s[h] - m[h]) : 0.f;
          l[h] += pr;
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            acc[h][2 * d] = __builtin_fmaf(pr, bf(vx[d] & 0xffffu), acc[h][2 * d]);
            acc[h][2 * d + 1] = __builtin_fmaf(pr, bf(vx[d] >> 16), acc[h][2 * d + 1]);
          }
        }
        load(i + kPf, kr[j], vr[j]);   // refill the slot; past the end: clamped, never used
      }
    }
    // Combine the four key groups of the wave (lanes l, l^16, l^32, l^48 hold
    // the same dims of different keys).
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float mm = m[h];
      mm = fmaxf(mm, __shfl_xor(mm, 16));
      mm = fmaxf(mm, __shfl_xor(mm, 32));
      const float a = mm == -INFINITY ? 0.f : exp2f(m[h] - mm);
      float lh = l[h] * a;
      lh += __shfl_xor(lh, 16);
      lh += __shfl_xor(lh, 32);
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        float x = acc[h][d] * a;
        x += __shfl_xor(x, 16);
        x += __shfl_xor(x, 32);
        if (kg == 0) s_acc[wave][h][8 * ds + d] = x;
      }
      if (lane == 0) {
        s_m[wave][h] = mm;
        s_l[wave][h] = lh;
      }
    }
    __syncthreads();
    // Combine the waves: one partial (unnormalised acc, max, sum) per head.
    float* po = p.part_o + slot * G * kD;
    float* pml = p.part_ml + slot * G * 2;
    for (int i = tid; i < G * kD; i += 256) {
      const int h = i / kD, d = i - h * kD;
      float mm = -INFINITY;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) mm = fmaxf(mm, s_m[w][h]);
      float a = 0.f;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w)
        if (s_m[w][h] != -INFINITY) a += exp2f(s_m[w][h] - mm) * s_acc[w][h][d];
      po[i] = a;
    }
    if (tid < G) {
      float mm = -INFINITY, lh = 0.f;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) mm = fmaxf(mm, s_m[w][tid]);
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w)
        if (s_m[w][tid] != -INFINITY) lh += exp2f(s_m[w][tid] - mm) * s_l[w][tid];
      pml[2 * tid] = mm;
      pml[2 * tid + 1] = lh;
    }
    }
    // The rest of the share continues at the start of the next pair (the
    // share ends inside this one otherwise).
    if (left == 0u) return;
    key = 0;
    if (++kvh == p.hkv) {
      kvh = 0;
      ++r;
    }
    __syncthreads();   // the next piece's combine writes the same LDS
  }
}

// One workgroup per output row (b, head): merge the split partials.  Thread
// (g, q) = (tid / 32, tid % 32) takes dims 4q .. +3 of splits g, g + 8, ...;
// the first kMergeAhead of them are loaded before the weights are known, so
// that a row of up to 32 splits costs one memory latency.  Latency-bound:
// each row reads its splits' 512-byte rows once.
constexpr int kMergeAhead = 4;
__global__ __launch_bounds__(256) void decode_merge_kernel(const DecodeParams p) {
  __shared__ float s_w[kMaxSplitsDev];
  __shared__ float s_red[8];
  __shared__ float4 s_part[8][kD / 4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = static_cast<int>(row / p.hq), hq = static_cast<int>(row - static_cast<int64_t>(b) * p.hq);
  const int kvh = hq / p.group, h = hq - kvh * p.group;
  // The pair's place on the line, the workgroups that share it and its slots.
  const SeqPlace seq = seq_place(p.plan[1 + b]);
  const uint32_t share = p.plan[0].x;
  const uint64_t off = seq.off + static_cast<uint64_t>(kvh) * seq.len;
  const uint32_t wg0 = quotient(off, share);
  const int nch = seq.n > 0 ? static_cast<int>(quotient(off + seq.n - 1, share) - wg0) + 1 : 0;   // at most 256
  const int64_t slot0 = static_cast<int64_t>(wg0) + static_cast<int64_t>(seq.rank) * p.hkv + kvh;
  const int g = tid >> 5, q = tid & 31;
  const float4* base = reinterpret_cast<const float4*>(p.part_o + (slot0 * p.group + h) * kD) + q;
  const int64_t cstride = static_cast<int64_t>(p.group) * (kD / 4);
  float2 ml = make_float2(-INFINITY, 0.f);   // split tid's maximum and sum
  if (tid < nch) ml = *reinterpret_cast<const float2*>(p.part_ml + ((slot0 + tid) * p.group + h) * 2);
  float4 ahead[kMergeAhead];
#pragma unroll
  for (int i = 0; i < kMergeAhead; ++i) {
    ahead[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (g + 8 * i < nch) ahead[i] = base[(g + 8 * i) * cstride];
  }
  // Maximum over the non-empty splits.
  float mx = ml.y > 0.f ? ml.x : -INFINITY;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  const float M = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  // Split weights 2^(m_c - M) (0 for empty splits) and the weighted sum of l.
  const float wt = (ml.y > 0.f && M != -INFINITY) ? __builtin_amdgcn_exp2f(ml.x - M) : 0.f;
  s_w[tid] = wt;
  float lsum = wt * ml.y;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) lsum += __shfl_xor(lsum, off);
  if (lane == 0) s_red[4 + wave] = lsum;
  __syncthreads();
  const float L = (s_red[4] + s_red[5]) + (s_red[6] + s_red[7]);
  // Weighted sum of the unnormalised partial outputs.
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  auto add = [&](int c, const float4& x) {
    const float w = s_w[c];
    if (w != 0.f) {
      a.x += w * x.x;
      a.y += w * x.y;
      a.z += w * x.z;
      a.w += w * x.w;
    }
  };
#pragma unroll
  for (int i = 0; i < kMergeAhead; ++i)
    if (g + 8 * i < nch) add(g + 8 * i, ahead[i]);
#pragma unroll 4
  for (int c = g + 8 * kMergeAhead; c < nch; c += 8) add(c, base[c * cstride]);
  s_part[g][q] = a;
  __syncthreads();
  if (tid < kD) {
    const float* part = reinterpret_cast<const float*>(s_part) + tid;
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc += part[i * kD];
    const float o = acc / L;   // empty row: 0 / 0 = NaN, as the prefill writes it
    p.out[row * kD + tid] = __builtin_bit_cast(uint16_t, static_cast<__bf16>(o));
    if (tid == 0) p.lse[row] = M == -INFINITY ? -INFINITY : M + log2f(L);
  }
}

}  // namespace
}  // namespace swattn

using namespace swattn;

extern "C" {

// Workgroups the line of routed keys is shared out over: two per CU, as many
// as are resident at once for the larger query groups.  The workspace holds
// four per CU plus one per (sequence, KV head) pair partials; shares number
// at most that many and each pair adds at most one piece.
constexpr int kSplitTarget = 2;   // workgroups per CU
constexpr int kSplitRoom = 4;     // partials per CU in the workspace
static_assert(2 * kSplitTarget <= kSplitRoom, "every share has its partial");

static int decode_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    return 256;
  return n;
}

struct DecodeLayout {
  int64_t slots, off_ml, off_list, off_plan, bytes;   // byte offsets
};

static DecodeLayout decode_layout(int64_t batch, int64_t heads_q, int64_t heads_kv, int cus) {
  DecodeLayout L{};
  L.slots = static_cast<int64_t>(kSplitRoom) * cus + batch * heads_kv;
  const int64_t group = heads_q / heads_kv;
  auto al = [](int64_t x) { return (x + 255) & ~static_cast<int64_t>(255); };
  int64_t o = al(L.slots * group * kD * 4);               // part_o
  L.off_ml = o;    o = al(o + L.slots * group * 2 * 4);
  L.off_list = o;  o = al(o + batch * 4);
  L.off_plan = o;  o = al(o + (1 + batch) * 16);
  L.bytes = o;
  return L;
}

size_t swattn_decode_workspace_bytes(int32_t batch, int64_t cache_len, int32_t heads_q,
                                     int32_t heads_kv) {
  if (batch < 1 || cache_len < 1 || heads_q < 1 || heads_kv < 1 || heads_q % heads_kv) return 0;
  return static_cast<size_t>(decode_layout(batch, heads_q, heads_kv, decode_cus()).bytes);
}

}  // extern "C"

// Argument checks shared by both decode entry points (name = the entry point).
static int decode_check(const char* name, const void* q, const void* k_cache,
                        const void* v_cache, const int32_t* cache_lens, const uint8_t* full,
                        void* out, float* lse, int32_t batch, int64_t cache_len,
                        int32_t heads_q, int32_t heads_kv, int32_t head_dim, int32_t window) {
  const std::string n(name);
  if (head_dim != kD) return invalid(n + ": head_dim must be 128");
  if (batch < 1 || cache_len < 1 || heads_q < 1 || heads_kv < 1) return invalid(n + ": bad shape");
  if (heads_q % heads_kv) return invalid(n + ": heads_q must be a multiple of heads_kv");
  if (heads_q / heads_kv > kMaxG) return invalid(n + ": heads_q / heads_kv must be at most 8");
  if (window <= 0) return invalid(n + ": window must be positive");
  if (batch > 65535 || heads_kv > 65535 || cache_len > INT32_MAX ||
      static_cast<int64_t>(batch) * heads_q > INT32_MAX)
    return invalid(n + ": batch, heads_kv or cache_len too large");
  if (q == nullptr || k_cache == nullptr || v_cache == nullptr || cache_lens == nullptr ||
      full == nullptr || out == nullptr || lse == nullptr)
    return invalid(n + ": null pointer");
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return invalid(n + ": q, k_cache, v_cache and out must be 16-byte aligned");
  return SWATTN_OK;
}

template <int G>
static void launch_split(bool inline_plan, dim3 grid, hipStream_t st, const DecodeParams& p) {
  if (inline_plan)
    hipLaunchKernelGGL((decode_split_kernel<G, true>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((decode_split_kernel<G, false>), grid, dim3(256), 0, st, p);
}

// Split and merge kernels (and the plan kernel for many sequences) on `stream`
// with the (checked) workspace ws.
static int decode_launch(const char* name, const void* q, const void* k_cache,
                         const void* v_cache, const int32_t* cache_lens, const uint8_t* full,
                         void* out, float* lse, int32_t batch, int64_t cache_len,
                         int32_t heads_q, int32_t heads_kv, int32_t window, float scale_log2,
                         char* ws, void* stream) {
  const int group = heads_q / heads_kv;
  DecodeParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k_cache);
  p.v = static_cast<const uint16_t*>(v_cache);
  p.lens = cache_lens;
  p.full = full;
  const int cus = decode_cus();
  const DecodeLayout L = decode_layout(batch, heads_q, heads_kv, cus);
  if (L.slots > INT32_MAX) return invalid(std::string(name) + ": too many work items");
  p.part_o = reinterpret_cast<float*>(ws);
  p.part_ml = reinterpret_cast<float*>(ws + L.off_ml);
  p.list = reinterpret_cast<int32_t*>(ws + L.off_list);
  p.plan = reinterpret_cast<uint4*>(ws + L.off_plan);
  p.target = kSplitTarget * cus;
  // A share is at most the line over the resident workgroups, and has to fit 32
  // bits: with 256 CUs the limit is 128 TiB of K, the size of the address space.
  const int64_t rows = static_cast<int64_t>(batch) * cache_len * heads_kv;
  if (rows / p.target >= (int64_t{1} << 30))
    return invalid(std::string(name) + ": the K cache is larger than the address space");
  // (Padding positions of the line stay below 2^30 beside at most 2^31 keys.)
  p.pad = static_cast<int64_t>(batch) * heads_kv < (int64_t{1} << 30) / kPairPad ? kPairPad : 0;
  p.batch = batch;
  p.out = static_cast<uint16_t*>(out);
  p.lse = lse;
  p.cache_len = static_cast<int>(cache_len);
  p.hq = heads_q;
  p.hkv = heads_kv;
  p.group = group;
  p.window = window;
  p.c = scale_log2;
  const hipStream_t st = as_stream(stream);
  // Up to kInlineSeqs sequences the split workgroups plan for themselves, at
  // up to kInlinePer sequences per thread; beyond that each of them would
  // read too many lengths and the plan kernel's few us no longer count
  // beside the thousands of pairs.  (Caches of 2^31 rows, which only a sparsely
  // mapped address range can hold, need the plan kernel's 64-bit positions.)
  const bool inline_plan = batch <= kInlineSeqs && rows <= INT32_MAX;
  if (!inline_plan) hipLaunchKernelGGL(decode_plan_kernel, dim3(1), dim3(kPlanThreads), 0, st, p);
  // Grid: one workgroup per share, no more of them than whole caches can fill
  // at kMinShare positions each.
  const int64_t pairs = static_cast<int64_t>(batch) * heads_kv;
  const int64_t most = pairs * ((cache_len + p.pad + kMinShare - 1) / kMinShare);
  const dim3 grid(static_cast<uint32_t>(most < 2 * p.target ? most : 2 * p.target));
  switch (group) {
    case 1: launch_split<1>(inline_plan, grid, st, p); break;
    case 2: launch_split<2>(inline_plan, grid, st, p); break;
    case 3: launch_split<3>(inline_plan, grid, st, p); break;
    case 4: launch_split<4>(inline_plan, grid, st, p); break;
    case 5: launch_split<5>(inline_plan, grid, st, p); break;
    case 6: launch_split<6>(inline_plan, grid, st, p); break;
    case 7: launch_split<7>(inline_plan, grid, st, p); break;
    default: launch_split<8>(inline_plan, grid, st, p); break;
  }
  const int64_t out_rows = static_cast<int64_t>(batch) * heads_q;
  hipLaunchKernelGGL(decode_merge_kernel, dim3(static_cast<uint32_t>(out_rows)), dim3(256), 0, st, p);
  return launch_status(name);
}

extern "C" {

int swattn_decode_fwd(const void* q, const void* k_cache, const void* v_cache,
                      const int32_t* cache_lens, const uint8_t* full, void* out, float* lse,
                      int32_t batch, int64_t cache_len, int32_t heads_q, int32_t heads_kv,
                      int32_t head_dim, int32_t window, float scale_log2, void* workspace,
                      size_t workspace_bytes, void* stream) {
  const char* name = "swattn_decode_fwd";
  const int st = decode_check(name, q, k_cache, v_cache, cache_lens, full, out, lse, batch,
                              cache_len, heads_q, heads_kv, head_dim, window);
  if (st != SWATTN_OK) return st;
  const size_t need = swattn_decode_workspace_bytes(batch, cache_len, heads_q, heads_kv);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("swattn_decode_fwd: workspace smaller than swattn_decode_workspace_bytes()");
    return SWATTN_EWORKSPACE;
  }
  if (!aligned256(workspace)) return invalid("swattn_decode_fwd: workspace must be 256-byte aligned");
  return decode_launch(name, q, k_cache, v_cache, cache_lens, full, out, lse, batch, cache_len,
                       heads_q, heads_kv, window, scale_log2, static_cast<char*>(workspace),
                       stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The same decode with library-owned scratch, for callers that cannot
// allocate device memory (code under HIP graph capture, tight serving loops).
// `scratch` is a file-scope device array: every GPU the library runs on gets
// its own copy, held until the process ends.  In host code its name is only a
// host-side stand-in, so its device address is looked up once per device
// (hipGetSymbolAddress, with that device current) and only that address is
// ever handed to kernels.  The decode kernels write every scratch byte they
// read within the same call (plan, list of sequences, partials), so nothing
// needs clearing between calls; two calls that overlap on one GPU share the
// array and race.
// ---------------------------------------------------------------------------
constexpr size_t kDecodeScratchBytes = SWATTN_DECODE_NOALLOC_MAX_BYTES;   // 16 MiB per GPU
static_assert(kDecodeScratchBytes % 256 == 0, "whole 256-byte lines");
static __device__ __align__(256) char scratch[kDecodeScratchBytes];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxScratchDevices];   // per device, nullptr until looked up

// Device address of this GPU's scratch array (the current device's), or
// nullptr with the error set.
static void* scratch_for_current_device(const char* name) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices) {
    set_error(std::string(name) + ": no usable current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      set_error(std::string(name) + ": hipGetSymbolAddress(scratch): " + hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

extern "C" {

int swattn_decode_fwd_noalloc(const void* q, const void* k_cache, const void* v_cache,
                              const int32_t* cache_lens, const uint8_t* full, void* out,
                              float* lse, int32_t batch, int64_t cache_len, int32_t heads_q,
                              int32_t heads_kv, int32_t head_dim, int32_t window,
                              float scale_log2, void* stream) {
  const char* name = "swattn_decode_fwd_noalloc";
  const int st = decode_check(name, q, k_cache, v_cache, cache_lens, full, out, lse, batch,
                              cache_len, heads_q, heads_kv, head_dim, window);
  if (st != SWATTN_OK) return st;
  const size_t need = swattn_decode_workspace_bytes(batch, cache_len, heads_q, heads_kv);
  if (need > kDecodeScratchBytes) {
    set_error("swattn_decode_fwd_noalloc: this shape needs " + std::to_string(need) +
              " bytes of scratch, more than the library's " +
              std::to_string(kDecodeScratchBytes) + " (use swattn_decode_fwd with a workspace)");
    return SWATTN_EINVAL;
  }
  void* ws = scratch_for_current_device(name);
  if (ws == nullptr) return SWATTN_EINVAL;
  return decode_launch(name, q, k_cache, v_cache, cache_lens, full, out, lse, batch, cache_len,
                       heads_q, heads_kv, window, scale_log2, static_cast<char*>(ws), stream);
}

}  // extern "C"
