// Integer kernels of the routed prefill: router-mask compaction, index-list
// validation and varlen position metadata.  gfx950, wave64.
//
// Reference tags: V = swiattn_gqa_prefill_varlen.py, F = swiattn_gqa_prefill.py.

#include <limits.h>
#include <string.h>

#include <atomic>
#include <chrono>
#include <string>

#include "common.h"
#include "swattn_internal.h"

namespace swattn {

static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }

namespace {

// ---------------------------------------------------------------------------
// Compaction (V:306-322).
//
// A block of 16 waves owns 4096 or (long masks) 16384 consecutive mask bytes;
// wave w owns 4 or 16 groups of 64 bytes.  Lane l of group e reads byte base +
// 64e + l, so each group is one coalesced 64-byte read and one 64-bit ballot.
// popcount(ballot) gives the
// group's full count and mbcnt(ballot) a lane's rank inside the group; the
// ballots stay in scalar registers between the counting pass and the write
// pass, so the mask is read once per kernel.  Full position i lands at
// index excl(i) and local position i at nf + i - excl(i), where excl(i) is the
// number of full positions before i: both lists come out ascending and the
// whole output is exactly arange(n)[mask] ++ arange(n)[~mask].
// ---------------------------------------------------------------------------
constexpr int kCompactWaves = 16;
constexpr int kCompactThreads = kCompactWaves * 64;
constexpr int kCompactGroups = 16;
constexpr int kCompactChunk = kCompactThreads * kCompactGroups;  // 16384 bytes per block

// What decides "full" for position i: a byte mask, or router logits above a
// threshold (compared in fp32; bf16 and fp16 convert exactly, NaN is never
// above the threshold).
// count16: how many of the 16 bytes' values are full (kPer of them).
struct MaskSource {
  static constexpr int kPer = 16;
  const uint8_t* p;
  __device__ __forceinline__ bool operator()(int64_t i) const { return p[i] != 0; }
  __device__ __forceinline__ int count16(const uint4& v) const {
    auto nonzero = [](uint32_t x) {   // bytes of x that are not 0
      return __builtin_popcount((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u);
    };
    return nonzero(v.x) + nonzero(v.y) + nonzero(v.z) + nonzero(v.w);
  }
};
struct F32LogitSource {
  static constexpr int kPer = 4;
  const float* p;
  float thr;
  __device__ __forceinline__ bool operator()(int64_t i) const { return p[i] > thr; }
  __device__ __forceinline__ int count16(const uint4& v) const {
    return (__uint_as_float(v.x) > thr) + (__uint_as_float(v.y) > thr) +
           (__uint_as_float(v.z) > thr) + (__uint_as_float(v.w) > thr);
  }
};
struct BF16LogitSource {
  static constexpr int kPer = 8;
  const uint16_t* p;
  float thr;
  __device__ __forceinline__ bool operator()(int64_t i) const {
    return __uint_as_float(static_cast<uint32_t>(p[i]) << 16) > thr;
  }
  __device__ __forceinline__ int count16(const uint4& v) const {
    auto both = [this](uint32_t x) {
      return (__uint_as_float(x << 16) > thr) + (__uint_as_float(x & 0xffff0000u) > thr);
    };
    return both(v.x) + both(v.y) + both(v.z) + both(v.w);
  }
};
struct F16LogitSource {
  static constexpr int kPer = 8;
  const _Float16* p;
  float thr;
  __device__ __forceinline__ bool operator()(int64_t i) const {
    return static_cast<float>(p[i]) > thr;
  }
  __device__ __forceinline__ int count16(const uint4& v) const {
    auto both = [this](uint32_t x) {
      const auto h = __builtin_bit_cast(__attribute__((ext_vector_type(2))) _Float16, x);
      return (static_cast<float>(h.x) > thr) + (static_cast<float>(h.y) > thr);
    };
    return both(v.x) + both(v.y) + both(v.z) + both(v.w);
  }
};

// Position of lane `lane` of group e of wave `wave`, kGroups groups per wave.
template <int kGroups>
__device__ __forceinline__ int64_t compact_elem(int wave, int e, int lane) {
  return (static_cast<int64_t>(blockIdx.x) * kCompactWaves + wave) * (64 * kGroups) + 64 * e + lane;
}

// The write pass of a block: its ballots, the full positions before the wave
// (all of the mask's before the block included) and in all of the mask.
template <int kGroups>
__device__ __forceinline__ void compact_write(const uint64_t (&bal)[kGroups], int64_t full_before,
                                              int64_t nf, int64_t n, int32_t* __restrict__ indices) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int e = 0; e < kGroups; ++e) {
    const int64_t i = compact_elem<kGroups>(wave, e, lane);
    const uint64_t b = bal[e];
    const int64_t fb = full_before + count_below(b);
    if (i < n) {
      if ((b >> lane) & 1ull)
        indices[fb] = static_cast<int32_t>(i);
      else
        indices[nf + (i - fb)] = static_cast<int32_t>(i);
    }
    full_before += __builtin_popcountll(b);
  }
}

// One launch, for masks that every block can afford to read whole: a block
// writes 4096 positions and counts the full ones of all the mask, those before
// its own apart, from L2 (16 bytes per lane and load where the mask is
// 16-byte aligned).  Latency-bound: against one block for all 16384 positions
// this spreads the loads and the stores over CUs, and against a counting
// kernel first it saves that launch.  Back to back, byte mask: 1024 positions
// 4.6 -> 2.8 us, 16384 5.9 -> 4.1, 65536 9.6 (two kernels) -> 4.6, 262144 10.1 ->
// 6.6; fp32 logits: 16384 6.0 -> 4.5, 65536 10.0 -> 6.2.
constexpr int kWholeGroups = 4;
constexpr int kWholeChunk = kCompactThreads * kWholeGroups;   // 4096 positions per block
constexpr int64_t kWholeBytes = 256 << 10;   // a block reads at most this much (10 us, as two kernels)
constexpr int64_t kWholeUnaligned = 64 << 10;   // positions, read one by one (8 us; 131072: 12)
static_assert(kWholeBytes / kWholeChunk + 2 <= SWATTN_COMPACT_HOST_WORDS, "one word per block");
//
// kHost: counts is pinned host memory that a host thread polls, with one word
// per block after the counts.  A block sets its word when its indices are in
// memory, so that a host that has seen all of them may hand the lists to any
// stream, as after a synchronisation: every wave waits for its own stores, and
// after the barrier one thread's system-scope release writes the L2 back for
// all of them.  (With a system-scope fence in each of the 16 waves a block
// wrote it back 16 times over: prefill B1 S1024 38.2 -> 34.9 us per call, S2999
// 100.3 -> 95.4, B2 S4096 206.2 -> 200.9.  Stores through the caches, with no
// release, take the same time.)
template <typename Src, bool kVec, bool kHost>
__global__ __launch_bounds__(kCompactThreads) void compact_whole_kernel(
    const Src src, int64_t n, int32_t* __restrict__ indices, int32_t* __restrict__ counts) {
  __shared__ int s_own[kCompactWaves], s_before[kCompactWaves], s_all[kCompactWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint64_t bal[kWholeGroups];
  int own = 0;
#pragma unroll
  for (int e = 0; e < kWholeGroups; ++e) {
    const int64_t i = compact_elem<kWholeGroups>(wave, e, lane);
    const bool f = i < n && src(i);
    bal[e] = wave_ballot(f);
    own += __builtin_popcountll(bal[e]);
  }
  int before = 0, all = 0;
  if (gridDim.x > 1) {
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kWholeChunk;
    int64_t done = 0;
    if constexpr (kVec) {   // kPer divides the chunk: a load is before it or not
      const int64_t whole = n / Src::kPer;
      const uint4* p = reinterpret_cast<const uint4*>(src.p);
#pragma unroll 4
      for (int64_t v = tid; v < whole; v += kCompactThreads) {
        const int c = src.count16(p[v]);
        all += c;
        before += v * Src::kPer < first ? c : 0;
      }
      done = whole * Src::kPer;
    }
#pragma unroll 4
    for (int64_t i = done + tid; i < n; i += kCompactThreads) {
      const int c = src(i) ? 1 : 0;
      all += c;
      before += i < first ? c : 0;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      all += __shfl_xor(all, off);
      before += __shfl_xor(before, off);
    }
  }
  if (lane == 0) {
    s_own[wave] = own;
    s_before[wave] = before;
    s_all[wave] = all;
  }
  __syncthreads();
  int64_t full_before = 0, nf = 0;
#pragma unroll
  for (int w = 0; w < kCompactWaves; ++w) {
    full_before += s_before[w] + (w < wave ? s_own[w] : 0);
    nf += gridDim.x > 1 ? s_all[w] : s_own[w];
  }
  if (blockIdx.x == 0 && tid == 0) {
    counts[0] = static_cast<int32_t>(nf);
    counts[1] = static_cast<int32_t>(n - nf);
  }
  compact_write<kWholeGroups>(bal, full_before, nf, n, indices);
  if constexpr (kHost) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's own stores
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(counts + 2 + blockIdx.x, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <typename Src>
__global__ __launch_bounds__(kCompactThreads) void compact_count_kernel(
    const Src src, int64_t n, int32_t* __restrict__ block_counts) {
  __shared__ int s_wave[kCompactWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int cnt = 0;
#pragma unroll
  for (int e = 0; e < kCompactGroups; ++e) {
    const int64_t i = compact_elem<kCompactGroups>(wave, e, lane);
    const bool f = i < n && src(i);
    cnt += __builtin_popcountll(wave_ballot(f));
  }
  if (lane == 0) s_wave[wave] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int w = 0; w < kCompactWaves; ++w) tot += s_wave[w];
    block_counts[blockIdx.x] = tot;
  }
}

template <typename Src>
__global__ __launch_bounds__(kCompactThreads) void compact_scatter_kernel(
    const Src src, int64_t n, const int32_t* __restrict__ block_counts,
    int nblocks, int32_t* __restrict__ indices, int32_t* __restrict__ counts) {
  __shared__ int s_wave[kCompactWaves];
  __shared__ int s_prefix, s_total;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t bal[kCompactGroups];
  int cnt = 0;
#pragma unroll
  for (int e = 0; e < kCompactGroups; ++e) {
    const int64_t i = compact_elem<kCompactGroups>(wave, e, lane);
    const bool f = i < n && src(i);
    bal[e] = wave_ballot(f);
    cnt += __builtin_popcountll(bal[e]);
  }
  if (lane == 0) s_wave[wave] = cnt;
  if (wave == 0) {
    int pre = 0, tot = 0;
    for (int j = lane; j < nblocks; j += 64) {
      const int c = block_counts[j];
      tot += c;
      pre += (j < static_cast<int>(blockIdx.x)) ? c : 0;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      pre += __shfl_xor(pre, off);
      tot += __shfl_xor(tot, off);
    }
    if (lane == 0) {
      s_prefix = pre;
      s_total = tot;
    }
  }
  __syncthreads();
  int wave_prefix = s_prefix;
  for (int w = 0; w < wave; ++w) wave_prefix += s_wave[w];
  const int64_t nf = s_total;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    counts[0] = static_cast<int32_t>(nf);
    counts[1] = static_cast<int32_t>(n - nf);
  }
  compact_write<kCompactGroups>(bal, wave_prefix, nf, n, indices);
}

// ---------------------------------------------------------------------------
// Index validation (V:299-302 on both lists, disjointness of V:341-342).
// One thread per slot; a slot checks its full entry (range, order against the
// previous entry, binary search in the local list) and its local entry (range,
// order).  Any failure ORs its bit into *flags, which flags_clear_kernel zeroes
// first.  The binary search is only meaningful when the local list is sorted;
// when it is not, ERR_LOCAL_ORDER is raised and the caller reports that first.
// ---------------------------------------------------------------------------
__global__ void flags_clear_kernel(int32_t* flags) { flags[0] = 0; }

__global__ __launch_bounds__(256) void check_indices_kernel(
    const int32_t* __restrict__ full, int64_t nf, const int32_t* __restrict__ local, int64_t nl,
    int64_t seq_len, int32_t* __restrict__ flags) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  int f = 0;
  if (i < nf) {
    const int32_t x = full[i];
    if (x < 0 || x >= seq_len) f |= SWATTN_ERR_FULL_RANGE;
    if (i > 0 && x <= full[i - 1]) f |= SWATTN_ERR_FULL_ORDER;
    int64_t lo = 0, hi = nl;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (local[mid] < x)
        lo = mid + 1;
      else
        hi = mid;
    }
    if (lo < nl && local[lo] == x) f |= SWATTN_ERR_OVERLAP;
  }
  if (i < nl) {
    const int32_t x = local[i];
    if (x < 0 || x >= seq_len) f |= SWATTN_ERR_LOCAL_RANGE;
    if (i > 0 && x <= local[i - 1]) f |= SWATTN_ERR_LOCAL_ORDER;
  }
  // One atomic per wave that saw a failure.
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) f |= __shfl_xor(f, off);
  if (f != 0 && (threadIdx.x & 63) == 0) atomicOr(flags, f);
}

// ---------------------------------------------------------------------------
// Varlen metadata (the fields V validates at V:360-383; F's rule per segment).
// One thread per token; the segment is found by binary search in cu_seqlens.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int find_segment(const int32_t* cu, int nseq, int64_t t) {
  int lo = 0, hi = nseq;  // invariant: cu[lo] <= t < cu[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu[mid] <= t)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

struct MetadataOut {
  int32_t *q_pos, *kv_pos, *q_seg, *kv_seg, *full_starts, *local_starts, *causal_ends;
};

__device__ __forceinline__ void metadata_entry(const int32_t* cu_q, const int32_t* cu_kv, int nseq,
                                               int64_t total_q, int64_t total_kv, int window,
                                               const MetadataOut& o) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < total_q) {
    const int s = find_segment(cu_q, nseq, t);
    const int64_t i = t - cu_q[s];
    const int64_t ks = cu_kv[s], klen = static_cast<int64_t>(cu_kv[s + 1]) - ks;
    o.q_pos[t] = static_cast<int32_t>(i);
    o.q_seg[t] = s;
    o.full_starts[t] = static_cast<int32_t>(ks);
    const int64_t lo = i - window + 1;
    o.local_starts[t] = static_cast<int32_t>(ks + (lo > 0 ? lo : 0));
    o.causal_ends[t] = static_cast<int32_t>(ks + (i + 1 < klen ? i + 1 : klen));
  }
  if (t < total_kv) {
    const int s = find_segment(cu_kv, nseq, t);
    o.kv_pos[t] = static_cast<int32_t>(t - cu_kv[s]);
    o.kv_seg[t] = s;
  }
}

__global__ __launch_bounds__(256) void metadata_kernel(const int32_t* __restrict__ cu_q,
                                                       const int32_t* __restrict__ cu_kv, int nseq,
                                                       int64_t total_q, int64_t total_kv,
                                                       int window, const MetadataOut o) {
  metadata_entry(cu_q, cu_kv, nseq, total_q, total_kv, window, o);
}

// The same with the offsets as kernel arguments (up to kCuMax - 1 sequences),
// staged in LDS for the searches.  The caller's offsets live on the host: as
// device arrays they took two blocking copies of about 15 us before the launch.
constexpr int kCuMax = 257;
struct CuArgs {
  int32_t q[kCuMax], kv[kCuMax];
};
static_assert(sizeof(CuArgs) <= 3072, "kernel arguments end at 4 KiB");
__global__ __launch_bounds__(256) void metadata_args_kernel(const CuArgs cu, int nseq,
                                                            int64_t total_q, int64_t total_kv,
                                                            int window, const MetadataOut o) {
  __shared__ int32_t s_q[kCuMax], s_kv[kCuMax];
  for (int i = threadIdx.x; i <= nseq; i += 256) {
    s_q[i] = cu.q[i];
    s_kv[i] = cu.kv[i];
  }
  __syncthreads();
  metadata_entry(s_q, s_kv, nseq, total_q, total_kv, window, o);
}

// Whether each list's key bounds are non-decreasing along it (a start past its
// row's end counts as the end): what the backward's searches need.  One thread
// per entry of both lists and its successor; a listed position outside
// [0, total_q) is never dereferenced and fails the check.
__global__ __launch_bounds__(256) void check_bounds_kernel(
    const int32_t* __restrict__ full, int64_t nf, const int32_t* __restrict__ local, int64_t nl,
    const int32_t* __restrict__ full_starts, const int32_t* __restrict__ local_starts,
    const int32_t* __restrict__ ends, int64_t total_q, int32_t* __restrict__ flags) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  auto falls = [&](const int32_t* list, int64_t n, const int32_t* starts) {
    if (i >= n) return false;
    const int32_t a = list[i];
    if (a < 0 || a >= total_q) return true;
    if (i + 1 >= n) return false;
    const int32_t b = list[i + 1];
    if (b < 0 || b >= total_q) return true;
    const int32_t ea = ends[a], eb = ends[b];
    return eb < ea || min(starts[b], eb) < min(starts[a], ea);
  };
  const bool f = falls(full, nf, full_starts) || falls(local, nl, local_starts);
  if (wave_ballot(f) != 0 && (threadIdx.x & 63) == 0) atomicOr(flags, 1);
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int compact_logits_impl(const void* logits, int32_t dtype, int64_t n, float threshold,
                        int32_t* indices, int32_t* counts, void* workspace, size_t workspace_bytes,
                        void* stream, const char* name, int* host_blocks);

static_assert(kCuMax == SWATTN_METADATA_HOST_MAX_SEQS + 1, "offsets of the header's limit");

// Argument checks shared by both metadata entry points.
int metadata_check(const char* name, const int32_t* cu_q, const int32_t* cu_kv, int32_t num_seqs,
                   int64_t total_q, int64_t total_kv, int32_t window, const MetadataOut& o) {
  const std::string n(name);
  if (num_seqs < 1 || total_q < 0 || total_kv < 0 || total_q > INT32_MAX || total_kv > INT32_MAX)
    return invalid(n + ": bad sizes");
  if (window <= 0) return invalid(n + ": window must be positive");
  if (cu_q == nullptr || cu_kv == nullptr) return invalid(n + ": null cu_seqlens");
  if ((total_q > 0 && (o.q_pos == nullptr || o.q_seg == nullptr || o.full_starts == nullptr ||
                       o.local_starts == nullptr || o.causal_ends == nullptr)) ||
      (total_kv > 0 && (o.kv_pos == nullptr || o.kv_seg == nullptr)))
    return invalid(n + ": null output");
  return SWATTN_OK;
}

template <typename Src>
int compact_impl(const Src& src, bool src_null, int64_t n, int32_t* indices, int32_t* counts,
                 void* workspace, size_t workspace_bytes, void* stream, const char* name,
                 int* host_blocks = nullptr);

}  // namespace
}  // namespace swattn

using namespace swattn;

extern "C" {

int swattn_version(void) { return (0 << 16) | 2; }

const char* swattn_last_error(void) { return g_last_error.c_str(); }

size_t swattn_compact_workspace_bytes(int64_t n) {
  const int64_t nb = ceil_div(n, kCompactChunk);
  return nb > 1 ? static_cast<size_t>(nb) * sizeof(int32_t) : 0;
}

int swattn_compact(const uint8_t* mask, int64_t n, int32_t* indices, int32_t* counts,
                   void* workspace, size_t workspace_bytes, void* stream) {
  return compact_impl(MaskSource{mask}, mask == nullptr, n, indices, counts, workspace,
                      workspace_bytes, stream, "swattn_compact");
}

int swattn_compact_logits(const void* logits, int32_t dtype, int64_t n, float threshold,
                          int32_t* indices, int32_t* counts, void* workspace,
                          size_t workspace_bytes, void* stream) {
  const char* name = "swattn_compact_logits";
  return compact_logits_impl(logits, dtype, n, threshold, indices, counts, workspace,
                             workspace_bytes, stream, name, nullptr);
}

int swattn_compact_wait(const void* x, int32_t dtype, int64_t n, float threshold, int32_t* indices,
                        int32_t* host, void* workspace, size_t workspace_bytes, void* stream) {
  const char* name = dtype < 0 ? "swattn_compact" : "swattn_compact_logits";
  if (host == nullptr) return invalid(std::string(name) + ": null pointer");
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(as_stream(stream), &capture) == hipSuccess &&
      capture != hipStreamCaptureStatusNone)   // before a launch that nothing could wait for
    return invalid(std::string(name) + ": waits for its result and cannot be captured");
  for (int i = 0; i < SWATTN_COMPACT_HOST_WORDS; ++i) host[i] = 0;
  int blocks = 0;
  const int status =
      dtype < 0 ? compact_impl(MaskSource{static_cast<const uint8_t*>(x)}, x == nullptr, n, indices,
                               host, workspace, workspace_bytes, stream, name, &blocks)
                : compact_logits_impl(x, dtype, n, threshold, indices, host, workspace,
                                      workspace_bytes, stream, name, &blocks);
  if (status != SWATTN_OK) {
    // A HIP error, perhaps one that an earlier call left pending: the kernel may
    // be queued all the same, and must not report into the next call's words.
    if (status > 0) (void)hipStreamSynchronize(as_stream(stream));
    return status;
  }
  // Poll the blocks' words for a while; then, or where none report, wait for
  // the stream (it may hold any amount of earlier work, or have failed).
  volatile int32_t* word = host + 2;
  const auto t0 = std::chrono::steady_clock::now();
  for (int done = 0; blocks > 0;) {
    while (done < blocks && word[done] != 0) ++done;
    if (done == blocks) {
      std::atomic_thread_fence(std::memory_order_acquire);
      return SWATTN_OK;
    }
    __builtin_ia32_pause();
    if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) break;
  }
  const hipError_t e = hipStreamSynchronize(as_stream(stream));
  if (e != hipSuccess) {
    set_error(std::string(name) + ": " + hipGetErrorString(e));
    return static_cast<int>(e);
  }
  return SWATTN_OK;
}

}  // extern "C"

namespace swattn {
namespace {

int compact_logits_impl(const void* logits, int32_t dtype, int64_t n, float threshold,
                        int32_t* indices, int32_t* counts, void* workspace, size_t workspace_bytes,
                        void* stream, const char* name, int* host_blocks) {
  switch (dtype) {
    case SWATTN_DTYPE_F32:
      return compact_impl(F32LogitSource{static_cast<const float*>(logits), threshold},
                          logits == nullptr, n, indices, counts, workspace, workspace_bytes,
                          stream, name, host_blocks);
    case SWATTN_DTYPE_BF16:
      return compact_impl(BF16LogitSource{static_cast<const uint16_t*>(logits), threshold},
                          logits == nullptr, n, indices, counts, workspace, workspace_bytes,
                          stream, name, host_blocks);
    case SWATTN_DTYPE_F16:
      return compact_impl(F16LogitSource{static_cast<const _Float16*>(logits), threshold},
                          logits == nullptr, n, indices, counts, workspace, workspace_bytes,
                          stream, name, host_blocks);
    default:
      return invalid("swattn_compact_logits: dtype must be SWATTN_DTYPE_F32, _BF16 or _F16");
  }
}

}  // namespace
}  // namespace swattn

extern "C" {

int swattn_check_indices(const int32_t* full, int64_t n_full, const int32_t* local,
                         int64_t n_local, int64_t seq_len, int32_t* flags, void* stream) {
  if (n_full < 0 || n_local < 0 || seq_len < 0 || seq_len > INT32_MAX)
    return invalid("swattn_check_indices: bad sizes");
  if (flags == nullptr || (n_full > 0 && full == nullptr) || (n_local > 0 && local == nullptr))
    return invalid("swattn_check_indices: null pointer");
  const hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(flags_clear_kernel, dim3(1), dim3(1), 0, st, flags);
  const int64_t n = n_full > n_local ? n_full : n_local;
  if (n > 0) {
    hipLaunchKernelGGL(check_indices_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, full,
                       n_full, local, n_local, seq_len, flags);
  }
  return launch_status("swattn_check_indices");
}

int swattn_check_bounds(const int32_t* full, int64_t n_full, const int32_t* local, int64_t n_local,
                        const int32_t* full_starts, const int32_t* local_starts,
                        const int32_t* causal_ends, int64_t total_q, int32_t* flags,
                        void* stream) {
  if (n_full < 0 || n_local < 0 || total_q < 0 || total_q > INT32_MAX)
    return invalid("swattn_check_bounds: bad sizes");
  if (flags == nullptr || (n_full > 0 && (full == nullptr || full_starts == nullptr)) ||
      (n_local > 0 && (local == nullptr || local_starts == nullptr)) ||
      (n_full + n_local > 0 && causal_ends == nullptr))
    return invalid("swattn_check_bounds: null pointer");
  const hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(flags_clear_kernel, dim3(1), dim3(1), 0, st, flags);
  const int64_t n = n_full > n_local ? n_full : n_local;
  if (n > 0)
    hipLaunchKernelGGL(check_bounds_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, full, n_full,
                       local, n_local, full_starts, local_starts, causal_ends, total_q, flags);
  return launch_status("swattn_check_bounds");
}

int swattn_build_metadata(const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                          int32_t num_seqs, int64_t total_q, int64_t total_kv, int32_t window,
                          int32_t* q_positions, int32_t* kv_positions, int32_t* q_segment_ids,
                          int32_t* kv_segment_ids, int32_t* full_starts, int32_t* local_starts,
                          int32_t* causal_ends, void* stream) {
  const MetadataOut o{q_positions, kv_positions, q_segment_ids, kv_segment_ids,
                      full_starts, local_starts, causal_ends};
  const char* name = "swattn_build_metadata";
  const int st = metadata_check(name, cu_seqlens_q, cu_seqlens_kv, num_seqs, total_q, total_kv,
                                window, o);
  const int64_t n = total_q > total_kv ? total_q : total_kv;
  if (st != SWATTN_OK || n == 0) return st;
  hipLaunchKernelGGL(metadata_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, as_stream(stream),
                     cu_seqlens_q, cu_seqlens_kv, num_seqs, total_q, total_kv, window, o);
  return launch_status(name);
}

int swattn_build_metadata_host(const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                               int32_t num_seqs, int64_t total_q, int64_t total_kv, int32_t window,
                               int32_t* q_positions, int32_t* kv_positions,
                               int32_t* q_segment_ids, int32_t* kv_segment_ids,
                               int32_t* full_starts, int32_t* local_starts, int32_t* causal_ends,
                               void* stream) {
  const MetadataOut o{q_positions, kv_positions, q_segment_ids, kv_segment_ids,
                      full_starts, local_starts, causal_ends};
  const char* name = "swattn_build_metadata_host";
  const int st = metadata_check(name, cu_seqlens_q, cu_seqlens_kv, num_seqs, total_q, total_kv,
                                window, o);
  if (st != SWATTN_OK) return st;
  if (num_seqs > SWATTN_METADATA_HOST_MAX_SEQS)
    return invalid("swattn_build_metadata_host: too many sequences (use swattn_build_metadata)");
  CuArgs cu{};
  memcpy(cu.q, cu_seqlens_q, (num_seqs + 1) * sizeof(int32_t));
  memcpy(cu.kv, cu_seqlens_kv, (num_seqs + 1) * sizeof(int32_t));
  const int64_t n = total_q > total_kv ? total_q : total_kv;
  if (n == 0) return SWATTN_OK;
  hipLaunchKernelGGL(metadata_args_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, as_stream(stream),
                     cu, num_seqs, total_q, total_kv, window, o);
  return launch_status(name);
}

}  // extern "C"

namespace swattn {
namespace {

// host_blocks: counts is pinned host memory; set to the blocks that report
// there (0: the stream has to be synchronised instead).
template <typename Src>
int compact_impl(const Src& src, bool src_null, int64_t n, int32_t* indices, int32_t* counts,
                 void* workspace, size_t workspace_bytes, void* stream, const char* name,
                 int* host_blocks) {
  if (n < 0 || n > INT32_MAX) return invalid(std::string(name) + ": n must be in [0, 2^31)");
  if (counts == nullptr || (n > 0 && (src_null || indices == nullptr)))
    return invalid(std::string(name) + ": null pointer");
  const hipStream_t st = as_stream(stream);
  if (n == 0) {
    hipLaunchKernelGGL(flags_clear_kernel, dim3(1), dim3(1), 0, st, counts);
    hipLaunchKernelGGL(flags_clear_kernel, dim3(1), dim3(1), 0, st, counts + 1);
    return launch_status(name);
  }
  const int64_t nb = ceil_div(n, kCompactChunk);
  if (nb > 1) {
    if (workspace == nullptr || workspace_bytes < swattn_compact_workspace_bytes(n)) {
      set_error(std::string(name) + ": workspace too small");
      return SWATTN_EWORKSPACE;
    }
    if (!aligned256(workspace)) return invalid(std::string(name) + ": workspace must be 256-byte aligned");
  }
  // Masks of up to kWholeBytes (kWholeUnaligned positions where 16-byte loads
  // cannot be used) go through one kernel whose blocks each read all of it;
  // beyond that those reads take longer than a second launch.
  const bool vec = aligned16(src.p);
  if (vec ? n * 16 <= kWholeBytes * Src::kPer : n <= kWholeUnaligned) {
    const dim3 grid(static_cast<uint32_t>(ceil_div(n, kWholeChunk)));
    const auto kernel = host_blocks != nullptr
                            ? (vec ? compact_whole_kernel<Src, true, true> : compact_whole_kernel<Src, false, true>)
                            : (vec ? compact_whole_kernel<Src, true, false> : compact_whole_kernel<Src, false, false>);
    if (host_blocks != nullptr) *host_blocks = static_cast<int>(grid.x);
    hipLaunchKernelGGL(kernel, grid, dim3(kCompactThreads), 0, st, src, n, indices, counts);
  } else {
    int32_t* bc = static_cast<int32_t*>(workspace);
    hipLaunchKernelGGL(compact_count_kernel<Src>, dim3(nb), dim3(kCompactThreads), 0, st, src, n,
                       bc);
    hipLaunchKernelGGL(compact_scatter_kernel<Src>, dim3(nb), dim3(kCompactThreads), 0, st, src,
                       n, static_cast<const int32_t*>(bc), static_cast<int>(nb), indices, counts);
  }
  return launch_status(name);
}

}  // namespace
}  // namespace swattn
