// Entry points of libswattn.so for the package's own Python layer: not part of
// the public C ABI (include/swattn.h), whose conventions they follow.
#pragma once

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * swattn_compact (dtype -1: x is a byte mask) or swattn_compact_logits, waiting
 * for the result: on return the lists are complete, for any stream, and host[0]
 * and host[1] hold the counts.
 *   host  SWATTN_COMPACT_HOST_WORDS int32 of pinned host memory, one call at a
 *         time.  The kernel reports there; a device copy of the counts and a
 *         stream synchronisation would take about 8 us more.  After a HIP error
 *         (a positive status) the stream was synchronised if it could be; if not,
 *         a kernel may report later, so that host is not to be used again.
 * A stream under capture is refused (SWATTN_EINVAL) before anything is launched.
 */
#define SWATTN_COMPACT_HOST_WORDS 66
int swattn_compact_wait(const void* x, int32_t dtype, int64_t n, float threshold, int32_t* indices,
                        int32_t* host, void* workspace, size_t workspace_bytes, void* stream);

/*
 * swattn_build_metadata with the offsets in host memory (read before the call
 * returns, so that no device copy of them is needed), for up to
 * SWATTN_METADATA_HOST_MAX_SEQS sequences.  They must be ascending and end at
 * the totals, as for swattn_build_metadata.
 */
#define SWATTN_METADATA_HOST_MAX_SEQS 256
int swattn_build_metadata_host(const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                               int32_t num_seqs, int64_t total_q, int64_t total_kv, int32_t window,
                               int32_t* q_positions, int32_t* kv_positions,
                               int32_t* q_segment_ids, int32_t* kv_segment_ids,
                               int32_t* full_starts, int32_t* local_starts, int32_t* causal_ends,
                               void* stream);

/*
 * Whether each list's key bounds are non-decreasing along the list, which
 * swattn_prefill_bwd needs of caller-supplied bounds; no counterpart in the
 * reference, which is forward-only.  A start past its row's end counts as the
 * end.  full / local as swattn_check_indices, bounds per query row as
 * swattn_prefill_fwd.
 *   flags  1 int32 output: 0 if both lists' bounds are (and every listed
 *          position lies in [0, total_q)), 1 otherwise.
 */
int swattn_check_bounds(const int32_t* full, int64_t n_full, const int32_t* local, int64_t n_local,
                        const int32_t* full_starts, const int32_t* local_starts,
                        const int32_t* causal_ends, int64_t total_q, int32_t* flags,
                        void* stream);

#ifdef __cplusplus
}  // extern "C"
#endif
