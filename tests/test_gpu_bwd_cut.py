"""Which (key tile, KV head) pairs the backward cuts, and where their shares run.

A share of a cut pair leaves 256 KiB of fp32 partials at its workgroup's place
in the workspace; pairs left whole write none.  The tests call the C ABI with a
workspace filled with one pattern and read from the partials which workgroups
were shares, so they see the path as well as the result.  Gradients: the bars
of test_gpu_backward against the oracle, and 2e-3 (relative L2) between sums
of the same terms in another order, as the 64-key and the eight-wave kernels.
"""

from __future__ import annotations

import pytest
import torch

from switchattentionkernels_amd import (_lib, build_switch_attention_metadata,
                                        build_switch_query_indices, switch_gqa_prefill_backward,
                                        switch_gqa_prefill_forward)

from test_gpu_backward import _grad_close, _oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
LOG2E = 1.4426950408889634


def _problem(b, s, hq, hkv, mask, window, skv=None, cu=None):
    gen = torch.Generator().manual_seed(s + hq)
    skv = s if skv is None else skv
    q, do = (torch.randn(b, s, hq, 128, generator=gen).bfloat16().to(DEV) for _ in range(2))
    k, v = (torch.randn(b, skv, hkv, 128, generator=gen).bfloat16().to(DEV) for _ in range(2))
    md = None if cu is None else build_switch_attention_metadata(s, s, device=DEV,
                                                                 window_size=window, cu_seqlens=cu)
    full, local = build_switch_query_indices(mask.to(DEV))
    o, lse = switch_gqa_prefill_forward(q, k, v, full, local, metadata=md, window_size=window)
    return q, k, v, do, o, lse, full, local, md


def _backward(problem, window):
    """(dq, dk, dv) through the C ABI and, per share slot of the dK/dV grid
    ([slots, pairs]), whether a share wrote its partials there."""
    q, k, v, do, o, lse, full, local, md = problem
    b, s, hq, _ = q.shape
    skv, hkv = k.shape[1:3]
    L = _lib.lib()
    shape = (b, skv, hq, hkv, 128, window, full.numel(), local.numel())
    need = L.swattn_prefill_bwd_workspace_bytes(*shape)
    ws = torch.full((need // 4,), -1, dtype=torch.int32, device=DEV)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    bounds = [None] * 3 if md is None else [t.data_ptr() for t in (md.full_starts, md.local_starts,
                                                                   md.causal_ends)]
    st = L.swattn_prefill_bwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), do.data_ptr(),
        full.data_ptr(), full.numel(), local.data_ptr(), local.numel(), *bounds, dq.data_ptr(),
        dk.data_ptr(), dv.data_ptr(), b, s, skv, hq, hkv, 128, window, 128 ** -0.5 * LOG2E,
        ws.data_ptr(), need, _lib.stream_handle(DEV))
    assert st == 0, L.swattn_last_error()
    # 1 KiB of row info per 32-row block, a 256-byte zero row and the block
    # ranges come before the partials.
    tiles, g = -(-b * skv // 256), hq // hkv
    pairs = tiles * hkv
    slots = min(16, -(-512 // pairs))
    blocks = hkv * sum(-(-n.numel() * g // 32) for n in (full, local))
    start = blocks * 1024 + 256 + -(-(2 * tiles * 2 * 4) // 256) * 256
    part = ws[start // 4:start // 4 + slots * pairs * 65536].view(slots, pairs, 65536)
    return (dq, dk, dv), (part[:, :, :1024] != -1).any(-1).cpu()


def test_shares_of_recurring_long_pairs_spread_over_the_xcds():
    """Four sequences whose last key tile straddles the next sequence and is
    seen by far more row blocks than the rest (late rows without keys): the
    long pairs recur every fourth tile, with two KV heads every eighth
    workgroup.  Their shares must not all run on the same XCDs (workgroup i
    runs on XCD i % 8)."""
    mask = torch.zeros(4, 8000, dtype=torch.bool)
    mask[:, 7200:] = True
    problem = _problem(4, 8000, 8, 2, mask, 318, skv=963)
    _, shares = _backward(problem, 318)
    per_xcd = shares.reshape(-1, 8).sum(0)
    print("[cut] shares per XCD", per_xcd.tolist(), flush=True)
    assert int(shares.sum()) >= 32
    assert int(per_xcd.max()) <= 1.5 * int(shares.sum()) / 8


