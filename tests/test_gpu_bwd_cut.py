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


def _rows_blocks(cu, group, tiles):
    """Row blocks that see each 256-key tile, every row full: 32-row blocks of
    the rows whose range [sequence start, position] overlaps the tile."""
    rows = [(a, p) for a, e in zip(cu, cu[1:]) for p in range(a, e)]
    out = []
    for t in range(tiles):
        seen = [p for a, p in rows if p >= 256 * t and a < 256 * (t + 1)]
        out.append(-(-(seen[-1] + 1) * group // 32) - seen[0] * group // 32)
    return out


def test_packed_sequences_are_cut_by_what_their_tiles_see():
    """Eight short sequences, every row full: a tile is seen by its own
    sequence's rows only, many fewer than the list lengths allow for.  A
    pair that takes longer than the grid's time per CU must be cut, and the
    gradients are those of the sequences one by one."""
    cu = [0, 300, 700, 1000, 1300, 1500, 1800, 2143, 3564]
    s, hq, hkv, w = cu[-1], 64, 8, 473
    problem = _problem(1, s, hq, hkv, torch.ones(1, s, dtype=torch.bool), w, cu=cu)
    grads, shares = _backward(problem, w)
    n = _rows_blocks(cu, hq // hkv, shares.shape[1] // hkv)
    per_cu = 2.7 * hkv * sum(n) / 256   # us: a row block 1.6, its part of dQ 1.1
    cut = shares.sum(0).view(-1, hkv)   # (8 KV heads: every row holds the pairs in order)
    print("[cut] blocks", n, "time per CU", round(per_cu), "shares", cut[:, 0].tolist(), flush=True)
    for tile, blocks in enumerate(n):
        if 1.6 * blocks > 2 * per_cu:
            assert int(cut[tile].min()) >= 2, (tile, blocks)
        if 1.6 * blocks < 0.5 * per_cu:
            assert int(cut[tile].max()) == 0, (tile, blocks)
    assert int(cut.max()) >= 2
    q, k, v, do, o, lse = problem[:6]
    for a, e in zip(cu, cu[1:]):
        full, local = build_switch_query_indices(torch.ones(1, e - a, dtype=torch.bool, device=DEV))
        one = [t[:, a:e].contiguous() for t in (q, k, v, o, lse, do)]
        ref = switch_gqa_prefill_backward(*one, full, local, window_size=w)
        for name, got, want in zip(("dq", "dk", "dv"), grads, ref):
            g, r = got[:, a:e].float(), want.float()
            assert float((g - r).norm() / r.norm()) <= 2e-3, (name, a)


@pytest.mark.parametrize("b,s,hq,hkv,w,p", [
    (2, 2048, 8, 4, 256, 0.9),      # whole 256-key tiles of two sequences, few shares
    (2, 1792, 16, 2, 200, 0.25),
    (3, 1000, 8, 2, 300, 0.5)])     # tiles that straddle the sequences
def test_cut_pairs_of_several_sequences(b, s, hq, hkv, w, p):
    gen = torch.Generator().manual_seed(b * s)
    mask = torch.rand(b, s, generator=gen) < p
    problem = _problem(b, s, hq, hkv, mask, w)
    grads, shares = _backward(problem, w)
    per_slot = shares.sum(1).tolist()
    print(f"[cut] B{b} S{s} shares per slot, last slot first", per_slot, flush=True)
    assert per_slot[-1] > 0 and per_slot == sorted(per_slot)   # some cut, few of them finely
    assert per_slot[0] < shares.shape[1]
    q, k, v, do = (t.cpu() for t in problem[:4])
    for got, ref, name in zip(grads, _oracle(q, k, v, do, mask, w), ("dq", "dk", "dv")):
        _grad_close(got, ref, f"cut b{b} s{s} {name}")
