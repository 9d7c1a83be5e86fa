"""What the native host path keeps of the calls' behaviour in Python: the type
of a tensor subclass, torch's out-of-memory error, torch's synchronization
debug mode, and metadata fields that are tensors of their own."""

from __future__ import annotations

import pytest
import torch

from switchattentionkernels_amd import (build_switch_attention_metadata,
                                        build_switch_query_indices,
                                        build_switch_query_indices_from_logits,
                                        switch_gqa_decode_forward, switch_gqa_prefill_backward,
                                        switch_gqa_prefill_forward)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


class Tagged(torch.Tensor):
    pass


def _qkv(s=200, hq=8, hkv=2):
    return [torch.randn(1, s, h, 128, device=DEV).bfloat16() for h in (hq, hkv, hkv)]


def _lists(s=200):
    return build_switch_query_indices(torch.arange(s, device=DEV) % 3 == 0)


def test_subclasses_come_back():
    """Outputs are made like the tensors they belong to, as torch.empty_like makes them."""
    q, k, v = _qkv()
    full, local = _lists()
    tq, tk = q.as_subclass(Tagged), k.as_subclass(Tagged)
    o, lse = switch_gqa_prefill_forward(q, k, v, full, local, window_size=50)
    to, tlse = switch_gqa_prefill_forward(tq, tk, v, full, local, window_size=50)
    assert type(o) is torch.Tensor and type(to) is Tagged
    assert type(lse) is torch.Tensor and type(tlse) is torch.Tensor
    assert torch.equal(o, to.as_subclass(torch.Tensor)) and torch.equal(lse, tlse)
    want = switch_gqa_prefill_backward(q, k, v, o, lse, q, full, local, window_size=50)
    got = switch_gqa_prefill_backward(tq, tk, v, o, lse, q, full, local, window_size=50)
    assert [type(t) for t in got] == [Tagged, Tagged, torch.Tensor]
    for a, b in zip(want, got):
        assert torch.equal(a, b.as_subclass(torch.Tensor))
    lens = torch.tensor([200], dtype=torch.int32, device=DEV)
    route = torch.ones(1, dtype=torch.bool, device=DEV)
    for qd in (q[:, -1:].contiguous(), q[:, -1].contiguous()):
        o, _ = switch_gqa_decode_forward(qd, k, v, lens, route)
        to, _ = switch_gqa_decode_forward(qd.as_subclass(Tagged), k, v, lens, route)
        assert type(to) is Tagged and torch.equal(o, to.as_subclass(torch.Tensor))


def test_out_of_memory_is_torchs_error():
    q, k, v = _qkv(s=65536, hq=8, hkv=8)   # 128 MiB each
    full, local = _lists(65536)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 2 ** 20) / total)
    held = []
    try:
        while True:   # what earlier tests left free inside the reserved segments
            try:
                held.append(torch.empty(2 ** 25, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                break
        with pytest.raises(torch.OutOfMemoryError):
            switch_gqa_prefill_forward(q, k, v, full, local)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        held.clear()
    o, _ = switch_gqa_prefill_forward(q, k, v, full, local)
    assert bool(torch.isfinite(o).all())


@pytest.mark.parametrize("make", [
    lambda m: build_switch_query_indices(m),
    lambda m: build_switch_query_indices_from_logits(m.float(), 0.5)])
def test_sync_debug_mode_sees_the_wait(make):
    mask = torch.arange(5000, device=DEV) % 3 == 0
    make(mask)
    try:
        torch.cuda.set_sync_debug_mode("error")
        with pytest.raises(RuntimeError, match="synchroniz"):
            make(mask)
        torch.cuda.set_sync_debug_mode("warn")
        with pytest.warns(UserWarning, match="synchroniz"):
            full, local = make(mask)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    assert full.numel() == 1667 and local.numel() == 3333


@pytest.mark.parametrize("nseq", [1, 7, 256, 257])
@pytest.mark.parametrize("extra", [0, 3])
def test_metadata_fields_are_tensors_of_their_own(nseq, extra):
    """Whole storages, aligned as torch allocates, with version counters of their own."""
    n = 5 * nseq + 2
    cu = [5 * i for i in range(nseq)] + [n]
    ck = cu[:-1] + [n + extra]
    md = build_switch_attention_metadata(n, n + extra, device=DEV, window_size=3, cu_seqlens=cu,
                                         cu_seqlens_kv=ck)
    fields = (md.q_positions, md.kv_positions, md.q_segment_ids, md.kv_segment_ids,
              md.full_starts, md.local_starts, md.causal_ends)
    assert len({t.untyped_storage().data_ptr() for t in fields}) == 7
    for t in fields:
        assert t.data_ptr() % 256 == 0 and t.storage_offset() == 0
        assert t.untyped_storage().nbytes() == 4 * t.numel()
    before = [t._version for t in fields]
    md.causal_ends.add_(0)
    assert [t._version for t in fields] == before[:-1] + [before[-1] + 1]
