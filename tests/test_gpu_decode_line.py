"""The decode's work split: the line of routed keys and its shares.

Cases sit where the plan can go wrong: the batch sizes at which a thread
plans one or several sequences and at which the plan kernel takes over, empty
sequences at the ends and in between, pairs that fill a share exactly, and
both layouts (few long pairs, many short ones).  Tolerances are the parity
bars of the decode tests: O within 2e-2 / 2e-3 mean, LSE 1e-3 relative.
"""

from __future__ import annotations

import pytest
import torch

import oracle
from switchattentionkernels_amd import _lib, switch_gqa_decode_forward

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _lens(kind: str, batch: int, cache: int, gen: torch.Generator) -> torch.Tensor:
    if kind == "whole":
        return torch.full((batch,), cache, dtype=torch.int32)
    lens = torch.randint(0, cache + 1, (batch,), generator=gen, dtype=torch.int32)
    if kind == "holes":   # empty at both ends and in runs
        lens[::3] = 0
        lens[-1] = 0
    if kind == "one":     # a single sequence with keys
        lens[:] = 0
        lens[batch // 2] = cache
    return lens


@pytest.mark.parametrize("batch,cache,hq,hkv,w,p,kind", [
    (1, 1, 8, 1, 5, 1.0, "whole"), (1, 128, 4, 4, 64, 1.0, "whole"),
    (1, 4096, 8, 2, 256, 1.0, "whole"), (3, 4097, 8, 1, 1, 0.5, "random"),
    (2, 130, 5, 1, 17, 0.0, "random"), (64, 1024, 8, 8, 1024, 0.0, "whole"),
    (255, 70, 4, 2, 33, 0.5, "holes"), (256, 70, 3, 1, 33, 0.5, "random"),
    (257, 70, 7, 1, 33, 0.5, "one"), (700, 40, 6, 2, 16, 0.3, "holes"),
    (1024, 40, 2, 1, 16, 0.5, "random"), (1025, 40, 2, 1, 16, 0.5, "holes"),
    (1025, 600, 1, 1, 64, 1.0, "one"), (16, 6000, 4, 2, 700, 0.5, "random"),
    (5, 300, 8, 2, 64, 0.5, "empty"), (1500, 300, 2, 1, 64, 0.5, "empty")])
def test_decode_line(batch, cache, hq, hkv, w, p, kind):
    gen = torch.Generator().manual_seed(batch * 7 + cache)
    q = torch.randn(batch, 1, hq, 128, generator=gen).bfloat16()
    k = torch.randn(batch, cache, hkv, 128, generator=gen).bfloat16()
    v = torch.randn(batch, cache, hkv, 128, generator=gen).bfloat16()
    lens = (torch.zeros(batch, dtype=torch.int32) if kind == "empty"
            else _lens(kind, batch, cache, gen))
    full = torch.rand(batch, generator=gen) < p
    print(f"[decode line] B{batch} L{cache} {hq}/{hkv} W{w} {kind}", flush=True)
    o, lse = switch_gqa_decode_forward(q.to(DEV), k.to(DEV), v.to(DEV), lens.to(DEV),
                                       full.to(DEV), window_size=w)
    o_r, lse_r = oracle.decode_attention(q[:, 0], k, v, lens.tolist(), full.tolist(),
                                         window_size=w)
    o, lse = o[:, 0].float().cpu(), lse[:, 0].cpu()
    o_r, lse_r = o_r.float().view(o.shape), lse_r.view(lse.shape)
    empty = lens == 0
    assert bool(torch.isnan(o[empty]).all()) and bool((lse[empty] == -torch.inf).all())
    live = ~empty
    if bool(live.any()):
        d = (o[live] - o_r[live]).abs()
        assert float(d.max()) <= 2e-2 and float(d.mean()) <= 2e-3
        rel = (lse[live] - lse_r[live]).abs() / lse_r[live].abs().clamp_min(1.0)
        assert float(rel.max()) <= 1e-3


@pytest.mark.parametrize("batch,cache", [(3, 1 << 30), (1100, 1 << 22), (2, 2 ** 31 - 1)])
def test_decode_over_a_sparse_address_range(batch, cache):
    """Caches of more than 2^31 rows of address range, of which only the first
    sequence's are there and only they have keys, as a caller that maps its
    cache by need can have through the C ABI: the plan's positions are 64-bit
    for these."""
    hq, hkv, w, n = 8, 2, 100, 300
    gen = torch.Generator().manual_seed(batch)
    q = torch.randn(batch, hq, 128, generator=gen).bfloat16().to(DEV)
    k, v = (torch.randn(1, n, hkv, 128, generator=gen).bfloat16().to(DEV) for _ in range(2))
    full = torch.ones(batch, dtype=torch.bool, device=DEV)
    lens = torch.zeros(batch, dtype=torch.int32, device=DEV)
    lens[0] = n
    assert batch * cache * hkv > 2 ** 31
    L = _lib.lib()
    need = L.swattn_decode_workspace_bytes(batch, cache, hq, hkv)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    o = torch.empty_like(q)
    lse = torch.empty(batch, hq, device=DEV)
    print(f"[decode line] B{batch} L{cache} sparse", flush=True)
    st = L.swattn_decode_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), lens.data_ptr(),
                             full.data_ptr(), o.data_ptr(), lse.data_ptr(), batch, cache, hq, hkv,
                             128, w, 128 ** -0.5 * 1.4426950408889634, ws.data_ptr(), need,
                             _lib.stream_handle(DEV))
    assert st == 0, L.swattn_last_error()
    o_r, lse_r = oracle.decode_attention(q[:1].cpu(), k.cpu(), v.cpu(), [n], [True], window_size=w)
    d = (o[0].float().cpu() - o_r.float().view(hq, 128)).abs()
    assert float(d.max()) <= 2e-2 and float(d.mean()) <= 2e-3
    assert torch.allclose(lse[0].cpu(), lse_r.view(hq), rtol=1e-3)
    assert bool(torch.isnan(o[1:]).all()) and bool((lse[1:] == -torch.inf).all())
