"""The backward's one grid for dK/dV and dQ: which pairs and row tiles are cut.

Shapes sit on both sides of every rule: pairs that stay whole, pairs cut into a
few and into the most shares, 512 pairs (never cut), a KV-head count that is
no multiple of the XCDs, several sequences of whole and of partial key tiles,
one list empty.  Compared with the fp32 oracle at the backward's bars
(relative L2 1e-2, largest error 3e-2 of the largest gradient), and rerun bit
for bit.
"""

from __future__ import annotations

import pytest
import torch

import oracle
from switchattentionkernels_amd import (build_switch_query_indices, switch_gqa_prefill_backward,
                                        switch_gqa_prefill_forward)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("b,s,hq,hkv,w,p", [
    (1, 1, 2, 1, 4, 1.0), (1, 255, 4, 1, 64, 0.5), (1, 257, 3, 3, 100, 0.5),
    (1, 1500, 8, 2, 128, 0.3), (2, 512, 4, 2, 100, 0.0), (2, 512, 4, 2, 100, 1.0),
    (3, 500, 10, 2, 700, 0.6), (1, 2048, 4, 4, 256, 0.25), (4, 256, 128, 128, 64, 0.4),
    (1, 3000, 2, 1, 64, 0.9)])
def test_backward_grid(b, s, hq, hkv, w, p):
    gen = torch.Generator().manual_seed(s + hq)
    q, do = (torch.randn(b, s, hq, 128, generator=gen).bfloat16() for _ in range(2))
    k, v = (torch.randn(b, s, hkv, 128, generator=gen).bfloat16() for _ in range(2))
    mask = torch.rand(b, s, generator=gen) < p
    print(f"[bwd grid] B{b} S{s} {hq}/{hkv} W{w} p{p}", flush=True)
    fi, li = build_switch_query_indices(mask.to(DEV))
    dev = [t.to(DEV) for t in (q, k, v, do)]
    o, lse = switch_gqa_prefill_forward(*dev[:3], fi, li, window_size=w)
    got = switch_gqa_prefill_backward(*dev[:3], o, lse, dev[3], fi, li, window_size=w)
    again = switch_gqa_prefill_backward(*dev[:3], o, lse, dev[3], fi, li, window_size=w)
    for x, y in zip(got, again):
        assert torch.equal(x, y)
    ref = oracle.routed_attention_backward(q, k, v, do, fi.cpu(), li.cpu(), window_size=w,
                                           out=o.float().cpu())
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        g, r = g.float().cpu(), r.float()
        if float(r.abs().max()) < 1e-3:   # a row that sees one key: zero in exact arithmetic
            assert float(g.abs().max()) <= 1e-2, name
            continue
        assert float((g - r).norm() / r.norm()) <= 1e-2, name
        assert float((g - r).abs().max()) <= 3e-2 * float(r.abs().max()), name
