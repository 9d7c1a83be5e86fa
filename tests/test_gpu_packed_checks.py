"""Packed sequences: metadata around the number of sequences whose offsets
travel as kernel arguments (256), with empty sequences and separate key
offsets, and the bounds check of the backward against its definition in
torch.  Integers: exact."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import routing as R
from switchattentionkernels_amd import _lib, build_switch_attention_metadata

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("same", [True, False])
@pytest.mark.parametrize("nseq", [1, 2, 255, 256, 257, 600])
def test_metadata_sequence_counts(nseq, same):
    rng = np.random.default_rng(nseq)

    def offsets():
        lens = rng.integers(0, 9, nseq)
        lens[-1] += 1
        return [0] + np.cumsum(lens).tolist()

    cq = offsets()
    ck = cq if same else offsets()
    md = build_switch_attention_metadata(cq[-1], ck[-1], device=DEV, window_size=3, cu_seqlens=cq,
                                         cu_seqlens_kv=None if same else ck)
    ref = R.varlen_metadata(cq, ck, 3)
    for name, want in ref.items():
        got = getattr(md, name)
        assert got.is_contiguous() and np.array_equal(got.cpu().numpy(), want), name


@pytest.mark.parametrize("nf,nl,fault", [
    (0, 1, None), (1, 0, None), (257, 300, None), (64, 65, "full_end"), (1000, 513, "full_start"),
    (2, 256, "local_start"), (256, 2, "local_end"), (300, 300, "empty_start"),
    (300, 300, "range"), (0, 1, "range"), (1, 1, "range"), (300, 1, "range")])
def test_check_bounds(nf, nl, fault):
    n = nf + nl
    gen = torch.Generator().manual_seed(n)
    perm = torch.randperm(n, generator=gen)
    full, local = perm[:nf].sort().values.int(), perm[nf:].sort().values.int()
    ends = torch.arange(1, n + 1, dtype=torch.int32)
    fs, ls = torch.zeros(n, dtype=torch.int32), (ends - 5).clamp_min(0)
    if fault == "full_end":
        ends[full[-1]] = 0
    elif fault == "full_start":
        fs[full[nf // 2]] = 3                 # the next full row starts at 0 again
    elif fault == "local_start":
        ls[local[0]] = ends[local[0]]
        ls[local[1]] = 0
    elif fault == "local_end":
        ends[local[0]] = n + 7
    elif fault == "empty_start":              # a start past its row's end counts as the end: fine
        ls[local[10]] = n + 100
        ends[local[10]], ends[local[11]] = 4, max(4, int(ends[local[11]]))
        ls[local[11]:] = ls[local[11]:].clamp_min(4)
        ls[local[:10].long()] = 0
        ends[local[:10].long()] = torch.arange(10, dtype=torch.int32).clamp_max(4)
    if fault == "range":
        local[-1] = n
        want = True
    else:
        want = False
        for lst, st in ((full, fs), (local, ls)):
            li = lst.long()
            e = ends[li]
            for b in (torch.minimum(st[li], e), e):
                want |= bool((b[1:] < b[:-1]).any())
        assert want == (fault in ("full_end", "full_start", "local_start", "local_end"))
    d = [t.to(DEV) for t in (full, local, fs, ls, ends)]
    flags = torch.full((1,), 7, dtype=torch.int32, device=DEV)
    st = _lib.lib().swattn_check_bounds(d[0].data_ptr(), nf, d[1].data_ptr(), nl, d[2].data_ptr(),
                                        d[3].data_ptr(), d[4].data_ptr(), n, flags.data_ptr(),
                                        _lib.stream_handle(DEV))
    assert st == 0 and bool(flags.item()) == want
