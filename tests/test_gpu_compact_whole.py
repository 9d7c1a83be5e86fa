"""Compaction sizes at which the kernels change: the edges of a wave's groups,
of a block's 4096 positions, of the one-launch limits (256 KiB of mask or
logits, 65536 unaligned positions), each on aligned and unaligned inputs, bit
for bit against torch."""

from __future__ import annotations

import pytest
import torch

from switchattentionkernels_amd import (build_switch_query_indices,
                                        build_switch_query_indices_from_logits)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype,sizes", [
    (torch.bool, (1, 63, 64, 65, 4095, 4096, 4097, 65536, 65537, 262144, 262145)),
    (torch.float32, (1, 4095, 4097, 16387, 65536, 65537)),
    (torch.bfloat16, (7, 4097, 65535, 131072, 131073)),
    (torch.float16, (9, 4096, 65537, 131071, 131073))])
def test_compact_sizes(dtype, sizes, offset):
    gen = torch.Generator().manual_seed(offset)
    for n in sizes:
        x = torch.randn(n + offset, generator=gen)
        x[::7] = float("nan")   # never full
        for shift in (0.0, 100.0, -100.0):   # mixed, all but the NaNs full, none full
            y = x + shift
            t = (y > 0.5 if dtype == torch.bool else y.to(dtype)).to(DEV)[offset:]
            if dtype == torch.bool:
                full, local = build_switch_query_indices(t)
                mask = t
            else:
                full, local = build_switch_query_indices_from_logits(t, 0.5)
                mask = t > 0.5
            assert torch.equal(full, mask.nonzero().flatten().int()), (n, shift)
            assert torch.equal(local, (~mask).nonzero().flatten().int()), (n, shift)
