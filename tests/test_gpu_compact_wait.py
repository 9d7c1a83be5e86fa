"""What the compaction promises when it returns: the lists are complete for
any stream, whatever was queued before it, from any host thread, and a call
that failed leaves nothing behind for the next.  Integers: exact."""

from __future__ import annotations

import ctypes
import os
import threading

import pytest
import torch

from switchattentionkernels_amd import (build_switch_query_indices,
                                        build_switch_query_indices_from_logits)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _mask(seed, n, p=0.3):
    return torch.rand(n, generator=torch.Generator().manual_seed(seed)) < p


def _expect(mask):
    return mask.nonzero().flatten().int(), (~mask).nonzero().flatten().int()


def _queue_work(ms=3):
    """Several ms of matrix products on the current stream."""
    a = torch.randn(4096, 4096, device=DEV).bfloat16()
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    torch.mm(a, a)
    start.record()
    torch.mm(a, a)
    end.record()
    end.synchronize()
    for _ in range(int(ms / max(start.elapsed_time(end), 1e-3)) + 1):
        torch.mm(a, a)


# One block, several blocks, the most blocks that report by themselves, and the
# two-kernel path.
SIZES = (1000, 4096, 20000, 262144, 300000)


@pytest.mark.parametrize("n", SIZES)
def test_lists_are_complete_for_another_stream(n):
    """Lists made on one stream and read on another with no event between."""
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    masks = [_mask(s, n, 0.1 + 0.2 * s) for s in range(4)]
    want = [_expect(m) for m in masks]
    dev = [m.to(DEV) for m in masks]
    torch.cuda.synchronize()
    got = []
    for i in range(60):
        with torch.cuda.stream(a):
            full, local = build_switch_query_indices(dev[i % 4])
        with torch.cuda.stream(b):
            got.append((i % 4, full.clone(), local.clone()))
        b.synchronize()   # the lists' memory is reused by the next pass on stream a
    for i, full, local in got:
        assert torch.equal(full.cpu(), want[i][0]) and torch.equal(local.cpu(), want[i][1])


@pytest.mark.parametrize("n", SIZES)
def test_work_queued_before(n):
    """More work before the compaction than it polls for."""
    mask = _mask(n, n)
    dev = mask.to(DEV)
    for _ in range(3):
        _queue_work()
        full, local = build_switch_query_indices(dev)
        want = _expect(mask)
        assert torch.equal(full.cpu(), want[0]) and torch.equal(local.cpu(), want[1])


def test_two_threads():
    errors = []

    def work(seed):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for i in range(150):
                    n = SIZES[(i + seed) % len(SIZES)]
                    mask = _mask(1000 * seed + i % 7, n, 0.1 + 0.1 * (i % 7))
                    logits = torch.where(mask, 1.0, -1.0)
                    full, local = (build_switch_query_indices_from_logits(logits.to(DEV)) if i % 2
                                   else build_switch_query_indices(mask.to(DEV)))
                    want = _expect(mask)
                    assert torch.equal(full.cpu(), want[0]), (seed, i)
                    assert torch.equal(local.cpu(), want[1]), (seed, i)
        except BaseException as e:   # noqa: BLE001  -- reported by the test's thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("n", SIZES)
def test_failed_call_leaves_the_next_alone(n):
    """An error that another HIP call of this thread left pending fails the
    compaction although its kernel is queued.  The next call, made while that
    kernel still waits behind other work, must not take its counts."""
    first, second = _mask(1, n, 0.9), _mask(2, n, 0.2)
    f_dev, s_dev = first.to(DEV), second.to(DEV)
    want = _expect(second)
    a = torch.randn(2048, 2048, device=DEV).bfloat16()
    build_switch_query_indices(s_dev)
    hip = ctypes.CDLL(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))
    wrong = []
    for i in range(60):
        torch.cuda.synchronize()
        for _ in range(1 + i % 20):   # the queued kernel starts at another time in each pass
            torch.mm(a, a)
        assert hip.hipSetDevice(9999) != 0
        failed = False
        try:
            build_switch_query_indices(f_dev)
        except RuntimeError:
            failed = True
        full, local = build_switch_query_indices(s_dev)
        assert failed
        if full.numel() != want[0].numel():
            wrong.append((i, full.numel()))
        else:
            assert torch.equal(full.cpu(), want[0]) and torch.equal(local.cpu(), want[1])
    assert not wrong, (want[0].numel(), wrong)


@pytest.mark.parametrize("n", [0, 5000, 300000])
def test_capture_is_refused(n):
    """A call under capture raises and leaves the capture as it was."""
    mask = _mask(3, n)
    dev = mask.to(DEV)
    x = torch.zeros(8, device=DEV)
    build_switch_query_indices(dev)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1)
        with pytest.raises(RuntimeError, match="captur"):
            build_switch_query_indices(dev)
    for _ in range(3):
        graph.replay()
    full, local = build_switch_query_indices(dev)
    want = _expect(mask)
    assert torch.equal(full.cpu(), want[0]) and torch.equal(local.cpu(), want[1])
    assert x.tolist() == [3.0] * 8
