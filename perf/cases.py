"""Performance cases of the routed attention framework.

Every case is one call sequence that a program using this package makes, from
the router's output to the finished tensors, through the package's public
entry points (``switchattentionkernels_amd/__init__.py``):

* ``prefill``: a serving prefill of one attention layer.  The router's bool
  mask is compacted (``build_switch_query_indices``) and the routed attention
  runs (``switch_gqa_prefill_forward``, or ``switch_gqa_prefill_varlen_forward``
  for packed sequences).  Returns the output and the log2 LSE.
* ``train``: one attention layer of a training step.  Router logits are
  thresholded and compacted (``build_switch_query_indices_from_logits``), the
  forward runs under autograd (``switch_gqa_prefill`` /
  ``switch_gqa_prefill_varlen``) and the gradients of q, k and v follow.
* ``decode``: one routed decode step over a batch of KV caches
  (``switch_gqa_decode_forward``).

head_dim is 128 throughout (the kernels' only one) and all row tensors are
bf16.  Sizes come from ``switchattentionkernels_amd/workloads.py`` and
``bench.py`` or are generic.  The module gives, per case, its inputs, one pass,
the work that the pass cannot do without, the tolerance of its outputs, and a
plain 64-bit evaluation that shares no code with the package.
"""

from __future__ import annotations

import math
import random
import statistics

import torch

import switchattentionkernels_amd as swa

D = 128


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _attention(kind, batch, seq, heads_q, heads_kv, window, p_full, routing="bernoulli",
               nseq=0, len_lo=0, len_hi=0, len_seed=0):
    """``nseq`` > 0: that many packed sequences with lengths uniform in
    ``[len_lo, len_hi]`` drawn from ``len_seed`` (``batch`` 1, ``seq`` unused)."""
    return {"kind": kind, "batch": batch, "seq": seq, "heads_q": heads_q, "heads_kv": heads_kv,
            "window": window, "p_full": p_full, "routing": routing, "nseq": nseq,
            "len_lo": len_lo, "len_hi": len_hi, "len_seed": len_seed}


def _decode(batch, cache, heads_q, heads_kv, window, p_full):
    return {"kind": "decode", "batch": batch, "cache": cache, "heads_q": heads_q,
            "heads_kv": heads_kv, "window": window, "p_full": p_full}


def listed():
    return [
        # A short prompt on a small layer: the smallest prefill, where launches,
        # the list read-back and the longest row's chain of keys count.
        dict(_attention("prefill", 1, 1024, 8, 2, 256, 0.25), name="prefill_s1024"),
        # An ordinary chat-length prompt whose length is no multiple of any tile,
        # five query heads per KV head, half of the tokens routed full.
        dict(_attention("prefill", 1, 2999, 40, 8, 512, 0.5), name="prefill_ragged_s2999"),
        # A small batch of ordinary prompts.
        dict(_attention("prefill", 2, 4096, 32, 8, 1024, 0.25), name="prefill_b2_s4096"),
        # Long-context prefill: the benchmark's shape.
        dict(_attention("prefill", 1, 16384, 32, 8, 1024, 0.25), name="prefill_s16k"),
        # Continuous-batching prefill: packed sequences of mixed lengths, eight
        # query heads per KV head, clustered routing, metadata built per call.
        dict(_attention("prefill", 1, 0, 64, 8, 2048, 0.3, "markov", 8, 512, 8192, 1),
             name="prefill_varlen"),
        # A very long document, full routing rising towards its end: the largest.
        dict(_attention("prefill", 1, 65536, 40, 8, 4096, 0.15, "ramp"), name="prefill_s64k"),
        # Training on short sequences with a small layer: the smallest step.
        dict(_attention("train", 1, 1024, 8, 2, 256, 0.25), name="train_s1024"),
        # Training at an ordinary sequence length.
        dict(_attention("train", 2, 4096, 32, 8, 1024, 0.25), name="train_b2_s4096"),
        # Long-context training.
        dict(_attention("train", 1, 16384, 32, 8, 1024, 0.25), name="train_s16k"),
        # One GPU's share of the long-context layer when its KV heads are split
        # over eight GPUs: few heads, long chains of keys.
        dict(_attention("train", 1, 16384, 4, 1, 1024, 0.25), name="train_kvh1_s16k"),
        # A serving batch in decode: mixed cache lengths and routes.
        dict(_decode(64, 8192, 32, 8, 1024, 0.25), name="decode_b64_l8192"),
        # One user's decode step: the smallest call of all, latency only.
        dict(_decode(1, 4096, 32, 8, 1024, 1.0), name="decode_b1_l4096"),
    ]


_HEADS = [(8, 2), (32, 8), (40, 8), (64, 8), (4, 1)]
_MAX_FLOPS = {"prefill": 4.0e12, "train": 6.0e12}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["prefill", "prefill", "train", "train", "decode"])
    heads_q, heads_kv = rng.choice(_HEADS)
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        cache = _log_int(rng, 512, min(32768, 64 * 8192 // batch))
        return _decode(batch, cache, heads_q, heads_kv, _log_int(rng, 256, 4096),
                       rng.choice([0.0, 0.25, 0.5, 1.0]))
    while True:
        window = _log_int(rng, 256, 4096)
        p_full = round(rng.uniform(0.1, 0.5), 2)
        if rng.random() < 0.3:
            nseq = rng.randint(2, 8)
            hi = _log_int(rng, 1024, 8192)
            case = _attention(kind, 1, 0, heads_q, heads_kv, window, p_full, "markov", nseq,
                              hi // 16, hi, rng.randint(0, 10 ** 6))
        else:
            case = _attention(kind, rng.choice([1, 1, 2, 4]), _log_int(rng, 512, 16384), heads_q,
                              heads_kv, window, p_full,
                              rng.choice(["bernoulli", "bernoulli", "markov", "ramp"]))
        if work(case)["flops"] <= _MAX_FLOPS[kind]:
            return case


def _lengths(case):
    """Sequence lengths of an attention case (equal ones for a batch)."""
    if case["nseq"]:
        rng = random.Random(case["len_seed"])
        return [rng.randint(case["len_lo"], case["len_hi"]) for _ in range(case["nseq"])]
    return [case["seq"]] * case["batch"]


# ---------------------------------------------------------------------------
# Inputs and the pass
# ---------------------------------------------------------------------------
def _full_mask(case, gen, dev):
    """Router decisions, one per position of the flattened rows."""
    lens = _lengths(case)
    n, p = sum(lens), case["p_full"]
    u = torch.rand(n, generator=gen, device=dev)
    if case["routing"] == "markov":
        # Keep the previous state with probability 0.95, else redraw it; each
        # sequence starts with a fresh draw.
        fresh = torch.rand(n, generator=gen, device=dev) >= 0.95
        start = 0
        for length in lens:
            fresh[start] = True
            start += length
        pos = torch.arange(n, device=dev)
        last = torch.cummax(torch.where(fresh, pos, torch.zeros_like(pos)), 0).values
        return u[last] < p
    if case["routing"] == "ramp":   # from p/3 at the start to 5p/3 at the end
        ps = torch.cat([torch.linspace(p / 3, 5 * p / 3, length, device=dev) for length in lens])
        return u < ps
    return u < p


def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def rows(*shape):
        return torch.randn(*shape, generator=gen, device=dev).to(torch.bfloat16)

    hq, hkv = case["heads_q"], case["heads_kv"]
    if case["kind"] == "decode":
        b, cache = case["batch"], case["cache"]
        lens = torch.randint(cache // 2, cache + 1, (b,), generator=gen, device=dev,
                             dtype=torch.int32)
        full = torch.rand(b, generator=gen, device=dev) < case["p_full"]
        return {"q": rows(b, 1, hq, D), "k": rows(b, cache, hkv, D), "v": rows(b, cache, hkv, D),
                "lens": lens, "full": full}
    lens = _lengths(case)
    batch = 1 if case["nseq"] else case["batch"]
    seq = sum(lens) // batch
    mask = _full_mask(case, gen, dev).view(batch, seq)
    st = {"q": rows(batch, seq, hq, D), "k": rows(batch, seq, hkv, D),
          "v": rows(batch, seq, hkv, D), "mask": mask, "cu": None}
    if case["nseq"]:
        st["cu"] = [0]
        for length in lens:
            st["cu"].append(st["cu"][-1] + length)
    if case["kind"] == "train":
        # Router logits whose sign is the decision.
        z = torch.randn(batch, seq, generator=gen, device=dev).abs() + 0.01
        st["logits"] = torch.where(mask, z, -z)
        st["grad"] = rows(batch, seq, hq, D)
    return st


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = dict(case)
    if case["kind"] == "train":
        for name in ("q", "k", "v"):
            st[name].requires_grad_()
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "decode":
        return swa.switch_gqa_decode_forward(st["q"], st["k"], st["v"], st["lens"], st["full"],
                                             window_size=case["window"])
    q, k, v, window = st["q"], st["k"], st["v"], case["window"]
    if case["kind"] == "prefill":
        full, local = swa.build_switch_query_indices(st["mask"])
        if st["cu"] is not None:
            return swa.switch_gqa_prefill_varlen_forward(q, k, v, full, local, st["cu"],
                                                         window_size=window)
        return swa.switch_gqa_prefill_forward(q, k, v, full, local, window_size=window)
    full, local = swa.build_switch_query_indices_from_logits(st["logits"])
    if st["cu"] is not None:
        out, lse = swa.switch_gqa_prefill_varlen(q, k, v, full, local, st["cu"],
                                                 window_size=window)
    else:
        out, lse = swa.switch_gqa_prefill(q, k, v, full, local, window_size=window)
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), st["grad"])
    return out.detach(), lse, dq, dk, dv


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------
def _expected_pairs(case):
    """Legal (query position, key) pairs expected from the routing's probabilities."""
    p, w, total = case["p_full"], case["window"], 0.0
    for n in _lengths(case):
        m = min(n, w)
        local = m * (m + 1) / 2 + (n - m) * w
        if case["routing"] == "ramp":   # full with probability p (1/3 + 4/3 i / (n - 1))
            step = 4 / 3 / max(n - 1, 1)
            more = sum((1 / 3 + step * i) * (i + 1 - w) for i in range(m, n))
            total += local + p * more   # a full row sees i + 1 - w keys more than a local one
        else:
            total += local + p * (n * (n + 1) / 2 - local)
    return total


def work(case):
    hq, hkv = case["heads_q"], case["heads_kv"]
    if case["kind"] == "decode":
        b, cache, w, p = case["batch"], case["cache"], case["window"], case["p_full"]
        lo = cache // 2
        mean = (lo + cache) / 2
        local = sum(min(n, w) for n in range(lo, cache + 1)) / (cache - lo + 1)
        keys = b * (p * mean + (1 - p) * local)
        return {"bytes": keys * 2 * hkv * D * 2 + b * hq * (2 * D * 2 + 4) + b * 5,
                "flops": 4 * D * hq * keys}
    rows = sum(_lengths(case))
    flops = 4 * D * hq * _expected_pairs(case)
    io = rows * (2 * hq + 2 * hkv) * D * 2 + rows * hq * 4   # q, out, k, v and the LSE
    if case["kind"] == "prefill":
        return {"bytes": io + rows, "flops": flops}
    # The backward reads dO and writes dq, dk, dv; five products against two.
    return {"bytes": io + rows * (2 * hq + 2 * hkv) * D * 2 + 4 * rows, "flops": 3.5 * flops}


def tolerance(case):
    # bf16 outputs from fp32 sums with bf16 P and dS.  Measured against the
    # 64-bit result over the listed and drawn cases: O 1.6e-3 (decode, whose P
    # stays fp32) to 2.3e-3, gradients 2.3e-3 to 2.5e-3, the LSE 5e-8.
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------
# 64-bit evaluation in plain torch
# ---------------------------------------------------------------------------
def _blocks(positions, size):
    for i in range(0, positions.numel(), size):
        yield positions[i:i + size]


def _exact_attention(st, case, backward):
    hq, hkv, w = case["heads_q"], case["heads_kv"], case["window"]
    g = hq // hkv
    batch, seq = st["q"].shape[:2]
    dev = st["q"].device
    lens = _lengths(case)

    def flat(name, heads):
        return st[name].detach().reshape(batch * seq, heads, D)

    q, k, v = flat("q", hq), flat("k", hkv), flat("v", hkv)
    mask = st["mask"].reshape(-1)
    out = torch.empty(batch * seq, hq, D, dtype=torch.float64, device=dev)
    lse = torch.empty(batch * seq, hq, dtype=torch.float64, device=dev)
    if backward:
        grad = flat("grad", hq)
        dq = torch.empty_like(out)
        dk = torch.zeros(batch * seq, hkv, D, dtype=torch.float64, device=dev)
        dv = torch.zeros_like(dk)
    scale = D ** -0.5
    start = 0

    def grouped(x, idx):   # rows idx as [hkv, rows * g, D] in 64 bits
        n = idx.numel()
        return (x[idx].double().view(n, hkv, g, D).permute(1, 0, 2, 3).reshape(hkv, n * g, D)
                .contiguous())

    def ungrouped(x, n):
        return x.view(hkv, n, g, -1).permute(1, 0, 2, 3).reshape(n, hq, -1)

    for length in lens:
        seg = slice(start, start + length)
        kk = k[seg].double().permute(1, 0, 2).contiguous()    # [hkv, length, D]
        vv = v[seg].double().permute(1, 0, 2).contiguous()
        kt, vt = kk.transpose(1, 2).contiguous(), vv.transpose(1, 2).contiguous()
        routes = mask[seg]
        for is_full in (True, False):
            pos = torch.nonzero(routes if is_full else ~routes).flatten()
            for blk in _blocks(pos, 256 if is_full else 1024):
                n = blk.numel()
                first, last = int(blk[0]), int(blk[-1])
                k0 = 0 if is_full else max(first - w + 1, 0)
                k1 = last + 1
                keys = torch.arange(k0, k1, device=dev)
                legal = keys[None] <= blk[:, None]
                if not is_full:
                    legal &= keys[None] > blk[:, None] - w
                legal = legal.repeat_interleave(g, 0)[None]
                qq = grouped(q, blk + start)
                s = torch.bmm(qq, kt[:, :, k0:k1].contiguous()).mul_(scale)
                s.masked_fill_(~legal, -math.inf)
                m = s.amax(-1, keepdim=True)
                p = s.sub_(m).exp_()
                z = p.sum(-1, keepdim=True)
                p.div_(z)
                o = torch.bmm(p, vv[:, k0:k1].contiguous())
                out[blk + start] = ungrouped(o, n)
                lse[blk + start] = ungrouped((m + z.log()) / math.log(2.0), n)[..., 0]
                if backward:
                    do = grouped(grad, blk + start)
                    dp = torch.bmm(do, vt[:, :, k0:k1].contiguous())
                    ds = dp.sub_((do * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                    dq[blk + start] = ungrouped(torch.bmm(ds, kk[:, k0:k1].contiguous()), n)
                    a, b = start + k0, start + k1
                    dk[a:b] += torch.bmm(ds.transpose(1, 2).contiguous(), qq).permute(1, 0, 2)
                    dv[a:b] += torch.bmm(p.transpose(1, 2).contiguous(), do).permute(1, 0, 2)
        start += length
    shape = (batch, seq)
    res = [out.view(*shape, hq, D), lse.view(*shape, hq)]
    if backward:
        res += [dq.view(*shape, hq, D), dk.view(*shape, hkv, D), dv.view(*shape, hkv, D)]
    return tuple(res)


def exact(case, seed):
    st = _inputs(case, seed)
    if case["kind"] != "decode":
        return _exact_attention(st, case, case["kind"] == "train")
    hq, hkv = case["heads_q"], case["heads_kv"]
    g = hq // hkv
    out = torch.empty(st["q"].shape, dtype=torch.float64, device=st["q"].device)
    lse = torch.empty(st["q"].shape[:3], dtype=torch.float64, device=st["q"].device)
    for b, (n, full) in enumerate(zip(st["lens"].tolist(), st["full"].tolist())):
        lo = 0 if full else max(n - case["window"], 0)
        q = st["q"][b, 0].double().view(hkv, g, D)
        k = st["k"][b, lo:n].double().permute(1, 2, 0).contiguous()
        v = st["v"][b, lo:n].double().permute(1, 0, 2).contiguous()
        s = torch.bmm(q, k) * D ** -0.5
        out[b, 0] = torch.bmm(torch.softmax(s, -1), v).reshape(hq, D)
        lse[b, 0] = (torch.logsumexp(s, -1) / math.log(2.0)).reshape(hq)
    return out, lse
