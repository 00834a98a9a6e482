"""The work a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values:

``kind``               "forward" (one ``HBSAttention`` call) or "train" (the call and the gradients of q, k and v)
``dtype``              "bf16", "fp16" or "fp32"
``batch``              sequences of the packed batch
``q_lo``, ``q_hi``     their query lengths lie in this range (drawn from the case itself, so a case has fixed sizes)
``k_lo``, ``k_hi``     their key lengths; 0: equal to the query lengths
``hq``, ``hk``, ``d``  query heads, key/value heads, head dim
``qbs``, ``kbs``       block sizes
``keep``               probability that a block of the mask is kept (every kv head has its own mask)
``diag``               the block a q block is aligned with is always kept
``causal``, ``scale``  as in the call (scale ``None``: 1 / sqrt(d))
``metadata``           the block metadata is passed in (as a program that calls more than once does), or left to the call
"""
import math
import random

import numpy as np
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.workloads import make_problem

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def _case(name=None, *, kind="forward", dtype="bf16", batch, q_lo, q_hi, k_lo=0, k_hi=0, hq, hk, d, qbs, kbs, keep, diag=True,
          causal=True, scale=None, metadata=True):
    c = dict(kind=kind, dtype=dtype, batch=batch, q_lo=q_lo, q_hi=q_hi, k_lo=k_lo, k_hi=k_hi, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs,
             keep=keep, diag=diag, causal=causal, scale=scale, metadata=metadata)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # The reference README's worked example, called the way it is shown there: without block metadata.
        # The smallest call; launches and host work are all there is to it.
        _case("readme", batch=5, q_lo=32, q_hi=32, k_lo=23, k_hi=39, hq=8, hk=2, d=32, qbs=32, kbs=16, keep=0.7, diag=False,
              metadata=False),
        # A serving batch of short ragged prompts, grouped-query heads, small blocks: latency and occupancy.
        _case("short prompts", batch=16, q_lo=40, q_hi=500, hq=32, hk=8, d=128, qbs=64, kbs=64, keep=0.5),
        # A head dim between the usual powers of two, ordinary lengths, non-causal (an encoder), fp16.
        _case("head dim 192", dtype="fp16", batch=8, q_lo=1800, q_hi=2300, hq=16, hk=16, d=192, qbs=128, kbs=128, keep=0.3,
              causal=False),
        # One decode step of a ragged serving batch: one query a sequence against its whole key cache, few blocks kept.
        _case("decode", batch=32, q_lo=1, q_hi=1, k_lo=2000, k_hi=32000, hq=32, hk=8, d=128, qbs=16, kbs=64, keep=0.25),
        # Chunked prefill: the next few hundred tokens of two long sequences against everything before them.
        _case("prefill chunk", batch=2, q_lo=300, q_hi=512, k_lo=60000, k_hi=70000, hq=32, hk=8, d=128, qbs=128, kbs=128, keep=0.2),
        # The speed sweep's ordinary length: uniform 8K sequences, 90 % sparse (workload C2).
        _case("prefill 8K", batch=8, q_lo=8192, q_hi=8192, hq=32, hk=32, d=128, qbs=128, kbs=128, keep=0.1),
        # Ragged prefill with grouped-query heads and unequal blocks (workload C3).
        _case("prefill ragged", batch=8, q_lo=2048, q_hi=16384, hq=32, hk=8, d=128, qbs=64, kbs=128, keep=0.3),
        # Query and key lengths that differ, block sizes that are no powers of two, head dim 64 (workload C5).
        _case("unequal lengths", batch=4, q_lo=777, q_hi=5120, k_lo=4100, k_hi=8192, hq=16, hk=2, d=64, qbs=80, kbs=48, keep=0.5,
              diag=False, scale=0.1),
        # The long end: uniform 32K sequences, 90 % sparse (workload T, the benchmark's default).
        _case("prefill 32K", batch=8, q_lo=32768, q_hi=32768, hq=32, hk=32, d=128, qbs=128, kbs=128, keep=0.1),
        # A training step's attention at the sweep's ordinary shape: forward, then the gradients.
        _case("train 8K", kind="train", batch=4, q_lo=8192, q_hi=8192, hq=32, hk=32, d=128, qbs=128, kbs=128, keep=0.1),
        # Training on ragged packed documents with grouped-query heads, head dim 64, fp16.
        _case("train ragged", kind="train", dtype="fp16", batch=6, q_lo=300, q_hi=4000, hq=16, hk=4, d=64, qbs=64, kbs=64, keep=0.4),
        # fp32 tensors (the reference's accuracy grid runs in fp32), ragged, multiplied in fp32.
        _case("fp32", dtype="fp32", batch=4, q_lo=500, q_hi=3000, hq=8, hk=4, d=64, qbs=64, kbs=64, keep=0.5),
    ]


# ---------------------------------------------------------------------------------------------------------------
# more cases of the same ranges
# ---------------------------------------------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lengths_about(rng, mid):
    """A range of lengths around mid: one length for all, or ragged."""
    if rng.random() < 0.3:
        return mid, mid
    return max(1, int(mid * rng.uniform(0.3, 0.9))), max(1, int(mid * rng.uniform(1.0, 1.6)))


def _heads(rng, most):
    hk = rng.choice([h for h in (1, 2, 4, 8, 16, 32) if h <= most])
    ratio = rng.choice([r for r in (1, 1, 2, 4, 8) if r * hk <= most])
    return hk * ratio, hk


def _short(rng):
    lo, hi = _lengths_about(rng, _log_int(rng, 24, 900))
    hq, hk = _heads(rng, 32)
    return _case(dtype=rng.choice(("bf16", "fp16")), batch=_log_int(rng, 1, 16), q_lo=lo, q_hi=hi, hq=hq, hk=hk,
                 d=rng.choice((32, 64, 128)), qbs=16 * rng.randint(1, 8), kbs=16 * rng.randint(1, 8), keep=round(rng.uniform(0.3, 0.9), 2),
                 diag=rng.random() < 0.7, causal=rng.random() < 0.7, metadata=rng.random() < 0.5)


def _prefill(rng):
    lo, hi = _lengths_about(rng, _log_int(rng, 1000, 20000))
    hq, hk = _heads(rng, 32)
    return _case(dtype=rng.choice(("bf16", "bf16", "fp16")), batch=_log_int(rng, 1, 8), q_lo=lo, q_hi=hi, hq=hq, hk=hk,
                 d=rng.choice((64, 128, 128)), qbs=rng.choice((64, 80, 128, 128)), kbs=rng.choice((48, 64, 128, 128)),
                 keep=round(rng.uniform(0.08, 0.4), 2), causal=rng.random() < 0.7)


def _decode(rng):
    mid = _log_int(rng, 1500, 40000)
    hq, hk = _heads(rng, 32)
    return _case(dtype=rng.choice(("bf16", "fp16")), batch=_log_int(rng, 1, 64), q_lo=1, q_hi=rng.choice((1, 1, 1, 4)),
                 k_lo=int(mid * rng.uniform(0.2, 1.0)), k_hi=int(mid * rng.uniform(1.0, 1.6)), hq=hq, hk=hk, d=rng.choice((64, 128, 128)),
                 qbs=16, kbs=rng.choice((16, 32, 64, 128)), keep=round(rng.uniform(0.1, 0.6), 2))


def _chunk(rng):
    q_mid, k_mid = _log_int(rng, 64, 1500), _log_int(rng, 8000, 90000)
    hq, hk = _heads(rng, 32)
    return _case(dtype=rng.choice(("bf16", "bf16", "fp16")), batch=rng.randint(1, 4), q_lo=max(1, q_mid // 2), q_hi=q_mid,
                 k_lo=int(k_mid * rng.uniform(0.5, 1.0)), k_hi=k_mid, hq=hq, hk=hk, d=rng.choice((64, 128, 128)),
                 qbs=rng.choice((64, 128)), kbs=rng.choice((64, 128)), keep=round(rng.uniform(0.1, 0.5), 2))


def _odd_head_dim(rng):
    lo, hi = _lengths_about(rng, _log_int(rng, 300, 4000))
    hq, hk = _heads(rng, 16)
    return _case(dtype=rng.choice(("bf16", "fp16")), batch=_log_int(rng, 1, 8), q_lo=lo, q_hi=hi, hq=hq, hk=hk,
                 d=rng.choice((48, 80, 96, 160, 192, 256)), qbs=rng.choice((64, 128)), kbs=rng.choice((64, 128)),
                 keep=round(rng.uniform(0.1, 0.5), 2), causal=rng.random() < 0.5)


def _train(rng):
    lo, hi = _lengths_about(rng, _log_int(rng, 200, 8000))
    hq, hk = _heads(rng, 32)
    return _case(kind="train", dtype=rng.choice(("bf16", "bf16", "fp16")), batch=_log_int(rng, 1, 8), q_lo=lo, q_hi=hi, hq=hq, hk=hk,
                 d=rng.choice((64, 128, 128)), qbs=rng.choice((64, 80, 128)), kbs=rng.choice((48, 64, 128)),
                 keep=round(rng.uniform(0.1, 0.6), 2), causal=rng.random() < 0.7)


def _fp32(rng):
    lo, hi = _lengths_about(rng, _log_int(rng, 64, 3000))
    hq, hk = _heads(rng, 16)
    return _case(dtype="fp32", batch=_log_int(rng, 1, 8), q_lo=lo, q_hi=hi, hq=hq, hk=hk, d=rng.choice((32, 64, 128)),
                 qbs=rng.choice((32, 64, 128)), kbs=rng.choice((16, 64, 128)), keep=round(rng.uniform(0.3, 0.7), 2),
                 causal=rng.random() < 0.5)


# each family with the most arithmetic (in FLOP) and the most bytes that a case of it may need
_FAMILIES = ((_short, 2e11, 1e9), (_prefill, 6e12, 6e9), (_decode, 6e11, 6e9), (_chunk, 3e12, 6e9), (_odd_head_dim, 6e11, 4e9),
             (_train, 4e12, 6e9), (_fp32, 1e11, 2e9))


def draw(rng):
    family, most_flops, most_bytes = rng.choice(_FAMILIES)
    while True:
        c = family(rng)
        w = work(c)
        if w["flops"] <= most_flops and w["bytes"] <= most_bytes and _mask_elements(c) <= 1 << 28:
            return c


# ---------------------------------------------------------------------------------------------------------------
# inputs, one pass
# ---------------------------------------------------------------------------------------------------------------
def _lengths(c):
    rng = random.Random(":".join(str(c[k]) for k in ("batch", "q_lo", "q_hi", "k_lo", "k_hi")))
    q = [rng.randint(c["q_lo"], c["q_hi"]) for _ in range(c["batch"])]
    k = [rng.randint(c["k_lo"], c["k_hi"]) for _ in range(c["batch"])] if c["k_hi"] else list(q)
    return q, k


def _mask_elements(c):
    q, k = _lengths(c)
    return c["hk"] * sum(-(-n // c["qbs"]) for n in q) * sum(-(-n // c["kbs"]) for n in k)


def prepare(case, seed):
    q_lens, k_lens = _lengths(case)
    w = make_problem(seed=seed, q_lens=q_lens, k_lens=k_lens, hq=case["hq"], hk=case["hk"], d=case["d"], qbs=case["qbs"],
                     kbs=case["kbs"], keep=case["keep"], diag=case["diag"], causal=case["causal"], scale=case["scale"],
                     device="cuda", dtype=_DTYPES[case["dtype"]], gen_device="device")
    dout = None
    if case["kind"] == "train":
        for t in (w.q, w.k, w.v):
            t.requires_grad_(True)
        g = torch.Generator(device="cuda")
        g.manual_seed(seed + 1)
        dout = torch.randn(w.q.shape, generator=g, device="cuda", dtype=torch.float32).to(w.q.dtype)
    return {"args": w.args(with_meta=case["metadata"]), "dout": dout}


def run(state):
    args, dout = state["args"], state["dout"]
    out = HBSAttention(*args)
    if dout is None:
        return out
    return (out,) + torch.autograd.grad(out, args[:3], dout)


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------
def work(case):
    """Arithmetic of the block pairs that are visited (kept, same sequence, not wholly above the causal diagonal; 4 * d FLOP
    a score element, and 2.5 times that more for the gradients), and every input and output once; of K and V, the
    blocks that some kept pair needs.  Expected values over the random mask."""
    q_lens, k_lens = _lengths(case)
    qbs, kbs, keep, d, esize = case["qbs"], case["kbs"], case["keep"], case["d"], _BYTES[case["dtype"]]
    elements = keys = mask = 0.0
    for q_len, k_len in zip(q_lens, k_lens):
        r0, c0 = np.arange(0, q_len, qbs), np.arange(0, k_len, kbs)
        rows, cols = np.minimum(qbs, q_len - r0), np.minimum(kbs, k_len - c0)
        p = np.full((len(r0), len(c0)), keep)
        if case["diag"]:
            p[np.arange(len(r0)), np.clip(r0 + (k_len - q_len), 0, k_len - 1) // kbs] = 1.0
        if case["causal"]:
            p[(r0 + rows - 1 + (k_len - q_len))[:, None] < c0[None, :]] = 0.0
        elements += float(rows @ p @ cols)
        keys += float((1.0 - np.prod(1.0 - p, axis=0)) @ cols)
        mask += float(p.size)
    q_values = sum(q_lens) * case["hq"] * d
    kv_values = 2.0 * keys * case["hk"] * d
    nbytes = (2.0 * q_values + kv_values) * esize + mask * case["hk"]
    flops = 4.0 * d * elements * case["hq"]
    if case["kind"] == "train":   # dout read, dq written; dk and dv written
        nbytes += (2.0 * q_values + 2.0 * sum(k_lens) * case["hk"] * d) * esize
        flops *= 3.5
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # operands (the probabilities among them) and results carry 8, 11 or 24 significant bits; sums are fp32
    return {"bf16": {"rel": 1e-2}, "fp16": {"rel": 2e-3}, "fp32": {"rel": 1e-5}}[case["dtype"]]
