"""Performance cases of the attention forward: what a program that uses this
framework has it do, through ``fa_amd.binding.Operator``.

A case is one call shape:

  batch, heads_q, heads_kv, seq_q, seq_k   the geometry (128 dims per head)
  acc       accumulation variant, "fp32" or "fp16"
  causal    "none", "top_left" (a whole prompt) or "bottom_right" (new rows
            behind a cache of earlier keys)
  split     True: the key-split forward with the library's own part count,
            which is what decode and short query ranges are meant to use;
            False: the one-pass forward, the default
  layout    "bhnd", or "bnhd": sequence-major tensors viewed as [B, H, N, 128]
  lse       True: the per-row log-sum-exp is returned as well
  dist      "normal" N(0,1), or "stress" (queries and keys of standard
            deviation 3, one value row in twenty scaled by 8)

The listed cases run from one decode step over a short cache to the
131072-token forward; ``draw`` spreads the same four kinds of call (decode,
a short query range behind a cache, a prompt, cross attention) over their
whole ranges.
"""

import torch

from fa_amd import build
from fa_amd.binding import AttentionConfig, Operator

DIM = 128


def _case(name, batch, heads_q, heads_kv, seq_q, seq_k, acc="fp32", causal="none", split=False,
          layout="bhnd", lse=False, dist="normal"):
    return {"name": name, "batch": batch, "heads_q": heads_q, "heads_kv": heads_kv,
            "seq_q": seq_q, "seq_k": seq_k, "acc": acc, "causal": causal, "split": split,
            "layout": layout, "lse": lse, "dist": dist}


def listed():
    return [
        # One decode step early in a generation: a short cache whose length is
        # whatever the step happens to be, the smallest call of all.
        _case("decode_4k", 1, 12, 1, 1, 4099, split=True),
        # One decode step behind the longest context.
        _case("decode_131k", 1, 12, 1, 1, 131072, split=True),
        # A decode step of a serving batch with eight KV heads, its cache kept
        # sequence-major and of an arbitrary length.
        _case("decode_batch", 8, 64, 8, 1, 8005, split=True, layout="bnhd"),
        # A few tokens at once behind a cache (drafted tokens being checked).
        _case("extend_16", 1, 12, 1, 16, 50001, causal="bottom_right", split=True),
        # One chunk of a long prompt that is prefilled in pieces.
        _case("extend_256", 1, 12, 1, 256, 131072, causal="bottom_right", split=True, lse=True),
        # A short prompt of an odd length.
        _case("prefill_1k", 1, 12, 1, 1000, 1000, causal="top_left"),
        # The 4096-token configuration (B=1, 12 query heads on one KV head).
        _case("prefill_4k", 1, 12, 1, 4096, 4096),
        # A batch of prompts in the sequence-major layout of training and
        # serving code, with the log-sum-exp a backward or a merge needs.
        _case("prefill_batch", 4, 32, 8, 2048, 2048, causal="top_left", layout="bnhd", lse=True),
        # Cross attention with odd lengths, FP16-accumulated.
        _case("cross_odd", 2, 24, 2, 3001, 7777, acc="fp16", lse=True),
        # The 32768-token configuration.
        _case("prefill_32k", 1, 12, 1, 32768, 32768),
        # The 65536-token configuration with the stress distribution, through
        # the FP16-accumulated variant.
        _case("stress_64k", 2, 12, 1, 65536, 65536, acc="fp16", dist="stress"),
        # The headline configuration, the largest.
        _case("prefill_131k", 2, 12, 1, 131072, 131072),
    ]


# (query heads, KV heads): groups of 1 to 12 on 1 to 16 KV heads.
HEADS = [(12, 1), (12, 1), (8, 1), (24, 2), (32, 8), (64, 8), (16, 16)]
MAX_KEYS = 1 << 21        # batch * KV heads * keys of a drawn case: 512 MiB each of K and V
MAX_ROWS = 1 << 22        # batch * query heads * query rows: 1 GiB each of Q and O
MAX_FLOPS = 5.0e13


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], both ends included."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "extend", "prefill", "prefill", "cross"])
    heads_q, heads_kv = rng.choice(HEADS)
    causal, split = "none", False
    if kind == "decode":
        seq_q, seq_k, split = 1, _log(rng, 64, 131072), True
    elif kind == "extend":
        seq_k = _log(rng, 512, 131072)
        seq_q, causal, split = _log(rng, 2, 512), "bottom_right", True
    elif kind == "prefill":
        seq_q = seq_k = _log(rng, 64, 65536)
        causal = rng.choice(["none", "top_left", "top_left"])
    else:
        seq_q, seq_k = _log(rng, 64, 8192), _log(rng, 16, 32768)
    batch = _log(rng, 1, 32)
    case = _case("", batch, heads_q, heads_kv, seq_q, seq_k,
                 acc="fp16" if rng.random() < 0.25 else "fp32", causal=causal, split=split,
                 layout=rng.choice(["bhnd", "bhnd", "bnhd"]), lse=rng.random() < 0.3,
                 dist="stress" if rng.random() < 0.15 else "normal")
    del case["name"]
    while case["batch"] > 1 and (case["batch"] * heads_kv * seq_k > MAX_KEYS
                                 or case["batch"] * heads_q * seq_q > MAX_ROWS
                                 or work(case)["flops"] > MAX_FLOPS):
        case["batch"] -= 1
    return case


def _tensors(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(heads, n):
        shape = (case["batch"], heads, n, DIM) if case["layout"] == "bhnd" else \
            (case["batch"], n, heads, DIM)
        t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)
        return t if case["layout"] == "bhnd" else t.transpose(1, 2)

    q = rand(case["heads_q"], case["seq_q"])
    k = rand(case["heads_kv"], case["seq_k"])
    v = rand(case["heads_kv"], case["seq_k"])
    if case["dist"] == "stress":
        q.mul_(3.0)
        k.mul_(3.0)
        rows = torch.rand(v.shape[:3], generator=g, device="cuda") < 0.05
        v.mul_(torch.where(rows, 8.0, 1.0).half().unsqueeze(-1))
    return q, k, v


def prepare(case, seed):
    q, k, v = _tensors(case, seed)
    op = Operator(build.LIBRARY, AttentionConfig(acc=case["acc"], causal=case["causal"],
                                                 splits=0 if case["split"] else None))
    return {"op": op, "q": q, "k": k, "v": v, "lse": case["lse"]}


def run(state):
    return state["op"](state["q"], state["k"], state["v"], return_lse=state["lse"])


def _offset(case):
    """Row i sees keys j <= i + offset under the case's mask."""
    return case["seq_k"] - case["seq_q"] if case["causal"] == "bottom_right" else 0


def _pairs(case):
    """(query, key) pairs of one head that the mask lets through."""
    nq, nk = case["seq_q"], case["seq_k"]
    if case["causal"] == "none":
        return nq * nk
    first = 1 + _offset(case)                       # keys row 0 sees, were there enough
    skip = max(0, 1 - first)                        # rows before it see nothing
    rows = nq - skip
    first += skip
    ramp = max(0, min(rows, nk - first + 1))        # rows that see first, first + 1, ... keys
    return ramp * first + ramp * (ramp - 1) // 2 + max(0, rows - ramp) * nk


def work(case):
    pairs = _pairs(case)
    keys = case["seq_k"] if case["causal"] == "none" else \
        max(0, min(case["seq_k"], case["seq_q"] + _offset(case)))
    rows = case["batch"] * case["heads_q"] * case["seq_q"]
    return {"bytes": 2 * rows * DIM * 2 + 2 * case["batch"] * case["heads_kv"] * keys * DIM * 2
            + (4 * rows if case["lse"] else 0),
            "flops": 4 * case["batch"] * case["heads_q"] * pairs * DIM}


def tolerance(case):
    # The probabilities enter the second product as FP16 and O leaves as FP16
    # (FP16 accumulation rounds O every 512 keys as well): 2.9e-4 and 6.8e-4
    # from the float64 result at most, measured.
    if case["acc"] == "fp16":
        return {"rel": 3e-3, "max": 6e-2}
    return {"rel": 1.2e-3, "max": 3e-2}


# float64 work above this takes too long.
EXACT_FLOPS = 1.0e13


def exact(case, seed):
    if work(case)["flops"] > EXACT_FLOPS:
        return None
    q, k, v = _tensors(case, seed)
    nq, nk, group = case["seq_q"], case["seq_k"], case["heads_q"] // case["heads_kv"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.full(q.shape[:3], float("-inf"), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // nk)                  # rows at a time: at most 1 GiB of scores
    cols = torch.arange(nk, device="cuda")
    for b in range(case["batch"]):
        for hk in range(case["heads_kv"]):
            kt = k[b, hk].double().t().contiguous()
            vd = v[b, hk].double().contiguous()
            for h in range(hk * group, (hk + 1) * group):
                for r0 in range(0, nq, step):
                    r1 = min(nq, r0 + step)
                    s = torch.mm(q[b, h, r0:r1].double().contiguous(), kt) * DIM ** -0.5
                    if case["causal"] != "none":
                        last = torch.arange(r0, r1, device="cuda") + _offset(case)
                        s.masked_fill_(cols > last.unsqueeze(1), float("-inf"))
                    top = s.amax(dim=1, keepdim=True)
                    top = torch.where(torch.isinf(top), torch.zeros_like(top), top)
                    s.sub_(top).exp_()
                    total = s.sum(dim=1, keepdim=True)
                    seen = total > 0
                    out[b, h, r0:r1] = torch.where(
                        seen, torch.mm(s, vd) / torch.where(seen, total, torch.ones_like(total)),
                        torch.zeros((), dtype=torch.float64, device="cuda"))
                    lse[b, h, r0:r1] = (total.log() + top).squeeze(1)
    return (out, lse) if case["lse"] else out
