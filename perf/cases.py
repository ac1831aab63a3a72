"""The calls whose speed this framework is judged by: attention forward, attention forward + backward, RetNet's parallel
form (mask tensor and decay rates, forward and forward + backward) and RetNet's recurrent form, each through the public
operators.

A call never starts a tuning run here: like the benchmark and any serving process, a problem without an entry in the tuning
cache launches what the framework picks for it (AAT_TUNE_ON_MISS=0).

Sequence lengths of the parallel operators are multiples of 64 (the operators' granularity), of the recurrent one multiples
of 32; head sizes are the pairs the framework is built for ahead of time.
"""
import math
import os

import torch

import attention_autotuner_amd as aat

os.environ.setdefault("AAT_TUNE_ON_MISS", "0")

_ARCH = aat.MI355X()

_ATTN_DIMS = ((64, 64), (128, 128), (128, 128), (192, 192), (256, 256))
_RET_DIMS = ((64, 64), (128, 128), (192, 192), (256, 256), (256, 512), (256, 512))


def listed():
    return [
        # A short prompt through a small model: the call's own cost (host path, launch, one wave of blocks) is what a user waits for.
        dict(name="attn_small", op="attn", b=2, h=8, sq=512, sk=512, dqk=64, dv=64, causal=False, train=False),
        # The benchmark's headline problem: bidirectional attention at an ordinary batch.
        dict(name="attn_infer", op="attn", b=4, h=32, sq=2048, sk=2048, dqk=128, dv=128, causal=False, train=False),
        # Prefill of one long prompt.
        dict(name="attn_prefill", op="attn", b=1, h=32, sq=8192, sk=8192, dqk=128, dv=128, causal=True, train=False),
        # Few query rows against a long context: cross-attention, or a block of drafted tokens checked at once.
        dict(name="attn_long_kv", op="attn", b=1, h=32, sq=256, sk=16384, dqk=128, dv=128, causal=False, train=False),
        # Chunked prefill: a ragged chunk of new tokens against what is cached, causal along the bottom-right diagonal.
        dict(name="attn_chunk", op="attn", b=3, h=12, sq=192, sk=4160, dqk=128, dv=128, causal=True, train=False),
        # A training step of a decoder layer at an ordinary length.
        dict(name="attn_train", op="attn", b=4, h=32, sq=2048, sk=2048, dqk=128, dv=128, causal=True, train=True),
        # A training step on a packed batch padded to a ragged length, small heads.
        dict(name="attn_train_ragged", op="attn", b=3, h=12, sq=1088, sk=1088, dqk=64, dv=64, causal=True, train=True),
        # RetNet forward with an arbitrary (dense) mask at a ragged length.
        dict(name="ret_mask_ragged", op="ret", b=3, h=8, sq=1344, sk=1344, dqk=256, dv=256, mask="normal", mode="auto", train=False),
        # RetNet training step with its decay mask handed over as a tensor: the benchmark's RetNet problem.
        dict(name="ret_train", op="ret", b=4, h=8, sq=2048, sk=2048, dqk=256, dv=512, mask="decay", mode="auto", train=True),
        # RetNet training step with the decay rates instead of a mask tensor, ragged length.
        dict(name="ret_decay_train_ragged", op="ret_decay", b=2, h=8, sq=2112, sk=2112, dqk=256, dv=512, train=True),
        # RetNet's recurrent form over a batch of sequences: the benchmark's problem.
        dict(name="recurrent", op="recurrent", b=8, h=32, l=2048, kd=128, vd=128),
        # The recurrent form at the parallel form's larger head sizes, few and ragged sequences.
        dict(name="recurrent_wide_ragged", op="recurrent", b=2, h=8, l=1056, kd=256, vd=512),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _length(rng, lo, hi, step=64):
    return max(lo, min(hi, step * round(_log_uniform(rng, lo, hi) / step)))


def _heads(rng, most):
    return rng.randint(1, 8), rng.choice([h for h in (4, 6, 8, 12, 16, 20, 32) if h <= most])


def _drawn(rng):
    kind = rng.choice(("attn", "few_rows", "attn_train", "ret", "ret_train", "ret_decay", "recurrent"))
    if kind == "recurrent":
        b, h = _heads(rng, 32)
        return dict(op="recurrent", b=b, h=h, l=_length(rng, 64, 4096, 32), kd=rng.choice((64, 128, 128, 192, 256)),
                    vd=rng.choice((64, 128, 192, 256, 512)))
    if kind in ("attn", "few_rows", "attn_train"):
        b, h = _heads(rng, 32)
        dqk, dv = rng.choice(_ATTN_DIMS)
        causal = rng.random() < 0.6
        if kind == "few_rows":
            sq, sk = _length(rng, 64, 512), _length(rng, 1024, 32768)
        else:
            sq = sk = _length(rng, 64, 8192)
        return dict(op="attn", b=b, h=h, sq=sq, sk=sk, dqk=dqk, dv=dv, causal=causal, train=kind == "attn_train")
    b, h = _heads(rng, 16)
    dqk, dv = rng.choice(_RET_DIMS)
    s = _length(rng, 64, 4096)
    train = kind == "ret_train" or rng.random() < 0.5
    if kind == "ret_decay":
        return dict(op="ret_decay", b=b, h=h, sq=s, sk=s, dqk=dqk, dv=dv, train=train)
    mask = rng.choice(("decay", "decay", "normal"))
    mode = rng.choice(("auto", "kept_scan", "promise") if mask == "decay" else ("auto", "dense"))
    return dict(op="ret", b=b, h=h, sq=s, sk=s, dqk=dqk, dv=dv, mask=mask, mode=mode, train=kind == "ret_train")


def draw(rng):
    """A case of the same ranges that costs no more than the largest listed ones of its kind (half of their operations: wide
    heads and unfavourable lengths run at lower rates)."""
    parallel = [work(c) for c in listed() if c["op"] != "recurrent"]
    most = {"flops": 0.5 * max(w["flops"] for w in parallel), "bytes": max(w["bytes"] for w in parallel)}
    recurrent = [work(c) for c in listed() if c["op"] == "recurrent"]
    most_recurrent = {k: max(w[k] for w in recurrent) for k in most}
    while True:
        case = _drawn(rng)
        w, limit = work(case), most_recurrent if case["op"] == "recurrent" else most
        if w["flops"] <= limit["flops"] and w["bytes"] <= limit["bytes"]:
            return case


def _gamma(heads):
    return 1.0 - torch.pow(2.0, -5.0 - torch.arange(heads, dtype=torch.float64))


def _decay_mask(heads, sq, sk):
    """gamma_h^(i + sk - sq - j) on and below that diagonal, 0 above."""
    i = torch.arange(sq, device="cuda").unsqueeze(1) + (sk - sq)
    dist = (i - torch.arange(sk, device="cuda").unsqueeze(0)).float()
    gamma = _gamma(heads).float().cuda().view(-1, 1, 1)
    return (torch.pow(gamma, dist.clamp(min=0).unsqueeze(0)) * (dist >= 0)).half()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    b, h = case["b"], case["h"]
    state = {"case": case}
    if case["op"] == "recurrent":
        kd, vd, l = case["kd"], case["vd"], case["l"]

        def uniform(*shape):
            return torch.rand(*shape, generator=g, device="cuda") * 2 - 1
        state.update(q=uniform(b, h, kd, l), k=uniform(b, h, kd, l), v=uniform(b, h, vd, l),
                     decay=_gamma(h).float().cuda().unsqueeze(1).expand(h, l).contiguous())
        return state

    sq, sk, dqk, dv = case["sq"], case["sk"], case["dqk"], case["dv"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda").half()
    state.update(q=normal(b, h, sq, dqk), k=normal(b, h, sk, dqk), v=normal(b, h, sk, dv))
    if case["train"]:
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
        state["do"] = normal(b, h, sq, dv)
    if case["op"] == "ret_decay":
        state["gamma"] = _gamma(h)
    elif case["op"] == "ret":
        state["mask"] = _decay_mask(h, sq, sk) if case["mask"] == "decay" else normal(h, sq, sk)
        # how much of the mask is walked: found by the call, found once for all layers and steps, promised, or all of it
        state["walk"] = {"auto": lambda: None, "kept_scan": lambda: aat.retnet_mask_scan(state["mask"], _ARCH),
                         "promise": lambda: True, "dense": lambda: False}[case["mode"]]()
    return state


def run(state):
    case = state["case"]
    q, k, v = state["q"], state["k"], state["v"]
    if case["op"] == "recurrent":
        return aat.retnet_recurrent_fwd(q, k, v, state["decay"])
    if case["op"] == "attn":
        o = aat.flash_attn_func(q, k, v, _ARCH, case["causal"])
    elif case["op"] == "ret_decay":
        o = aat.RetNetDecayAttnFunc(q, k, v, state["gamma"], _ARCH)
    else:
        o = aat.RetNetAttnFunc(q, k, v, state["mask"], _ARCH, state["walk"])
    if not case["train"]:
        return o
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


def work(case):
    b, h = case["b"], case["h"]
    if case["op"] == "recurrent":
        kd, vd, l = case["kd"], case["vd"], case["l"]
        # per position: the state's decay and update and its product with q, for every (key dim, value dim)
        return {"bytes": 4.0 * b * h * l * (2 * kd + 2 * vd) + 4.0 * h * l, "flops": 5.0 * b * h * l * kd * vd}
    sq, sk, dqk, dv = case["sq"], case["sk"], case["dqk"], case["dv"]
    lower = case.get("causal", False) or case["op"] == "ret_decay" or case.get("mask") == "decay"
    if lower:                    # row i sees the columns up to i + sk - sq
        pairs = sum(min(sk, max(0, i + sk - sq + 1)) for i in range(sq))
    else:
        pairs = sq * sk
    flops = 2.0 * b * h * pairs * (dqk + dv)
    nbytes = 2.0 * b * h * (sq * dqk + sk * dqk + sk * dv + sq * dv)
    if case["train"]:
        flops += 2.0 * b * h * pairs * (3 * dqk + 2 * dv)
        nbytes += 2.0 * b * h * (sq * dqk + sk * dqk + sk * dv + sq * dv)
    if case["op"] == "ret":      # a scanning or dense call reads the whole mask, a kept scan or a promise its lower half
        nbytes += 2.0 * h * (pairs if case["mode"] in ("kept_scan", "promise") else sq * sk)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Four times the distance of a result from the same sums in 64 bits: 2.6e-4 to 3.1e-4 over the parallel cases (fp16 inputs,
    # P / S / dS and results rounded to fp16), 2.7e-7 over the recurrent ones (fp32 throughout; longer sums stray further).
    if case["op"] == "recurrent":
        return {"rel": 2e-6}
    return {"rel": 1.2e-3}
