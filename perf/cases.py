"""The calls whose speed is measured, as a program that serves a model makes them.

Three producers and consumers of logits meet here: the sampler (one row of an
interactive decode, batches of a server, every filter), the lm_heads that feed
it (bf16 with the final softcap, and the int2 quantised head) and the scorers
beside it (log-probabilities, grammar masks). `listed()` holds one case per
use; `draw()` gives others of the same ranges.

  family "sample"   gs_sample over logits in HBM
  family "step"     a constrained decode step: masks of the rows' DFA states, then the sampler
  family "head"     the bf16 lm_head
  family "headstep" the bf16 lm_head and the sampler in one call
  family "qat"      the int2 lm_head
  family "score"    tokenLogProbability of one token a row
"""
import math
import os
import sys

import numpy as np
import torch

_PACKAGES = os.path.join(os.getcwd(), "gemma-webgpu-engine_amd")
if _PACKAGES not in sys.path:
    sys.path.insert(0, _PACKAGES)

import gsample as gs  # noqa: E402
from gsample import runtime as rt  # noqa: E402
from gsample import workloads as wl  # noqa: E402

V = 262144

# Decoding options by name. "default" is the session's own default, "penalties"
# the batched serving mix, "multinomial" a temperature and nothing else over
# generate()'s defaults, "typical" typical-p over the same defaults.
POLICIES = {
    "default": gs.DecodingConfig(),
    "greedy": gs.DecodingConfig(temperature=0.0, topK=0, topP=1.0, repetitionPenalty=1.0, repetitionWindow=0),
    "penalties": wl.PENALTY_CONFIG,
    "nucleus": wl.HEAVY_TAIL_CONFIG,
    "topk_deep": wl.TOPK_DEEP_CONFIG,
    "minp": wl.HEAVY_TAIL_CONFIG.merged(topP=1.0, minP=0.05),
    "multinomial": wl.MULTINOMIAL_CONFIG,
    "typical": wl.MULTINOMIAL_CONFIG.merged(typicalP=0.9),
    "head": wl.LMHEAD_CONFIG,
}


def listed():
    return [
        # one row of an interactive decode through the whole host call, with the session's default options
        {"name": "decode_row", "family": "sample", "call": "whole", "rows": 1, "vocab": V, "dtype": "f32",
         "policy": "default"},
        # a server's ordinary batch: penalties over 512-id histories, top-k and top-p
        {"name": "serve_batch", "family": "sample", "call": "launch", "rows": 256, "vocab": V, "dtype": "f32",
         "policy": "penalties"},
        # a server's largest batch: heavy-tailed bf16 logits and a nucleus alone
        {"name": "nucleus_bf16", "family": "sample", "call": "launch", "rows": 1024, "vocab": V, "dtype": "bf16",
         "policy": "nucleus"},
        # generate() with a temperature alone: a draw from the whole vocabulary
        {"name": "multinomial", "family": "sample", "call": "launch", "rows": 256, "vocab": V, "dtype": "f32",
         "policy": "multinomial"},
        # typical-p alone, on a vocabulary that no tile divides
        {"name": "typical_odd", "family": "sample", "call": "launch", "rows": 24, "vocab": 151643, "dtype": "f32",
         "policy": "typical"},
        # one step of grammar-constrained decoding: new states each step, so masks and samples
        {"name": "grammar_step", "family": "step", "call": "whole", "rows": 64, "vocab": V, "dtype": "f32",
         "policy": "nucleus"},
        # a decode step of a batch of 64: hidden states to logits and tokens
        {"name": "head_step_64", "family": "headstep", "rows": 64, "vocab": V, "width": 2048, "policy": "head"},
        # logits of a prompt's positions (scoring a prompt, checking drafted tokens)
        {"name": "head_prompt", "family": "head", "rows": 512, "vocab": V, "width": 2048},
        # a few rows at a wider hidden state and a vocabulary of odd size
        {"name": "head_wide_odd", "family": "head", "rows": 12, "vocab": 151643, "width": 3840},
        # one decode row of the quantised head, in the layout that a GPU host keeps
        {"name": "qat_row", "family": "qat", "rows": 1, "vocab": V, "width": 1536, "layout": "block",
         "in_scale": 0.0, "out_scale": 0.125},
        # a batch through the quantised head in the checkpoint's layout, activations quantised too
        {"name": "qat_batch", "family": "qat", "rows": 48, "vocab": V, "width": 1536, "layout": "row",
         "in_scale": 0.03, "out_scale": 0.02},
        # log-probabilities of a sequence's tokens
        {"name": "score_rows", "family": "score", "rows": 128, "vocab": V, "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng):
    return V if rng.random() < 0.5 else rng.randrange(32001, V)


def draw(rng):
    family = rng.choice(["sample", "sample", "sample", "step", "headstep", "head", "head", "qat", "qat", "score"])
    vocab = _vocab(rng)
    if family == "sample":
        whole = rng.random() < 0.25
        return {"family": "sample", "call": "whole" if whole else "launch",
                "rows": _log_int(rng, 1, 16 if whole else 512), "vocab": vocab,
                "dtype": rng.choice(["f32", "f32", "bf16"]),
                "policy": rng.choice([p for p in sorted(POLICIES) if p != "head"])}
    if family == "step":
        return {"family": "step", "call": "whole", "rows": _log_int(rng, 1, 128), "vocab": vocab, "dtype": "f32",
                "policy": rng.choice(["nucleus", "greedy", "penalties"])}
    if family == "headstep":
        return {"family": "headstep", "rows": _log_int(rng, 1, 128), "vocab": vocab,
                "width": 64 * rng.randrange(8, 41), "policy": "head"}
    if family == "head":
        width = 64 * rng.randrange(8, 41)
        return {"family": "head", "rows": _log_int(rng, 1, 512 if width <= 2048 else 256), "vocab": vocab,
                "width": width}
    if family == "qat":
        quantised = rng.random() < 0.5
        return {"family": "qat", "rows": _log_int(rng, 1, 64), "vocab": vocab,
                "width": rng.choice([256 * rng.randrange(2, 9), 64 * rng.randrange(8, 33)]),
                "layout": rng.choice(["block", "row"]),
                "in_scale": 0.03 if quantised else 0.0, "out_scale": 0.02 if quantised else 0.125}
    return {"family": "score", "rows": _log_int(rng, 1, 256), "vocab": vocab, "dtype": rng.choice(["f32", "bf16"])}


# ---------------------------------------------------------------- inputs

_ZIPF = {}
_STREAM = []


def _stream():
    """The one stream the program serves from (not torch's default stream,
    whose null handle the library reads as "the context's own")."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0].cuda_stream


def _histories(rng, rows, vocab, n):
    """n Zipf(1.1) ids a row: the ids a text repeats most are the lowest."""
    if vocab not in _ZIPF:
        cdf = np.cumsum(np.arange(1, vocab + 1, dtype=np.float64) ** -1.1)
        _ZIPF[vocab] = cdf / cdf[-1]
    ids = np.searchsorted(_ZIPF[vocab], rng.random((rows, n)), side="right")
    return np.minimum(ids, vocab - 1).astype(np.int32)


def _logits(case, gen, device):
    """N(0, 3^2) in f32; in bf16 8 ln(rank^-1.1) + N(0, 0.5^2) in an order of
    each row's own, the heavy tail of a language model's logits."""
    rows, vocab = case["rows"], case["vocab"]
    if case["dtype"] == "f32":
        return torch.randn(rows, vocab, generator=gen, device=device).mul_(3.0)
    base = -8.8 * torch.log(torch.arange(1, vocab + 1, device=device, dtype=torch.float32))
    out = torch.empty(rows, vocab, dtype=torch.bfloat16, device=device)
    for r in range(rows):
        x = base + 0.5 * torch.randn(vocab, generator=gen, device=device)
        out[r, torch.randperm(vocab, generator=gen, device=device)] = x.to(torch.bfloat16)
    return out


def _options(case, rng, states=None):
    policy = POLICIES[case["policy"]]
    draws = rng.random(case["rows"])
    conf = np.stack([rt.row_config(policy, uniform=float(u), mask_slot=-1 if states is None else r)
                     for r, u in enumerate(draws)])
    hist = None
    if policy.repetitionWindow > 0:
        hist = _histories(rng, case["rows"], case["vocab"], policy.repetitionWindow)
    return policy, conf, hist, draws


def prepare(case, seed):
    device = torch.device("cuda", 0)
    gen = torch.Generator(device=device).manual_seed(seed)
    rng = np.random.default_rng(seed)
    rows, vocab, family = case["rows"], case["vocab"], case["family"]
    s = gs.Sampler(vocab_size=vocab, max_rows=rows)
    state = {"case": case, "sampler": s}
    if family == "score":
        state["logits"] = _logits(case, gen, device)
        state["tokens"] = rng.integers(0, vocab, rows).astype(np.int32)
        return state
    if family == "qat":
        width = case["width"]
        state["x"] = torch.randn(rows, width, generator=gen, device=device).mul_(1.5)
        state["codes"] = torch.randint(-2 ** 31, 2 ** 31, (vocab * width // 16,), generator=gen, device=device,
                                       dtype=torch.int64).to(torch.int32)
        state["scales"] = 0.0008 + (torch.arange(vocab, device=device) % 29).float() * 0.000025
        state["out"] = torch.empty(rows, vocab, device=device)
        return state
    if family in ("head", "headstep"):
        width = case["width"]
        state["hidden"] = torch.randn(rows, width, generator=gen, device=device).to(torch.bfloat16)
        state["weight"] = torch.empty(vocab, width, dtype=torch.bfloat16, device=device)
        for v in range(0, vocab, 32768):
            w = torch.randn(min(32768, vocab - v), width, generator=gen, device=device)
            state["weight"][v:v + 32768] = w.mul_(0.02).to(torch.bfloat16)
        state["out"] = torch.empty(rows, vocab, device=device)
        if family == "headstep":
            state["policy"], conf, hist, state["draws"] = _options(case, rng)
            state["histories"] = hist
            state["batch"], state["keep"] = s.prepare(state["out"], conf, histories=list(hist))
        return state
    state["logits"] = _logits(case, gen, device)
    states = rng.integers(0, 64, rows) if family == "step" else None
    state["policy"], conf, hist, state["draws"] = _options(case, rng, states)
    state["histories"] = hist
    if family == "step":
        offsets, data = wl.synthetic_vocab(vocab=vocab)
        s.set_vocab(offsets, data)
        s.set_dfa(*wl.synthetic_dfa())
        state["states"], state["config"] = states, conf
    elif case["call"] == "whole":
        state["config"] = conf
    else:
        state["batch"], state["keep"] = s.prepare(state["logits"], conf,
                                                  histories=None if hist is None else list(hist))
    return state


# ----------------------------------------------------------------- calls


def _results(keep):
    """Tokens and probabilities as the sampler left them (16 bytes a row)."""
    raw = keep[-1]
    return {"tokens": raw.view(torch.int32)[:, 0], "probabilities": raw[:, 1]}


def run(state):
    case, s = state["case"], state["sampler"]
    family = case["family"]
    if family == "score":
        return s.token_log_probability(state["logits"], state["tokens"])
    if family == "qat":
        layout = rt.GS_QAT_BLOCK_MAJOR if case["layout"] == "block" else rt.GS_QAT_ROW_MAJOR
        return s.qat_lmhead(state["x"], state["codes"], state["scales"], layout=layout,
                            input_scale=case["in_scale"], output_scale=case["out_scale"], out=state["out"],
                            stream=_stream())
    if family == "head":
        return s.lmhead(state["hidden"], state["weight"], softcap_value=30.0, out=state["out"], stream=_stream())
    if family == "headstep":
        s.lmhead_sample_launch(state["hidden"], state["weight"], 30.0, state["out"], state["batch"], _stream())
        return {"logits": state["out"], **_results(state["keep"])}
    hist = None if state["histories"] is None else list(state["histories"])
    if family == "step":
        table = s.build_masks(state["states"])
        out = s.sample(state["logits"], state["config"], histories=hist, mask_table=table)
        return {"masks": table, "tokens": out.tokens, "probabilities": out.probabilities}
    if case["call"] == "whole":
        out = s.sample(state["logits"], state["config"], histories=hist)
        return {"tokens": out.tokens, "probabilities": out.probabilities}
    s.launch(state["batch"], _stream())
    return _results(state["keep"])


def work(case):
    rows, vocab, family = case["rows"], case["vocab"], case["family"]
    if family == "qat":
        width = case["width"]
        return {"bytes": vocab * width / 4 + 4 * vocab + 4 * rows * width + 4 * rows * vocab,
                "flops": 2.0 * rows * vocab * width}
    if family in ("head", "headstep"):
        width = case["width"]
        return {"bytes": 2.0 * vocab * width + 2 * rows * width + 4.0 * rows * vocab,
                "flops": 2.0 * rows * vocab * width}
    size = rows * vocab * (2 if case["dtype"] == "bf16" else 4)
    if family == "score":
        return {"bytes": size + 12.0 * rows, "flops": 3.0 * rows * vocab}
    window = POLICIES[case["policy"]].repetitionWindow
    masks = rows * vocab / 4.0 + 14.5 * vocab if family == "step" else 0.0
    return {"bytes": size + masks + rows * (4 * window + 112 + 16.0), "flops": 3.0 * rows * vocab}


def tolerance(case):
    if case["family"] == "qat":
        return "exact"  # the head's contract: its logits equal the reference's bit for bit
    if case["family"] == "score":
        return {"rel": 1e-13}
    return {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------- the same in 64 bits


def _sampled_probability(x, policy, u, history):
    """The chosen item's probability of the reference's sampler over one row of
    64-bit logits (masked ids are -inf)."""
    if history is not None and policy.repetitionWindow > 0:
        ids, counts = np.unique(history[-policy.repetitionWindow:], return_counts=True)
        at = torch.from_numpy(ids.astype(np.int64)).to(x.device)
        n = torch.from_numpy(counts.astype(np.float64)).to(x.device)
        l = x[at]
        l = torch.where(l < 0, l * policy.repetitionPenalty, l / policy.repetitionPenalty)
        x = x.clone()
        x[at] = l - (policy.presencePenalty + n * policy.frequencyPenalty)
    if policy.temperature == 0:
        return 1.0
    v = torch.sort(x / policy.temperature, descending=True, stable=True).values
    p = torch.exp(v - v[0])
    p = p / p.sum()
    if policy.topK > 0:
        p = p[:policy.topK]
    if policy.minP > 0:
        p = p[p >= p[0] * policy.minP]
    if policy.typicalP < 1:
        p = p[p > 0]
        entropy = -(p * p.log()).sum()
        order = torch.sort((-p.log() - entropy).abs(), stable=True).indices
        kept = int((torch.cumsum(p[order], 0) < policy.typicalP).sum()) + 1
        p = torch.sort(p[order[:kept]], descending=True, stable=True).values
    if policy.topP < 1:
        p = p[:int((torch.cumsum(p, 0) < policy.topP).sum()) + 1]
    c = torch.cumsum(p, 0)
    return float(p[min(int((c < u * c[-1]).sum()), p.numel() - 1)])


def _srq(x, scale):
    if scale == 0:
        return x
    return torch.clamp(torch.round(x / scale), -128, 127).mul(scale).to(torch.float32).double()


def _codes(state, lo, hi):
    """Rows lo .. hi of the weights, code - 2, in 64 bits."""
    case = state["case"]
    vocab, width = case["vocab"], case["width"]
    if case["layout"] == "block":
        words = state["codes"].view(width // 64, vocab, 4)[:, lo:hi].permute(1, 0, 2).reshape(hi - lo, -1)
    else:
        words = state["codes"].view(vocab, width // 16)[lo:hi]
    shift = 2 * torch.arange(16, device=words.device, dtype=torch.int32)
    return (((words.unsqueeze(-1) >> shift) & 3) - 2).reshape(hi - lo, width).double()


def exact(case, seed):
    state = prepare(case, seed)
    rows, vocab, family = case["rows"], case["vocab"], case["family"]
    if family == "score":
        out = np.empty(rows)
        for r in range(rows):
            x = state["logits"][r].double()
            d = x - x.max()
            out[r] = float(d[int(state["tokens"][r])] - d.exp().sum().log())
        return out
    if family == "qat":
        a = _srq(state["x"].double(), np.float32(case["in_scale"]).item())
        out = torch.empty(rows, vocab, dtype=torch.float64, device=a.device)
        scale_out = np.float32(case["out_scale"]).item()
        for lo in range(0, vocab, 32768):
            hi = min(vocab, lo + 32768)
            dot = a @ _codes(state, lo, hi).t().contiguous()
            out[:, lo:hi] = _srq(dot * state["scales"][lo:hi].double(), scale_out)
        return out
    if family in ("head", "headstep"):
        out = torch.empty(rows, vocab, dtype=torch.float64, device=state["out"].device)
        for lo in range(0, vocab, 32768):
            w = state["weight"][lo:lo + 32768].double().t().contiguous()
            out[:, lo:lo + 32768] = 30.0 * torch.tanh((state["hidden"].double() @ w) / 30.0)
        if family == "head":
            return out
        p = torch.tensor([_sampled_probability(out[r], state["policy"], state["draws"][r], state["histories"][r])
                          for r in range(rows)], dtype=torch.float64)
        return {"logits": out, "tokens": None, "probabilities": p}
    hist = state["histories"]
    p = torch.empty(rows, dtype=torch.float64)
    allowed = None
    if family == "step":
        offsets, data = wl.synthetic_vocab(vocab=vocab)
        allowed = _legal(offsets, data, *wl.synthetic_dfa(), states=state["states"])
    for r in range(rows):
        x = state["logits"][r].double()
        if allowed is not None:
            x = x.masked_fill(~torch.from_numpy(allowed[r]).to(x.device), -math.inf)
        p[r] = _sampled_probability(x, state["policy"], state["draws"][r], None if hist is None else hist[r])
    if family == "step":
        return {"masks": None, "tokens": None, "probabilities": p}
    return {"tokens": None, "probabilities": p}


def _legal(offsets, data, nxt, finals, states):
    """Which tokens each state's bytes allow: every step has an edge to a state
    that still reaches a final one."""
    viable = finals.astype(bool)
    while True:
        more = viable | ((nxt >= 0) & viable[nxt]).any(axis=1)
        if (more == viable).all():
            break
        viable = more
    step = np.where((nxt >= 0) & viable[nxt], nxt, -1)
    lengths = np.diff(offsets)
    out = {}
    for s0 in sorted(set(int(s) for s in states)):
        s = np.where(lengths > 0, s0, -1)
        for i in range(int(lengths.max())):
            live = np.flatnonzero((s >= 0) & (lengths > i))
            s[live] = step[s[live], data[offsets[live] + i]]
        out[s0] = s >= 0
    return [out[int(s)] for s in states]
