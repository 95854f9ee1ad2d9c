"""The calls whose speed this repository answers for, as a user's program makes them.

A case is a dict of plain values.  Its ``path`` says which public entry points
one pass goes through:

* ``decode``      one token for every live sequence: the Q/K/V convolution on
                  its cached history (``conv``), the slot-pool state update,
                  the gated norm (``conv``); or the state update alone;
* ``prefill``     prompts through the chunked forward into pool slots;
* ``train``       ``chunk_pkda`` with a per-head log decay, forward and
                  backward (rows, packed documents, an initial state);
* ``production``  ``pkda_recurrence``, the training operator with the raw
                  per-channel gate and the preconditioner, both ways;
* ``mixer``       the mixer between its projections: convolution, controls,
                  ``chunk_pkda`` with the decay expansion, gated norm, both ways;
* ``conv``        ``pkda_qkv_conv`` both ways;
* ``norm_gate``   ``pkda_norm_gate`` both ways.

Sizes and draws are those of ``bench.py`` and ``tests/``: heads 4 to 32 of 64
or 128 channels, the bench's rows of 4,096 and 16,384 tokens, its geometric
documents, its 512-slot decode pool, and ragged lengths between.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from delta_feedback_experiment_amd import (chunk_pkda, pkda_controls, pkda_decode_step_,
                                           pkda_norm_gate, pkda_prefill_, pkda_qkv_conv, pkda_qkv_conv_cached_,
                                           pkda_recurrence)

SQUASH_X, EPS = 1.5, 1e-6
TAPS = 4
CHUNK = 64


# -- the cases -----------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # a chat server between requests: four sequences decode, so the calls
        # and launches of one layer are the whole cost
        _decode("decode_few", live=4, slots=16, H=8, D=128, gate="raw", conv=True),
        # the bench's loaded server: 256 of 512 slots, 1 GiB of state per step
        _decode("decode_full", live=256, slots=512, H=32, D=128, gate="head", conv=False),
        # one prompt of a few pages, the time to its first token
        _prefill("prefill_prompt", prompts=1, tokens=1531, H=8, D=128, gate="raw"),
        # a batch of prompts of mixed lengths, packed
        _prefill("prefill_packed", prompts=13, tokens=12001, H=16, D=128, gate="raw"),
        # the headline step: rows of 4,096 tokens, per-head decay
        _train("train_rows", B=8, T=4096, H=16, D=128),
        # the same tokens as packed documents of geometric lengths
        _train("train_packed", B=1, T=32768, H=16, D=128, docs=32),
        # long rows that continue from a state, a tenth of the tokens decaying hard
        _train("train_long", B=2, T=16384, H=32, D=128, state=True, strong=True),
        # the model's own training operator at the headline geometry
        _production("production_rows", B=8, T=4096, H=16, D=128),
        # the same in FP32, as a numerics check or a small study runs it: short ragged rows
        _production("production_fp32", B=4, T=777, H=4, D=64, dtype="float32"),
        # a whole mixer at the smaller geometry, rows that fill no last chunk
        {"name": "mixer_ragged", "path": "mixer", "B": 3, "T": 1000, "H": 8, "D": 128, "dtype": "bfloat16",
         "lean": True},
        # the recurrence's producer and consumer in a training step
        {"name": "conv_rows", "path": "conv", "B": 8, "T": 4096, "H": 8, "D": 128, "dtype": "bfloat16"},
        {"name": "norm_gate_rows", "path": "norm_gate", "B": 8, "T": 4096, "H": 16, "D": 128, "dtype": "bfloat16"},
    ]


def _decode(name, *, live, slots, H, D, gate, conv, dtype="bfloat16"):
    return _named(name, path="decode", live=live, slots=slots, H=H, D=D, gate=gate, conv=conv, dtype=dtype)


def _prefill(name, *, prompts, tokens, H, D, gate, resume=False, dtype="bfloat16"):
    return _named(name, path="prefill", prompts=prompts, tokens=tokens, H=H, D=D, gate=gate, resume=resume,
                  dtype=dtype)


def _train(name, *, B, T, H, D, docs=0, state=False, strong=False, lean=False, dtype="bfloat16"):
    return _named(name, path="train", B=B, T=T, H=H, D=D, docs=docs, state=state, strong=strong, lean=lean,
                  dtype=dtype)


def _production(name, *, B, T, H, D, lean=False, dtype="bfloat16"):
    return _named(name, path="production", B=B, T=T, H=H, D=D, lean=lean, dtype=dtype)


def _named(name, **case):
    return case if name is None else {"name": name, **case}


def draw(rng) -> dict:
    """One more case of the same ranges: sizes spread over their logarithm,
    at most a quarter of the largest listed case's token-heads."""
    path = rng.choice(("decode", "decode", "prefill", "prefill", "train", "train", "production", "production",
                       "mixer", "conv", "norm_gate"))
    H, D = rng.choice((4, 8, 16, 32)), rng.choice((64, 128, 128, 128))
    if path == "decode":
        live = _log_int(rng, 1, 256)
        conv = rng.random() < 0.5
        return _decode(None, live=live, slots=live + _log_int(rng, 1, 256), H=H, D=D,
                       gate="raw" if conv else rng.choice(("raw", "head")), conv=conv,
                       dtype="float32" if rng.random() < 0.15 else "bfloat16")
    if path == "prefill":
        prompts = _log_int(rng, 1, 24)
        tokens = _log_int(rng, max(16, 4 * prompts), min(32768, 2 ** 18 // H))
        return _prefill(None, prompts=prompts, tokens=tokens, H=H, D=D, gate=rng.choice(("raw", "raw", "head")),
                        resume=rng.random() < 0.3)
    fp32 = rng.random() < 0.2 and path in ("train", "production")  # built for 64 channels
    if fp32:
        H, D = min(H, 8), 64
    tokens = _log_int(rng, 200, min(8192, 2 ** 15 // H) if fp32 else 2 ** 18 // H)
    B = min(_log_int(rng, 1, 16), max(1, tokens // 50))
    T = max(1, tokens // B)
    dtype = "float32" if fp32 else "bfloat16"
    if path == "train":
        docs = _log_int(rng, 2, 64) if rng.random() < 0.4 else 0
        if docs:
            B, T = 1, max(B * T, 8 * docs)
        return _train(None, B=B, T=T, H=H, D=D, docs=docs, state=rng.random() < 0.3, strong=rng.random() < 0.3,
                      lean=rng.random() < 0.25, dtype=dtype)
    if path == "production":
        return _production(None, B=B, T=T, H=H, D=D, lean=rng.random() < 0.4, dtype=dtype)
    case = {"path": path, "B": B, "T": T, "H": H, "D": D, "dtype": dtype}
    return {**case, "lean": rng.random() < 0.5} if path == "mixer" else case


def _log_int(rng, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(max(low, high)))))))


# -- inputs --------------------------------------------------------------------

def _device() -> torch.device:
    return torch.device("cuda", torch.cuda.current_device())


class _Draw:
    """The bench's distributions from one seeded generator on the device."""

    def __init__(self, seed: int, dtype: torch.dtype):
        self.dev, self.dtype = _device(), dtype
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=self.dev)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=self.dev)

    def act(self, *shape, scale: float = 1.0):
        return (scale * self.normal(*shape)).to(self.dtype)

    def unit(self, *shape):
        t = self.normal(*shape)
        return (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)).to(self.dtype)

    def raw_gate(self, lead, H, D):
        """Raw decay projection, A_log, dt_bias; the preconditioner's decay,
        strength and log-space center."""
        return dict(
            g=self.act(*lead, H, D, scale=0.2),
            A_log=(1.0 + 15.0 * self.uniform(H)).log(),
            dt_bias=0.1 * self.normal(H * D),
            g_atk=-F.softplus(0.2 * self.normal(*lead, H) + 0.3),
            beta_atk=torch.sigmoid(self.normal(*lead, H)),
            center=-0.2 + 0.1 * self.normal(H),
        )


def _dtype(case) -> torch.dtype:
    return {"bfloat16": torch.bfloat16, "float32": torch.float32}[case["dtype"]]


def _lengths(parts: int, total: int, seed: int) -> list[int]:
    """``parts`` positive lengths that sum to ``total``, exponentially spread."""
    u = torch.rand(parts, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    w = -torch.log1p(-u) + 0.02
    cuts = (torch.cumsum(w, 0) / w.sum() * (total - parts)).round().long().tolist()
    cuts[-1] = total - parts
    return [b - a + 1 for a, b in zip([0] + cuts[:-1], cuts)]


def _cu(lengths: list[int], dev) -> torch.Tensor:
    return torch.tensor([0] + lengths, dtype=torch.int64).cumsum(0).to(torch.int32).to(dev)


def _slots(n: int, pool: int, seed: int, dev) -> torch.Tensor:
    return torch.randperm(pool, generator=torch.Generator().manual_seed(seed))[:n].to(torch.int32).to(dev)


def _leaves(**tensors):
    return {n: t.requires_grad_() for n, t in tensors.items()}


def prepare(case: dict, seed: int) -> dict:
    r = _Draw(seed, _dtype(case))
    state = _PREPARE[case["path"]](case, seed, r)
    return {"case": case, **state}


def _prepare_decode(c, seed, r):
    n, P, H, D = c["live"], c["slots"], c["H"], c["D"]
    s = dict(
        slot=_slots(n, P, seed, r.dev), pool=0.02 * r.normal(P, H, D, D), q=r.unit(n, H, D), k=r.unit(n, H, D),
        v=r.act(n, H, D), beta=torch.sigmoid(0.2 * r.normal(n, H)),
    )
    if c["gate"] == "raw":
        s.update(r.raw_gate((n,), H, D), a_pool=r.uniform(P, H, D) / D)
    else:
        s["g"] = -F.softplus(r.normal(n, H))
    if c["conv"]:
        s.update(x=r.act(n, 1, 3 * H * D), conv_weight=0.5 * r.normal(3 * H * D, TAPS),
                 conv_pool=r.act(P, TAPS - 1, 3 * H * D), out_gate=r.act(n, H, D), norm=1.0 + 0.1 * r.normal(D))
    return s


def _prepare_prefill(c, seed, r):
    N, T, H, D = c["prompts"], c["tokens"], c["H"], c["D"]
    P = 2 * N + 3
    s = dict(
        slot=_slots(N, P, seed, r.dev), pool=0.02 * r.normal(P, H, D, D), q=r.unit(1, T, H, D), k=r.unit(1, T, H, D),
        v=r.act(1, T, H, D), lengths=_lengths(N, T, seed),
    )
    s["cu"] = None if N == 1 else _cu(s["lengths"], r.dev)
    if c["gate"] == "raw":
        s.update(r.raw_gate((1, T), H, D), a_pool=r.uniform(P, H, D) / D, beta=torch.sigmoid(0.2 * r.normal(1, T, H)))
    else:
        s.update(g=-F.softplus(r.normal(1, T, H)), beta=torch.sigmoid(r.normal(1, T, H)))
    return s


def _prepare_train(c, seed, r):
    B, T, H, D = c["B"], c["T"], c["H"], c["D"]
    lengths = _lengths(c["docs"], T, seed) if c["docs"] else [T] * B
    g = -F.softplus(r.normal(B, T, H))
    if c["strong"]:
        g = torch.where((r.uniform(B, T) < 0.1)[:, :, None], torch.full_like(g, -8.0), g)
    leaves = _leaves(q=r.unit(B, T, H, D), k=r.unit(B, T, H, D), v=r.act(B, T, H, D), g=g,
                     beta=torch.sigmoid(r.normal(B, T, H)))
    s = dict(do=r.act(B, T, H, D), lengths=lengths, cu=_cu(lengths, r.dev) if c["docs"] else None)
    if c["state"]:
        leaves.update(_leaves(s0=0.02 * r.normal(len(lengths), H, D, D)))
        s["dS"] = 0.02 * r.normal(len(lengths), H, D, D)
    return dict(s, leaves=leaves)


_PRODUCTION = ("q", "k", "v", "g", "g_atk", "beta_atk", "beta", "A_log", "dt_bias", "center")


def _prepare_production(c, seed, r):
    B, T, H, D = c["B"], c["T"], c["H"], c["D"]
    t = dict(q=r.unit(B, T, H, D), k=r.unit(B, T, H, D), v=r.act(B, T, H, D),
             beta=torch.sigmoid(0.2 * r.normal(B, T, H)), **r.raw_gate((B, T), H, D))
    return dict(leaves=_leaves(**{n: t[n] for n in _PRODUCTION}), do=r.act(B, T, H, D))


def _prepare_mixer(c, seed, r):
    B, T, H, D = c["B"], c["T"], c["H"], c["D"]
    bound = D ** -0.5
    leaves = _leaves(
        x=r.act(B, T, 3 * H * D), conv_weight=0.5 * r.normal(3 * H * D, TAPS),
        packed=r.act(B, T, 2 * D + 3 * H, scale=3 ** -0.5),
        decay_up=(bound * (2 * r.uniform(H * D, D) - 1)).to(r.dtype),
        A_log=(1.0 + 15.0 * r.uniform(H)).log(), dt_bias=0.1 * r.normal(H * D),
        A_log_p=(1.0 + r.uniform(H)).log(), dt_bias_p=0.1 * r.normal(H), center=-0.2 + 0.1 * r.normal(H),
        out_gate=r.act(B, T, H, D), norm=1.0 + 0.1 * r.normal(D),
    )
    return dict(leaves=leaves, dy=r.act(B, T, H, D), d_gate_hidden=r.act(B, T, D))


def _prepare_conv(c, seed, r):
    B, T, W = c["B"], c["T"], c["H"] * c["D"]
    leaves = _leaves(x=r.act(B, T, 3 * W), conv_weight=0.5 * r.normal(3 * W, TAPS))
    return dict(leaves=leaves, grads=[r.act(B, T, W) for _ in range(3)])


def _prepare_norm_gate(c, seed, r):
    shape = (c["B"], c["T"], c["H"], c["D"])
    leaves = _leaves(o=r.act(*shape), out_gate=r.act(*shape), norm=1.0 + 0.1 * r.normal(c["D"]))
    return dict(leaves=leaves, dy=r.act(*shape))


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "train": _prepare_train,
            "production": _prepare_production, "mixer": _prepare_mixer, "conv": _prepare_conv,
            "norm_gate": _prepare_norm_gate}


# -- one pass ------------------------------------------------------------------

def run(state: dict) -> dict:
    return _RUN[state["case"]["path"]](state["case"], state)


def _raw_gate_args(s) -> dict:
    return dict(g_atk=s["g_atk"], beta_atk=s["beta_atk"], log_atk_scale=s["center"], A_log=s["A_log"],
                dt_bias=s["dt_bias"], use_gate_in_kernel=True, x=SQUASH_X, eps=EPS)


def _run_decode(c, s):
    H, D = c["H"], c["D"]
    q, k, v, out = s["q"], s["k"], s["v"], {}
    if c["conv"]:
        qkv = pkda_qkv_conv_cached_(s["x"], s["conv_weight"], D, 2 * H * D, EPS, s["conv_pool"], s["slot"])
        q, k, v = (t.reshape(-1, H, D) for t in qkv)
        out["conv_pool"] = s["conv_pool"]
    if c["gate"] == "raw":
        o = pkda_decode_step_(q, k, v, s["g"], s["beta"], s["pool"], s["slot"], a_pool=s["a_pool"],
                              **_raw_gate_args(s))
        out["a_pool"] = s["a_pool"]
    else:
        o = pkda_decode_step_(q, k, v, s["g"], s["beta"], s["pool"], s["slot"])
    if c["conv"]:
        o = pkda_norm_gate(o, s["out_gate"], s["norm"], EPS)[0]
    return {**out, "o": o, "pool": s["pool"]}


def _run_prefill(c, s):
    more = dict(_raw_gate_args(s), a_pool=s["a_pool"]) if c["gate"] == "raw" else {}
    o = pkda_prefill_(s["q"], s["k"], s["v"], s["g"], s["beta"], s["pool"], s["slot"], cu_seqlens=s["cu"],
                      continue_state=c["resume"], **more)
    return {"o": o, "pool": s["pool"], **({"a_pool": s["a_pool"]} if more else {})}


def _gradients(outputs, leaves, grads) -> dict:
    return dict(zip(("d" + n for n in leaves), torch.autograd.grad(outputs, list(leaves.values()), grads)))


def _run_train(c, s):
    p = s["leaves"]
    o, S, _ = chunk_pkda(p["q"], p["k"], p["v"], p["g"], p["beta"], initial_state=p.get("s0"),
                         output_final_state=c["state"], cu_seqlens=s["cu"], lean=c["lean"])
    outputs, grads = ([o, S], [s["do"], s["dS"]]) if c["state"] else ([o], [s["do"]])
    got = _gradients(outputs, p, grads)
    return {"o": o.detach(), **({"S": S.detach()} if c["state"] else {}), **got}


def _run_production(c, s):
    p = s["leaves"]
    o, _ = pkda_recurrence(*(p[n] for n in _PRODUCTION), c["D"] ** -0.5, SQUASH_X, EPS, c["lean"])
    return {"o": o.detach(), **_gradients([o], p, [s["do"]])}


def _run_mixer(c, s):
    p, lead = s["leaves"], (c["B"], c["T"], c["H"], c["D"])
    H, D = c["H"], c["D"]
    q, k, v = (t.reshape(lead) for t in pkda_qkv_conv(p["x"], p["conv_weight"], D, 2 * H * D, EPS))
    hidden, beta, g_atk, beta_atk, gate_hidden = pkda_controls(p["packed"], p["A_log_p"], p["dt_bias_p"], D, H)
    o, _, _ = chunk_pkda(q, k, v, hidden, beta, decay_up=p["decay_up"], A_log=p["A_log"], dt_bias=p["dt_bias"],
                         use_gate_in_kernel=True, g_atk=g_atk, beta_atk=beta_atk, log_atk_scale=p["center"],
                         x=SQUASH_X, eps=EPS, lean=c["lean"])
    y = pkda_norm_gate(o, p["out_gate"], p["norm"], EPS)[0]
    return {"y": y.detach(), **_gradients([y, gate_hidden], p, [s["dy"], s["d_gate_hidden"]])}


def _run_conv(c, s):
    p = s["leaves"]
    qkv = pkda_qkv_conv(p["x"], p["conv_weight"], c["D"], 2 * c["H"] * c["D"], EPS)
    got = _gradients(list(qkv), p, s["grads"])
    return {**dict(zip("qkv", (t.detach() for t in qkv))), **got}


def _run_norm_gate(c, s):
    p = s["leaves"]
    y, _ = pkda_norm_gate(p["o"], p["out_gate"], p["norm"], EPS)
    return {"y": y.detach(), **_gradients([y], p, [s["dy"]])}


_RUN = {"decode": _run_decode, "prefill": _run_prefill, "train": _run_train, "production": _run_production,
        "mixer": _run_mixer, "conv": _run_conv, "norm_gate": _run_norm_gate}


# -- what a pass cannot do without ----------------------------------------------

def work(case: dict) -> dict:
    """Each input read once, each output written once; the recurrence's chunked
    products (chunks of 64 tokens: forward 6 d^2 + 10 C d per token and head,
    forward and backward three times that)."""
    H, D, a = case["H"], case["D"], _dtype(case).itemsize
    path = case["path"]
    if path == "decode":
        n, raw = case["live"], case["gate"] == "raw"
        per_head = 8 * D * D + 4 * D * a + 4 + (D * a + 8 * D + 8 if raw else 4)
        # the convolution reads x, its history and the taps, and leaves the history
        conv = n * 3 * H * D * a * (2 * TAPS - 1) + 3 * H * D * TAPS * 4 + n * H * D * a if case["conv"] else 0
        return {"bytes": n * H * per_head + 4 * n + conv, "flops": 6 * n * H * D * D}
    tokens = case["tokens"] if path == "prefill" else case["B"] * case["T"]
    th, act = tokens * H, tokens * H * D * a
    forward = th * (6 * D * D + 10 * CHUNK * D)
    if path == "prefill":
        raw = case["gate"] == "raw"
        states = case["prompts"] * H * (D * D + (D if raw else 0)) * 4 * (2 if case["resume"] else 1)
        return {"bytes": 4 * act + (act + 12 * th if raw else 8 * th) + states, "flops": forward}
    if path == "train":
        states = 4 * (case["docs"] or case["B"]) * H * D * D * 4 if case["state"] else 0
        return {"bytes": 8 * act + 16 * th + states, "flops": 3 * forward}
    if path == "production":
        return {"bytes": 10 * act + 24 * th, "flops": 3 * forward}
    if path == "mixer":
        packed = tokens * (2 * D + 3 * H) * a
        return {"bytes": 10 * act + 2 * packed + tokens * D * a + 2 * H * D * (D * a + 4 * 3 * TAPS),
                "flops": 3 * forward + 6 * th * D * D}
    if path == "conv":
        return {"bytes": 12 * act + 2 * 3 * H * D * TAPS * 4, "flops": 3 * act // a * (6 * TAPS + 12)}
    return {"bytes": 6 * act, "flops": 20 * act // a}


def tolerance(case: dict) -> dict:
    """About four times the largest error against ``exact`` of any output: FP32
    4.4e-6 (the gate's bias gradient), the single BF16 roundings of the
    convolution and the norm 1.7e-3, the BF16 recurrence 3.7e-3.  The mixer's
    ``dA_log`` sums a gate gradient whose terms cancel over rounded queries and
    keys: 1.2e-2 to 2.7e-2 from ``exact``."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-3}
    if case["path"] in ("conv", "norm_gate"):
        return {"rel": 6e-3, "max": 5e-2}
    return {"rel": 3e-2 if case["path"] == "mixer" else 1.2e-2, "max": 0.4}


# -- 64-bit results --------------------------------------------------------------

def exact(case: dict, seed: int):
    """``run``'s outputs in 64 bits, token by token."""
    s = prepare(case, seed)
    for name, t in list(s.get("leaves", {}).items()):
        s["leaves"][name] = t.detach().double().requires_grad_()
    for name, t in list(s.items()):
        if torch.is_tensor(t) and t.is_floating_point():
            s[name] = t.double()
    if "grads" in s:
        s["grads"] = [t.double() for t in s["grads"]]
    return _EXACT[case["path"]](case, s)


def _segment(q, k, v, g, beta, S, A, g_atk, beta_atk, center, scale):
    """Tokens one after another from the states ``S [N, H, K, V]``, ``A [N, H, K]``."""
    kw = k
    if g_atk is not None:
        decay, gain, A_t = g_atk.exp().unbind(1), (beta_atk.unsqueeze(-1) * k * k).unbind(1), []
        for a, b in zip(decay, gain):
            A = a.unsqueeze(-1) * A + b
            A_t.append(A)
        rise = torch.log(torch.stack(A_t, 1) + EPS) - center[:, None]
        kw = k * torch.exp(-math.log(SQUASH_X) * rise / (1 + rise.abs()))
    alpha = (g if g.dim() == 4 else g.unsqueeze(-1)).exp()
    out = []
    for q_t, k_t, w_t, v_t, a_t, b_t in zip(*(t.unbind(1) for t in ((scale * q), k, kw, v, alpha, beta))):
        S = S * a_t.unsqueeze(-1)
        miss = v_t - (S * k_t.unsqueeze(-1)).sum(-2)
        S = S + w_t.unsqueeze(-1) * (b_t.unsqueeze(-1) * miss).unsqueeze(-2)
        out.append((S * q_t.unsqueeze(-1)).sum(-2))
    return torch.stack(out, 1), S, A


class _Recurrence(torch.autograd.Function):
    """:func:`_segment` over whole rows, holding one segment's graph at a time."""

    LENGTH = 32

    @staticmethod
    def forward(ctx, scale, S, A, center, *tokens):
        ctx.scale, entering, out = scale, [], []
        for at in range(0, tokens[0].shape[1], _Recurrence.LENGTH):
            entering += [S, A]
            o, S, A = _Recurrence.part(scale, S, A, center, tokens, at)
            out.append(o)
        ctx.save_for_backward(center, *tokens, *entering)
        ctx.count = len(tokens)
        return torch.cat(out, 1), S, A

    @staticmethod
    def part(scale, S, A, center, tokens, at):
        cut = [None if t is None else t[:, at:at + _Recurrence.LENGTH] for t in tokens]
        q, k, v, g, beta, g_atk, beta_atk = cut
        return _segment(q, k, v, g, beta, S, A, g_atk, beta_atk, center, scale)

    @staticmethod
    def backward(ctx, do, dS, dA):
        center, *rest = ctx.saved_tensors
        tokens, entering = rest[:ctx.count], rest[ctx.count:]
        grads = [None if t is None else torch.zeros_like(t) for t in tokens]
        dcenter = torch.zeros_like(center)
        dS = torch.zeros_like(entering[0]) if dS is None else dS
        dA = torch.zeros_like(entering[1]) if dA is None else dA
        for i in reversed(range(len(entering) // 2)):
            at = i * _Recurrence.LENGTH
            cut = [None if t is None else t[:, at:at + _Recurrence.LENGTH].detach().requires_grad_() for t in tokens]
            S, A, c = (t.detach().requires_grad_() for t in (*entering[2 * i:2 * i + 2], center))
            with torch.enable_grad():
                q, k, v, g, beta, g_atk, beta_atk = cut
                made = _segment(q, k, v, g, beta, S, A, g_atk, beta_atk, c, ctx.scale)
            wanted = [S, A, c] + [t for t in cut if t is not None]
            got = torch.autograd.grad(made, wanted, (do[:, at:at + _Recurrence.LENGTH], dS, dA), allow_unused=True)
            got = [torch.zeros_like(t) if x is None else x for t, x in zip(wanted, got)]
            dS, dA = got[0], got[1]
            dcenter += got[2]
            left = iter(got[3:])
            for grad in grads:
                if grad is not None:
                    grad[:, at:at + _Recurrence.LENGTH] = next(left)
        return (None, dS, dA, dcenter, *grads)


def _exact_recurrence(q, k, v, g, beta, lengths=None, S0=None, A0=None, g_atk=None, beta_atk=None, center=None):
    """``(o, S_T, A_T)`` of rows ``[B, T, H, D]`` or, with ``lengths``, of one
    packed row whose documents run side by side, padded with tokens that leave
    the state as it is (zero log decay, nothing written)."""
    H, D = q.shape[2:]
    tokens = [q, k, v, g, beta, g_atk, beta_atk]
    packed = lengths is not None and q.shape[0] == 1 and len(lengths) > 1
    if packed:
        longest = max(lengths)
        at = torch.zeros(len(lengths), longest, dtype=torch.int64)
        live = torch.zeros(len(lengths), longest, dtype=torch.bool)
        first = 0
        for n, length in enumerate(lengths):
            at[n, :length] = torch.arange(first, first + length)
            live[n, :length] = True
            first += length
        at, live = at.to(q.device), live.to(q.device)
        tokens = [None if t is None else t[0][at] * live.reshape(*live.shape, *(1,) * (t.dim() - 2)).to(t.dtype)
                  for t in tokens]
    N = tokens[0].shape[0]
    S0 = q.new_zeros(N, H, D, D) if S0 is None else S0
    A0 = q.new_zeros(N, H, D) if A0 is None else A0
    center = q.new_zeros(H) if center is None else center
    o, S, A = _Recurrence.apply(D ** -0.5, S0, A0, center, *tokens)
    return (o[live].unsqueeze(0) if packed else o), S, A


def _log_decay(raw, A_log, dt_bias):
    H, D = raw.shape[-2:]
    return -A_log.exp()[:, None] * F.softplus(raw + dt_bias.reshape(H, D))


def _exact_conv(x, weight, history, H, D):
    """Q, K and V slabs: the causal taps, SiLU, unit queries and keys."""
    B, T, _ = x.shape
    rows = torch.cat((history, x), 1)
    y = F.silu(sum(weight[:, w] * rows[:, w:w + T] for w in range(TAPS)))
    q, k, v = y.reshape(B, T, 3, H, D).unbind(2)
    q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + EPS) for t in (q, k))
    return tuple(t.reshape(B, T, H * D) for t in (q, k, v)), rows[:, T:]


def _exact_norm_gate(o, gate, weight):
    return o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS) * weight * torch.sigmoid(gate)


def _exact_decode(c, s):
    H, D, i = c["H"], c["D"], s["slot"].long()
    q, k, v, out = s["q"], s["k"], s["v"], {}
    if c["conv"]:
        qkv, history = _exact_conv(s["x"], s["conv_weight"], s["conv_pool"][i], H, D)
        q, k, v = (t.reshape(-1, H, D) for t in qkv)
        out["conv_pool"] = s["conv_pool"].index_copy(0, i, history)
    tokens = [t.unsqueeze(1) for t in (q, k, v)]
    beta, pool = s["beta"].unsqueeze(1), s["pool"]
    if c["gate"] == "raw":
        g = _log_decay(s["g"], s["A_log"], s["dt_bias"]).unsqueeze(1)
        o, S, A = _exact_recurrence(*tokens, g, beta, S0=pool[i], A0=s["a_pool"][i], g_atk=s["g_atk"].unsqueeze(1),
                                    beta_atk=s["beta_atk"].unsqueeze(1), center=s["center"])
        out["a_pool"] = s["a_pool"].index_copy(0, i, A)
    else:
        o, S, _ = _exact_recurrence(*tokens, s["g"].unsqueeze(1), beta, S0=pool[i])
    o = o.squeeze(1)
    if c["conv"]:
        o = _exact_norm_gate(o, s["out_gate"], s["norm"])
    return {**out, "o": o, "pool": pool.index_copy_(0, i, S)}


def _exact_prefill(c, s):
    i, more, g = s["slot"].long(), {}, s["g"]
    if c["gate"] == "raw":
        g = _log_decay(g, s["A_log"], s["dt_bias"])
        more = dict(g_atk=s["g_atk"], beta_atk=s["beta_atk"], center=s["center"],
                    A0=s["a_pool"][i] if c["resume"] else None)
    o, S, A = _exact_recurrence(s["q"], s["k"], s["v"], g, s["beta"], s["lengths"],
                                S0=s["pool"][i] if c["resume"] else None, **more)
    out = {"o": o, "pool": s["pool"].index_copy(0, i, S)}
    return {**out, "a_pool": s["a_pool"].index_copy(0, i, A)} if more else out


def _exact_train(c, s):
    p = s["leaves"]
    o, S, _ = _exact_recurrence(p["q"], p["k"], p["v"], p["g"], p["beta"], s["lengths"] if c["docs"] else None,
                                S0=p.get("s0"))
    outputs, grads = ([o, S], [s["do"], s["dS"]]) if c["state"] else ([o], [s["do"]])
    got = _gradients(outputs, p, grads)
    return {"o": o.detach(), **({"S": S.detach()} if c["state"] else {}), **got}


def _exact_production(c, s):
    p = s["leaves"]
    o, _, _ = _exact_recurrence(p["q"], p["k"], p["v"], _log_decay(p["g"], p["A_log"], p["dt_bias"]), p["beta"],
                                g_atk=p["g_atk"], beta_atk=p["beta_atk"], center=p["center"])
    return {"o": o.detach(), **_gradients([o], p, [s["do"]])}


def _exact_mixer(c, s):
    p, lead, H, D = s["leaves"], (c["B"], c["T"], c["H"], c["D"]), c["H"], c["D"]
    zeros = p["x"].new_zeros(c["B"], TAPS - 1, 3 * H * D)
    q, k, v = (t.reshape(lead) for t in _exact_conv(p["x"], p["conv_weight"], zeros, H, D)[0])
    hidden, beta, g_atk, beta_atk, gate_hidden = p["packed"].split((D, H, H, H, D), -1)
    g = _log_decay((hidden @ p["decay_up"].t()).reshape(lead), p["A_log"], p["dt_bias"])
    g_atk = -p["A_log_p"].exp() * F.softplus(g_atk + p["dt_bias_p"])
    o, _, _ = _exact_recurrence(q, k, v, g, torch.sigmoid(beta), g_atk=g_atk, beta_atk=torch.sigmoid(beta_atk),
                                center=p["center"])
    y = _exact_norm_gate(o, p["out_gate"], p["norm"])
    return {"y": y.detach(), **_gradients([y, gate_hidden], p, [s["dy"], s["d_gate_hidden"]])}


def _exact_conv_rows(c, s):
    p = s["leaves"]
    zeros = p["x"].new_zeros(c["B"], TAPS - 1, p["x"].shape[-1])
    qkv, _ = _exact_conv(p["x"], p["conv_weight"], zeros, c["H"], c["D"])
    got = _gradients(list(qkv), p, s["grads"])
    return {**dict(zip("qkv", (t.detach() for t in qkv))), **got}


def _exact_norm_gate_rows(c, s):
    p = s["leaves"]
    y = _exact_norm_gate(p["o"], p["out_gate"], p["norm"])
    return {"y": y.detach(), **_gradients([y], p, [s["dy"]])}


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "train": _exact_train, "production": _exact_production,
          "mixer": _exact_mixer, "conv": _exact_conv_rows, "norm_gate": _exact_norm_gate_rows}
