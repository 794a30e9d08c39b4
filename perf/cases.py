"""What the framework's performance is measured on: a user's calls through the public entry points.

``listed()`` holds the calls that matter in serving and training a Gated DeltaNet layer at the two head layouts
this framework is used with (4 qk / 8 v heads and 16 qk / 32 v heads, head dim 128); ``draw`` gives more of the
same ranges.  ``prepare`` makes a call's inputs on the GPU, ``run`` is one pass, ``exact`` its results in 64 bits
by plain torch.

Kinds:
  decode   one token per sequence, state out of place    (``decode.run`` / ``decode.gdn_decode``)
  multi    T tokens per sequence, as draft verification  (``decode.gdn_decode_multi``)
  pool     one token per sequence, states in a slot pool (``decode.decode_pool_``)
  update   the decode conv1d, conv states in place       (``conv.qkv_conv1d_update``)
  conv     the prefill conv1d over packed sequences      (``conv.qkv_conv1d``)
  prefill  packed sequences through the chunked rule     (``prefill.run`` / ``prefill.gdn_prefill``)
  train    forward and backward of the prefill           (``backward.chunk_gated_delta_rule``)
"""

import importlib
import math
import random

import torch

import __graft_entry__

_PACKAGE = __graft_entry__.load_package().__name__
_decode, _prefill, _conv, _backward = (importlib.import_module(f"{_PACKAGE}.{m}")
                                       for m in ("decode", "prefill", "conv", "backward"))

D = 128          # head dimension
CHUNK = 64       # tokens per chunk of the exact form (any size gives the same values)
WIDTH = 4        # conv taps
SCALE = 1.0 / math.sqrt(D)


def listed():
    return [
        # one user's stream: a single decode step, where the call itself is what counts
        {"name": "decode_b1", "kind": "decode", "batch": 1, "hq": 4, "hv": 8, "l2norm": False},
        # the decode step of a full serving batch
        {"name": "decode_b256", "kind": "decode", "batch": 256, "hq": 4, "hv": 8, "l2norm": False},
        # verification of four draft tokens and their successor, an odd batch, q and k normalised in the call
        {"name": "multi_b61_t5", "kind": "multi", "batch": 61, "tokens": 5, "hq": 16, "hv": 32, "l2norm": True},
        # the largest decode: a continuous-batching server's pool with spare slots
        {"name": "pool_b1024", "kind": "pool", "batch": 1024, "hq": 16, "hv": 32},
        # the decode conv1d of the same batch
        {"name": "update_b1024", "kind": "update", "batch": 1024, "hq": 16, "hv": 32},
        # the conv1d ahead of the largest prefill
        {"name": "conv_t32768", "kind": "conv", "n": 8, "tokens": 32768, "spread": 0.5, "hq": 16, "hv": 32},
        # short prompts of odd lengths joining a running batch, states carried, q and k normalised in the call
        {"name": "prefill_ragged24", "kind": "prefill", "n": 24, "tokens": 6143, "spread": 0.95, "hq": 16, "hv": 32,
         "state": True, "l2norm": True, "int32": True},
        # one prompt
        {"name": "prefill_t4096", "kind": "prefill", "n": 1, "tokens": 4096, "spread": 0.0, "hq": 4, "hv": 8,
         "state": False, "l2norm": False, "int32": False},
        # sixteen prompts of very different lengths
        {"name": "prefill_varlen16", "kind": "prefill", "n": 16, "tokens": 59289, "spread": 0.95, "hq": 4, "hv": 8,
         "state": True, "l2norm": False, "int32": True},
        # the largest prefill
        {"name": "prefill_t32768", "kind": "prefill", "n": 8, "tokens": 32768, "spread": 0.5, "hq": 16, "hv": 32,
         "state": True, "l2norm": False, "int32": False},
        # a training step of a layer on one sequence, and on a large packed batch
        {"name": "train_t4096", "kind": "train", "n": 1, "tokens": 4096, "spread": 0.0, "hq": 4, "hv": 8,
         "state": False, "int32": False},
        {"name": "train_t32768", "kind": "train", "n": 8, "tokens": 32768, "spread": 0.5, "hq": 16, "hv": 32,
         "state": False, "int32": False},
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], its logarithm uniform."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "multi", "pool", "update", "conv", "prefill", "prefill", "train"])
    hq, hv = rng.choice([(4, 8), (16, 32)])
    small = 1 if hv == 32 else 4                     # batches of the smaller layout reach further
    case = {"kind": kind, "hq": hq, "hv": hv}
    if kind == "decode":
        return {**case, "batch": _between(rng, 1, 256 * small), "l2norm": rng.random() < 0.5}
    if kind == "multi":
        return {**case, "batch": _between(rng, 1, 64 * small), "tokens": rng.randint(2, 8),
                "l2norm": rng.random() < 0.5}
    if kind in ("pool", "update"):
        return {**case, "batch": _between(rng, 1, 1024)}
    tokens = _between(rng, 32, 32768 if kind != "prefill" or hv == 32 else 65536)
    case.update(n=min(_between(rng, 1, 32), 1 + tokens // 16), tokens=tokens, spread=rng.choice([0.0, 0.5, 0.95]))
    if kind == "conv":
        return case
    case.update(state=rng.random() < 0.5, int32=rng.random() < 0.5)
    if kind == "prefill":
        case["l2norm"] = rng.random() < 0.5
    return case


def _lengths(case):
    """``n`` lengths of 1 or more that sum to ``tokens``, within ``spread`` of their mean before rescaling; the case
    alone decides them."""
    n, total = case["n"], case["tokens"]
    rng = random.Random(1000003 * total + n)
    w = [1.0 + case["spread"] * rng.uniform(-1.0, 1.0) for _ in range(n)]
    got = [max(1, int(x / sum(w) * total)) for x in w]
    got[got.index(max(got))] += total - sum(got)
    return got


def _inputs(case, seed):
    """The inputs by name, made on the GPU from the seed: q and k of unit length (raw where the call normalises
    them), v, a and b normal, states of standard deviation 0.02, per-head gate parameters."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.bfloat16):
        x = torch.randn(*shape, generator=gen, device="cuda")
        return (x.mul_(std) if std != 1.0 else x).to(dtype)

    kind, hq, hv = case["kind"], case["hq"], case["hv"]
    if kind in ("conv", "update"):
        channels = (2 * hq + hv) * D
        rows = case["tokens"] if kind == "conv" else case["batch"]
        x = {"x": normal(rows, channels), "weight": normal(channels, WIDTH, std=0.5, dtype=torch.float32),
             "bias": normal(channels, std=0.1, dtype=torch.float32)}
        if kind == "update":
            pool = case["batch"] + case["batch"] // 4
            x["slots"] = torch.randperm(pool, generator=gen, device="cuda")[:case["batch"]].to(torch.int32)
            x["conv_state"] = normal(pool, channels, WIDTH - 1)
            return x
        x["conv_state"] = normal(case["n"], channels, WIDTH - 1)
    else:
        batch = case.get("batch")
        lead = (case["tokens"],) if batch is None else (batch, case.get("tokens", 1))
        x = {"q": normal(*lead, hq, D, dtype=torch.float32), "k": normal(*lead, hq, D, dtype=torch.float32)}
        for name in ("q", "k"):
            if not case.get("l2norm"):
                x[name] /= x[name].norm(dim=-1, keepdim=True)
            x[name] = x[name].to(torch.bfloat16)
        x["v"] = normal(*lead, hv, D)
        x["a"], x["b"] = normal(*lead, hv), normal(*lead, hv)
        x["A_log"] = torch.rand(hv, generator=gen, device="cuda") * 2.0 - 2.0
        x["dt_bias"] = normal(hv, std=0.1, dtype=torch.float32)
        if kind == "pool":
            pool = batch + batch // 4
            x["slots"] = torch.randperm(pool, generator=gen, device="cuda")[:batch].to(torch.int32)
            x["state"] = normal(pool, hv, D, D, std=0.02, dtype=torch.float32)
        else:
            rows = case["n"] if batch is None else batch
            x["state"] = normal(rows, hv, D, D, std=0.02, dtype=torch.float32) if case.get("state", True) else None
        if batch is not None:
            return x
    ends = [0]
    for length in _lengths(case):
        ends.append(ends[-1] + length)
    x["cu"] = torch.tensor(ends, dtype=torch.int32 if case.get("int32") else torch.int64, device="cuda")
    if kind == "train":
        x["d_out"] = normal(case["tokens"], hv, D)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    x["case"] = case
    if case["kind"] == "train":
        x["wrt"] = [x[n] for n in ("q", "k", "v", "A_log", "a", "dt_bias", "b", "state") if x[n] is not None]
        for t in x["wrt"]:
            t.requires_grad_()
    return x


def run(s):
    case = s["case"]
    kind, hq, hv = case["kind"], case["hq"], case["hv"]
    if kind == "update":
        return _conv.qkv_conv1d_update(s["x"], s["conv_state"], s["weight"], s["bias"], num_q_heads=hq,
                                       num_v_heads=hv, slot_ids=s["slots"]) + (s["conv_state"],)
    if kind == "conv":
        return _conv.qkv_conv1d(s["x"], s["weight"], s["bias"], s["cu"], s["conv_state"], num_q_heads=hq,
                                num_v_heads=hv)
    gates = (s["A_log"], s["a"], s["dt_bias"], s["b"])
    if kind == "train":
        out, final = _backward.chunk_gated_delta_rule(s["q"], s["k"], s["v"], *gates, s["cu"], s["state"], SCALE)
        return (out.detach(), final.detach()) + torch.autograd.grad(out, s["wrt"], s["d_out"])
    if kind == "pool":
        return _decode.decode_pool_(s["q"], s["k"], s["v"], s["state"], s["slots"], *gates, SCALE), s["state"]
    if kind == "multi":
        return _decode.gdn_decode_multi(s["q"], s["k"], s["v"], s["state"], *gates, SCALE, qk_l2norm=case["l2norm"])
    own = (hq, hv) == (4, 8) and not case["l2norm"]      # the layout of the plain entry points
    if kind == "decode":
        if own:
            return _decode.run(s["q"], s["k"], s["v"], s["state"], *gates, SCALE)
        return _decode.gdn_decode(s["q"], s["k"], s["v"], s["state"], *gates, SCALE, qk_l2norm=case["l2norm"])
    if own:
        return _prefill.run(s["q"], s["k"], s["v"], s["state"], *gates, s["cu"], SCALE)
    return _prefill.gdn_prefill(s["q"], s["k"], s["v"], s["state"], *gates, s["cu"], SCALE, qk_l2norm=case["l2norm"])


def work(case):
    """Inputs read once, outputs written once, and the recurrence's three products with the state per token and
    v-head (``S k``, the rank-1 update and ``S q``), which a chunked form adds to; the gradients take twice that."""
    kind, hq, hv = case["kind"], case["hq"], case["hv"]
    if kind in ("conv", "update"):
        channels = (2 * hq + hv) * D
        rows = case["tokens"] if kind == "conv" else case["batch"]
        states = case["n"] if kind == "conv" else case["batch"]
        size = rows * channels * 4 + states * channels * (WIDTH - 1) * 4 + channels * (WIDTH + 1) * 4
        return {"bytes": size, "flops": 2 * WIDTH * rows * channels}
    batch = case.get("batch")
    tokens = case["tokens"] if batch is None else batch * case.get("tokens", 1)
    rows = case["n"] if batch is None else batch
    activations = tokens * (2 * hq * D + hv * D + 2 * hv) * 2           # q, k, v, a, b
    out = tokens * hv * D * 2
    state = rows * hv * D * D * 4
    size = activations + out + state * (2 if case.get("state", True) else 1)
    flops = 6 * D * D * tokens * hv
    if kind == "train":                       # the backward: the inputs and the output's gradient again, gradients out
        return {"bytes": size + 2 * activations + out + (state if case["state"] else 0), "flops": 3 * flops}
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Four times the error against ``exact`` (bf16 outputs: half a unit in the last place is 1.6e-3 of a value in
    the mean; gradients also carry the bf16 operands of their products)."""
    if case["kind"] == "train":
        return {"rel": 2e-2}
    return {"rel": 1e-2 if case["kind"] == "prefill" else 7e-3}


# ---------------------------------------------------------------------------------------------------------------
# The results in 64 bits


def _silu(y):
    return y * torch.sigmoid(y)


def _normalised(x, l2norm):
    x = x.double()
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) if l2norm else x


def _gates64(A_log, a, dt_bias, b):
    """The log-decay and beta."""
    return -A_log.double().exp() * torch.nn.functional.softplus(a.double() + dt_bias.double()), torch.sigmoid(b.double())


def _steps64(q, k, v, state, g, beta):
    """Token by token: q, k, v [B, T, HV, D], state [B, HV, D, D]."""
    outs = []
    for t in range(q.shape[1]):
        state = state * g[:, t].exp()[..., None, None]
        delta = beta[:, t, :, None] * (v[:, t] - (state * k[:, t, :, None, :]).sum(-1))
        state = state + delta[..., None] * k[:, t, :, None, :]
        outs.append(SCALE * (state * q[:, t, :, None, :]).sum(-1))
    return torch.stack(outs, 1), state


def _chunks64(q, k, v, state, g, beta, lengths):
    """The same recurrence chunk by chunk over packed sequences: q, k, v [T, HV, D], state [N, HV, D, D] or None."""
    n, hv, total = len(lengths), v.shape[1], sum(lengths)
    nc = -(-max(lengths) // CHUNK)
    at = torch.full((n, nc * CHUNK), total, dtype=torch.int64)            # row `total` is a row of zeros
    begin = 0
    for i, length in enumerate(lengths):
        at[i, :length] = torch.arange(begin, begin + length)
        begin += length
    at = at.to(q.device)

    def padded(x):                                                        # -> [nc, N * HV, CHUNK, ...]
        x = torch.cat([x, x.new_zeros(1, *x.shape[1:])])[at]
        x = x.reshape(n, nc, CHUNK, hv, -1).permute(1, 0, 3, 2, 4)
        return x.reshape(nc, n * hv, CHUNK, -1).contiguous()

    q, k, v, beta = padded(q), padded(k), padded(v), padded(beta)
    gam = padded(g).cumsum(2)
    s = v.new_zeros(n * hv, D, D) if state is None else state.reshape(n * hv, D, D)
    eye = torch.eye(CHUNK, dtype=v.dtype, device=v.device)
    lower = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=v.device).tril()
    outs = []
    for c in range(nc):
        kt = k[c].transpose(1, 2).contiguous()
        e, last = gam[c].exp(), gam[c][:, -1:]
        decay = (gam[c] - gam[c].transpose(1, 2)).masked_fill(~lower, -math.inf).exp()
        power = -(beta[c] * decay * (k[c] @ kt)).tril(-1)
        inverse = eye + power                                             # (I - power)^-1, power^64 = 0
        for _ in range(5):
            power = power @ power
            inverse = inverse + inverse @ power
        st = s.transpose(1, 2).contiguous()
        vn = inverse @ (beta[c] * (v[c] - e * (k[c] @ st)))
        outs.append(SCALE * (e * (q[c] @ st) + (decay * (q[c] @ kt)) @ vn))
        s = last.exp() * s + ((last - gam[c]).exp() * vn).transpose(1, 2).contiguous() @ k[c]
    out = torch.stack(outs).reshape(nc, n, hv, CHUNK, D).permute(1, 0, 3, 2, 4).reshape(n * nc * CHUNK, hv, D)
    return out[(at.reshape(-1) < total).nonzero().flatten()], s.reshape(n, hv, D, D)


def exact(case, seed):
    x = _inputs(case, seed)
    kind, hq, hv = case["kind"], case["hq"], case["hv"]
    if kind in ("conv", "update"):
        weight, bias = x["weight"].double(), x["bias"].double()
        if kind == "update":
            rows = x["slots"].long()
            window = torch.cat([x["conv_state"][rows].double(), x["x"].double()[..., None]], -1)
            y = _silu((window * weight).sum(-1) + bias)
            state = x["conv_state"].double()
            state[rows] = window[..., 1:]
            parts = [p.reshape(p.shape[0], 1, -1, D) for p in y.split([hq * D, hq * D, hv * D], -1)]
            return tuple(parts) + (state,)
        ys, states, begin = [], [], 0
        for i, length in enumerate(_lengths(case)):
            u = torch.cat([x["conv_state"][i].double().t(), x["x"][begin:begin + length].double()])
            ys.append(_silu(sum(u[j:j + length] * weight[:, j] for j in range(WIDTH)) + bias))
            states.append(u[length:].t().contiguous())
            begin += length
        parts = [p.reshape(p.shape[0], -1, D) for p in torch.cat(ys).split([hq * D, hq * D, hv * D], -1)]
        return tuple(parts) + (torch.stack(states),)
    if kind == "train":
        names = [n for n in ("q", "k", "v", "A_log", "a", "dt_bias", "b", "state") if x[n] is not None]
        wide = {n: x[n].double().requires_grad_() for n in names}
    else:
        wide = x
    q, k = (_normalised(wide[n], case.get("l2norm")).repeat_interleave(hv // hq, -2) for n in ("q", "k"))
    v = wide["v"].double()
    g, beta = _gates64(wide["A_log"], wide["a"], wide["dt_bias"], wide["b"])
    if kind == "pool":
        rows = x["slots"].long()
        out, new = _steps64(q, k, v, x["state"][rows].double(), g, beta)
        state = x["state"].double()
        state[rows] = new
        return out, state
    if kind in ("decode", "multi"):
        return _steps64(q, k, v, x["state"].double(), g, beta)
    state = wide.get("state")
    out, final = _chunks64(q, k, v, None if state is None else state.double(), g, beta, _lengths(case))
    if kind != "train":
        return out, final
    grads = torch.autograd.grad(out, [wide[n] for n in names], x["d_out"].double())
    return (out.detach(), final.detach()) + grads
