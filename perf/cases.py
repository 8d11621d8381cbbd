"""Performance cases of the gated delta-rule library.

Each case is one call (or one short chain of calls) that a program using
rhizome_amd makes: prompts of one user and of many, one decode position,
speculative windows, and the Local block's mixer around the op.  Head sizes
are those of the model configurations (head_dim 32, 64 and 128), with 16
heads as in the benchmark, 32 heads in its long context.

A case is a dict of plain values:
  op       prefill | decode | multistep | block_prefill | block_decode
  dtype    dtype of q, k, v and o ("bf16" or "f32"); gates and states are fp32
  batch, seq_len      dense batch (seq_len: positions of a multistep window)
  lengths             packed batch instead: comma-separated sequence lengths
  heads, d_k, d_v
  gate     what the caller holds: "log" (g = ln alpha) or "alpha"
  g_mean   mean of the decay logits: g = -softplus(N(g_mean, 1))
  init     whether the sequences continue from a state
"""
import math

import torch
import torch.nn.functional as F

import rhizome_amd

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _case(op, dtype, batch, seq_len, heads, d_k, d_v, *, lengths="", gate="log", g_mean=0.0, init=False):
    return dict(op=op, dtype=dtype, batch=batch, seq_len=seq_len, lengths=lengths, heads=heads, d_k=d_k, d_v=d_v,
                gate=gate, g_mean=g_mean, init=init)


def listed():
    named = {
        # one user's next token in one layer: the smallest call, all latency
        "decode_one": _case("decode", "bf16", 1, 1, 16, 128, 128),
        # a serving batch's next token
        "decode_batch": _case("decode", "bf16", 48, 1, 16, 128, 128),
        # the benchmark's decode step, fp32 throughout
        "decode_large": _case("decode", "f32", 256, 1, 16, 128, 128),
        # speculative decoding: a window of 8 positions with a snapshot after each
        "speculate": _case("multistep", "bf16", 32, 8, 16, 128, 128),
        # one user's prompt, a length that fills no last chunk
        "prompt_one": _case("prefill", "bf16", 1, 2043, 16, 128, 128),
        # the benchmark's headline: a training or prompt batch that fills the chip
        "prefill_batch": _case("prefill", "bf16", 4, 4096, 16, 128, 128),
        # prompts of several users packed without padding, each continuing from its state
        "prefill_packed": _case("prefill", "bf16", 9, 0, 16, 128, 128, init=True,
                                lengths="1187,129,64,733,2048,351,1,918,1502"),
        # long context with slow decay and wide values
        "prefill_long": _case("prefill", "bf16", 1, 32768, 32, 128, 256, g_mean=-2.0),
        # the fp32 path (checks of a model, and its training at full precision)
        "prefill_fp32": _case("prefill", "f32", 4, 4096, 16, 128, 128),
        # a small model (head_dim 64) at full precision, packed, alpha as the caller holds it
        "small_fp32": _case("prefill", "f32", 5, 0, 8, 64, 64, gate="alpha", lengths="300,77,512,1,190"),
        # the Local block's mixer on a prompt: conv1d and the op's inputs, the op, the per-head norm
        "block_prefill": _case("block_prefill", "bf16", 2, 3001, 16, 128, 128),
        # the same mixer on one position of a serving batch, conv and op states carried
        "block_decode": _case("block_decode", "bf16", 64, 1, 16, 128, 128),
    }
    return [dict(name=n, **c) for n, c in named.items()]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """One more case of the listed ones' ranges; its cost stays below theirs
    by a bound on tokens x heads (prefill), on the sequential length of a
    call, and on the state's bytes (decode, multistep)."""
    op = rng.choice(["decode", "decode", "multistep", "prefill", "prefill", "prefill", "prefill", "block_prefill",
                     "block_decode"])
    d_k = rng.choice([32, 64, 128, 128, 128])
    d_v = rng.choice([d_k, d_k, d_k, 2 * d_k])
    heads = rng.choice([2, 4, 8, 16, 16, 16, 32])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    gate = rng.choice(["log", "log", "alpha"])
    g_mean = rng.choice([0.0, 0.0, -2.0])
    init = rng.random() < 0.5
    state = heads * d_k * d_v * 4
    if op in ("decode", "block_decode"):
        batch = _log_int(rng, 1, max(1, min(256, (256 << 20) // state)))
        return _case(op, dtype, batch, 1, heads, d_k, d_v, gate="log" if op == "block_decode" else gate, g_mean=g_mean)
    if op == "multistep":
        n = rng.randint(2, 8)
        batch = _log_int(rng, 1, max(1, min(64, (320 << 20) // (n * state))))
        return _case(op, dtype, batch, n, heads, d_k, d_v, gate=gate, g_mean=g_mean)
    tokens = _log_int(rng, 64, 2600 if dtype == "f32" else 16384)
    tokens = min(tokens, (96000 if dtype == "f32" else 400000) // heads)
    if op == "block_prefill":
        batch = rng.randint(1, 3)
        return _case(op, dtype, batch, max(1, tokens // batch), heads, d_k, d_v, g_mean=g_mean)
    if rng.random() < 0.5:
        batch = _log_int(rng, 1, 8)
        return _case(op, dtype, batch, max(1, tokens // batch), heads, d_k, d_v, gate=gate, g_mean=g_mean, init=init)
    n = rng.randint(2, 16)
    cuts = sorted(rng.randint(0, tokens) for _ in range(n - 1))
    lens = [b - a for a, b in zip([0] + cuts, cuts + [tokens])]
    return _case(op, dtype, n, 0, heads, d_k, d_v, gate=gate, g_mean=g_mean, init=init,
                 lengths=",".join(str(x) for x in lens))


def _lengths(case):
    if case["lengths"]:
        return [int(x) for x in case["lengths"].split(",")]
    return [case["seq_len"]] * case["batch"]


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _inputs(case, seed):
    """The tensors of the call, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, T, H, dk, dv = case["batch"], case["seq_len"], case["heads"], case["d_k"], case["d_v"]
    packed = bool(case["lengths"])
    lead = (sum(_lengths(case)),) if packed else ((B,) if case["op"] == "decode" else (B, T))

    def normal(*shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=gen, device="cuda") * std + mean

    s = {}
    if packed:
        cu = [0]
        for n in _lengths(case):
            cu.append(cu[-1] + n)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
    if case["op"].startswith("block"):
        C = H * (2 * dk + dv)
        s["x"] = normal(*lead, C).to(dt)
        s["w"] = normal(C, 4, std=0.5)
        s["bias"] = normal(C, std=0.1)
        s["beta_logit"], s["alpha_logit"] = normal(*lead, H), normal(*lead, H, mean=case["g_mean"])
        s["a_log"] = normal(H, std=0.3)
        s["scale"] = normal(dv, mean=1.0, std=0.1)
        if case["op"] == "block_decode":
            s["conv_state"] = normal(B, C, 3)
            s["state"] = normal(B, H, dv, dk, std=0.05)
        return s
    s["q"] = (_unit(normal(*lead, H, dk)) * math.sqrt(dk)).to(dt)
    s["k"] = _unit(normal(*lead, H, dk)).to(dt)
    s["v"] = normal(*lead, H, dv).to(dt)
    g = -F.softplus(normal(*lead, H, mean=case["g_mean"]))
    s["gate"] = g if case["gate"] == "log" else torch.exp(g)
    s["beta"] = torch.sigmoid(normal(*lead, H))
    if case["init"] or case["op"] in ("decode", "multistep"):
        s["state"] = normal(B, H, dv, dk, std=0.05)
    return s


def prepare(case, seed):
    return {"case": dict(case), **_inputs(case, seed)}


def run(state):
    s, case = state, state["case"]
    op, H, dk, dv = case["op"], case["heads"], case["d_k"], case["d_v"]
    if op.startswith("block"):
        q, k, v, beta, g, conv = rhizome_amd.conv_prepare(
            s["x"], s["w"], s["bias"], s["beta_logit"], s["alpha_logit"], s["a_log"], heads=H, d_k=dk, d_v=dv,
            initial_state=s.get("conv_state"), output_final_state=True)
        if op == "block_decode":
            o = rhizome_amd.decode_step(q[:, 0], k[:, 0], v[:, 0], g[:, 0], beta[:, 0], state=s["state"])
            fin = s["state"]
        else:
            o, fin = rhizome_amd.prefill(q, k, v, g, beta)
        return rhizome_amd.rmsnorm_heads(o, s["scale"]), fin, conv
    gate = {"g" if case["gate"] == "log" else "alpha": s["gate"]}
    if op == "decode":  # the state is updated in place, as a serving loop keeps it
        return rhizome_amd.decode_step(s["q"], s["k"], s["v"], beta=s["beta"], state=s["state"], **gate), s["state"]
    if op == "multistep":
        return rhizome_amd.multistep(s["q"], s["k"], s["v"], beta=s["beta"], state=s["state"], **gate)
    return rhizome_amd.prefill(s["q"], s["k"], s["v"], beta=s["beta"], cu_seqlens=s.get("cu"),
                               initial_state=s.get("state"), **gate)


def work(case):
    """Bytes: every input and output once.  Flops of a prefill: the chunked
    form's, per (chunk of c tokens, head) 6 c^2 d_k + 4 c^2 d_v + 6 c d_k d_v
    with c = 64, or the recurrence's 8 d_k d_v per token-head for fp32,
    decode and multistep."""
    H, dk, dv, n_seq = case["heads"], case["d_k"], case["d_v"], len(_lengths(case))
    tokens = sum(_lengths(case))
    e = 2 if case["dtype"] == "bf16" else 4
    unit = tokens * H
    state = n_seq * H * dk * dv * 4
    flops = 8.0 * unit * dk * dv
    if case["op"] in ("prefill", "block_prefill") and case["dtype"] == "bf16":
        flops = 0.0
        for n in _lengths(case):
            for c, times in ((64, n // 64), (n % 64, 1)):
                flops += H * times * (6.0 * c * c * dk + 4.0 * c * c * dv + 6.0 * c * dk * dv)
    io = unit * ((2 * dk + 2 * dv) * e + 8)
    if case["op"] == "multistep":
        return {"bytes": io + state + state * case["seq_len"], "flops": flops}
    if case["op"] == "decode":
        return {"bytes": io + 2 * state, "flops": flops}
    if case["op"] == "prefill":
        return {"bytes": io + state * (2 if case["init"] else 1), "flops": flops}
    # the mixer: x, the logits and the parameters in, the normed output and
    # the states out
    C = H * (2 * dk + dv)
    conv_state = n_seq * C * 3 * 4
    both = 2 if case["op"] == "block_decode" else 1
    return {"bytes": unit * ((2 * dk + 2 * dv) * e + 8) + C * 20 + both * (state + conv_state),
            "flops": flops + unit * (8.0 * (2 * dk + dv) + 4.0 * dv)}


def tolerance(case):
    """Of the 2-norm: fp32 sums of a few hundred terms carried along a
    sequence differ by about 1e-7 from 64 bits (measured); a bf16 output by
    1.8e-3, nearly all from its own rounding, a mixer's by up to 4.5e-3 (q, k,
    v and o are rounded on the way).  Each bound is about four times that."""
    if case["dtype"] == "f32":
        return {"rel": 5e-7}
    if case["op"].startswith("block"):
        return {"rel": 2e-2}
    return {"rel": 8e-3}


def _recurrence(q, k, v, alpha, beta, S, states=None):
    """S_t = alpha_t S (I - beta_t k k^T) + beta_t v k^T, o_t = S_t q_t over
    dim 1 of [N, T, H, ...], f64."""
    o = torch.empty(v.shape, dtype=torch.float64, device=v.device)
    for t in range(q.shape[1]):
        kt, a, b = k[:, t], alpha[:, t, :, None], beta[:, t, :, None]
        u = b * (v[:, t] - a * torch.matmul(S, kt[..., None])[..., 0])
        S = a[..., None] * S + u[..., None] * kt[..., None, :]
        o[:, t] = torch.matmul(S, q[:, t, ..., None])[..., 0]
        if states is not None:
            states[:, t] = S
    return o, S


def exact(case, seed):
    s = _inputs(case, seed)
    op, H, dk, dv = case["op"], case["heads"], case["d_k"], case["d_v"]
    d = {n: t.double() for n, t in s.items() if n != "cu"}
    N = len(_lengths(case))
    S = d["state"] if "state" in d else torch.zeros(N, H, dv, dk, dtype=torch.float64, device="cuda")
    if op.startswith("block"):
        x, conv = d["x"], d.get("conv_state")
        B, T, C = x.shape
        if conv is None:
            conv = torch.zeros(B, C, 3, dtype=torch.float64, device="cuda")
        xx = torch.cat([conv.transpose(1, 2), x], dim=1)
        y = d["bias"] + sum(d["w"][:, j] * xx[:, j:j + T] for j in range(4))
        q = _unit(y[..., :H * dk].reshape(B, T, H, dk)) * math.sqrt(dk)
        k = _unit(y[..., H * dk:2 * H * dk].reshape(B, T, H, dk))
        v = y[..., 2 * H * dk:].reshape(B, T, H, dv)
        alpha = torch.exp(-F.softplus(d["a_log"]) * F.softplus(d["alpha_logit"]))
        o, S = _recurrence(q, k, v, alpha, torch.sigmoid(d["beta_logit"]), S)
        o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6) * d["scale"]
        return (o[:, 0] if op == "block_decode" else o), S, xx[:, T:].transpose(1, 2).contiguous()
    alpha = torch.exp(d["gate"]) if case["gate"] == "log" else d["gate"]
    q, k, v, beta = d["q"], d["k"], d["v"], d["beta"]
    if op == "decode":
        o, S = _recurrence(q[:, None], k[:, None], v[:, None], alpha[:, None], beta[:, None], S)
        return o[:, 0], S
    if op == "multistep":
        states = torch.empty(*q.shape[:3], dv, dk, dtype=torch.float64, device="cuda")
        o, _ = _recurrence(q, k, v, alpha, beta, S, states)
        return o, states
    if not case["lengths"]:
        return _recurrence(q, k, v, alpha, beta, S)
    # packed: the sequences side by side, padded by positions that leave the
    # state alone (alpha 1, beta 0)
    lens = _lengths(case)
    T = max(lens)

    def pad(x, fill):
        out = torch.full((N, T) + tuple(x.shape[1:]), fill, dtype=torch.float64, device="cuda")
        at = 0
        for i, n in enumerate(lens):
            out[i, :n] = x[at:at + n]
            at += n
        return out

    o, S = _recurrence(pad(q, 0.0), pad(k, 0.0), pad(v, 0.0), pad(alpha, 1.0), pad(beta, 0.0), S)
    return torch.cat([o[i, :n] for i, n in enumerate(lens)]), S
