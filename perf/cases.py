"""Measured workloads of the BASED kernels, through the functions that a program calls.

Every case is one call of the ``kernels`` package (or one forward of its attention module) on
tensors that are resident on the GPU: ``prepare`` makes them from a seed, ``run`` is the call,
``exact`` the same function in plain torch in 64 bits, ``work`` the bytes and operations the call
cannot do without.  The inputs are N(0, 1), with q and k divided by sqrt(d) for the BASED kernels
(the benchmark's inputs); the softmax branch takes them undivided.

The kinds:

* ``parallel`` -- ``solution_nki``, the fused causal kernel (a training-length forward).
* ``chunked``  -- ``chunked_nki_numerator`` / ``chunked_based_attn``, the linear-time kernel.
* ``prefill``  -- ``based_chunked(return_state=True)``: a prompt, and the state decoding starts from.
* ``continue`` -- ``based_chunked(state_in=..., return_state=True)``: the next piece of a long prompt.
* ``decode``   -- ``based_decode_step``: one token for every sequence of a batch.
* ``sliding``  -- ``nki_sliding_window_attn``, the softmax companion.
* ``layer``    -- ``based_layer_attn``: both branches summed.
* ``module``   -- ``TrainiumBasedLinearAttention{,NKI}``: projections around the kernels.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "trainium-linear-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import kernels as K  # noqa: E402

EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one decoding step of a small batch: latency, launches and host work
        dict(name="decode_b2h16", kind="decode", b=2, h=16, n=1, d=16, dv=64, dtype="bf16", past=300),
        # one decoding step of a serving batch: the states' bytes
        dict(name="decode_b64h16", kind="decode", b=64, h=16, n=1, d=16, dv=64, dtype="bf16", past=300),
        # the smallest benchmark forward, 32-bit
        dict(name="parallel_f32_b1h4n1024", kind="parallel", b=1, h=4, n=1024, d=16, dv=64, dtype="f32"),
        # an ordinary training-length forward
        dict(name="parallel_b2h16n2048", kind="parallel", b=2, h=16, n=2048, d=16, dv=64, dtype="bf16"),
        # the headline benchmark
        dict(name="parallel_b2h16n8192", kind="parallel", b=2, h=16, n=8192, d=16, dv=64, dtype="bf16"),
        # the same length on the linear-time kernel, as the reference calls it (numerator)
        dict(name="chunked_b2h16n8192", kind="chunked", b=2, h=16, n=8192, d=16, dv=64, dtype="bf16",
             normalize=False, chunk=64),
        # a long prompt, with the state that decoding goes on from
        dict(name="prefill_b1h16n65536", kind="prefill", b=1, h=16, n=65536, d=16, dv=64, dtype="bf16",
             normalize=True, chunk=128),
        # the reference's default head dim for the chunked kernel, d = 64 (2145 features)
        dict(name="chunked_d64_b2h16n8192", kind="chunked", b=2, h=16, n=8192, d=64, dv=64, dtype="bf16",
             normalize=True, chunk=64),
        # the next piece of a prompt that is taken in pieces, d = 64, a length that no tile divides
        dict(name="continue_d64_b1h16n3001", kind="continue", b=1, h=16, n=3001, d=64, dv=64, dtype="bf16",
             normalize=True, chunk=64, past=500),
        # the softmax companion at its benchmark shape
        dict(name="sliding_b2h16n4096", kind="sliding", b=2, h=16, n=4096, d=64, dv=64, dtype="bf16", window=64),
        # the whole BASED layer, a ragged length
        dict(name="layer_b2h16n3001", kind="layer", b=2, h=16, n=3001, d=16, dv=64, d_sw=64, dtype="bf16", window=64),
        # an attention module as a model holds it: 16 heads of 64
        dict(name="module_dim1024h16n2048", kind="module", b=2, h=16, n=2048, d=64, dv=64, dtype="bf16",
             dispatch="fused"),
    ]


def _features(d):
    return 1 + d + d * (d + 1) // 2


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cost(c):
    w = work(c)
    return max(w["bytes"], w["flops"] * (8 if c["dtype"] == "f32" else 1) / 50)


def draw(rng):
    """One more case: any kind, head counts, lengths and dims over the ranges above."""
    kind = rng.choice(["decode", "parallel", "parallel", "chunked", "chunked", "prefill", "continue", "sliding",
                       "layer", "module"])
    c = dict(kind=kind, b=_log_int(rng, 1, 8), h=rng.choice([2, 4, 8, 12, 16, 16, 24, 32]),
             n=_log_int(rng, 200, 16384), d=rng.choice([16, 16, 16, 32, 64]), dv=rng.choice([32, 64, 64, 64, 128]),
             dtype=rng.choice(["bf16", "bf16", "bf16", "bf16", "f32"]))
    if kind == "decode":
        c.update(n=1, b=_log_int(rng, 1, 64), past=rng.randint(100, 400))
    if kind in ("chunked", "prefill", "continue"):
        c.update(n=_log_int(rng, 256, 65536), normalize=rng.random() < 0.7, chunk=rng.choice([64, 128]))
    if kind == "continue":
        c.update(past=rng.randint(100, 600))
    if kind == "sliding":
        c.update(d=rng.choice([32, 64, 64, 128]), window=_log_int(rng, 16, 256))
    if kind == "layer":
        c.update(d=16, dv=rng.choice([32, 64, 64]), d_sw=rng.choice([16, 32, 64, 64]), window=rng.randint(16, 64))
    if kind == "module":
        c.update(h=rng.choice([8, 16]), n=_log_int(rng, 200, 4096), dispatch=rng.choice(["fused", "auto"]))
        c["dv"] = c["d"]
    if rng.random() < 0.4 and c["n"] > 256:
        c["n"] -= c["n"] % 64      # lengths in practice are often whole tiles, and often not
    most = max(_cost(x) for x in listed() if x["dtype"] == "bf16")
    while _cost(c) > most:
        if c["b"] > 1:
            c["b"] = (c["b"] + 1) // 2
        elif c["n"] > 1:
            c["n"] = c["n"] * 2 // 3 + 1
        else:
            c["h"] = max(1, c["h"] // 2)
    return c


# ---- inputs

def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _phi(x):
    """[1, x / d^(1/4), x_i^2 / sqrt(2 d), x_i x_j / sqrt(d) (i < j)] in x's own type."""
    d = x.shape[-1]
    i, j = torch.triu_indices(d, d, 1, device=x.device)
    return torch.cat([torch.ones_like(x[..., :1]), x / d ** 0.25, x * x / math.sqrt(2 * d),
                      x[..., i] * x[..., j] / math.sqrt(d)], -1)


def _state(g, c):
    """The (b, h, F, dv + 1) fp32 state of ``past`` earlier tokens."""
    b, h, d, dv, past = (c[x] for x in ("b", "h", "d", "dv", "past"))
    k = (_randn(g, b * h, past, d) / math.sqrt(d)).to(DTYPES[c["dtype"]]).float()
    v = _randn(g, b * h, past, dv).to(DTYPES[c["dtype"]]).float()
    out = torch.empty(b * h, _features(d), dv + 1, device="cuda")
    for r in range(0, b * h, 64):
        ph = _phi(k[r:r + 64]).transpose(1, 2).contiguous()
        out[r:r + 64, :, :dv] = torch.bmm(ph, v[r:r + 64])
        out[r:r + 64, :, dv] = ph.sum(-1)
    out[:, 0, dv] = past
    return out.view(b, h, _features(d), dv + 1)


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = DTYPES[c["dtype"]]
    b, h, n, d, dv = (c[x] for x in ("b", "h", "n", "d", "dv"))
    if c["kind"] == "module":
        dim = h * d
        cls = K.TrainiumBasedLinearAttention if c["dispatch"] == "auto" else K.TrainiumBasedLinearAttentionNKI
        m = cls(dim, heads=h).to(device="cuda", dtype=dt)
        with torch.no_grad():
            for p in (m.q_proj, m.k_proj, m.v_proj, m.o_proj):
                p.weight.copy_(_randn(g, dim, dim) / math.sqrt(dim))
        return {"case": c, "module": m, "x": _randn(g, b, n, dim).to(dt)}
    scale = 1.0 if c["kind"] == "sliding" else 1.0 / math.sqrt(d)
    s = {"case": c, "q": (_randn(g, b, h, n, d) * scale).to(dt), "k": (_randn(g, b, h, n, d) * scale).to(dt),
         "v": _randn(g, b, h, n, dv).to(dt)}
    if c["kind"] == "layer":
        s.update(q_sw=_randn(g, b, h, n, c["d_sw"]).to(dt), k_sw=_randn(g, b, h, n, c["d_sw"]).to(dt))
    if c["kind"] in ("decode", "continue"):
        s["state"] = _state(g, c)
    return s


# ---- the calls

def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "module":
        with torch.no_grad():
            return s["module"](s["x"])
    q, k, v = s["q"], s["k"], s["v"]
    if kind == "parallel":
        return K.solution_nki(q, k, v)
    if kind == "chunked":
        if c["normalize"]:
            return K.chunked_based_attn(q, k, v, chunk_size=c["chunk"])
        return K.chunked_nki_numerator(q, k, v, chunk_size=c["chunk"])
    if kind == "prefill":
        return K.based_chunked(q, k, v, chunk_size=c["chunk"], normalize=c["normalize"], return_state=True)
    if kind == "continue":
        return K.based_chunked(q, k, v, chunk_size=c["chunk"], normalize=c["normalize"], return_state=True,
                               state_in=s["state"], prev_tokens=c["past"])
    if kind == "decode":
        return K.based_decode_step(q, k, v, s["state"]), s["state"]
    if kind == "sliding":
        return K.nki_sliding_window_attn(q, k, v, window_size=c["window"])
    return K.based_layer_attn(q, k, v, window_size=c["window"], q_sw=s["q_sw"], k_sw=s["k_sw"])


# ---- the same in 64 bits

def _based64(q, k, v, normalize, num0=None, den0=None):
    """sum_{u <= t} (1 + s + s^2 / 2) v_u, and its division by the sum of weights; (bh, n, .) in fp64."""
    bh, n, d = q.shape
    out = torch.empty(bh, n, v.shape[-1], dtype=torch.float64, device=q.device)
    rows = 512
    for t0 in range(0, n, rows):
        t1 = min(n, t0 + rows)
        p = torch.bmm(q[:, t0:t1], k[:, :t1].transpose(1, 2).contiguous()).mul_(1.0 / math.sqrt(d))
        p.addcmul_(p, p, value=0.5).add_(1.0)
        p[:, :, t0:].tril_()
        num = torch.bmm(p, v[:, :t1])
        den = p.sum(-1, keepdim=True)
        if num0 is not None:
            num += num0[:, t0:t1]
            den += den0[:, t0:t1]
        out[:, t0:t1] = num / (den + EPS) if normalize else num
    return out


def _softmax64(q, k, v, window):
    bh, n, d = q.shape
    out = torch.empty(bh, n, v.shape[-1], dtype=torch.float64, device=q.device)
    rows = 512
    for t0 in range(0, n, rows):
        t1, u0 = min(n, t0 + rows), max(0, t0 - window + 1)
        s = torch.bmm(q[:, t0:t1], k[:, u0:t1].transpose(1, 2).contiguous()) / math.sqrt(d)
        gap = torch.arange(t0, t1, device=q.device)[:, None] - torch.arange(u0, t1, device=q.device)[None, :]
        s.masked_fill_((gap < 0) | (gap >= window), float("-inf"))
        out[:, t0:t1] = torch.bmm(torch.softmax(s, -1), v[:, u0:t1])
    return out


def _phi_sum64(k, v):
    """[sum phi(k) v^T | sum phi(k)] in fp64, one block of tokens at a time."""
    bh, n, d = k.shape
    s = torch.zeros(bh, _features(d), v.shape[-1] + 1, dtype=torch.float64, device=k.device)
    one = torch.ones(bh, n, 1, dtype=torch.float64, device=k.device)
    vx = torch.cat([v, one], -1)
    for t0 in range(0, n, 1024):
        s += torch.bmm(_phi(k[:, t0:t0 + 1024]).transpose(1, 2).contiguous(), vx[:, t0:t0 + 1024])
    return s


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    b, h, n, d, dv = (c[x] for x in ("b", "h", "n", "d", "dv"))
    if c["kind"] == "module":
        m, x = s["module"], s["x"].double()
        with torch.no_grad():
            q, k, v = ((x @ p.weight.double().T).view(b, n, h, d).transpose(1, 2).reshape(b * h, n, d)
                       for p in (m.q_proj, m.k_proj, m.v_proj))
            y = _based64(q, k, v, True).view(b, h, n, d).transpose(1, 2).reshape(b, n, h * d)
            return y @ m.o_proj.weight.double().T
    q, k, v = (s[x].double().reshape(b * h, n, -1) for x in ("q", "k", "v"))
    if c["kind"] == "sliding":
        return _softmax64(q, k, v, c["window"]).view(b, h, n, dv)
    if c["kind"] == "layer":
        qs, ks = (s[x].double().reshape(b * h, n, -1) for x in ("q_sw", "k_sw"))
        return (_based64(q, k, v, True) + _softmax64(qs, ks, v, c["window"])).view(b, h, n, dv)
    normalize = c.get("normalize", True)
    if c["kind"] in ("parallel", "chunked"):
        return _based64(q, k, v, normalize).view(b, h, n, dv)
    F = _features(d)
    if c["kind"] == "prefill":
        return _based64(q, k, v, normalize).view(b, h, n, dv), _phi_sum64(k, v).view(b, h, F, dv + 1)
    st = s["state"].double().view(b * h, F, dv + 1)
    ext = torch.cat([torch.bmm(_phi(q[:, t:t + 1024]), st) for t in range(0, n, 1024)], 1)
    y = _based64(q, k, v, normalize, ext[..., :dv], ext[..., dv:])
    return y.view(b, h, n, dv), (st + _phi_sum64(k, v)).view(b, h, F, dv + 1)


# ---- what a call cannot do without

def work(case):
    c = case
    b, h, n, d, dv = (c[x] for x in ("b", "h", "n", "d", "dv"))
    e, bh, F = (2 if c["dtype"] == "bf16" else 4), b * h, _features(d)
    pairs = n * (n + 1) / 2
    qkvo = e * bh * n * (2 * d + 2 * dv)
    state = 4 * bh * F * (dv + 1)
    # per token: the cheaper of all causal pairs and of the recurrence (state in and out, and the
    # pairs of a 64-token chunk); two operations for each multiply and add
    quadratic = 2 * (d + dv) * pairs
    linear = n * (4 * F * dv + 65 * (d + dv))
    if c["kind"] == "decode":
        return {"bytes": 2 * state + qkvo, "flops": bh * 4 * F * (dv + 1)}
    if c["kind"] == "parallel":
        return {"bytes": qkvo, "flops": bh * quadratic}
    if c["kind"] == "chunked":
        return {"bytes": qkvo, "flops": bh * min(quadratic, linear)}
    if c["kind"] == "prefill":
        return {"bytes": qkvo + state, "flops": bh * min(quadratic + n * 2 * F * dv, linear)}
    if c["kind"] == "continue":
        return {"bytes": qkvo + 2 * state, "flops": bh * min(quadratic + n * 4 * F * dv, linear)}
    w = c.get("window", 0)
    near = sum(min(t + 1, w) for t in range(min(n, w))) + max(0, n - w) * w
    if c["kind"] == "sliding":
        return {"bytes": qkvo, "flops": bh * 2 * (d + dv) * near}
    if c["kind"] == "layer":
        return {"bytes": qkvo + e * bh * n * 2 * c["d_sw"],
                "flops": bh * (min(quadratic, linear) + 2 * (c["d_sw"] + dv) * near)}
    dim = h * d
    return {"bytes": e * (2 * b * n * dim + 4 * dim * dim), "flops": 8 * b * n * dim * dim + bh * quadratic}


# Relative error (2-norm).  bf16 outputs are 1.5e-3 to 1.7e-3 off 64 bits, which is the rounding of the
# result (the chunked kernels' fp16 operands and state stay below it), so two kernels differ by up to
# 2.4e-3; the module, which rounds q, k, v and the attention's output between its products, is 3.2e-3
# off.  fp32 outputs are 1.3e-7 to 1.9e-7 off at these sizes; sums of up to 65536 terms in another
# order and products split in three reach 1e-6 and more.
def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 7e-3} if case["kind"] != "module" else {"rel": 1.3e-2}
