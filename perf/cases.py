"""The work that users of the GatedDeltaNet path have it do, as timed cases.

Serving: single-token decode (one sequence, a batch through several layers' caches, the
whole layer with its projections), a short prompt continued from a cache, ordinary and
packed prefills, a long document.  Training: forward and backward of the chunked rule, of
the layer between its projections, and of the whole layer.  Head layouts: 16 key heads and
32 or 64 value heads of dim 128, and smaller layouts of dim 64, in bf16, with fp32 inputs
for the chunked rule alone.  ``exact`` restates every case in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import omegalax_amd as om

CONV_K = 4
EPS = 1e-6
CHUNK = 64


def listed():
    return [
        # one user's next token: nothing but latency
        dict(name="decode_one", kind="decode", batch=1, layers=1, hk=16, hv=32, d=128),
        # a serving batch's next token through four layers' caches, whose state together is
        # larger than any cache of the chip, as in a model
        dict(name="decode_batch", kind="decode", batch=64, layers=4, hk=16, hv=32, d=128),
        # a small serving batch's next token through one whole layer, projections included
        dict(name="module_decode", kind="module_decode", batch=17, hidden=2048, hk=16, hv=32, d=128),
        # a short turn of a conversation, continued from its cache
        dict(name="prefill_turn", kind="prefill", batch=1, tokens=77, packed=0, carry=True,
             hk=16, hv=32, d=128),
        # one prompt of ordinary length into an empty cache
        dict(name="prefill_prompt", kind="prefill", batch=1, tokens=1900, packed=0, carry=False,
             hk=16, hv=32, d=128),
        # a batch of long prompts
        dict(name="prefill_batch", kind="prefill", batch=4, tokens=4096, packed=0, carry=False,
             hk=16, hv=32, d=128),
        # eight documents of uneven lengths, each continued from its own state
        dict(name="prefill_packed", kind="prefill", batch=1, tokens=32768, packed=8, carry=True,
             hk=16, hv=32, d=128),
        # the rule alone on fp32 inputs with small heads: parity runs and small models
        dict(name="core_fp32", kind="core", batch=2, tokens=512, hk=4, hv=4, d=64, dtype="fp32",
             long_memory=False),
        # a long document with slowly decaying memory and the wide head layout
        dict(name="core_long", kind="core", batch=1, tokens=65536, hk=16, hv=64, d=128,
             dtype="bf16", long_memory=True),
        # a training step of the rule at the benchmark's batch
        dict(name="core_train", kind="core_train", batch=4, tokens=4096, hk=16, hv=32, d=128,
             dtype="bf16", long_memory=False),
        # fine-tuning on one row of packed documents: few sequences, ragged lengths
        dict(name="layer_train", kind="layer_train", batch=1, tokens=3001, packed=5, hk=16,
             hv=32, d=128),
        # a training step of the whole layer of a small model, projections included
        dict(name="module_train", kind="module_train", batch=4, tokens=500, hidden=1024, hk=8,
             hv=16, d=64),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """A case of the listed kinds; tokens x value heads x dim and the length of one sequence
    (a serial chain of chunks) are bounded so that none is dearer than the largest listed."""
    kind = rng.choice(["decode", "module_decode", "prefill", "prefill", "core", "core_train",
                       "layer_train", "module_train"])
    d = rng.choice([128, 128, 64])
    hk = rng.choice([4, 8, 16])
    c = dict(kind=kind, hk=hk, hv=hk * rng.choice([1, 2, 2, 4]), d=d)
    if kind == "decode":
        c.update(batch=_log_int(rng, 1, 200), layers=rng.choice([1, 2, 4]))
        while c["batch"] * c["layers"] * c["hv"] > 64 * 4 * 32:
            c["batch"] = max(1, c["batch"] // 2)
        return c
    if kind == "module_decode":
        c.update(batch=_log_int(rng, 1, 64), hidden=rng.choice([1024, 2048]))
        return c
    most, longest = {"prefill": (32768 * 32 * 128, 16384), "core": (65536 * 64 * 128, 32768),
                     "core_train": (16384 * 32 * 128, 8192), "layer_train": (8192 * 32 * 128, 8192),
                     "module_train": (4096 * 32 * 128, 4096)}[kind]
    dtype = "bf16"
    if kind in ("core", "core_train"):
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        c.update(dtype=dtype, long_memory=rng.random() < 0.5)
        if dtype == "fp32":
            c["d"] = 64
            most, longest = most // 4, longest // 4
    total = _log_int(rng, 40, min(65536, most // (c["hv"] * c["d"])))
    c["batch"] = 1
    if kind in ("prefill", "layer_train") and rng.random() < 0.4 and total >= 64:
        c["packed"] = rng.randint(2, 9)
    else:
        if kind in ("prefill", "layer_train"):
            c["packed"] = 0
        if rng.random() < 0.5:
            c["batch"] = rng.randint(1, min(8, max(1, total // 16)))
    c["tokens"] = max(1, min(longest, total // c["batch"]))
    if kind == "prefill":
        c["carry"] = rng.random() < 0.5
    if kind == "module_train":
        c["hidden"] = rng.choice([1024, 2048])
    return c


# ---------------------------------------------------------------- inputs


class _Draws:
    """Seeded normal and uniform draws on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _dims(case):
    return dict(num_k_heads=case["hk"], head_k_dim=case["d"], num_v_heads=case["hv"],
                head_v_dim=case["d"])


def _conv_dim(case):
    return (2 * case["hk"] + case["hv"]) * case["d"]


def _layer_params(r, case):
    """Conv, gate and norm parameters: conv N(0, 0.1), A in [1, 16], dt_bias in [-2, 0]."""
    hv = case["hv"]
    return dict(conv_w=r.normal(_conv_dim(case), CONV_K, scale=0.1),
                A_log=r.uniform(0.0, math.log(16.0), hv), dt_bias=r.uniform(-2.0, 0.0, hv),
                norm_w=r.uniform(0.5, 1.5, case["d"]))


def _projected(r, case, *lead):
    """Projection outputs (mixed_qkv, z, a, b) in bf16."""
    bf = torch.bfloat16
    return dict(mixed_qkv=r.normal(*lead, _conv_dim(case), dtype=bf),
                z=r.normal(*lead, case["hv"], case["d"], dtype=bf),
                a=r.normal(*lead, case["hv"], dtype=bf), b=r.normal(*lead, case["hv"], dtype=bf))


def _lengths(case, seed):
    """`packed` lengths that sum to the tokens: a seeded uneven split, each at least one."""
    n, total = case["packed"], case["tokens"]
    gen = torch.Generator()
    gen.manual_seed(seed)
    w = -torch.log(torch.rand(n, generator=gen, dtype=torch.float64))
    least = max(1, total // (16 * n))
    lens = (w / w.sum() * (total - least * n)).floor().to(torch.int64) + least
    lens[0] += total - int(lens.sum())
    return lens.tolist()


def _offsets(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _module_weights(r, case):
    """Projection weights of one layer, N(0, 0.02) in bf16."""
    D, bf, value = case["hidden"], torch.bfloat16, case["hv"] * case["d"]
    w = lambda n, m: r.normal(n, m, scale=0.02, dtype=bf)
    return dict(in_proj_qkv=w(_conv_dim(case), D), in_proj_z=w(value, D),
                in_proj_b=w(case["hv"], D), in_proj_a=w(case["hv"], D), out_proj=w(D, value),
                **_layer_params(r, case))


def _config(case):
    return om.GDNConfig(hidden_size=case["hidden"], num_k_heads=case["hk"], head_k_dim=case["d"],
                        num_v_heads=case["hv"], head_v_dim=case["d"], conv_kernel=CONV_K,
                        rms_norm_eps=EPS)


def _leaves(ts):
    return {k: t.requires_grad_(True) for k, t in ts.items()}


def prepare(case, seed):
    r = _Draws(seed)
    kind, hv, d = case["kind"], case["hv"], case["d"]
    s = dict(kind=kind, kw=dict(_dims(case), eps=EPS))
    if kind == "decode":
        s["layers"] = []
        for _ in range(case["layers"]):
            B = case["batch"]
            s["layers"].append(dict(
                **_projected(r, case, B), **_layer_params(r, case),
                conv_state=r.normal(B, _conv_dim(case), CONV_K - 1, dtype=torch.bfloat16),
                state=r.normal(B, hv, d, d, scale=0.02)))
        return s
    if kind == "module_decode":
        B = case["batch"]
        s["params"] = om.GDNParams(**_module_weights(r, case))
        s["cfg"] = _config(case)
        s["hidden"] = r.normal(B, case["hidden"], dtype=torch.bfloat16)
        s["cache"] = om.make_gdn_cache(s["cfg"], 1, B)[0]
        s["cache"].conv_state.copy_(r.normal(B, _conv_dim(case), CONV_K - 1))
        s["cache"].recurrent_state.copy_(r.normal(B, hv, d, d, scale=0.02))
        return s
    B, T = case["batch"], case["tokens"]
    if kind in ("prefill", "layer_train"):
        s["x"] = dict(**_projected(r, case, B, T), **_layer_params(r, case))
        n = case["packed"] or B
        if case["packed"]:
            s["lens"] = _lengths(case, seed)
            s["kw"]["cu_seqlens"] = torch.tensor(_offsets(s["lens"]), dtype=torch.int32, device="cuda")
        if kind == "prefill":
            s["kw"]["output_final_state"] = True
            if case["carry"]:
                s["kw"]["initial_state"] = r.normal(n, hv, d, d, scale=0.02)
                s["kw"]["conv_state"] = r.normal(n, _conv_dim(case), CONV_K - 1, dtype=torch.bfloat16)
        else:
            s["x"] = _leaves(s["x"])
            s["d_out"] = r.normal(B, T, hv * d, dtype=torch.bfloat16)
        return s
    if kind in ("core", "core_train"):
        dt = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        hk = case["hk"]
        x = dict(q=r.normal(B, T, hk, d, dtype=dt), k=r.normal(B, T, hk, d, dtype=dt),
                 v=r.normal(B, T, hv, d, dtype=dt))
        if case["long_memory"]:
            x["g"] = torch.log(r.uniform(0.9, 0.9999, B, T, hv))
        else:
            A, dt_bias = torch.exp(r.uniform(0.0, math.log(16.0), hv)), r.uniform(-2.0, 0.0, hv)
            x["g"] = -A * F.softplus(r.normal(B, T, hv) + dt_bias)
        x["beta"] = torch.sigmoid(r.normal(B, T, hv))
        s["x"] = x
        if kind == "core_train":
            s["x"] = _leaves(x)
            s["d_out"] = r.normal(B, T, hv, d)
        return s
    assert kind == "module_train"
    w = _leaves(_module_weights(r, case))
    s["weights"], s["params"], s["cfg"] = w, om.GDNParams(**w), _config(case)
    s["hidden"] = r.normal(B, T, case["hidden"], dtype=torch.bfloat16).requires_grad_(True)
    s["d_out"] = r.normal(B, T, case["hidden"], dtype=torch.bfloat16)
    return s


# ---------------------------------------------------------------- one pass


_LAYER_ARGS = ("mixed_qkv", "z", "a", "b", "conv_w", "A_log", "dt_bias", "norm_w")
_CORE_ARGS = ("q", "k", "v", "g", "beta")


def run(s):
    kind = s["kind"]
    if kind == "decode":
        outs = []
        for l in s["layers"]:
            o = om.gdn_decode_step(*(l[n] for n in _LAYER_ARGS), l["conv_state"], l["state"], **s["kw"])
            outs += [o, l["conv_state"], l["state"]]
        return outs
    if kind == "module_decode":
        o = om.gated_deltanet_decode(s["params"], s["cfg"], s["hidden"], s["cache"])
        return [o, s["cache"].conv_state, s["cache"].recurrent_state]
    if kind == "prefill":
        return list(om.gdn_prefill(*(s["x"][n] for n in _LAYER_ARGS), **s["kw"]))
    if kind == "layer_train":
        x = [s["x"][n] for n in _LAYER_ARGS]
        o = om.gdn_prefill(*x, **s["kw"])
        return [o.detach(), *torch.autograd.grad(o, x, s["d_out"])]
    x = [s["x"][n] for n in _CORE_ARGS] if "x" in s else None
    if kind == "core":
        return list(om.chunk_gated_delta_rule(*x, output_final_state=True))
    if kind == "core_train":
        o = om.chunk_gated_delta_rule(*x)
        return [o.detach(), *torch.autograd.grad(o, x, s["d_out"])]
    o = om.gated_deltanet_forward(s["params"], s["cfg"], s["hidden"])
    return [o.detach(), *torch.autograd.grad(o, [s["hidden"], *s["weights"].values()], s["d_out"])]


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind, hk, hv, d = case["kind"], case["hk"], case["hv"], case["d"]
    cd, value = _conv_dim(case), case["hv"] * case["d"]
    params = (cd * CONV_K + 2 * hv + d) * 4
    state = hv * d * d * 4
    window = cd * (CONV_K - 1) * 2
    io = (cd + 2 * value + 2 * hv) * 2          # mixed_qkv, z, out, a, b of one token
    rule = hv * (2 * CHUNK * 5 * d + 6 * d * d)  # products of one token in chunks of 64
    if kind == "decode":
        n = case["batch"] * case["layers"]
        return dict(bytes=n * (2 * state + 2 * window + io) + case["layers"] * params,
                    flops=n * hv * 8 * d * d)
    proj = 0
    if "hidden" in case:
        proj = (cd + 2 * value + 2 * hv) * case["hidden"]  # weights of the five projections
    if kind == "module_decode":
        n = case["batch"]
        return dict(bytes=n * (2 * state + 2 * window + 4 * case["hidden"]) + params + 2 * proj,
                    flops=n * (hv * 8 * d * d + 2 * proj))
    n = case["batch"] * case["tokens"]
    if kind == "prefill":
        seqs = case["packed"] or case["batch"]
        states = seqs * (state + window) * (2 if case["carry"] else 1)
        return dict(bytes=n * io + states + params, flops=n * rule)
    if kind == "layer_train":
        # out written, d_out read; every input read and its gradient written
        return dict(bytes=n * (2 * (cd + value + 2 * hv) * 2 + 2 * value * 2) + 2 * params,
                    flops=3 * n * rule)
    if kind in ("core", "core_train"):
        size = 4 if case["dtype"] == "fp32" else 2
        inputs, out = ((2 * hk + hv) * d * size + 2 * hv * 4), value * 4
        if kind == "core":
            return dict(bytes=n * (inputs + out) + case["batch"] * state, flops=n * rule)
        return dict(bytes=n * 2 * (inputs + out), flops=3 * n * rule)
    return dict(bytes=n * 8 * case["hidden"] + 4 * proj + 2 * params,
                flops=3 * n * (rule + 2 * proj))


def tolerance(case):
    """About four times the error against ``exact`` at the listed and drawn sizes."""
    if case.get("dtype") == "fp32":  # sums in split bf16 products: 6e-6 to 9e-6
        return {"rel": 4e-5}
    if case["kind"] in ("core", "core_train"):  # bf16 inputs and operands: 1.7e-3 to 3.3e-3
        return {"rel": 1.2e-2}
    # bf16 at the conv, the gates, the norm and the output too: 4e-3 to 9e-3
    return {"rel": 2e-2}


# ---------------------------------------------------------------- the same in 64 bits


def _rule64(q, k, v, g, beta, S):
    """The gated delta rule in chunks on [B, T, H, *] float64 (q, k normalised, q scaled);
    returns (o, final state)."""
    B, T, H, A = q.shape
    J = -(-T // CHUNK)

    def chunks(x):
        x = F.pad(x.movedim(2, 1).flatten(3), (0, 0, 0, J * CHUNK - T)) if x.dim() == 4 else \
            F.pad(x.movedim(2, 1), (0, J * CHUNK - T))
        return x.reshape(B, H, J, CHUNK, *x.shape[3:]).contiguous()

    q, k, v, g, beta = (chunks(x) for x in (q, k, v, g, beta))
    G = g.cumsum(-1)
    low = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    decay = torch.exp((G[..., :, None] - G[..., None, :]).masked_fill(~low, float("-inf")))
    kt = k.transpose(-1, -2).contiguous()
    L = (k @ kt * decay * beta[..., None]).tril(-1)
    eye = torch.eye(CHUNK, dtype=q.dtype, device=q.device)
    X = torch.linalg.solve_triangular(L + eye, eye.expand_as(L), upper=False, unitriangular=True)
    U = X @ (v * beta[..., None])
    W = X @ (k * (beta * G.exp())[..., None])
    P = q @ kt * decay
    qe = q * G.exp()[..., None]
    ke = (k * torch.exp(G[..., -1:] - G)[..., None]).transpose(-1, -2).contiguous()
    last = G[..., -1].exp()[..., None, None]
    o = []
    for j in range(J):
        vn = U[:, :, j] - W[:, :, j] @ S
        o.append(qe[:, :, j] @ S + P[:, :, j] @ vn)
        S = last[:, :, j] * S + ke[:, :, j] @ vn
    o = torch.stack(o, 2).reshape(B, H, J * CHUNK, -1)[:, :, :T].movedim(1, 2)
    return o, S


def _unit(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + EPS)


def _core64(q, k, v, g, beta, S=None):
    H, d = v.shape[2], q.shape[3]
    rep = H // q.shape[2]
    q, k = (_unit(x).repeat_interleave(rep, dim=2) for x in (q, k))
    if S is None:
        S = torch.zeros(q.shape[0], H, d, v.shape[3], dtype=q.dtype, device=q.device)
    return _rule64(q * d ** -0.5, k, v, g, beta, S)


def _layer64(case, x, z, a, b, conv_w, A_log, dt_bias, norm_w, window=None, S=None):
    """Conv + SiLU, gates, the rule and the gated norm; (out, final state, conv window)."""
    B, T, C = x.shape
    hk, hv, d = case["hk"], case["hv"], case["d"]
    if window is None:
        window = torch.zeros(B, C, CONV_K - 1, dtype=x.dtype, device=x.device)
    xx = torch.cat([window.transpose(1, 2), x], 1)
    y = F.silu(sum(xx[:, i:i + T] * conv_w[:, i] for i in range(CONV_K)))
    q, k, v = y.split([hk * d, hk * d, hv * d], -1)
    g = -A_log.exp() * F.softplus(a + dt_bias)
    o, S = _core64(q.reshape(B, T, hk, d), k.reshape(B, T, hk, d), v.reshape(B, T, hv, d), g,
                   b.sigmoid(), S)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * norm_w
    o = o * F.silu(z.reshape(o.shape))
    return o.reshape(B, T, hv * d), S, xx[:, T:].transpose(1, 2)


def _sequences64(s, case, x):
    """_layer64 over the batch or over each packed sequence."""
    window, S = (t if t is None else t.double() for t in (s["kw"].get("conv_state"), s["kw"].get("initial_state")))
    if "lens" not in s:
        return _layer64(case, *x, window, S)
    cu, parts = _offsets(s["lens"]), []
    for i in range(len(s["lens"])):
        seq = [t[:, cu[i]:cu[i + 1]] for t in x[:4]] + x[4:]
        parts.append(_layer64(case, *seq, *(t if t is None else t[i:i + 1] for t in (window, S))))
    o, S, window = zip(*parts)
    return torch.cat(o, 1), torch.cat(S), torch.cat(window)


def _leaf64(t):
    return t.detach().double().requires_grad_(t.requires_grad)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode":
        outs = []
        for l in s["layers"]:
            x = [l[n].double() for n in _LAYER_ARGS]
            x = [t[:, None] for t in x[:4]] + x[4:]
            o, S, window = _layer64(case, *x, l["conv_state"].double(), l["state"].double())
            outs += [o[:, 0], window, S]
        return outs
    if kind == "module_decode":
        p, c = s["params"], s["cache"]
        h = s["hidden"].double()[:, None]
        x = [h @ getattr(p, n).double().t() for n in ("in_proj_qkv", "in_proj_z", "in_proj_a", "in_proj_b")]
        o, S, window = _layer64(case, *x, *(getattr(p, n).double() for n in _LAYER_ARGS[4:]),
                                c.conv_state.double(), c.recurrent_state.double())
        return [o[:, 0] @ p.out_proj.double().t(), window, S]
    if kind == "prefill":
        return list(_sequences64(s, case, [s["x"][n].double() for n in _LAYER_ARGS]))
    if kind == "layer_train":
        x = [_leaf64(s["x"][n]) for n in _LAYER_ARGS]
        o = _sequences64(s, case, x)[0]
        return [o.detach(), *torch.autograd.grad(o, x, s["d_out"].double())]
    if kind == "core":
        return list(_core64(*(s["x"][n].double() for n in _CORE_ARGS)))
    if kind == "core_train":
        x = [_leaf64(s["x"][n]) for n in _CORE_ARGS]
        o = _core64(*x)[0]
        return [o.detach(), *torch.autograd.grad(o, x, s["d_out"].double())]
    w = {n: _leaf64(t) for n, t in s["weights"].items()}
    h = _leaf64(s["hidden"])
    x = [h @ w[n].t() for n in ("in_proj_qkv", "in_proj_z", "in_proj_a", "in_proj_b")]
    o = _layer64(case, *x, *(w[n] for n in _LAYER_ARGS[4:]))[0] @ w["out_proj"].t()
    return [o.detach(), *torch.autograd.grad(o, [h, *w.values()], s["d_out"].double())]
