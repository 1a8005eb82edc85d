"""Performance cases of the framework: what its users call, from one decoded token to whole prompts.

Every case goes through the torch front end (nemotron_infer_amd/ops.py) on the sizes of this
repository's model configuration (hidden 3136, MLP 12544, 40 / 8 attention heads of 128, Mamba-2
96 heads of 80 in 8 groups) or, among the drawn cases, two generic smaller models.  Kinds:

  linear         one fp8 projection (a program's own projection, or a head)
  mlp            the fp8 MLP block
  attn_decode    the fp8 attention block on one new token, against a KV cache
  attn_prefill   the fp8 attention block over a prompt, filling the KV caches
  mamba_decode   the fp8 Mamba-2 block on one new token of each of `batch` sequences
  mamba_prefill  the fp8 Mamba-2 block over `batch` prompts, with their final states
  step           a whole decode step of a stack of blocks, captured in a HIP graph as a serving
                 loop keeps it ("m" Mamba-2, "f" MLP, "a" attention)

Inputs: seeded N(0, 0.02) weights quantised to e4m3 with a per-tensor scale (or per-row
log-uniform scales), N(0, 1) activations, relu(z)^2 or x50 outliers where a case says so.
"""
import math

import torch

from nemotron_infer_amd import ops, synth

DEV = "cuda:0"
D = 128          # attention head dimension
N_STATE = 128    # Mamba-2 state size
EPS = 1e-5

# hidden, MLP width, query heads, KV heads, Mamba heads, Mamba head dimension, Mamba groups
MODELS = {
    "h3136": (3136, 12544, 40, 8, 96, 80, 8),
    "h2048": (2048, 8192, 16, 4, 64, 64, 8),
    "h2560": (2560, 10240, 32, 8, 80, 64, 4),
}


def listed():
    return [
        # one projection of one token: the smallest call (attention output projection)
        {"name": "linear_m1", "kind": "linear", "M": 1, "N": 3136, "K": 5120, "act": "normal", "scales": "per_tensor"},
        # one token through an MLP block: interactive decode
        {"name": "mlp_m1", "kind": "mlp", "model": "h3136", "M": 1},
        # a small decode batch, an odd number of sequences
        {"name": "mlp_m13", "kind": "mlp", "model": "h3136", "M": 13},
        # a chat turn's short prompt
        {"name": "mlp_m100", "kind": "mlp", "model": "h3136", "M": 100},
        # a chunk of a longer prompt, a ragged number of tokens
        {"name": "mlp_m777", "kind": "mlp", "model": "h3136", "M": 777},
        # a full prompt: the prefill workload of the benchmark
        {"name": "mlp_m2048", "kind": "mlp", "model": "h3136", "M": 2048},
        # one token against a conversation of some thousand tokens
        {"name": "attn_decode_s4000", "kind": "attn_decode", "model": "h3136", "S": 4000},
        # a medium prompt, ragged
        {"name": "attn_prefill_s700", "kind": "attn_prefill", "model": "h3136", "S": 700},
        # a long prompt: attention's quadratic part counts
        {"name": "attn_prefill_s4096", "kind": "attn_prefill", "model": "h3136", "S": 4096},
        # batched serving: one token of each of 24 sequences, each with its own state
        {"name": "mamba_decode_b24", "kind": "mamba_decode", "model": "h3136", "batch": 24},
        # two prompts at once
        {"name": "mamba_prefill_b2_s500", "kind": "mamba_prefill", "model": "h3136", "batch": 2, "S": 500},
        # a decode step of eight layers in the model's mix, one HIP graph
        {"name": "step_8_layers", "kind": "step", "model": "h3136", "layers": "mfmfmamf", "S": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "mlp", "attn_decode", "attn_prefill", "mamba_decode", "mamba_prefill", "step"])
    model = rng.choice(["h3136", "h3136", "h2048", "h2560"])
    if kind == "linear":
        hidden, inter, hq, hkv, mh, mp, mg = MODELS[model]
        N, K = rng.choice([(hidden, hq * D), (inter, hidden), (hidden, inter), (hq * D, hidden),
                           (2 * mh * mp + 2 * mg * N_STATE + mh, hidden), (hidden, mh * mp)])
        return {"kind": kind, "M": _log(rng, 1, 2048), "N": N, "K": K,
                "act": rng.choice(["normal", "relu2", "outliers"]), "scales": rng.choice(["per_tensor", "log_uniform"])}
    case = {"kind": kind, "model": model}
    if kind == "mlp":
        case["M"] = _log(rng, 1, 2048)
    elif kind == "attn_decode":
        case["S"] = _log(rng, 16, 32768)
    elif kind == "attn_prefill":
        case["S"] = _log(rng, 16, 4096)
    elif kind == "mamba_decode":
        case["batch"] = _log(rng, 1, 64)
    elif kind == "mamba_prefill":
        case["batch"] = rng.randint(1, 4)
        case["S"] = _log(rng, 16, 2048 // case["batch"])
    else:
        case["layers"] = "".join(rng.choice("mmmffa") for _ in range(rng.randint(2, 8)))
        case["S"] = _log(rng, 16, 8192)
    return case


# --- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _norm_w(n, g):
    return 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _mlp_layer(model, seed):
    hidden, inter = MODELS[model][:2]
    return {"norm": _norm_w(hidden, _gen(seed)), "up": synth.make_weight(inter, hidden, seed + 1, DEV),
            "down": synth.make_weight(hidden, inter, seed + 2, DEV)}


def _attn_layer(model, seed):
    hidden, _, hq, hkv = MODELS[model][:4]
    shapes = [(hq * D, hidden), (hkv * D, hidden), (hkv * D, hidden), (hidden, hq * D)]
    return {"norm": _norm_w(hidden, _gen(seed)),
            "mats": [synth.make_weight(n, k, seed + 1 + i, DEV) for i, (n, k) in enumerate(shapes)]}


def _mamba_layer(model, seed):
    hidden = MODELS[model][0]
    H, P, G = MODELS[model][4:]
    inter, conv_dim = H * P, H * P + 2 * G * N_STATE
    g = _gen(seed)
    f = {"device": DEV, "dtype": torch.float32, "generator": g}
    return {"norm": _norm_w(hidden, g), "in": synth.make_weight(inter + conv_dim + H, hidden, seed + 1, DEV),
            "out": synth.make_weight(hidden, inter, seed + 2, DEV),
            "conv_w": 0.3 * torch.randn((conv_dim, 4), **f), "conv_b": 0.1 * torch.randn(conv_dim, **f),
            "A_log": torch.rand(H, **f) * 2.5 - 1.0, "D": torch.randn(H, **f), "dt_bias": 0.5 * torch.randn(H, **f),
            "gnorm": 1.0 + 0.1 * torch.randn(inter, **f)}


def _mamba_states(model, batch, seed):
    """States in mid conversation: the conv window holds activations, the SSM state sums of them."""
    H, P, G = MODELS[model][4:]
    g = _gen(seed)
    conv = torch.randn((batch, H * P + 2 * G * N_STATE, 3), generator=g, device=DEV)
    ssm = 0.5 * torch.randn((batch, H, P, N_STATE), generator=g, device=DEV)
    return conv, ssm


def _caches(model, cap, seed):
    hkv = MODELS[model][3]
    g = _gen(seed)
    return [torch.randn((hkv, cap, D), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)]


def _stack(case, base):
    """The layers of a "step" case: [(kind, layer, state tensors)]."""
    layers = []
    for i, c in enumerate(case["layers"]):
        seed = base + 100 + 20 * i
        if c == "m":
            layers.append((c, _mamba_layer(case["model"], seed), _mamba_states(case["model"], 1, seed + 10)))
        elif c == "f":
            layers.append((c, _mlp_layer(case["model"], seed), ()))
        else:
            layers.append((c, _attn_layer(case["model"], seed), _caches(case["model"], case["S"] + 1, seed + 10)))
    return layers


def _inputs(case, seed):
    """The tensors of a case: what prepare() and exact() both start from."""
    base = 1000 * (seed % 1000003)
    kind = case["kind"]
    if kind == "linear":
        w, s = synth.make_weight(case["N"], case["K"], base + 1, DEV, scales=case["scales"])
        x = synth.make_act(case["M"], case["K"], base + 2, DEV, kind="relu2" if case["act"] == "relu2" else "normal",
                           outlier_frac=0.001 if case["act"] == "outliers" else 0.0)
        return {"x": x, "w": w, "s": s}
    model = case["model"]
    hidden, hkv = MODELS[model][0], MODELS[model][3]
    rows = {"mlp": case.get("M"), "attn_decode": 1, "attn_prefill": case.get("S"), "mamba_decode": case.get("batch"),
            "mamba_prefill": case.get("batch", 0) * case.get("S", 0), "step": 1}[kind]
    st = {"x": synth.make_act(rows, hidden, base + 1, DEV)}
    if kind == "mlp":
        st["layer"] = _mlp_layer(model, base + 10)
    elif kind in ("attn_decode", "attn_prefill"):
        st["layer"] = _attn_layer(model, base + 10)
        if kind == "attn_decode":
            st["caches"] = _caches(model, case["S"] + 1, base + 50)
        else:
            st["caches"] = [torch.zeros((hkv, case["S"], D), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    elif kind in ("mamba_decode", "mamba_prefill"):
        st["layer"] = _mamba_layer(model, base + 10)
        st["states"] = _mamba_states(model, case["batch"], base + 50)
    else:
        st["stack"] = _stack(case, base)
    return st


# --- one pass -------------------------------------------------------------------------------


def _mlp(x, L, out):
    return ops.mlp_forward_fp8(x, L["norm"], *L["up"], *L["down"], out=out)


def _attn_weights(L):
    return [t for m in L["mats"] for t in m]


def _mamba_weights(L):
    return (L["norm"], *L["in"], L["conv_w"], L["conv_b"], L["A_log"], L["D"], L["dt_bias"], L["gnorm"], *L["out"])


def _step(st, case):
    cur, nxt = st["x"], st["hidden"][0]
    for i, (c, L, state) in enumerate(st["stack"]):
        if c == "m":
            ops.mamba_decode_fp8(cur, *_mamba_weights(L), *state, *MODELS[case["model"]][4:], out=nxt)
        elif c == "f":
            _mlp(cur, L, nxt)
        else:
            ops.attn_decode_fp8(cur, L["norm"], *_attn_weights(L), *state, case["S"], out=nxt)
        cur, nxt = nxt, st["hidden"][(i + 1) % 2]
    return cur


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    if case["kind"] == "linear":
        st["out"] = torch.empty((case["M"], case["N"]), dtype=torch.bfloat16, device=DEV)
        return st
    st["out"] = torch.empty_like(st["x"])
    if case["kind"] == "step":
        # A serving loop captures its decode step once: an eager pass first (workspaces), the
        # states put back afterwards, then the capture.
        st["hidden"] = [torch.empty_like(st["x"]) for _ in range(2)]
        kept = [[t.clone() for t in state] for _, _, state in st["stack"]]
        _step(st, case)
        for (_, _, state), old in zip(st["stack"], kept):
            for t, o in zip(state, old):
                t.copy_(o)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            st["out"] = _step(st, case)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.linear_fp8_w8a16(st["x"], st["w"], st["s"], out=st["out"])
    if kind == "mlp":
        return _mlp(st["x"], st["layer"], st["out"])
    if kind == "attn_decode":
        L = st["layer"]
        ops.attn_decode_fp8(st["x"], L["norm"], *_attn_weights(L), *st["caches"], case["S"], out=st["out"])
        return [st["out"], *st["caches"]]
    if kind == "attn_prefill":
        L = st["layer"]
        k_cache, v_cache = st["caches"]
        ops.attn_forward_fp8(st["x"], L["norm"], *_attn_weights(L), k_cache=k_cache, v_cache=v_cache, out=st["out"])
        return [st["out"], k_cache, v_cache]
    if kind == "mamba_decode":
        ops.mamba_decode_fp8(st["x"], *_mamba_weights(st["layer"]), *st["states"], *MODELS[case["model"]][4:],
                             out=st["out"])
        return [st["out"], *st["states"]]
    if kind == "mamba_prefill":
        conv, ssm = st["states"]
        ops.mamba_forward_fp8(st["x"], *_mamba_weights(st["layer"]), *MODELS[case["model"]][4:], batch=case["batch"],
                              conv_state_out=conv, ssm_state_out=ssm, out=st["out"])
        return [st["out"], conv, ssm]
    st["graph"].replay()
    return [st["out"], *[t for _, _, state in st["stack"] for t in state]]


# --- what a pass cannot do without ----------------------------------------------------------


def _layer_work(kind, model, rows, batch, S):
    """(bytes, flops) of one block over `rows` tokens; S the prompt length or the cached positions."""
    hidden, inter, hq, hkv, H, P, G = MODELS[model]
    io = 4 * rows * hidden + 4 * hidden                      # x in, out, norm weight
    if kind == "f":
        n = 2 * inter * hidden
        return n + 4 * (inter + hidden) + io, 2 * rows * n
    if kind == "a":
        n = 2 * hq * D * hidden + 2 * hkv * D * hidden
        nbytes = n + 4 * (hq * D + 2 * hkv * D + hidden) + io
        pairs = S if rows == 1 else S * (S + 1) // 2         # (query, key) pairs of a head
        kv = 4 * hkv * D * (S + 1 if rows == 1 else S)       # K and V, read or written
        return nbytes + kv, 2 * rows * n + 4 * pairs * D * hq
    conv_dim = H * P + 2 * G * N_STATE
    n = hidden * (2 * H * P + 2 * G * N_STATE + H) + hidden * H * P
    nbytes = n + 4 * (H * P + conv_dim + H + hidden) + io + 4 * (5 * conv_dim + 3 * H + H * P)
    state = 4 * batch * (conv_dim * 3 + H * P * N_STATE)
    # decode reads and writes the states; prefill writes them
    return nbytes + state * (2 if S == 0 else 1), 2 * rows * n + rows * (8 * conv_dim + 6 * H * P * N_STATE)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K + 4 * N + 2 * M * K + 2 * M * N, "flops": 2 * M * N * K}
    model = case["model"]
    if kind == "mlp":
        b, f = _layer_work("f", model, case["M"], 1, 0)
    elif kind == "attn_decode":
        b, f = _layer_work("a", model, 1, 1, case["S"])
    elif kind == "attn_prefill":
        b, f = _layer_work("a", model, case["S"], 1, case["S"])
    elif kind == "mamba_decode":
        b, f = _layer_work("m", model, case["batch"], case["batch"], 0)
    elif kind == "mamba_prefill":
        b, f = _layer_work("m", model, case["batch"] * case["S"], case["batch"], case["S"])
    else:
        each = [_layer_work(c, model, 1, 1, case["S"] if c == "a" else 0) for c in case["layers"]]
        b, f = sum(e[0] for e in each), sum(e[1] for e in each)
    return {"bytes": b, "flops": f}


# About four times what another order of the float32 sums was measured to change: bf16 outputs that
# fall on the other side of a rounding tie (single blocks up to 5.3e-4 in the 2-norm and 0.015 in
# one value), carried from block to block in a step (7.2e-3 and 0.062 after eight).
def tolerance(case):
    if case["kind"] == "linear":
        return {"rel": 1e-3, "max": 0.04}
    if case["kind"] == "step":
        return {"rel": 2.5e-2, "max": 0.25}
    return {"rel": 2e-3, "max": 0.06}


# --- the same in 64 bits --------------------------------------------------------------------


def _lin64(x, w):
    codes, scale = w
    out = []
    for r in range(0, codes.shape[0], 4096):
        w64 = codes[r:r + 4096].view(torch.float8_e4m3fn).to(torch.float64)
        out.append(x @ w64.t())
    return torch.cat(out, dim=1) * scale.double()


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _mlp64(x, L):
    up = torch.relu(_lin64(_rms64(x, L["norm"]), L["up"]))
    return x + _lin64(up * up, L["down"])


def _qkv64(x, L):
    h = _rms64(x, L["norm"])
    return [_lin64(h, m).view(x.shape[0], -1, D) for m in L["mats"][:3]]


def _attn_decode64(x, L, caches, S):
    q, k, v = _qkv64(x, L)
    kc, vc = (c.double().clone() for c in caches)
    ratio = q.shape[1] // kc.shape[0]
    o = torch.empty((q.shape[1], D), dtype=torch.float64, device=x.device)
    for h in range(q.shape[1]):
        p = torch.softmax((kc[h // ratio, :S] @ q[0, h]) / math.sqrt(D), dim=0)
        o[h] = p @ vc[h // ratio, :S]
    kc[:, S], vc[:, S] = k[0], v[0]
    return x + _lin64(o.view(1, -1), L["mats"][3]), kc, vc


def _attn_prefill64(x, L):
    q, k, v = _qkv64(x, L)
    S = x.shape[0]
    ratio = q.shape[1] // k.shape[1]
    o = torch.empty_like(q)
    mask = torch.ones((S, S), dtype=torch.bool, device=x.device).tril()
    for h in range(q.shape[1]):
        sc = (q[:, h] @ k[:, h // ratio].t()) / math.sqrt(D)
        o[:, h] = torch.softmax(sc.masked_fill(~mask, -math.inf), dim=1) @ v[:, h // ratio]
    return x + _lin64(o.view(S, -1), L["mats"][3]), k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()


def _mamba64(x, L, model, batch, conv, ssm):
    """The block over x [batch * S, hidden] token by token, from the given states."""
    H, P, G = MODELS[model][4:]
    inter = H * P
    proj = _lin64(_rms64(x, L["norm"]), L["in"]).view(batch, x.shape[0] // batch, -1)
    z, xbc, dt = proj.split([inter, inter + 2 * G * N_STATE, H], dim=2)
    conv, ssm = conv.double().clone(), ssm.double().clone()
    seq = torch.cat([conv.transpose(1, 2), xbc], dim=1)
    S = xbc.shape[1]
    taps = L["conv_w"].double()
    c = L["conv_b"].double() + sum(seq[:, t:t + S] * taps[:, t] for t in range(4))
    c = c * torch.sigmoid(c)
    dt = torch.nn.functional.softplus(dt + L["dt_bias"].double())
    dA = torch.exp(-torch.exp(L["A_log"].double()) * dt)
    xs = c[..., :inter].reshape(batch, S, H, P)
    B = c[..., inter:inter + G * N_STATE].reshape(batch, S, G, N_STATE).repeat_interleave(H // G, dim=2)
    C = c[..., inter + G * N_STATE:].reshape(batch, S, G, N_STATE).repeat_interleave(H // G, dim=2)
    y = torch.empty_like(xs)
    for t in range(S):
        ssm = ssm * dA[:, t, :, None, None] + (dt[:, t, :, None] * xs[:, t])[..., None] * B[:, t, :, None, :]
        y[:, t] = (ssm * C[:, t, :, None, :]).sum(dim=3)
    y = y + L["D"].double()[:, None] * xs
    u = (y.reshape(batch * S, inter) * (z * torch.sigmoid(z)).reshape(batch * S, inter)).view(batch * S, G, -1)
    g = _rms64(u, torch.ones((), device=x.device)).view(batch * S, inter) * L["gnorm"].double()
    return x + _lin64(g, L["out"]), seq[:, -3:].transpose(1, 2).contiguous(), ssm


def exact(case, seed):
    st = _inputs(case, seed)
    kind = case["kind"]
    x = st["x"].double()
    if kind == "linear":
        return _lin64(x, (st["w"], st["s"]))
    if kind == "mlp":
        return _mlp64(x, st["layer"])
    if kind == "attn_decode":
        return list(_attn_decode64(x, st["layer"], st["caches"], case["S"]))
    if kind == "attn_prefill":
        return list(_attn_prefill64(x, st["layer"]))
    if kind in ("mamba_decode", "mamba_prefill"):
        conv, ssm = st["states"]
        if kind == "mamba_prefill":
            conv, ssm = torch.zeros_like(conv), torch.zeros_like(ssm)
        return list(_mamba64(x, st["layer"], case["model"], case["batch"], conv, ssm))
    states = []
    for c, L, state in st["stack"]:
        if c == "f":
            x = _mlp64(x, L)
        elif c == "m":
            x, *new = _mamba64(x, L, case["model"], 1, *state)
            states += new
        else:
            x, *new = _attn_decode64(x, L, state, case["S"])
            states += new
    return [x, *states]
