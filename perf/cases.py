"""Cases for timing the framework through its public entry points: training steps of the operators and of a
layer, prompt processing, and single-token decoding, from the smallest calls to the longest sequences.

A case is a dict of plain values:

  op      "clean"  fused_ccq_clean_read            "gdn"  fused_chunk_ccq_gdn       "gla"  fused_chunk_ccq_gla
          "decode" fused_recurrent_ccq_gdn          "graph" CapturedDecode over DecodeStep layers
          "layer"  CCQGDN forward and backward      "layer_decode" GDNLayerDecode in a captured graph
  train   forward and the gradients of every input (True), or forward with final states, no gradients (False)
  B T H K V   batch, tokens, heads, key and value channels per head
  gate    lambda from the fused per-head gate (True) or handed in (False)
  l2norm  raw q and k, normalised by the operator (True), or normalised by the caller (False)
  seqs    > 0: one packed row of T tokens holding that many sequences (cu_seqlens)
  past    tokens already seen: initial states of that many tokens are handed in
  dtype   activations' type
"""

import math

import torch

CHUNK = 64
DEV = "cuda"


def listed():
    return [
        # The cleaning operator alone on one short fp32 sequence (the first benchmark configuration's sizes): an
        # experiment at a small scale, where launches and host work count.
        dict(name="clean_small", op="clean", train=True, B=1, T=512, H=4, K=64, V=0, gate=False, l2norm=False,
             seqs=0, past=0, dtype="float32"),
        # The cleaning operator alone at training size (the benchmark's fused cleaning configuration).
        dict(name="clean_train", op="clean", train=True, B=8, T=4096, H=8, K=128, V=0, gate=True, l2norm=False,
             seqs=0, past=0, dtype="bfloat16"),
        # The headline workload: fused cleaning + gated delta rule, forward and backward.
        dict(name="gdn_train", op="gdn", train=True, B=8, T=4096, H=8, K=128, V=128, gate=True, l2norm=False,
             seqs=0, past=0, dtype="bfloat16"),
        # Fine-tuning on a packed row of ragged documents with small heads: odd lengths, normalisation in the operator.
        dict(name="gdn_train_packed", op="gdn", train=True, B=1, T=6001, H=6, K=64, V=128, gate=False, l2norm=True,
             seqs=13, past=0, dtype="bfloat16"),
        # One 32K-token sequence with the default layer's heads (the published overhead shape): the longest calls.
        dict(name="gdn_train_long", op="gdn", train=True, B=1, T=32768, H=6, K=256, V=512, gate=True, l2norm=False,
             seqs=0, past=0, dtype="bfloat16"),
        # A prompt of odd length on one sequence with those heads, its states kept for decoding: time to first token.
        dict(name="gdn_prefill", op="gdn", train=False, B=1, T=1531, H=6, K=256, V=512, gate=False, l2norm=True,
             seqs=0, past=0, dtype="bfloat16"),
        # The gated-linear-attention operator at its layer configuration's training size.
        dict(name="gla_train", op="gla", train=True, B=4, T=8192, H=4, K=128, V=256, gate=False, l2norm=True,
             seqs=0, past=0, dtype="bfloat16"),
        # The next part of two prompts, continued from cached states.
        dict(name="gla_prefill", op="gla", train=False, B=2, T=777, H=4, K=128, V=256, gate=False, l2norm=True,
             seqs=0, past=1000, dtype="bfloat16"),
        # One token of sixteen sequences through the recurrent operator, as the layer calls it in generation.
        dict(name="gdn_decode", op="decode", train=False, B=16, T=1, H=4, K=256, V=512, gate=False, l2norm=True,
             seqs=0, past=4096, dtype="bfloat16"),
        # The captured decode step of eight layers' recurrent states for the same sixteen sequences.
        dict(name="gdn_decode_graph", op="graph", train=False, B=16, T=1, H=4, K=256, V=512, gate=True, l2norm=True,
             seqs=0, past=4096, dtype="bfloat16", layers=8),
        # A whole layer's training step (projections, short convolutions, gates, operator, gated norm).
        dict(name="gdn_layer_train", op="layer", train=True, B=4, T=4096, H=4, K=256, V=512, gate=False,
             l2norm=False, seqs=0, past=0, dtype="bfloat16", hidden=1024),
        # A whole layer's token step for a few sequences, captured: serving at low batch.
        dict(name="gdn_layer_decode", op="layer_decode", train=False, B=4, T=1, H=4, K=256, V=512, gate=False,
             l2norm=False, seqs=0, past=2048, dtype="bfloat16", hidden=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["clean", "gdn", "gdn", "gdn", "gla", "gla", "decode", "graph", "layer", "layer_decode"])
    c = dict(op=op, train=True, gate=False, l2norm=True, seqs=0, past=0, dtype="bfloat16")
    if op in ("clean", "gdn", "gla"):
        K = rng.choice([64, 128, 128, 256])
        V = 0 if op == "clean" else rng.choice({64: [64, 128], 128: [128, 256], 256: [256, 512]}[K])
        H = rng.choice([2, 3, 4, 6, 8])
        c.update(H=H, K=K, V=V, train=rng.random() < 0.6, gate=rng.random() < 0.4, l2norm=op != "clean")
        if op == "gdn":
            c["l2norm"] = rng.random() < 0.5
        # up to the headline workload's tokens x heads, and less than the longest call's work
        units = min(8 * 4096 * 8, 32768 * 6 * 256 * (256 + 512) // (K * (K + V)))
        tokens = _log(rng, 300, units // H)
        c["B"] = min(rng.choice([1, 1, 2, 4, 8]), max(1, tokens // 200))
        c["T"] = tokens // c["B"]
        if c["B"] == 1 and rng.random() < 0.5:
            c["seqs"] = rng.randint(2, max(2, min(24, c["T"] // 64)))
        elif not c["train"] and rng.random() < 0.5:
            c["past"] = _log(rng, 64, 4096)
        if op == "clean" and rng.random() < 0.3:
            c["dtype"] = "float32"
        if not c["train"]:
            c["gate"] = False
    elif op in ("decode", "graph"):
        K = rng.choice([64, 128, 256])
        c.update(train=False, B=_log(rng, 1, 32), T=1, H=rng.choice([2, 4, 6, 8]), K=K, V=K * rng.choice([1, 2]),
                 past=_log(rng, 64, 16384), gate=op == "graph")
        if op == "graph":
            c["layers"] = rng.choice([2, 4, 8])
    else:
        K = rng.choice([128, 256])
        c.update(H=rng.choice([2, 4]), K=K, V=2 * K, hidden=rng.choice([512, 1024]), l2norm=False)
        if op == "layer":
            c.update(B=rng.choice([1, 2, 4]), T=_log(rng, 200, 4096))
        else:
            c.update(train=False, B=_log(rng, 1, 16), T=1, past=_log(rng, 64, 16384))
    return c


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------

def _unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _bounds(c, seed):
    """Boundaries of the packed sequences: random lengths of at least one token."""
    if not c["seqs"]:
        return None
    gen = torch.Generator().manual_seed(seed)
    cut = torch.randperm(c["T"] - 1, generator=gen)[:c["seqs"] - 1].sort().values + 1
    return [0] + cut.tolist() + [c["T"]]


def _past(c, n, rnd):
    """States after c["past"] tokens: a delta-rule state of ordinary size, sums of unit keys' products and keys."""
    H, K, V = c["H"], c["K"], c["V"]
    keys = _unit(rnd(n, H, 256, K)) * math.sqrt(c["past"] / 256)
    st = dict(h0=keys.transpose(-1, -2) @ keys, m0=keys.sum(-2) * math.sqrt(c["past"] / 256))
    if V:
        st["s0"] = 0.1 * rnd(n, H, K, V)
    return st


def _op_inputs(c, seed):
    gen = torch.Generator(DEV).manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    def uni(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=gen, device=DEV)

    B, T, H, K, V = c["B"], c["T"], c["H"], c["K"], c["V"]
    dt = getattr(torch, c["dtype"])
    x = {}
    for name in ("q", "k"):
        t = rnd(B, T, H, K)
        x[name] = (t if c["l2norm"] else _unit(t)).to(dt)
    if c["gate"]:
        x["w"], x["b"] = 0.02 * rnd(H, K), uni(-1.0, 1.0, H)
    else:
        x["lam"] = torch.sigmoid(rnd(B, T, H, 1)).to(dt)
    if V:
        x["v"] = rnd(B, T, H, V).to(dt)
    if c["op"] in ("gdn", "decode", "graph"):
        rate = torch.exp(uni(0.0, math.log(16.0), H))
        x["g"] = -torch.nn.functional.softplus(rnd(B, T, H)) * rate
        x["beta"] = torch.sigmoid(rnd(B, T, H))
    if c["op"] == "gla":
        x["g"] = torch.nn.functional.logsigmoid(rnd(B, T, H, K)) / 16.0
    leaves = list(x)
    x["do"] = rnd(B, T, H, V or K).to(dt)
    cu = _bounds(c, seed)
    if c["past"]:
        x.update(_past(c, B, rnd))
    return x, leaves, cu


def _layer(c, seed):
    from ccq_amd import CCQGDN
    torch.manual_seed(seed)
    with torch.device(DEV):
        layer = CCQGDN(hidden_size=c["hidden"], head_dim=c["K"], num_heads=c["H"], expand_v=c["V"] // c["K"],
                       mode="fused_chunk", layer_idx=0)
    layer = layer.to(torch.bfloat16)
    gen = torch.Generator(DEV).manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    st = dict(layer=layer, x=rnd(c["B"], c["T"], c["hidden"]).to(torch.bfloat16))
    if c["op"] == "layer":
        st["dy"] = rnd(c["B"], c["T"], c["hidden"]).to(torch.bfloat16)
        st["x"].requires_grad_()
    else:
        st.update(_past(c, c["B"], rnd))
        H, K, V = c["H"], c["K"], c["V"]
        st["convs"] = tuple(0.5 * rnd(c["B"], d, layer.conv_size - 1) for d in (H * K, H * K, H * V))
        st["convs"] = tuple(t.to(torch.bfloat16) for t in st["convs"])
    return st


def prepare(case, seed):
    c = case
    st = dict(case=c)
    if c["op"] == "layer":
        st.update(_layer(c, seed))
        st["params"] = [p for p in st["layer"].parameters() if p.requires_grad]
    elif c["op"] == "layer_decode":
        from ccq_amd.graph import GDNLayerDecode
        with torch.no_grad():
            st.update(_layer(c, seed))
            step = GDNLayerDecode(st["layer"], c["B"])
            entry = dict(recurrent_state=(st.pop("s0"), st.pop("h0"), st.pop("m0"), c["past"]),
                         conv_state=st.pop("convs"))
            step.load(entry)
            step(st["x"], st["x"])  # the kernels are loaded before the capture
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                st["y"] = step(st["x"], st["x"])
            step.load(entry)
        st.update(step=step, graph=graph)
    elif c["op"] == "graph":
        from ccq_amd.graph import CapturedDecode, DecodeStep
        steps = []
        for i in range(c["layers"]):
            x, _, _ = _op_inputs(c, seed * 64 + i)
            s = DecodeStep(c["B"], c["H"], c["K"], c["V"], mode="gdn", gate=True, device=DEV)
            for name, src in (("q", "q"), ("k", "k"), ("v", "v"), ("g", "g"), ("beta", "beta"), ("gate_w", "w"),
                              ("gate_b", "b")):
                getattr(s, name).copy_(x[src])
            s.load_state(x["s0"], x["h0"], x["m0"], c["past"])
            steps.append(s)
        st.update(steps=steps, captured=CapturedDecode(steps).capture())
    else:
        x, leaves, cu = _op_inputs(c, seed)
        if c["train"]:
            for n in leaves:
                x[n].requires_grad_()
        st.update(x=x, leaves=leaves, cu=None if cu is None else torch.tensor(cu, device=DEV))
    return st


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------

def run(state):
    c = state["case"]
    if c["op"] == "layer":
        y = state["layer"](state["x"])[0]
        grads = torch.autograd.grad(y, [state["x"]] + state["params"], state["dy"])
        return (y,) + grads
    if c["op"] == "layer_decode":
        state["graph"].replay()
        s = state["step"].step
        return state["y"], s.S, s.C, s.m
    if c["op"] == "graph":
        state["captured"].replay()
        return [(s.o, s.S, s.C, s.m) for s in state["steps"]]
    import ccq_amd
    x = state["x"]
    kw = dict(initial_cov_state=x.get("h0"), initial_mean_state=x.get("m0"), position_offset=c["past"],
              cu_seqlens=state["cu"], output_final_state=not c["train"])
    if c["op"] != "decode" and c["gate"]:
        kw.update(gate_w=x["w"], gate_b=x["b"])
    if c["op"] == "clean":
        def op():
            return ccq_amd.fused_ccq_clean_read(x["q"], x["k"], x.get("lam"), **kw)
    elif c["op"] == "gdn":
        def op():
            return ccq_amd.fused_chunk_ccq_gdn(x["q"], x["k"], x["v"], x.get("lam"), x["g"], x["beta"],
                                               initial_state=x.get("s0"), use_qk_l2norm_in_kernel=c["l2norm"], **kw)
    elif c["op"] == "gla":
        def op():
            return ccq_amd.fused_chunk_ccq_gla(x["q"], x["k"], x["v"], x.get("lam"), x["g"],
                                               initial_state=x.get("s0"), **kw)
    else:
        def op():
            return ccq_amd.fused_recurrent_ccq_gdn(x["q"], x["k"], x["v"], x["lam"], g=x["g"], beta=x["beta"],
                                                   initial_state=x.get("s0"), use_qk_l2norm_in_kernel=c["l2norm"],
                                                   **kw)
    if not c["train"]:
        with torch.no_grad():
            return op()
    o = op()[0]
    return (o,) + torch.autograd.grad(o, [x[n] for n in state["leaves"]], x["do"])


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------

def _op_work(c):
    """(bytes, flops) of one operator call: each input read once, each output written once; every contraction
    of the 64-token chunked form once, a backward as twice its forward."""
    B, T, H, K, V = c["B"], c["T"], c["H"], c["K"], c["V"]
    n = B * T * H
    e = 4 if c["dtype"] == "float32" else 2
    scalars = {"clean": 1, "gdn": 3, "gla": 1 + K, "decode": 3, "graph": 3}[c["op"]]
    if c["gate"]:
        scalars -= 1
    io = n * (e * (2 * K + V) + 4 * scalars)      # inputs
    out = n * e * (V or K)
    if c["op"] in ("decode", "graph"):
        state = 4 * B * H * (K * K + K + K * V)
        return io + out + 2 * state, n * (6 * K * V + 4 * K * K)
    flops = n * (4 * K * K + 4 * CHUNK * K)
    if c["op"] == "gdn":
        flops += n * (6 * K * V + CHUNK * (6 * K + 4 * V) + 2 * CHUNK * CHUNK // 3)
    if c["op"] == "gla":
        flops += n * (4 * K * V + CHUNK * (2 * K + 2 * V))
    byts = io + out
    if c["train"]:
        byts += io + out + io                      # the inputs again, the upstream gradient, the inputs' gradients
        flops *= 3
    else:
        state = 4 * max(c["seqs"], B) * H * (K * K + K + K * V)
        byts += state * (2 if c["past"] else 1)
    return byts, flops


def work(case):
    c = case
    if c["op"] in ("layer", "layer_decode"):
        n = c["B"] * c["T"]
        key, val, d = c["H"] * c["K"], c["H"] * c["V"], c["hidden"]
        weights = d * (2 * key + 3 * val + 2 * c["H"]) + key * c["H"]
        f = 2 * n * weights
        if c["op"] == "layer":
            _, of = _op_work(dict(c, op="gdn"))
            return dict(bytes=2 * (2 * weights + 6 * n * d), flops=3 * f + of)
        # the projections' weights and the states
        ob, of = _op_work(dict(c, op="decode"))
        return dict(bytes=2 * weights + ob + 4 * n * d, flops=f + of)
    b, f = _op_work(c)
    m = c.get("layers", 1)
    return dict(bytes=b * m, flops=f * m)


def tolerance(case):
    # Measured against 64 bits: outputs of an operator 0.2 to 0.35 % off (bf16 operands and results); a layer's
    # gradients 0.6 to 1.4 %, the decay parameters' most, since a rounding travels through every later product.
    if case["op"] == "layer":
        return {"rel": 2.5e-2, "max": 0.25}
    return {"rel": 8e-3, "max": 0.1}


# ---------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------------

def _heads_first(t, pad):
    """[B, T, H, ...] -> [B, H, chunks, 64, ...], padded with zeros."""
    t = t.transpose(1, 2)
    if pad:
        t = torch.cat([t, t.new_zeros(*t.shape[:2], pad, *t.shape[3:])], 2)
    return t.reshape(*t.shape[:2], -1, CHUNK, *t.shape[3:])


def _tokens_first(t, T):
    t = t.reshape(*t.shape[:2], -1, *t.shape[4:])
    return t[:, :, :T].transpose(1, 2)


def _clean64(q, k, lam, h0, m0, offset):
    """q_clean, the final sum of k k^T and the final sum of k; q, k [B, H, n, 64, K], lam [B, H, n, 64]."""
    Bn, H, n, _, K = q.shape
    mask = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    kk = k.transpose(-1, -2) @ k
    tot = kk.cumsum(2)
    pre = tot - kk
    msum = k.reshape(Bn, H, n * CHUNK, K).cumsum(2)
    if h0 is not None:
        pre, tot, msum = pre + h0[:, :, None], tot + h0[:, :, None], msum + m0[:, :, None]
    z = q @ pre + ((q @ k.transpose(-1, -2)) * mask) @ k
    m = msum.reshape(q.shape)
    pos = (torch.arange(1, n * CHUNK + 1, device=q.device, dtype=q.dtype) + offset).reshape(n, CHUNK, 1)
    corr = z / pos - (m * q).sum(-1, keepdim=True) * m / (pos * pos)
    return q - lam[..., None] * corr, tot[:, :, -1], msum[:, :, -1]


def _gdn64(q, k, v, g, beta, s0):
    """Gated delta rule in its chunked form; g, beta [B, H, n, 64].  Returns o and the final state."""
    Bn, H, n, _, K = q.shape
    one = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device)
    G = g.cumsum(-1)
    diff = G[..., :, None] - G[..., None, :]
    decay = torch.exp(diff.masked_fill(~one.tril(), -math.inf))
    A = beta[..., None] * (k @ k.transpose(-1, -2)) * decay.masked_fill(~one.tril(-1), 0.0)
    # (I + A)^-1 of the nilpotent A: (I - A)(I + A^2)(I + A^4) ... (I + A^32)
    eye = torch.eye(CHUNK, dtype=q.dtype, device=q.device)
    inv, power = eye - A, A
    for _ in range(5):
        power = power @ power
        inv = inv + inv @ power
    w, u = inv @ ((beta * torch.exp(G))[..., None] * k), inv @ (beta[..., None] * v)
    last = torch.exp(G[..., -1:] - G)[..., None] * k
    S = q.new_zeros(Bn, H, K, v.shape[-1]) if s0 is None else s0
    states, us = [], []
    for i in range(n):
        states.append(S)
        U = u[:, :, i] - w[:, :, i] @ S
        us.append(U)
        S = torch.exp(G[:, :, i, -1])[..., None, None] * S + last[:, :, i].transpose(-1, -2) @ U
    P = (q @ k.transpose(-1, -2)) * decay
    o = torch.exp(G)[..., None] * (q @ torch.stack(states, 2)) + P @ torch.stack(us, 2)
    return o * K ** -0.5, S


def _gla64(q, k, v, gk, s0):
    """Gated linear attention in its chunked form; gk [B, H, n, 64, K]."""
    Bn, H, n, _, K = q.shape
    mask = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    G = gk.cumsum(-2)
    qe = q * torch.exp(G)
    add = (k * torch.exp(G[..., -1:, :] - G)).transpose(-1, -2) @ v
    S = q.new_zeros(Bn, H, K, v.shape[-1]) if s0 is None else s0
    states = []
    for i in range(n):
        states.append(S)
        S = torch.exp(G[:, :, i, -1])[..., None] * S + add[:, :, i]
    o = qe @ torch.stack(states, 2) + ((qe @ (k * torch.exp(-G)).transpose(-1, -2)) * mask) @ v
    return o * K ** -0.5, S


def _op64(op, x, l2norm, offset):
    """One dense operator call on float64 tensors laid out [B, T, H, ...]; (o, S, C, m) or (q_clean, C, m)."""
    T = x["q"].shape[1]
    pad = -T % CHUNK
    q, k = x["q"], x["k"]
    if l2norm:
        q, k = _unit(q), _unit(k)
    lam = torch.sigmoid((q * x["w"]).sum(-1) + x["b"]) if "w" in x else x["lam"].squeeze(-1)
    q, k, lam = (_heads_first(t, pad) for t in (q, k, lam))
    qc, C, m = _clean64(q, k, lam, x.get("h0"), x.get("m0"), offset)
    if op == "clean":
        return _tokens_first(qc, T), C, m
    v, g = _heads_first(x["v"], pad), _heads_first(x["g"], pad)
    if op == "gla":
        o, S = _gla64(qc, k, v, g, x.get("s0"))
    else:
        o, S = _gdn64(qc, k, v, g, _heads_first(x["beta"], pad), x.get("s0"))
    return _tokens_first(o, T), S, C, m


def _conv64(x, weight, before):
    """Causal short convolution over time and SiLU; before [B, D, W - 1] or None."""
    W = weight.shape[-1]
    head = x.new_zeros(x.shape[0], W - 1, x.shape[2]) if before is None else before.transpose(1, 2)
    full = torch.cat([head, x], 1)
    y = sum(full[:, i:i + x.shape[1]] * weight[:, 0, i] for i in range(W))
    return torch.nn.functional.silu(y)


def _layer64(c, p, x, state=None, convs=None):
    H, K, V = c["H"], c["K"], c["V"]
    lin = lambda t, name: t @ p[name + ".weight"].T  # noqa: E731
    cq, ck, cv = convs or (None, None, None)
    q = _conv64(lin(x, "q_proj"), p["q_conv1d.weight"], cq)
    k = _conv64(lin(x, "k_proj"), p["k_conv1d.weight"], ck)
    v = _conv64(lin(x, "v_proj"), p["v_conv1d.weight"], cv)
    lam = torch.sigmoid(lin(q, "erase_lambda_proj") + p["erase_lambda_proj.bias"])
    heads = lambda t, d: t.reshape(*t.shape[:2], H, d)  # noqa: E731
    g = -torch.exp(p["A_log"]) * torch.nn.functional.softplus(lin(x, "a_proj") + p["dt_bias"])
    t = dict(q=heads(q, K), k=heads(k, K), v=heads(v, V), lam=lam[..., None], g=g,
             beta=torch.sigmoid(lin(x, "b_proj")), **(state or {}))
    o, S, C, m = _op64("gdn", t, True, c["past"])
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5) * p["o_norm.weight"]
    o = o * torch.nn.functional.silu(heads(lin(x, "g_proj"), V))
    return lin(o.reshape(*o.shape[:2], H * V), "o_proj"), S, C, m


def exact(case, seed):
    c = case
    if c["op"] in ("layer", "layer_decode"):
        st = _layer(c, seed)
        p = {n: t.detach().double() for n, t in st["layer"].named_parameters()}
        x = st["x"].detach().double()
        if c["op"] == "layer":
            wanted = [x] + list(p.values())
            for t in wanted:
                t.requires_grad_()
            y = _layer64(c, p, x)[0]
            return (y,) + torch.autograd.grad(y, wanted, st["dy"].double())
        with torch.no_grad():
            y, S, C, m = _layer64(c, p, x, {n: st[n].double() for n in ("s0", "h0", "m0")},
                                  [t.double() for t in st["convs"]])
            return x + y, S, C, m
    if c["op"] == "graph":
        with torch.no_grad():
            out = []
            for i in range(c["layers"]):
                x, _, _ = _op_inputs(c, seed * 64 + i)
                # (the recurrent step's gate reads the normalised query, as the operators' does)
                out.append(_op64("gdn", {n: t.double() for n, t in x.items()}, True, c["past"]))
            return out
    raw, leaves, cu = _op_inputs(c, seed)
    x = {n: t.double() for n, t in raw.items()}
    if c["train"]:
        for n in leaves:
            x[n].requires_grad_()
    parts = []
    with torch.set_grad_enabled(c["train"]):
        for a, b in zip(cu[:-1], cu[1:]) if cu else [(0, c["T"])]:
            part = {n: t if n in ("w", "b", "h0", "m0", "s0") else t[:, a:b] for n, t in x.items()}
            parts.append(_op64("gdn" if c["op"] == "decode" else c["op"], part, c["l2norm"], c["past"]))
        outs = tuple(torch.cat(t, 1 if i == 0 else 0) for i, t in enumerate(zip(*parts)))
    if not c["train"]:
        return outs
    return (outs[0],) + torch.autograd.grad(outs[0], [x[n] for n in leaves], x["do"])
