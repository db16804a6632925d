"""The work whose speed is measured: calls that programs using this package make,
over the sizes they make them with.

Each kind of call below has an `_<kind>_inputs` (tensors from the seed alone), a
`_<kind>_prepare` (what a program holds before the call), a `_<kind>_run` (one call
through the public entry points), a `_<kind>_work` (bytes and operations the call
cannot do without) and a `_<kind>_exact` (the same outputs in 64 bits by plain
torch).  `listed()` names one to three sizes of each kind, `draw()` others of the
same ranges.
"""
import math

import torch
import torch.nn.functional as F

from __graft_entry__ import load_package

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DTYPES = {"bf16": BF16, "fp32": F32}
BYTES = {"bf16": 2, "fp32": 4}

# FovealPattentionMLP shapes: the module's defaults and the benchmark's 8B-class layer.
MLPS = {
    "default": dict(hidden=2048, inter=6144, base=4, remote=20),
    "8b": dict(hidden=4096, inter=14336, base=8, remote=56),
}
BLOCK = 64


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=F32):
    t = torch.randn(*shape, device="cuda", generator=g)
    return (t.mul_(std) if std != 1.0 else t).to(dtype)


# --- the routed MLP, inference --------------------------------------------------------
# A layer of a served model: its active blocks were routed when the sequence began, and
# each later call streams them.  1..64 tokens are decode batches, 65..255 short prompts
# and drafts to verify, 256 and more prompts.


def _mlp_inputs(c, seed):
    s, g = MLPS[c["layer"]], _gen(seed)
    D, I = s["hidden"], s["inter"]
    w = {n: _randn(g, *shape, std=0.02, dtype=BF16) for n, shape in
         (("k_gate", (I, D)), ("k_up", (I, D)), ("v", (D, I)))}
    remote = torch.randperm(I // BLOCK - s["base"], device="cuda", generator=g)[:s["remote"]] + s["base"]
    active = torch.cat([torch.arange(s["base"], device="cuda"), remote])
    x = _randn(g, c["tokens"], D, dtype=BF16)
    return w, active, x


def _mlp_module(c, w, train):
    s = MLPS[c["layer"]]
    with torch.device("meta"):
        m = load_package().FovealPattentionMLP(hidden_dim=s["hidden"], intermediate_dim=s["inter"],
                                               base_blocks=s["base"], remote_blocks=s["remote"],
                                               use_fused_kernel=c["fused"])
    m = m.to_empty(device="cuda").train(train)
    m.offsets = torch.arange(BLOCK, device="cuda")
    with torch.no_grad():
        m.q_proj_16d.weight.zero_()
        m.block_keys_16d.zero_()
        m.out_proj_16d.weight.zero_()
        m.k_gate.copy_(w["k_gate"])
        m.k_up.copy_(w["k_up"])
        m.v.copy_(w["v"].t())
    return m


def _mlp_prepare(c, seed):
    w, active, x = _mlp_inputs(c, seed)
    m = _mlp_module(c, w, train=False)
    m.set_active_blocks(active)
    # (batch, 1, D) as a decode step passes it, (1, tokens, D) as a prompt does
    return m, (x[:, None] if c["tokens"] <= 64 else x[None])


def _mlp_run(state):
    m, x = state
    with torch.no_grad():
        return m(x)


def _mlp_work(c):
    s, M = MLPS[c["layer"]], c["tokens"]
    w = 3 * (s["base"] + s["remote"]) * BLOCK * s["hidden"]
    return {"bytes": 2 * (w + 2 * M * s["hidden"]), "flops": 2 * M * w}


def _mlp_exact(c, seed):
    w, active, x = _mlp_inputs(c, seed)
    ch = (active[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).flatten()
    x = x.double()
    y = (F.silu(x @ w["k_gate"][ch].double().t()) * (x @ w["k_up"][ch].double().t())) @ w["v"].t()[ch].double()
    return y[:, None] if c["tokens"] <= 64 else y[None]


# --- the routed MLP, training ---------------------------------------------------------
# Forward and backward of the layer in training mode: routing from the tokens, gradients
# for the input and every parameter.  The inputs have a common direction that some block
# keys point along (what a calibrated router shows), so the routed set is clear cut.


def _mlp_train_inputs(c, seed):
    s = MLPS[c["layer"]]
    D, I = s["hidden"], s["inter"]
    w, _, x = _mlp_inputs(c, seed)
    g = _gen(seed + 7_000_003)
    qw = torch.linalg.qr(_randn(g, D, 16))[0].t().contiguous()
    u = F.normalize(_randn(g, 16), dim=0)
    keys = _randn(g, I // BLOCK, 16, std=0.15)
    hot = torch.randperm(I // BLOCK - s["base"], device="cuda", generator=g)[:s["remote"]] + s["base"]
    keys[hot] += 1.5 * u
    x = (x.float() + 4.0 * (u @ qw)).to(BF16)
    p = {"q": qw.to(BF16), "keys": keys.to(BF16), "o": _randn(g, D, 16, std=0.02, dtype=BF16)}
    return w, p, hot, x, _randn(g, c["tokens"], D, dtype=BF16)


_MLP_GRADS = ("x", "k_gate", "k_up", "v", "q", "keys", "o")


def _mlp_train_prepare(c, seed):
    w, p, _, x, dy = _mlp_train_inputs(c, seed)
    m = _mlp_module(c, w, train=True)
    with torch.no_grad():
        m.q_proj_16d.weight.copy_(p["q"])
        m.block_keys_16d.copy_(p["keys"])
        m.out_proj_16d.weight.copy_(p["o"])
    return m, x[None].requires_grad_(), dy[None]


def _mlp_train_run(state):
    m, x, dy = state
    params = (x, m.k_gate, m.k_up, m.v, m.q_proj_16d.weight, m.block_keys_16d, m.out_proj_16d.weight)
    y = m(x)
    return dict(zip(_MLP_GRADS, torch.autograd.grad(y, params, dy)), y=y.detach())


def _mlp_train_work(c):
    s, M = MLPS[c["layer"]], c["tokens"]
    D, I = s["hidden"], s["inter"]
    w = 3 * (s["base"] + s["remote"]) * BLOCK * D
    # active weights, x and dy in; y, dx and the dense weight gradients out
    return {"bytes": 2 * (w + 4 * M * D + 3 * I * D), "flops": 3 * 2 * M * w}


def _mlp_train_exact(c, seed):
    s = MLPS[c["layer"]]
    w, p, hot, x, dy = _mlp_train_inputs(c, seed)
    leaf = {n: t.double().requires_grad_() for n, t in
            (("x", x), ("k_gate", w["k_gate"]), ("k_up", w["k_up"]), ("v", w["v"].t()), *p.items())}
    ch = (torch.cat([torch.arange(s["base"], device="cuda"), hot.sort().values])[:, None] * BLOCK
          + torch.arange(BLOCK, device="cuda")).flatten()
    x = leaf["x"]
    z = F.rms_norm(x @ leaf["q"].t(), (16,), eps=torch.finfo(BF16).eps)
    soft = F.softmax(z @ leaf["keys"].t() / 4.0, dim=-1)
    act = F.silu(x @ leaf["k_gate"][ch].t()) * (x @ leaf["k_up"][ch].t())
    y = act @ leaf["v"][ch] + (soft @ leaf["keys"]) @ leaf["o"].t()
    grads = dict(zip(_MLP_GRADS, torch.autograd.grad(y, [leaf[n] for n in _MLP_GRADS], dy.double())))
    return dict({n: t[None] if n == "x" else t for n, t in grads.items()}, y=y.detach()[None])


# --- routing queries to blocks --------------------------------------------------------
# Scores and the top-p selection in one call, as a prefill routes all its query blocks
# over all key blocks (the benchmark's indexer workload is the listed size).


def _route_inputs(c, seed):
    g = _gen(seed)
    Q, N, B = c["queries"], c["keys"], c["batch"]
    k = F.normalize(_randn(g, B, N, 16), dim=-1)
    pick = torch.randint(0, N, (B, Q, 4), device="cuda", generator=g)
    w = torch.rand(B, Q, 4, device="cuda", generator=g).pow(3.0)
    w = w / w.sum(-1, keepdim=True)
    near = torch.stack([k[b][pick[b]] for b in range(B)])
    q = (w[..., None] * near).sum(2) + _randn(g, B, Q, 16, std=0.1)
    return q.to(DTYPES[c["dtype"]]), k.to(DTYPES[c["dtype"]])


def _route_prepare(c, seed):
    q, k = _route_inputs(c, seed)
    return q, k, dict(causal=c["causal"], local_window_blocks=c["window"], top_p=c["top_p"], min_remote_blocks=4,
                      max_remote_blocks=c["k_max"], remote_capacity=c["k_max"], return_mass=True)


def _route_run(state):
    q, k, kw = state
    return load_package().score_and_route(q, k, **kw)


def _route_work(c):
    rows, n = c["batch"] * c["queries"], c["keys"]
    return {"bytes": 16 * BYTES[c["dtype"]] * (rows + c["batch"] * n) + rows * (4 * c["k_max"] + 8),
            "flops": rows * n * 33}


def _route_exact(c, seed):
    q, k = _route_inputs(c, seed)
    s = F.normalize(q.double(), dim=-1) @ F.normalize(k.double(), dim=-1).transpose(1, 2).contiguous() / 4.0
    Q, N = c["queries"], c["keys"]
    if c["causal"]:
        qi, ki = torch.arange(Q, device="cuda")[:, None], torch.arange(N, device="cuda")[None]
        valid, remote = ki < qi, ki < (qi - c["window"]).clamp_min(0)
    else:
        valid = torch.ones(Q, N, dtype=torch.bool, device="cuda")
        remote = (torch.arange(N, device="cuda") >= c["window"]).expand(Q, N)
    p = torch.nan_to_num(torch.softmax(s.masked_fill(~valid, -math.inf), dim=-1))
    local = (p * (valid & ~remote)).sum(-1)
    target = (c["top_p"] - local).clamp_min(0)
    cum = p.masked_fill(~remote, 0.0).topk(min(c["k_max"], N), dim=-1).values.cumsum(-1)
    avail = remote.sum(-1)
    need = ((cum < target[..., None]).sum(-1) + (target > 0)).clamp_min(4)
    count = torch.minimum(need, avail.expand_as(need)).clamp_max(c["k_max"])
    far = cum.gather(-1, (count - 1).clamp_min(0)[..., None])[..., 0]
    return [None, None, local + torch.where(count > 0, far, torch.zeros_like(far))]


# --- the indexer, training ------------------------------------------------------------
# One distillation step of the indexer on hidden states: queries at the block anchors,
# pooled keys and values, block scores, the KL loss against a teacher's block mass and
# the additive stream; gradients of its four projections (the modules' fp32 default, and
# bf16).


def _indexer_inputs(c, seed):
    g = _gen(seed)
    D, dt = c["hidden"], DTYPES[c["dtype"]]
    x = _randn(g, c["batch"], c["blocks"] * BLOCK, D, dtype=dt)
    w = {n: _randn(g, 16, D, std=D ** -0.5, dtype=dt) for n in ("q", "k", "v")}
    w["o"] = _randn(g, D, 16, std=0.02, dtype=dt)
    teacher = torch.softmax(_randn(g, c["batch"], c["blocks"], c["blocks"], std=2.0), dim=-1)
    return x, w, teacher, _randn(g, *x.shape, std=1e-3, dtype=dt)


def _indexer_prepare(c, seed):
    x, w, teacher, dy = _indexer_inputs(c, seed)
    m = load_package().FovealIndexer(hidden_size=c["hidden"], block_size=BLOCK).to("cuda", DTYPES[c["dtype"]])
    with torch.no_grad():
        for n, p in (("q", m.q_proj), ("k", m.k_proj), ("v", m.v_proj), ("o", m.out_proj)):
            p.weight.copy_(w[n])
    return m, x, teacher, dy


def _indexer_run(state):
    m, x, teacher, dy = state
    q = m.compute_query_16d(x[:, ::BLOCK])
    k, v = m.compute_kv_blocks_16d(x)
    scores = m.compute_block_scores(q, k)
    loss = m.distillation_loss(scores, teacher)
    add = m.additive_stream(scores, v)
    params = (m.q_proj.weight, m.k_proj.weight, m.v_proj.weight, m.out_proj.weight)
    grads = torch.autograd.grad((loss, add), params, (torch.ones_like(loss), dy))
    return dict(zip("qkvo", grads), loss=loss.detach(), add=add.detach())


def _indexer_work(c):
    e, n = BYTES[c["dtype"]], c["batch"] * c["blocks"] * BLOCK * c["hidden"]
    nb = c["batch"] * c["blocks"] ** 2
    # x in for the projections and again for their gradients' products with it, which a
    # pass over x cannot give before the scores are known; dy in, the stream out
    return {"bytes": e * 4 * n + 4 * nb, "flops": 2 * n * 16 * 2 * 2 + nb * 16 * 2 * 6}


def _indexer_exact(c, seed):
    x, w, teacher, dy = _indexer_inputs(c, seed)
    if x.numel() > 1 << 28:
        return None
    eps = torch.finfo(DTYPES[c["dtype"]]).eps if c["dtype"] == "bf16" else torch.finfo(F32).eps
    leaf = {n: t.double().requires_grad_() for n, t in w.items()}
    x, teacher = x.double(), teacher.double()
    B, nb, D = c["batch"], c["blocks"], c["hidden"]
    q = F.rms_norm(x[:, ::BLOCK] @ leaf["q"].t(), (16,), eps=eps)
    k = F.rms_norm(x @ leaf["k"].t(), (16,), eps=eps).view(B, nb, BLOCK, 16).mean(2)
    v = (x @ leaf["v"].t()).view(B, nb, BLOCK, 16).mean(2)
    s = F.normalize(q, dim=-1) @ F.normalize(k, dim=-1).transpose(1, 2).contiguous() / 4.0
    valid = torch.arange(nb, device="cuda")[None] < torch.arange(nb, device="cuda")[:, None]
    z = s.masked_fill(~valid, -math.inf)[:, 1:]
    t = (teacher * valid)[:, 1:]
    loss = -(t / t.sum(-1, keepdim=True) * torch.log_softmax(z, -1).masked_fill(~valid[1:], 0.0)).sum(-1).mean()
    ctx = torch.cat([torch.zeros_like(v[:, :1]), torch.softmax(z, -1) @ v], dim=1)
    add = (ctx @ leaf["o"].t()).repeat_interleave(BLOCK, dim=1)
    grads = torch.autograd.grad((loss, add), [leaf[n] for n in "qkvo"], (torch.ones_like(loss), dy.double()))
    return dict(zip("qkvo", grads), loss=loss.detach(), add=add.detach())


# --- attention of one decode step -----------------------------------------------------
# Routing and attention of one new token per sequence over a long cache: the paged bf16
# cache in one call, and the modules' default fp32 cache as routing and then attention.

DECODE = dict(window=1024, top_p=0.9, k_max=32)


def _decode_inputs(c, seed):
    g = _gen(seed)
    B, n, hd, dt = c["batch"], c["context"], c["head_dim"], DTYPES[c["dtype"]]
    k, v = (_randn(g, B, c["kv_heads"], n, hd, dtype=dt) for _ in range(2))
    P = -(-n // BLOCK)
    kp = F.normalize(_randn(g, B, P, 16), dim=-1)
    vp = _randn(g, B, P, 16, dtype=dt)
    q = _randn(g, B, c["heads"], hd, dtype=dt)
    qi = F.rms_norm(_randn(g, B, 16), (16,)).to(dt)
    table = torch.randperm(B * P, device="cuda", generator=g).view(B, P).to(torch.int32)
    return k, v, kp, vp, q, qi, table


def _decode_prepare(c, seed):
    k, v, kp, vp, q, qi, table = _decode_inputs(c, seed)
    cache = load_package().FovealKVCache(c["batch"], c["context"], c["kv_heads"], c["head_dim"], 16, BLOCK,
                                         torch.device("cuda"), DTYPES[c["dtype"]],
                                         page_table=table if c["dtype"] == "bf16" else None)
    cache.load_dense(k, v)
    cache.kp_cache.copy_(kp)
    cache.vp_cache.copy_(vp)
    cache.seq_len, cache.completed_pages = c["context"], c["context"] // BLOCK
    return cache, q, qi


def _decode_run(state):
    cache, q, qi = state
    fsi = load_package()
    pos, scale = cache.seq_len - 1, cache.head_dim ** -0.5
    route = dict(completed_pages=cache.completed_pages, top_p=DECODE["top_p"], min_remote_blocks=0,
                 max_remote_blocks=DECODE["k_max"], return_context=True)
    if cache.paged:
        return fsi.decode_step_attention(q, qi, cache, pos=pos, window=DECODE["window"], scale=scale, **route)
    pages, counts, ctx = fsi.decode_route(qi, cache.kp_cache, cache.vp_cache, pos=pos, page_size=cache.page_size,
                                          local_window=DECODE["window"], **route)
    out = fsi.decode_attention(q, cache, pos=pos, window=DECODE["window"], remote_pages=pages, remote_counts=counts,
                               scale=scale)
    return out, pages, counts, ctx


def _decode_work(c):
    e, B, n = BYTES[c["dtype"]], c["batch"], c["context"]
    far = max(0, n - DECODE["window"]) // BLOCK
    keys = min(n, DECODE["window"]) + BLOCK * min(far, DECODE["k_max"])
    P = n // BLOCK
    return {"bytes": B * (2 * keys * c["kv_heads"] * c["head_dim"] * e + P * 16 * (4 + e)
                          + 2 * c["heads"] * c["head_dim"] * e),
            "flops": B * (4 * keys * c["heads"] * c["head_dim"] + 2 * P * 16 * 2)}


def _decode_exact(c, seed):
    k, v, kp, vp, q, qi, _ = _decode_inputs(c, seed)
    B, n, hd, G = c["batch"], c["context"], c["head_dim"], c["heads"] // c["kv_heads"]
    done, lo = n // BLOCK, max(0, n - DECODE["window"])
    far = lo // BLOCK
    s = (F.normalize(qi.double(), dim=-1)[:, None] * kp[:, :done].double()).sum(-1) / 4.0
    ctx = (torch.softmax(s, -1)[..., None] * vp[:, :done].double()).sum(1)
    out = torch.zeros(B, c["heads"], hd, dtype=F64, device="cuda")
    for b in range(B):
        toks = torch.arange(lo, n, device="cuda")
        if far > 0 and done > far:
            p, order = torch.softmax(s[b, :far], -1).sort(descending=True)
            need = min(int((p.cumsum(-1) < DECODE["top_p"]).sum()) + 1, DECODE["k_max"], far)
            pages = order[:need]
            toks = torch.cat([toks, (pages[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).flatten()])
        kk, vv = (t[b][:, toks].double().repeat_interleave(G, 0) for t in (k, v))
        w = torch.softmax((kk * q[b].double()[:, None]).sum(-1) * hd ** -0.5, -1)
        out[b] = (w[..., None] * vv).sum(1)
    return [out, None, None, ctx]


# --- attention over a prompt ----------------------------------------------------------
# Block-sparse causal attention of a whole prompt (local window plus routed pages):
# forward as a served prefill runs it, forward and backward as training does.


def _attn_inputs(c, seed):
    g = _gen(seed)
    B, T, hd, dt = c["batch"], c["tokens"], c["head_dim"], DTYPES[c["dtype"]]
    q, k, v, dy = (_randn(g, B, T, h, hd, dtype=dt) for h in (c["heads"], c["kv_heads"], c["kv_heads"], c["heads"]))
    nb = -(-T // BLOCK)
    # pages below the local window, best first, as a route lists them
    far = (torch.arange(nb, device="cuda") - c["window"] // BLOCK).clamp_min(0)
    s = torch.rand(B, nb, nb, device="cuda", generator=g)
    s = s.masked_fill(torch.arange(nb, device="cuda")[None, None] >= far[None, :, None], -1.0)
    cap = min(c["pages"], nb)
    lists = s.topk(cap, dim=-1).indices.to(torch.int32)
    counts = far.clamp_max(cap).expand(B, nb).to(torch.int32).contiguous()
    return [t.transpose(1, 2) for t in (q, k, v, dy)], lists, counts


def _attn_prepare(c, seed):
    (q, k, v, dy), lists, counts = _attn_inputs(c, seed)
    if c["train"]:
        q, k, v = (t.requires_grad_() for t in (q, k, v))
    return q, k, v, dy, lists, counts, c["window"], c["train"]


def _attn_run(state):
    q, k, v, dy, lists, counts, window, train = state
    out = load_package().sparse_attention(q, k, v, lists, counts, block=BLOCK, window=window)
    if not train:
        return out
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), dy))


def _attn_pairs(c):
    """Attended (query, key) pairs of one head: the window plus the whole listed pages."""
    T, w = c["tokens"], c["window"]
    local = sum(min(t + 1, w) for t in range(T))
    nb = -(-T // BLOCK)
    cap = min(c["pages"], nb)
    far = sum(min(cap, max(0, b - w // BLOCK)) * min(BLOCK, T - b * BLOCK) for b in range(nb))
    return c["batch"] * (local + far * BLOCK)


def _attn_work(c):
    e, n = BYTES[c["dtype"]], c["batch"] * c["tokens"] * c["head_dim"]
    io = (2 * c["heads"] + 2 * c["kv_heads"]) * n * e
    if c["train"]:  # q, k, v, dy in; out, dq, dk, dv out
        io = (4 * c["heads"] + 4 * c["kv_heads"]) * n * e
    return {"bytes": io, "flops": _attn_pairs(c) * c["heads"] * c["head_dim"] * (14 if c["train"] else 4)}


def _attn_exact(c, seed):
    (q, k, v, dy), lists, counts = _attn_inputs(c, seed)
    B, T, hd, G, scale = c["batch"], c["tokens"], c["head_dim"], c["heads"] // c["kv_heads"], c["head_dim"] ** -0.5
    nb = counts.shape[1]
    out, dq = (torch.zeros(B, c["heads"], T, hd, dtype=F64, device="cuda") for _ in range(2))
    dk, dv = (torch.zeros(B, c["kv_heads"], T, hd, dtype=F64, device="cuda") for _ in range(2))
    step = 2048
    for b in range(B):
        page = torch.zeros(nb, nb, dtype=torch.bool, device="cuda")
        used = torch.arange(lists.shape[2], device="cuda")[None] < counts[b][:, None]
        page[torch.arange(nb, device="cuda")[:, None].expand_as(used)[used], lists[b].long()[used]] = True
        page = page.repeat_interleave(BLOCK, 1)[:, :T]
        for t0 in range(0, T, step):
            t = torch.arange(t0, min(T, t0 + step), device="cuda")
            s = torch.arange(T, device="cuda")[None]
            seen = ((s <= t[:, None]) & (s > t[:, None] - c["window"])) | page[t // BLOCK]
            for h in range(c["heads"]):
                kk, vv, qq = k[b, h // G].double(), v[b, h // G].double(), q[b, h, t0:t0 + step].double()
                p = torch.softmax((qq @ kk.t() * scale).masked_fill_(~seen, -math.inf), -1)
                o = p @ vv
                out[b, h, t0:t0 + step] = o
                if c["train"]:
                    g = dy[b, h, t0:t0 + step].double()
                    ds = p * (g @ vv.t() - (g * o).sum(-1, keepdim=True)) * scale
                    dq[b, h, t0:t0 + step] = ds @ kk
                    dk[b, h // G] += ds.t() @ qq
                    dv[b, h // G] += p.t() @ g
    return [out, dq, dk, dv] if c["train"] else out


# --- tile-sparse linear, training -----------------------------------------------------
# x (W o mask)^T with one tile mask for each group of 128 rows, or one for all rows (what
# the 2-D tile-sparse layer passes), and its gradients for x and W.


def _tile_inputs(c, seed):
    g = _gen(seed)
    M, K, N, t, dt = c["rows"], c["k"], c["n"], c["tile"], DTYPES[c["dtype"]]
    groups = -(-M // 128) if c["grouped"] else 1
    tiles = (K // t) * (N // t)
    mask = torch.zeros(groups, tiles, dtype=torch.bool, device="cuda")
    rank = torch.rand(groups, tiles, device="cuda", generator=g)
    mask.scatter_(1, rank.topk(max(1, int(c["density"] * tiles)), dim=1).indices, True)
    return (_randn(g, M, K, dtype=dt), _randn(g, N, K, std=0.01, dtype=dt), mask, _randn(g, M, N, dtype=dt))


def _tile_prepare(c, seed):
    x, w, mask, dy = _tile_inputs(c, seed)
    return x.requires_grad_(), w.requires_grad_(), mask, dy, c["tile"]


def _tile_run(state):
    x, w, mask, dy, tile = state
    y = load_package().blockwise_matmul(x, w, mask, tile, tile, rows_per_group=128)
    return (y.detach(), *torch.autograd.grad(y, (x, w), dy))


def _tile_work(c):
    M, K, N = c["rows"], c["k"], c["n"]
    tiles = (K // c["tile"]) * (N // c["tile"])
    share = max(1, int(c["density"] * tiles)) / tiles
    return {"bytes": BYTES[c["dtype"]] * (2 * M * K + 2 * M * N + 2 * N * K), "flops": int(6 * M * K * N * share)}


def _tile_exact(c, seed):
    x, w, mask, dy = _tile_inputs(c, seed)
    M, K, N, t = c["rows"], c["k"], c["n"], c["tile"]
    rows = 128 if c["grouped"] else M
    y, dx, dw = (torch.zeros(*s, dtype=F64, device="cuda") for s in ((M, N), (M, K), (N, K)))
    for i, m in enumerate(mask):
        em = m.view(K // t, N // t).t().repeat_interleave(t, 0).repeat_interleave(t, 1)
        r = slice(i * rows, min(M, (i + 1) * rows))
        we = w.double() * em
        y[r] = x[r].double() @ we.t()
        dx[r] = dy[r].double() @ we
        dw += (dy[r].double().t() @ x[r].double()) * em
    return [y, dx, dw]


# --- the cases ------------------------------------------------------------------------

_KINDS = {n: tuple(globals()["_%s_%s" % (n, part)] for part in ("prepare", "run", "work", "exact"))
          for n in ("mlp", "mlp_train", "route", "indexer", "decode", "attn", "tile")}


def listed():
    heads = dict(heads=32, kv_heads=8, head_dim=128)
    return [
        # one sequence being decoded: the least work a layer is called with
        dict(name="mlp_decode_1", kind="mlp", layer="default", tokens=1, fused=True),
        # a full decode batch of the benchmark's layer
        dict(name="mlp_decode_64", kind="mlp", layer="8b", tokens=64, fused=True),
        # a short prompt of an odd length
        dict(name="mlp_prompt_150", kind="mlp", layer="8b", tokens=150, fused=True),
        # a long prompt
        dict(name="mlp_prefill_4096", kind="mlp", layer="8b", tokens=4096, fused=True),
        # one training micro-batch of the default layer
        dict(name="mlp_train_2048", kind="mlp_train", layer="default", tokens=2048, fused=True),
        # the benchmark's routing: every query against every block
        dict(name="route_8192x4096", kind="route", batch=1, queries=8192, keys=4096, dtype="bf16", causal=False,
             window=0, top_p=0.9, k_max=64),
        # one distillation step over a batch of sequences, in the modules' default type
        dict(name="indexer_train_fp32", kind="indexer", batch=4, blocks=64, hidden=2048, dtype="fp32"),
        # one decode step of a served batch with long contexts
        dict(name="decode_bf16_32x32768", kind="decode", batch=32, context=32768, dtype="bf16", **heads),
        # one decode step of a few sequences on the default cache, mid page
        dict(name="decode_fp32_4x9001", kind="decode", batch=4, context=9001, dtype="fp32", **heads),
        # a long prompt served
        dict(name="attn_prefill_16384", kind="attn", batch=1, tokens=16384, dtype="bf16", window=1024, pages=32,
             train=False, **heads),
        # a training sequence
        dict(name="attn_train_8192", kind="attn", batch=1, tokens=8192, dtype="bf16", window=1024, pages=32, train=True,
             **heads),
        # a training step of the benchmark's tile-sparse product
        dict(name="tile_train_4096", kind="tile", rows=4096, k=8192, n=8192, tile=128, density=0.25, grouped=True,
             dtype="bf16"),
    ]


def _span(rng, lo, hi, step=1):
    """A whole number of steps in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def draw(rng):
    kind = rng.choice(("mlp", "mlp", "mlp", "mlp_train", "route", "indexer", "decode", "decode", "attn", "attn", "tile"))
    if kind == "mlp":
        lo, hi = rng.choice(((1, 64), (65, 255), (256, 4096)))
        return dict(kind=kind, layer=rng.choice(("default", "8b")), tokens=_span(rng, lo, hi), fused=rng.random() < 0.8)
    if kind == "mlp_train":
        return dict(kind=kind, layer="default", tokens=_span(rng, 128, 2048), fused=rng.random() < 0.8)
    if kind == "route":
        causal = rng.random() < 0.5
        n = _span(rng, 64, 4096)
        return dict(kind=kind, batch=rng.choice((1, 1, 2)), queries=n if causal else _span(rng, 64, 4096), keys=n,
                    dtype=rng.choice(("bf16", "fp32")), causal=causal, window=rng.choice((0, 8)) if causal else 0,
                    top_p=rng.choice((0.8, 0.9, 0.95)), k_max=rng.choice((8, 16, 64)))
    if kind == "indexer":
        blocks = _span(rng, 4, 128)
        return dict(kind=kind, batch=rng.randint(1, max(1, 256 // blocks)) if blocks > 32 else rng.randint(1, 4),
                    blocks=blocks, hidden=rng.choice((1024, 2048)), dtype=rng.choice(("fp32", "bf16")))
    if kind == "decode":
        dtype = rng.choice(("bf16", "bf16", "fp32"))
        batch = _span(rng, 1, 32)
        kv = rng.choice((2, 8))
        return dict(kind=kind, batch=batch, context=_span(rng, 1500, min(65536, (1 << 20) // batch)), dtype=dtype,
                    heads=4 * kv, kv_heads=kv, head_dim=rng.choice((64, 128)))
    if kind == "attn":
        train = rng.random() < 0.5
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp32"))
        top = {("bf16", False): 16384, ("bf16", True): 8192, ("fp32", False): 4096, ("fp32", True): 2048}[dtype, train]
        kv = rng.choice((2, 8))
        return dict(kind=kind, batch=1, tokens=_span(rng, 512, top), dtype=dtype, window=rng.choice((256, 512, 1024)),
                    pages=rng.choice((8, 16, 32)), train=train, heads=4 * kv, kv_heads=kv,
                    head_dim=rng.choice((64, 128)))
    tile = rng.choice((64, 128))
    return dict(kind=kind, rows=_span(rng, 100, 2048), k=_span(rng, 1024, 8192, 256), n=_span(rng, 1024, 8192, 256),
                tile=tile, density=rng.choice((0.1, 0.25, 0.5)), grouped=rng.random() < 0.5, dtype="bf16")


def prepare(case, seed):
    return case["kind"], _KINDS[case["kind"]][0](case, seed)


def run(state):
    kind, own = state
    return _KINDS[kind][1](own)


def work(case):
    return _KINDS[case["kind"]][2](case)


def exact(case, seed):
    return _KINDS[case["kind"]][3](case, seed)


# About four times the largest relative error against `exact` seen over the ranges, of any
# output: 3.9e-3 for the MLP in bf16, 7.2e-3 for its training (the router's gradient),
# 5e-8 for the route's mass, 6.6e-3 / 1.4e-6 for the indexer, 2.7e-3 / 4.6e-7 for a decode
# step (bf16 / fp32), 1.8e-3 / 1.1e-6 for attention, 4.2e-3 for the tile product.  Single
# values in cancelling sums are further off: "max" is four times the largest seen there.
# Ranks of equal probabilities may change places.
_TOLERANCE = {
    ("mlp", "bf16"): {"rel": 1.5e-2, "max": 0.08},
    ("mlp_train", "bf16"): {"rel": 2.8e-2, "max": 0.2},
    ("route", "bf16"): {"rel": 4e-7, "max": 1e-6, "differ": 1e-3},
    ("route", "fp32"): {"rel": 4e-7, "max": 1e-6, "differ": 1e-3},
    ("indexer", "bf16"): {"rel": 2.6e-2, "max": 0.16},
    ("indexer", "fp32"): {"rel": 6e-6, "max": 4e-5},
    ("decode", "bf16"): {"rel": 1e-2, "max": 0.03, "differ": 1e-3},
    ("decode", "fp32"): {"rel": 2e-6, "max": 2e-5, "differ": 1e-3},
    ("attn", "bf16"): {"rel": 7e-3, "max": 0.6},
    ("attn", "fp32"): {"rel": 4.5e-6, "max": 3e-5},
    ("tile", "bf16"): {"rel": 1.6e-2, "max": 0.16},
}


def tolerance(case):
    return _TOLERANCE[case["kind"], case.get("dtype", "bf16")]
