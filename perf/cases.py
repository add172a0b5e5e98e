"""The workloads whose speed is watched: the calls a training or serving program
makes of this library, over the range of sizes it is used at.

Every tensor is float32.  Four groups:

  core          causal attention forward + backward of one layer (a training
                step's core), recomputing or keeping the scores, heads-first or
                the reference's per-position [B][T][H*D] layout; from_probs
                takes the attention weights as given (the reference's
                attention_backward contract)
  layer         the whole projection + core + projection layer, forward and
                backward with weight gradients
  decode        one query per sequence against a K/V cache (serving)
  wave*         harmonic coherence attention: a training step, a prompt's
                prefill into the KV cache, one decoded token per sequence

Sizes are those of the library's own configurations (168-, 384-, 768- and
4096-dim) and ragged ones between them.
"""
import math

import torch

from __graft_entry__ import load_package

wha = load_package()


def _dev():
    return torch.device("cuda:0")


def listed():
    return [
        # the research configuration's training step: the smallest call, a few
        # microseconds of work, where latency and launches count
        dict(name="core_168", kind="core", B=4, H=4, T=256, D=42, layout="bhtd", keep=False),
        # the grammar configuration's training step, scores kept (the plan's default)
        dict(name="core_384_kept", kind="core", B=16, H=8, T=512, D=48, layout="bhtd", keep=True),
        # the production configuration's training step, scores recomputed
        dict(name="core_768", kind="core", B=8, H=12, T=1024, D=64, layout="bhtd", keep=False),
        # odd batch, length and head dim in the per-position layout the reference uses
        dict(name="core_ragged", kind="core", B=3, H=10, T=1531, D=56, layout="bthd", keep=False),
        # the 4096-dim preset, scores kept: the largest listed work
        dict(name="core_4096_kept", kind="core", B=4, H=32, T=2048, D=128, layout="bhtd", keep=True),
        # attention_backward as the reference's trait has it: weights given, used as they are
        dict(name="from_probs_768", kind="probs", B=8, H=12, T=1024, D=64),
        # a whole attention layer (c_attn, core, c_proj) in training
        dict(name="layer_768", kind="layer", B=8, H=12, T=1024, D=64),
        # serving: 64 sequences, one token each, against 8192 cached positions
        dict(name="decode_768", kind="decode", B=64, H=12, T=8192, D=64),
        # a wave-attention training step at the research size ...
        dict(name="wave_168", kind="wave", B=4, H=4, T=256, D=42, C=16),
        # ... and at the production size
        dict(name="wave_768", kind="wave", B=8, H=12, T=1024, D=64, C=16),
        # serving the wave model: prompts into the cache ...
        dict(name="wave_prefill_768", kind="wave_prefill", B=4, H=12, T=2048, D=64, C=16),
        # ... and one token for each of 32 sequences
        dict(name="wave_decode_768", kind="wave_decode", B=32, H=12, T=4096, D=64, C=16),
    ]


def _loguniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


_HEAD_DIMS = (32, 40, 42, 48, 56, 64, 64, 80, 96, 100, 128)


def draw(rng):
    """One more case of the listed kinds: sizes spread over their logarithm."""
    kind = rng.choice(("core", "core", "core", "probs", "layer", "decode", "wave", "wave", "wave_prefill",
                       "wave_decode"))
    for _ in range(1000):
        c = dict(kind=kind, B=_loguniform(rng, 1, 16), H=rng.choice((1, 2, 4, 6, 8, 10, 12, 16, 32)),
                 D=rng.choice(_HEAD_DIMS))
        if kind == "core":
            c.update(T=_loguniform(rng, 33, 3000), layout=rng.choice(("bhtd", "bthd")), keep=rng.random() < 0.5)
            limit = 4e11
        elif kind == "probs":
            c.update(T=_loguniform(rng, 33, 2048))
            limit = 1e11
        elif kind == "layer":
            c.update(T=_loguniform(rng, 64, 2048))
            limit = 4e11
        elif kind == "decode":
            c.update(B=_loguniform(rng, 1, 64), T=_loguniform(rng, 128, 16384))
            limit = 2e9
        elif kind == "wave":
            c.update(T=_loguniform(rng, 64, 2500), C=rng.choice((0, 5, 8, 16, 30)))
            limit = 2e11
        elif kind == "wave_prefill":
            c.update(T=_loguniform(rng, 64, 3000), C=rng.choice((0, 16)))
            limit = 2e11
        else:
            c.update(B=_loguniform(rng, 1, 64), T=_loguniform(rng, 128, 8192), C=rng.choice((0, 16)))
            limit = 4e9
        w = work(c)
        if w["flops"] <= limit and w["bytes"] <= 3.3e9:
            return c
    raise RuntimeError("no size of this kind is within the limits")


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


def _normal(g, *shape, sd=1.0):
    return torch.randn(*shape, generator=g, device=_dev()) * sd


def _heads(buf, c, H, D):
    """Heads view [B][H][T][D] of columns c*H*D .. of buf [B][T][n*H*D]."""
    B, T = buf.shape[:2]
    return buf[:, :, c * H * D:(c + 1) * H * D].unflatten(2, (H, D)).permute(0, 2, 1, 3)


def _qkv(case, seed):
    """Queries, keys and values of unit variance (projections of a normed
    hidden state), so that scores q.k/sqrt(D) are of unit variance too, and the
    upstream gradient."""
    B, H, T, D = (case[k] for k in "BHTD")
    g = _gen(seed)
    if case.get("layout", "bhtd") == "bhtd":
        return tuple(_normal(g, B, H, T, D) for _ in range(4))
    return tuple(_heads(_normal(g, B, T, H * D), 0, H, D) for _ in range(4))


def _layer_inputs(case, seed):
    B, H, T, D = (case[k] for k in "BHTD")
    E, M = H * D, B * T
    g = _gen(seed)
    return dict(x=_normal(g, M, E), wa=_normal(g, 3 * E, E, sd=E ** -0.5), ba=_normal(g, 3 * E, sd=0.1),
                wp=_normal(g, E, E, sd=E ** -0.5), bp=_normal(g, E, sd=0.1), dy=_normal(g, M, E, sd=M ** -0.5))


def _decided(x, pw, pb):
    """Which rows of x [N][E] have every head's phase decided: not within
    float32 rounding of the edge between two buckets (either side would be
    right, and moves a key in or out of its neighbours' rows) and not at the
    origin, where the phase has no direction."""
    H, _, E = pw.shape
    rs = torch.matmul(x.double(), pw[:, :2].double().reshape(H * 2, E).t().contiguous()).view(-1, H, 2)
    rs = rs + pb[:, :2].double()
    edge = torch.atan2(rs[..., 1], rs[..., 0]) / (math.pi / 4)
    dist = (edge - edge.round()).abs() * (math.pi / 4)
    mag = rs.norm(dim=-1)
    return ((mag > 0.01) & (dist * mag > 4e-6)).all(-1)


def _wave_inputs(case, seed):
    """Weights as an initialised model has them (projections of a unit-variance
    input are O(1)) and a normed hidden state; the few positions whose phases
    rounding would decide are drawn again."""
    B, H, T, D, C = (case[k] for k in "BHTDC")
    E = H * D
    g = _gen(seed)
    w = (_normal(g, H), _normal(g, H, 2 + C, E, sd=E ** -0.5), _normal(g, H, 2 + C, sd=0.1),
         _normal(g, H, D, D, sd=D ** -0.5), _normal(g, H, D, sd=0.1), _normal(g, E, E, sd=E ** -0.5),
         _normal(g, E, sd=0.1))
    x = _normal(g, B if case["kind"] == "wave_decode" else B * T, E)
    for _ in range(8):
        again = ~_decided(x, w[1], w[2])
        x = torch.where(again[:, None], _normal(g, *x.shape), x)
    return g, w, x if case["kind"] == "wave_decode" else x.view(B, T, E)


def _wave_cache_entries(case, g, hraw):
    """A filled KV cache: phases over the circle and value rows."""
    B, H, T, D = (case[k] for k in "BHTD")
    phase = (torch.rand(B, H, T, generator=g, device=_dev()) * 2 - 1) * math.pi
    values = _normal(g, B, H, T, D)
    return phase, values


def _bucket(phase):
    """phase_to_bucket: the eighth of the circle a phase falls into."""
    tau = torch.tensor(2 * math.pi, dtype=phase.dtype, device=phase.device)
    nrm = torch.fmod(torch.fmod(phase, tau) + tau, tau)
    return (nrm / (tau / 8)).floor().clamp(0, 7).to(torch.int32)


def prepare(case, seed):
    kind = case["kind"]
    B, H, T, D = (case[k] for k in "BHTD")
    if kind == "core":
        q, k, v, do = _qkv(case, seed)
        st = dict(kind=kind)
        if case["keep"]:
            like = lambda: torch.empty_strided(q.shape, q.stride(), device=q.device)
            o, dq, dk, dv = like(), like(), like(), like()
            lse = torch.empty(B, H, T, device=q.device)
            st.update(plan=wha.AttnPlan(q, k, v, o, lse, do, dq, dk, dv), out=(o, lse, dq, dk, dv))
        else:
            ws = torch.empty(wha.attn_bwd_workspace_bytes(wha.layout_of(q)) // 4 + 64, device=q.device)
            st.update(plan=None, q=q, k=k, v=v, do=do, ws=ws)
        return st
    if kind == "probs":
        q, k, v, do = _qkv(case, seed)
        att = torch.empty(B, H, T, T, device=q.device)
        mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
        for b in range(B):
            s = torch.matmul(q[b], k[b].transpose(1, 2).contiguous()) / math.sqrt(D)
            att[b] = torch.softmax(s.masked_fill_(mask, -math.inf), -1)
        L = wha.layout_of(q)
        ws = torch.empty(int(wha.lib().wha_attn_bwd_from_probs_workspace_size(L)) // 4 + 64, device=q.device)
        return dict(kind=kind, q=q, k=k, v=v, do=do, att=att, ws=ws)
    if kind == "layer":
        st = _layer_inputs(case, seed)
        E, M = H * D, B * T
        e = lambda *s: torch.empty(*s, device=_dev())
        qkv, obuf, dobuf, d_qkv = (e(M, 3 * E) for _ in range(4))  # o and d_o share q's strides
        hv = lambda buf, c: _heads(buf.view(B, T, 3 * E), c, H, D)
        q = hv(qkv, 0)
        L = wha.layout_of(q)
        dw_ws = max(int(wha.lib().wha_linear_bwd_dw_workspace_size(M, n, E)) for n in (E, 3 * E))
        st.update(kind=kind, E=E, qkv=qkv, obuf=obuf, dobuf=dobuf, d_qkv=d_qkv, q=q, k=hv(qkv, 1), v=hv(qkv, 2),
                  o=hv(obuf, 0), do=hv(dobuf, 0), dq=hv(d_qkv, 0), dk=hv(d_qkv, 1), dv=hv(d_qkv, 2), out=e(M, E),
                  dx=e(M, E), lse=e(B, H, T), sc=wha.attn_scores_buffer(L, _dev()),
                  wsa=e(wha.attn_bwd_workspace_bytes(L) // 4 + 64), wsl=e(dw_ws // 4 + 64))
        return st
    if kind == "decode":
        g = _gen(seed)
        q = _normal(g, B, H, D)
        kc, vc = _normal(g, B, H, T, D), _normal(g, B, H, T, D)
        ws = torch.empty(int(wha.lib().wha_decode_workspace_size(wha.layout_of(kc))) // 4 + 64, device=_dev())
        return dict(kind=kind, q=q, k=kc, v=vc, ws=ws)
    C = case["C"]
    E = H * D
    g, w, x = _wave_inputs(case, seed)
    W = wha.WaveAttnWeights(*w)
    e = lambda n: torch.empty(n // 4 + 64, device=_dev())
    if kind == "wave":
        shape = wha.WaveShape(B, T, E, H, C)
        return dict(kind=kind, W=W, x=x, dy=_normal(g, B, T, E, sd=(B * T) ** -0.5),
                    wsf=e(wha.wave_fwd_workspace_bytes(shape)), wsb=e(wha.wave_bwd_workspace_bytes(shape)))
    if kind == "wave_prefill":
        shape = wha.WaveShape(B, T, E, H, C)
        return dict(kind=kind, W=W, x=x, cache=wha.WaveKvCache(B, H, D, T, _dev()),
                    ws=e(int(wha.lib().wha_wave_kv_prefill_workspace_size(shape))))
    cache = wha.WaveKvCache(B, H, D, T + 1, _dev())
    phase, values = _wave_cache_entries(case, g, w[0])
    n = torch.nn.functional.softplus(w[0])[None, :, None]
    cache.phase[:, :, :T] = phase
    cache.bucket[:, :, :T] = _bucket(phase)
    cache.cs[:, :, :T, 0] = torch.cos(n * phase)
    cache.cs[:, :, :T, 1] = torch.sin(n * phase)
    cache.values[:, :, :T] = values
    return dict(kind=kind, W=W, x=x, cache=cache, T=T, B=B,
                ws=e(wha.wave_kv_decode_workspace_bytes(wha.WaveShape(B, 1, E, H, C), T + 1)))


# ---------------------------------------------------------------- one pass


def run(st):
    kind = st["kind"]
    if kind == "core":
        if st["plan"] is not None:
            st["plan"].fwd()
            st["plan"].bwd()
            return st["out"]
        o, lse = wha.attn_fwd(st["q"], st["k"], st["v"])
        dq, dk, dv = wha.attn_bwd(st["q"], st["k"], st["v"], o, st["do"], lse, workspace=st["ws"])
        return o, lse, dq, dk, dv
    if kind == "probs":
        return wha.attn_bwd_from_probs(st["do"], st["q"], st["k"], st["v"], st["att"], workspace=st["ws"])
    if kind == "layer":
        E, o2, do2 = st["E"], st["obuf"][:, :st["E"]], st["dobuf"][:, :st["E"]]
        wha.linear_fwd(st["x"], st["wa"], st["ba"], out=st["qkv"])
        wha.attn_fwd(st["q"], st["k"], st["v"], out=st["o"], lse=st["lse"], scores=st["sc"])
        wha.linear_fwd(o2, st["wp"], st["bp"], out=st["out"])
        wha.linear_bwd_dx(st["dy"], st["wp"], out=do2)
        dwp, dbp = wha.linear_bwd_dw(st["dy"], o2, workspace=st["wsl"])
        wha.attn_bwd(st["q"], st["k"], st["v"], st["o"], st["do"], st["lse"], workspace=st["wsa"], dq=st["dq"],
                     dk=st["dk"], dv=st["dv"], scores=st["sc"])
        wha.linear_bwd_dx(st["d_qkv"], st["wa"], out=st["dx"])
        dwa, dba = wha.linear_bwd_dw(st["d_qkv"], st["x"], workspace=st["wsl"])
        return st["out"], st["dx"], dwa, dba, dwp, dbp
    if kind == "decode":
        return wha.decode_fwd(st["q"], st["k"], st["v"], workspace=st["ws"])
    if kind == "wave":
        out, _, cache = wha.wave_attention_forward(st["W"], st["x"], workspace=st["wsf"])
        g = wha.wave_attention_backward_full(st["W"], cache, st["dy"], workspace=st["wsb"])
        return (out, g.d_normed, g.d_harmonic_raw, g.d_proj_w, g.d_proj_b, g.d_v_w, g.d_v_b, g.out_proj_w,
                g.out_proj_b)
    cache = st["cache"]
    if kind == "wave_prefill":
        out = wha.prefill_attention(st["W"], st["x"], cache, workspace=st["ws"])
        return out, cache.cs, cache.phase, cache.bucket, cache.values
    cache.lengths = [st["T"]] * st["B"]  # the same position again on each pass
    out = wha.forward_one_attention(st["W"], st["x"], cache, workspace=st["ws"])
    # the entries the call appends: all that it writes of the cache
    T = st["T"]
    return out, cache.cs[:, :, T], cache.phase[:, :, T], cache.bucket[:, :, T], cache.values[:, :, T]


# ---------------------------------------------------------------- least work


def work(case):
    kind = case["kind"]
    B, H, T, D = (case[k] for k in "BHTD")
    pairs = B * H * T * (T + 1) // 2
    act = 4 * B * H * T * D  # bytes of one [B][H][T][D] tensor
    rows = 4 * B * H * T
    E, M = H * D, B * T
    if kind == "core":
        # q, k, v in, o and lse out; q, k, v, o, do, lse in, dq, dk, dv out
        return dict(bytes=13 * act + 2 * rows, flops=12 * D * pairs)
    if kind == "probs":
        return dict(bytes=7 * act + 4 * pairs, flops=8 * D * pairs)
    if kind == "layer":
        lin = 2 * M * E * 4 * E
        weights = 4 * 4 * E * E
        return dict(bytes=27 * act + 2 * rows + 3 * weights, flops=3 * lin + 12 * D * pairs)
    if kind == "decode":
        return dict(bytes=2 * act + 8 * B * H * D, flops=4 * D * B * H * T)
    C = case["C"]
    P = 2 + C
    seen = 3 / 8  # share of the pairs in neighbouring buckets
    weights = 4 * (H * P * E + H * D * D + E * E)
    if kind == "wave":
        proj = 2 * M * (E * H * P + E * D + E * E)
        core = seen * pairs * 2 * (2 + C + D)
        return dict(bytes=int(9 * act + 6 * M * H * P * 4 + 3 * weights), flops=int(3 * proj + 3 * core))
    if kind == "wave_prefill":
        proj = 2 * M * (E * H * 2 + E * D + E * E)
        return dict(bytes=int(5 * act + 4 * rows + weights), flops=int(proj + seen * pairs * 2 * (2 + D)))
    proj = 2 * B * (E * H * 2 + E * D + E * E)
    return dict(bytes=int(seen * (act + 2 * rows) + rows + weights + 8 * B * E),
                flops=int(proj + seen * B * H * T * 2 * (2 + D)))


# ---------------------------------------------------------------- 64-bit results


def _core64(q, k, v, do, att=None):
    """Causal attention of one sequence's heads [H][T][D] in 64 bits: o, lse,
    dq, dk, dv (att given: its weights are used as they are)."""
    T, D = q.shape[1:]
    mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    scale = 1 / math.sqrt(D)
    lse = None
    if att is None:
        s = (torch.matmul(q, k.transpose(1, 2).contiguous()) * scale).masked_fill_(mask, -math.inf)
        lse = torch.logsumexp(s, -1)
        att = torch.exp(s - lse[..., None])
    else:
        att = att.masked_fill(mask, 0)
    o = torch.matmul(att, v)
    dp = torch.matmul(do, v.transpose(1, 2).contiguous())
    ds = att * (dp - (att * dp).sum(-1, keepdim=True)) * scale
    dq = torch.matmul(ds, k)
    dk = torch.matmul(ds.transpose(1, 2).contiguous(), q)
    dv = torch.matmul(att.transpose(1, 2).contiguous(), do)
    return o, lse, dq, dk, dv


def _wave64(w, x, dy=None, content=True):
    """The wave attention in 64 bits: out, values and phases, and with dy the
    gradients of x and of every weight."""
    hraw, pw, pb, vw, vb, ow, ob = w
    B, T, E = x.shape
    H, P = pw.shape[:2]
    D, C = E // H, P - 2
    xd = x.double().requires_grad_(dy is not None)
    ws = [t.double().requires_grad_(dy is not None) for t in w]
    hraw, pw, pb, vw, vb, ow, ob = ws
    causal = torch.ones(T, T, dtype=torch.bool, device=x.device).tril()
    prev = torch.ones(T, T, dtype=torch.bool, device=x.device).tril(-1).triu(-1)
    eye = torch.eye(T, dtype=torch.bool, device=x.device)
    outs, vals, phases, grads = [], [], [], None
    for b in range(B):  # a sequence at a time: the [H][T][T] weights in 64 bits
        n = torch.nn.functional.softplus(hraw)
        pr = torch.matmul(xd[b], pw.reshape(H * P, E).t().contiguous()).view(T, H, P) + pb
        pr = pr.permute(1, 0, 2)
        phi = torch.atan2(pr[..., 1], pr[..., 0])
        bk = _bucket(phi.detach())
        near = torch.remainder(bk[:, None, :] - bk[:, :, None] + 1, 8) <= 2
        see = causal & (near | prev | eye)
        s = torch.cos(n[:, None, None] * (phi[:, :, None] - phi[:, None, :]))
        if C > 0 and content:
            c = pr[..., 2:]
            s = s + torch.matmul(c, c.transpose(1, 2).contiguous()) / math.sqrt(C)
        att = torch.softmax(s.masked_fill(~see, -math.inf), -1)
        xv = xd[b].view(T, H, D).permute(1, 0, 2)
        val = torch.matmul(xv, vw.transpose(1, 2).contiguous()) + vb[:, None, :]
        merged = torch.matmul(att, val).permute(1, 0, 2).reshape(T, E)
        out = torch.matmul(merged, ow.t().contiguous()) + ob
        if dy is not None:
            gb = torch.autograd.grad(out, [xd] + ws, dy[b].double(), allow_unused=True)
            gb = [torch.zeros_like(t) if g is None else g for t, g in zip([xd] + ws, gb)]
            grads = gb if grads is None else [p + q for p, q in zip(grads, gb)]
        outs.append(out.detach())
        vals.append(val.detach())
        phases.append(phi.detach())
    return torch.stack(outs), torch.stack(vals), torch.stack(phases), grads


def exact(case, seed):
    kind = case["kind"]
    B, H, T, D = (case[k] for k in "BHTD")
    if kind == "core":
        q, k, v, do = _qkv(case, seed)
        per_seq = [_core64(q[b].double(), k[b].double(), v[b].double(), do[b].double()) for b in range(B)]
        return tuple(torch.stack([r[i] for r in per_seq]) for i in range(5))
    if kind == "probs":
        st = prepare(case, seed)
        per_seq = [_core64(*(st[n][b].double() for n in ("q", "k", "v", "do", "att"))) for b in range(B)]
        return tuple(torch.stack([r[i] for r in per_seq]) for i in (2, 3, 4))
    if kind == "layer":
        i = {n: t.double() for n, t in _layer_inputs(case, seed).items()}
        E = H * D
        mm = lambda a, b: torch.matmul(a, b.contiguous())
        qkv = (mm(i["x"], i["wa"].t()) + i["ba"]).view(B, T, 3 * E)
        do = mm(i["dy"], i["wp"]).view(B, T, E)
        o, d_qkv = torch.empty_like(do), torch.empty_like(qkv)
        for b in range(B):
            h = lambda t, c: _heads(t[b:b + 1], c, H, D)[0].contiguous()
            r = _core64(h(qkv, 0), h(qkv, 1), h(qkv, 2), h(do, 0))
            _heads(o[b:b + 1], 0, H, D)[0].copy_(r[0])
            for c in range(3):
                _heads(d_qkv[b:b + 1], c, H, D)[0].copy_(r[2 + c])
        o, d_qkv = o.view(B * T, E), d_qkv.view(B * T, 3 * E)
        return (mm(o, i["wp"].t()) + i["bp"], mm(d_qkv, i["wa"]), mm(d_qkv.t(), i["x"]), d_qkv.sum(0),
                mm(i["dy"].t(), o), i["dy"].sum(0))
    if kind == "decode":
        st = prepare(case, seed)
        o = torch.empty(B, H, D, dtype=torch.float64, device=_dev())
        for b in range(B):
            s = torch.matmul(st["k"][b].double(), st["q"][b].double()[:, :, None])[..., 0] / math.sqrt(D)
            o[b] = torch.matmul(torch.softmax(s, -1)[:, None, :], st["v"][b].double())[:, 0]
        return o
    g, w, x = _wave_inputs(case, seed)
    if kind == "wave":
        dy = _normal(g, B, T, H * D, sd=(B * T) ** -0.5)
        out, _, _, gr = _wave64(w, x, dy)
        return (out, *gr)
    n = torch.nn.functional.softplus(w[0].double())
    if kind == "wave_prefill":
        out, vals, phi, _ = _wave64(w, x, content=False)
        a = n[None, :, None] * phi
        return out, torch.stack((torch.cos(a), torch.sin(a)), -1), phi, _bucket(phi), vals
    phase, values = _wave_cache_entries(case, g, w[0])
    hraw, pw, pb, vw, vb, ow, ob = (t.double() for t in w)
    E, xd = H * D, x.double()
    rs = torch.matmul(xd, pw[:, :2].reshape(H * 2, E).t().contiguous()).view(B, H, 2) + pb[:, :2]
    phi = torch.atan2(rs[..., 1], rs[..., 0])
    val = torch.matmul(xd.view(B, H, 1, D), vw.transpose(1, 2).contiguous())[:, :, 0] + vb
    bk, near_bk = _bucket(phi), _bucket(phase)
    see = torch.remainder(near_bk - bk[..., None] + 1, 8) <= 2
    see[:, :, T - 1] = True  # the previous position always counts
    s = torch.cos(n[None, :, None] * (phi[..., None] - phase.double())).masked_fill(~see, -math.inf)
    s = torch.cat((s, torch.ones(B, H, 1, dtype=torch.float64, device=s.device)), -1)
    p = torch.softmax(s, -1)
    merged = torch.empty(B, H, D, dtype=torch.float64, device=s.device)
    for b in range(B):
        merged[b] = torch.matmul(p[b, :, None, :T], values[b].double())[:, 0]
    merged += p[..., T:] * val
    out = torch.matmul(merged.view(B, E), ow.t().contiguous()) + ob
    a = n[None, :] * phi
    return out, torch.stack((torch.cos(a), torch.sin(a)), -1), phi, bk, val


def tolerance(case):
    """About four times the difference measured between two orders of the same
    float32 sums.  The wave kinds' gradients pass through atan2, which divides
    the rounding of a projection by its distance from the origin."""
    if case["kind"] in ("wave", "wave_prefill"):
        return {"rel": 2e-4}
    return {"rel": {"core": 6e-6, "probs": 2e-6, "layer": 8e-6, "decode": 2e-6, "wave_decode": 2e-5}[case["kind"]]}
