"""The attention forward on the bf16 matrix cores (attn_fwd_split.hip) against 64-bit
arithmetic, at the edges of its tiles: 32 keys, 128 queries a block, one kernel per head
dim class (32, 48, 64, 96, 128).

The bound, with u = 2^-24: a score is a sum of D exact-product terms in three-part form,
the dropped parts below 1.001 u of |q||k|, summed in fp32 in any order, so its error e is at
most (D + 8) u |q|.|k| scale; the exponent and exp2 add u (|s| + |m|) + 4u.  A row's
probabilities then move by P (e + mean e), its output by that times |v|, plus the
rounding of the sums over at most T keys in tiles of 32: (T / 32 + 40) u sum P |v|.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def exact(q, k, v, scale, adds=None, drop=None):
    """O, LSE and their bounds, in 64 bits; without key `drop`."""
    q, k, v = (x.double() for x in (q, k, v))
    T, D = q.shape[-2:]
    adds = T / 32 + 40 if adds is None else adds
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    e = (q.abs() @ k.abs().transpose(-1, -2).contiguous()) * scale * (D + 8) * U
    mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    if drop is not None:
        mask[:, drop] = True
    s = s.masked_fill(mask, -math.inf)
    lse = torch.logsumexp(s, -1, keepdim=True)
    p = torch.exp(s - lse)
    e = e + U * (s.abs().masked_fill(mask, 0) + s.amax(-1, keepdim=True).abs()) + 4 * U
    pe = p * e
    mean = pe.sum(-1, keepdim=True)
    vmag = v.abs()
    o_tol = pe @ vmag + (mean + adds * U) * (p @ vmag)
    return p @ v, lse[..., 0], o_tol, (mean + adds * U)[..., 0] + U * lse[..., 0].abs()


def check(o, lse, q, k, v, scale):
    want_o, want_l, tol_o, tol_l = exact(q, k, v, scale)
    assert ((o.double() - want_o).abs() <= tol_o).all()
    assert ((lse.double() - want_l).abs() <= tol_l).all()


def draw(B, H, T, D, seed, mixed=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    q, k, v = (torch.randn(B, H, T, D, device="cuda", generator=g) for _ in range(3))
    if mixed:  # rows from 2^-12 to 2^2 beside each other, and a common offset
        e = torch.randint(-12, 3, (3, B, H, T, 1), device="cuda", generator=g).float().exp2()
        q, k, v = q * e[0], k * e[1] + 0.5, v * e[2] + 3.0
    return q, k, v


@pytest.mark.parametrize("D", [4, 32, 33, 36, 48, 50, 64, 65, 96, 100, 127, 128])
@pytest.mark.parametrize("T", [513, 640, 671, 1000])
def test_tile_edges(pkg, T, D):
    q, k, v = draw(2, 17, T, D, T * 1000 + D, mixed=True)
    o, lse = pkg.attn_fwd(q, k, v)
    check(o, lse, q, k, v, 1 / math.sqrt(D))
    # the element loads (a base 4 bytes off) stage the same tiles: bit-identical
    parts = []
    for x in (q, k, v):
        buf = torch.empty(x.numel() + 4, device="cuda")
        parts.append(buf[1:1 + x.numel()].view_as(x).copy_(x))
    o2, lse2 = pkg.attn_fwd(*parts)
    assert torch.equal(o, o2) and torch.equal(lse, lse2)


@pytest.mark.parametrize("D,T,waves", [(68, 33, 2), (80, 64, 2), (80, 65, 2), (96, 127, 2), (96, 129, 2), (72, 256, 2),
                                       (80, 257, 4), (100, 33, 2), (128, 64, 2), (128, 65, 4), (128, 128, 4),
                                       (104, 129, 2), (128, 192, 2), (128, 193, 4)])
def test_short_rows_of_wide_heads(pkg, D, T, waves):
    """Blocks of two waves (two_waves): tile edges, the kept scores and the gradients from them;
    the same bits as blocks of four."""
    from torch.profiler import ProfilerActivity, profile
    q, k, v = draw(9, 32, T, D, T + D, mixed=True)
    o, lse = pkg.attn_fwd(q, k, v)
    torch.cuda.synchronize()
    sc = pkg.attn_scores_buffer(pkg.layout_of(q), torch.device("cuda:0"))
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        o2, lse2 = pkg.attn_fwd(q, k, v, scores=sc)
        torch.cuda.synchronize()
    ran = [e.name for e in prof.events() if "attn_fwd_split_kernel" in e.name]
    assert len(ran) == 1 and f", {waves}, true, true>" in ran[0], ran
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    check(o, lse, q, k, v, 1 / math.sqrt(D))
    do = draw(9, 32, T, D, 1)[0]
    whole = pkg.attn_bwd(q, k, v, o, do, lse, scores=sc)
    plain = pkg.attn_bwd(q, k, v, o, do, lse)
    for a, b in zip(whole, plain):
        assert (a - b).norm() <= 1e-5 * b.norm()
    # one load per element: always four waves
    parts = []
    for x in (q, k, v):
        buf = torch.empty(x.numel() + 4, device="cuda")
        parts.append(buf[1:1 + x.numel()].view_as(x).copy_(x))
    o3, lse3 = pkg.attn_fwd(*parts)
    assert torch.equal(o, o3) and torch.equal(lse, lse3)


def fp32_sums(q, k, v, scale):
    """O and LSE with every sum a chain of fp32 fused multiply-adds (exact in 64 bits, rounded)."""
    T, D = q.shape[-2:]
    s = torch.zeros(*q.shape[:-1], T, device=q.device)
    for d in range(D):
        s = (s.double() + q[..., d, None].double() * k[..., None, :, d].double()).float()
    s = (s * scale).masked_fill(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    m = s.amax(-1, keepdim=True)
    p = torch.exp(s - m)
    o, l = torch.zeros_like(q), torch.zeros_like(m)
    for j in range(T):
        o = (o.double() + p[..., j, None].double() * v[..., j, None, :].double()).float()
        l = l + p[..., j, None]
    return o / l, (m + torch.log(l))[..., 0]


@pytest.mark.parametrize("kind", ["step", "half"])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_error_no_larger_than_fp32_sums(pkg, D, kind):
    """Operands where a three-part split does worst (test_gpu_gemm_split.py): the 2-norm error of O
    and LSE is no larger than that of fp32 sums."""
    from test_gpu_gemm_split import beside_a_step
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    q, k, v = (beside_a_step(g, kind, 2, 17, 544, D) for _ in range(3))
    q = q * (torch.randint(0, 2, q.shape, generator=g, device="cuda").float() * 2 - 1)
    scale = 1 / math.sqrt(D)
    o, lse = pkg.attn_fwd(q, k, v)
    o32, lse32 = fp32_sums(q, k, v, scale)
    want_o, want_l, _, _ = exact(q, k, v, scale)
    for name, got, other, want in (("O", o, o32, want_o), ("LSE", lse, lse32, want_l)):
        e, e32 = ((t.double() - want).norm() / want.norm() for t in (got, other))
        print(f"  {name} {kind} D {D}: {float(e):.2e}, fp32 sums {float(e32):.2e}", flush=True)
        assert e <= e32


@pytest.mark.parametrize("D", [48, 64, 128])
def test_token_major_rows(pkg, D):
    """[B,T,H,D] memory (row stride H*D), as the layer holds it."""
    q, k, v = draw(2, 32, 777, D, D)
    qt, kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    o, lse = pkg.attn_fwd(q, k, v)
    ot, lset = pkg.attn_fwd(qt, kt, vt)
    assert torch.equal(o, ot) and torch.equal(lse, lset)


@pytest.mark.parametrize("D", [48, 128])
@pytest.mark.parametrize("over", [False, True])
def test_rows_two_gib_apart(pkg, D, over):
    """A head's rows up to and past 2 GiB: 32-bit or 64-bit offsets, the same results, kept
    scores and their backward included."""
    T = 1061
    st = ((2 ** 31 // 4) // (T + 32) & ~3) + (4 if over else -4)
    q, k, v = draw(1, 2, T, D, D)
    do = draw(1, 2, T, D, D + 1)[0]
    far = []
    for x in (q, k, v, do):
        f = torch.empty(T * st, device="cuda").as_strided((1, 2, T, D), (T * st, D, st, 1))
        far.append(f.copy_(x))
    out = []
    for a in ((q, k, v, do), far):
        L = pkg.layout_of(a[0])
        sc = pkg.attn_scores_buffer(L, torch.device("cuda:0"))
        assert sc is not None
        o = torch.empty_strided(a[0].shape, a[0].stride(), device="cuda")
        o, lse = pkg.attn_fwd(a[0], a[1], a[2], out=o, scores=sc)
        g = [torch.empty_strided(a[0].shape, a[0].stride(), device="cuda") for _ in range(3)]
        g = pkg.attn_bwd(a[0], a[1], a[2], o, a[3], lse, dq=g[0], dk=g[1], dv=g[2], scores=sc)
        out.append([x.contiguous() for x in (o, lse, *g)])
        del o, g, sc
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_rows_that_are_not_finite(pkg, D):
    """A row sees an infinity or NaN of the keys and values up to its own only.  Rows whose
    32-key tile holds one are summed again in fp32, key by key: at most T additions, so the
    bound has T u where it had (T / 32 + 40) u."""
    T, at, ch = 700, 333, 1
    q, k, v = draw(3, 32, T, D, 7)
    o, lse = pkg.attn_fwd(q, k, v)
    v2 = v.clone()
    v2[0, 0, at, ch] = math.inf
    k2 = k.clone()
    k2[0, 1, at, 0] = math.nan
    k2[0, 2, at, 0] = math.inf      # a score of -inf where q is negative there: weight 0
    o2, lse2 = pkg.attn_fwd(q, k2, v2)
    same = torch.ones_like(lse, dtype=torch.bool)
    same[0, :3, at // 32 * 32:] = False
    assert torch.equal(o[same], o2[same]) and torch.equal(lse[same], lse2[same])
    scale = 1 / math.sqrt(D)
    want, want_l, tol, tol_l = exact(q[0, :3], k[0, :3], v[0, :3], scale, adds=T)
    for h in range(3):  # the rows before it
        assert ((o2[0, h, :at].double() - want[h, :at]).abs() <= tol[h, :at]).all()
        assert ((lse2[0, h, :at].double() - want_l[h, :at]).abs() <= tol_l[h, :at]).all()
    assert (o2[0, 0, at:, ch] == math.inf).all()
    rest = [d for d in range(D) if d != ch]
    assert ((o2[0, 0].double() - want[0]).abs() <= tol[0])[:, rest].all()
    assert o2[0, 1, at:].isnan().all() and lse2[0, 1, at:].isnan().all()
    pos = torch.nonzero(q[0, 2, at:, 0] > 0)[:, 0] + at
    neg = torch.nonzero(q[0, 2, at:, 0] < 0)[:, 0] + at
    assert o2[0, 2, pos].isnan().all()
    want, want_l, tol, tol_l = exact(q[0, 2], k[0, 2], v[0, 2], scale, adds=T, drop=at)
    assert ((o2[0, 2].double() - want).abs() <= tol)[neg].all()
    assert ((lse2[0, 2].double() - want_l).abs() <= tol_l)[neg].all()


@pytest.mark.parametrize("D", [48, 64, 96, 128])
def test_kept_scores_that_are_not_finite(pkg, D):
    """The kept pair on the same data: the forward gives the same bits, and the backward that
    reads the scores the same infinities and NaN as the one that forms them; the rest agrees
    within 1e-4 of the largest value, the parity tests' tolerance."""
    T, at = 700, 333
    q, k, v = draw(3, 32, T, D, 11)
    do = draw(3, 32, T, D, 12)[0]
    v[0, 0, at, 1] = math.inf
    k[0, 1, at, 0] = math.nan
    k[0, 2, at, 0] = math.inf
    q[0, 3, at, 2] = -math.inf
    q[0, 4] = math.nan
    sc = pkg.attn_scores_buffer(pkg.layout_of(q), torch.device("cuda:0"))
    assert sc is not None
    o, lse = pkg.attn_fwd(q, k, v)
    o2, lse2 = pkg.attn_fwd(q, k, v, scores=sc)
    for a, b in ((o, o2), (lse, lse2)):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(nan=0.0), b.nan_to_num(nan=0.0))
    assert o2[0, 4].isnan().all() and o2[0, 3, at].isnan().all() and o2[0, 3, :at].isfinite().all()
    g = pkg.attn_bwd(q, k, v, o, do, lse)
    g2 = pkg.attn_bwd(q, k, v, o2, do, lse2, scores=sc)
    for name, a, b in zip(("dQ", "dK", "dV"), g, g2):
        assert torch.equal(a.isnan(), b.isnan()), name
        assert torch.equal(a.isinf(), b.isinf()), name
        both = a.isfinite()
        assert both[1:].all()
        assert (a - b)[both].abs().max() <= 1e-4 * a[both].abs().max(), name


def test_rows_that_are_not_finite_keep_their_pace(pkg):
    """All NaN, or one infinity or NaN that every row of a head meets: at most 16 times
    the finite forward (6.7 were measured; one row after another it was 270)."""
    from test_gpu_gemm_split import gpu_ms
    q, k, v = draw(8, 12, 1024, 64, 3)
    k1, v1 = k.clone(), v.clone()
    k1[:, :, 0, 0] = math.nan
    v1[:, :, 0, 0] = math.inf
    base = gpu_ms(torch, lambda: pkg.attn_fwd(q, k, v))
    for name, a in (("all NaN", (q, k, torch.full_like(v, math.nan))), ("NaN key", (q, k1, v)),
                    ("infinite value", (q, k, v1))):
        t = gpu_ms(torch, lambda: pkg.attn_fwd(*a))
        print(f"  {name}: {t:.3f} ms, finite {base:.3f}", flush=True)
        assert t < 16 * base
