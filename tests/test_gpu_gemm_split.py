"""The projections' bf16-matrix-core GEMMs (csrc/gemm_split.hip, products of at
least 2^24 multiply-adds, weight gradients 2^29) against 64-bit sums: partial tiles, k remainders,
unaligned rows, split-K weight gradients, infinities and NaN.

Bound per element, with S = sum_k |a_k b_k|: the three dropped partial products
are below 1.001 x 2^-24 S, and each of the K/16 + 4 additions of a sum no larger
than S rounds by at most 2^-23 S (twice the fp32 unit roundoff, whichever way the
matrix core rounds)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available()
    return torch, torch.device("cuda:0")


def _check(name, got, a, b, extra=0.0, adds=0):
    """got against a @ b (+ extra) within the bound of the module docstring; adds: further fp32 additions."""
    import torch
    ref = a.double() @ b.double() + extra
    s = a.double().abs() @ b.double().abs() + (extra.abs() if torch.is_tensor(extra) else extra)
    bound = 2.0 ** -23 * (0.51 + a.shape[1] / 16 + 4 + adds) * s
    bad = (got.double() - ref).abs() > bound
    assert not bool(bad.any()), f"{name}: {int(bad.sum())} elements past the bound"
    print(f"  {name} rel {float((got.double() - ref).norm() / ref.norm()):.2e}", flush=True)


# (M, N, K): whole tiles, one row / column past them, 64-column and few-column
# outputs, odd k (unaligned rows), a k remainder of 4, few rows (mostly 64 x 64
# tiles; every other instance: INSTANCES)
SHAPES = [(512, 256, 256), (513, 257, 260), (129, 1025, 132), (4100, 64, 64), (700, 36, 1000), (301, 203, 333),
          (33, 768, 768), (2048, 130, 70), (4100, 513, 260), (8200, 64, 1028)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("pad", [0, 1])
def test_linear_pair_within_fp32_bound(pkg, torch_dev, M, N, K, pad):
    torch, dev = torch_dev
    print(f"gemm split M{M} N{N} K{K} pad{pad}", flush=True)
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    # rows of very different sizes: each output row keeps its own precision
    x = (rnd(M, K) * 10.0 ** torch.linspace(-8, 8, M, device=dev)[:, None])
    x = torch.nn.functional.pad(x, (0, pad))[:, :K]   # pad: a row stride that is no multiple of four
    w, b, dy = rnd(N, K), rnd(N), torch.nn.functional.pad(rnd(M, N), (0, pad))[:, :N]
    _check("y", pkg.linear_fwd(x, w, b), x, w.t().contiguous(), b.double()[None, :], adds=1)
    _check("dx", pkg.linear_bwd_dx(dy, w), dy, w)
    dw, db = pkg.linear_bwd_dw(dy, x)
    _check("dw", dw, dy.t().contiguous(), x, adds=32)
    _check("db", db[:, None], dy.t().contiguous(), torch.ones(M, 1, device=dev), adds=M)


# One shape for every instance that a call can reach: (entry, M, N, K, tile rows, tile
# columns, 128-bit loads, split-K).  Rows, columns and k just past whole tiles and stages.
INSTANCES = [("y", 6001, 517, 36, 128, 128, True, False), ("y", 6001, 517, 133, 128, 128, False, False),
             ("y", 8193, 129, 36, 128, 64, True, False), ("y", 8193, 129, 133, 128, 64, False, False),
             ("y", 6001, 129, 36, 64, 128, True, False), ("y", 6001, 129, 133, 64, 128, False, False),
             ("y", 257, 129, 516, 64, 64, True, False), ("y", 257, 257, 261, 64, 64, False, False),
             ("dx", 4097, 68, 516, 128, 128, True, False), ("dx", 12289, 65, 132, 128, 128, False, False),
             ("dx", 6001, 68, 260, 128, 64, True, False), ("dx", 8193, 65, 133, 128, 64, False, False),
             ("dx", 6001, 68, 132, 64, 128, True, False), ("dx", 6001, 65, 133, 64, 128, False, False),
             ("dx", 257, 260, 260, 64, 64, True, False), ("dx", 257, 129, 517, 64, 64, False, False),
             ("dw", 4097, 516, 516, 128, 128, True, True), ("dw", 4097, 517, 516, 128, 128, False, True),
             ("dw", 4097, 516, 260, 128, 64, True, True), ("dw", 4097, 517, 260, 128, 64, False, True),
             ("dw", 2049, 516, 516, 64, 128, True, True), ("dw", 4097, 257, 517, 64, 128, False, True),
             ("dw", 16001, 192, 192, 64, 64, True, True), ("dw", 300, 1028, 2052, 128, 128, True, False),
             ("dw", 300, 1028, 2049, 128, 128, False, False), ("dw", 513, 1540, 772, 64, 128, True, False),
             ("dw", 513, 1540, 773, 64, 128, False, False)]


@pytest.mark.parametrize("entry,M,N,K,bm,bn,vec,partial", INSTANCES)
def test_every_instance(pkg, torch_dev, entry, M, N, K, bm, bn, vec, partial):
    """Each instance of the kernel at partial tiles and a k remainder, and that it is the one that
    ran; split-K sums repeat bit for bit."""
    from torch.profiler import ProfilerActivity, profile
    torch, dev = torch_dev
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w, b, dy = rnd(M, K), rnd(N, K), rnd(N), rnd(M, N)
    call = {"y": lambda: pkg.linear_fwd(x, w, b), "dx": lambda: pkg.linear_bwd_dx(dy, w),
            "dw": lambda: pkg.linear_bwd_dw(dy, x)}[entry]
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    ran = [e.name for e in prof.events() if "gemm_split_kernel" in e.name]
    kc = {"y": "true, true", "dx": "true, false", "dw": "false, false"}[entry]
    assert len(ran) == 1 and f"gemm_split_kernel<{bm}, {bn}, " in ran[0], ran
    assert f", {kc}, {str(vec).lower()}, {str(partial).lower()}>" in ran[0], ran
    if entry == "y":
        _check("y", out, x, w.t().contiguous(), b.double()[None, :], adds=1)
    elif entry == "dx":
        _check("dx", out, dy, w)
    else:
        _check("dw", out[0], dy.t().contiguous(), x, adds=32)
        _check("db", out[1][:, None], dy.t().contiguous(), torch.ones(M, 1, device=dev), adds=M)
        again = call()
        assert torch.equal(out[0], again[0]) and torch.equal(out[1], again[1])


def beside_a_step(g, kind, *shape):
    """Numbers where a three-part split does worst: just below a bf16 step (cut off, all parts
    of a product lose in one direction) or just below half a step, and the remainder below half
    a step again (rounded, all remainders are largest)."""
    import torch
    r = lambda lo, hi: torch.randint(lo, hi, shape, generator=g, device=g.device).float()
    x = 1 + r(1, 9) * 2.0 ** -7 - r(1, 5) * 2.0 ** -23
    if kind == "half":
        x = x + 2.0 ** -8 - 2.0 ** -16 + 2.0 ** -17
    return x * r(-2, 3).exp2() * (r(0, 2) * 2 - 1 if kind == "signed" else 1)


def fma_chain(a, b):
    """a @ b as fp32 fused multiply-adds in order (a product of two floats is exact in 64 bits)."""
    import torch
    acc = torch.zeros(a.shape[0], b.shape[1], device=a.device)
    for k in range(a.shape[1]):
        acc = (acc.double() + a[:, k, None].double() * b[None, k].double()).float()
    return acc


@pytest.mark.parametrize("kind", ["step", "signed", "half"])
@pytest.mark.parametrize("K", [32, 64, 128, 768])
def test_error_no_larger_than_fp32_sums(pkg, torch_dev, kind, K):
    """The 2-norm error of each product is no larger than that of fp32 sums of the same length."""
    torch, dev = torch_dev
    g = torch.Generator(device=dev)
    g.manual_seed(K)
    M = max(1024, 2 ** 24 // (512 * K))
    a, w = beside_a_step(g, kind, M, K), beside_a_step(g, kind, 512, K)
    D = max(K, 128) * 16                       # positions of the weight gradient, 2^29 multiply-adds or more
    dy, x = beside_a_step(g, kind, D, 512), beside_a_step(g, kind, D, -(-2 ** 20 // D))
    for name, got, p, q in (("y", pkg.linear_fwd(a, w), a, w.t().contiguous()),
                            ("dx", pkg.linear_bwd_dx(a, w.t().contiguous()), a, w.t().contiguous()),
                            ("dw", pkg.linear_bwd_dw(dy, x)[0], dy.t().contiguous(), x)):
        ref = p.double() @ q.double()
        e, e32 = ((t.double() - ref).norm() / ref.norm() for t in (got, fma_chain(p, q)))
        print(f"  {name} {kind} K {K}: {float(e):.2e}, fp32 sums {float(e32):.2e}", flush=True)
        assert e <= e32


@pytest.mark.parametrize("M,N,K", [(2049, 516, 520), (2050, 1024, 260), (2051, 768, 512), (4099, 64, 2052)])
def test_weight_gradient_of_any_number_of_positions(pkg, torch_dev, M, N, K):
    """Positions that are no multiple of four: the 128-bit loads of both operands stop at the last
    one, one k at a time, whatever lies behind it (NaN, as below)."""
    torch, dev = torch_dev
    bufs = [torch.full(((1 << 29) + (1 << 20),), float("nan"), device=dev) for _ in range(2)]
    dy, x = bufs[0][:M * N].view(M, N), bufs[1][:M * K].view(M, K)
    dy.copy_(torch.randn(M, N, device=dev))
    x.copy_(torch.randn(M, K, device=dev))
    dw, db = pkg.linear_bwd_dw(dy, x)
    _check("dw", dw, dy.t().contiguous(), x.clone(), adds=32)
    _check("db", db[:, None], dy.t().contiguous(), torch.ones(M, 1, device=dev), adds=M)


def test_odd_positions_keep_the_weight_gradients_pace(pkg, torch_dev):
    """4001 positions against 4004: at most 1.3 times the time (1.0 was measured; with one load per
    element 1.6)."""
    torch, dev = torch_dev
    x, dy = torch.randn(4004, 576, device=dev), torch.randn(4004, 1728, device=dev)
    even = gpu_ms(torch, lambda: pkg.linear_bwd_dw(dy, x), passes=20)
    odd = gpu_ms(torch, lambda: pkg.linear_bwd_dw(dy[:4001], x[:4001]), passes=20)
    print(f"  4004: {even:.4f} ms, 4001: {odd:.4f}", flush=True)
    assert odd < 1.3 * even


@pytest.mark.parametrize("M,N,K", [(700, 36, 1000), (4096, 68, 260)])
def test_k_remainder_reads_nothing_past_the_operand(pkg, torch_dev, M, N, K):
    """A last k stage of four rows: the piece past them reads as zero, wherever the memory
    after the operand lies.  All of it up to 2 GiB on (the lane offset that marks the piece)
    holds NaN, which a stray read would carry into the sums."""
    torch, dev = torch_dev
    buf = torch.full(((1 << 29) + (1 << 20),), float("nan"), device=dev)
    w = buf[:N * K].view(N, K)             # dx sums over its rows
    w.copy_(torch.randn(N, K, device=dev))
    dy = torch.randn(M, N, device=dev)
    _check("dx", pkg.linear_bwd_dx(dy, w), dy, w.clone())


def fp32_ref(a, b):
    """What the formula gives where an operand is not finite: the sum of the products in order."""
    import torch
    acc = torch.zeros(a.shape[0], b.shape[1], device=a.device, dtype=torch.float64)
    for k in range(a.shape[1]):
        acc += a[:, k, None].double() * b[None, k].double()
    return acc.float()


def same_where_not_finite(name, got, a, b, extra=None):
    """Infinities and NaN as the formula gives them, the rest within the bound."""
    import torch
    want = fp32_ref(a, b)
    odd = ~torch.isfinite(want)
    assert bool(odd.any()) and bool((~odd).any()), name
    assert torch.equal(torch.isnan(got), torch.isnan(want)), name
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf]), name
    z = lambda t: torch.where(torch.isfinite(t), t, torch.zeros_like(t)).double()
    S = z(a).abs() @ z(b).abs()
    bad = (got.double() - want.double()).abs() > 2.0 ** -23 * (a.shape[1] + 40) * S
    assert not bool((bad & ~odd).any()), name


# (M, N, K): weight gradients and products with whole and partial tiles; k splits of the weight gradient
@pytest.mark.parametrize("M,N,K", [(2049, 516, 520), (2050, 513, 521)])
def test_operands_that_are_not_finite(pkg, torch_dev, M, N, K):
    """dX, split-K dW with db, y: each output sees the infinities and NaN of its own row and column
    only, and numbers that round to a bf16 infinity stay what they are."""
    torch, dev = torch_dev
    g = torch.Generator(device=dev)
    g.manual_seed(M)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    inf, nan = float("inf"), float("nan")
    x, w, dy = rnd(M, K), rnd(N, K), rnd(M, N)
    x[3, 7], x[M - 1, 9], x[8, K - 1], x[70, 0] = inf, -inf, nan, 3.3999e38
    w[N - 1, 5], w[1, 3] = inf, nan
    w[:, 0] = w[:, 0].abs() * 0.1 * 2.0 ** -40
    dy[70] = dy[70].clamp(-0.9, 0.9)       # times x[70, 0]: no overflow, which 64 bits would not show
    dy[5, 1], dy[M - 2, N - 1], dy[64, 2] = nan, inf, -inf
    same_where_not_finite("y", pkg.linear_fwd(x, w), x, w.t().contiguous())
    same_where_not_finite("dx", pkg.linear_bwd_dx(dy, w), dy, w)
    dw, db = pkg.linear_bwd_dw(dy, x)
    same_where_not_finite("dw", dw, dy.t().contiguous(), x)
    want = fp32_ref(dy.t().contiguous(), torch.ones(M, 1, device=dev))[:, 0]
    assert torch.equal(torch.isnan(db), torch.isnan(want)) and torch.equal(db[torch.isinf(want)], want[torch.isinf(want)])


def gpu_ms(torch, call, passes=5):
    call()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    a.record()
    for _ in range(passes):
        call()
    b.record()
    torch.cuda.synchronize()
    return a.elapsed_time(b) / passes


def test_nan_does_not_slow_a_product_down_without_bound(pkg, torch_dev):
    """All-NaN operands and one NaN: at most 12 times the finite call (5 to 7 were measured; summed
    element by element it was 87)."""
    torch, dev = torch_dev
    M, N, K = 4096, 768, 768
    x, w, dy = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev), torch.randn(M, N, device=dev)
    bad = torch.full_like(x, float("nan"))
    one = w.clone()
    one[5, 5] = float("nan")
    for name, call in (("y", lambda a, b: pkg.linear_fwd(a, b)), ("dx", lambda a, b: pkg.linear_bwd_dx(dy, b)),
                       ("dw", lambda a, b: pkg.linear_bwd_dw(dy, a))):
        base = gpu_ms(torch, lambda: call(x, w))
        t = [gpu_ms(torch, lambda: call(bad, torch.full_like(w, float("nan")))), gpu_ms(torch, lambda: call(x, one))]
        print(f"  {name}: {base:.4f} ms, all NaN {t[0]:.4f}, one NaN in w {t[1]:.4f}", flush=True)
        assert max(t) < 12 * base


def test_infinities_and_nan_reach_the_outputs_they_should(pkg, torch_dev):
    torch, dev = torch_dev
    M, N, K = 300, 256, 256
    x, w = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev)
    w[:, 7] = w[:, 7].abs() + 0.5
    w[:, 9] = 1.0                       # parts below the first are zero: infinity times them
    x[3, 7], x[5, 9], x[8, 7], x[10, 1] = float("inf"), float("-inf"), float("nan"), 3.0e38
    x[10, 2], w[:, 1], w[:, 2] = 3.0e38, 2.0, 2.0   # overflows
    y = pkg.linear_fwd(x, w)
    assert bool((y[3] == float("inf")).all()) and bool((y[5] == float("-inf")).all())
    assert bool(torch.isnan(y[8]).all()) and bool((y[10] == float("inf")).all())
    keep = torch.ones(M, dtype=torch.bool, device=dev)
    keep[[3, 5, 8, 10]] = False
    _check("finite rows", y[keep], x[keep], w.t().contiguous())
