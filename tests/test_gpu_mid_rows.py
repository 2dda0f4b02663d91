"""The multiplies of up to 64 rows (MI355X only): w8g with bf16 / binary16 X, which splits K over waves and blocks, and q8 in
both activation-scale modes, at the edges of the kernels' row tiles (16, 32, 48, 64), of their blocks of 2 to 8 weight
tiles (a last block with tiles missing), of the K-parts and of the waves (fewer groups than waves), with padded strides.

Reference: float64 of the dequantized operands. Bound: a float32 sum of K products and G group links is within
(K + G + 8) 2^-24 sum |x_k w_k| of it (each product and addition rounds once; the q8 sums of a group are exact); SwiGLU
adds |d silu(g) u| <= 1.1 |u| dg + |silu(g)| du and a few ulp of its own."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def sm():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import sepal_mlp
    sepal_mlp.library()
    return sepal_mlp


def _swiglu(z):
    t, n = z.shape
    z = z.view(t, n // 128, 2, 64)
    gate, up = z[:, :, 0, :], z[:, :, 1, :]
    return (gate.reshape(t, n // 2), up.reshape(t, n // 2))


def _check(y, ref, mag, u):
    """|y - ref| within u * mag of the sums, elementwise."""
    assert torch.isfinite(y).all()
    excess = (y.double() - ref).abs() - u * mag
    assert (excess <= 0).all(), excess.max().item()


def _check_swiglu(h, z, mag, u, type_eps):
    g, up = _swiglu(z)
    dg, du = _swiglu(u * mag)
    silu = g / (1 + torch.exp(-g))
    ref = silu * up
    bound = 1.1 * up.abs() * dg + silu.abs() * du + dg * du + 2.0**-20 * ref.abs() + type_eps * ref.abs() + 1e-7
    assert ((h.double() - ref).abs() <= bound).all()


SHAPES = [
    # t, n, k: one tile and one group; tiles short of a block; groups short of the waves; K-parts; a wide grid; NT 2 / 3 / 5
    (17, 16, 128), (20, 144, 128), (31, 48, 640), (32, 2560, 9728), (33, 80, 1152), (48, 1008, 512), (49, 128, 384),
    (63, 12288, 256), (64, 2576, 1280), (40, 20608, 256), (64, 256, 9728), (5, 640, 384), (16, 2048, 3200),
]


@pytest.mark.parametrize("t,n,k", SHAPES)
def test_up_to_64_rows(sm, t, n, k):
    print("[case] mid rows", t, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(1000 * t + n + k)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).half()
    x = torch.randn(t, k + 16, generator=g, device="cuda")[:, :k]
    u = (k + k // 128 + 8) * 2.0**-24
    q, s = sm.quantize_group_s8(w)
    wpad = torch.zeros(n, k + 32, dtype=torch.int8, device="cuda")
    wpad[:, :k] = q
    deq = (q.double().view(n, k // 128, 128) * s.double()[:, :, None]).view(n, k)
    for dt in (torch.bfloat16, torch.float16):
        xp = torch.zeros(t, k + 16, dtype=dt, device="cuda")
        xp[:, :k] = x.to(dt)
        xb = xp[:, :k]
        ref, mag = xb.double() @ deq.T, xb.double().abs() @ deq.abs().T
        y = torch.full((t, n + 4), 7.0, device="cuda")
        sm.gemm_w8g(xb, wpad[:, :k], s, y=y[:, :n])
        _check(y[:, :n], ref, mag, u)
        assert (y[:, n:] == 7.0).all()
        y0 = torch.randn(t, n, generator=g, device="cuda")
        ya = sm.gemm_w8g(xb, q, s, y=y0.clone(), epilogue=sm.ADD)
        _check(ya, ref + y0.double(), mag + y0.double().abs() + ref.abs(), u)
        if n % 128 == 0:
            for yt, eps in ((torch.float32, 0.0), (torch.float16, 2.0**-11), (torch.bfloat16, 2.0**-8)):
                _check_swiglu(sm.gemm_w8g(xb, q, s, epilogue=sm.SWIGLU, y_dtype=yt), ref, mag, u, eps)
    for block in (k, 128):
        xq, xs = sm.quantize_rows_s8(x.contiguous(), block=block)
        xd = (xq.double().view(t, k // block, block) * xs.double()[:, :, None]).view(t, k)
        ref, mag = xd @ deq.T, xd.abs() @ deq.abs().T
        _check(sm.gemm_q8(xq, xs, q, s, act_block=block), ref, mag, u)
        if n % 128 == 0:
            _check_swiglu(sm.gemm_q8(xq, xs, q, s, act_block=block, epilogue=sm.SWIGLU), ref, mag, u, 0.0)
        if n % 256 == 0:
            hq, hs = sm.gemm_q8_swiglu_quantize(xq, xs, q, s, act_block=block)
            h = sm.gemm_q8(xq, xs, q, s, act_block=block, epilogue=sm.SWIGLU)
            rq, rs = sm.quantize_rows_s8(h, block=128)
            assert torch.equal(hq, rq) and torch.equal(hs, rs)


@pytest.mark.parametrize("t", [17, 48, 64])
def test_rows_do_not_see_each_other(sm, t):
    """A row's bits depend on that row alone at one T; a row of infinities stays in its row; the second call repeats the
    first one's bits (the K-parts and waves are added in a fixed order)."""
    n, k = 2560, 2560
    g = torch.Generator(device="cuda").manual_seed(t)
    q, s = sm.quantize_group_s8((torch.randn(n, k, generator=g, device="cuda") * 0.02).half())
    x = torch.randn(t, k, generator=g, device="cuda").bfloat16()
    a = sm.gemm_w8g(x, q, s)
    assert torch.equal(a, sm.gemm_w8g(x, q, s))
    x2 = torch.randn(t, k, generator=g, device="cuda").bfloat16()
    x2[t // 2] = x[t // 2]
    x2[0] = float("inf")
    b = sm.gemm_w8g(x2, q, s)
    assert torch.equal(a[t // 2], b[t // 2])
    assert torch.isfinite(b[1:]).all() and not torch.isfinite(b[0]).any()


# t, n, k: one row; one tile and one group; tiles short of a block; K-parts; both sides of 24 rows and of N = 8192
@pytest.mark.parametrize("t,n,k", [(1, 16, 128), (5, 144, 384), (16, 2560, 9728), (17, 48, 640), (24, 2576, 1280),
                                   (24, 8176, 256), (24, 256, 9728), (25, 2560, 1152), (24, 8192, 512)])
def test_float32_x(sm, t, n, k):
    """A float32 X up to 24 rows as its hi and lo bf16 rows in one multiply: hi + lo is within 2^-17 of x."""
    print("[case] mid rows float32", t, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(t + n + k)
    q, s = sm.quantize_group_s8((torch.randn(n, k, generator=g, device="cuda") * 0.02).half())
    x = torch.randn(t, k + 4, generator=g, device="cuda")[:, :k]
    deq = (q.double().view(n, k // 128, 128) * s.double()[:, :, None]).view(n, k)
    ref, mag = x.double() @ deq.T, x.double().abs() @ deq.abs().T
    u = (2 * k + k // 128 + 16) * 2.0**-24 + 2.0**-17
    y = torch.full((t, n + 4), 7.0, device="cuda")
    sm.gemm_w8g(x, q, s, y=y[:, :n])
    _check(y[:, :n], ref, mag, u)
    assert (y[:, n:] == 7.0).all()
    first = y[:, :n].clone()
    sm.gemm_w8g(x, q, s, y=y[:, :n], epilogue=sm.ADD)
    _check(y[:, :n], 2 * ref, 2 * mag, u)
    assert torch.equal(sm.gemm_w8g(x, q, s), first)


@pytest.mark.parametrize("t,n", [(1, 128), (17, 128), (18, 384), (32, 4096), (32, 8064)])
def test_swiglu_of_exact_sums(sm, t, n):
    """One product a sum and weight scales of powers of two: gate and up are exact, so the default SwiGLU up to 32 rows with
    N < 8192 differs from the weight-streaming path's (config 1) only in its silu, which is the same function: equal
    bits, also where gate times up leaves float32 beside a vanishing silu."""
    print("[case] mid swiglu", t, n, flush=True)
    k = 128
    g = torch.Generator(device="cuda").manual_seed(t + n)
    w = torch.zeros(n, k, dtype=torch.int8, device="cuda")
    gate = (torch.arange(n, device="cuda") // 64) % 2 == 0
    w[gate, 0], w[~gate, 1] = 1, 1
    s = torch.exp2(torch.randint(-3, 3, (n, 1), generator=g, device="cuda").float())
    x = torch.zeros(t, k, device="cuda")
    x[:, 0] = torch.randn(t, generator=g, device="cuda") * 8
    x[:, 1] = torch.randn(t, generator=g, device="cuda")
    x[0, 0], x[0, 1] = -1e4, 3e37
    if t > 1:
        x[1, 0], x[1, 1] = -90.0, 1e37
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        y = sm.gemm_w8g(x.bfloat16(), w, s, epilogue=sm.SWIGLU, y_dtype=dt)
        assert not torch.isnan(y).any()
        assert torch.equal(y, sm.gemm_w8g(x.bfloat16(), w, s, epilogue=sm.SWIGLU, y_dtype=dt, config=1))
