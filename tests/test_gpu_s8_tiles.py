"""gemm_s8 and gemm_q8y on each tile of the whole-K kernel (MI355X only): ragged rows and columns, K tails of 16 .. 112
values, K below one group, int8 -128. The int32 sum is exact and each of the two float32 products rounds once, so the
results equal torch's float32 products of the exact sum bit for bit."""
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


# t, n, k: 32, 64, 96, 128 x 128 and 128 x 256 tiles; full rounds and a rest; one row; K under a group; parts of the rest's
# tiles wholly past T (sub-tiles of 128 x 256, halves of 256 x 256); 64, 96 and 128 x 128 tiles of which a block takes
# several in turn (test_launch_rules.py holds the plan to these)
SHAPES = [(65, 2560, 400), (33, 130, 144), (511, 2560, 1040), (640, 2574, 272), (1024, 2560, 1136), (1500, 2560, 528),
          (2100, 2560, 256), (1024, 7168, 1024), (4096, 2560, 1152), (1, 34, 128), (70, 300, 112), (300, 514, 16),
          (3872, 2560, 2560), (3104, 2574, 2560), (3104, 7168, 128), (65, 2560, 2576), (90, 2574, 1296), (257, 21808, 400),
          (6494, 1330, 1792), (8221, 784, 272)]


@pytest.mark.parametrize("t,n,k", SHAPES)
def test_whole_k_tiles(sm, t, n, k):
    print("[case] s8 tile", t, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(t + n + k)
    wq = torch.randint(-128, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    xq = torch.randint(-128, 128, (t, k), generator=g, device="cuda", dtype=torch.int8)
    sx = torch.rand(t, generator=g, device="cuda") * 1e-3
    sw = torch.rand(n, generator=g, device="cuda") * 1e-3
    s = (xq.double() @ wq.double().T).float()  # exact, below 2^24 or rounded to float32 once, as the kernel's conversion
    ref = (s * sx[:, None]) * sw[None, :]
    assert torch.equal(sm.gemm_s8(xq, sx, wq, sw), ref)
    assert torch.equal(sm.gemm_s8(xq, sx, wq, sw, y_dtype=torch.float16), ref.half())
    refy = (s * sw[None, :]) * sx[:, None]
    assert torch.equal(sm.gemm_q8y(xq, sx, wq, sw), refy)
    base = torch.randn(t, n + 6, generator=g, device="cuda")
    y = base.clone()
    sm.gemm_q8y(xq, sx, wq, sw, y=y[:, :n], epilogue=sm.ADD)
    assert torch.equal(y[:, :n], base[:, :n] + refy) and torch.equal(y[:, n:], base[:, n:])
    if n % 128 == 0:
        h = sm.gemm_q8y(xq, sx, wq, sw, epilogue=sm.SWIGLU)
        z = refy.view(t, n // 128, 2, 64)
        gate, up = z[:, :, 0, :].reshape(t, n // 2).double(), z[:, :, 1, :].reshape(t, n // 2).double()
        want = gate / (1 + torch.exp(-gate)) * up  # the silu polynomial is within a few ulp
        assert ((h.double() - want).abs() <= 1e-6 * want.abs() + 1e-30).all()


# t, n, k, ld_y: whole and ragged tiles of each kind with padded Y rows; a row stride of 2^20, past which the stores of an
# edge tile go by 64-bit addresses (a T of one edge tile: Y is a view of t 2^20 values)
@pytest.mark.parametrize("t,n,k,ld", [(65, 2560, 2576, 2564), (640, 2574, 272, 2580), (1024, 2560, 1136, 2562),
                                      (1500, 2560, 528, 2568), (2100, 2560, 256, 2576), (33, 130, 144, 1 << 20),
                                      (45, 258, 1040, (1 << 20) + 2)])
@pytest.mark.parametrize("dt", ["float32", "float16"])
def test_padded_y(sm, t, n, k, ld, dt):
    """gemm_s8 into rows longer than N: the values of the product, and nothing between the rows written."""
    print("[case] s8 padded y", t, n, k, ld, dt, flush=True)
    dt = getattr(torch, dt)
    g = torch.Generator(device="cuda").manual_seed(t + n + k)
    wq = torch.randint(-128, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    xq = torch.randint(-128, 128, (t, k), generator=g, device="cuda", dtype=torch.int8)
    sx = torch.rand(t, generator=g, device="cuda") * 1e-3
    sw = torch.rand(n, generator=g, device="cuda") * 1e-3
    ref = ((xq.double() @ wq.double().T).float() * sx[:, None]) * sw[None, :]
    y = torch.full((t, ld), 7.0, device="cuda", dtype=dt)
    torch.cuda.synchronize()
    rc = sm.library().sepal_hip_gemm_s8(xq.data_ptr(), k, sx.data_ptr(), wq.data_ptr(), k, sw.data_ptr(), y.data_ptr(),
                                        sm.F32 if dt == torch.float32 else sm.F16, ld, t, n, k, None)
    assert rc == sm.OK
    torch.cuda.synchronize()
    assert torch.equal(y[:, :n], ref.to(dt)) and (y[:, n:] == 7.0).all()
