"""GPU parity of the GEMV with the bf16 input rotation inside the launch: the values of rot followed by the GEMV, bit for
bit."""
import importlib

import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pk():
    return load_package()


# one row with and without a 16-lane group per block of the split (17,408: without), ragged splits, one bit width and
# mixed ones, the layouts' register limits (K = 6) and the largest K
@pytest.mark.parametrize("k,ns,Ks,cb", [(5120, [6144, 1024, 1024], 6, 0), (6144, [5120], 8, 0), (17408, [5120], 3, 1),
                                        (128, [128], 1, 0), (2048, [640, 128], [5, 2], 2), (768, [128], 7, 0),
                                        (5120, [1024, 256, 256], [4, 6, 8], 0)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_gemv_rotate_bf16_bitwise(pk, k, ns, Ks, cb, out_dtype):
    g = torch.Generator(device="cuda").manual_seed(k + sum(ns))
    each = Ks if isinstance(Ks, list) else [Ks] * len(ns)
    trs = [torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device="cuda", generator=g)
           for n, K in zip(ns, each)]
    half = lambda *s: torch.randn(s, device="cuda", generator=g).half()
    svh, suh, bias = half(sum(ns)) / k ** 0.5, half(len(ns), k), half(sum(ns)).to(out_dtype)
    for rows in (1, 2, 8, 16):
        plan = pk.kernels.TrellisGemvPlan(k, ns, Ks, cb, svh, rows, out_dtype)
        x = (2 * half(rows, k)).bfloat16()
        x[0, :8] = torch.tensor([0.0, -0.0, 1e-40, 3e4, -3e4, 1e-8, 1.0, -1.0], device="cuda").bfloat16()
        assert torch.equal(plan.rotate_bf16(x, suh, trs, bias=bias), plan(pk.kernels.rot(x, suh), trs, bias=bias)), rows


def test_bf16_linear_is_one_launch(pk, monkeypatch):
    syn = importlib.import_module(pk.__name__ + ".synthetic")
    lin_mod = importlib.import_module(pk.__name__ + ".linear")
    g = torch.Generator(device="cuda").manual_seed(1)
    lin = syn.random_exl3_linear(512, 256, 4, 0, g, "cuda")
    x = torch.randn(3, 512, device="cuda", generator=g).bfloat16()
    want = lin.gemv_rotated(pk.kernels.rot(x, lin.rot_suh), torch.bfloat16)
    with monkeypatch.context() as mp:
        mp.setattr(lin_mod, "rot", None)
        assert torch.equal(lin(x), want)
    lin.arm_residual(torch.zeros(3, 256, dtype=torch.float16, device="cuda"))
    with pytest.raises(ValueError):          # an fp16 epilogue armed for a bf16 call is refused
        lin(x)


@pytest.mark.parametrize("rows,inside", [(1, True), (4, True), (8, False)])
def test_linear_on_both_sides_of_the_rotation_rule(pk, rows, inside):
    """17408 -> 7680: one launch and two launches give rot followed by the GEMV bit for bit, armed or not."""
    syn = importlib.import_module(pk.__name__ + ".synthetic")
    g = torch.Generator(device="cuda").manual_seed(rows)
    lin = syn.random_exl3_linear(17408, 7680, 2, 0, g, "cuda")
    for dt in (torch.float16, torch.bfloat16):
        x = torch.randn(rows, 17408, device="cuda", generator=g).to(dt)
        assert lin._plan(rows, dt).rotates_inside == inside
        assert torch.equal(lin(x), lin.gemv_rotated(pk.kernels.rot(x, lin.rot_suh), dt))
    x, res = x.half(), torch.randn(rows, 7680, device="cuda", generator=g).half()
    y = lin(x)
    lin.arm_residual(res)
    assert torch.equal(lin(x), (y.float() + res.float()).half()) and lin.take_armed_output() is not None


@pytest.mark.parametrize("k,n,rows,inside", [(14592, 4736, 8, True), (5120, 15616, 8, True), (5120, 15744, 8, False),
                                             (2304, 36736, 8, False), (1664, 98432, 2, True), (1664, 98432, 4, False)])
def test_rotation_rule_by_elements_and_weights(pk, k, n, rows, inside):
    """Up to 4.25 M rotated elements or below 80 M weights the rotation is inside the launch; the bits are the same."""
    assert inside == (rows * k * n // 128 <= 4_250_000 or k * n < 80_000_000)
    syn = importlib.import_module(pk.__name__ + ".synthetic")
    g = torch.Generator(device="cuda").manual_seed(n)
    lin = syn.random_exl3_linear(k, n, 2, 0, g, "cuda")
    for dt in (torch.float16, torch.bfloat16):
        x = torch.randn(rows, k, device="cuda", generator=g).to(dt)
        assert lin._plan(rows, dt).rotates_inside == inside
        assert torch.equal(lin(x), lin.gemv_rotated(pk.kernels.rot(x, lin.rot_suh), dt))


@pytest.mark.parametrize("rows", [1, 3, 16])
def test_gemv_rotate_fp16_entry(pk, rows):
    """exl3_gemv_rotate takes fp16 input too (the package calls exl3_gemv_fused for it): the same bits."""
    k, ns, Ks = 1024, [256, 128], [4, 6]
    g = torch.Generator(device="cuda").manual_seed(rows)
    trs = [torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device="cuda", generator=g)
           for n, K in zip(ns, Ks)]
    half = lambda *s: torch.randn(s, device="cuda", generator=g).half()
    plan = pk.kernels.TrellisGemvPlan(k, ns, Ks, 0, half(sum(ns)) / k ** 0.5, rows, torch.float16)
    x, suh, c = half(rows, k), half(2, k), pk._capi
    y = plan._rotate_args(x, torch.float16, suh, trs, None, None)
    c.check(c.lib().exl3_gemv_rotate(c.ptr(x), c.DTYPE_CODE[x.dtype], c.ptr(suh), plan._tr_c, 2, plan._ns_c, plan._Ks_c, k,
                                     0, c.ptr(plan.svh), None, c.ptr(y), c.DTYPE_CODE[y.dtype], rows,
                                     c.ptr(plan.workspace), plan.workspace.numel(), c.stream_handle(x.device)),
            "exl3_gemv_rotate")
    assert torch.equal(y, plan.rotate(x, suh, trs))
