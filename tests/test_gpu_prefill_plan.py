"""GPU parity of the prefill GEMM on shapes whose plan splits k at each tile height, and of a call done in column
windows.

Bars as for the other prefill GEMM tests (fp32 torch product of the same fp16 operands, rotation and svh in fp32)."""
import math

import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pk():
    return load_package()


def _had128(x):
    h = torch.ones(1, 1, device=x.device)
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (x.reshape(-1, 128) @ (h / math.sqrt(128.0))).reshape(x.shape)


def _operands(rows, k, n):
    g = torch.Generator(device="cuda").manual_seed(rows + k + n)
    return ((torch.randn((rows, k), device="cuda", generator=g) * 0.5).half(),
            (torch.randn((n, k), device="cuda", generator=g) / math.sqrt(k)).half(),
            (torch.randn(n, device="cuda", generator=g) * 0.1).half(),
            torch.randn(n, device="cuda", generator=g) * 0.1)


# shapes that split k, at tile heights of 256, 192 and 128 rows when this was written (the plan may be fitted anew): even
# and ragged splits, ragged rows and columns
@pytest.mark.parametrize("rows,k,n", [(777, 17408, 5120), (1536, 17408, 5120), (3000, 8192, 1024), (1000, 5120, 1152),
                                      (641, 5184, 640)])
def test_prefill_matmul_split_plans(pk, rows, k, n):
    nbytes = pk._capi.lib().exl3_prefill_matmul_workspace_bytes(rows, k, n)
    assert nbytes > 0 and nbytes % (rows * n * 4) == 0
    xh, wt, svh, bias = _operands(rows, k, n)
    for dt, bar in ((torch.float16, 2e-3), (torch.float32, 2e-3)):
        b = bias.to(dt)
        y = pk.kernels.prefill_matmul(xh, wt, svh, b, torch.empty((rows, n), dtype=dt, device="cuda"))
        ref = (_had128(xh.float() @ wt.float().t()) * svh.float()).to(dt).float() + b.float()
        assert ((y.float() - ref).abs().max() / ref.abs().max()).item() < bar
        assert torch.equal(y, pk.kernels.prefill_matmul(xh, wt, svh, b, torch.empty_like(y)))


def test_prefill_matmul_windows_of_a_split_call(pk):
    """Windows of a call whose plan splits k give the call's bits, also where a window alone would split otherwise."""
    rows, k, n = 700, 8192, 1024
    lib = pk._capi.lib()
    assert lib.exl3_prefill_matmul_workspace_bytes(rows, k, n) // (rows * n * 4) != \
        lib.exl3_prefill_matmul_workspace_bytes(rows, k, 256) // (rows * 256 * 4)
    xh, wt, svh, _ = _operands(rows, k, n)
    whole = pk.kernels.prefill_matmul(xh, wt, svh, None, torch.empty((rows, n), device="cuda"))
    parts = torch.empty((rows, n), device="cuda")
    for c in range(0, n, 256):
        pk.kernels.prefill_matmul(xh, wt[c:c + 256], svh[c:c + 256], None, parts[:, c:c + 256], n_call=n)
    assert torch.equal(whole, parts)
