"""GPU parity of the few-row prefill (exl3_prefill_rows: weights decoded into MFMA operands) against the CPU oracle.

Bars: an fp32 result differs from the fp64 oracle by fp32 accumulation alone (products of fp16 values are exact in
fp32), at most k * 2^-24 of the largest result (k <= 1088: 6.5e-5, bar 1e-4); fp16 and bf16 results add their
rounding, twice with a bias (2e-3, 1e-2: the bars of the other prefill forms)."""
import importlib

import numpy as np
import pytest

from conftest import load_package
from oracle import exl3_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BAR = {torch.float32: 1e-4, torch.float16: 2e-3, torch.bfloat16: 1e-2}


@pytest.fixture(scope="module")
def pk():
    return load_package()


def _case(k, n, K, cb, rows, seed):
    rng = np.random.default_rng(seed)
    tr = O.random_trellis(k, n, K, seed)
    svh = (rng.standard_normal(n) * 0.05).astype(np.float16)
    xh = rng.standard_normal((rows, k)).astype(np.float16)
    ref = O.gemv_ref(xh, O.reconstruct_inner(tr, k, n, K, cb), svh)
    return (*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (tr, svh, xh)), ref)


def _run(pk, tr, svh, xh, k, n, K, cb, dt, splits=0, bias=None):
    out = torch.full((xh.shape[0], n), float("nan"), dtype=dt, device="cuda")
    return pk.kernels.prefill_rows(xh, tr, k, n, K, cb, svh, bias, out, splits)


# every tile count (16, 32, 48, 64, 96, 128, 192, 256 rows) full and with one row more than the one before, several
# row blocks; splits: one (epilogue in the launch), uneven (7 steps over 2, 3), one step each, automatic
@pytest.mark.parametrize("rows", [1, 9, 16, 17, 33, 49, 64, 65, 97, 128, 129, 192, 193, 256, 257, 513])
@pytest.mark.parametrize("splits", [0, 1, 3, 7])
def test_prefill_rows_tile_and_split_edges(pk, rows, splits):
    k, n, K = 448, 256, 6
    tr, svh, xh, ref = _case(k, n, K, 0, rows, rows)
    y = _run(pk, tr, svh, xh, k, n, K, 0, torch.float32, splits)
    assert O.max_abs_rel(y.cpu().numpy(), ref) < BAR[torch.float32]
    assert torch.equal(y, _run(pk, tr, svh, xh, k, n, K, 0, torch.float32, splits))


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_prefill_rows_bitrates_codebooks(pk, K, cb):
    k, n = 1088, 384
    for rows, splits in ((40, 1), (150, 2)):
        tr, svh, xh, ref = _case(k, n, K, cb, rows, 10 * K + cb)
        y = _run(pk, tr, svh, xh, k, n, K, cb, torch.float32, splits)
        assert O.max_abs_rel(y.cpu().numpy(), ref) < BAR[torch.float32], (rows, splits)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("splits", [1, 4])
def test_prefill_rows_bias_and_dtypes(pk, dt, splits):
    """The bias is added after the rounding to the output type; both epilogues (in the launch, in the reduction)."""
    k, n, K, rows = 512, 256, 4, 77
    tr, svh, xh, ref = _case(k, n, K, 0, rows, 3)
    bias = torch.randn(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(dt)
    plain = _run(pk, tr, svh, xh, k, n, K, 0, dt, splits)
    y = _run(pk, tr, svh, xh, k, n, K, 0, dt, splits, bias)
    assert O.max_abs_rel(plain.float().cpu().numpy(), ref) < BAR[dt]
    assert torch.equal(y, (plain.float() + bias.float()).to(dt))


def test_prefill_rows_infinite_row_stays_alone(pk):
    k, n, K, rows = 256, 128, 5, 35
    tr, svh, xh, _ = _case(k, n, K, 0, rows, 8)
    y = _run(pk, tr, svh, xh, k, n, K, 0, torch.float32, 2)
    xh[34] = float("inf")
    yi = _run(pk, tr, svh, xh, k, n, K, 0, torch.float32, 2)
    assert torch.equal(yi[:34], y[:34]) and not torch.isfinite(yi[34]).any()


@pytest.mark.parametrize("rows,k,n", [(9, 256, 256), (640, 256, 256), (641, 256, 256), (1024, 512, 256), (1025, 512, 256)])
def test_prefill_auto_route(pk, rows, k, n):
    """prefill_gemm's "auto" gives the bits of the form its rule names, on both sides of the rule's edges."""
    K = 6
    tr, svh, xh, ref = _case(k, n, K, 0, rows, rows)
    y = pk.kernels.prefill_gemm(xh, tr, k, n, K, 0, svh, out_dtype=torch.float32)
    rows_form = pk.kernels.takes_rows_form(rows, k, n, K)
    assert rows_form == (rows <= 640 or (rows <= 1024 and k >= 2 * n))
    want = _run(pk, tr, svh, xh, k, n, K, 0, torch.float32) if rows_form else \
        pk.kernels.prefill_gemm(xh, tr, k, n, K, 0, svh, out_dtype=torch.float32, path="matmul")
    assert torch.equal(y, want) and O.max_abs_rel(y.cpu().numpy(), ref) < BAR[torch.float32]


# three members of different widths and bits; a strided input; both prefill forms (k = 1024: rows form up to 640 rows)
@pytest.mark.parametrize("rows", [9, 33, 700])
@pytest.mark.parametrize("dt", ["float16", "bfloat16", "float32"])
def test_group_prefill_equals_its_members(pk, rows, dt):
    syn = importlib.import_module(pk.__name__ + ".synthetic")
    lin_mod = importlib.import_module(pk.__name__ + ".linear")
    g = torch.Generator(device="cuda").manual_seed(rows)
    lins = [syn.random_exl3_linear(1024, n, K, 0, g, "cuda") for n, K in ((1280, 5), (256, 6), (128, 8))]
    x = torch.randn(2, rows, 1024, device="cuda", generator=g).to(getattr(torch, dt)).transpose(0, 1)
    want = [lin(x) for lin in lins]
    group = lin_mod.EXL3SiblingGroup(lins)
    for got, w in zip(group(x), want):
        assert got.shape == w.shape and got.dtype == w.dtype and torch.equal(got, w)
    calls = []
    hook = lins[1].register_forward_hook(lambda *a: calls.append(1))
    assert all(torch.equal(a, b) for a, b in zip(group(x), want)) and calls
    hook.remove()
    with pytest.raises(ValueError):
        group(x.reshape(-1, 512))


@pytest.mark.parametrize("rows", [33, 246])
def test_prefill_rows_output_head(pk, rows):
    """The 27B output head, 5120 -> 151936 at K = 6, through the default form of few rows: one launch over all columns,
    against the fp32 product of decode_wt's weights (bar 2e-3), its transient memory the splits' sums alone (128 MiB at
    most)."""
    k, n, K = 5120, 151936, 6
    F = pk.kernels
    assert F.takes_rows_form(rows, k, n, K)
    g = torch.Generator(device="cuda").manual_seed(rows)
    tr = torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device="cuda", generator=g)
    svh = (torch.randn(n, device="cuda", generator=g) * 0.01).half()
    xh = torch.randn((rows, k), device="cuda", generator=g).half()
    out = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    F.prefill_gemm(xh, tr, k, n, K, 0, svh, out_dtype=torch.float32, out=out)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - base <= 128 << 20
    h = torch.ones(1, 1, device="cuda")
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    for c0 in range(0, n, 25344):
        cn = min(25344, n - c0)
        W = F.decode_wt(tr, k, n, K, 0, nt0=c0 // 16, ntc=cn // 16).float()
        y = xh.float() @ W.T
        del W
        ref = (y.reshape(-1, 128) @ (h / 128 ** 0.5)).reshape(rows, cn) * svh[c0:c0 + cn].float()
        err = ((out[:, c0:c0 + cn] - ref).abs().max() / ref.abs().max()).item()
        assert err < 2e-3, (c0, err)
