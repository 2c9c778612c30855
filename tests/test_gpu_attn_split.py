"""GPU parity of the split decode attention (exl3_attn_decode_rotate_ws), in one launch (arrival counters) and in two,
against torch attention in fp64 from the same fp16 rows.

Bar: the output is the fp64 result rounded once to fp16 (2^-11 relative) after fp32 sums over at most 8,192 positions;
1e-3 of the largest output."""
import math

import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pk():
    return load_package()


@pytest.fixture(autouse=True)
def _no_kept_workspace(pk, monkeypatch):
    """A call without a workspace takes the two launches, as when it is captured (eager it would use the thread's)."""
    monkeypatch.setattr(pk.kernels._attn_scratch, "get", lambda *a: None)


def _inputs(n_heads, n_kv, pos, max_len):
    g = torch.Generator(device="cuda").manual_seed(pos + n_heads + max_len)

    def half(*s):
        return torch.randn(*s, device="cuda", generator=g).half()
    ang = torch.rand(max_len, 64, device="cuda", generator=g) * 6.0
    kc, vc = half(n_kv, max_len, 128), half(n_kv, max_len, 128)
    kc[:, pos + 1:], vc[:, pos + 1:] = float("nan"), float("nan")      # rows past the position hold anything
    return (half(n_heads * 128), half(n_kv * 128), half(n_kv * 128), kc, vc,
            torch.tensor([pos], dtype=torch.int64, device="cuda"), ang.cos().contiguous(), ang.sin().contiguous(),
            half(n_heads * 128))


def _rope(x, c, s):
    lo, hi = x[:, :64].float(), x[:, 64:].float()
    return torch.cat((lo * c - hi * s, hi * c + lo * s), 1).half()


# positions: first, both sides of a 64-position pass and of a workgroup's second pass (48 / 8 heads: 5 workgroups of a
# head at 1,024 and 2,048), last; head groups of 1, 2, 3, 4, 6, 7 and 8 heads, a group size that does not divide
@pytest.mark.parametrize("n_heads,n_kv,max_len", [(48, 8, 1024), (48, 8, 2048), (48, 8, 8192), (8, 8, 1024),
                                                 (6, 1, 600), (10, 2, 2048), (64, 4, 4096), (7, 1, 1024),
                                                 (64, 4, 8192), (96, 16, 8192), (112, 16, 8192), (128, 16, 8192)])
@pytest.mark.parametrize("where", ["0", "63", "64", "319", "320", "640", "639", "-1"])
def test_attn_split_vs_torch(pk, n_heads, n_kv, max_len, where):
    pos = int(where) if int(where) >= 0 else max_len - 1
    if pos >= max_len:
        pytest.skip("position past this capacity")
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(n_heads, n_kv, pos, max_len)
    qr, kr = _rope(q.view(-1, 128), cos[pos], sin[pos]), _rope(k.view(-1, 128), cos[pos], sin[pos])
    K, V = kc[:, :pos + 1].double(), vc[:, :pos + 1].double()
    K[:, pos], V[:, pos] = kr.double(), v.view(-1, 128).double()
    grp = n_heads // n_kv
    sc = torch.matmul(qr.double().view(n_kv, grp, 128), K.transpose(1, 2).contiguous()) / math.sqrt(128)
    ref = torch.matmul(torch.softmax(sc, -1), V).reshape(-1)
    for ws in (None, pk.kernels.attn_workspace(n_heads, n_kv, max_len, "cuda")):
        a, b = kc.clone(), vc.clone()
        xh, o = pk.kernels.attn_decode_rotate(q, k, v, a, b, p, cos, sin, suh, want_o=True, workspace=ws)
        assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3
        assert torch.equal(xh.view(1, -1), pk.kernels.rot(o, suh.view(1, -1)).view(1, -1))
        assert torch.equal(a[:, pos], kr) and torch.equal(b[:, pos], v.view(-1, 128))
        rows = torch.arange(max_len, device="cuda") != pos
        assert torch.equal(a[:, rows].view(torch.int16), kc[:, rows].view(torch.int16))
        assert torch.equal(b[:, rows].view(torch.int16), vc[:, rows].view(torch.int16))
        xh2, o2 = pk.kernels.attn_decode_rotate(q, k, v, a, b, p, cos, sin, suh, want_o=True, workspace=ws)
        assert torch.equal(o2, o) and torch.equal(xh2, xh)
        if ws is not None:
            assert not ws[:256 * n_heads].any()          # the counters are at zero at rest


@pytest.mark.parametrize("held", [False, True])
def test_attn_split_out_of_range_position_writes_nothing(pk, held):
    n_heads, n_kv, max_len = 4, 2, 1024
    q, k, v, kc, vc, _, cos, sin, suh = _inputs(n_heads, n_kv, max_len - 1, max_len)
    ws = pk.kernels.attn_workspace(n_heads, n_kv, max_len, "cuda") if held else None
    for bad in (-1, max_len, 1 << 40):
        a, b = kc.clone(), vc.clone()
        p = torch.tensor([bad], dtype=torch.int64, device="cuda")
        xh, o = pk.kernels.attn_decode_rotate(q, k, v, a, b, p, cos, sin, suh, want_o=True, workspace=ws)
        assert not o.any() and not xh.any() and torch.equal(a, kc) and torch.equal(b, vc)


def test_attn_split_workspace_of_another_shape_is_refused(pk):
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(4, 2, 5, 1024)
    ws = pk.kernels.attn_workspace(8, 2, 1024, "cuda")
    with pytest.raises(ValueError):
        pk.kernels.attn_decode_rotate(q, k, v, kc, vc, p, cos, sin, suh, workspace=ws)


@pytest.mark.parametrize("n_heads,n_kv", [(48, 8), (8, 8), (7, 1)])
def test_attn_split_workgroup_of_minus_infinity_scores(pk, n_heads, n_kv):
    """A 64-position pass whose scores are all -inf has probability zero, as with one workgroup per head."""
    pos, max_len = 300, 1024
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(n_heads, n_kv, pos, max_len)
    cos[pos], sin[pos] = 1.0, 0.0
    q.view(-1, 128)[:, 0] = 1.0
    kc[:, 64:128, 0] = -math.inf
    keep = [i for i in range(pos) if not 64 <= i < 128]
    K = torch.cat((kc[:, keep], k.view(-1, 1, 128)), 1).double()
    V = torch.cat((vc[:, keep], v.view(-1, 1, 128)), 1).double()
    sc = torch.matmul(q.double().view(n_kv, -1, 128), K.transpose(1, 2).contiguous()) / math.sqrt(128)
    ref = torch.matmul(torch.softmax(sc, -1), V).reshape(-1)
    for ws in (None, pk.kernels.attn_workspace(n_heads, n_kv, max_len, "cuda")):
        _, o = pk.kernels.attn_decode_rotate(q, k, v, kc.clone(), vc.clone(), p, cos, sin, suh, want_o=True, workspace=ws)
        assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3
