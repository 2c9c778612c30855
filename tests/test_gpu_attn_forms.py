"""GPU parity of every way a decode attention call runs: with a held workspace (one launch), eager without one (the
thread's), captured without one (two launches), and one workgroup per head (exl3_attn_decode_rotate), against torch
attention in fp64 from the same fp16 rows.

Bar: the output is the fp64 result rounded once to fp16 (2^-11 relative) after fp32 sums over at most 8,192 positions;
1e-3 of the largest output."""
import math
import threading

import pytest

from conftest import load_package
from test_gpu_attn_split import _inputs, _rope

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def pk():
    return load_package()


def _ref(q, k, v, kc, vc, pos, cos, sin, n_kv):
    qr, kr = _rope(q.view(-1, 128), cos[pos], sin[pos]), _rope(k.view(-1, 128), cos[pos], sin[pos])
    K, V = kc[:, :pos + 1].double(), vc[:, :pos + 1].double()
    K[:, pos], V[:, pos] = kr.double(), v.view(-1, 128).double()
    sc = torch.matmul(qr.double().view(n_kv, -1, 128), K.transpose(1, 2).contiguous()) / math.sqrt(128)
    return torch.matmul(torch.softmax(sc, -1), V).reshape(-1), kr


def _unsplit(pk, q, k, v, kc, vc, p, cos, sin, suh):
    n_kv, max_len, _ = kc.shape
    xh, o = torch.empty(1, 1, q.numel(), dtype=torch.float16, device="cuda"), torch.empty_like(q).view(1, -1)
    c = pk._capi
    c.check(c.lib().exl3_attn_decode_rotate(c.ptr(q), c.ptr(k), c.ptr(v), c.ptr(kc), c.ptr(vc), c.ptr(p), c.ptr(cos),
                                            c.ptr(sin), q.numel() // 128, n_kv, 128, max_len, c.ptr(suh), c.ptr(o),
                                            c.ptr(xh), c.stream_handle(q.device)), "exl3_attn_decode_rotate")
    return xh, o


def _call(pk, form, args):
    """(xh, o) of one call; a captured one is replayed three times, with eager work between the replays."""
    if form == "unsplit":
        return _unsplit(pk, *args)
    if form != "captured":
        q, kc = args[0], args[3]
        ws = pk.kernels.attn_workspace(q.numel() // 128, kc.shape[0], kc.shape[1], "cuda") if form == "held" else None
        return pk.kernels.attn_decode_rotate(*args, want_o=True, workspace=ws)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        xh, o = pk.kernels.attn_decode_rotate(*args, want_o=True)
    torch.cuda.current_stream().wait_stream(side)
    for i in range(3):
        xh.fill_(float("nan"))
        o.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        out = (xh.clone(), o.clone())
        assert i == 0 or torch.equal(out[1], last)
        last = out[1]
    return out


# both sides of a 64-position pass and of the positions one workgroup per head still holds: 3 to 7 passes with head groups of
# 1 (48 / 8 at 1,024), 2, 3, 4, 6, 7 and 8 heads; five workgroups of eight heads have no workgroup per head
@pytest.mark.parametrize("n_heads,n_kv,max_len", [(48, 8, 1024), (48, 8, 4096), (48, 8, 8192), (64, 8, 8192), (96, 16, 8192),
                                                 (112, 16, 8192), (128, 16, 8192), (384, 48, 600), (600, 40, 4096),
                                                 (48, 8, 512)])
@pytest.mark.parametrize("pos", [0, 63, 64, 127, 128, 191, 192, 255, 256, 319, 320, 383, 384, 448, 511])
def test_attn_forms_vs_torch(pk, n_heads, n_kv, max_len, pos):
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(n_heads, n_kv, pos, max_len)
    ref, kr = _ref(q, k, v, kc, vc, pos, cos, sin, n_kv)
    for form in ("held", "eager", "captured", "unsplit"):
        a, b = kc.clone(), vc.clone()
        xh, o = _call(pk, form, (q, k, v, a, b, p, cos, sin, suh))
        assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3, form
        assert torch.equal(xh.view(1, -1), pk.kernels.rot(o, suh.view(1, -1)).view(1, -1)), form
        assert torch.equal(a[:, pos], kr) and torch.equal(b[:, pos], v.view(-1, 128)), form
        rows = torch.arange(max_len, device="cuda") != pos
        assert torch.equal(a[:, rows].view(torch.int16), kc[:, rows].view(torch.int16)), form
        assert torch.equal(b[:, rows].view(torch.int16), vc[:, rows].view(torch.int16)), form


# one workgroup per head over several steps of its loop (512 positions each), up to the last position of the longest cache;
# the other forms at the same positions
@pytest.mark.parametrize("n_heads,n_kv,pos,max_len", [(48, 8, 1500, 2048), (48, 8, 8191, 8192), (8, 2, 1023, 1024),
                                                     (4, 4, 4500, 5000), (14, 2, 2049, 8192)])
@pytest.mark.parametrize("form", ["unsplit", "captured", "eager", "held"])
def test_attn_forms_long(pk, n_heads, n_kv, pos, max_len, form):
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(n_heads, n_kv, pos, max_len)
    ref, _ = _ref(q, k, v, kc, vc, pos, cos, sin, n_kv)
    xh, o = _call(pk, form, (q, k, v, kc, vc, p, cos, sin, suh))
    assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3
    assert torch.equal(xh.view(1, -1), pk.kernels.rot(o, suh.view(1, -1)).view(1, -1))


@pytest.mark.parametrize("form", ["held", "eager", "captured", "unsplit"])
@pytest.mark.parametrize("bad", [-1, 1024, 1 << 40, -(1 << 40)])
def test_attn_forms_invalid_position_yields_zeros(pk, form, bad):
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(48, 8, 1023, 1024)
    a, b = kc.clone(), vc.clone()
    p.fill_(bad)
    xh, o = _call(pk, form, (q, k, v, a, b, p, cos, sin, suh))
    assert not o.any() and not xh.any()
    assert torch.equal(a.view(torch.int16), kc.view(torch.int16)) and torch.equal(b.view(torch.int16), vc.view(torch.int16))


@pytest.mark.parametrize("form", ["held", "eager", "captured", "unsplit"])
@pytest.mark.parametrize("pos", [150, 300, 700])
def test_attn_forms_minus_infinity_scores(pk, form, pos):
    """A pass whose scores are all -inf has probability zero, whoever adds it."""
    q, k, v, kc, vc, p, cos, sin, suh = _inputs(48, 8, pos, 1024)
    cos[pos], sin[pos] = 1.0, 0.0
    q.view(-1, 128)[:, 0] = 1.0
    kc[:, 64:128, 0] = -math.inf
    keep = [i for i in range(pos) if not 64 <= i < 128]
    K = torch.cat((kc[:, keep], k.view(-1, 1, 128)), 1).double()
    V = torch.cat((vc[:, keep], v.view(-1, 1, 128)), 1).double()
    sc = torch.matmul(q.double().view(8, -1, 128), K.transpose(1, 2).contiguous()) / math.sqrt(128)
    ref = torch.matmul(torch.softmax(sc, -1), V).reshape(-1)
    _, o = _call(pk, form, (q, k, v, kc, vc, p, cos, sin, suh))
    assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3


def test_attn_scratch_streams_threads_and_bound(pk):
    """Calls without a workspace on two streams of two threads each, shapes in turn: every result is the held form's, the
    counters are left at zero, and a thread keeps at most ENTRIES workspaces, none for a shape past ENTRY_BYTES."""
    K = pk.kernels
    shapes = [(48, 8, 700, 1024), (8, 2, 1500, 2048), (48, 8, 6000, 8192), (4, 4, 900, 1024), (6, 1, 599, 600)]
    sets = []
    for h, kv, pos, L in shapes:
        a = _inputs(h, kv, pos, L)
        sets.append((a, K.attn_decode_rotate(*a, want_o=True, workspace=K.attn_workspace(h, kv, L, "cuda"))))
    torch.cuda.synchronize()
    errors = []

    def work():
        try:
            streams = [torch.cuda.Stream() for _ in range(2)]
            own = [[tuple(t.clone() for t in a) for a, _ in sets] for _ in streams]
            for s in streams:
                s.wait_stream(torch.cuda.current_stream())
            got = []
            for i in range(30):
                for s, inputs in zip(streams, own):
                    with torch.cuda.stream(s):
                        j = i % len(sets)
                        got.append((K.attn_decode_rotate(*inputs[j], want_o=True), sets[j][1]))
            torch.cuda.synchronize()
            assert all(torch.equal(x, y) for g, w in got for x, y in zip(g, w))
            held = K._attn_scratch.held
            assert 0 < len(held) <= K._attn_scratch.ENTRIES
            for (_, _, h, _, _), ws in held.items():
                assert ws.numel() <= K._attn_scratch.ENTRY_BYTES and not ws[:256 * h].any()
        except BaseException as e:      # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    h, kv, pos, L = 1024, 8, 40, 8192                      # 8,192 positions of 1,024 heads: past what is kept
    assert 256 * h + K._attn_workspace_bytes(h, kv, L) > K._attn_scratch.ENTRY_BYTES
    before = list(K._attn_scratch.held)
    a = _inputs(h, kv, pos, L)
    ref, _ = _ref(*a[:5], pos, a[6], a[7], kv)
    _, o = K.attn_decode_rotate(*a, want_o=True)
    assert ((o.view(-1).double() - ref).abs().max() / ref.abs().max()).item() < 1e-3
    assert list(K._attn_scratch.held) == before
