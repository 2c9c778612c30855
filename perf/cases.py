# SPDX-License-Identifier: Apache-2.0
"""Measured cases: the work that a program using these EXL3 layers has them do, through the package's public
entry points (EXL3Linear, EXL3SiblingGroup, attn_decode_rotate, SyntheticDecoder).

Kinds of case
  linear   one EXL3Linear call: decode and speculative verify (1..8 rows), short prompts, batched decode and
           prompt chunks (9..~1000 rows), whole prompts
  group    same-input siblings (q/k/v, gate/up) called as one EXL3SiblingGroup, 1..8 rows, one or several bitrates
  mlp      down(silu(gate(x)) * up(x)) of three EXL3 layers with gate / up grouped: the prompt pass of a block
  attn     batch-1 decode attention with rotary embedding, KV-cache append and o_proj's input rotation
  decoder  one decode step of a whole decoder (layers + head) with its KV cache, replayed from a captured graph

Sizes are those of the repository's own configurations: the single 4096 x 4096 layer, the 27B-class layer shapes
(hidden 5120, MLP 17408, 48 / 8 heads of 128, head 5120 -> 151936) and a 4,608-token prompt. The trellis words are
uniformly random (the codebook makes them near-Gaussian weights), the signs carry scales as checkpoints do, and
the activations have channels of different size.
"""
import importlib.util
import math
import os
import sys

import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _package():
    """The package directory omlx-exl3_amd/, imported under the module name omlx_exl3_amd."""
    name = "omlx_exl3_amd"
    if name not in sys.modules:
        pkg = os.path.join(_ROOT, "omlx-exl3_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------------
def _linear(name, k, n, K, rows, dtype="fp16", cb=0, bias=False):
    c = {"kind": "linear", "k": k, "n": n, "K": K, "rows": rows, "dtype": dtype, "cb": cb, "bias": bias}
    return {"name": name, **c} if name else c


def _group(name, k, ns, Ks, rows, dtype="fp16", cb=0):
    """ns, Ks: two or three members (a third of width 0 is absent)."""
    c = {"kind": "group", "k": k, "n0": ns[0], "n1": ns[1], "n2": ns[2], "K0": Ks[0], "K1": Ks[1], "K2": Ks[2],
         "rows": rows, "dtype": dtype, "cb": cb}
    return {"name": name, **c} if name else c


def _mlp(name, hidden, inter, K, rows, dtype="fp16", cb=0):
    c = {"kind": "mlp", "hidden": hidden, "inter": inter, "K": K, "rows": rows, "dtype": dtype, "cb": cb}
    return {"name": name, **c} if name else c


def _attn(name, heads, kv, pos, max_len):
    c = {"kind": "attn", "heads": heads, "kv": kv, "pos": pos, "max_len": max_len}
    return {"name": name, **c} if name else c


def _decoder(name, layers, K, pos, max_len, vocab=151936):
    c = {"kind": "decoder", "layers": layers, "K": K, "pos": pos, "max_len": max_len, "vocab": vocab}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one small layer at batch 1: the smallest call, all latency
        _linear("linear_4096_K4_row1", 4096, 4096, 4, 1),
        # the attention output projection of a bf16 model at batch 1
        _linear("o_bf16_row1", 6144, 5120, 6, 1, "bf16"),
        # speculative verify of 4 tokens through the q/k/v projections of a mixed-bitrate checkpoint
        _group("qkv_mixed_rows4", 5120, (6144, 1024, 1024), (5, 6, 8), 4),
        # the gate/up projections at batch 1: the largest launch of a decode step's layer
        _group("gate_up_row1", 5120, (17408, 17408, 0), (6, 6, 0), 1),
        # the widest verify step, of a low-bitrate MCG checkpoint
        _linear("down_mcg_K3_rows8", 17408, 5120, 3, 8, cb=1),
        # the output head at batch 1
        _linear("head_row1", 5120, 151936, 6, 1),
        # a short prompt, or a decode batch of 33 requests
        _linear("gate_rows33", 5120, 17408, 6, 33),
        # a prompt chunk of odd length through the MLP of a 4-bit bf16 model
        _mlp("mlp_bf16_K4_rows211", 5120, 17408, 4, 211, "bf16"),
        # a mid-sized prompt through the down projection (long k, narrow output)
        _linear("down_rows777", 17408, 5120, 6, 777),
        # a 4,608-token prompt through the MLP: the largest contraction
        _mlp("mlp_rows4608", 5120, 17408, 6, 4608),
        # decode attention deep into a long context
        _attn("attn_pos6143", 48, 8, 6143, 8192),
        # a whole decode step at a usual context length
        _decoder("decoder_step_pos700", 4, 6, 700, 1024),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng, lo, hi):
    """A layer width: a multiple of 128, spread over the logarithm of the range (odd multiples among them)."""
    return 128 * _log_int(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(["decode", "decode", "chunk", "chunk", "group", "group", "prompt", "mlp", "attn", "decoder"])
    cb = rng.choice([0, 0, 1, 2])
    dtype = rng.choice(["fp16", "fp16", "bf16"])
    K = rng.randint(2, 8)
    if kind in ("decode", "chunk", "prompt"):
        k = _dim(rng, 1024, 17408)
        n = _dim(rng, 512, min(17408, 5120 * 17408 // k))
        rows = rng.randint(1, 8) if kind == "decode" else _log_int(rng, 9, 1000) if kind == "chunk" \
            else _log_int(rng, 1000, 4608)
        return _linear(None, k, n, K, rows, dtype, cb, rng.random() < 0.25)
    if kind == "group":
        k = _dim(rng, 1024, 8192)
        same = rng.random() < 0.5
        Ks = [K if same else rng.randint(2, 8) for _ in range(3)]
        if rng.random() < 0.5:                                   # gate / up
            n = _dim(rng, 1024, 17408)
            return _group(None, k, (n, n, 0), (Ks[0], Ks[1], 0), rng.randint(1, 8), dtype, cb)
        kv = _dim(rng, 256, 2048)                                 # q / k / v
        return _group(None, k, (kv * rng.randint(2, 8), kv, kv), Ks, rng.randint(1, 8), dtype, cb)
    if kind == "mlp":
        return _mlp(None, _dim(rng, 1024, 5120), _dim(rng, 2048, 17408), K, _log_int(rng, 9, 4608), dtype, cb)
    if kind == "attn":
        kv = rng.choice([2, 4, 8])
        max_len = rng.choice([512, 1024, 2048, 4096, 8192])
        return _attn(None, kv * rng.choice([1, 2, 4, 6, 8]), kv, _log_int(rng, 16, max_len) - 1, max_len)
    max_len = rng.choice([1024, 2048, 4096])
    return _decoder(None, rng.randint(1, 3), rng.randint(3, 8), _log_int(rng, 16, max_len) - 1, max_len,
                    _dim(rng, 32000 // 128 * 128, 151936))


# ------------------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ------------------------------------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + salt)
    return g


def _scales(n, gen, size):
    """Signs with magnitudes around `size`."""
    sign = torch.randint(0, 2, (n,), generator=gen, device="cuda").to(torch.float32) * 2 - 1
    return (sign * size * (0.75 + 0.5 * torch.rand(n, generator=gen, device="cuda"))).to(torch.float16)


def _layer_tensors(k, n, K, cb, gen, bias=False):
    """The checkpoint tensors of one EXL3 layer."""
    t = {"trellis": torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), generator=gen, device="cuda",
                                  dtype=torch.int16),
         "suh": _scales(k, gen, 1.0), "svh": _scales(n, gen, 0.8 / math.sqrt(k))}
    if cb:
        t["mcg" if cb == 1 else "mul1"] = torch.zeros(1, dtype=torch.int16, device="cuda")
    if bias:
        t["bias"] = (0.1 * torch.randn(n, generator=gen, device="cuda")).to(torch.float16)
    return t


def _activations(rows, k, dtype, gen):
    """Normal values on channels whose sizes differ (a few of them several times the rest)."""
    size = torch.exp(0.5 * torch.randn(k, generator=gen, device="cuda"))
    return (torch.randn(rows, k, generator=gen, device="cuda") * size).to(_DTYPES[dtype])


def _case_layers(case):
    """(k, n, K, bias) of each layer of a linear, group or mlp case."""
    if case["kind"] == "linear":
        return [(case["k"], case["n"], case["K"], case["bias"])]
    if case["kind"] == "group":
        return [(case["k"], case["n%d" % i], case["K%d" % i], False) for i in range(3) if case["n%d" % i]]
    h, m, K = case["hidden"], case["inter"], case["K"]
    return [(h, m, K, False), (h, m, K, False), (m, h, K, False)]


def _layer_inputs(case, seed):
    gen = _gen(seed)
    layers = [_layer_tensors(k, n, K, case["cb"], gen, bias) for k, n, K, bias in _case_layers(case)]
    return layers, _activations(case["rows"], _case_layers(case)[0][0], case["dtype"], gen)


def _attn_inputs(case, seed):
    gen = _gen(seed, 1)
    nh, nkv, L = case["heads"], case["kv"], case["max_len"]

    def half(*shape):
        return torch.randn(*shape, generator=gen, device="cuda").to(torch.float16)
    inv = 1.0 / (1e6 ** (torch.arange(0, 128, 2, device="cuda", dtype=torch.float32) / 128))
    f = torch.outer(torch.arange(L, device="cuda", dtype=torch.float32), inv)
    return {"q": half(nh * 128), "k": half(nkv * 128), "v": half(nkv * 128), "kc": half(nkv, L, 128),
            "vc": half(nkv, L, 128), "pos": torch.tensor([case["pos"]], dtype=torch.int64, device="cuda"),
            "cos": f.cos(), "sin": f.sin(), "suh": _scales(nh * 128, gen, 1.0)}


def _decoder_model(case, seed):
    """A synthetic decoder with its KV caches filled up to the position, and the step's token and position."""
    pk = _package()
    S = importlib.import_module("omlx_exl3_amd.synthetic")
    cfg = S.DecoderConfig(n_layers=case["layers"], K=case["K"], max_len=case["max_len"], vocab=case["vocab"])
    model = S.SyntheticDecoder(cfg, seed=int(seed), device="cuda")
    gen = _gen(seed, 2)
    for layer in model.model.layers:
        for c in (layer.self_attn.k_cache, layer.self_attn.v_cache):
            c[:, :case["pos"]] = torch.randn(c.shape[0], case["pos"], c.shape[2], generator=gen,
                                             device="cuda").to(torch.float16)
    tok = torch.randint(0, cfg.vocab, (1,), generator=gen, device="cuda")
    return pk, model, tok, torch.tensor([case["pos"]], dtype=torch.int64, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    pk = _package()
    if kind == "attn":
        return {"kind": kind, "call": pk.kernels.attn_decode_rotate, **_attn_inputs(case, seed)}
    if kind == "decoder":
        _, model, tok, pos = _decoder_model(case, seed)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(tok, pos)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            logits = model(tok, pos)
        return {"kind": kind, "graph": graph, "model": model, "tok": tok, "pos": pos, "logits": logits,
                "caches": [(a.self_attn.k_cache, a.self_attn.v_cache) for a in model.model.layers]}
    tensors, x = _layer_inputs(case, seed)
    L = importlib.import_module("omlx_exl3_amd.linear")
    lins = []
    for (k, n, _, _), t in zip(_case_layers(case), tensors):
        lin = L.EXL3Linear(k, n, {p: (tuple(v.shape), v.dtype) for p, v in t.items()}, device="cuda")
        lin.load_state_dict(t)
        lins.append(lin)
    group = L.EXL3SiblingGroup(lins[:2] if kind == "mlp" else lins) if kind != "linear" else None
    return {"kind": kind, "lins": lins, "group": group, "x": x}


def run(state):
    kind = state["kind"]
    if kind == "decoder":
        state["graph"].replay()
        return [state["logits"], state["caches"]]
    if kind == "attn":
        xh, o = state["call"](state["q"], state["k"], state["v"], state["kc"], state["vc"], state["pos"], state["cos"],
                              state["sin"], state["suh"], want_o=True)
        return [xh, o, state["kc"], state["vc"]]
    if kind == "linear":
        return state["lins"][0](state["x"])
    if kind == "group":
        return list(state["group"](state["x"]))
    gate, up, down = state["lins"]
    x = state["x"]
    return down(F.silu(gate(x)) * up(x))


# ------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how near a correct result lies
# ------------------------------------------------------------------------------------------------------
def _layer_work(k, n, K, rows, size):
    return K * k * n // 8 + 2 * (k + n) + size * rows * (k + n), 2 * rows * k * n


def work(case):
    kind = case["kind"]
    if kind == "attn":
        kv = 2 * 2 * 128 * case["kv"] * (case["pos"] + 1)
        return {"bytes": kv + 128 * (8 * case["heads"] + 8 * case["kv"]), "flops": 4 * 128 * case["heads"] * (case["pos"] + 1)}
    if kind == "decoder":
        shapes = [(5120, 6144), (5120, 1024), (5120, 1024), (6144, 5120), (5120, 17408), (5120, 17408), (17408, 5120)]
        shapes = shapes * case["layers"] + [(5120, case["vocab"])]
        ws = [_layer_work(k, n, case["K"], 1, 2) for k, n in shapes]
        kv = 2 * 2 * 1024 * (case["pos"] + 1) * case["layers"]
        return {"bytes": sum(b for b, _ in ws) + kv, "flops": sum(f for _, f in ws) + 4 * 6144 * (case["pos"] + 1) * case["layers"]}
    size = 4 if case["dtype"] == "fp32" else 2
    layers, rows = _case_layers(case), case["rows"]
    ws = [_layer_work(k, n, K, rows, size) for k, n, K, _ in layers]
    nbytes = sum(b for b, _ in ws)
    if kind == "group":                                           # one input for all members
        nbytes -= (len(layers) - 1) * size * rows * case["k"]
    elif kind == "mlp":                                           # x once; gate, up and their product never needed in memory
        nbytes -= size * rows * (case["hidden"] + 3 * case["inter"])
    return {"bytes": nbytes, "flops": sum(f for _, f in ws)}


def tolerance(case):
    """About four times the error against 64 bits that the present path shows: the rotated input and the result
    are rounded to 16 bits (2^-11 fp16, 2^-9 bf16 relative, at most), the sums are fp32."""
    kind = case["kind"]
    if kind == "attn":
        return {"rel": 1.5e-3, "max": 1e-2}
    if kind == "decoder":
        return {"rel": 6e-3, "max": 5e-2}
    if case["dtype"] == "bf16":
        return {"rel": 2e-2, "max": 8e-2} if kind == "mlp" else {"rel": 7e-3, "max": 2e-2}
    return {"rel": 3e-3, "max": 2e-2} if kind == "mlp" else {"rel": 1.5e-3, "max": 1e-2}


# ------------------------------------------------------------------------------------------------------
# the same results in 64 bits
# ------------------------------------------------------------------------------------------------------
_HASH = {0: (89226354, 64248484), 1: (0xCBAC1FED, 0), 2: (0x83DCD12D, 0)}


def _half_bits(v):
    """int64 tensor of 16-bit patterns -> the fp16 values."""
    v = v & 0xFFFF
    return torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16)


def _codebook(cb):
    """The 65,536 weight values (fp16 by the format's definition) as float64."""
    mul, add = _HASH[cb]
    h = (torch.arange(65536, dtype=torch.int64, device="cuda") * mul + add) & 0xFFFFFFFF
    if cb == 2:
        r = (1024 + (h & 255) + (h >> 8 & 255) + (h >> 16 & 255) + (h >> 24)).to(torch.float64)
        inv, bias = _half_bits(torch.tensor([0x1EEE, 0xC931], device="cuda")).to(torch.float64)
        return (r * inv + bias).to(torch.float32).to(torch.float16).to(torch.float64)
    u = (h & 0x8FFF8FFF) ^ 0x3B603B60
    return (_half_bits(u).float() + _half_bits(u >> 16).float()).to(torch.float16).to(torch.float64)


def _weights(trellis, cb):
    """W (k, n) float64 of a trellis [k/16, n/16, 16K]: position t of a tile's 256 has as its state the 16 stream
    bits that end at bit (t + 1) K, most significant first, around the tile's end."""
    KT, NT, w16 = trellis.shape
    K = w16 // 16
    half = trellis.to(torch.int64) & 0xFFFF
    words = (half[..., 0::2] | half[..., 1::2] << 16)
    table = _codebook(cb)
    out = torch.empty(KT, 16, NT, 16, dtype=torch.float64, device=trellis.device)
    for t in range(256):
        end = (t + 1) * K
        i = (end - 1) // 32
        two = words[..., i] | (words[..., (i - 1) % (8 * K)] & 0x7FFFFFFF) << 32
        state = two >> (32 * (i + 1) - end) & 0xFFFF
        g, p = divmod(t, 32)
        out[:, 2 * (p // 8) + p % 2 + 8 * ((p % 4) // 2), :, g + (8 if p % 8 >= 4 else 0)] = table[state]
    return out.reshape(KT * 16, NT * 16)


def _hadamard(v):
    """The orthonormal 128-point Hadamard transform of each block of the last dimension."""
    h = torch.ones(1, 1, dtype=torch.float64, device=v.device)
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (v.reshape(-1, 128) @ (h / math.sqrt(128.0))).reshape(v.shape)


def _layer64(x, t, cb):
    xh = _hadamard(x * t["suh"].double())
    step, parts = 512, []                                         # n-tiles decoded at a time
    for a in range(0, t["trellis"].shape[1], step):
        parts.append(xh @ _weights(t["trellis"][:, a:a + step], cb))
    y = _hadamard(torch.cat(parts, 1)) * t["svh"].double()
    return y + t["bias"].double() if "bias" in t else y


def _attention64(q, k, v, kc, vc, pos, cos, sin):
    """(o, updated caches) for one new position; q (heads * 128,), k and v (kv * 128,), all float64."""
    def rope(a):
        a = a.reshape(-1, 128)
        lo, hi = a[:, :64], a[:, 64:]
        return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), 1)
    kc, vc = kc.clone(), vc.clone()
    kc[:, pos], vc[:, pos] = rope(k), v.reshape(-1, 128)
    nkv = kc.shape[0]
    qh = rope(q).reshape(nkv, -1, 128)
    p = torch.softmax(torch.stack([qh[i] @ kc[i, :pos + 1].T for i in range(nkv)]) / math.sqrt(128.0), -1)
    return torch.stack([p[i] @ vc[i, :pos + 1] for i in range(nkv)]).reshape(1, -1), kc, vc


def _decoder64(case, seed):
    _, model, tok, pos_t = _decoder_model(case, seed)
    pos, eps = case["pos"], model.cfg.eps
    cos, sin = model.rope_cos_half[pos].double(), model.rope_sin_half[pos].double()

    def lin(m, x):
        return _layer64(x, {"trellis": m.trellis, "suh": m.suh, "svh": m.svh}, 0)

    def norm(m, x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * m.weight.double()
    h = model.model.embed_tokens.weight[tok].double()
    caches = []
    for layer in model.model.layers:
        a, m = layer.self_attn, layer.mlp
        x = norm(layer.input_layernorm, h)
        o, kc, vc = _attention64(lin(a.q_proj, x), lin(a.k_proj, x), lin(a.v_proj, x), a.k_cache.double(),
                                 a.v_cache.double(), pos, cos, sin)
        caches.append((kc, vc))
        h = h + lin(a.o_proj, o)
        x = norm(layer.post_attention_layernorm, h)
        h = h + lin(m.down_proj, F.silu(lin(m.gate_proj, x)) * lin(m.up_proj, x))
    return [lin(model.lm_head, norm(model.model.norm, h)).reshape(-1), caches]


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "decoder":
            return _decoder64(case, seed)
        if kind == "attn":
            s = {a: b.double() if b.is_floating_point() else b for a, b in _attn_inputs(case, seed).items()}
            pos = case["pos"]
            o, kc, vc = _attention64(s["q"], s["k"], s["v"], s["kc"], s["vc"], pos, s["cos"][pos], s["sin"][pos])
            return [_hadamard(o * s["suh"])[None], o, kc, vc]
        tensors, x = _layer_inputs(case, seed)
        ys = [_layer64(x.double(), t, case["cb"]) for t in tensors[:2 if kind == "mlp" else None]]
        if kind == "mlp":
            return _layer64(F.silu(ys[0]) * ys[1], tensors[2], case["cb"])
        return ys if kind == "group" else ys[0]
