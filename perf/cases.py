"""Performance cases: what a user of this library has it do, through its public
entry points (the ctypes mirror of include/anehip.h).

A case is a dict of plain values; `kind` names the entry points it goes through:

  linear    one quantised product y[b] = W x[b] (anehip_quant_gemm on GGUF
            blocks, anehip_quant_gemm_packed on the panel copy)
  mlp       one FFN block out of the kernel-level entries (RMSNorm, gate, up,
            SiLU-mul, down, residual add), captured once and replayed
  deltanet  one Gated DeltaNet step (anehip_deltanet_step)
  attention one attention step over an fp16 KV cache (anehip_attention_step)
  decode    one decode step of a model for `batch` sequences
  prefill   one prompt of `tokens` tokens into an empty sequence

Weights are N(0, 0.02) quantised by block absmax as GGUF files hold them,
activations N(0, 1); model tensors follow the library's random-init recipe.
Everything is made from the seed on the GPU.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ane-infer_amd"))
import anehip  # noqa: E402

Q4, Q8 = anehip.Q4_0, anehip.Q8_0
BLOCK = {Q4: 18, Q8: 34}
TYPE = {"q8_0": Q8, "q4_0": Q4}
HD = 256  # attention head width the kernels are built for
DK = 128  # DeltaNet head width
EPS = 1e-6
ROPE = 10000.0


def listed():
    shape = {"dim": 2048, "hidden": 6144, "heads": 8, "kv_heads": 2}  # the 2B hybrid's layers
    return [
        # one token's projection through one layer matrix: the smallest call, all latency
        {"name": "gemv_q8_6144x2048", "kind": "linear", "type": "q8_0", "layout": "panel", "m": 6144, "n": 2048, "batch": 1},
        # the vocabulary projection of a full decode batch
        {"name": "lm_head_q8_b32", "kind": "linear", "type": "q8_0", "layout": "panel", "m": 151936, "n": 2048, "batch": 32},
        # a caller that keeps the file's own blocks (the engine's add_gemv), a few rows at once
        {"name": "gguf_q8_12288x2048_b8", "kind": "linear", "type": "q8_0", "layout": "gguf", "m": 12288, "n": 2048, "batch": 8},
        # one chunk of a prompt through the widest layer matrix
        {"name": "chunk_q8_12288x2048_r256", "kind": "linear", "type": "q8_0", "layout": "panel", "m": 12288, "n": 2048, "batch": 256},
        # an FFN block in the smaller weight type, a small decode batch
        {"name": "mlp_q4_b4", "kind": "mlp", "type": "q4_0", "dim": 2048, "hidden": 6144, "batch": 4},
        # the recurrent mixer of a full decode batch
        {"name": "deltanet_b32", "kind": "deltanet", "heads": 16, "batch": 32},
        # attention of a full batch whose sequences stand at different lengths
        {"name": "attention_b32_8k", "kind": "attention", "heads": 8, "kv_heads": 2, "batch": 32, "max_seq": 8192},
        # attention of one long conversation
        {"name": "attention_b1_32k", "kind": "attention", "heads": 8, "kv_heads": 2, "batch": 1, "max_seq": 32768},
        # one token of one conversation through the whole 2B-shape model
        {"name": "decode_b1", "kind": "decode", "type": "q8_0", "layers": 24, "vocab": 151936, "batch": 1, "ctx": 1024, **shape},
        # one period of layers (three DeltaNet, one attention), a medium and a full batch
        {"name": "layers_b8", "kind": "decode", "type": "q8_0", "layers": 4, "vocab": 16384, "batch": 8, "ctx": 2048, **shape},
        {"name": "layers_b32", "kind": "decode", "type": "q8_0", "layers": 4, "vocab": 16384, "batch": 32, "ctx": 1024, **shape},
        # an ordinary prompt through the whole 2B-shape model (its last chunk is ragged)
        {"name": "prefill_1500", "kind": "prefill", "type": "q8_0", "layers": 24, "vocab": 151936, "tokens": 1500, **shape},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "deltanet", "attention", "attention", "decode", "decode", "prefill"])
    t = rng.choice(["q8_0", "q8_0", "q4_0"])
    if kind == "linear":
        layout = rng.choice(["panel", "panel", "gguf"])
        batch = _log(rng, 1, 256 if layout == "panel" else 32)
        n = 256 * rng.randint(4, 32)
        m = _log(rng, 1024, 160000 if n <= 2560 and batch <= 32 else 16384)
        return {"kind": kind, "type": t, "layout": layout, "m": m if batch == 1 else m // 4 * 4, "n": n, "batch": batch}
    if kind == "mlp":
        dim = 256 * rng.randint(4, 16)
        return {"kind": kind, "type": t, "dim": dim, "hidden": 256 * rng.randint(8, 48), "batch": _log(rng, 1, 256)}
    if kind == "deltanet":
        return {"kind": kind, "heads": rng.randint(4, 32), "batch": _log(rng, 1, 32)}
    kv = rng.choice([1, 2, 4])
    heads = kv * rng.choice([1, 2, 4])
    if kind == "attention":
        return {"kind": kind, "heads": heads, "kv_heads": kv, "batch": _log(rng, 1, 32), "max_seq": _log(rng, 200, 32768 if kv < 4 else 16384)}
    dim = 256 * rng.randint(4, 9)
    case = {"kind": kind, "type": t, "layers": 4, "vocab": 4 * rng.randint(1000, 8000), "dim": dim, "hidden": 256 * rng.randint(8, 32),
            "heads": heads, "kv_heads": kv}
    if kind == "decode":
        return {**case, "batch": _log(rng, 1, 32), "ctx": _log(rng, 50, 16384)}
    return {**case, "tokens": _log(rng, 16, 4096)}


# ---- inputs -----------------------------------------------------------------


class _Draws:
    """Seeded device draws; `at` names what is drawn."""

    def __init__(self, seed):
        self.seed = int(seed)

    def _gen(self, at):
        g = torch.Generator("cuda")
        g.manual_seed((self.seed * 1_000_003 + at) & 0x7FFFFFFFFFFFFFFF)
        return g

    def normal(self, at, shape, mean=0.0, std=1.0, dtype=torch.float32):
        return torch.randn(shape, generator=self._gen(at), device="cuda", dtype=dtype).mul_(std).add_(mean)

    def uniform(self, at, shape, lo, hi):
        return torch.rand(shape, generator=self._gen(at), device="cuda").mul_(hi - lo).add_(lo)

    def whole(self, at, shape, lo, hi):
        return torch.randint(lo, hi, shape, generator=self._gen(at), device="cuda")

    def blocks(self, at, t, m, n):
        """An [m, n] weight as GGUF blocks, uint8 [m, n / 32, 34 or 18]."""
        w = self.normal(at, (m, n // 32, 32), std=0.02)
        top = w.abs().amax(2, keepdim=True)
        if t == Q8:
            d = (top / 127.0).half()
            q = (w / d.float()).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        else:
            d = (top / 7.0).half()
            q = (w / d.float()).round_().add_(8).clamp_(0, 15).to(torch.uint8)
            q = q[..., :16] | (q[..., 16:] << 4)
        return torch.cat([d.view(torch.uint8), q], 2).contiguous()


def _weights64(blocks, t):
    """GGUF blocks as the 64-bit matrix they stand for."""
    m = blocks.shape[0]
    d = blocks[..., :2].contiguous().view(torch.float16).double()
    if t == Q8:
        q = blocks[..., 2:].contiguous().view(torch.int8).double()
    else:
        b = blocks[..., 2:]
        q = torch.cat([b & 15, b >> 4], 2).double() - 8.0
    return (q * d).reshape(m, -1)


_shared = None


def _ctx():
    """The program's one bare context (its stream orders all kernel-level calls)."""
    global _shared
    if _shared is None:
        _shared = anehip.Context(0)
    return _shared


class _Owner:
    """A model; closed when the state and every tensor that looks into the model's memory are gone."""

    def __init__(self, model):
        self.model = model

    def __del__(self):
        self.model.close()


class _State(dict):
    """What one case keeps; gives back its graph when it goes."""

    def __del__(self):
        if "graph" in self:
            anehip.Context.graph_destroy(self["graph"])


def _panel(ctx, t, blocks, m, n):
    out = torch.empty(anehip.lib().anehip_quant_packed_bytes(t, m, n), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    ctx.call("quant_pack", t, blocks.data_ptr(), m, n, out.data_ptr())
    ctx.sync()
    return out


def _spec(c):
    return anehip.Spec(dim=c["dim"], hidden_dim=c["hidden"], n_layers=c["layers"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                       head_dim=HD, vocab_size=c["vocab"], ssm_state_size=DK, ssm_conv_kernel=4, ssm_group_count=c["dim"] // DK,
                       rope_freq_base=ROPE, rms_norm_eps=EPS)


def _at(layer, kind):
    return 1000 + (layer + 1) * 64 + kind


def _vector(r, layer, kind, shape):
    dist, a, b = anehip.F32_RECIPE[kind]
    return r.normal(_at(layer, kind), shape, a, b) if dist == 0 else r.uniform(_at(layer, kind), shape, a, b)


class _DeviceArray:
    """A device buffer of a model, for torch.as_tensor: the tensor keeps this object, and so the model, alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 2}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_DeviceArray(owner, ptr, shape, typestr), device="cuda")


def _state_shapes(c, batch, max_seq):
    """{(layer, which): shape} of the model's per-sequence state."""
    out = {}
    for l in range(c["layers"]):
        if l % 4 == 3:
            out[l, 2] = out[l, 3] = (batch, c["kv_heads"], max_seq, HD)
        else:
            out[l, 0] = (batch, 3 * c["dim"], 4)
            out[l, 1] = (batch, c["dim"] // DK, DK, DK)
    return out


def _state_values(c, r, batch, max_seq):
    """State as a sequence some way on has it."""
    for (l, which), shape in _state_shapes(c, batch, max_seq).items():
        at = 500_000 + 8 * l + which
        if which >= 2:
            yield l, which, r.normal(at, shape, dtype=torch.float16)
        else:
            yield l, which, r.normal(at, shape, std=1.0 if which == 0 else 0.01)


def _capacity(c):
    return c["ctx"] + 256 if c["kind"] == "decode" else c["tokens"]


def _tokens(c, r):
    shape = (c["batch"],) if c["kind"] == "decode" else (c["tokens"],)
    return r.whole(7, shape, 0, c["vocab"])


def _model(c, r):
    t = TYPE[c["type"]]
    spec = _spec(c)
    batch, cap = c.get("batch", 1), _capacity(c)
    gm = anehip.Model(spec)
    owner = _Owner(gm)
    s = _State(model=gm, owner=owner, case=c)
    for layer in [-1] + list(range(spec.n_layers)):
        for kind, (rows, cols, quant) in spec.shapes(layer).items():
            v = r.blocks(_at(layer, kind), t, rows, cols) if quant else _vector(r, layer, kind, (rows, cols))
            ptr, nbytes = gm.tensor_ptr(layer, kind, t)
            assert nbytes == v.numel() * v.element_size()
            torch.cuda.synchronize()
            gm.d2d(ptr, v.data_ptr(), nbytes)
            gm.sync()
    gm.alloc_state(batch, cap)
    tokens = _tokens(c, r).cpu().numpy().astype(np.uint32)
    s["views"] = {}
    for (l, which), shape in _state_shapes(c, batch, cap).items():
        s["views"]["%d.%d" % (l, which)] = _view(owner, gm.state_ptr(l, which)[0], shape, "<f2" if which >= 2 else "<f4")
    s["tokens"] = tokens
    if c["kind"] == "decode":
        # one step first, as any session has had (it lays the weights out and records the step), then the sequences' states
        gm.step(tokens, want_logits=False)
        for l, which, v in _state_values(c, r, batch, cap):
            s["views"]["%d.%d" % (l, which)].copy_(v)
        for b in range(batch):
            gm.set_pos(b, c["ctx"])
        s["left"] = cap - c["ctx"]
        p = anehip.C.c_void_p()
        gm._check(anehip.lib().anehip_logits_ptr(gm.h, anehip.C.byref(p)))
        s["logits"] = _view(owner, p.value, (batch, c["vocab"]), "<f4")
    else:
        gm.prefill(0, tokens[:1], want_logits=False)  # lays the weights out
    torch.cuda.synchronize()
    return s


def _positions(c, r):
    return r.whole(6, (c["batch"],), c["max_seq"] // 4, c["max_seq"]) if c["batch"] > 1 else r.whole(6, (1,), c["max_seq"] * 15 // 16, c["max_seq"])


def _inputs(c, r):
    """The plain tensors of a kernel-level case."""
    if c["kind"] == "linear":
        return {"w": r.blocks(1, TYPE[c["type"]], c["m"], c["n"]), "x": r.normal(2, (c["batch"], c["n"]))}
    if c["kind"] == "mlp":
        d, f, t = c["dim"], c["hidden"], TYPE[c["type"]]
        return {"x": r.normal(1, (c["batch"], d)), "norm": r.normal(2, (d,), 1.0, 0.1), "gate": r.blocks(3, t, f, d),
                "up": r.blocks(4, t, f, d), "down": r.blocks(5, t, d, f)}
    if c["kind"] == "deltanet":
        b, h = c["batch"], c["heads"]
        ch = 3 * h * DK
        return {"qkv": r.normal(1, (b, ch)), "beta": r.normal(2, (b, h)), "alpha": r.normal(3, (b, h)), "conv_w": r.normal(4, (ch, 4), std=0.3),
                "ssm_a": r.uniform(5, (h,), -1.0, 0.0), "dt": r.normal(6, (h,)), "conv": r.normal(7, (b, ch, 4)),
                "S": r.normal(8, (b, h, DK, DK), std=0.01)}
    b, h, kv = c["batch"], c["heads"], c["kv_heads"]
    cache = (b, kv, c["max_seq"], HD)
    return {"qkv": r.normal(1, (b, h * 2 * HD + 2 * kv * HD)), "q_norm": r.normal(2, (HD,), 1.0, 0.1), "k_norm": r.normal(3, (HD,), 1.0, 0.1),
            "pos": _positions(c, r).to(torch.int32), "k": r.normal(4, cache, dtype=torch.float16), "v": r.normal(5, cache, dtype=torch.float16)}


def prepare(case, seed):
    r = _Draws(seed)
    c = case
    if c["kind"] in ("decode", "prefill"):
        return _model(c, r)
    ctx = _ctx()
    s = _State(_inputs(c, r))
    s["case"], s["ctx"] = c, ctx
    empty = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if c["kind"] == "linear":
        s["y"] = empty(c["batch"], c["m"])
        if c["layout"] == "panel":
            s["w"] = _panel(ctx, TYPE[c["type"]], s["w"], c["m"], c["n"])
    elif c["kind"] == "mlp":
        t, d, f, b = TYPE[c["type"]], c["dim"], c["hidden"], c["batch"]
        for name, (m, n) in {"gate": (f, d), "up": (f, d), "down": (d, f)}.items():
            s[name] = _panel(ctx, t, s[name], m, n)
        s["h"], s["g"], s["u"], s["y"] = empty(b, d), empty(b, f), empty(b, f), empty(b, d)
        x = s["x"].clone()
        torch.cuda.synchronize()

        def block():
            ctx.call("rmsnorm", s["x"].data_ptr(), s["norm"].data_ptr(), s["h"].data_ptr(), b, d, EPS)
            ctx.call("quant_gemm_packed", t, s["gate"].data_ptr(), f, d, s["h"].data_ptr(), b, s["g"].data_ptr())
            ctx.call("quant_gemm_packed", t, s["up"].data_ptr(), f, d, s["h"].data_ptr(), b, s["u"].data_ptr())
            ctx.call("silu_mul", s["g"].data_ptr(), s["u"].data_ptr(), b * f)
            ctx.call("quant_gemm_packed", t, s["down"].data_ptr(), d, f, s["g"].data_ptr(), b, s["y"].data_ptr())
            ctx.call("residual_add", s["x"].data_ptr(), s["y"].data_ptr(), b * d)

        block()  # sizes the context's workspace, as recording needs
        ctx.sync()
        s["x"].copy_(x)
        torch.cuda.synchronize()
        ctx.capture_begin()
        block()
        s["graph"] = ctx.capture_end()
    elif c["kind"] == "deltanet":
        s["o"] = empty(c["batch"], c["heads"] * DK)
    else:
        s["o"] = empty(c["batch"], c["heads"] * HD)
    torch.cuda.synchronize()
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "linear":
        name = "quant_gemm_packed" if c["layout"] == "panel" else "quant_gemm"
        s["ctx"].call(name, TYPE[c["type"]], s["w"].data_ptr(), c["m"], c["n"], s["x"].data_ptr(), c["batch"], s["y"].data_ptr())
        return s["y"]
    if kind == "mlp":
        s["ctx"].graph_launch(s["graph"])
        return s["x"]
    if kind == "deltanet":
        s["ctx"].call("deltanet_step", c["batch"], c["heads"], s["qkv"].data_ptr(), s["beta"].data_ptr(), s["alpha"].data_ptr(),
                      s["conv_w"].data_ptr(), s["ssm_a"].data_ptr(), s["dt"].data_ptr(), s["conv"].data_ptr(), s["S"].data_ptr(), s["o"].data_ptr())
        return {"o": s["o"], "conv": s["conv"], "S": s["S"]}
    if kind == "attention":
        s["ctx"].call("attention_step", c["batch"], c["heads"], c["kv_heads"], c["max_seq"], s["qkv"].data_ptr(), s["q_norm"].data_ptr(),
                      s["k_norm"].data_ptr(), ROPE, s["pos"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr())
        return {"o": s["o"], "k": s["k"], "v": s["v"]}
    gm = s["model"]
    if kind == "decode":
        if s["left"] == 0:  # the cache is full: back to where the sequences stood
            for b in range(c["batch"]):
                gm.set_pos(b, c["ctx"])
            s["left"] = _capacity(c) - c["ctx"]
        s["left"] -= 1
        gm.step(s["tokens"], want_logits=False)
        return {"logits": s["logits"], **s["views"]}
    gm.reset_state()
    return {"logits": gm.prefill(0, s["tokens"]), **s["views"]}


# ---- what a pass cannot do without -------------------------------------------


def _qbytes(t, m, n):
    return m * (n // 32) * BLOCK[t]


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        m, n, b = c["m"], c["n"], c["batch"]
        return {"bytes": _qbytes(TYPE[c["type"]], m, n) + 4 * b * (m + n), "flops": 2 * m * n * b}
    if kind == "mlp":
        d, f, b = c["dim"], c["hidden"], c["batch"]
        return {"bytes": 3 * _qbytes(TYPE[c["type"]], f, d) + 4 * (2 * b * d + d), "flops": 6 * b * d * f}
    if kind == "deltanet":
        b, h = c["batch"], c["heads"]
        # per sequence: S and the three kept window columns read, S and one column written, qkv in, heads out, beta / alpha
        return {"bytes": b * (2 * h * DK * DK + 3 * h * DK * (3 + 1 + 1) + h * DK + 2 * h) * 4 + 3 * h * DK * 16, "flops": b * h * DK * DK * 7}
    if kind == "attention":
        b, h, kv = c["batch"], c["heads"], c["kv_heads"]
        n = b * c["max_seq"] * (0.625 if b > 1 else 0.97)  # positions read, on average
        return {"bytes": n * kv * HD * 4 + b * 4 * (3 * h * HD + 2 * kv * HD), "flops": 4 * n * h * HD}
    t, d, f, h, kv = TYPE[c["type"]], c["dim"], c["hidden"], c["heads"], c["kv_heads"]
    b, steps, seen = (c["batch"], 1, c["ctx"] + 1) if kind == "decode" else (1, c["tokens"], c["tokens"])
    params, mixers, flops = 3 * f * d * c["layers"], 0, 0
    for l in range(c["layers"]):
        if l % 4 == 3:
            params += (3 * h * HD + 2 * kv * HD) * d
            mixers += b * 4 * kv * HD * (seen if kind == "decode" else 1)
            flops += b * 4 * h * HD * (seen if kind == "decode" else steps * (steps + 1) // 2)
            mixers += 0 if kind == "decode" else 4 * kv * HD * steps
        else:
            params += (5 * d + 2 * d // DK) * d
            mixers += b * (2 * d * DK + 3 * d * 5) * 4
            flops += b * steps * d * DK * 7
    head = c["vocab"] * d
    return {"bytes": _qbytes(t, 1, params) + _qbytes(t, 1, head) + mixers + 4 * (b * c["vocab"] + b * steps * d),
            "flops": 2 * b * (params * steps + head) + flops}


def tolerance(case):
    """Four times what the path's outputs are off 64 bits by, which is about what another order of its 32-bit sums moves them."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "mlp":
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "deltanet":
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "attention":
        # RoPE's angle position * frequency is a 32-bit product: 2e-4 off at 32k positions
        return {"rel": 8e-4, "max": 3e-2}
    # a cached key or value next to a rounding boundary of its 16 bits falls either way, and the layers after carry that on
    return {"rel": 1e-3, "max": 3e-2}


# ---- the same in 64 bits, in plain torch -------------------------------------


def _norm(x, w, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _delta(qkv, beta, alpha, conv_w, ssm_a, dt, conv, S):
    """Gated DeltaNet over T tokens: qkv [B, T, C], beta / alpha [B, T, H]; heads [B, T, H, 128] and the new window and state."""
    b, steps, ch = qkv.shape
    h = ch // (3 * DK)
    seen = torch.cat([conv, qkv.transpose(1, 2)], 2)  # [B, C, 4 + T]
    act = _silu(sum(seen[:, :, 1 + i:1 + i + steps] * conv_w[:, i, None] for i in range(4))).transpose(1, 2)
    q, k, v = act.reshape(b, steps, 3, h, DK).unbind(2)
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-12)  # noqa: E731
    q, k = unit(q) / math.sqrt(DK), unit(k)
    beta = torch.sigmoid(beta)
    decay = torch.exp(ssm_a * torch.nn.functional.softplus(alpha + dt, threshold=1e9))
    out = torch.empty(b, steps, h, DK, dtype=torch.float64, device=qkv.device)
    S = S.clone()
    for t in range(steps):
        S *= decay[:, t, :, None, None]
        delta = beta[:, t, :, None] * (v[:, t] - (k[:, t].unsqueeze(-2) @ S).squeeze(-2))
        S += k[:, t].unsqueeze(-1) * delta.unsqueeze(-2)
        out[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
    return out, seen[:, :, -4:].contiguous(), S


def _rope(x, pos):
    """x [..., T, 256] at positions pos [T]: adjacent pairs rotated."""
    inv = ROPE ** (-torch.arange(0, HD, 2, dtype=torch.float64, device=x.device) / HD)
    a = pos.double()[:, None] * inv
    c, s = a.cos(), a.sin()
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * s, e * s + o * c], -1).flatten(-2)


def _attend(qkv, pos, q_norm, k_norm, k_cache, v_cache, h, kv):
    """One sequence, T tokens from position pos: qkv [T, ...]; caches [kv, max_seq, 256] fp16, appended in place."""
    steps = qkv.shape[0]
    at = torch.arange(pos, pos + steps, device=qkv.device)
    q, gate = qkv[:, :h * 2 * HD].reshape(steps, h, 2, HD).unbind(2)
    k, v = qkv[:, h * 2 * HD:].reshape(steps, 2, kv, HD).unbind(1)
    q = _rope(_norm(q, q_norm).transpose(0, 1), at)
    k_cache[:, pos:pos + steps] = _rope(_norm(k, k_norm).transpose(0, 1), at).half()
    v_cache[:, pos:pos + steps] = v.transpose(0, 1).half()
    K, V = (x[:, :pos + steps].double() for x in (k_cache, v_cache))
    hidden = torch.arange(pos + steps, device=qkv.device)[None, :] > at[:, None]
    out = torch.empty(steps, h, HD, dtype=torch.float64, device=qkv.device)
    for i in range(h):
        p = (q[i] @ K[i // (h // kv)].T / math.sqrt(HD)).masked_fill_(hidden, -math.inf)
        out[:, i] = torch.softmax(p, -1) @ V[i // (h // kv)]
    return (out * torch.sigmoid(gate)).reshape(steps, -1)


def _forward64(c, r):
    """Decode: one token of each sequence; prefill: all tokens of one. Logits of each sequence's last token, and the states."""
    T = anehip.T
    t, d = TYPE[c["type"]], c["dim"]
    spec = _spec(c)
    cap = _capacity(c)
    batch = c.get("batch", 1)
    tokens = _tokens(c, r).reshape(batch, -1)
    steps, pos = tokens.shape[1], c.get("ctx", 0)
    state = {k: torch.zeros(s, dtype=torch.float16 if k[1] >= 2 else torch.float64, device="cuda") for k, s in _state_shapes(c, batch, cap).items()}
    if c["kind"] == "decode":
        for l, which, v in _state_values(c, r, batch, cap):
            state[l, which] = v if which >= 2 else v.double()

    def vec(layer, kind):
        rows, cols, _ = spec.shapes(layer)[T[kind]]
        v = _vector(r, layer, T[kind], (rows, cols)).double()
        return v[0] if rows == 1 else v

    def lin(x, layer, kind):
        rows, cols, _ = spec.shapes(layer)[T[kind]]
        return x @ _weights64(r.blocks(_at(layer, T[kind]), t, rows, cols), t).T

    rows, cols, _ = spec.shapes(-1)[T["EMBEDDING"]]
    x = _vector(r, -1, T["EMBEDDING"], (rows, cols))[tokens].double()
    for l in range(c["layers"]):
        h = _norm(x, vec(l, "ATTN_NORM"))
        if l % 4 == 3:
            qkv = torch.cat([lin(h, l, k) for k in ("WQ", "WK", "WV")], -1)
            o = torch.stack([_attend(qkv[b], pos, vec(l, "Q_NORM"), vec(l, "K_NORM"), state[l, 2][b], state[l, 3][b], c["heads"], c["kv_heads"])
                             for b in range(batch)])
            x = x + lin(o, l, "WO")
        else:
            o, state[l, 0], state[l, 1] = _delta(lin(h, l, "QKV"), lin(h, l, "SSM_BETA"), lin(h, l, "SSM_ALPHA"), vec(l, "SSM_CONV1D"),
                                                 vec(l, "SSM_A"), vec(l, "SSM_DT_BIAS"), state[l, 0], state[l, 1])
            o = _norm(o, vec(l, "SSM_NORM")).reshape(batch, steps, d) * _silu(lin(h, l, "ATTN_GATE"))
            x = x + lin(o, l, "SSM_OUT")
        h = _norm(x, vec(l, "POST_ATTN_NORM"))
        x = x + lin(_silu(lin(h, l, "FFN_GATE")) * lin(h, l, "FFN_UP"), l, "FFN_DOWN")
    logits = lin(_norm(x[:, -1], vec(-1, "FINAL_NORM")), -1, "LM_HEAD")
    views = {"%d.%d" % k: (v.double() if k[1] >= 2 else v) for k, v in state.items()}
    return {"logits": logits if c["kind"] == "decode" else logits[0], **views}


def exact(case, seed):
    r = _Draws(seed)
    c = case
    if c["kind"] in ("decode", "prefill"):
        return _forward64(c, r)
    v = _inputs(c, r)
    if c["kind"] == "linear":
        return v["x"].double() @ _weights64(v["w"], TYPE[c["type"]]).T
    if c["kind"] == "mlp":
        t = TYPE[c["type"]]
        x = v["x"].double()
        h = _norm(x, v["norm"].double())
        g, u = (h @ _weights64(v[k], t).T for k in ("gate", "up"))
        return x + (_silu(g) * u) @ _weights64(v["down"], t).T
    if c["kind"] == "deltanet":
        f = {k: x.double() for k, x in v.items()}
        o, conv, S = _delta(f["qkv"][:, None], f["beta"][:, None], f["alpha"][:, None], f["conv_w"], f["ssm_a"], f["dt"], f["conv"], f["S"])
        return {"o": o.reshape(c["batch"], -1), "conv": conv, "S": S}
    out = torch.stack([_attend(v["qkv"][b:b + 1].double(), int(v["pos"][b]), v["q_norm"].double(), v["k_norm"].double(), v["k"][b], v["v"][b],
                               c["heads"], c["kv_heads"])[0] for b in range(c["batch"])])
    return {"o": out, "k": v["k"].double(), "v": v["v"].double()}
