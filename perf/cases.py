"""The work a user of this library has it do, as cases that can be timed and compared.

A speculative decoder over an MLX-quantised model does five things with it: it runs the prompt
through the quantised layers (many rows), decodes one token (one row), verifies a drafted block
(2..16 rows, eagerly or as captured layer graphs), scores the block with the LM head and takes
the greedy accept, and, where activations and scales differ in dtype, runs the stock path with
fp32 outputs.  Shapes are those of the benchmark: a 5120-wide model (q|k|v 7168, MLP 17408,
vocabulary 151936) and the 4096 x 4096 projection.

Interface: listed(), draw(rng), prepare(case, seed), run(state), work(case), tolerance(case),
exact(case, seed).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "dflash-swift_amd"))
import dflash_qmm  # noqa: E402

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
MOST_WEIGHTS = 17408 * 5120  # codes of one weight at 4 bits; half as many at 8
MOST_WORK = 2048 * MOST_WEIGHTS  # multiply-adds of the largest listed case


def _case(name, kind, **kw):
    c = {"kind": kind, "rows": 1, "n": 0, "k": 0, "bits": 4, "gs": 64, "dtype": "bf16"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one decode row through one 4096 x 4096 projection, fp16
        _case("decode_proj_f16", "qmm", rows=1, n=4096, k=4096, dtype="f16"),
        # a decode step on a swapped layer: one row is below the fast kernel's window, so the
        # layer takes the stock path
        _case("decode_layer", "layer", rows=1, n=17408, k=5120),
        # a verify pass of 8 rows through an MLP projection: the benchmark's headline call
        _case("verify_up", "qmm", rows=8, n=17408, k=5120),
        # the widest verify pass through the down projection (long K)
        _case("verify_down_16", "qmm", rows=16, n=5120, k=17408),
        # a verify pass over an 8-bit q|k|v projection with a linear bias
        _case("verify_qkv_8bit", "qmm", rows=8, n=7168, k=5120, bits=8, lbias=True),
        # a verify pass of whole layers as a serving loop runs it: q|k|v, o, gate|up with the
        # activation, down, captured once as a graph and launched per pass
        _case("verify_layers", "chain", rows=8, k=5120, qkv=7168, hidden=17408, layers=4),
        # the same over the packed layout, with a wider block
        _case("verify_layers_packed_12", "chain", rows=12, k=5120, qkv=7168, hidden=17408,
              layers=2, packed=True),
        # the LM head of a verify pass with the greedy accept
        _case("lm_head_accept", "head", rows=8, n=151936, k=5120),
        # a 512-token prompt through an attention projection
        _case("prefill_proj_512", "layer", rows=512, n=5120, k=5120),
        # a ragged prompt through a whole MLP with 8-bit fp16 weights
        _case("prefill_mlp_333_8bit_f16", "mlp", rows=333, n=17408, k=5120, bits=8,
              dtype="f16"),
        # a long prompt through an MLP projection: the largest call
        _case("prefill_up_2048", "layer", rows=2048, n=17408, k=5120),
        # fp32 activations over bf16 scales: the result is fp32 (MLX's promotion)
        _case("mixed_f32_6", "mixed", rows=6, n=4096, k=4096, xdtype="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["qmm"] * 6 + ["layer"] * 6 + ["mlp"] * 2 + ["chain"] * 2 + ["mixed"] * 2 +
                      ["head"])
    bits = rng.choice([4, 4, 8])
    gs = rng.choice([32, 64, 64, 128])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    most = MOST_WEIGHTS * 4 // bits
    if kind == "qmm":
        # K a multiple of the kernel's step; not always of its preferred 8 groups
        k = _k(rng, 512, 17408, rng.choice([256, 512, 1024]))
        n = min(_log(rng, 256, 34816), most // k)
        return _case(None, kind, rows=rng.randint(1, 16), n=n, k=k, bits=bits, gs=gs,
                     dtype=dtype, lbias=rng.random() < 0.25)
    if kind == "layer":
        k = _k(rng, 512, 17408, rng.choice([128, 512]))
        n = min(_log(rng, 512, 17408), most // k)
        rows = _log(rng, 1, 2048)
        return _case(None, kind, rows=min(rows, MOST_WORK // (n * k * bits // 4)), n=n, k=k,
                     bits=bits, gs=gs, dtype=dtype, lbias=rng.random() < 0.25)
    if kind == "mlp":
        k = _k(rng, 1024, 5120, 512)
        n = min(_log(rng, 2048, 17408) // 256 * 256, most // k // 256 * 256)
        return _case(None, kind, rows=_log(rng, 17, 640), n=n, k=k, bits=bits, gs=gs,
                     dtype=dtype)
    if kind == "chain":
        k = _k(rng, 1024, 5120, 1024)
        return _case(None, kind, rows=rng.randint(1, 16), k=k, qkv=_log(rng, k, 2 * k) // 16 * 16,
                     hidden=_log(rng, 2 * k, min(4 * k, 17408)) // 1024 * 1024,
                     layers=rng.randint(1, 3), packed=rng.random() < 0.5)
    if kind == "head":
        k = _k(rng, 1024, 5120, 1024)
        return _case(None, kind, rows=rng.randint(2, 16), n=_log(rng, 32000, 151936), k=k)
    k = _k(rng, 512, 8192, 128)
    n = _log(rng, 256, 8192)
    rows = min(_log(rng, 1, 64), max(1, 10 ** 9 // (n * k)))
    xdtype, dtype = rng.choice([("f32", "bf16"), ("f32", "bf16"), ("f32", "f16"), ("bf16", "f16"),
                                ("f16", "bf16"), ("bf16", "f32")])
    return _case(None, "mixed", rows=rows, n=n, k=k, bits=rng.choice([2, 4, 8]), gs=gs,
                 dtype=dtype, xdtype=xdtype)


# ---- inputs -------------------------------------------------------------------------------

_ctx = None


def _context():
    """A program keeps one context per GPU."""
    global _ctx
    if _ctx is None:
        _ctx = dflash_qmm.Context(0)
    return _ctx


def _quantise(n, k, bits, gs, dtype, gen):
    """Normal weights (sd 0.02) quantised as MLX does: per group of gs, a scale and a bias."""
    per = 32 // bits
    top = (1 << bits) - 1
    w = torch.empty(n, k // per, dtype=torch.int32, device="cuda")
    s = torch.empty(n, k // gs, dtype=dtype, device="cuda")
    b = torch.empty(n, k // gs, dtype=dtype, device="cuda")
    step = max(1, (1 << 27) // k)
    for r in range(0, n, step):
        m = min(step, n - r)
        f = torch.randn(m, k // gs, gs, device="cuda", generator=gen) * 0.02
        lo, hi = f.amin(2), f.amax(2)
        s[r:r + m] = ((hi - lo) / top).to(dtype)
        b[r:r + m] = lo.to(dtype)
        q = (f - b[r:r + m].float()[:, :, None]) / s[r:r + m].float()[:, :, None]
        q = q.round_().clamp_(0, top).to(torch.int32).view(m, k // per, per)
        word = q[:, :, 0].clone()
        for t in range(1, per):
            word |= q[:, :, t] << (bits * t)
        w[r:r + m] = word
    return w, s, b


def _activations(rows, k, dtype, gen):
    """Normalised activations: unit normal, with one channel in 256 eight times larger."""
    x = torch.randn(rows, k, device="cuda", generator=gen)
    x[:, 17::256] *= 8.0
    return x.to(dtype)


def _dequant(w, s, b, bits, gs, rows=None):
    """Rows of the weight in 64 bits."""
    if rows is not None:
        w, s, b = w[rows], s[rows], b[rows]
    per = 32 // bits
    q = torch.stack([(w >> (bits * t)) & ((1 << bits) - 1) for t in range(per)], 2)
    n = w.shape[0]
    q = q.view(n, -1, gs).double()
    return (q * s.double()[:, :, None] + b.double()[:, :, None]).view(n, -1)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * (seed + 1))
    dt, kind = DT[case["dtype"]], case["kind"]
    rows, n, k, bits, gs = (case[f] for f in ("rows", "n", "k", "bits", "gs"))
    if kind == "chain":
        layers = []
        for _ in range(case["layers"]):
            layers.append({name: _quantise(nn, kk, bits, gs, dt, gen) for name, nn, kk in
                           (("qkv", case["qkv"], k), ("o", k, k), ("gate", case["hidden"], k),
                            ("up", case["hidden"], k), ("down", k, case["hidden"]))})
        return {"layers": layers, "x": _activations(rows, k, dt, gen),
                "a": _activations(rows, k, dt, gen), "x2": _activations(rows, k, dt, gen)}
    if kind == "mlp":
        return {"gu": _quantise(2 * n, k, bits, gs, dt, gen), "down": _quantise(k, n, bits, gs, dt,
                                                                                gen),
                "x": _activations(rows, k, dt, gen)}
    i = {"w": _quantise(n, k, bits, gs, dt, gen),
         "x": _activations(rows, k, DT[case.get("xdtype", case["dtype"])], gen)}
    if case.get("lbias"):
        i["lbias"] = (torch.randn(n, device="cuda", generator=gen) * 0.1).to(dt)
    if kind == "head":
        # a trained head's logits peak at one token: each row leans towards one vocabulary row
        target = torch.randperm(n, device="cuda", generator=gen)[:rows]
        lean = _dequant(*i["w"], bits, gs, rows=target) * (20.0 * 5120 / k)
        i["x"] = (i["x"].double() + lean).to(dt)
        # the draft agrees for the first half of the block
        prop = target[:rows - 1].to(torch.int32).clone()
        prop[rows // 2:] = (prop[rows // 2:] + 1) % n
        i["proposals"] = prop
    return i


def prepare(case, seed):
    ctx = _context()
    i = _inputs(case, seed)
    dt, kind = DT[case["dtype"]], case["kind"]
    rows, n, k, bits, gs = (case[f] for f in ("rows", "n", "k", "bits", "gs"))

    def workspace(nbytes):
        return torch.zeros(max(nbytes, 256), dtype=torch.uint8, device="cuda")

    st = {"kind": kind, "ctx": ctx, "bits": bits, "gs": gs, "i": i}
    if kind == "qmm":
        st["ws"] = workspace(ctx.workspace_bytes(rows, n, k, bits, gs))
        st["y"] = torch.empty(rows, n, dtype=dt, device="cuda")
    elif kind == "head":
        st["ws"] = workspace(ctx.qmm_argmax_accept_workspace_bytes(rows, n, k, bits, gs))
        st["logits"] = torch.empty(rows, n, dtype=dt, device="cuda")
        st["tokens"] = torch.empty(rows, dtype=torch.int32, device="cuda")
        st["accepted"] = torch.empty(1, dtype=torch.int32, device="cuda")
    elif kind in ("layer", "mixed"):
        stock = dflash_qmm.QuantizedLinear(ctx, *i["w"], i.get("lbias"), group_size=gs, bits=bits)
        # a model is swapped as a whole: an eligible layer becomes the drop-in one
        swap = kind == "layer" and dflash_qmm.SmallMQuantizedMatmul.is_eligible(stock)
        st["stock"] = stock
        st["layer"] = dflash_qmm.SmallMQuantizedLinear(stock) if swap else stock
    elif kind == "mlp":
        st["gu"] = dflash_qmm.QuantizedLinear(ctx, *i["gu"], None, group_size=gs, bits=bits)
        st["down"] = dflash_qmm.QuantizedLinear(ctx, *i["down"], None, group_size=gs, bits=bits)
    else:
        _prepare_chain(st, case)
    return st


def _prepare_chain(st, case):
    """The layers' calls captured as one graph, over buffers the program keeps."""
    ctx, i, bits, gs = st["ctx"], st["i"], case["bits"], case["gs"]
    rows, k, qkv, hid = case["rows"], case["k"], case["qkv"], case["hidden"]
    dt = i["x"].dtype
    calls, outs = [], []
    for layer in i["layers"]:
        gu = tuple(ctx.interleave_gate_up(g, u) for g, u in zip(layer["gate"], layer["up"]))
        ops = {"qkv": layer["qkv"], "o": layer["o"], "gu": gu, "down": layer["down"]}
        if case.get("packed"):
            ops = {name: ctx.pack(*w, bits, gs) for name, w in ops.items()}
        out = {name: torch.empty(rows, width, dtype=dt, device="cuda")
               for name, width in (("qkv", qkv), ("o", k), ("h", hid), ("y", k))}
        calls.append(ops)
        outs.append(out)
    need = max(ctx.workspace_bytes(rows, n, kk, bits, gs)
               for n, kk in ((qkv, k), (k, k), (2 * hid, k), (k, hid)))
    ws = torch.zeros(max(need, 256), dtype=torch.uint8, device="cuda")

    def issue(stream):
        for ops, out in zip(calls, outs):
            if isinstance(ops["qkv"], tuple):
                ctx.qmm(i["x"], *ops["qkv"], bits, gs, out=out["qkv"], ws=ws, stream=stream)
                ctx.qmm(i["a"], *ops["o"], bits, gs, out=out["o"], ws=ws, stream=stream)
                ctx.qmm_silu_gate_up(i["x2"], *ops["gu"], bits, gs, out=out["h"], ws=ws,
                                     stream=stream)
                ctx.qmm(out["h"], *ops["down"], bits, gs, out=out["y"], ws=ws, stream=stream)
            else:
                ctx.qmm_packed(i["x"], ops["qkv"], out=out["qkv"], ws=ws, stream=stream)
                ctx.qmm_packed(i["a"], ops["o"], out=out["o"], ws=ws, stream=stream)
                ctx.qmm_silu_gate_up_packed(i["x2"], ops["gu"], out=out["h"], ws=ws,
                                            stream=stream)
                ctx.qmm_packed(out["h"], ops["down"], out=out["y"], ws=ws, stream=stream)

    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    issue(stream)
    stream.synchronize()
    ctx.graph_begin(stream)
    issue(stream)
    st["graph"] = ctx.graph_end(stream)
    st["keep"] = (calls, ws, stream)
    st["outs"] = outs


def run(state):
    kind, ctx, i, bits, gs = (state[f] for f in ("kind", "ctx", "i", "bits", "gs"))
    if kind == "qmm":
        return ctx.qmm(i["x"], *i["w"], bits, gs, lbias=i.get("lbias"), out=state["y"],
                       ws=state["ws"])
    if kind == "head":
        tokens, accepted = ctx.qmm_argmax_accept(
            i["x"], *i["w"], bits, gs, proposals=i["proposals"], logits=state["logits"],
            tokens=state["tokens"], accepted=state["accepted"], ws=state["ws"])
        return {"logits": state["logits"], "tokens": tokens, "accepted": accepted}
    if kind in ("layer", "mixed"):
        return state["layer"](i["x"])
    if kind == "mlp":
        gu = state["gu"](i["x"])
        h = ctx.silu_mul(gu)
        return {"gu": gu, "h": h, "y": state["down"](h)}
    state["graph"].launch()
    return state["outs"]


# ---- what a pass cannot do without, and how close two right results come --------------------

def _weight_bytes(n, k, bits, gs, sbytes):
    return n * k * bits // 8 + 2 * n * (k // gs) * sbytes


def work(case):
    rows, n, k, bits, gs = (case[f] for f in ("rows", "n", "k", "bits", "gs"))
    sb = SIZE[case["dtype"]]
    kind = case["kind"]
    if kind == "chain":
        qkv, hid = case["qkv"], case["hidden"]
        shapes = ((qkv, k), (k, k), (2 * hid, k), (k, hid))
        per = sum(_weight_bytes(a, b, bits, gs, sb) for a, b in shapes)
        acts = rows * (qkv + k + 2 * hid + k) * sb  # h is written, and read by down
        return {"bytes": case["layers"] * (per + acts) + 3 * rows * k * sb,
                "flops": case["layers"] * 2 * rows * sum(a * b for a, b in shapes)}
    if kind == "mlp":
        w = _weight_bytes(2 * n, k, bits, gs, sb) + _weight_bytes(k, n, bits, gs, sb)
        return {"bytes": w + rows * sb * (k + 2 * n + n + k), "flops": 2 * rows * 3 * n * k}
    xb = SIZE[case.get("xdtype", case["dtype"])]
    yb = xb if case.get("xdtype", case["dtype"]) == case["dtype"] else 4
    extra = n * sb if case.get("lbias") else 0
    return {"bytes": _weight_bytes(n, k, bits, gs, sb) + rows * k * xb + rows * n * yb + extra,
            "flops": 2 * rows * n * k}


# Measured against exact() (2-norm of the difference over 2-norm of the result): bf16 outputs
# 1.7e-3 (their rounding), fp16 2.1e-4, fp32 sums in another order 1e-6 or less.  The MLP and
# the layer graphs feed a rounded activation into the next product, which adds a like error.
# Stated at about four times that.
REL = {"bf16": 7e-3, "f16": 9e-4, "f32": 1e-5}


def tolerance(case):
    if case["kind"] == "mixed":
        return {"rel": REL["f32"]}
    r = REL[case["dtype"]]
    return {"rel": 1.5 * r if case["kind"] in ("mlp", "chain") else r}


def exact(case, seed):
    i = _inputs(case, seed)
    kind, bits, gs = case["kind"], case["bits"], case["gs"]

    def lin(x, w, lbias=None):
        n, out = w[0].shape[0], []
        step = max(1, (1 << 28) // x.shape[1])
        for r in range(0, n, step):
            rows = slice(r, min(n, r + step))
            out.append(x.double() @ _dequant(*w, bits, gs, rows=rows).t())
        y = torch.cat(out, 1)
        return y if lbias is None else y + lbias.double()

    def silu_mul(g, u):
        # g and u as the library holds them: rounded to the activations' dtype
        dt = i["x"].dtype
        g, u = g.to(dt).double(), u.to(dt).double()
        return g / (1.0 + torch.exp(-g)) * u

    if kind == "chain":
        outs = []
        for layer in i["layers"]:
            h = silu_mul(lin(i["x2"], layer["gate"]), lin(i["x2"], layer["up"]))
            outs.append({"qkv": lin(i["x"], layer["qkv"]), "o": lin(i["a"], layer["o"]), "h": h,
                         "y": lin(h.to(i["x"].dtype), layer["down"])})
        return outs
    if kind == "mlp":
        gu = lin(i["x"], i["gu"])
        n = gu.shape[1] // 2
        h = silu_mul(gu[:, :n], gu[:, n:])
        return {"gu": gu, "h": h, "y": lin(h.to(i["x"].dtype), i["down"])}
    y = lin(i["x"], i["w"], i.get("lbias"))
    if kind != "head":
        return y
    tokens = y.argmax(1).to(torch.int32)
    run_len = (tokens[:-1] == i["proposals"]).to(torch.int32).cumprod(0).sum().to(torch.int32)
    return {"logits": y, "tokens": tokens, "accepted": run_len.view(1)}
