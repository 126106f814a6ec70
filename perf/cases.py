"""The engine's calls as a program that runs a Q4_0 model makes them, for timing and comparing builds.

A case is one of these, at the shapes of Llama-3.2-1B (kv260gemv/configs.py) where it is listed and at generic
ones where it is drawn:

  gemv    one matrix, one token: quantize and GEMV in one call, x as float32, engine layout or Q8_0 blocks, or
          rmsnorm in front (q|k|v, gate|up) -- the calls of a decode that is issued matrix by matrix
  mlp     the MLP of one token: gate|up with silu as its epilogue, then down
  head    the LM head with its greedy pick
  topk    the sampler's candidates of the logits
  step    a whole decode step as a chain plan, launched and waited for: per layer q|k|v, o, gate|up, down, then
          the LM head; `fused` with rmsnorm, silu and the greedy pick inside, else plain GEMVs on float32 vectors
  layer   a layer's matrices for m tokens at once (a prompt, or a few tokens decoded together): rmsnorm and
          quantize, the four GEMMs, silu between the last two; `graph`: captured once and replayed, as a program
          that decodes a fixed batch does
  build   float32 weights to Q4_0 (a model loaded from float weights)

Every result's bytes are fixed by the contract (block sums exact, every float32 operation and its order given), so
another correct build gives the same bits: tolerance() is "exact". Activations are normal with a few outlier
channels, as a transformer's hidden states have; weights are normal with a standard deviation of 0.02.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-kv260_amd"))
import kv260gemv as kv  # noqa: E402

HIDDEN, FFN, QKV, VOCAB, LAYERS = 2048, 8192, 3072, 128256, 16
EPS = 1e-5
ENGINE, F32, Q8_0, RMS = "engine", "f32", "q8_0", "rms"


def _layer(m, **more):
    return dict(dict(kind="layer", m=m, hidden=HIDDEN, qkv=QKV, ffn=FFN, graph=False), **more)


def listed():
    return [
        # One small matrix: a decode issued call by call is made of these.
        dict(name="o_gemv", kind="gemv", rows=HIDDEN, k=HIDDEN, x=F32),
        # q|k|v of a decode layer with its rmsnorm.
        dict(name="qkv_rmsnorm_gemv", kind="gemv", rows=QKV, k=HIDDEN, x=RMS),
        # A decode layer's MLP, activation quantized between the two.
        dict(name="mlp_decode", kind="mlp", hidden=HIDDEN, ffn=FFN),
        # The last matrix of every decoded token, greedy decoding.
        dict(name="lm_head_greedy", kind="head", vocab=VOCAB, hidden=HIDDEN),
        # The sampler's candidates, 40 of the vocabulary.
        dict(name="topk_40", kind="topk", n=VOCAB, k=40),
        # A token of the whole model: the framework's headline.
        dict(name="decode_step", kind="step", layers=LAYERS, hidden=HIDDEN, qkv=QKV, ffn=FFN, vocab=VOCAB, fused=True),
        # Eight tokens together: batched decode, or drafted tokens being verified, replayed token by token.
        _layer(8, name="layer_8_tokens", graph=True),
        # A short prompt.
        _layer(24, name="layer_24_tokens"),
        # A prompt of no round length, on a model of other sizes (k no multiple of 512, odd row counts).
        _layer(333, name="layer_333_ragged", hidden=2304, qkv=3333, ffn=5888),
        # A paragraph or a chunk of a chunked prefill.
        _layer(512, name="layer_512_tokens"),
        # A long prompt.
        _layer(2048, name="layer_2048_tokens"),
        # One fused gate|up matrix quantized at load time.
        dict(name="build_gate_up", kind="build", rows=2 * FFN, k=HIDDEN),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "mlp", "head", "topk", "step", "layer", "layer", "layer", "layer", "build"])
    if kind == "gemv":
        x = rng.choice([F32, F32, ENGINE, Q8_0, RMS])
        return dict(kind=kind, rows=_log_int(rng, 64, 32768), k=256 * _log_int(rng, 1, 32), x=x)
    if kind == "mlp":   # the fused epilogue's shapes: whole tiles of rows in each half
        return dict(kind=kind, hidden=2048, ffn=256 * _log_int(rng, 4, 56))
    if kind == "head":
        return dict(kind=kind, vocab=_log_int(rng, 8000, 160000), hidden=256 * rng.randint(4, 12))
    if kind == "topk":
        return dict(kind=kind, n=_log_int(rng, 4000, 262144), k=rng.randint(1, 64))
    if kind == "step":
        return dict(kind=kind, layers=rng.randint(2, LAYERS), hidden=2048, qkv=8 * rng.randint(288, 512),
                    ffn=256 * rng.randint(16, 32), vocab=_log_int(rng, 16000, VOCAB), fused=rng.random() < 0.5)
    if kind == "layer":
        m = _log_int(rng, 2, 2048)
        return _layer(m, hidden=256 * rng.randint(2, 8), qkv=_log_int(rng, 700, 3072), ffn=256 * _log_int(rng, 6, 32),
                      graph=m <= 16 and rng.random() < 0.5)
    return dict(kind=kind, rows=_log_int(rng, 1000, 16384), k=32 * _log_int(rng, 16, 64))


# ------------------------------------------------------------------ inputs


class _Inputs:
    """Seeded inputs on the GPU, drawn in order (the same sequence in prepare and exact)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def hidden(self, *shape):
        """Activations: normal, every 61st channel ten times larger."""
        x = self.normal(*shape)
        x[..., 7::61] *= 10.0
        return x

    def norm(self, k):
        return 1.0 + 0.1 * self.normal(k)

    def dense(self, rows, k):
        return self.normal(rows, k).mul_(0.02)

    def weights(self, rows, k):
        """[rows, k / 32 * 18] Q4_0 bytes: fp16 scale, then 16 bytes of two 4-bit weights (j low, j + 16 high)."""
        w = self.dense(rows, k).view(rows, k // 32, 32)
        hi, lo = w.amax(-1, keepdim=True), w.amin(-1, keepdim=True)
        d = torch.where(hi > -lo, hi, lo) / -8.0
        n = w.mul_(torch.where(d == 0, 0.0, 1.0 / d)).add_(8.5).clamp_(0.0, 15.0).to(torch.uint8)
        q = n[..., :16] | (n[..., 16:] << 4)
        return torch.cat([d.to(torch.float16).view(torch.uint8), q], dim=-1).reshape(rows, k // 32 * 18)


class _Plan:
    """A chain plan; destroyed with its state."""

    def __init__(self, steps):
        self.handle = ctypes.c_void_p()
        kv.check("w4a8_chain_plan_create_steps", kv.lib().w4a8_chain_plan_create_steps(
            ctypes.cast(steps, ctypes.c_void_p), len(steps), ctypes.byref(self.handle)))

    def __del__(self):
        if self.handle:
            kv.lib().w4a8_chain_plan_destroy(self.handle)


def _layer_inputs(i, c):
    m, h, f = c["m"], c["hidden"], c["ffn"]
    return dict(x=i.hidden(m, h), attn=i.normal(m, h), x2=i.hidden(m, h), n1=i.norm(h), n2=i.norm(h),
                wqkv=i.weights(c["qkv"], h), wo=i.weights(h, h), wgu=i.weights(2 * f, h), wd=i.weights(h, f))


def _step_inputs(i, c):
    h, f = c["hidden"], c["ffn"]
    layers = [dict(x=i.hidden(h), attn=i.normal(h), x2=i.hidden(h), act=i.normal(f), n1=i.norm(h), n2=i.norm(h),
                   wqkv=i.weights(c["qkv"], h), wo=i.weights(h, h), wgu=i.weights(2 * f, h), wd=i.weights(h, f))
              for _ in range(c["layers"])]
    return layers, dict(x=i.hidden(h), n=i.norm(h), w=i.weights(c["vocab"], h))


def _prepare_step(c, s, i):
    layers, head = _step_inputs(i, c)
    n, h, f, fused = c["layers"], c["hidden"], c["ffn"], c["fused"]

    def out(*shape, dtype=torch.float32):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    y = dict(qkv=out(n, c["qkv"]), o=out(n, h), down=out(n, h), logits=out(c["vocab"]))
    y["act" if fused else "gate_up"] = out(n, f + f // 8, dtype=torch.uint8) if fused else out(n, 2 * f)
    steps = []

    def add(kind, w, x, yt, rows, k, norm=None, best=None, ws=None):
        steps.append(kv.PlanStep(kind, w.data_ptr(), x.data_ptr(), yt.data_ptr(), rows, k,
                                 norm.data_ptr() if norm is not None else None, EPS,
                                 best.data_ptr() if best is not None else None,
                                 ws.data_ptr() if ws is not None else None))

    for j, t in enumerate(layers):
        add(kv.PLAN_GEMV, t["wqkv"], t["x"], y["qkv"][j], c["qkv"], h, t["n1"] if fused else None)
        add(kv.PLAN_GEMV, t["wo"], t["attn"], y["o"][j], h, h)
        if fused:
            add(kv.PLAN_GATE_UP_SILU_Q8, t["wgu"], t["x2"], y["act"][j], 2 * f, h, t["n2"])
            add(kv.PLAN_GEMV_ENGINE, t["wd"], y["act"][j], y["down"][j], h, f)
        else:
            add(kv.PLAN_GEMV, t["wgu"], t["x2"], y["gate_up"][j], 2 * f, h)
            add(kv.PLAN_GEMV, t["wd"], t["act"], y["down"][j], h, f)
    if fused:
        y["best"], s["ws"] = out(1, dtype=torch.int32), kv.argmax_workspace()
        add(kv.PLAN_ARGMAX, head["w"], head["x"], y["logits"], c["vocab"], h, head["n"], y["best"], s["ws"])
    else:
        add(kv.PLAN_GEMV, head["w"], head["x"], y["logits"], c["vocab"], h)
    s.update(inputs=(layers, head), y=y)
    torch.cuda.synchronize()   # a plan is not stream-ordered: what it reads is complete before it is launched
    s["plan"] = _Plan((kv.PlanStep * len(steps))(*steps))


def prepare(case, seed):
    c, i, s = case, _Inputs(seed), {}
    kind = s["kind"] = c["kind"]
    s["case"] = c
    if kind == "gemv":
        s.update(x=i.hidden(c["k"]), norm=i.norm(c["k"]), w=i.weights(c["rows"], c["k"]))
        if c["x"] == ENGINE:
            s["xq"] = kv.quantize_q8_0_engine(s["x"])
        elif c["x"] == Q8_0:   # ggml's blocks, as another program of its family hands them over
            xq, xd = kv.quantize_q8_0(s["x"])
            s["xq"] = torch.cat([xd.view(torch.uint8).view(-1, 2), xq.view(torch.uint8).view(-1, 32)], 1).reshape(-1)
        s["y"] = torch.empty(c["rows"], device="cuda")
    elif kind == "mlp":
        s.update(x=i.hidden(c["hidden"]), norm=i.norm(c["hidden"]), wgu=i.weights(2 * c["ffn"], c["hidden"]),
                 wd=i.weights(c["hidden"], c["ffn"]), ws=None)
        s["act"] = torch.empty(c["ffn"] + c["ffn"] // 8, dtype=torch.uint8, device="cuda")
        s["y"] = torch.empty(c["hidden"], device="cuda")
    elif kind == "head":
        s.update(x=i.hidden(c["hidden"]), norm=i.norm(c["hidden"]), w=i.weights(c["vocab"], c["hidden"]),
                 ws=kv.argmax_workspace(), y=torch.empty(c["vocab"], device="cuda"))
    elif kind == "topk":
        s["logits"] = 3.0 * i.normal(c["n"])
        s["ws"] = torch.empty(max(kv.lib().w4a8_topk_workspace_bytes(c["n"]), 8), dtype=torch.uint8, device="cuda")
    elif kind == "step":
        _prepare_step(c, s, i)
    elif kind == "layer":
        s.update(_layer_inputs(i, c))
        if c["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _run_layer(s)
            torch.cuda.current_stream().wait_stream(side)
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["y"] = _run_layer(s)
    else:
        s["w"] = i.dense(c["rows"], c["k"])
    return s


# -------------------------------------------------------------------- run


def _run_layer(s):
    h, f = s["case"]["hidden"], s["case"]["ffn"]
    qkv = kv.gemm_engine(s["wqkv"], h, kv.rmsnorm_q8_0_engine(s["x"], s["n1"], EPS))
    o = kv.gemm_engine(s["wo"], h, kv.quantize_q8_0_engine(s["attn"]))
    gate_up = kv.gemm_engine(s["wgu"], h, kv.rmsnorm_q8_0_engine(s["x2"], s["n2"], EPS))
    down = kv.gemm_engine(s["wd"], f, kv.silu_mul_q8_0_engine(gate_up))
    return dict(qkv=qkv, o=o, gate_up=gate_up, down=down)


def run(s):
    c, kind = s["case"], s["kind"]
    if kind == "gemv":
        if c["x"] == F32:
            return kv.gemv_q4_0_f32(s["w"], c["k"], s["x"], out=s["y"])
        if c["x"] == ENGINE:
            return kv.gemv_engine(s["w"], c["k"], s["xq"], out=s["y"])
        if c["x"] == Q8_0:
            return kv.gemv_q8_0_blocks(s["w"], c["k"], s["xq"], out=s["y"])
        return kv.gemv_rmsnorm(s["w"], c["k"], s["x"], s["norm"], EPS, out=s["y"])
    if kind == "mlp":
        act = kv.gemv_gate_up_silu(s["wgu"], c["hidden"], s["x"], s["norm"], EPS, out=s["act"], q8=True)
        return act, kv.gemv_engine(s["wd"], c["ffn"], act, out=s["y"])
    if kind == "head":
        return kv.gemv_rmsnorm_argmax(s["w"], c["hidden"], s["x"], s["norm"], EPS, s["ws"], out=s["y"])
    if kind == "topk":
        return kv.topk(s["logits"], c["k"], s["ws"])
    if kind == "step":
        L = kv.lib()
        kv.check("w4a8_chain_plan_launch", L.w4a8_chain_plan_launch(s["plan"].handle, 1))
        kv.check("w4a8_chain_plan_wait", L.w4a8_chain_plan_wait(s["plan"].handle, 10000))
        return s["y"]
    if kind == "layer":
        if c["graph"]:
            s["graph"].replay()
            return s["y"]
        return _run_layer(s)
    return kv.quantize_q4_0(s["w"])


# ------------------------------------------------------------------- work


def _q4(rows, k):
    return rows * (k // 32) * 18


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        k, x = c["k"], {F32: 4, ENGINE: 1.125, Q8_0: 34 / 32, RMS: 8}[c["x"]]
        return dict(bytes=_q4(c["rows"], k) + x * k + 4 * c["rows"], flops=2 * c["rows"] * k)
    if kind == "mlp":
        h, f = c["hidden"], c["ffn"]
        return dict(bytes=_q4(2 * f, h) + _q4(h, f) + 8 * h + 1.125 * f + 4 * h, flops=6 * h * f)
    if kind == "head":
        h, v = c["hidden"], c["vocab"]
        return dict(bytes=_q4(v, h) + 8 * h + 4 * v + 4, flops=2 * v * h)
    if kind == "topk":
        return dict(bytes=4 * c["n"] + 8 * c["k"], flops=0)
    if kind == "step":
        h, f, n, q, v = c["hidden"], c["ffn"], c["layers"], c["qkv"], c["vocab"]
        io = 8 * h + 4 * q + 4 * h + 4 * h + 8 * h + 1.125 * f + 4 * h if c["fused"] else \
            12 * h + 4 * q + 8 * h + 12 * f
        per = _q4(q, h) + _q4(h, h) + _q4(2 * f, h) + _q4(h, f)
        return dict(bytes=n * (per + io) + _q4(v, h) + 8 * h + 4 * v, flops=2 * (n * (q + h + 3 * f) + v) * h)
    if kind == "layer":
        m, h, f, q = c["m"], c["hidden"], c["ffn"], c["qkv"]
        per = _q4(q, h) + _q4(h, h) + _q4(2 * f, h) + _q4(h, f)
        return dict(bytes=per + m * (12 * h + 4 * q + 4 * h + 8 * f + 4 * h) + 8 * h, flops=2 * m * (q + h + 3 * f) * h)
    return dict(bytes=4 * c["rows"] * c["k"] + _q4(c["rows"], c["k"]), flops=0)


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ exact


def _dense(q):
    """Q4_0 bytes as float64 weights."""
    rows = q.shape[0]
    b = q.view(rows, -1, 18)
    d = b[..., :2].contiguous().view(torch.float16).double()
    n = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], dim=-1)
    return ((n.double() - 8.0) * d).view(rows, -1)


def _q8(x):
    """float64 activations as Q8_0 holds them: 32 values to a scale of amax / 127, the scale in fp16."""
    b = x.view(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    s = b * torch.where(d == 0, 0.0, 1.0 / d)
    return (torch.sign(s) * torch.floor(s.abs() + 0.5) * d.half().double()).view(x.shape)


def _rms(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _silu(gate_up):
    g, u = gate_up.chunk(2, -1)
    return g / (1.0 + torch.exp(-g)) * u


def _mul(w, x):
    return x @ _dense(w).t()


def exact(case, seed):
    c, kind, i = case, case["kind"], _Inputs(seed)
    if kind == "gemv":
        x, norm, w = i.hidden(c["k"]), i.norm(c["k"]), i.weights(c["rows"], c["k"])
        return _mul(w, _q8(_rms(x, norm) if c["x"] == RMS else x.double()))
    if kind == "mlp":
        h, f = c["hidden"], c["ffn"]
        x, norm, wgu, wd = i.hidden(h), i.norm(h), i.weights(2 * f, h), i.weights(h, f)
        return None, _mul(wd, _q8(_silu(_mul(wgu, _q8(_rms(x, norm))))))
    if kind == "head":
        h = c["hidden"]
        x, norm, w = i.hidden(h), i.norm(h), i.weights(c["vocab"], h)
        return _mul(w, _q8(_rms(x, norm))), None
    if kind == "topk":
        v = 3.0 * i.normal(c["n"])
        return torch.sort(v.double(), descending=True).values[: c["k"]], None
    if kind == "step":
        layers, head = _step_inputs(i, c)
        got = dict(qkv=[], o=[], gate_up=[], down=[])
        for t in layers:
            x, x2 = (_rms(t["x"], t["n1"]), _rms(t["x2"], t["n2"])) if c["fused"] else (t["x"].double(), t["x2"].double())
            got["qkv"].append(_mul(t["wqkv"], _q8(x)))
            got["o"].append(_mul(t["wo"], _q8(t["attn"].double())))
            got["gate_up"].append(_mul(t["wgu"], _q8(x2)))
            got["down"].append(_mul(t["wd"], _q8(_silu(got["gate_up"][-1]) if c["fused"] else t["act"].double())))
        got = {n: torch.stack(v) for n, v in got.items()}
        x = _rms(head["x"], head["n"]) if c["fused"] else head["x"].double()
        got["logits"] = _mul(head["w"], _q8(x))
        if c["fused"]:
            del got["gate_up"]
            got.update(act=None, best=None)
        return got
    if kind == "layer":
        t = _layer_inputs(i, c)
        gate_up = _mul(t["wgu"], _q8(_rms(t["x2"], t["n2"])))
        return dict(qkv=_mul(t["wqkv"], _q8(_rms(t["x"], t["n1"]))), o=_mul(t["wo"], _q8(t["attn"].double())),
                    gate_up=gate_up, down=_mul(t["wd"], _q8(_silu(gate_up))))
    return None   # Q4_0 bytes: whole numbers
