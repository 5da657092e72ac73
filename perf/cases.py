"""What the engine's speed is measured on: decode steps, prompts and chat turns
of packed models, the batched projections and the attention of single layers,
and the fused unpack-matvec, each through the calls that a program makes
(`GPUMistralV2Model`, the C ABI of `gsdlq.hip`).

Models are random: codes drawn with the probabilities that a Gaussian weight
gives the points of the hexagon, fp16 scales around 0.02 per weight, norms
around one.  Shapes are the Mistral-7B shape of the benchmark and two smaller
ones of the tests; modes are "turbo" (radius 8, one byte per code) and
"precision" (radius 6, rank 2).  Whole calls run two to four layers, so that the
head and the host's part weigh more than in a 32-layer model.

The oracle (`exact`) dequantises to float64 and runs the reference's formulas;
what the format itself rounds (K and V rows in fp16, RoPE angles in float32)
is rounded there too.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "gsd-lq_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

SHAPES = {
    "7b": dict(hidden=4096, ffn=14336, n_heads=32, n_kv_heads=8, head_dim=128, vocab=32768),
    "mid": dict(hidden=2048, ffn=5056, n_heads=16, n_kv_heads=4, head_dim=128, vocab=512),
    "small": dict(hidden=256, ffn=512, n_heads=4, n_kv_heads=2, head_dim=64, vocab=512),
}
MODES = {"turbo": dict(radius=8, k_dim=0), "precision": dict(radius=6, k_dim=2)}
LAYER = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")
SETS = {"qkv": LAYER[:3], "o": LAYER[3:4], "gate_up": LAYER[4:6], "down": LAYER[6:]}
EPS, THETA, SIGMA = 1e-5, 1e6, 0.02


def listed():
    return [
        # the least a call can cost: one sampled token of a small model with kinks
        dict(name="step_small", kind="step", shape="small", mode="precision", kinks=2, layers=2, pos=33, max_seq=64),
        # a chat's reply, token by token with the logits on the host, early in the context
        dict(name="step_7b", kind="step", shape="7b", mode="precision", kinks=0, layers=2, pos=100, max_seq=2048),
        # the same near the end of a full context, the other mode
        dict(name="step_7b_late", kind="step", shape="7b", mode="turbo", kinks=0, layers=2, pos=1733, max_seq=2048),
        # a short user turn on top of a cached conversation
        dict(name="turn_7b", kind="prompt", shape="7b", mode="turbo", kinks=0, layers=2, start=301, n=37, max_seq=2048),
        # a first prompt: system rules and a long question
        dict(name="prompt_7b", kind="prompt", shape="7b", mode="precision", kinks=0, layers=4, start=0, n=923, max_seq=2048),
        # batched projections of one layer: a few sequences at once, a batch, a prefill chunk
        dict(name="qkv_16", kind="matmul", shape="7b", mode="turbo", kinks=0, tensors="qkv", m=16),
        dict(name="gate_up_128", kind="matmul", shape="7b", mode="precision", kinks=0, tensors="gate_up", m=128),
        dict(name="down_512", kind="matmul", shape="7b", mode="turbo", kinks=0, tensors="down", m=512),
        # a prompt chunk's causal attention behind a long prefix
        dict(name="attend_512", kind="attend", n_heads=32, n_kv_heads=8, head_dim=128, pos0=1024, m=512),
        # one token's RoPE, K/V append and attention over eight layers' caches: mid context, long context
        dict(name="decode_700", kind="decode", n_heads=32, n_kv_heads=8, head_dim=128, ctx=700, layers=8),
        dict(name="decode_8192", kind="decode", n_heads=32, n_kv_heads=8, head_dim=128, ctx=8192, layers=8),
        # one packed tensor in the file's layout: rank projection, then the fused unpack-matvec
        dict(name="matvec_4096", kind="matvec", rows=4096, cols=4096, radius=6, k_dim=2, kinks=1),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "prompt", "matmul", "matmul", "attend", "decode", "matvec"))
    mode = rng.choice(("turbo", "precision"))
    if kind == "step":
        shape = rng.choice(("7b", "7b", "mid", "small"))
        return dict(kind=kind, shape=shape, mode=mode, kinks=rng.choice((0, 0, 1)), layers=rng.choice((1, 2)),
                    pos=_log_int(rng, 8, 2000), max_seq=2048)
    if kind == "prompt":
        shape = rng.choice(("7b", "7b", "mid"))
        n = _log_int(rng, 2, 900)
        # (the listed prompt stands for precision: a shallow model's head takes some hundred prompts only)
        return dict(kind=kind, shape=shape, mode="turbo", kinks=rng.choice((0, 0, 1)), layers=rng.choice((1, 2)),
                    start=rng.randrange(0, 1024), n=n, max_seq=2048)
    if kind == "matmul":
        return dict(kind=kind, shape=rng.choice(("7b", "7b", "mid")), mode=mode, kinks=rng.choice((0, 0, 1)),
                    tensors=rng.choice(tuple(SETS)), m=_log_int(rng, 2, 512))
    if kind in ("attend", "decode"):
        h, kv, hd = rng.choice(((32, 8, 128), (32, 8, 128), (16, 4, 128), (16, 8, 64)))
        if kind == "attend":
            return dict(kind=kind, n_heads=h, n_kv_heads=kv, head_dim=hd, pos0=rng.randrange(0, 1024), m=_log_int(rng, 8, 512))
        return dict(kind=kind, n_heads=h, n_kv_heads=kv, head_dim=hd, ctx=_log_int(rng, 16, 8192), layers=8)
    rows, cols = rng.choice(((4096, 4096), (1024, 4096), (4096, 14336), (14336, 4096), (2048, 5056), (520, 192)))
    radius = rng.choice((6, 8))
    return dict(kind=kind, rows=rows - rng.randrange(0, 9), cols=cols, radius=radius, k_dim=2 if radius == 6 else 0,
                kinks=rng.choice((0, 1, 3)))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, stream):
    return torch.Generator("cuda").manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFF)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _points(radius):
    """float64 [n, 2]: the hexagon's points in the order of the codes."""
    return np.array([(a + 0.5 * b, b * math.sqrt(3.0) / 2.0) for a in range(-radius, radius + 1)
                     for b in range(-radius, radius + 1) if abs(a + b) <= radius])


def _tensor(seed, stream, rows, cols, radius, k_dim, kinks):
    """A packed tensor's fields on the GPU, typed as in a .gsd2 file."""
    g = _gen(seed, stream)
    pts = torch.from_numpy(_points(radius)).cuda()
    spread = radius / 2.9   # the largest of a block's 32 Gaussian pairs lies on the rim
    cdf = torch.softmax(-(pts ** 2).sum(1) / (2 * spread ** 2), 0).cumsum(0).float()
    u = torch.rand(rows * cols // 2, generator=g, device="cuda")
    codes = torch.searchsorted(cdf, u, out_int32=True).clamp_(max=len(pts) - 1).to(torch.uint8)
    scales = (SIGMA / spread * torch.exp(0.12 * _randn(g, rows * cols // 64))).half()
    f = dict(codes=codes, scales=scales, row_ptr=torch.arange(rows + 1, device="cuda", dtype=torch.int32) * kinks)
    at = torch.rand(rows, cols, generator=g, device="cuda").topk(kinks, 1).indices.sort(1).values if kinks else torch.zeros(0)
    f["kink_cols"] = at.reshape(-1).to(torch.int32).to(torch.uint16)
    f["kink_deltas"] = 3 * SIGMA * _randn(g, rows * kinks)
    if k_dim:
        f["U"] = (_randn(g, rows, k_dim) / math.sqrt(rows)).half()
        f["S"] = 0.2 * SIGMA * (math.sqrt(rows) + math.sqrt(cols)) * (1 + 0.1 * _randn(g, k_dim).abs())
        f["Vt"] = (_randn(g, k_dim, cols) / math.sqrt(cols)).half()
    return f


_FIELD = dict(codes=np.uint8, scales=np.uint16, row_ptr=np.uint32, kink_cols=np.uint16, kink_deltas=np.float32,
              U=np.uint16, S=np.float32, Vt=np.uint16)


class _Source:
    """A random packed model with the accessors of an open .gsd2 file."""

    def __init__(self, case, seed):
        from gsdlq import synth
        s = SHAPES[case["shape"]]
        if "layers" not in case:   # single-layer cases: the vocabulary plays no part
            s = dict(s, vocab=512)
        self.seed, self.kinks = int(seed), int(case["kinks"])
        spec = synth.SynthSpec(n_layers=case.get("layers", 1), mode=case["mode"], rms_eps=EPS, rope_theta=THETA, **s)
        self.config = synth.make_config(spec)
        self.header = {"avg_bpw": None}
        self.shape = dict(s)
        self.tensors = {n: dict(MODES[case["mode"]], rows=r, cols=c) for n, (r, c) in synth.tensor_shapes(spec).items()}
        self.names = list(self.tensors)
        self._last = (None, None)

    def fields(self, name):
        t = self.tensors[name]
        return _tensor(self.seed, 16 + self.names.index(name), t["rows"], t["cols"], t["radius"], t["k_dim"], self.kinks)

    def hex_field(self, name, field):
        if self._last[0] != name:
            self._last = (name, {k: v.cpu().numpy().reshape(-1).view(_FIELD[k]) for k, v in self.fields(name).items()})
        return self._last[1][field]

    def values(self, name):
        """A dense tensor on the GPU: the embedding in fp16, norms in float32."""
        if name == "token_embd.weight":
            return (SIGMA * _randn(_gen(self.seed, 1), self.shape["vocab"], self.shape["hidden"])).half()
        layer = 2 * int(name.split(".")[1]) + (".ffn_norm." in name) if name.startswith("blk.") else -1
        return 1 + 0.2 * _randn(_gen(self.seed, 1000 + layer), self.shape["hidden"])

    def dense(self, name, dtype):
        return self.values(name).cpu().numpy().view(dtype)

    def close(self):
        self._last = (None, None)


class _State:
    pass


def _model(case, seed, max_seq):
    import run_gpu_native_chat as chat
    src = _Source(case, seed)
    model = chat.GPUMistralV2Model(src, max_seq_len=max_seq, verbose=False)
    src.close()
    return src, model


def _tokens(seed, n, vocab):
    return np.random.default_rng((int(seed), 5)).integers(0, vocab, n).astype(np.int32)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _activations(seed, m, cols):
    """Rows as a norm or a SwiGLU leaves them: unit scale, a few columns far larger."""
    g = _gen(seed, 3)
    col = torch.exp(0.5 * _randn(g, cols))
    return (_randn(g, m, cols) * col).to(torch.bfloat16)


def _attention_inputs(case, seed, tokens, positions, layers):
    """Queries of `tokens` tokens and K/V caches filled to `positions`, for `layers` layers."""
    g = _gen(seed, 4)
    h, kv, hd = case["n_heads"], case["n_kv_heads"], case["head_dim"]
    q = 1.5 * _randn(g, layers, tokens, h, hd)
    kc = _randn(g, layers, positions, kv, hd).half()
    vc = _randn(g, layers, positions, kv, hd).half()
    return g, q, kc, vc


def prepare(case, seed):
    from gsdlq import hip
    s = _State()
    s.kind, s.lib = case["kind"], hip.lib()
    if s.kind in ("step", "prompt"):
        src, s.model = _model(case, seed, case["max_seq"])
        n0 = case["pos"] if s.kind == "step" else case["start"]
        ids = _tokens(seed, n0 + case.get("n", 1), src.shape["vocab"])
        s.before, s.ids, s.at = ids[:n0], ids[n0:], n0
        if n0:
            s.model.prefill(s.before, 0, return_logits=False)
    elif s.kind == "matmul":
        src, s.model = _model(case, seed, 16)
        names = SETS[case["tensors"]]
        shapes = [src.tensors[f"blk.0.{n}.weight"] for n in names]
        s.m, s.n = case["m"], len(names)
        s.stream = torch.cuda.ExternalStream(s.lib.gsdh_model_stream(s.model._m))
        s.x = _activations(seed, s.m, shapes[0]["cols"])
        s.y = [torch.empty(s.m, t["rows"], device="cuda") for t in shapes]
        s.slots = (ctypes.c_int * s.n)(*[hip.SLOTS[n] for n in names])
        s.out = (ctypes.c_void_p * s.n)(*[y.data_ptr() for y in s.y])
    elif s.kind == "attend":
        s.m, s.pos0 = case["m"], case["pos0"]
        _, q, s.kc, s.vc = _attention_inputs(case, seed, s.m, s.pos0 + s.m, 1)
        s.q, s.y = q[0], torch.empty_like(q[0])
        s.dims = (case["n_heads"], case["n_kv_heads"], case["head_dim"], s.pos0 + s.m)
        s.scale = 1.0 / math.sqrt(case["head_dim"])
    elif s.kind == "decode":
        g, q, s.kc, s.vc = _attention_inputs(case, seed, 1, case["ctx"], case["layers"])
        s.q, s.y = q[:, 0], torch.empty_like(q[:, 0])
        s.k, s.v = _randn(g, *s.kc[:, 0].shape), _randn(g, *s.kc[:, 0].shape)
        s.layers, s.pos = case["layers"], case["ctx"] - 1
        s.dims = (case["n_heads"], case["n_kv_heads"], case["head_dim"], case["ctx"])
        s.scale = 1.0 / math.sqrt(case["head_dim"])
    else:
        rows, cols, k = case["rows"], case["cols"], case["k_dim"]
        s.f = _tensor(seed, 2, rows, cols, case["radius"], k, case["kinks"])
        s.x = _activations(seed, 1, cols)[0].float()
        s.points = torch.from_numpy(_points(case["radius"])).cuda().float().contiguous()
        s.tmp, s.y = torch.empty(max(k, 1), device="cuda"), torch.empty(rows, device="cuda")
        s.rows, s.cols, s.k = rows, cols, k
    return s


def run(s):
    lib = s.lib
    if s.kind == "step":
        return s.model.forward_token(int(s.ids[0]), s.at)
    if s.kind == "prompt":
        return s.model.prefill(s.ids, s.at)
    if s.kind == "matmul":   # (on the model's stream, between what made its input and what reads its outputs)
        here = torch.cuda.current_stream()
        s.stream.wait_stream(here)
        lib.gsdh_model_matmul_shared(s.model._m, 0, s.slots, s.n, s.x.data_ptr(), s.m, s.out)
        here.wait_stream(s.stream)
        return s.y
    st = _stream()
    if s.kind == "attend":
        lib.gsdh_prefill_attention(st, s.q.data_ptr(), s.kc.data_ptr(), s.vc.data_ptr(), s.y.data_ptr(), 0, s.pos0, s.m,
                                   *s.dims, s.scale)
        return s.y
    if s.kind == "decode":
        qp, kp, vp, op = s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), s.y.data_ptr()
        kc, vc = s.kc.data_ptr(), s.vc.data_ptr()
        nq, nkv = 4 * s.q[0].numel(), 4 * s.k[0].numel()
        for layer in range(s.layers):
            lib.gsdh_rope_store_gqa_attention(st, qp + layer * nq, kp + layer * nkv, vp + layer * nkv, kc, vc,
                                              op + layer * nq, layer, s.pos, *s.dims, THETA, 1, s.scale)
        return {"out": s.y, "q": s.q, "k": s.kc[:, s.pos], "v": s.vc[:, s.pos]}
    f = s.f
    at = {k: v.data_ptr() if v.numel() else None for k, v in f.items()}
    if s.k:
        lib.gsdh_lowrank_proj(st, s.x.data_ptr(), at["Vt"], at["S"], s.tmp.data_ptr(), s.k, s.cols)
    lib.gsdh_hex2d_matvec(st, s.x.data_ptr(), at["codes"], at["scales"], s.points.data_ptr(), at.get("U"),
                          s.tmp.data_ptr(), at["row_ptr"], at["kink_cols"], at["kink_deltas"], s.y.data_ptr(),
                          s.rows, s.cols, s.k, len(s.points))
    return s.y


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far off a correct one may be
# ---------------------------------------------------------------------------
def _packed_bytes(rows, cols, radius, k_dim, kinks):
    codes = rows * cols // 2
    codes = (7 * codes + 7) // 8 if radius <= 6 else codes   # 127 points take seven bits
    return codes + rows * cols // 32 + 4 * (rows + 1) + 6 * rows * kinks + 2 * k_dim * (rows + cols) + 4 * k_dim


def work(case):
    if case["kind"] == "attend":
        h, kv, hd, m, p0 = case["n_heads"], case["n_kv_heads"], case["head_dim"], case["m"], case["pos0"]
        return dict(bytes=8 * m * h * hd + 4 * (p0 + m) * kv * hd, flops=4 * h * hd * (m * p0 + m * (m + 1) // 2))
    if case["kind"] == "decode":
        h, kv, hd, n, nl = case["n_heads"], case["n_kv_heads"], case["head_dim"], case["ctx"], case["layers"]
        return dict(bytes=nl * (12 * h * hd + 8 * kv * hd + 4 * n * kv * hd), flops=nl * 4 * h * hd * n)
    if case["kind"] == "matvec":
        r, c = case["rows"], case["cols"]
        return dict(bytes=_packed_bytes(r, c, case["radius"], case["k_dim"], case["kinks"]) + 4 * (r + c), flops=2 * r * c)
    s, mode, kinks = SHAPES[case["shape"]], MODES[case["mode"]], case["kinks"]
    hid, qd, kvd, hd = s["hidden"], s["n_heads"] * s["head_dim"], s["n_kv_heads"] * s["head_dim"], s["head_dim"]
    dims = dict(zip(LAYER, ((qd, hid), (kvd, hid), (kvd, hid), (hid, qd), (s["ffn"], hid), (s["ffn"], hid), (hid, s["ffn"]))))
    packed = lambda r, c: _packed_bytes(r, c, mode["radius"], mode["k_dim"], kinks)  # noqa: E731
    if case["kind"] == "matmul":
        ts, m = [dims[n] for n in SETS[case["tensors"]]], case["m"]
        return dict(bytes=sum(packed(*t) + 4 * m * t[0] for t in ts) + 2 * m * ts[0][1], flops=sum(2 * m * r * c for r, c in ts))
    m, p0 = (1, case["pos"]) if case["kind"] == "step" else (case["n"], case["start"])
    nl, vocab = case["layers"], s["vocab"]
    seen = m * p0 + m * (m + 1) // 2
    return dict(bytes=nl * (sum(packed(*t) for t in dims.values()) + 4 * kvd * (p0 + 2 * m) + 8 * hid)
                + packed(vocab, hid) + 2 * m * hid + 4 * vocab,
                flops=nl * (2 * m * sum(r * c for r, c in dims.values()) + 4 * s["n_heads"] * hd * seen) + 2 * vocab * hid)


def tolerance(case):
    # about four times what each path is off exact() over its range of sizes
    if case["kind"] == "matmul":    # 1.7e-4: one fp16 rounding of each input pair
        return {"rel": 7e-4, "max": 7e-3}
    if case["kind"] in ("step", "prompt"):   # 5e-5: fp32, and K/V elements that round to the other fp16 value
        return {"rel": 2e-4, "max": 2e-3}
    if case["kind"] == "decode":    # 5e-7, and more where an element of the appended row rounds the other way
        return {"rel": 2e-5, "max": 2e-3}
    return {"rel": 5e-6, "max": 1e-4}   # 1e-7 (matvec), 6e-7 (attention of a prompt)


# ---------------------------------------------------------------------------
# the oracle, in 64 bits
# ---------------------------------------------------------------------------
def _dense(f, rows, cols, radius, k_dim):
    pts = torch.from_numpy(_points(radius)).cuda()
    w = torch.empty(rows, cols, device="cuda", dtype=torch.float64)
    codes, scales = f["codes"].reshape(rows, -1), f["scales"].reshape(rows, -1, 1)
    for r in range(0, rows, 1024):   # (an index of all of a head's codes exceeds torch's grid)
        part = w[r:r + 1024].view(-1, cols // 64, 64)
        torch.mul(pts[codes[r:r + 1024].long()].reshape(part.shape), scales[r:r + 1024].double(), out=part)
    if f["kink_cols"].numel():
        per = f["kink_cols"].numel() // rows
        at = torch.from_numpy(f["kink_cols"].cpu().numpy().astype(np.int64)).cuda().reshape(rows, per)
        w.scatter_add_(1, at, f["kink_deltas"].double().reshape(rows, per))
    if k_dim:
        w += f["U"].double() @ (f["S"].double()[:, None] * f["Vt"].double())
    return w


def _angles(positions, hd):
    """cos and sin [positions, hd / 2] of the reference's float32 angles."""
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, (ctypes.c_float, ctypes.c_float)
    freq = np.array([np.float32(1.0) / np.float32(powf(THETA, np.float32(2 * i) / np.float32(hd))) for i in range(hd // 2)],
                    np.float32)
    a = torch.from_numpy(np.asarray(positions, np.float32)[:, None] * freq).cuda().double()
    return a.cos(), a.sin()


def _rotate(x, cs):
    """Interleaved RoPE of x [tokens, heads, hd]."""
    c, s = cs[0][:, None], cs[1][:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).reshape(x.shape)


def _attend(q, k, v, p0, scale):
    """Causal attention in 64 bits: q [m, h, hd] at positions p0.., k and v [ctx, kv, hd]."""
    m, h, _ = q.shape
    ctx, kv, _ = k.shape
    out = torch.empty_like(q)
    ahead = torch.arange(ctx, device="cuda")[None] > p0 + torch.arange(m, device="cuda")[:, None]
    for i in range(h):
        j = i // (h // kv)
        p = (q[:, i] @ k[:, j].T * scale).masked_fill_(ahead, -math.inf).softmax(1)
        out[:, i] = p @ v[:, j]
    return out


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _forward(case, seed):
    """The last token's logits of the whole context."""
    src = _Source(case, seed)
    s, mode = src.shape, MODES[case["mode"]]
    n0 = case["pos"] if case["kind"] == "step" else case["start"]
    ids = torch.from_numpy(_tokens(seed, n0 + case.get("n", 1), s["vocab"]).astype(np.int64)).cuda()
    n, hd = len(ids), s["head_dim"]
    w = lambda name: _dense(src.fields(name), src.tensors[name]["rows"], src.tensors[name]["cols"], mode["radius"], mode["k_dim"])  # noqa: E731
    x, cs = src.values("token_embd.weight")[ids].double(), _angles(range(n), hd)
    for layer in range(case["layers"]):
        p = f"blk.{layer}."
        y = _rms(x, src.values(p + "attn_norm.weight"))
        q = _rotate((y @ w(p + "attn_q.weight").T).reshape(n, -1, hd), cs)
        k = _rotate((y @ w(p + "attn_k.weight").T).reshape(n, -1, hd), cs).half().double()
        v = (y @ w(p + "attn_v.weight").T).reshape(n, -1, hd).half().double()
        x = x + _attend(q, k, v, 0, 1.0 / math.sqrt(hd)).reshape(n, -1) @ w(p + "attn_output.weight").T
        y = _rms(x, src.values(p + "ffn_norm.weight"))
        gate = y @ w(p + "ffn_gate.weight").T
        x = x + (gate / (1 + (-gate).exp()) * (y @ w(p + "ffn_up.weight").T)) @ w(p + "ffn_down.weight").T
    return w("output.weight") @ _rms(x[-1], src.values("output_norm.weight"))


def exact(case, seed):
    if case["kind"] in ("step", "prompt"):
        return _forward(case, seed)
    if case["kind"] == "matmul":
        src = _Source(case, seed)
        out = []
        for n in SETS[case["tensors"]]:
            t = src.tensors[f"blk.0.{n}.weight"]
            x = _activations(seed, case["m"], t["cols"]).double()
            out.append(x @ _dense(src.fields(f"blk.0.{n}.weight"), t["rows"], t["cols"], t["radius"], t["k_dim"]).T)
        return out
    if case["kind"] == "attend":
        _, q, kc, vc = _attention_inputs(case, seed, case["m"], case["pos0"] + case["m"], 1)
        return _attend(q[0].double(), kc[0].double(), vc[0].double(), case["pos0"], 1.0 / math.sqrt(case["head_dim"]))
    if case["kind"] == "decode":
        g, q, kc, vc = _attention_inputs(case, seed, 1, case["ctx"], case["layers"])
        k, v, pos = _randn(g, *kc[:, 0].shape), _randn(g, *kc[:, 0].shape), case["ctx"] - 1
        cs, out, qs = _angles([pos], case["head_dim"]), [], []
        for layer in range(case["layers"]):
            kc[layer, pos] = _rotate(k[layer][None].double(), cs)[0].half()
            vc[layer, pos] = v[layer].half()
            qs.append(_rotate(q[layer].double(), cs))
            out.append(_attend(qs[-1], kc[layer].double(), vc[layer].double(), pos, 1.0 / math.sqrt(case["head_dim"]))[0])
        return {"out": torch.stack(out), "q": torch.cat(qs), "k": None, "v": None}
    f = _tensor(seed, 2, case["rows"], case["cols"], case["radius"], case["k_dim"], case["kinks"])
    return _dense(f, case["rows"], case["cols"], case["radius"], case["k_dim"]) @ _activations(seed, 1, case["cols"])[0].double()
