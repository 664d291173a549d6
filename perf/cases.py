"""Performance cases of the framework: the calls its users make, through the
public entry points of parakeet_wgsl_amd.palette_abi, with seeded synthetic
inputs made on the GPU.

A case is a dict of plain values; `kind` says which entry points it goes
through:

  encoder   one pass of pk_encoder (fbank, subsampling, every layer, the
            projector), replayed from its graph: what a transcription service
            runs per batch of 15-second windows
  layer     pk_encoder over subsampled features without front end or
            projector: the FastConformer layer as a block
  decode    pk_tdt: the greedy TDT decode of a batch of windows
  ff        the feed-forward block: two palette GEMMs back to back
  mha       the relative-position attention block: QKV GEMM, the rel-pos
            linear over the sinusoid rows, attention, output GEMM + residual
  conv      the convolution module: pointwise 1 with the GLU epilogue, the
            depthwise tail, pointwise 2 + residual
  gemm      one palette GEMM
  stream    pk_gemm_group over all eight matrices of 24 layers: few rows, every
            weight read once

`f16` is the reference's default execution profile, `f32` its fp32 one.
"""
import math

import numpy as np
import torch

import parakeet_wgsl_amd.palette_abi as abi

FRAMES = 188        # encoder frames of a 15-second window (1501 fbank frames)
MAX_TOKENS = 1024   # token slots per window of the decoder
D, HIDDEN, HEADS = 1024, 4096, 8
# name: (bits, inner, columns, palette groups), the package's layer matrices
MATRICES = {
    "ff1_linear1": (5, 1024, 4096, 1), "ff1_linear2": (5, 4096, 1024, 1), "qkv": (5, 1024, 3072, 3),
    "o_proj": (6, 1024, 1024, 1), "pointwise1": (5, 1024, 2048, 1), "pointwise2": (5, 1024, 1024, 1),
    "ff2_linear1": (5, 1024, 4096, 1), "ff2_linear2": (5, 4096, 1024, 1),
}


def listed():
    return [
        # the service's full batch: 16 windows of 15 s through the whole encoder
        {"name": "encoder-16x15s", "kind": "encoder", "precision": "f16", "windows": 16, "frames": FRAMES,
         "layers": 24},
        # one live utterance: the same pass where every launch is small
        {"name": "encoder-1x15s", "kind": "encoder", "precision": "f16", "windows": 1, "frames": FRAMES,
         "layers": 24},
        # a layer of the fp32 profile at the full batch
        {"name": "layer-f32-16x188", "kind": "layer", "precision": "f32", "windows": 16, "frames": FRAMES,
         "layers": 1},
        # decoding the full batch's projector output
        {"name": "decode-16x188", "kind": "decode", "precision": "f16", "windows": 16, "frames": FRAMES},
        # decoding one live utterance
        {"name": "decode-1x188", "kind": "decode", "precision": "f16", "windows": 1, "frames": FRAMES},
        # decoding a small batch in the fp32 profile
        {"name": "decode-f32-4x188", "kind": "decode", "precision": "f32", "windows": 4, "frames": FRAMES},
        # the feed-forward block of 8 windows (half of a layer's GEMM work)
        {"name": "ff-1504", "kind": "ff", "precision": "f16", "rows": 1504},
        # attention over one-minute windows (quadratic part at its largest)
        {"name": "mha-4x750", "kind": "mha", "precision": "f16", "windows": 4, "frames": 750},
        # the convolution module at the full batch
        {"name": "conv-16x188", "kind": "conv", "precision": "f16", "windows": 16, "frames": FRAMES},
        # a single fp32 GEMM with bias, 6-bit
        {"name": "gemm-f32-256", "kind": "gemm", "precision": "f32", "rows": 256, "inner": 1024, "columns": 4096,
         "bits": 6, "activation": "none", "bias": True},
        # a single small GEMM: the launch-latency regime
        {"name": "gemm-f16-16", "kind": "gemm", "precision": "f16", "rows": 16, "inner": 1024, "columns": 4096,
         "bits": 5, "activation": "silu", "bias": False},
        # all encoder weights streamed once at few rows
        {"name": "stream-16", "kind": "stream", "precision": "f16", "rows": 16, "layers": 24},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["encoder", "layer", "decode", "decode", "ff", "ff", "mha", "conv", "gemm", "gemm", "stream"])
    precision = rng.choice(["f16", "f16", "f32"])
    if kind == "encoder":
        frames = rng.choice([rng.randint(94, FRAMES), _log_int(rng, 24, 400)])
        return {"kind": kind, "precision": "f16", "windows": _log_int(rng, 1, min(40, 3008 // frames)),
                "frames": frames, "layers": 24}
    if kind == "layer":
        frames = _log_int(rng, 24, 400)
        return {"kind": kind, "precision": precision, "windows": _log_int(rng, 1, max(1, 3008 // frames)),
                "frames": frames, "layers": rng.randint(1, 2)}
    if kind == "decode":
        return {"kind": kind, "precision": precision,
                "windows": _log_int(rng, 1, 16 if precision == "f32" else 40),
                "frames": rng.randint(40, FRAMES)}
    if kind == "ff":
        return {"kind": kind, "precision": precision,
                "rows": _log_int(rng, 8, 3008 if precision == "f32" else 7520)}
    if kind in ("mha", "conv"):
        frames = _log_int(rng, 24, 750)
        return {"kind": kind, "precision": precision, "windows": _log_int(rng, 1, max(1, 3008 // frames)),
                "frames": frames}
    if kind == "gemm":
        bits, inner, columns, _ = rng.choice([m for m in MATRICES.values() if m[3] == 1] +
                                             [(6, 1024, 4096, 1), (5, 1024, 640, 1), (5, 4096, 1024, 1)])
        return {"kind": kind, "precision": precision, "rows": _log_int(rng, 1, 3008), "inner": inner,
                "columns": columns, "bits": bits, "activation": rng.choice(["none", "silu", "relu"]),
                "bias": rng.random() < 0.5}
    return {"kind": "stream", "precision": "f16", "rows": _log_int(rng, 1, 188), "layers": rng.randint(4, 24)}


# ------------------------------------------------------------------ inputs

class Buffer:
    """A torch tensor as a device buffer of the ABI (pointer, bytes, numpy type)."""

    _TYPES = {torch.float16: np.float16, torch.float32: np.float32, torch.int32: np.uint32}

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr, self.nbytes = tensor.data_ptr(), tensor.numel() * tensor.element_size()
        self.dtype, self.shape = np.dtype(self._TYPES[tensor.dtype]), tuple(tensor.shape)


_context = None


def context():
    """The process's library context on the first GPU."""
    global _context
    if _context is None:
        torch.cuda.current_device()
        _context = abi.Context(0)
    return _context


class Inputs:
    """Seeded tensors of one case, made on the GPU."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = torch.float16 if case.get("precision", "f16") == "f16" else torch.float32

    def normal(self, *shape, std=1.0, mean=0.0, dtype=None):
        t = torch.randn(shape, generator=self.g, device="cuda") * std + mean
        return t.to(self.dtype if dtype is None else dtype)

    def vector(self, n, std, mean=0.0):
        return self.normal(n, std=std, mean=mean, dtype=torch.float32)

    def lengths(self, n, low, high):
        return torch.randint(low, high + 1, (n,), generator=self.g, device="cuda", dtype=torch.int32)

    def matrix(self, bits, inner, columns, groups=1, std=0.02, centred=False):
        """A palette matrix: uniform codes (every bit of the packed words is
        a code bit) and a LUT per palette group."""
        words = inner * columns * bits // 32
        packed = torch.randint(-2**31, 2**31, (words,), generator=self.g, device="cuda", dtype=torch.int64)
        lut = torch.randn((groups, 1 << bits), generator=self.g, device="cuda") * std
        if centred:  # these multiply ReLU outputs: a LUT mean would shift every output
            lut = lut - lut.mean()
        return packed.to(torch.int32), lut.to(self.dtype), (bits, inner, columns, groups)


def layer_weights(make, frames):
    w = {"norm_gamma": make.normal(5, D, std=0.1, mean=1.0, dtype=torch.float32),
         "norm_beta": make.normal(5, D, std=0.1, dtype=torch.float32)}
    for name, (bits, inner, columns, groups) in MATRICES.items():
        w[name] = make.matrix(bits, inner, columns, groups)
    w["positions"] = make.normal(2 * frames - 1, D, std=0.6)
    w["bias_u"] = make.normal(HEADS, 128, std=0.02, dtype=torch.float32)
    w["bias_v"] = make.normal(HEADS, 128, std=0.02, dtype=torch.float32)
    w["depthwise"] = make.normal(9, D, std=0.05)
    w["bn_scale"] = make.vector(D, 0.1, 1.0)
    w["bn_shift"] = make.vector(D, 0.1)
    return w


def front_weights(make):
    w = {}
    for conv in ("conv0", "depthwise2", "depthwise5"):
        w[conv + "_weights"] = make.normal(3, 3, 256, std=0.3)
        w[conv + "_bias"] = make.vector(256, 0.05)
    for name, inner, columns, std in (("pointwise3", 256, 256, 0.05), ("pointwise6", 256, 256, 0.05),
                                      ("linear", 4096, 1024, 0.08)):
        w[name] = make.matrix(5, inner, columns, std=std, centred=True)
        w[name + "_bias"] = make.vector(columns, 0.05)
    return w


def subsampled(n, steps):
    for _ in range(steps):
        n = (n + 1) // 2
    return n


def sinusoids(frames):
    """The Transformer-XL position rows: row p is relative distance frames - 1 - p."""
    at = torch.arange(frames - 1, -frames, -1, device="cuda", dtype=torch.float32)[:, None]
    rate = torch.exp(torch.arange(0, D, 2, device="cuda", dtype=torch.float32) * (-math.log(10000.0) / D))
    table = torch.empty(2 * frames - 1, D, device="cuda")
    table[:, 0::2], table[:, 1::2] = torch.sin(at * rate), torch.cos(at * rate)
    return table


def tensors_of(case, seed):
    """Every input tensor of a case, by name."""
    make, kind = Inputs(case, seed), case["kind"]
    if kind in ("encoder", "layer"):
        windows, frames = case["windows"], case["frames"]
        t = {"layers": [layer_weights(make, frames) for _ in range(case["layers"])]}
        if kind == "encoder":
            feature_frames = 8 * frames - 3
            t["input"] = make.normal(windows, 128, feature_frames, dtype=torch.float32)
            t["feature_lengths"] = make.lengths(windows, (feature_frames + 1) // 2, feature_frames)
            t["valid"] = subsampled(t["feature_lengths"], 3).to(torch.int32)
            t["front"] = front_weights(make)
            t["projector"], t["projector_bias"] = make.matrix(5, D, 640), make.vector(640, 0.01)
        else:
            t["input"] = make.normal(windows * frames, D)
            t["valid"] = make.lengths(windows, (frames + 1) // 2, frames)
        return t
    if kind == "decode":
        windows, frames = case["windows"], case["frames"]
        head, head_bias = make.normal(640, 1032, std=0.05), make.vector(1032, 0.1)
        head[:, 1030:] = 0
        head_bias[1024] += 2.0  # random heads otherwise hardly ever choose blank
        head_bias[1030:] = 0
        weights = {"embedding": make.normal(1025, 640, std=0.5), "head_weight": head, "head_bias": head_bias,
                   "lstm_weight_l0": make.normal(1280, 2560, std=0.03), "lstm_bias_l0": make.vector(2560, 0.1),
                   "lstm_weight_l1": make.normal(1280, 2560, std=0.03), "lstm_bias_l1": make.vector(2560, 0.1),
                   "projector_weight": make.normal(640, 640, std=0.04), "projector_bias": make.vector(640, 0.1)}
        return {"weights": weights, "encoder_projected": make.normal(windows, frames, 640, std=0.5),
                "encoded_lengths": make.lengths(windows, (frames + 1) // 2, frames)}
    if kind == "ff":
        return {"x": make.normal(case["rows"], D), "w1": make.matrix(5, D, HIDDEN), "w2": make.matrix(5, HIDDEN, D)}
    if kind == "mha":
        windows, frames = case["windows"], case["frames"]
        return {"x": make.normal(windows * frames, D), "wqkv": make.matrix(6, D, 3 * D, 3),
                "wpos": make.matrix(6, D, D), "wo": make.matrix(6, D, D),
                "table": sinusoids(frames).to(make.dtype), "bias_u": make.vector(D, 0.02), "bias_v": make.vector(D, 0.02),
                "valid": make.lengths(windows, (frames + 1) // 2, frames)}
    if kind == "conv":
        windows, frames = case["windows"], case["frames"]
        return {"x": make.normal(windows * frames, D), "pw1": make.matrix(6, D, 2 * D), "pw2": make.matrix(6, D, D),
                "depthwise": make.normal(9, D, std=0.05), "scale": make.vector(D, 0.1, 1.0),
                "shift": make.vector(D, 0.1), "valid": make.lengths(windows, (frames + 1) // 2, frames)}
    if kind == "gemm":
        return {"x": make.normal(case["rows"], case["inner"]),
                "w": make.matrix(case["bits"], case["inner"], case["columns"]),
                "bias": make.vector(case["columns"], 0.01) if case["bias"] else None}
    if kind == "stream":
        return {"x": {k: make.normal(case["rows"], k) for k in (D, HIDDEN)},
                "layers": [{n: make.matrix(*m) for n, m in MATRICES.items()} for _ in range(case["layers"])]}
    raise ValueError(kind)


# ----------------------------------------------------------------- passes

class State:
    """What a user's program holds between calls: buffers and library objects."""

    def __init__(self):
        self.objects, self.keep, self.steps, self.outputs = [], [], [], {}

    def buf(self, tensor):
        b = Buffer(tensor)
        self.keep.append(b)
        return b

    def new(self, *shape, dtype):
        return self.buf(torch.zeros(shape, dtype=dtype, device="cuda"))

    def own(self, obj):
        self.objects.append(obj)
        return obj

    def gemm(self, a, matrix, out, **more):
        packed, lut, (bits, inner, columns, _) = matrix
        return self.own(abi.GemmOp(context(), a=a, packed=self.buf(packed), palette=self.buf(lut), output=out,
                                   bits=bits, rows=a.shape[0], inner=inner, columns=columns, **more))

    def __del__(self):
        torch.cuda.synchronize()
        for obj in reversed(self.objects):
            obj.release()


def _encoder(s, case, t):
    windows, frames = case["windows"], case["frames"]
    dtype = torch.float16 if case["precision"] == "f16" else torch.float32
    put = s.buf

    def mat(m):
        return put(m[0]), put(m[1])
    layers = []
    for w in t["layers"]:
        d = {n: mat(w[n]) for n in MATRICES}
        for n in ("norm_gamma", "norm_beta"):
            d[n] = [put(row) for row in w[n]]
        d["projected_positions"] = put(w["positions"].reshape(-1, HEADS, 32, 4).permute(1, 2, 0, 3).contiguous())
        for n in ("bias_u", "bias_v", "depthwise", "bn_scale", "bn_shift"):
            d[n] = put(w[n])
        layers.append(d)
    out = s.new(windows * frames, D, dtype=dtype)
    s.outputs = {"output": out.tensor}
    more = {}
    if case["kind"] == "encoder":
        projected = s.new(windows * frames, 640, dtype=dtype)
        s.outputs["projected"] = projected.tensor
        front = {n: mat(v) if isinstance(v, tuple) else put(v) for n, v in t["front"].items()}
        more = dict(subsampling=front, feature_frames=8 * frames - 3, feature_lengths=put(t["feature_lengths"]),
                    projector=mat(t["projector"]), projector_bias=put(t["projector_bias"]),
                    projected_output=projected, projected_channels=640)
    op = s.own(abi.EncoderOp(context(), layers=layers, valid_lengths=put(t["valid"]), input=put(t["input"]),
                             output=out, batch_size=windows, frames=frames, precision=case["precision"], **more))
    s.steps = [lambda: op.enqueue(graph=True)]


def _decode(s, case, t):
    windows, frames = case["windows"], case["frames"]

    def u32(*shape, value=0):
        return s.buf(torch.full(shape, value, dtype=torch.int32, device="cuda"))
    outs = {"tokens": u32(windows, MAX_TOKENS), "token_frames": u32(windows, MAX_TOKENS),
            "token_durations": u32(windows, MAX_TOKENS), "metadata": u32(2 * windows),
            "state": s.new(windows, 4, 640, dtype=torch.float32),
            "predictor_scratch": s.new(windows, 5, 640, dtype=torch.float32)}
    op = s.own(abi.TdtDecoderOp(context(), weights={n: s.buf(w) for n, w in t["weights"].items()},
                                encoder_projected=s.buf(t["encoder_projected"]),
                                encoded_lengths=s.buf(t["encoded_lengths"]), decode_starts=u32(windows),
                                decode_ends=u32(windows, value=frames), flush_finals=u32(windows, value=1),
                                batch_size=windows, frames=frames, max_tokens=MAX_TOKENS,
                                precision=case["precision"], **outs))
    s.outputs = {n: b.tensor for n, b in outs.items()}
    s.steps = [op.enqueue]


def _blocks(s, case, t):
    kind, dtype = case["kind"], torch.float16 if case["precision"] == "f16" else torch.float32
    f16 = dtype == torch.float16
    if kind == "ff":
        x, h, y = s.buf(t["x"]), s.new(case["rows"], HIDDEN, dtype=dtype), s.new(case["rows"], D, dtype=dtype)
        expand = s.gemm(x, t["w1"], h, activation="silu")
        contract = s.gemm(h, t["w2"], y, residual=x, residual_scale=0.5)
        s.steps, s.outputs = [expand.enqueue, contract.enqueue], {"hidden": h.tensor, "output": y.tensor}
    elif kind == "mha":
        windows, frames = case["windows"], case["frames"]
        rows = windows * frames
        x, qkv = s.buf(t["x"]), s.new(rows, 3 * D, dtype=dtype)
        positions = s.new(2 * frames - 1, D, dtype=dtype)
        ctx, y = s.new(rows, D, dtype=dtype), s.new(rows, D, dtype=dtype)
        first = s.gemm(x, t["wqkv"], qkv)
        linear = s.gemm(s.buf(t["table"]), t["wpos"], positions)
        attention = s.own(abi.RelativeAttentionOp(
            context(), qkv=qkv, projected_positions=positions, bias_u=s.buf(t["bias_u"]), bias_v=s.buf(t["bias_v"]),
            valid_lengths=s.buf(t["valid"]), output=ctx, batch_size=windows, frames=frames,
            positions_row_major=True))
        last = s.gemm(ctx, t["wo"], y, residual=x, residual_scale=1.0)
        s.steps = [first.enqueue, linear.enqueue, attention.enqueue, last.enqueue]
        s.outputs = {"context": ctx.tensor, "output": y.tensor}
    elif kind == "conv":
        windows, frames = case["windows"], case["frames"]
        rows = windows * frames
        x, p = s.buf(t["x"]), s.new(rows, D if f16 else 2 * D, dtype=dtype)
        z, y = s.new(rows, D, dtype=dtype), s.new(rows, D, dtype=dtype)
        first = s.gemm(x, t["pw1"], p, glu=f16)  # the GLU epilogue is the f16 profile's
        tail = s.own(abi.ConformerConvOp(
            context(), pointwise_input=p, depthwise_weights=s.buf(t["depthwise"]),
            batch_norm_scale=s.buf(t["scale"]), batch_norm_shift=s.buf(t["shift"]), valid_lengths=s.buf(t["valid"]),
            output=z, batch_size=windows, frames=frames, input_glu=f16))
        last = s.gemm(z, t["pw2"], y, residual=x, residual_scale=1.0)
        s.steps = [first.enqueue, tail.enqueue, last.enqueue]
        s.outputs = {"conv": z.tensor, "output": y.tensor}
    elif kind == "gemm":
        y = s.new(case["rows"], case["columns"], dtype=dtype)
        op = s.gemm(s.buf(t["x"]), t["w"], y, activation=case["activation"],
                    bias=s.buf(t["bias"]) if case["bias"] else None)
        s.steps, s.outputs = [op.enqueue], {"output": y.tensor}
    else:
        x = {k: s.buf(v) for k, v in t["x"].items()}
        rows, total = case["rows"], sum(m[2] for m in MATRICES.values())
        whole = torch.zeros(case["layers"], total * rows, dtype=dtype, device="cuda")
        ops = []
        for layer, out in zip(t["layers"], whole):
            at = 0
            for n, (_, inner, columns, _) in MATRICES.items():
                y = s.buf(out[at:at + rows * columns].view(rows, columns))
                ops.append(s.gemm(x[inner], layer[n], y))
                at += rows * columns
        group = s.own(abi.GemmGroup(context(), ops))
        s.steps, s.outputs = [group.enqueue], {"outputs": whole}


def prepare(case, seed):
    s = State()
    t = tensors_of(case, seed)
    {"encoder": _encoder, "layer": _encoder, "decode": _decode}.get(case["kind"], _blocks)(s, case, t)
    s.keep.append(t)
    torch.cuda.synchronize()  # the library's stream starts after the inputs are there
    context().synchronize()
    return s


def run(state):
    for step in state.steps:
        step()
    return state.outputs


# ------------------------------------------------------------------- work

def _gemm_work(rows, inner, columns, bits, groups, e, residual=False):
    return (2 * rows * inner * columns,
            inner * columns * bits / 8 + groups * 2**bits * e + rows * (inner + columns * (2 if residual else 1)) * e)


def work(case):
    kind, e = case["kind"], 2 if case["precision"] == "f16" else 4
    if kind in ("encoder", "layer"):
        windows, frames, layers = case["windows"], case["frames"], case["layers"]
        rows = windows * frames
        weights = sum(k * n * b / 8 for b, k, n, _ in MATRICES.values()) + (2 * frames - 1) * D * e
        # mean valid length 3/4 of the frames: three products per live key
        attention = windows * (0.5833 * frames * frames) * D * 2 * 3
        flops = layers * (sum(2 * rows * k * n for _, k, n, _ in MATRICES.values()) + attention)
        nbytes = layers * weights + 2 * rows * D * e
        if kind == "encoder":
            f = 8 * frames - 3
            h1, h2 = subsampled(f, 1), subsampled(f, 2)
            flops += 2 * 9 * 256 * windows * (h1 * 64 + h2 * 32 + frames * 16)
            flops += 2 * windows * (h2 * 32 + frames * 16) * 256 * 256 + 2 * rows * 4096 * D + 2 * rows * D * 640
            nbytes += windows * 128 * f * 4 + (4096 * D + D * 640) * 5 / 8 + rows * 640 * e - rows * D * e
        return {"bytes": nbytes, "flops": flops}
    if kind == "decode":
        windows, frames = case["windows"], case["frames"]
        # about 0.3 tokens and 0.6 joint steps per frame with these weights
        joint, predictor = 2 * 640 * 1032, 2 * (2 * 1280 * 2560 + 640 * 640)
        flops = windows * frames * (0.6 * joint + 0.3 * predictor)
        nbytes = (1025 * 640 + 2 * 1280 * 2560 + 640 * 640 + 640 * 1032) * e + windows * (frames * 640 * e + 9 * 640 * 4)
        return {"bytes": nbytes, "flops": flops}
    if kind == "stream":
        parts = [_gemm_work(case["rows"], k, n, b, g, e) for b, k, n, g in MATRICES.values()]
        return {"flops": case["layers"] * sum(p[0] for p in parts), "bytes": case["layers"] * sum(p[1] for p in parts)}
    if kind == "gemm":
        f, b = _gemm_work(case["rows"], case["inner"], case["columns"], case["bits"], 1, e)
        return {"flops": f, "bytes": b}
    if kind == "ff":
        rows = case["rows"]
        parts = [_gemm_work(rows, D, HIDDEN, 5, 1, e), _gemm_work(rows, HIDDEN, D, 5, 1, e)]
        return {"flops": sum(p[0] for p in parts), "bytes": sum(p[1] for p in parts)}
    rows, frames = case["windows"] * case["frames"], case["frames"]
    if kind == "mha":
        parts = [_gemm_work(rows, D, 3 * D, 6, 3, e), _gemm_work(2 * frames - 1, D, D, 6, 1, e),
                 _gemm_work(rows, D, D, 6, 1, e)]
        attention = case["windows"] * (0.5833 * frames * frames) * D * 2 * 3
        return {"flops": sum(p[0] for p in parts) + attention, "bytes": 3 * D * D * 2 * 6 / 8 + 3 * rows * D * e}
    return {"flops": 2 * rows * D * 3 * D + rows * D * 9 * 2, "bytes": 3 * D * D * 6 / 8 + 3 * rows * D * e}


def tolerance(case):
    kind, f16 = case["kind"], case["precision"] == "f16"
    if kind == "decode":
        return "exact"  # tokens, and the state that the token sequence fixes to the bit
    if kind == "encoder":
        return {"rel": 1e-2}  # f16 activations through 24 layers: each side is 2e-3 from 64 bits
    return {"rel": 2e-3 if f16 else 1e-5}


# ------------------------------------------------------------------ exact

def dense(matrix):
    """The float64 [inner, columns] matrix of a palette matrix: codes LSB first
    in little-endian words, 32 codes in 5 words or 16 codes in 3."""
    packed, lut, (bits, inner, columns, groups) = matrix
    per, words = {5: (32, 5), 6: (16, 3)}[bits]
    w = packed.to(torch.int64).reshape(-1, words) & 0xFFFFFFFF
    w = torch.cat([w, torch.zeros_like(w[:, :1])], 1)
    codes = [((w[:, i * bits // 32] | w[:, i * bits // 32 + 1] << 32) >> (i * bits % 32)) & ((1 << bits) - 1)
             for i in range(per)]
    codes = torch.stack(codes, 1).reshape(inner, columns)
    group = torch.clamp(torch.arange(columns, device="cuda") // (columns // groups), max=groups - 1)
    return lut.double().reshape(-1)[codes + group[None, :] * (1 << bits)]


def _silu(v):
    return v * torch.sigmoid(v)


def _norm(x, gamma, beta):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), gamma.double(), beta.double(), 1e-5)


def _attend(qkv, positions, bias_u, bias_v, valid, windows, frames):
    x = qkv.reshape(windows, frames, 3, HEADS, 128).permute(2, 0, 3, 1, 4)      # [3, B, H, T, 128]
    pos = positions.reshape(2 * frames - 1, HEADS, 128).permute(1, 2, 0).contiguous()
    at = torch.arange(frames, device="cuda")
    index = frames - 1 - at[:, None] + at[None, :]
    u, v = (b.double().reshape(HEADS, 1, 128) for b in (bias_u, bias_v))
    out = torch.zeros(windows, frames, HEADS, 128, dtype=torch.float64, device="cuda")
    for b in range(windows):
        n = int(valid[b])
        q, k, val = x[0, b], x[1, b], x[2, b]
        near = torch.matmul(q + u, k.transpose(1, 2).contiguous())
        far = torch.matmul(q + v, pos).gather(2, index.expand(HEADS, frames, frames))
        p = torch.softmax(((near + far) / math.sqrt(128.0))[:, :n, :n], -1)
        out[b, :n] = torch.matmul(p, val[:, :n].contiguous()).permute(1, 0, 2)
    return out.reshape(windows * frames, D)


def _conv_tail(pointwise, depthwise, scale, shift, valid, windows, frames):
    glu = pointwise[:, :D] * torch.sigmoid(pointwise[:, D:])
    live = torch.arange(frames, device="cuda")[None, :] < valid[:, None]
    glu = torch.nn.functional.pad(glu.reshape(windows, frames, D) * live[:, :, None], (0, 0, 4, 4))
    y = sum(glu[:, tap:tap + frames] * depthwise[tap].double() for tap in range(9))
    return _silu(y * scale.double() + shift.double()).reshape(windows * frames, D)


def _layer(x, w, valid, windows, frames):
    def lin(a, name):
        return a @ dense(w[name])

    def norm(a, i):
        return _norm(a, w["norm_gamma"][i], w["norm_beta"][i])
    x = x + 0.5 * lin(_silu(lin(norm(x, 0), "ff1_linear1")), "ff1_linear2")
    c = _attend(lin(norm(x, 1), "qkv"), w["positions"].double(), w["bias_u"], w["bias_v"], valid, windows, frames)
    x = x + lin(c, "o_proj")
    c = _conv_tail(lin(norm(x, 2), "pointwise1"), w["depthwise"], w["bn_scale"], w["bn_shift"], valid, windows, frames)
    x = x + lin(c, "pointwise2")
    x = x + 0.5 * lin(_silu(lin(norm(x, 3), "ff2_linear1")), "ff2_linear2")
    return norm(x, 4)


def _front(t, windows):
    """[windows * frames, 1024] of the fbank; every stage is channel-last [B, time, bins, C]."""
    w, lengths = t["front"], t["feature_lengths"].to(torch.int64)

    def masked(a, steps):
        live = torch.arange(a.shape[1], device="cuda")[None, :] < subsampled(lengths, steps)[:, None]
        return a * live[:, :, None, None]

    def conv(a, name):
        rows, bins = subsampled(a.shape[1], 1), subsampled(a.shape[2], 1)
        a = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        y = w[name + "_bias"].double().expand(windows, rows, bins, 256).clone()
        for ky in range(3):
            for kx in range(3):
                part = a[:, ky:ky + 2 * rows - 1:2, kx:kx + 2 * bins - 1:2]
                y += part * w[name + "_weights"][ky, kx].double()
        return y

    def point(a, name):
        return torch.relu(a @ dense(w[name]) + w[name + "_bias"].double())
    a = t["input"].double().permute(0, 2, 1)[..., None]
    a = masked(torch.relu(conv(a, "conv0")), 1)
    a = point(masked(conv(a, "depthwise2"), 2), "pointwise3")
    a = masked(point(masked(conv(masked(a, 2), "depthwise5"), 3), "pointwise6"), 3)
    return a.reshape(-1, 4096) @ dense(w["linear"]) + w["linear_bias"].double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return None  # one token that 64 bits choose differently changes all that follows
    t = tensors_of(case, seed)
    if kind in ("encoder", "layer"):
        windows, frames = case["windows"], case["frames"]
        x = _front(t, windows) if kind == "encoder" else t["input"].double()
        for w in t["layers"]:
            x = _layer(x, w, t["valid"], windows, frames)
        if kind == "layer":
            return {"output": x}
        return {"output": x, "projected": x @ dense(t["projector"]) + t["projector_bias"].double()}
    if kind == "ff":
        x = t["x"].double()
        h = _silu(x @ dense(t["w1"]))
        return {"hidden": h, "output": x + 0.5 * (h @ dense(t["w2"]))}
    if kind == "mha":
        x = t["x"].double()
        c = _attend(x @ dense(t["wqkv"]), t["table"].double() @ dense(t["wpos"]), t["bias_u"], t["bias_v"],
                    t["valid"], case["windows"], case["frames"])
        return {"context": c, "output": x + c @ dense(t["wo"])}
    if kind == "conv":
        x = t["x"].double()
        z = _conv_tail(x @ dense(t["pw1"]), t["depthwise"], t["scale"], t["shift"], t["valid"], case["windows"],
                       case["frames"])
        return {"conv": z, "output": x + z @ dense(t["pw2"])}
    if kind == "gemm":
        y = t["x"].double() @ dense(t["w"])
        if case["bias"]:
            y = y + t["bias"].double()
        return {"output": {"none": lambda v: v, "silu": _silu, "relu": torch.relu}[case["activation"]](y)}
    x = {k: v.double() for k, v in t["x"].items()}
    rows = [torch.cat([(x[MATRICES[n][1]] @ dense(m)).reshape(-1) for n, m in layer.items()]) for layer in t["layers"]]
    return {"outputs": torch.stack(rows)}
