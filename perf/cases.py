"""Performance cases of the quantized-weight matmul path: what a program that runs models on this library has it do.

Every case goes through the public Python binding (`oxinfer_amd.HipBackend`), on weights of the formats and shapes of the
repository's benchmark and tests (Llama-8B-like layers, a 128-expert MoE layer, the 7168 x 18432 FP8 matrix). Five paths:

  matvec   one matrix alone at decode size: quantize the input, run the decode kernel (a head, a projection on its own)
  layer    one decode step over a few dense layers, recorded once as a plan and replayed for every step, as a decode loop
           does: norm + quantize, q / k / v in one batch, output projection (residual add), norm + quantize, gate / up pair,
           quantize, down projection (residual add)
  gemm     prefill: a matrix (or an MLP's up and down matrices) over many tokens on the matrix cores
  moe      routing and the routed experts of one MoE layer in one call
  host     the `Backend` surface: host activations in, host results out, several matrices sharing one input
"""
import ctypes

import numpy as np
import torch

from oxinfer_amd import HipBackend, hip

DEV = "cuda"
# stored bits per weight
BITS = {"mlx4": 4.5, "q4_0": 4.5, "q8_0": 8.5, "q4_k": 4.5, "q5_k": 5.5, "q6_k": 6.5625, "mxfp4": 4.25, "nvfp4": 4.5, "fp8": 8.0, "bf16": 16.0}
GGML = {"q4_0": hip.GGML_Q4_0, "q8_0": hip.GGML_Q8_0, "q4_k": hip.GGML_Q4_K, "q5_k": hip.GGML_Q5_K, "q6_k": hip.GGML_Q6_K, "mxfp4": hip.GGML_MXFP4}
FLOAT_STORED = ("fp8", "nvfp4", "bf16")  # decode takes f32 rows
# a layer's formats: (most matrices, the v and down projections), as quantized files mix them
MIXES = {"q4_k_m": ("q4_k", "q6_k"), "q5_k_m": ("q5_k", "q6_k"), "q6_k": ("q6_k", "q6_k"), "q8_0": ("q8_0", "q8_0"), "mlx4": ("mlx4", "mlx4"),
         "q4_0": ("q4_0", "q4_0"), "mxfp4": ("mxfp4", "mxfp4")}
VARIANT = {"bf16": 0, "i8": 1, "fp8": 2}

_shared = {}


def backend():
    """One backend per process, as a program keeps it."""
    if "be" not in _shared:
        _shared["be"] = HipBackend(0)
    return _shared["be"]


def decode_stream():
    """The stream of the decode loop (a plan records on a stream of its own)."""
    if "stream" not in _shared:
        _shared["stream"] = torch.cuda.Stream()
    return _shared["stream"]


def listed():
    return [
        # the smallest call: one 4096 x 4096 projection for one token; latency and launches are what counts
        dict(name="matvec_mlx4_t1", path="matvec", fmt="mlx4", n_out=4096, n_in=4096, t=1),
        # single-stream chat: a token through two Llama-8B layers of a Q4_K_M file
        dict(name="layer_q4_k_m_t1", path="layer", mix="q4_k_m", h=4096, kv=1024, inter=14336, layers=2, t=1),
        # a server decoding eight sequences together on Q8_0 weights
        dict(name="layer_q8_0_t8", path="layer", mix="q8_0", h=4096, kv=1024, inter=14336, layers=2, t=8),
        # the widest decode step (16 sequences) on MLX 4-bit weights
        dict(name="layer_mlx4_t16", path="layer", mix="mlx4", h=4096, kv=1024, inter=14336, layers=2, t=16),
        # FP8 block-scaled weights, a batch of 32 sequences: still one pass over the weights
        dict(name="fp8_t32", path="gemm", fmt="fp8", n_out=7168, n_in=18432, both=False, t=32, x="bf16", y="bf16", variant="bf16"),
        # a short ragged prompt over a matrix of odd height, Q6_K
        dict(name="gemm_q6_k_t43", path="gemm", fmt="q6_k", n_out=5001, n_in=4352, both=False, t=43, x="f32", y="f32", variant="bf16"),
        # an ordinary prompt: an MLP's two matrices over 512 tokens
        dict(name="gemm_mlx4_t512", path="gemm", fmt="mlx4", n_out=14336, n_in=4096, both=True, t=512, x="bf16", y="f32", variant="bf16"),
        # a long prompt, or one chunk of it: 2048 tokens over a Q4_K file's MLP
        dict(name="gemm_q4_k_t2048", path="gemm", fmt="q4_k", n_out=14336, n_in=4096, both=True, t=2048, x="f32", y="f32", variant="bf16"),
        # MoE decode of one token
        dict(name="moe_mlx4_t1", path="moe", fmt="mlx4", experts=128, k=8, h=2048, inter=768, t=1),
        # MoE decode of a batch of 24 sequences: most experts are touched, by one or two rows each
        dict(name="moe_mlx4_t24", path="moe", fmt="mlx4", experts=128, k=8, h=2048, inter=768, t=24),
        # MoE prefill
        dict(name="moe_mlx4_t256", path="moe", fmt="mlx4", experts=128, k=8, h=2048, inter=768, t=256),
        # the Backend surface: a 512-token prompt through gate and up, activations in and results out over the host link
        dict(name="host_q4_k_t512", path="host", fmt="q4_k", n_out=14336, n_in=4096, jobs=2, t=512),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["matvec", "layer", "layer", "layer", "gemm", "gemm", "gemm", "gemm", "moe", "moe", "moe", "host"])
    if path == "matvec":
        fmt = rng.choice(list(BITS))
        return dict(path=path, fmt=fmt, n_out=_log_int(rng, 512, 32003), n_in=256 * rng.randint(4, 56), t=rng.choice([1, 1, 2, 4, 8, rng.randint(1, 16)]))
    if path == "layer":
        h = 256 * rng.randint(6, 20)
        return dict(path=path, mix=rng.choice(list(MIXES)), h=h, kv=rng.choice([h // 4, 128 * rng.randint(2, 8)]), inter=256 * rng.randint(16, 56),
                    layers=rng.randint(1, 3), t=rng.choice([1, 1, 2, 4, 8, 16, rng.randint(1, 16)]))
    if path == "gemm":
        fmt = rng.choice(["mlx4", "mlx4", "q4_k", "q4_k", "q6_k", "q8_0", "q5_k", "q4_0", "mxfp4", "nvfp4", "fp8", "fp8"])
        n_out, n_in = rng.choice([(14336, 4096), (4096, 14336), (_log_int(rng, 1000, 14336), 128 * rng.randint(16, 112))])
        if fmt in ("q4_k", "q5_k", "q6_k"):
            n_in = n_in // 256 * 256
        if fmt == "fp8":
            n_out, n_in = rng.choice([(7168, 18432), (n_out, n_in)])
        t = min(_log_int(rng, 17, 2048), 2048 * 14336 * 4096 // (n_out * n_in))
        variant = "bf16"
        if fmt in ("mlx4", "fp8") and rng.random() < 0.2:
            variant = "i8" if fmt == "mlx4" else "fp8"
            t = min(t, 512)
        return dict(path=path, fmt=fmt, n_out=n_out, n_in=n_in, both=False, t=t, x=rng.choice(["bf16", "f32"]), y=rng.choice(["bf16", "f32"]), variant=variant)
    if path == "moe":
        h, inter = rng.choice([(2048, 768), (2048, 768), (128 * rng.randint(8, 24), 128 * rng.randint(3, 12))])
        fmt = rng.choice(["mlx4", "mlx4", "mlx4", "q4_k", "q8_0", "q4_0", "mxfp4"])
        if fmt == "q4_k":
            h, inter = h // 256 * 256, inter // 256 * 256
        return dict(path=path, fmt=fmt, experts=rng.choice([128, 128, 64, 32]), k=rng.choice([8, 8, 4, 6]), h=h, inter=inter,
                    t=rng.choice([1, _log_int(rng, 1, 256), _log_int(rng, 2, 256)]))
    return dict(path=path, fmt=rng.choice(["q4_k", "mlx4", "q8_0", "q6_k"]), n_out=256 * rng.randint(4, 56), n_in=256 * rng.randint(4, 16),
                jobs=rng.randint(1, 3), t=_log_int(rng, 1, 340))


# ---- weights, made on the device and handed over from the host as a loader does -----------------------------------------


class Gen:
    """Seeded random tensors with the distributions of the benchmark's weights (uniform codes, |N| scales), centred."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=self.g)

    def normal(self, *shape):
        return torch.randn(shape, device=DEV, generator=self.g)

    def half_bytes(self, n, sd, signed=False):
        v = self.normal(n) * sd
        return (v if signed else v.abs()).to(torch.float16).view(torch.uint8).reshape(n, 2)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, dtype=torch.int32, device=DEV, generator=self.g)

    def k4_header(self, nb, mid):
        """d, dmin and the twelve packed bytes of eight 6-bit (scale, min) pairs; the mins centre the codes (about `mid` on
        average), so that the weights have no common mean, as those of a model have none."""
        sc = self.ints(0, 64, nb, 8)
        mn = (sc + self.ints(-2, 3, nb, 8)).clamp_(0, 63)
        d = (self.normal(nb).abs() * 0.005).to(torch.float16)
        dmin = (d.float() * mid).to(torch.float16)
        packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
        return torch.cat([v.view(torch.uint8).reshape(nb, 2) for v in (d, dmin)] + [packed.to(torch.uint8)], 1)

    def mlx4(self, n_out, n_in, group=64):
        w = self.bytes(n_out, n_in // 2)
        s = (self.normal(n_out, n_in // group).abs() * (0.02 / 7.5)).to(torch.bfloat16)
        return [w.cpu().numpy().view(np.uint32)] + [v.view(torch.int16).cpu().numpy().view(np.uint16) for v in (s, s * -7.5)]

    def blocks(self, fmt, n_out, n_in):
        n = n_out * n_in
        if fmt == "q4_0":
            b = torch.cat([self.half_bytes(n // 32, 0.01), (self.ints(1, 16, n // 32, 16) | self.ints(1, 16, n // 32, 16) << 4).to(torch.uint8)], 1)
        elif fmt == "q8_0":
            b = torch.cat([self.half_bytes(n // 32, 0.01), self.ints(-127, 128, n // 32, 32).to(torch.int8).view(torch.uint8)], 1)
        elif fmt in ("q4_k", "q5_k"):
            b = torch.cat([self.k4_header(n // 256, 7.5 if fmt == "q4_k" else 15.5), self.bytes(n // 256, 128 if fmt == "q4_k" else 160)], 1)
        elif fmt == "q6_k":
            b = torch.cat([self.bytes(n // 256, 208), self.half_bytes(n // 256, 0.005, signed=True)], 1)
        elif fmt == "mxfp4":
            b = torch.cat([self.ints(116, 124, n // 32, 1).to(torch.uint8), self.bytes(n // 32, 16)], 1)
        else:  # nvfp4: four unsigned e4m3 scales, then the codes
            b = torch.cat([(self.ints(0, 7, n // 64, 4) << 3 | self.ints(0, 8, n // 64, 4)).to(torch.uint8), self.bytes(n // 64, 32)], 1)
        return b.reshape(-1).cpu().numpy()

    def upload(self, fmt, n_out, n_in):
        be = backend()
        if fmt == "mlx4":
            w = be.upload_mlx_q4(*self.mlx4(n_out, n_in), 64, n_out, n_in)
        elif fmt == "fp8":
            data = self.normal(n_out, n_in).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
            scales = self.normal(-(-n_out // 128), -(-n_in // 128)).abs() * 0.01
            w = be.upload_fp8(data.cpu().numpy(), scales.cpu().numpy(), n_out, n_in)
        elif fmt == "bf16":
            w = be.upload_bf16((self.normal(n_out, n_in) * 0.02).to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16), n_out, n_in)
        elif fmt == "nvfp4":
            w = be.upload_nvfp4(self.blocks(fmt, n_out, n_in), n_out, n_in, scales=0.75)
        else:
            w = be.upload_gguf(GGML[fmt], self.blocks(fmt, n_out, n_in), n_out, n_in)
        if w is None:
            raise RuntimeError(be.last_error())
        return w

    def experts(self, fmt, count, n_out, n_in):
        """(descriptor, kept arrays) of each expert."""
        be = backend()
        if fmt == "mlx4":
            w, s, b = self.mlx4(count * n_out, n_in)
            rows = [slice(e * n_out, (e + 1) * n_out) for e in range(count)]
            return [be.desc_mlx_q4(w[r], s[r], b[r], 64, n_out, n_in) for r in rows]
        raw = self.blocks(fmt, count * n_out, n_in).reshape(count, -1)
        return [be.desc_gguf(GGML[fmt], raw[e], n_out, n_in) for e in range(count)]


# ---- one decode step over dense layers ----------------------------------------------------------------------------------


class DecodeStep:
    """The buffers, weights and recorded plan of a decode step over `layers` dense layers."""

    def __init__(self, case, seed):
        be, g = backend(), Gen(seed)
        t, h, kv, inter = case["t"], case["h"], case["kv"], case["inter"]
        big, small = MIXES[case["mix"]]
        self.t, self.h = t, h
        self.token = g.normal(t, h)  # the step's input: embeddings of the tokens
        self.layers = []
        for _ in range(case["layers"]):
            spec = dict(q=(big, h, h), k=(big, kv, h), v=(small, kv, h), o=(big, h, h), gate=(big, inter, h), up=(big, inter, h), down=(small, h, inter))
            w = {n: g.upload(*s) for n, s in spec.items()}
            # norm weights scaled so that the matrices that read a normed row yield values of unit size
            unit = 1 / (h**0.5 * be.dequantize(w["q"], 0, 64).std())
            w["n1"], w["n2"] = ((1 + 0.1 * g.normal(h)) * unit for _ in range(2))
            self.layers.append(w)
        f32 = dict(dtype=torch.float32, device=DEV)
        self.x = torch.zeros((t, h), **f32)
        self.q, self.k, self.v = (torch.zeros((t, n), **f32) for n in (h, kv, kv))
        self.act = torch.zeros((t, inter), **f32)
        self.qa, self.qo, self.qd = hip.QAct(t, h, DEV), hip.QAct(t, h, DEV), hip.QAct(t, inter, DEV)
        for w in self.layers:
            w["qkv"] = be.decode_jobs([(w[n], self.qa, None, t, y, None, None) for n, y in (("q", self.q), ("k", self.k), ("v", self.v))])
        torch.cuda.synchronize()
        with torch.cuda.stream(decode_stream()):
            self.x.copy_(self.token)
            self.chain()  # brings the stream's scratch into being
            decode_stream().synchronize()
            self.plan = be.plan_record(self.chain)
            decode_stream().synchronize()

    def norm(self, w):
        be = backend()
        if not be.lib.oxhip_dev_norm(be.ctx, self.x.data_ptr(), None, w.data_ptr(), None, 1.0, self.h, self.t, 0, 0, 1e-6, 0, ctypes.byref(self.qa.c), be._stream()):
            raise RuntimeError(be.last_error())

    def linear(self, w, y, xa, mode, w2=None):
        be = backend()
        if not be.linear(w, y, xa=xa, t=self.t, mode=mode, w2=w2):
            raise RuntimeError(be.last_error())

    def chain(self):
        be = backend()
        for w in self.layers:
            self.norm(w["n1"])
            be.decode_batch(w["qkv"])
            be.quantize_act(self.q, out=self.qo)  # (attention is the caller's: its output has q's shape)
            self.linear(w["o"], self.x, self.qo, hip.LIN_ADD)
            self.norm(w["n2"])
            self.linear(w["gate"], self.act, self.qa, hip.LIN_SILU_PAIR, w2=w["up"])
            be.quantize_act(self.act, out=self.qd)
            self.linear(w["down"], self.x, self.qd, hip.LIN_ADD)

    def step(self):
        with torch.cuda.stream(decode_stream()):
            self.x.copy_(self.token)
            self.plan.replay()
        return [self.x, self.q, self.k, self.v, self.act]


# ---- the interface ------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    path = case["path"]
    be = backend()
    if path == "layer":
        return dict(case=case, step=DecodeStep(case, seed))
    g, t = Gen(seed), case["t"]
    if path == "moe":
        ne, h, inter = case["experts"], case["h"], case["inter"]
        layer = be.upload_moe(g.experts(case["fmt"], ne, 2 * inter, h), g.experts(case["fmt"], ne, h, inter), h, inter)
        if layer is None:
            raise RuntimeError(be.last_error())
        return dict(case=case, layer=layer, x=g.normal(t, h), logits=g.normal(t, ne), y=torch.zeros((t, h), device=DEV),
                    sel=torch.empty((2, t, case["k"]), dtype=torch.int32, device=DEV))
    n_out, n_in = case["n_out"], case["n_in"]
    if path == "host":
        ws = [g.upload(case["fmt"], n_out, n_in) for _ in range(case["jobs"])]
        return dict(case=case, x=g.normal(t, n_in).cpu().numpy(), jobs=[(w, np.zeros((t, n_out), np.float32)) for w in ws])
    if path == "matvec":
        quantized = case["fmt"] not in FLOAT_STORED
        return dict(case=case, w=g.upload(case["fmt"], n_out, n_in), x=g.normal(t, n_in), y=torch.zeros((t, n_out), device=DEV),
                    xa=hip.QAct(t, n_in, DEV) if quantized else None)
    dtype = torch.bfloat16 if case["x"] == "bf16" else torch.float32
    shapes = [(n_out, n_in)] + ([(n_in, n_out)] if case["both"] else [])
    return dict(case=case, pairs=[(g.upload(case["fmt"], n, k), g.normal(t, k).to(dtype)) for n, k in shapes])


def run(state):
    case, be = state["case"], backend()
    path = case["path"]
    if path == "layer":
        return state["step"].step()
    if path == "moe":
        be.moe_routed(state["layer"], state["x"], state["logits"], case["k"], state["y"], sel=state["sel"], add=False)
        return [state["y"], state["sel"][0], state["sel"][1].view(torch.float32)]
    if path == "host":
        if not be.matmul(state["x"], case["t"], case["n_in"], state["jobs"]):
            raise RuntimeError(be.last_error())
        return [y for _, y in state["jobs"]]
    if path == "matvec":
        if state["xa"] is None:
            return be.decode(state["w"], x=state["x"], y=state["y"])
        return be.decode(state["w"], xa=be.quantize_act(state["x"], out=state["xa"]), y=state["y"])
    return [be.gemm(w, x, variant=VARIANT[case["variant"]], out_bf16=case["y"] == "bf16") for w, x in state["pairs"]]


def work(case):
    path, t = case["path"], case["t"]
    if path == "layer":
        big, small = (BITS[f] / 8 for f in MIXES[case["mix"]])
        h, kv, inter = case["h"], case["kv"], case["inter"]
        n_big, n_small = 2 * h * h + kv * h + 2 * inter * h, kv * h + h * inter
        return {"bytes": case["layers"] * (n_big * big + n_small * small + 8 * h) + t * 4 * (3 * h + 2 * kv + inter),
                "flops": 2 * t * case["layers"] * (n_big + n_small)}
    if path == "moe":
        ne, k, h, inter = case["experts"], case["k"], case["h"], case["inter"]
        touched = ne * (1 - (1 - k / ne) ** t)  # experts that t tokens' independent routes reach, on average
        return {"bytes": touched * 3 * h * inter * BITS[case["fmt"]] / 8 + t * (8 * h + 4 * ne + 8 * k), "flops": 2 * t * k * 3 * h * inter}
    n_out, n_in = case["n_out"], case["n_in"]
    many = 2 if case.get("both") else case.get("jobs", 1)
    xs, ys = 2 if case.get("x") == "bf16" else 4, 2 if case.get("y") == "bf16" else 4
    io = t * (xs * n_in + ys * n_out) + (t * (xs * n_out + ys * n_in) if case.get("both") else (many - 1) * t * ys * n_out)
    return {"bytes": many * n_out * n_in * BITS[case["fmt"]] / 8 + io, "flops": 2 * t * many * n_out * n_in}


def tolerance(case):
    """About four times what was measured: decode of one matrix against itself on inputs moved by an f32 rounding (2e-7; FP8
    rows go in as two bf16 planes, 2.5e-6), the bf16 products against the same product in 64 bits (1.5e-3 to 2.9e-3 by the
    operands' and the result's types), a layer's step and a MoE pass against themselves with such a moved input (a sum that
    moves by one rounding can move an int8 code of the next matrix's input, and what that moves then moves others: 7e-3 after
    two layers, 2e-4 over one MoE layer)."""
    path, t = case["path"], case["t"]
    if path == "layer":
        return {"rel": 3e-2, "max": 0.6}
    if path == "moe":
        # six and more routed rows per expert run on bf16 operands (2.9e-3)
        return {"rel": 1e-2, "max": 6e-2} if t * case["k"] // case["experts"] >= 6 else {"rel": 1e-3, "max": 2e-2}
    if path == "matvec" or (path == "host" and t <= 16):
        return {"rel": 1e-5, "max": 5e-5}
    if case.get("variant", "bf16") == "bf16":
        return {"rel": 1e-2, "max": 6e-2}
    return {"rel": 1e-5, "max": 1e-4} if case["y"] == "f32" else {"rel": 1e-3, "max": 1e-2}
