"""Workloads of the quantized decode and prefill path, as a program that runs a
model on this library calls them.

Five kinds, each a dict of plain sizes:

  gemv    `count` matrix-vector products with MLX-affine weights, one after
          another (a decode step's products, or the head)
  proj    the attention projections of `layers` layers: matrices that share
          the hidden state in one call, the output projection in another
  dense   `layers` dense decoder layers: q/k/v, o, the gate/up pair with its
          SwiGLU, down
  moe     `layers` routed-expert blocks (routing, experts, combine, shared
          expert) on resident banks
  llama   `layers` whole dense decode layers with norms, RoPE, attention over
          the cache and residuals
  island  the host-pointer interface an engine links: the route island
          (begin, shared expert in between, finish) on host f32 activations

Decode passes of the device-native calls are captured once in a HIP graph and
replayed, as a serving loop does; prefill passes and the host-pointer calls
are made directly. Every case has its own weights per layer and matrix, so
that a pass reads them from HBM.
"""
import ctypes
import math

import numpy as np
import torch

from logan_amd import _lib, backend, device

GROUP = 64


def listed():
    return [
        # one decode step's 4-bit products at the smallest size in use: launch
        # and load latency
        dict(name="gemv_q4_m1", kind="gemv", bits=4, gs=64, I=2048, O=4096, M=1, count=32, out="bf16", fp16=False),
        # token generation, one sequence: MoE blocks of a 4-bit sparse model
        dict(name="moe_q4_b1", kind="moe", bits=4, E=512, k=10, D=2048, inter=512, B=1, layers=8, zipf=0.0, shared=True, out="bf16", fp16=False),
        # token generation for a small batch of sequences
        dict(name="moe_q4_b16", kind="moe", bits=4, E=512, k=10, D=2048, inter=512, B=16, layers=4, zipf=0.0, shared=True, out="f32", fp16=False),
        # the same at 6 bits with skewed expert popularity, a larger batch
        dict(name="moe_q6_b32_zipf", kind="moe", bits=6, E=512, k=10, D=2048, inter=512, B=32, layers=2, zipf=1.1, shared=True, out="bf16", fp16=False),
        # a prefill chunk through one MoE block
        dict(name="moe_q4_b512", kind="moe", bits=4, E=512, k=10, D=2048, inter=512, B=512, layers=1, zipf=0.0, shared=True, out="bf16", fp16=False),
        # a long prompt in one chunk, not a round number of tokens
        dict(name="moe_q4_b1999", kind="moe", bits=4, E=512, k=10, D=2048, inter=512, B=1999, layers=1, zipf=0.0, shared=True, out="bf16", fp16=False),
        # dense 8-bit model, decode for eight sequences
        dict(name="dense_q8_m8", kind="dense", bits=8, gs=64, H=4096, Q=6144, F=14336, M=8, layers=2, fp16=False),
        # the same model, a short prompt
        dict(name="dense_q8_m100", kind="dense", bits=8, gs=64, H=4096, Q=6144, F=14336, M=100, layers=1, fp16=False),
        # the same model, a long prompt chunk
        dict(name="dense_q8_m2048", kind="dense", bits=8, gs=64, H=4096, Q=6144, F=14336, M=2048, layers=1, fp16=False),
        # 4-bit attention projections of a hybrid model over a prefill chunk:
        # a linear-attention layer (qkvz, ba, out) and a full-attention layer
        dict(name="proj_q4_m512", kind="proj", bits=4, gs=64, D=2048, att=4096, shared_cols="12288,64;8192,512,512", M=512, fp16=False),
        # a dense 8-bit model's decode step with a context of some length
        dict(name="llama_q8_pos1500", kind="llama", fmt=15, D=4096, inter=14336, heads=32, kv_heads=8, hd=128, pos=1500, layers=2),
        # an engine linking the host-pointer interface, MXFP4 experts
        dict(name="island_mxfp4", kind="island", fmt=7, k=10, D=2048, inter=512, layers=4),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemv", "proj", "proj", "dense", "dense", "moe", "moe", "moe", "llama", "island"])
    fp16 = rng.random() < 0.2
    if kind == "gemv":
        I = 64 * _spread(rng, 8, 128)
        return dict(kind=kind, bits=rng.choice([4, 4, 5, 6, 8]), gs=rng.choice([32, 64, 64]), I=I,
                    O=_spread(rng, 257, 40000), M=rng.choice([1, 1, 1, 2, 3]), count=rng.randint(4, 16),
                    out=rng.choice(["bf16", "f32"]), fp16=fp16)
    if kind == "proj":
        D, att = rng.choice([(2048, 4096), (2048, 2048), (4096, 4096), (1536, 3072), (2880, 4096)])
        cols = rng.choice(["12288,64;8192,512,512", "8192,512,512", "4096,1024,1024", "6151,33"])
        return dict(kind=kind, bits=rng.choice([4, 4, 5, 6, 8]), gs=64, D=D, att=att, shared_cols=cols,
                    M=_spread(rng, 1, 2048), fp16=fp16)
    if kind == "dense":
        H, Q, F = rng.choice([(4096, 6144, 14336), (2048, 3072, 8192), (3072, 5120, 8192), (2560, 3584, 9728)])
        return dict(kind=kind, bits=rng.choice([4, 6, 8, 8]), gs=64, H=H, Q=Q, F=F, M=_spread(rng, 1, 2000), layers=1,
                    fp16=fp16)
    if kind == "moe":
        E, k, D, inter = rng.choice([(512, 10, 2048, 512), (512, 10, 2048, 512), (128, 8, 2048, 768), (64, 6, 1024, 512)])
        B = _spread(rng, 1, 1999)
        return dict(kind=kind, bits=rng.choice([4, 4, 5, 6, 8]), E=E, k=k, D=D, inter=inter, B=B, layers=4 if B <= 32 else 1,
                    zipf=rng.choice([0.0, 1.1]), shared=rng.random() < 0.8, out=rng.choice(["bf16", "f32"]), fp16=fp16)
    if kind == "llama":
        return dict(kind=kind, fmt=rng.choice([5, 15]), D=4096, inter=14336, heads=32, kv_heads=8, hd=128,
                    pos=_spread(rng, 1, 4000), layers=2)
    return dict(kind=kind, fmt=rng.choice([7, 21]), k=rng.randint(4, 12), D=2048, inter=rng.choice([512, 768]),
                layers=rng.randint(2, 4))


# ------------------------------------------------------------------ inputs


def _gen(seed, dev="cuda"):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _codes(g, shape, dev="cuda"):
    """Uniform packed words: every b-bit code is uniform."""
    return torch.randint(-(2**31), 2**31, shape, dtype=torch.int32, device=dev, generator=g)


def _affine(g, O, I, bits, gs, fp16, E=None, dev="cuda"):
    """Packed weights and their sidecar with weights of about 1 / sqrt(I)
    (bias = -2^(bits-1) * scale, exact in either 16-bit type)."""
    lead = () if E is None else (E,)
    w = _codes(g, lead + (O, I * bits // 32), dev).view(torch.uint8).reshape(lead + (O, I * bits // 8))
    t = torch.float16 if fp16 else torch.bfloat16
    s = torch.randn(lead + (O, I // gs), device=dev, generator=g).abs() * (math.sqrt(12.0) / (2**bits * math.sqrt(I)))
    s = s.to(t)
    b = (s.float() * -(2 ** (bits - 1))).to(t)
    return w, s.view(torch.int16), b.view(torch.int16)


def _matrix(g, O, I, bits, gs, fp16):
    return device.AffineMatrix(*_affine(g, O, I, bits, gs, fp16), O, I, bits, gs, fp16)


def _bank(g, E, O, I, bits, fp16):
    return device.AffineBank(*_affine(g, O, I, bits, GROUP, fp16, E=E), E, O, I, bits, GROUP, fp16)


def _x(g, *shape):
    return torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)


def _logits(g, B, E, zipf):
    """Router logits; zipf > 0: popularity rank^-zipf (Gumbel-max)."""
    if not zipf:
        return torch.randn((B, E), device="cuda", generator=g).to(torch.bfloat16)
    prior = -zipf * torch.log(torch.randperm(E, device="cuda", generator=g).float() + 1.0)
    u = torch.rand((B, E), device="cuda", generator=g).clamp_(1e-9, 1 - 1e-7)
    return (prior - torch.log(-torch.log(u))).to(torch.bfloat16)


def _dtype(case):
    return torch.bfloat16 if case.get("out", "bf16") == "bf16" else torch.float32


def _groups(case):
    return [[int(c) for c in layer.split(",")] for layer in case["shared_cols"].split(";")]


def _inputs(case, seed):
    """Everything of a state that is made from the seed."""
    kind = case["kind"]
    g = _gen(seed)
    s = {}
    if kind == "gemv":
        s["mats"] = [_matrix(g, case["O"], case["I"], case["bits"], case["gs"], case["fp16"]) for _ in range(case["count"])]
        s["x"] = [_x(g, case["M"], case["I"]) for _ in range(case["count"])]
    elif kind == "proj":
        s["layers"] = [([_matrix(g, c, case["D"], case["bits"], case["gs"], case["fp16"]) for c in cols],
                        _matrix(g, case["D"], case["att"], case["bits"], case["gs"], case["fp16"])) for cols in _groups(case)]
        s["x"] = _x(g, case["M"], case["D"])
        s["att"] = _x(g, case["M"], case["att"])
    elif kind == "dense":
        H, Q, F = case["H"], case["Q"], case["F"]
        s["layers"] = [{n: _matrix(g, O, I, case["bits"], case["gs"], case["fp16"])
                        for n, O, I in (("qkv", Q, H), ("o", H, H), ("gate", F, H), ("up", F, H), ("down", H, F))}
                       for _ in range(case["layers"])]
        s["x"] = [_x(g, case["M"], H) for _ in range(case["layers"])]
        s["att"] = [_x(g, case["M"], H) for _ in range(case["layers"])]
    elif kind == "moe":
        E, D, n, bits, fp16 = case["E"], case["D"], case["inter"], case["bits"], case["fp16"]
        s["layers"], s["x"], s["logits"] = [], [], []
        for _ in range(case["layers"]):
            banks = [_bank(g, E, n, D, bits, fp16), _bank(g, E, n, D, bits, fp16), _bank(g, E, D, n, bits, fp16)]
            sh = []
            if case["shared"]:
                sh = [_bank(g, 1, n, D, bits, fp16), _bank(g, 1, n, D, bits, fp16), _bank(g, 1, D, n, bits, fp16),
                      (torch.randn(D, device="cuda", generator=g) * 0.05).to(torch.bfloat16)]
            s["layers"].append(device.MoeLayer(*banks, case["k"], *sh))
            s["x"].append(_x(g, case["B"], D))
            s["logits"].append(_logits(g, case["B"], E, case["zipf"]))
    elif kind == "llama":
        D, n, qd, kv = case["D"], case["inter"], case["heads"] * case["hd"], case["kv_heads"] * case["hd"]
        s["layers"] = []
        for _ in range(case["layers"]):
            mats = []
            for O, I in ((qd, D), (kv, D), (kv, D), (D, qd), (n, D), (n, D), (D, n)):
                if case["fmt"] == 15:
                    w, sc, bi = _affine(g, O, I, 8, 64, False)
                    mats.append(device.DenseMatrix(w, O, I, 15, sc, bi))
                else:
                    w = (torch.randn((O, I), device="cuda", generator=g) / math.sqrt(I)).to(torch.bfloat16)
                    mats.append(device.DenseMatrix(w.view(torch.int16), O, I, 5))
            norms = [1 + 0.1 * torch.randn(D, device="cuda", generator=g) for _ in range(2)]
            cache = [torch.randn((case["pos"] + 1, kv), device="cuda", generator=g) for _ in range(2)]
            s["layers"].append(device.LlamaLayer(mats, *norms, *cache, D, n, case["heads"], case["kv_heads"], case["hd"],
                                                 500000.0, 1e-5))
        s["x0"] = torch.randn(D, device="cuda", generator=g)
    else:
        h = _gen(seed, "cpu")
        s["x"] = [torch.randn(case["D"], generator=h).numpy() for _ in range(case["layers"])]
        s["weights"] = []  # per layer: (k + 1) experts of gate, up, down; the last one is the shared expert
        for _ in range(case["layers"]):
            layer = []
            for _ in range(case["k"] + 1):
                for O, I in ((case["inter"], case["D"]), (case["inter"], case["D"]), (case["D"], case["inter"])):
                    if case["fmt"] == 7:
                        w = _codes(h, (O, I // 8), "cpu").numpy().view(np.uint8)
                        aux = torch.randint(118, 122, (O, I // 32), dtype=torch.uint8, generator=h).numpy()
                    else:
                        w, sc, bi = (t.numpy() for t in _affine(h, O, I, 4, 64, True, dev="cpu"))
                        aux = np.concatenate([sc.reshape(-1), bi.reshape(-1)]).view(np.uint8)
                    layer.append((w, aux, O, I))
            s["weights"].append(layer)
    return s


class _Handles:
    """The tensor handles an engine keeps per weight; freed with the state."""

    def __init__(self, descs):
        self.descs = descs

    def __del__(self):
        for d in self.descs:
            if d.tensor:
                _lib.lib().logan_hip_tensor_free(ctypes.c_void_p(d.tensor))


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    s["case"] = case
    new = lambda *shape, dtype=torch.bfloat16: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    if kind == "gemv":
        s["y"] = [new(case["M"], case["O"], dtype=_dtype(case)) for _ in s["mats"]]
    elif kind == "proj":
        M = case["M"]
        s["y"] = [([new(M, m.O) for m in ms], new(M, o.O)) for ms, o in s["layers"]]
    elif kind == "dense":
        M, H, Q, F = case["M"], case["H"], case["Q"], case["F"]
        s["y"] = [dict(qkv=new(M, Q), o=new(M, H), h=new(M, F), up=new(M, F), y=new(M, H)) for _ in s["layers"]]
    elif kind == "moe":
        s["y"] = [new(case["B"], case["D"], dtype=_dtype(case)) for _ in s["layers"]]
        s["ws"] = new(s["layers"][0].workspace_bytes(case["B"]), dtype=torch.uint8)
    elif kind == "llama":
        s["x"] = s["x0"].clone()
        s["ws"] = new(device.llama_workspace_bytes(s["layers"][0], case["pos"]), dtype=torch.uint8)
    else:
        if not backend.hip_init():
            raise RuntimeError("no device")
        s["calls"] = []
        for x, layer in zip(s["x"], s["weights"]):
            descs = (_lib.MatmulDesc * len(layer))()
            for d, (w, aux, O, I) in zip(descs, layer):
                d.weights, d.scales, d.fmt = w.ctypes.data, aux.ctypes.data, case["fmt"]
                d.I, d.O, d.gs, d.S = I, O, 0 if case["fmt"] == 7 else 64, 1
            ys, sy = np.zeros(case["k"] * case["D"], np.float32), np.zeros(case["D"], np.float32)
            s["calls"].append((descs, x, ys, sy, _Handles(descs)))
        _island(s)  # the weights become resident behind their handles
    if _decode(case):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
    return s


def _decode(case):
    """Whether the pass is a decode step (replayed from a graph)."""
    return case["kind"] in ("gemv", "llama") or (case["kind"] != "island" and case.get("M", case.get("B")) <= 32)


def _step(s):
    case, kind = s["case"], s["case"]["kind"]
    few = _decode(case)
    if kind == "gemv":
        for w, x, y in zip(s["mats"], s["x"], s["y"]):
            device.affine_gemv(w, x, out=y)
    elif kind == "proj":
        many, one = (device.affine_gemv_multi, device.affine_gemv) if few else (device.affine_qmm_multi, device.affine_qmm)
        for (ms, o), (ys, yo) in zip(s["layers"], s["y"]):
            many(ms, s["x"], outs=ys)
            one(o, s["att"], out=yo)
    elif kind == "dense":
        one = device.affine_gemv if few else device.affine_qmm
        for L, x, att, y in zip(s["layers"], s["x"], s["att"], s["y"]):
            one(L["qkv"], x, out=y["qkv"])
            one(L["o"], att, out=y["o"])
            if few:
                device.affine_gemv_swiglu(L["gate"], L["up"], y["o"], out=y["h"])
            else:
                device.affine_qmm_multi([L["gate"], L["up"]], y["o"], outs=[y["h"], y["up"]])
                device.silu_mul(y["h"], y["up"])
            one(L["down"], y["h"], out=y["y"])
    elif kind == "moe":
        for L, x, lg, y in zip(s["layers"], s["x"], s["logits"], s["y"]):
            device.moe_block(L, x, lg, out=y, workspace=s["ws"])
    elif kind == "llama":
        s["x"].copy_(s["x0"])
        for L in s["layers"]:
            device.llama_layer(L, s["x"], case["pos"], workspace=s["ws"])


def _island(s):
    lib, case = _lib.lib(), s["case"]
    k, D, n = case["k"], case["D"], case["inter"]
    for i, (descs, x, ys, sy, _) in enumerate(s["calls"]):
        shared = ctypes.cast(ctypes.byref(descs, 3 * k * ctypes.sizeof(_lib.MatmulDesc)), ctypes.POINTER(_lib.MatmulDesc))
        p = lib.logan_hip_moe_route_begin(1, i, descs, k, x.ctypes.data, D, n)
        if not p:
            raise RuntimeError("route island declined")
        if lib.logan_hip_shared_expert(1, i, shared, 3, x.ctypes.data, sy.ctypes.data, D, n) != 1:
            raise RuntimeError("shared expert declined")
        if lib.logan_hip_moe_route_finish(ctypes.c_void_p(p), ys.ctypes.data, k) != 1:
            raise RuntimeError("route island failed")


def run(state):
    kind = state["case"]["kind"]
    if kind == "island":
        _island(state)
        return [(ys, sy) for _, _, ys, sy, _ in state["calls"]]
    if "graph" in state:
        state["graph"].replay()
    else:
        _step(state)
    if kind == "dense":
        return [{n: y[n] for n in ("qkv", "o", "h", "y")} for y in state["y"]]
    if kind == "llama":
        return {"x": state["x"], "cache": [(L.k_cache, L.v_cache) for L in state["layers"]]}
    return state["y"]


# ------------------------------------------------------------- work, bounds


def _wbytes(O, I, bits, gs=GROUP):
    return O * I * bits // 8 + 4 * O * (I // gs)


def _experts_hit(case):
    """Distinct experts a batch is expected to touch."""
    E, k, B = case["E"], case["k"], case["B"]
    if not case["zipf"]:
        return E * (1 - (1 - k / E) ** B)
    r = np.random.default_rng(0)
    p = -case["zipf"] * np.log(np.arange(E) + 1.0) + r.gumbel(size=(B, E))
    return float(len(np.unique(np.argpartition(-p, k, axis=1)[:, :k])))


def work(case):
    kind, by, fl = case["kind"], 0.0, 0.0
    if kind == "gemv":
        by = _wbytes(case["O"], case["I"], case["bits"], case["gs"]) + case["M"] * (2 * case["I"] + case["O"] * (2 if case["out"] == "bf16" else 4))
        by, fl = by * case["count"], 2.0 * case["M"] * case["O"] * case["I"] * case["count"]
    elif kind == "proj":
        for cols in _groups(case):
            for O, I in [(c, case["D"]) for c in cols] + [(case["D"], case["att"])]:
                by += _wbytes(O, I, case["bits"], case["gs"]) + 2 * case["M"] * O
                fl += 2.0 * case["M"] * O * I
        by += 2 * case["M"] * (case["D"] + case["att"])
    elif kind == "dense":
        H, Q, F, M = case["H"], case["Q"], case["F"], case["M"]
        for O, I in ((Q, H), (H, H), (F, H), (F, H), (H, F)):
            by += _wbytes(O, I, case["bits"], case["gs"])
            fl += 2.0 * M * O * I
        by = (by + 2 * M * (Q + 3 * H + F + H)) * case["layers"]
        fl *= case["layers"]
    elif kind == "moe":
        per = 2 * _wbytes(case["inter"], case["D"], case["bits"]) + _wbytes(case["D"], case["inter"], case["bits"])
        sh = 1 if case["shared"] else 0
        by = (_experts_hit(case) + sh) * per + case["B"] * (2 * case["E"] + 2 * case["D"] + case["D"] * (2 if case["out"] == "bf16" else 4))
        fl = 2.0 * case["B"] * (case["k"] + sh) * 3 * case["inter"] * case["D"]
        by, fl = by * case["layers"], fl * case["layers"]
    elif kind == "llama":
        D, n, qd, kv = case["D"], case["inter"], case["heads"] * case["hd"], case["kv_heads"] * case["hd"]
        for O, I in ((qd, D), (kv, D), (kv, D), (D, qd), (n, D), (n, D), (D, n)):
            by += _wbytes(O, I, 8) if case["fmt"] == 15 else 2 * O * I
            fl += 2.0 * O * I
        by = (by + 8.0 * kv * (case["pos"] + 1) + 16 * D) * case["layers"]
        fl = (fl + 4.0 * qd * (case["pos"] + 1)) * case["layers"]
    else:
        per = 0
        for O, I in ((case["inter"], case["D"]), (case["inter"], case["D"]), (case["D"], case["inter"])):
            per += O * I // 2 + (O * I // 32 if case["fmt"] == 7 else 4 * O * (I // 64))
            fl += 2.0 * O * I
        by = (per + 4 * case["D"]) * (case["k"] + 1) * case["layers"]
        fl *= (case["k"] + 1) * case["layers"]
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """Sums in another order move a result by about 1e-6 of its norm before it
    is rounded; bf16 results then differ where a rounding falls the other way
    (one part in 256 of those values)."""
    if case["kind"] == "llama":
        return {"rel": 2e-5, "max": 2e-3}
    if case["kind"] == "island":
        return {"rel": 4e-5, "max": 4e-3}
    if case.get("out") == "f32":
        return {"rel": 4e-5, "max": 4e-3}
    return {"rel": 4e-3, "max": 0.05}


# ----------------------------------------------------------------- in 64 bits


def _unpack(w, bits):
    """Codes of packed rows [..., I * bits / 8] (LSB-first bit stream)."""
    b = w.to(torch.int32)
    if bits == 8:
        return b
    if bits == 4:
        return torch.stack([b & 15, b >> 4], dim=-1).flatten(-2)
    n = w.shape[-1] * 8 // bits
    at = torch.arange(n, device=w.device) * bits
    lo, sh = at // 8, (at % 8).to(torch.int32)
    hi = torch.clamp(lo + 1, max=w.shape[-1] - 1)
    return ((b[..., lo] | (b[..., hi] << 8)) >> sh) & ((1 << bits) - 1)


def _dequant(w, sc, bi, bits, gs, fp16, rounded=False):
    t = torch.float16 if fp16 else torch.bfloat16
    c = _unpack(w, bits)
    s = sc.view(t).double().repeat_interleave(gs, dim=-1)
    b = bi.view(t).double().repeat_interleave(gs, dim=-1)
    v = c.double().mul_(s).add_(b)
    # the prefill product's weights are defined as bf16, rounded from f32
    return v.float().to(torch.bfloat16).double() if rounded else v


def _full(m, rounded=False):
    return _dequant(m.weights, m.scales, m.biases, m.bits, m.group_size, m.aux_fp16, rounded)


def _silu(v):
    return v / (1 + torch.exp(-v))


def _bf(v):
    return v.to(torch.bfloat16).double()


def _exact_moe(case, L, x, lg):
    x, lg = x.double(), lg.double()
    top, idx = torch.sort(lg, dim=1, descending=True, stable=True)
    top, idx = top[:, :case["k"]], idx[:, :case["k"]]
    wts = torch.softmax(top, dim=1)
    out = torch.zeros_like(x)

    def expert(banks, e, v):
        g, u, d = (_dequant(b.weights[e], b.scales[e], b.biases[e], b.bits, b.group_size, b.aux_fp16) for b in banks)
        return (_silu(v @ g.T) * (v @ u.T)) @ d.T

    for e in torch.unique(idx).tolist():
        tok, rank = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, tok, expert((L.gate, L.up, L.down), e, x[tok]) * wts[tok, rank, None])
    if L.shared_gate is not None:
        gate = torch.sigmoid(x @ L.shared_gate_vec.double())
        out += expert((L.shared_gate, L.shared_up, L.shared_down), 0, x) * gate[:, None]
    return out


def _exact_llama(case, s):
    H, KH, hd, pos = case["heads"], case["kv_heads"], case["hd"], case["pos"]
    x = s["x0"].double()
    cache = []
    # the angle is defined in f32: pos / theta^(2 j / hd)
    pw = torch.pow(torch.tensor(500000.0, dtype=torch.float64), (torch.arange(hd // 2).float() * 2 / hd).double()).float()
    ang = (torch.tensor(float(pos)) / pw).double().cuda()

    def rope(v):
        a, b = v[:, : hd // 2], v[:, hd // 2:]
        return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], dim=1)

    for L in s["layers"]:
        def mat(i):
            m = L.mats[i]
            if m.fmt == 5:
                return m.weights.view(torch.bfloat16).double()
            return _dequant(m.weights, m.scales, m.biases, 8, 64, False, rounded=True)

        def norm(v, w):
            return v / torch.sqrt((v * v).mean() + 1e-5) * w.double()

        h = norm(x, L.in_norm)
        q = rope((mat(0) @ h).view(H, hd))
        kc, vc = L.k_cache.double(), L.v_cache.double()
        kc[pos], vc[pos] = rope((mat(1) @ h).view(KH, hd)).reshape(-1), mat(2) @ h
        kk = kc.view(-1, KH, hd).repeat_interleave(H // KH, dim=1)
        vv = vc.view(-1, KH, hd).repeat_interleave(H // KH, dim=1)
        p = torch.softmax((kk * q).sum(-1) / math.sqrt(hd), dim=0)
        x = x + mat(3) @ (p[:, :, None] * vv).sum(0).reshape(-1)
        h = norm(x, L.post_norm)
        x = x + mat(6) @ (_silu(mat(4) @ h) * (mat(5) @ h))
        cache.append((kc, vc))
    return {"x": x, "cache": cache}


def _exact_island(case, s):
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64)
    out = []
    for x, layer in zip(s["x"], s["weights"]):
        ys, v = [], torch.from_numpy(x).double()

        def mat(t):
            w, aux, O, I = t
            w = torch.from_numpy(w).view(O, -1)
            if case["fmt"] == 7:
                sc = torch.pow(2.0, torch.from_numpy(aux).double() - 127).view(O, I // 32)
                return table[_unpack(w, 4).long()] * sc.repeat_interleave(32, dim=1)
            p = torch.from_numpy(aux).view(torch.int16).view(2, O, I // 64)
            return _dequant(w, p[0], p[1], 4, 64, True)

        for e in range(case["k"] + 1):
            g, u, d = (mat(t) for t in layer[3 * e:3 * e + 3])
            ys.append(d @ (_silu(g @ v) * (u @ v)))
        out.append((torch.cat(ys[:-1]), ys[-1]))
    return out


def exact(case, seed):
    """run()'s result for these inputs in float64. Where a call hands bf16 to
    the next one, the value handed on is rounded to bf16 as there."""
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gemv":
        return [x.double() @ _full(m).T for m, x in zip(s["mats"], s["x"])]
    q = not _decode(case)
    if kind == "proj":
        x, att = s["x"].double(), s["att"].double()
        return [([x @ _full(m, q).T for m in ms], att @ _full(o, q).T) for ms, o in s["layers"]]
    if kind == "dense":
        out = []
        for L, x, att in zip(s["layers"], s["x"], s["att"]):
            o = att.double() @ _full(L["o"], q).T
            g, u = _bf(o) @ _full(L["gate"], q).T, _bf(o) @ _full(L["up"], q).T
            h = _silu(_bf(g)) * _bf(u) if q else _silu(g) * u
            out.append(dict(qkv=x.double() @ _full(L["qkv"], q).T, o=o, h=h, y=_bf(h) @ _full(L["down"], q).T))
        return out
    if kind == "moe":
        return [_exact_moe(case, L, x, lg) for L, x, lg in zip(s["layers"], s["x"], s["logits"])]
    if kind == "llama":
        return _exact_llama(case, s)
    return _exact_island(case, s)
