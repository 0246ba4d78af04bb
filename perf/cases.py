"""Performance cases of the MoE layer framework: what its users have it do.

Every case is one pass through the public entry points (hip_backend over the
C ABI): MoE blocks of the two model shapes this repository is built around
(Qwen3-Next: h 2048, 512 experts, top 10, ff 512 and a shared expert;
Qwen3-30B-A3B: h 2048, 128 experts, top 8, ff 768), from one token to a
4096-token prefill, the dense affine products beside them, and the op-by-op
sequence of a host that composes the block itself.

A case holds `kind` ("block", "linear", "ops"), the shape, the token count,
`layers` (independent layers of one pass, each with weights and input rows of
its own) and the options.  Weights are N(0, 0.02) quantized to MLX affine codes (per
group min / max, bf16 scales and biases), activations N(0, 1).  Tokens whose
K-th and K+1-th router logits lie closer than F32 sums can tell apart are
drawn again, so that every correct F32 router selects the same experts.
"""
import ctypes
import os
import sys

import numpy as np
import torch

PKG = os.path.join(os.getcwd(), "llama-rs-metal_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

NEXT = {"shape": "next", "h": 2048, "E": 512, "K": 10, "ff": 512, "ffs": 512}
A3B = {"shape": "a3b", "h": 2048, "E": 128, "K": 8, "ff": 768, "ffs": 0}

# options of a block, and their defaults: bits/group of the routed experts,
# of the router (0: dense F32) and of the shared expert, routing skew, the
# MFMA tile-order weight copies, RMSNorm + residual, replay of a captured graph
BLOCK = {"kind": "block", "layers": 1, "bits": 4, "group": 64, "rbits": 0, "sbits": 4, "skew": "none",
         "packed": False, "norm": True, "graph": False}

GAP = 1e-4     # least distance of the K-th and K+1-th router logit
STD = 0.02


def listed():
    def block(name, base, tokens, **over):
        return dict(BLOCK, **base, name=name, tokens=tokens, **over)

    return [
        # one token through the MoE blocks of 12 layers: a chat's decode loop,
        # captured once and replayed for every token
        block("next_decode", NEXT, 1, layers=12, graph=True),
        block("a3b_decode", A3B, 1, layers=12, rbits=4, graph=True),
        # the same, issued call by call, of an 8-bit checkpoint
        block("next_decode_8bit", NEXT, 1, layers=12, bits=8, group=128, sbits=8),
        # a few chats served at once: 8-bit router and shared expert, some
        # tokens of one topic (a hot set of experts)
        block("next_batch8", NEXT, 8, layers=6, rbits=8, sbits=8, skew="hot", norm=False),
        block("next_batch64", NEXT, 64, layers=3, rbits=8, sbits=8, skew="hot", norm=False),
        block("a3b_batch24", A3B, 24, layers=4, rbits=4),
        # short prompts and chunks of a chunked prefill: too few rows per
        # expert for whole matrix tiles
        block("next_chunk500", NEXT, 500, norm=False),
        block("a3b_chunk1000_8bit", A3B, 1000, bits=8, group=128, rbits=8, skew="zipf"),
        # long prompts, with the tile-order copies made at load
        block("a3b_prefill4096", A3B, 4096, rbits=4, skew="zipf", packed=True, norm=False),
        block("next_prefill4096", NEXT, 4096, packed=True, norm=False),
        # dense affine projections of a 700-token prompt (Batch::matmul)
        {"kind": "linear", "name": "linear700", "tokens": 700, "bits": 4, "group": 64, "stype": "bf16", "rows": 2048,
         "outs": "4096,512,512,2048"},
        # a host that issues the block op by op, one token (drop-in use of the
        # backend's op surface)
        dict(BLOCK, **NEXT, name="next_ops", kind="ops", tokens=1, layers=4),
    ]


def draw(rng):
    def size(lo, hi):
        return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))

    what = rng.choice(["decode", "batch", "batch", "chunk", "chunk", "prefill", "linear", "ops"])
    if what == "linear":
        bits = rng.choice([2, 4, 8])
        outs = [rng.choice([256, 512, 1000, 2048, 4096]) for _ in range(rng.randint(1, 3))]
        return {"kind": "linear", "tokens": size(4, 2000), "bits": bits, "group": rng.choice([32, 64, 128]),
                "stype": rng.choice(["bf16", "f16", "f32"]), "rows": rng.choice([512, 1024, 2048, 4096]),
                "outs": ",".join(str(o) for o in outs)}
    base = rng.choice([NEXT, A3B])
    c = dict(BLOCK, **base)
    c["bits"], c["group"] = rng.choice([(4, 64), (4, 64), (4, 32), (8, 64), (8, 128), (2, 32)])
    c["rbits"] = rng.choice([0, 4, 8])
    c["sbits"] = rng.choice([c["bits"], 8])
    c["norm"] = rng.random() < 0.5
    c["skew"] = rng.choice(["none", "hot", "zipf"])
    if what in ("decode", "ops"):
        c["tokens"], c["layers"], c["skew"] = 1, rng.randint(2, 12), "none"
        if what == "ops":
            c["kind"], c["layers"] = "ops", rng.randint(1, 4)
        else:
            c["graph"] = rng.random() < 0.5
    elif what == "batch":
        c["tokens"], c["layers"] = size(2, 64), rng.randint(1, 4)
    else:
        c["tokens"] = size(65, 1024) if what == "chunk" else size(1025, 4096)
        c["packed"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ inputs --
def quantize(w, bits, group, stype="bf16"):
    """MLX affine codes of w [rows, in] (F32, on the GPU): packed int32 words
    (low bits first), scales and biases [rows, in / group]."""
    rows, n = w.shape
    g = w.view(rows, n // group, group)
    mn, mx = g.amin(2), g.amax(2)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[stype]
    s = ((mx - mn) / ((1 << bits) - 1)).to(dt)
    b = mn.to(dt)
    q = ((g - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, (1 << bits) - 1)
    q = q.to(torch.int32).view(rows, n * bits // 32, 32 // bits)
    words = torch.zeros(q.shape[:2], dtype=torch.int32, device=w.device)
    for i in range(32 // bits):
        words |= q[..., i] << (bits * i)
    return words, s, b


class Matrix:
    """One weight: `experts` matrices [out, in], dense F32 (bits 0) or affine."""

    def __init__(self, gen, n_in, out, experts, bits, group, stype="bf16"):
        self.n_in, self.out, self.experts, self.bits, self.group, self.stype = n_in, out, experts, bits, group, stype
        if bits == 0:
            self.parts = (torch.randn(experts * out, n_in, generator=gen, device="cuda") * STD,)
            return
        step = max(1, (1 << 26) // (out * n_in))  # experts quantized at a time
        parts = [quantize(torch.randn(min(step, experts - e) * out, n_in, generator=gen, device="cuda") * STD,
                          bits, group, stype) for e in range(0, experts, step)]
        self.parts = tuple(torch.cat(p) for p in zip(*parts))

    def bytes(self):
        return sum(p.numel() * p.element_size() for p in self.parts)

    def f64(self, e=0):
        """Matrix e in 64 bits: code * scale + bias."""
        lo, hi = e * self.out, (e + 1) * self.out
        if self.bits == 0:
            return self.parts[0][lo:hi].double()
        words, s, b = (p[lo:hi] for p in self.parts)
        at = torch.arange(0, 32, self.bits, device="cuda", dtype=torch.int32)
        q = (words[..., None] >> at) & ((1 << self.bits) - 1)
        q = q.reshape(self.out, self.n_in // self.group, self.group).double()
        return (q * s.double()[..., None] + b.double()[..., None]).view(self.out, self.n_in)


def rms(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w


class LayerInputs:
    """Weights, input rows and routing bias of one MoE block."""

    def __init__(self, c, gen):
        h, E, K, T = c["h"], c["E"], c["K"], c["tokens"]
        group = c["group"]
        self.router = Matrix(gen, h, E, 1, c["rbits"], 64)
        self.gate = Matrix(gen, h, c["ff"], E, c["bits"], group)
        self.up = Matrix(gen, h, c["ff"], E, c["bits"], group)
        self.down = Matrix(gen, c["ff"], h, E, c["bits"], group)
        self.shared = None
        if c["ffs"]:
            sg = group if c["sbits"] == c["bits"] else 64
            self.shared = [Matrix(gen, h, c["ffs"], 1, c["sbits"], sg), Matrix(gen, h, c["ffs"], 1, c["sbits"], sg),
                           Matrix(gen, c["ffs"], h, 1, c["sbits"], sg), Matrix(gen, h, 1, 1, 0, 64)]
        self.norm = 1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda") if c["norm"] else None
        n = T + T // 8 + 16
        x = torch.randn(n, h, generator=gen, device="cuda")
        bias = None
        if c["skew"] == "zipf":
            rank = torch.randperm(E, generator=gen, device="cuda").float() + 1
            bias = (-1.1 * torch.log(rank)).expand(n, E).contiguous()
        elif c["skew"] == "hot":
            hot = torch.randperm(E, generator=gen, device="cuda")[:16]
            tok = torch.rand(n, generator=gen, device="cuda") < 0.2
            bias = torch.zeros(n, E, device="cuda")
            bias[:, hot] = 8.0 * tok.float()[:, None]
        x64 = x.double() if self.norm is None else rms(x.double(), self.norm.double())
        logits = x64 @ self.router.f64().T
        if bias is not None:
            logits = logits + bias.double()
        top = logits.topk(K + 1, 1).values
        keep = torch.argsort((top[:, K - 1] - top[:, K] < GAP).int(), stable=True)[:T]
        keep = keep.sort().values
        self.x = x[keep].contiguous()
        self.bias = bias[keep].contiguous() if bias is not None else None
        self.logits = logits[keep]

    def exact(self, c):
        """The block's output in 64 bits."""
        K = c["K"]
        x = self.x.double()
        xn = x if self.norm is None else rms(x, self.norm.double())
        v, ids = self.logits.topk(K, 1)
        w = torch.softmax(v, 1)  # softmax over all experts, then renormalised over the selected
        out = torch.zeros_like(x)
        for e in torch.unique(ids).tolist():
            t, k = (ids == e).nonzero(as_tuple=True)
            a = xn[t]
            g, u = a @ self.gate.f64(e).T, a @ self.up.f64(e).T
            out.index_add_(0, t, (torch.sigmoid(g) * g * u) @ self.down.f64(e).T * w[t, k][:, None])
        if self.shared:
            sg, su, sd, gi = (m.f64() for m in self.shared)
            g, u = xn @ sg.T, xn @ su.T
            out = out + (torch.sigmoid(g) * g * u) @ sd.T * torch.sigmoid(xn @ gi.T)
        return out + x if c["norm"] else out


def generator(case, seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * seed + 17 * case["tokens"] + case["bits"])


def linear_inputs(c, seed):
    gen = generator(c, seed)
    ws = [Matrix(gen, c["rows"], int(o), 1, c["bits"], c["group"], c["stype"]) for o in c["outs"].split(",")]
    return torch.randn(c["tokens"], c["rows"], generator=gen, device="cuda"), ws


# ------------------------------------------------------------------- state --
_GPU = []


def gpu():
    from hip_backend import Gpu

    if not _GPU:
        _GPU.append(Gpu())
    return _GPU[0]


class State:
    """Torch device memory bound to the framework in place (moe_register) and
    what a pass is issued with."""

    def __init__(self):
        from hip_backend import load_library

        self.gpu, self.lib = gpu(), load_library()
        self.tensors, self.owned, self.graph = [], [], None

    def adopt(self, t):
        n = t.numel() * t.element_size()
        if self.lib.moe_register(self.gpu._h, ctypes.c_void_p(t.data_ptr()), n) != 0:
            raise RuntimeError(self.lib.moe_last_error(self.gpu._h).decode())
        self.tensors.append(t)
        return t

    def buffer(self, t):
        from hip_backend import Buffer
        from hip_backend.api import MoeBufferC

        self.adopt(t)
        c = MoeBufferC()
        c.ptr, c.len = t.data_ptr(), t.numel()
        return Buffer(self.gpu, c, t.data_ptr())

    def zeros(self, *shape):
        t = torch.zeros(*shape, device="cuda")
        return t, self.buffer(t)

    def weight(self, m, dims):
        from hip_backend import BF16, F16, F32, Weight
        from hip_backend.api import MoeRegionC, MoeWeightC

        c = MoeWeightC()
        regions = []
        for t in m.parts:
            self.adopt(t)
            r = MoeRegionC()
            r.ptr, r.bytes = t.data_ptr(), t.numel() * t.element_size()
            regions.append(r)
        c.data = regions[0]
        if m.bits:
            c.scales, c.biases = regions[1], regions[2]
            c.scale_type = {"bf16": BF16, "f16": F16, "f32": F32}[m.stype]
            c.group_size = m.group
        c.bits = m.bits
        c.ndims = len(dims)
        for i, d in enumerate(dims):
            c.dims[i] = d
        return Weight(c, regions, dims, m.bits)

    def packed(self, w):
        p = self.gpu.pack_weight(w)
        self.owned += p.buffers
        return p

    def __del__(self):
        try:
            if self.graph is not None:
                self.graph.destroy()
            for t in self.tensors:
                self.lib.moe_unregister(self.gpu._h, ctypes.c_void_p(t.data_ptr()))
            for b in self.owned:
                self.gpu.release(b)
        except Exception:
            pass


def prepare(case, seed):
    from hip_backend import BlockWeights

    s = State()
    s.case = case
    if case["kind"] == "linear":
        x, ws = linear_inputs(case, seed)
        s.x = s.buffer(x)
        s.weights = [s.weight(m, [m.n_in, m.out]) for m in ws]
        s.outs = [s.zeros(case["tokens"], m.out) for m in ws]
        torch.cuda.synchronize()
        return s
    gen = generator(case, seed)
    h, E, ff, ffs, T = case["h"], case["E"], case["ff"], case["ffs"], case["tokens"]
    s.layers, s.outs = [], []
    s.ws = None
    for _ in range(case["layers"]):
        n = LayerInputs(case, gen)
        lay = {}
        lay["router"] = s.weight(n.router, [h, E])
        ex = [s.weight(n.gate, [h, ff, E]), s.weight(n.up, [h, ff, E]), s.weight(n.down, [ff, h, E])]
        sh = sgi = None
        if n.shared:
            sh = [s.weight(m, d) for m, d in zip(n.shared[:3], ([h, ffs], [h, ffs], [ffs, h]))]
            sgi = s.weight(n.shared[3], [h])
        lay["x"] = s.buffer(n.x)
        lay["bias"] = s.buffer(n.bias) if n.bias is not None else None
        lay["norm"] = s.buffer(n.norm) if n.norm is not None else None
        out, lay["out"] = s.zeros(T, h)
        s.outs.append(out)
        if case["kind"] == "ops":
            lay.update(ops_buffers(s, n, lay, ex, sh, sgi))
        else:
            torch.cuda.synchronize()
            pk = [s.packed(w) for w in ex] if case["packed"] else None
            spk = [s.packed(w) for w in sh] if case["packed"] and sh else None
            lay["bw"] = BlockWeights(lay["router"], *ex, case["K"], True, sh, sgi, packed=pk, shared_packed=spk)
            if s.ws is None:
                _, s.ws = s.zeros(lay["bw"].workspace_elems(T))
        s.layers.append(lay)
    torch.cuda.synchronize()
    if case["graph"]:
        cap = s.gpu.capture()
        with cap as b:
            issue_block(s, b)
        s.graph = cap.graph
    return s


def ops_buffers(s, n, lay, ex, sh, sgi):
    from hip_backend import Weight

    c = s.case
    h, E, K, ff, ffs = c["h"], c["E"], c["K"], c["ff"], c["ffs"]
    d = {"ex": ex, "sh": sh}
    if sgi is not None:
        d["sgi"] = sgi.reshape([h, 1])
    sizes = {"xn": h, "logits": E, "ids": K, "w": K, "gates": K * ff, "ups": K * ff, "eo": K * h, "proj": h,
             "sg": max(ffs, 1), "su": max(ffs, 1), "so": h, "gv": 1}
    for k, v in sizes.items():
        d[k] = s.zeros(v)[1]
    if n.norm is not None:  # the op takes its weight as a tensor
        from hip_backend.api import MoeRegionC, MoeWeightC

        w = MoeWeightC()
        w.data = MoeRegionC()
        w.data.ptr, w.data.bytes = n.norm.data_ptr(), 4 * h
        w.ndims = 1
        w.dims[0] = h
        d["norm_w"] = Weight(w, [w.data], [h], 0)
    return d


# ------------------------------------------------------------------ passes --
def issue_block(s, b):
    c = s.case
    for lay in s.layers:
        b.moe_block(lay["bw"], lay["x"], lay["out"], c["tokens"], s.ws, logit_bias=lay["bias"],
                    norm_weight=lay["norm"], norm_eps=1e-6, residual=c["norm"])


def issue_ops(s, b):
    """The block of one token as its ops: norm, router, routing, expert
    products, mix, shared expert, residual."""
    for L in s.layers:
        x = L["x"]
        if s.case["norm"]:
            b.norm(x, L["norm_w"], L["xn"], 1, s.case["h"], 1e-6)
            x = L["xn"]
        b.matmul(L["router"], x, L["logits"], 1)
        b.route(L["logits"], L["ids"], L["w"], True)
        b.expert_matmul(L["ex"][0], x, L["ids"], L["gates"], False)
        b.expert_matmul(L["ex"][1], x, L["ids"], L["ups"], False)
        b.swiglu(L["gates"], L["ups"], L["gates"])
        b.expert_matmul(L["ex"][2], L["gates"], L["ids"], L["eo"], True)
        to = L["proj"] if L["sh"] or s.case["norm"] else L["out"]
        b.mix(L["eo"], L["w"], to)
        if L["sh"]:
            b.matmul(L["sh"][0], x, L["sg"], 1)
            b.matmul(L["sh"][1], x, L["su"], 1)
            b.swiglu(L["sg"], L["su"], L["sg"])
            b.matmul(L["sh"][2], L["sg"], L["so"], 1)
            b.matmul(L["sgi"], x, L["gv"], 1)
            b.gate_scalar(L["so"], L["gv"], L["so"])
            b.add(to, L["so"], L["proj"] if s.case["norm"] else L["out"])
        if s.case["norm"]:
            b.add(L["x"], L["proj"], L["out"])


def run(state):
    s = state
    with s.gpu.batch() as b:
        if s.graph is not None:
            b.graph(s.graph)
        elif s.case["kind"] == "block":
            issue_block(s, b)
        elif s.case["kind"] == "ops":
            issue_ops(s, b)
        else:
            for w, (_, y) in zip(s.weights, s.outs):
                b.matmul(w, s.x, y, s.case["tokens"])
            return [t for t, _ in s.outs]
    return list(s.outs)


# ------------------------------------------------------- work, tolerance, exact --
def matrix_bytes(n_in, out, bits, group, scale=2):
    return 4 * n_in * out if bits == 0 else n_in * out * bits // 8 + 2 * scale * (n_in * out // group)


def work(case):
    T = case["tokens"]
    if case["kind"] == "linear":
        outs = [int(o) for o in case["outs"].split(",")]
        sb = 4 if case["stype"] == "f32" else 2
        return {"bytes": sum(matrix_bytes(case["rows"], o, case["bits"], case["group"], sb) for o in outs)
                + 4 * T * (case["rows"] + sum(outs)),
                "flops": 2 * T * case["rows"] * sum(outs)}
    h, E, K, ff, ffs = case["h"], case["E"], case["K"], case["ff"], case["ffs"]
    distinct = E * (1.0 - (1.0 - K / E) ** T)  # of a routing without skew
    if case["skew"] == "hot":
        # a fifth of the tokens choose among 16 experts
        distinct = min(E, 16 * (T > 4) + (E - 16) * (1.0 - (1.0 - K / E) ** (0.8 * T)))
    elif case["skew"] == "zipf":
        p = np.arange(1, E + 1) ** -1.1
        distinct = float(np.sum(1.0 - (1.0 - np.minimum(1.0, K * p / p.sum())) ** T))
    by = distinct * 3 * matrix_bytes(h, ff, case["bits"], case["group"]) + matrix_bytes(h, E, case["rbits"], 64)
    fl = 2 * T * (3 * h * ff * K + h * E)
    if ffs:
        sg = case["group"] if case["sbits"] == case["bits"] else 64
        by += 3 * matrix_bytes(h, ffs, case["sbits"], sg) + 4 * h
        fl += 2 * T * (3 * h * ffs + h)
    by += 8 * T * h + (4 * T * E if case["skew"] != "none" else 0) + (4 * h if case["norm"] else 0)
    return {"bytes": int(by) * case["layers"], "flops": int(fl) * case["layers"]}


def tolerance(case):
    # segments of 16 pairs and more on average take bf16 operands, all else is
    # F32 (the rule moe_block documents for its default path).  Measured
    # against 64 bits: bf16 4.3e-3, F32 1.1e-6; with the residual (about seven
    # times the block's own output) 6.7e-4 and 1.5e-7.
    bf16 = case["kind"] == "block" and case["tokens"] * case["K"] >= 16 * case["E"] and case["tokens"] > 1
    residual = case["kind"] != "linear" and case["norm"]
    if bf16:
        return {"rel": 3e-3 if residual else 1.5e-2}
    return {"rel": 1e-6 if residual else 6e-6}


def exact(case, seed):
    if case["kind"] == "linear":
        x, ws = linear_inputs(case, seed)
        return [x.double() @ m.f64().T for m in ws]
    gen = generator(case, seed)
    return [LayerInputs(case, gen).exact(case) for _ in range(case["layers"])]
