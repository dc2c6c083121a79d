"""What the framework's speed is measured on: the layers and steps that an
engine has this library run, through the public calls of cuca_amd.hip.

Every case names its kind (a class below), one of the model shapes of
cuca_amd.workloads.CONFIGS, and its sizes.  `listed` are the fixed cases,
`draw` gives another one of the same ranges, `prepare` builds what a program
holds before the call (inputs, packed weights, pools, workspaces, a captured
graph), `run` makes one pass, `exact` computes the outputs in 64 bits with
plain torch.
"""

import math

import numpy as np
import torch

from cuca_amd import hip
from cuca_amd import workloads as W

DEV = "cuda"
DTYPE = {"f32": torch.float32, "f16": torch.float16}
CODE = {"f32": hip.F32, "f16": hip.F16}
SIZE = {"f32": 4, "f16": 2}
ACT = {"silu": hip.ACT_SILU, "gelu": hip.ACT_GELU_TANH}
ROPE = {"neox": hip.ROPE_NEOX, "norm": hip.ROPE_NORM}
# block scales that give a projection outputs of order one
SCALES = {"q4_0": {"up": (0.001, 0.01), "down": (0.0005, 0.005)},
          "q8_0": {"up": (0.0001, 0.0007), "down": (0.00005, 0.00035)}}

_context = None


def context():
    """The program's one context, on its own stream."""
    global _context
    if _context is None:
        _context = hip.Context(0)
    return _context


def qbytes(qtype, n, k):
    return n * W.row_bytes(qtype, k)


def dequantised(raw, qtype, n, k):
    """The weight's values in 64 bits, from the GGUF bytes."""
    blocks = raw.view(n, k // 32, W.BLOCK_BYTES[qtype])
    d = blocks[..., 0:2].contiguous().view(torch.float16).double()
    q = blocks[..., 2:]
    if qtype == "q4_0":
        q = torch.cat([(q & 15).to(torch.int8), (q >> 4).to(torch.int8)], -1).double() - 8.0
    else:
        q = q.contiguous().view(torch.int8).double()
    return (q * d).view(n, k)


def q8_rows(x):
    """Activations as the bit-exact matmul sees them: Q8_0 blocks of 32 (f32
    scale amax / 127, ties away from zero, the scale then held in f16)."""
    b = x.float().view(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    v = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = (torch.sign(v) * torch.floor(v.abs().double() + 0.5)).clamp(-128, 127)
    return (q * d.half().double()).view(x.shape)


def act64(kind, g):
    if kind == "silu":
        return g / (1.0 + torch.exp(-g))
    return 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))


def rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 if w is None else w.double())


def rope64(x, cos, sin, kind, pos):
    """x [rows, heads, d], all of d rotated."""
    c, s = cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
    half = x.shape[-1] // 2
    if kind == "neox":
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * c - b * s, a * s + b * c], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


class Base:
    def __init__(self, case, seed):
        self.case, self.cfg = case, W.CONFIGS[case["config"]]
        self.gen = torch.Generator(device=DEV).manual_seed(seed)
        self.rng = np.random.default_rng(seed)
        self.inputs()

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, device=DEV, generator=self.gen) * std).to(dtype)

    def gain(self, n):
        return 1.0 + 0.02 * torch.randn((n,), device=DEV, generator=self.gen)

    def raw(self, n, k, qtype, what="up"):
        return W.quant_table_torch(self.gen, n, k, qtype, SCALES[qtype][what])

    @staticmethod
    def packed(raw, n, k, qtype):
        out = torch.empty(hip.qweight_bytes(W.GGML_ID[qtype], n, k), dtype=torch.uint8, device=DEV)
        torch.cuda.synchronize()  # the context works on a stream of its own
        context().qweight_pack(raw.data_ptr(), W.GGML_ID[qtype], n, k, out.data_ptr())
        context().sync()
        return out

    def blocks(self, count):
        """`count` pool blocks in the order an engine's free list left them."""
        return self.rng.permutation(count).astype(np.int32)

    def rope_tables(self, positions):
        cos, sin = hip.rope_tables(ROPE[self.cfg["rope"]], self.cfg["head_dim"], self.cfg["theta"], positions)
        return torch.from_numpy(cos).to(DEV), torch.from_numpy(sin).to(DEV)

    def setup(self):
        torch.cuda.synchronize()
        return self

    def exact(self):
        return None


class DecodeStep(Base):
    """A whole decode step: gather, layers (norm, Q|K|V, RoPE and K/V store,
    paged attention, o, norm, gate/up, down), final norm, LM head, greedy id;
    f32 with the CPU engine's bits in every projection, captured in a graph
    once and replayed per token, as the engine does."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        H, F, d, nq, nk = cfg["hidden"], cfg["ff"], cfg["head_dim"], cfg["nq"], cfg["nk"]
        n, V, qt = c["rows"], cfg["vocab"], c["qtype"]
        self.table = W.quant_table_torch(self.gen, V, H, "q8_0", cfg["d_range"])
        self.head = self.packed(self.raw(V, H, "q8_0"), V, H, "q8_0")
        per = (c["keys"] + 15) // 16
        self.n_blocks, self.max_blocks = n * per, per
        self.layers = []
        for _ in range(c["layers"]):
            w = {}
            for name, rows, cols in (("qkv", (nq + 2 * nk) * d, H), ("o", H, nq * d), ("g", F, H), ("u", F, H),
                                     ("d", H, F)):
                w[name] = self.packed(self.raw(rows, cols, qt, "down" if name == "d" else "up"), rows, cols, qt)
            w["n1"], w["n2"] = self.gain(H), self.gain(H)
            w["pk"], w["pv"] = self.normal(n * per, nk, 16, d), self.normal(n * per, nk, 16, d)
            self.layers.append(w)
        self.nout = self.gain(H)
        self.ids = torch.randint(0, V, (n,), device=DEV, generator=self.gen, dtype=torch.int32)
        keys = self.rng.integers((c["keys"] + 1) // 2, c["keys"] + 1, n).astype(np.int32)
        keys[0] = c["keys"]
        tables = self.blocks(n * per).reshape(n, per)
        self.tables = torch.from_numpy(tables).to(DEV)
        self.pos = torch.from_numpy(keys - 1).to(DEV)
        self.slots = torch.from_numpy(np.concatenate(
            [hip.kv_slots(tables[r].astype(np.uint32), int(keys[r]) - 1, 1, n * per) for r in range(n)])).to(DEV)
        self.ranges = torch.from_numpy(np.stack([np.zeros(n, np.int32), keys], 1).copy()).to(DEV)
        self.positions = c["keys"]
        self.cos, self.sin = self.rope_tables(self.positions)

    def setup(self):
        c, cfg = self.case, self.cfg
        H, F, d, nq, nk = cfg["hidden"], cfg["ff"], cfg["head_dim"], cfg["nq"], cfg["nk"]
        n, V = c["rows"], cfg["vocab"]
        z = lambda *s: torch.zeros(s, device=DEV)  # noqa: E731
        self.x, self.mid, self.h, self.ffn, self.attn = z(n, H), z(n, H), z(n, H), z(n, H), z(n, H)
        self.qkv, self.o, self.act, self.logits = z(n, (nq + 2 * nk) * d), z(n, nq * d), z(n, F), z(n, V)
        self.out_ids = torch.zeros((n,), device=DEV, dtype=torch.int32)
        self.ws_bytes = hip.paged_decode_workspace(n, nq, d, self.max_blocks)
        self.ws = torch.empty(max(self.ws_bytes, 16), dtype=torch.uint8, device=DEV)
        torch.cuda.synchronize()
        context().graph_begin()
        self.issue()
        self.graph = context().graph_end()
        return super().setup()

    def issue(self):
        c, cfg, x = self.case, self.cfg, context()
        H, F, d, nq, nk, eps = (cfg[k] for k in ("hidden", "ff", "head_dim", "nq", "nk", "eps"))
        n, V, T, f32 = c["rows"], cfg["vocab"], W.GGML_ID[c["qtype"]], hip.F32
        wide, kind = (nq + 2 * nk) * d, ROPE[cfg["rope"]]
        p = lambda t: t.data_ptr()  # noqa: E731
        x.embed_gguf(p(self.table), hip.GGML_Q8_0, V, H, p(self.ids), n, 1.0, p(self.x), f32)
        q = p(self.qkv)
        for i, l in enumerate(self.layers):
            branch = p(self.ffn) if i else None
            if kind == hip.ROPE_NORM:
                x.add_rmsnorm_qmm_rope_store_kv(p(self.x), branch, p(l["n1"]), eps, 1.0, p(self.mid), p(self.h),
                                                p(l["qkv"]), T, H, n, nq, nk, d, d, kind, p(self.cos), p(self.sin),
                                                self.positions, p(self.pos), q, wide, p(l["pk"]), p(l["pv"]),
                                                self.n_blocks, p(self.slots), f32)
            else:
                x.add_rmsnorm_qmm(p(self.x), branch, p(l["n1"]), eps, 1.0, p(self.mid), p(self.h), p(l["qkv"]), T,
                                  wide, H, n, wide, q, wide, f32)
                x.rope_store_kv(q, wide, q + 4 * nq * d, wide, q + 4 * (nq + nk) * d, wide, n, nq, nk, d, d, kind,
                                p(self.cos), p(self.sin), self.positions, p(self.pos), None, None, 0, eps,
                                p(l["pk"]), p(l["pv"]), self.n_blocks, p(self.slots), f32)
            x.paged_decode(q, p(l["pk"]), p(l["pv"]), self.n_blocks, p(self.tables), self.max_blocks,
                           p(self.ranges), n, nq, nk, d, 1.0 / math.sqrt(d), p(self.ws), self.ws_bytes, p(self.o),
                           f32, q_ld=wide)
            x.qmm(p(l["o"]), T, H, nq * d, p(self.o), nq * d, n, H, p(self.attn), H, f32)
            x.add_rmsnorm_qmm_glu(p(self.mid), p(self.attn), p(l["n2"]), eps, 1.0, p(self.x), p(self.h), p(l["g"]),
                                  p(l["u"]), T, F, H, n, ACT[cfg["act"]], 0.0, p(self.act), F, f32)
            x.qmm(p(l["d"]), T, H, F, p(self.act), F, n, H, p(self.ffn), H, f32)
        x.add_rmsnorm_qmm(p(self.x), p(self.ffn), p(self.nout), eps, 1.0, None, p(self.h), p(self.head),
                          hip.GGML_Q8_0, V, H, n, V, p(self.logits), V, f32)
        x.argmax(p(self.logits), V, n, V, f32, p(self.out_ids))

    def run(self):
        self.graph.launch()
        return {"logits": self.logits, "h": self.h}

    @staticmethod
    def work(c, cfg):
        H, F, d, nq, nk, V = (cfg[k] for k in ("hidden", "ff", "head_dim", "nq", "nk", "vocab"))
        values = (nq + 2 * nk) * d * H + H * nq * d + 3 * F * H
        weights = qbytes(c["qtype"], values // 32, 32)
        keys = c["keys"] * (1 + 0.75 * (c["rows"] - 1))
        return {"bytes": c["layers"] * (weights + keys * 2 * nk * d * 4) + qbytes("q8_0", V, H)
                + c["rows"] * (V * 4 + H * 4),
                "flops": 2.0 * c["rows"] * (c["layers"] * values + V * H) + c["layers"] * 4.0 * keys * nq * d}

    # the sums of one attention, rounded in another order, flip a few of the
    # next projection's Q8_0 roundings, which every later layer carries on
    # (values perturbed by 2e-7 moved the logits by up to 5e-4)
    @staticmethod
    def tolerance(c):
        return {"rel": 0.006, "max": 0.06}


class MlpQmm(Base):
    """The gate/up + activation and down projections of a few rows with the
    CPU engine's bits: small decode batches, speculative verification."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        H, F, qt = cfg["hidden"], cfg["ff"], c["qtype"]
        self.raws = [self.raw(F, H, qt), self.raw(F, H, qt), self.raw(H, F, qt, "down")]
        self.x = self.normal(c["rows"], H)

    def setup(self):
        H, F, qt, n = self.cfg["hidden"], self.cfg["ff"], self.case["qtype"], self.case["rows"]
        g, u, d = self.raws
        self.raws = None
        self.g, self.u, self.d = self.packed(g, F, H, qt), self.packed(u, F, H, qt), self.packed(d, H, F, qt)
        self.act, self.out = torch.zeros((n, F), device=DEV), torch.zeros((n, H), device=DEV)
        return super().setup()

    def run(self):
        H, F, T, n = self.cfg["hidden"], self.cfg["ff"], W.GGML_ID[self.case["qtype"]], self.case["rows"]
        x = context()
        x.qmm_glu(self.g.data_ptr(), self.u.data_ptr(), T, F, H, self.x.data_ptr(), H, n, ACT[self.cfg["act"]],
                  0.0, self.act.data_ptr(), F, hip.F32)
        x.qmm(self.d.data_ptr(), T, H, F, self.act.data_ptr(), F, n, H, self.out.data_ptr(), H, hip.F32)
        return {"hidden": self.act, "out": self.out}

    def exact(self):
        H, F, qt = self.cfg["hidden"], self.cfg["ff"], self.case["qtype"]
        x = q8_rows(self.x)
        g, u = (x @ dequantised(r, qt, F, H).T for r in self.raws[:2])
        # down reads the rounded quants of the hidden row: no 64-bit value
        return {"hidden": act64(self.cfg["act"], g) * u, "out": None}

    @staticmethod
    def work(c, cfg):
        H, F, n = cfg["hidden"], cfg["ff"], c["rows"]
        return {"bytes": 3 * qbytes(c["qtype"], F, H) + n * (2 * H + 2 * F) * 4, "flops": 6.0 * n * F * H}

    # an activation a rounding apart can flip a Q8_0 quant of the hidden row
    @staticmethod
    def tolerance(c):
        return {"rel": 1e-3, "max": 0.02}


class Projections(Base):
    """A layer's four projections (Q|K|V, o, gate/up with the activation,
    down) for a batch of rows on the matrix cores, from the quantised weights
    (`resident` false) or from their resident f16 copy (true)."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        H, F, d, qt = cfg["hidden"], cfg["ff"], cfg["head_dim"], c["qtype"]
        dt = DTYPE[c["dtype"]]
        self.shapes = {"qkv": ((cfg["nq"] + 2 * cfg["nk"]) * d, H), "o": (H, cfg["nq"] * d), "g": (F, H),
                       "u": (F, H), "d": (H, F)}
        self.raws = {k: self.raw(*s, qt, "down" if k == "d" else "up") for k, s in self.shapes.items()}
        self.h, self.h2 = self.normal(c["rows"], H, dtype=dt), self.normal(c["rows"], H, dtype=dt)
        self.attn = self.normal(c["rows"], cfg["nq"] * d, std=0.3, dtype=dt)

    def setup(self):
        c, cfg, ctx = self.case, self.cfg, context()
        H, F, qt, n, dt = cfg["hidden"], cfg["ff"], c["qtype"], c["rows"], DTYPE[c["dtype"]]
        T = W.GGML_ID[qt]
        self.w = {k: self.packed(r, *self.shapes[k], qt) for k, r in self.raws.items()}
        self.raws = None
        if c["resident"]:
            full = {k: torch.empty(s, dtype=torch.float16, device=DEV) for k, s in self.shapes.items() if k in "qkvod"}
            full["gu"] = torch.empty((2 * F, H), dtype=torch.float16, device=DEV)
            for k, (rows, cols) in self.shapes.items():
                to = full["gu"][F if k == "u" else 0:] if k in "gu" else full[k]
                ctx.qweight_dequant(self.w[k].data_ptr(), T, rows, cols, to.data_ptr())
            ctx.sync()
            self.w = full
            sizes = [hip.gemm_w16_workspace(rows, cols, n, k == "g", CODE[c["dtype"]])
                     for k, (rows, cols) in self.shapes.items()]
        else:
            sizes = [hip.qgemm_workspace(T, rows, cols, n, k == "g") for k, (rows, cols) in self.shapes.items()]
        self.ws_bytes = max(sizes)
        self.ws = torch.empty(max(self.ws_bytes, 16), dtype=torch.uint8, device=DEV)
        z = lambda k: torch.zeros((n, k), device=DEV, dtype=dt)  # noqa: E731
        self.outs = {"qkv": z(self.shapes["qkv"][0]), "o": z(H), "act": z(F), "down": z(H)}
        return super().setup()

    def run(self):
        c, cfg, x, o = self.case, self.cfg, context(), self.outs
        H, F, n, T, code = cfg["hidden"], cfg["ff"], c["rows"], W.GGML_ID[c["qtype"]], CODE[c["dtype"]]
        ws = (self.ws.data_ptr(), self.ws_bytes)

        def plain(k, src, dst):
            rows, cols = self.shapes[k]
            if c["resident"]:
                x.gemm_w16(self.w[k].data_ptr(), rows, cols, src.data_ptr(), cols, n, rows, *ws, dst.data_ptr(),
                           rows, code)
            else:
                x.qgemm(self.w[k].data_ptr(), T, rows, cols, src.data_ptr(), cols, n, rows, *ws, dst.data_ptr(),
                        rows, code)

        plain("qkv", self.h, o["qkv"])
        plain("o", self.attn, o["o"])
        if c["resident"]:
            x.gemm_w16_glu(self.w["gu"].data_ptr(), F, H, self.h2.data_ptr(), H, n, ACT[cfg["act"]], 0.0, *ws,
                           o["act"].data_ptr(), F, code)
        else:
            x.qgemm_glu(self.w["g"].data_ptr(), self.w["u"].data_ptr(), T, F, H, self.h2.data_ptr(), H, n,
                        ACT[cfg["act"]], 0.0, *ws, o["act"].data_ptr(), F, code)
        plain("d", o["act"], o["down"])
        return o

    def exact(self):
        qt = self.case["qtype"]
        mul = lambda x, k: x.double() @ dequantised(self.raws[k], qt, *self.shapes[k]).T  # noqa: E731
        act = act64(self.cfg["act"], mul(self.h2, "g")) * mul(self.h2, "u")
        return {"qkv": mul(self.h, "qkv"), "o": mul(self.attn, "o"), "act": act, "down": mul(act, "d")}

    @staticmethod
    def work(c, cfg):
        H, F, d, n, s = cfg["hidden"], cfg["ff"], cfg["head_dim"], c["rows"], SIZE[c["dtype"]]
        wide = (cfg["nq"] + 2 * cfg["nk"]) * d
        values = wide * H + H * cfg["nq"] * d + 3 * F * H
        w = 2 * values if c["resident"] else qbytes(c["qtype"], values // 32, 32)
        return {"bytes": w + n * s * (2 * H + cfg["nq"] * d + wide + 2 * H + 2 * F), "flops": 2.0 * n * values}

    # one f16 rounding of each operand (and of f16 results), f32 sums
    @staticmethod
    def tolerance(c):
        return {"rel": 2e-3, "max": 0.04}


class AttendRows(Base):
    """Attention of a prefill chunk (or of verification rows) of one sequence
    over its paged cache: `rows` queries after `past` cached positions, causal,
    with a sliding window where `window` is not 0."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        d, nq, nk, dt = cfg["head_dim"], cfg["nq"], cfg["nk"], DTYPE[c["dtype"]]
        keys = c["past"] + c["rows"]
        self.per = (keys + 15) // 16
        self.pk, self.pv = (self.normal(self.per, nk, 16, d, dtype=dt) for _ in range(2))
        self.q = self.normal(c["rows"], nq, d, dtype=dt)
        self.order = self.blocks(self.per)
        hi = np.arange(c["past"] + 1, keys + 1, dtype=np.int32)
        lo = np.maximum(hi - c["window"], 0) if c["window"] else np.zeros_like(hi)
        self.lo, self.hi = lo.astype(np.int32), hi

    def setup(self):
        self.table = torch.from_numpy(self.order).to(DEV)
        self.ranges = torch.from_numpy(np.stack([self.lo, self.hi], 1).copy()).to(DEV)
        self.out = torch.zeros_like(self.q)
        return super().setup()

    def run(self):
        c, cfg = self.case, self.cfg
        d, nq, nk = cfg["head_dim"], cfg["nq"], cfg["nk"]
        context().attend_rows(self.q.data_ptr(), nq * d, self.pk.data_ptr(), self.pv.data_ptr(), self.per,
                              self.table.data_ptr(), self.per, self.ranges.data_ptr(), c["rows"], nq, nk, d,
                              1.0 / math.sqrt(d), self.out.data_ptr(), nq * d, CODE[c["dtype"]])
        return self.out

    def exact(self):
        c, cfg = self.case, self.cfg
        d, nq, nk = cfg["head_dim"], cfg["nq"], cfg["nk"]
        at = torch.from_numpy(self.order).to(DEV).long()
        keys = c["past"] + c["rows"]
        j = torch.arange(keys, device=DEV)
        lo, hi = torch.from_numpy(self.lo).to(DEV)[:, None], torch.from_numpy(self.hi).to(DEV)[:, None]
        seen = (j >= lo) & (j < hi)
        out = torch.empty(self.q.shape, dtype=torch.float64, device=DEV)
        for h in range(nq):
            g = h // (nq // nk)
            k, v = (t[at, g].reshape(-1, d)[:keys].double() for t in (self.pk, self.pv))
            s = (self.q[:, h].double() @ k.T) / math.sqrt(d)
            out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v
        return out

    @staticmethod
    def work(c, cfg):
        d, nq, nk, s = cfg["head_dim"], cfg["nq"], cfg["nk"], SIZE[c["dtype"]]
        hi = np.arange(c["past"] + 1, c["past"] + c["rows"] + 1, dtype=np.float64)
        seen = float((np.minimum(hi, c["window"]) if c["window"] else hi).sum())
        first = max(0, c["past"] + 1 - c["window"]) if c["window"] else 0
        return {"bytes": s * (2 * c["rows"] * nq * d + 2 * (c["past"] + c["rows"] - first) * nk * d),
                "flops": 4.0 * seen * nq * d}

    @staticmethod
    def tolerance(c):
        return {"rel": 1e-3, "max": 0.01} if c["dtype"] == "f16" else {"rel": 1e-5, "max": 2e-4}


class PagedDecode(Base):
    """Paged decode attention of a batch of sequences of ragged lengths (from
    half of `keys` up to `keys`), one query row each."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        d, nq, nk, dt = cfg["head_dim"], cfg["nq"], cfg["nk"], DTYPE[c["dtype"]]
        n, per = c["rows"], (c["keys"] + 15) // 16
        self.per = per
        self.pk, self.pv = (self.normal(n * per, nk, 16, d, dtype=dt) for _ in range(2))
        self.q = self.normal(n, nq, d, dtype=dt)
        self.order = self.blocks(n * per).reshape(n, per)
        self.keys = self.rng.integers((c["keys"] + 1) // 2, c["keys"] + 1, n).astype(np.int32)
        self.keys[0] = c["keys"]

    def setup(self):
        c, cfg = self.case, self.cfg
        n = c["rows"]
        self.tables = torch.from_numpy(self.order).to(DEV)
        self.ranges = torch.from_numpy(np.stack([np.zeros(n, np.int32), self.keys], 1).copy()).to(DEV)
        self.ws_bytes = hip.paged_decode_workspace(n, cfg["nq"], cfg["head_dim"], self.per)
        self.ws = torch.empty(max(self.ws_bytes, 16), dtype=torch.uint8, device=DEV)
        self.out = torch.zeros_like(self.q)
        return super().setup()

    def run(self):
        c, cfg = self.case, self.cfg
        d, nq, nk, n = cfg["head_dim"], cfg["nq"], cfg["nk"], c["rows"]
        context().paged_decode(self.q.data_ptr(), self.pk.data_ptr(), self.pv.data_ptr(), n * self.per,
                               self.tables.data_ptr(), self.per, self.ranges.data_ptr(), n, nq, nk, d,
                               1.0 / math.sqrt(d), self.ws.data_ptr(), self.ws_bytes, self.out.data_ptr(),
                               CODE[c["dtype"]])
        return self.out

    def exact(self):
        cfg = self.cfg
        d, nq, nk = cfg["head_dim"], cfg["nq"], cfg["nk"]
        out = torch.empty(self.q.shape, dtype=torch.float64, device=DEV)
        for r in range(self.case["rows"]):
            at, keys = torch.from_numpy(self.order[r]).to(DEV).long(), int(self.keys[r])
            k, v = (t[at].transpose(0, 1).reshape(nk, -1, d)[:, :keys].double() for t in (self.pk, self.pv))
            q = self.q[r].double().view(nk, nq // nk, d)
            s = torch.softmax((q @ k.transpose(1, 2).contiguous()) / math.sqrt(d), -1)
            out[r] = (s @ v).view(nq, d)
        return out

    @staticmethod
    def work(c, cfg):
        d, nq, nk, s = cfg["head_dim"], cfg["nq"], cfg["nk"], SIZE[c["dtype"]]
        keys = c["keys"] * (1 + 0.75 * (c["rows"] - 1))
        return {"bytes": s * (2 * c["rows"] * nq * d + 2 * keys * nk * d), "flops": 4.0 * keys * nq * d}

    tolerance = AttendRows.tolerance


class Experts(Base):
    """The routed experts of a MoE layer: up (gate/up + activation), down
    (times the routing weight) and the sum per token; `cores` false is the
    decode path with the CPU engine's bits, true the grouped matrix-core
    GEMMs of a prefill.  Zipf(1.1) routing, pairs grouped by expert."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        H, F, qt, n = cfg["hidden"], cfg["ff"], c["qtype"], c["tokens"]
        E, used = cfg["moe"]
        self.raws = [self.raw(E * F, H, qt), self.raw(E * F, H, qt), self.raw(E * H, F, qt, "down")]
        self.x = self.normal(n, H, dtype=DTYPE[c["dtype"]])
        self.offsets, tok = W.zipf_expert_rows(self.rng, n, E, used)
        self.tok = tok.astype(np.int32)
        self.weight = self.rng.uniform(0.05, 0.3, tok.size).astype(np.float32)
        # a token's pairs in expert order
        self.token_pairs = np.argsort(tok, kind="stable").astype(np.int32).reshape(n, used)

    def setup(self):
        c, cfg = self.case, self.cfg
        H, F, qt, dt = cfg["hidden"], cfg["ff"], c["qtype"], DTYPE[c["dtype"]]
        E, used = cfg["moe"]
        T = W.GGML_ID[qt]
        torch.cuda.synchronize()  # the context works on a stream of its own
        self.pools, self.strides = [], []
        for raw, rows, cols in zip(self.raws, (F, F, H), (H, H, F)):
            one = (hip.qweight_bytes(T, rows, cols) + 15) // 16 * 16
            pool = torch.empty(E * one, dtype=torch.uint8, device=DEV)
            for e in range(E):
                context().qweight_pack(raw.data_ptr() + e * qbytes(qt, rows, cols), T, rows, cols,
                                       pool.data_ptr() + e * one)
            self.pools.append(pool)
            self.strides.append(one)
        context().sync()
        self.raws = None
        up = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
        self.d_off, self.d_tok, self.d_wt, self.d_tp = (up(self.offsets), up(self.tok), up(self.weight),
                                                        up(self.token_pairs))
        pairs = self.tok.size
        self.hidden = torch.zeros((pairs, F), device=DEV, dtype=dt)
        self.scratch = torch.zeros((pairs, H), device=DEV)
        self.out = torch.zeros((c["tokens"], H), device=DEV, dtype=dt)
        if c["cores"]:
            self.ws_bytes = max(hip.moe_qgemm_workspace(T, H, E, pairs), hip.moe_qgemm_workspace(T, F, E, pairs))
            self.ws = torch.empty(max(self.ws_bytes, 16), dtype=torch.uint8, device=DEV)
        return super().setup()

    def run(self):
        c, cfg, x = self.case, self.cfg, context()
        H, F, n, T, code = cfg["hidden"], cfg["ff"], c["tokens"], W.GGML_ID[c["qtype"]], CODE[c["dtype"]]
        E, used = cfg["moe"]
        pairs, act = self.tok.size, ACT[cfg["act"]]
        (g, u, d), (sg, _, sd) = (t.data_ptr() for t in self.pools), self.strides
        ws = (self.ws.data_ptr(), self.ws_bytes) if c["cores"] else ()
        (x.moe_up_qgemm if c["cores"] else x.moe_up)(
            g, u, sg, T, F, H, E, self.x.data_ptr(), H, n, self.d_off.data_ptr(), self.d_tok.data_ptr(), pairs, act,
            0.0, *ws, self.hidden.data_ptr(), F, code)
        (x.moe_down_qgemm if c["cores"] else x.moe_down)(
            d, sd, T, H, F, E, self.hidden.data_ptr(), F, self.d_off.data_ptr(), self.d_wt.data_ptr(), pairs, *ws,
            self.scratch.data_ptr(), H, code)
        x.moe_sum(self.scratch.data_ptr(), H, pairs, self.d_tp.data_ptr(), used, n, H, self.out.data_ptr(), H, code)
        return {"hidden": self.hidden, "out": self.out}

    def exact(self):
        c, cfg = self.case, self.cfg
        H, F, qt = cfg["hidden"], cfg["ff"], c["qtype"]
        E, _ = cfg["moe"]
        x = self.x.double() if c["cores"] else q8_rows(self.x)
        tok, wt = torch.from_numpy(self.tok).to(DEV).long(), torch.from_numpy(self.weight).to(DEV).double()
        hidden = torch.zeros((self.tok.size, F), device=DEV, dtype=torch.float64)
        out = torch.zeros((c["tokens"], H), device=DEV, dtype=torch.float64)
        for e in range(E):
            a, b = int(self.offsets[e]), int(self.offsets[e + 1])
            if a == b:
                continue
            wg, wu, wd = (dequantised(r.view(E, -1)[e], qt, rows, cols)
                          for r, rows, cols in zip(self.raws, (F, F, H), (H, H, F)))
            rows = x[tok[a:b]]
            hidden[a:b] = act64(cfg["act"], rows @ wg.T) * (rows @ wu.T)
            out.index_add_(0, tok[a:b], (hidden[a:b] @ wd.T) * wt[a:b, None])
        # with the CPU engine's bits down reads the hidden row's rounded quants
        return {"hidden": hidden, "out": out if c["cores"] else None}

    @staticmethod
    def work(c, cfg):
        H, F, s = cfg["hidden"], cfg["ff"], SIZE[c["dtype"]]
        E, used = cfg["moe"]
        n = c["tokens"]
        p = 1.0 / np.arange(1, E + 1) ** 1.1
        touched = float((1.0 - (1.0 - np.minimum(used * p / p.sum(), 1.0)) ** n).sum())
        return {"bytes": touched * 3 * qbytes(c["qtype"], F, H) + n * s * (2 * H + 2 * used * F),
                "flops": 6.0 * n * used * F * H}

    @staticmethod
    def tolerance(c):
        return {"rel": 2e-3, "max": 0.04}


class LayerOps(Base):
    """A layer's non-matmul sequence: the gather with the first norm, residual
    + norm (with the post-norm sandwich where the shape has one), RoPE (with
    the QK-norm where it has one) and the paged K/V store, the gated
    activation (over expert-grouped rows where the shape routes), residual +
    norm."""

    def inputs(self):
        c, cfg = self.case, self.cfg
        H, F, d, nq, nk, n = (*(cfg[k] for k in ("hidden", "ff", "head_dim", "nq", "nk")), c["rows"])
        dt, std = DTYPE[c["dtype"]], cfg["std"]
        self.table = W.quant_table_torch(self.gen, cfg["vocab"], H, cfg["qtype"], cfg["d_range"])
        self.ids = torch.randint(0, cfg["vocab"], (n,), device=DEV, generator=self.gen, dtype=torch.int32)
        self.w = [self.gain(H) for _ in range(5)]
        self.attn, self.ffn = self.normal(n, H, std=std, dtype=dt), self.normal(n, H, std=std, dtype=dt)
        self.q, self.k, self.v = (self.normal(n, h, d, std=std, dtype=dt) for h in (nq, nk, nk))
        self.qw, self.kw = (self.gain(d), self.gain(d)) if cfg.get("qk_norm") else (None, None)
        self.offsets = None
        self.ff_rows = n
        if "moe" in cfg:
            off, _ = W.zipf_expert_rows(self.rng, n, *cfg["moe"])
            self.offsets, self.ff_rows = torch.from_numpy(off).to(DEV), n * cfg["moe"][1]
        self.gate, self.up = (self.normal(self.ff_rows, F, std=std, dtype=dt) for _ in range(2))
        self.per = (n + 15) // 16
        self.slots_host = hip.kv_slots(self.blocks(self.per).astype(np.uint32), 0, n, self.per)
        self.pos = torch.arange(n, device=DEV, dtype=torch.int32)
        self.cos, self.sin = self.rope_tables(n)

    def setup(self):
        dt, cfg = DTYPE[self.case["dtype"]], self.cfg
        z = lambda *s: torch.zeros(s, device=DEV, dtype=dt)  # noqa: E731
        n, H = self.case["rows"], cfg["hidden"]
        self.slots = torch.from_numpy(self.slots_host).to(DEV)
        self.x, self.x1, self.x2, self.h0, self.h1, self.h2 = (z(n, H) for _ in range(6))
        self.act = z(self.ff_rows, cfg["ff"])
        self.pk, self.pv = (z(self.per, cfg["nk"], 16, cfg["head_dim"]) for _ in range(2))
        return super().setup()

    def run(self):
        c, cfg, x = self.case, self.cfg, context()
        H, F, d, nq, nk, eps, n = (*(cfg[k] for k in ("hidden", "ff", "head_dim", "nq", "nk", "eps")), c["rows"])
        code, act = CODE[c["dtype"]], ACT[cfg["act"]]
        p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
        post = (self.w[3], self.w[4]) if cfg.get("sandwich") else (None, None)
        x.embed_gguf_rms(p(self.table), W.GGML_ID[cfg["qtype"]], cfg["vocab"], H, p(self.ids), n, cfg["embd_scale"],
                         p(self.w[0]), eps, p(self.x), p(self.h0), code)
        # q is rotated in place: each pass rotates what the last one left, as
        # a buffer that every layer writes anew would be
        x.rope_store_kv(p(self.q), nq * d, p(self.k), nk * d, p(self.v), nk * d, n, nq, nk, d, d, ROPE[cfg["rope"]],
                        p(self.cos), p(self.sin), n, p(self.pos), p(self.qw), p(self.kw), 0, eps, p(self.pk),
                        p(self.pv), self.per, p(self.slots), code)
        x.add_rmsnorm(p(self.x), p(self.attn), p(self.w[1]), p(post[0]), eps, eps, 1.0, n, H, p(self.x1), p(self.h1),
                      code)
        if self.offsets is None:
            x.glu(p(self.gate), F, p(self.up), F, n, F, act, 0.0, p(self.act), F, code)
        else:
            x.glu_ragged(p(self.gate), F, p(self.up), F, p(self.offsets), cfg["moe"][0], self.ff_rows, F, act, 0.0,
                         p(self.act), F, code)
        x.add_rmsnorm(p(self.x1), p(self.ffn), p(self.w[2]), p(post[1]), eps, eps, 1.0, n, H, p(self.x2), p(self.h2),
                      code)
        return {"x": self.x, "h0": self.h0, "x1": self.x1, "h1": self.h1, "act": self.act, "x2": self.x2,
                "h2": self.h2, "k": self.pk, "v": self.pv}

    def exact(self):
        c, cfg = self.case, self.cfg
        n, eps, nk, d = c["rows"], cfg["eps"], cfg["nk"], cfg["head_dim"]
        table = self.table.view(cfg["vocab"], -1)[self.ids.long()]
        x = dequantised(table, cfg["qtype"], n, cfg["hidden"]) * cfg["embd_scale"]
        branch = lambda b, w: rms64(b.double(), w, eps) if cfg.get("sandwich") else b.double()  # noqa: E731
        x1 = x + branch(self.attn, self.w[3])
        x2 = x1 + branch(self.ffn, self.w[4])
        k = self.k.double() if self.kw is None else rms64(self.k.double(), self.kw, eps)
        slots = torch.from_numpy(self.slots_host).to(DEV).long()
        pools = []
        for rows in (rope64(k, self.cos, self.sin, cfg["rope"], self.pos), self.v.double()):
            pool = torch.zeros((self.per, nk, 16, d), dtype=torch.float64, device=DEV)
            pool[slots // 16, :, slots % 16] = rows
            pools.append(pool)
        return {"x": x, "h0": rms64(x, self.w[0], eps), "x1": x1, "h1": rms64(x1, self.w[1], eps),
                "act": act64(cfg["act"], self.gate.double()) * self.up.double(), "x2": x2,
                "h2": rms64(x2, self.w[2], eps), "k": pools[0], "v": pools[1]}

    @staticmethod
    def work(c, cfg):
        H, F, d, nq, nk, n, s = (*(cfg[k] for k in ("hidden", "ff", "head_dim", "nq", "nk")), c["rows"],
                                 SIZE[c["dtype"]])
        ff_rows = n * (cfg["moe"][1] if "moe" in cfg else 1)
        per = (W.row_bytes(cfg["qtype"], H) + 2 * s * H) + 2 * 4 * s * H + 2 * s * (nq + 2 * nk) * d + 4 * d
        return {"bytes": n * per + 3 * s * ff_rows * F, "flops": n * 20.0 * H + ff_rows * 10.0 * F}

    @staticmethod
    def tolerance(c):
        return {"rel": 1e-3, "max": 0.01} if c["dtype"] == "f16" else {"rel": 1e-6, "max": 1e-4}


class Head(Base):
    """The end of a step: the LM head over the whole vocabulary with the CPU
    engine's bits, then the 40 candidates of every row for the sampler."""

    K = 40

    def inputs(self):
        c, cfg = self.case, self.cfg
        self.raws = self.raw(cfg["vocab"], cfg["hidden"], c["qtype"])
        self.x = self.normal(c["rows"], cfg["hidden"])

    def setup(self):
        n, V = self.case["rows"], self.cfg["vocab"]
        self.w = self.packed(self.raws, V, self.cfg["hidden"], self.case["qtype"])
        self.raws = None
        self.logits = torch.zeros((n, V), device=DEV)
        self.best = torch.zeros((n, self.K), device=DEV)
        self.ids = torch.zeros((n, self.K), device=DEV, dtype=torch.int32)
        self.count = torch.zeros((n,), device=DEV, dtype=torch.int32)
        return super().setup()

    def run(self):
        n, V, H, T = self.case["rows"], self.cfg["vocab"], self.cfg["hidden"], W.GGML_ID[self.case["qtype"]]
        x = context()
        x.lm_head(self.w.data_ptr(), T, V, H, self.x.data_ptr(), H, n, V, 1.0, 1.0, 0.0, self.logits.data_ptr(), V,
                  hip.F32)
        x.top_k(self.logits.data_ptr(), V, n, V, hip.F32, self.K, 0.8, self.best.data_ptr(), self.ids.data_ptr(),
                self.count.data_ptr())
        return {"logits": self.logits, "best": self.best, "ids": self.ids, "count": self.count}

    def exact(self):
        V, H = self.cfg["vocab"], self.cfg["hidden"]
        x, rows = q8_rows(self.x), self.raws.view(V, -1)
        logits = torch.cat([x @ dequantised(rows[a:a + 16384], self.case["qtype"], min(16384, V - a), H).T
                            for a in range(0, V, 16384)], -1)
        return {"logits": logits, "best": None, "ids": None, "count": None}

    @staticmethod
    def work(c, cfg):
        V, H, n = cfg["vocab"], cfg["hidden"], c["rows"]
        return {"bytes": qbytes(c["qtype"], V, H) + n * 4 * (H + V), "flops": 2.0 * n * V * H}

    # the header promises the CPU engine's bits and a full sort's candidates
    @staticmethod
    def tolerance(c):
        return "exact"


KINDS = {"decode_step": DecodeStep, "mlp_qmm": MlpQmm, "projections": Projections, "attend_rows": AttendRows,
         "paged_decode": PagedDecode, "experts": Experts, "layer_ops": LayerOps, "head": Head}


def listed():
    return [
        # a token of one 8B conversation of 4001 positions (four of its layers and the head)
        {"name": "decode_step_b1", "kind": "decode_step", "config": "B", "rows": 1, "keys": 4001, "layers": 4,
         "qtype": "q4_0"},
        # the element ops of a small decode batch: launches and latency
        {"name": "layer_ops_d8", "kind": "layer_ops", "config": "D", "rows": 8, "dtype": "f32"},
        # the element ops of a long prompt: HBM
        {"name": "layer_ops_c16384", "kind": "layer_ops", "config": "C", "rows": 16384, "dtype": "f16"},
        # verification rows, or a few concurrent conversations, through the FFN
        {"name": "mlp_rows4", "kind": "mlp_qmm", "config": "B", "rows": 4, "qtype": "q4_0"},
        # a serving batch's decode projections
        {"name": "projections_b32", "kind": "projections", "config": "B", "rows": 32, "dtype": "f32",
         "qtype": "q4_0", "resident": False},
        # a ragged prompt chunk on the quantised weights
        {"name": "projections_d777", "kind": "projections", "config": "D", "rows": 777, "dtype": "f16",
         "qtype": "q8_0", "resident": False},
        # a long prompt on the resident f16 weights
        {"name": "projections_c4096", "kind": "projections", "config": "C", "rows": 4096, "dtype": "f16",
         "qtype": "q4_0", "resident": True},
        # a long prompt's attention
        {"name": "attend_c4096", "kind": "attend_rows", "config": "C", "rows": 4096, "past": 0, "window": 0,
         "dtype": "f16"},
        # a serving batch's attention over ragged histories
        {"name": "paged_b32", "kind": "paged_decode", "config": "B", "rows": 32, "keys": 8000, "dtype": "f16"},
        # routed experts of a decode batch
        {"name": "experts_t32", "kind": "experts", "config": "E", "tokens": 32, "dtype": "f32", "qtype": "q4_0",
         "cores": False},
        # routed experts of a long prompt
        {"name": "experts_t8192", "kind": "experts", "config": "E", "tokens": 8192, "dtype": "f16", "qtype": "q4_0",
         "cores": True},
        # the head and the sampler's candidates of three conversations
        {"name": "head_b3", "kind": "head", "config": "B", "rows": 3, "qtype": "q8_0"},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(sorted(KINDS))
    qtype = rng.choice(["q4_0", "q8_0"])
    dtype = rng.choice(["f16", "f32"])
    case = {"kind": kind, "config": rng.choice("ABCD")}
    if kind == "decode_step":
        case.update(config=rng.choice("AB"), rows=rng.choice([1, 1, 2, 4]), keys=size(64, 8192),
                    layers=rng.randint(2, 4), qtype=qtype)
    elif kind == "mlp_qmm":
        case.update(config=rng.choice("ABD"), rows=size(1, 16), qtype=qtype)
    elif kind == "projections":
        resident = rng.random() < 0.4
        case.update(config=rng.choice("ACD"), rows=size(256 if resident else 17, 4096 if resident else 2048),
                    dtype=dtype, qtype=qtype, resident=resident)
    elif kind == "attend_rows":
        case.update(config=rng.choice("ACDE"), rows=size(2, 2048), past=rng.choice([0, size(16, 4096)]),
                    window=rng.choice([0, 0, 1024]), dtype=dtype)
    elif kind == "paged_decode":
        case.update(config=rng.choice("ABDE"), rows=size(1, 64), keys=size(64, 8192), dtype=dtype)
    elif kind == "experts":
        cores = rng.random() < 0.5
        case.update(config="E", tokens=size(256, 8192) if cores else size(1, 64), dtype=dtype, qtype=qtype,
                    cores=cores)
    elif kind == "layer_ops":
        half = rng.random() < 0.5
        case.update(config=rng.choice("ACDE"), rows=size(256, 8192) if half else size(1, 256),
                    dtype="f16" if half else "f32")
    else:
        case.update(config=rng.choice("ABD"), rows=size(1, 8), qtype=qtype)
    return case


def prepare(case, seed):
    return KINDS[case["kind"]](case, seed).setup()


def run(state):
    return state.run()


def exact(case, seed):
    return KINDS[case["kind"]](case, seed).exact()


def work(case):
    return KINDS[case["kind"]].work(case, W.CONFIGS[case["config"]])


def tolerance(case):
    return KINDS[case["kind"]].tolerance(case)
