"""Performance cases of the W4A8 decoder-linear path: what a serving host has it do, through the public binding.

Three kinds of work:
  linear  one quantised linear on bf16 rows: the fused launch where the law has one, else quantiser + GEMM
  layers  the linears of successive decoder layers with the activation producers between them, as a decode step (captured
          once as a HIP graph and replayed, the way a serving loop runs it) or as a prefill / verify chunk (plain calls)
  moe     the routed expert layer, from router logits to the weighted combine

`layers` comes in the two bases the library serves. "plain": per-token int8 codes of the rows as they are; the layer is
the 27B-class one of the benchmark (synth.LAYER_LINEARS) and its three inputs come from other parts of an engine (norms,
attention). "hadamard": the codes of the 32-point Hadamard basis, made by the producers that hold the norm, the output
gate or SiLU * up; the projections are the served 27B graph's (gated attention layers and gated delta-net layers).

Weights are random bytes: every byte is two int4 codes (or one int8 code), so a random byte string in the device order is
uniform random codes, and no host repack stands in front of a case. Several layers a pass keep decode steps on weights
that come from memory, as in a model of 64 layers.
"""
import functools
import math

import torch

from saber_engine_amd import iu8, synth
from saber_engine_amd.moe import MoeLayerIU8

INTER, HIDDEN = 17408, 5120            # the 27B-class MLP
GDN_HEADS, HEAD_DIM = 48, 256          # delta-net heads of 128; attention heads of 256
CORE = GDN_HEADS * 128                 # width of the attention / delta-net core output: 6144
QKVZ, BA, QKV_GATED = 16384, 96, 14336  # in_proj_qkvz, in_proj_ba, [q | gate] heads + k + v
Z_OFFSET = QKVZ - CORE                 # z is the last part of a qkvz row
EPS = 1e-6
EXPERTS, TOPK, MOE_HIDDEN, MOE_INTER = 128, 8, 4096, 1536


def listed():
    return [
        # one projection of one token, called by itself: the smallest call there is, its launch counts
        dict(name="linear_1row", kind="linear", m=1, n=5120, k=5120, w8=False),
        # a decode step of one sequence, the figure the path is quoted on (M = 1 GEMVs, weights from memory)
        dict(name="decode_1", kind="layers", basis="plain", m=1, layers=4, w8=False, graph=True),
        # a small batch, output-side projections kept at int8 weights (mixed-precision layers)
        dict(name="decode_5_mixed", kind="layers", basis="plain", m=5, layers=4, w8=True, graph=True),
        # a full decode batch of the served hybrid graph
        dict(name="decode_16_hadamard", kind="layers", basis="hadamard", m=16, layers=4, w8=False, graph=True),
        # a speculative verify step: a few drafted tokens for several sequences, ragged
        dict(name="verify_45_hadamard", kind="layers", basis="hadamard", m=45, layers=4, w8=False, graph=True),
        # a short prompt, or a chunk beside decoding
        dict(name="prefill_200", kind="layers", basis="plain", m=200, layers=2, w8=False, graph=False),
        dict(name="prefill_777_hadamard_mixed", kind="layers", basis="hadamard", m=777, layers=2, w8=True, graph=False),
        # the usual prefill chunk
        dict(name="prefill_2048", kind="layers", basis="plain", m=2048, layers=1, w8=False, graph=False),
        # a long prompt in one piece
        dict(name="prefill_8192", kind="layers", basis="plain", m=8192, layers=1, w8=False, graph=False),
        # the routed layer: a decode batch, a ragged mid-size batch with a shared expert, a prefill chunk
        dict(name="moe_16", kind="moe", m=16, shared=False),
        dict(name="moe_300_shared", kind="moe", m=300, shared=True),
        dict(name="moe_4096", kind="moe", m=4096, shared=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "layers", "layers", "moe"))
    if kind == "linear":
        return dict(kind="linear", m=_log_int(rng, 1, 4096), n=16 * _log_int(rng, 6, 1792), k=128 * _log_int(rng, 8, 136),
                    w8=rng.random() < 0.3)
    if kind == "layers":
        basis = rng.choice(("plain", "hadamard"))
        m = _log_int(rng, 1, 8192 if basis == "plain" else 6144)
        return dict(kind="layers", basis=basis, m=m, layers=4 if m <= 64 else 2 if m <= 1024 else 1, w8=rng.random() < 0.3, graph=m <= 64)
    return dict(kind="moe", m=_log_int(rng, 1, 4096), shared=rng.random() < 0.4)


@functools.lru_cache(maxsize=None)
def _ctx():
    return iu8.Context()


class _Rng:
    """Seeded operands made on the device, in the distributions of saber_engine_amd.synth."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def bytes(self, n):
        return torch.randint(0, 256, (n,), generator=self.g, dtype=torch.uint8, device="cuda")

    def scales(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(0.02).abs_().add_(1e-4)

    def rows(self, m, k):
        """bf16 rows N(0, 1), one channel in two hundred x20."""
        a = torch.randn(m, k, generator=self.g, device="cuda")
        cols = torch.randperm(k, generator=self.g, device="cuda")[: k // 200]
        a[:, cols] *= 20.0
        return a.to(torch.bfloat16)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda").to(torch.bfloat16)

    def signs(self, k):
        return torch.randint(0, 2, (k,), generator=self.g, device="cuda").mul_(2).sub_(1).float()


def _bf16(m, n):
    return torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")


class _Codes:
    """An A edge for m rows of k codes and the rows' scales."""

    def __init__(self, m, k):
        self.q = torch.zeros(iu8.a_bytes(m, k), dtype=torch.uint8, device="cuda")
        self.s = torch.zeros(m, dtype=torch.float32, device="cuda")


class _Linear:
    def __init__(self, r, m, n, k, w8):
        self.m, self.n, self.k, self.kind = m, n, k, iu8.W8 if w8 else iu8.W4
        self.w, self.ws = r.bytes(n * k // (1 if w8 else 2)), r.scales(n)
        if w8:
            self.w[self.w == 128] = 127    # codes are -127..127
        self.c = _bf16(m, n)
        pb, cb = iu8.gemm_workspace(self.kind, m, n, k)
        self.partial = torch.empty(pb, dtype=torch.uint8, device="cuda") if pb else None
        self.counter = torch.zeros(cb, dtype=torch.uint8, device="cuda") if cb else None
        self.fused = iu8.fused_holds(m, k)

    def gemm(self, a, stream):
        p, c = self.partial, self.counter
        _ctx().gemm(self.kind, a.q.data_ptr(), a.s.data_ptr(), self.w.data_ptr(), self.ws.data_ptr(), self.c.data_ptr(), self.m, self.n, self.k,
                    p.data_ptr() if p is not None else None, c.data_ptr() if c is not None else None, stream)
        return self.c

    def plain(self, x, a, stream):
        if self.fused:
            _ctx().linear_fused(self.kind, x.data_ptr(), self.w.data_ptr(), self.ws.data_ptr(), self.c.data_ptr(), self.m, self.n, self.k,
                                stream=stream)
            return self.c
        _ctx().quant(x.data_ptr(), a.q.data_ptr(), a.s.data_ptr(), self.m, self.k, stream)
        return self.gemm(a, stream)


class _PlainLayer:
    def __init__(self, r, m, w8):
        self.m = m
        self.lin = {name: _Linear(r, m, n, k, w8 and name in ("o", "down")) for name, n, k in synth.LAYER_LINEARS}
        self.x = [r.rows(m, HIDDEN) for _ in range(3)]    # normed input, attention output, normed residual stream
        self.a, self.a_mlp = _Codes(m, HIDDEN), _Codes(m, INTER)
        self.chain = not w8 and iu8.mlp_chain_pays(m, HIDDEN, INTER)
        self.act = not self.chain and m >= 5 and iu8.gate_up_act_holds(m, HIDDEN, INTER)
        self.p = _bf16(m, INTER) if self.chain or self.act else None
        self.state = torch.zeros(iu8.MLP_CHAIN_STATE_BYTES, dtype=torch.uint8, device="cuda") if self.chain else None
        self.silu = iu8.resolve_silu_mul_quant(m, INTER)

    def run(self, stream):
        ctx, m, gu, dn, a2 = _ctx(), self.m, self.lin["gate_up"], self.lin["down"], self.a_mlp
        out = [self.lin["qkv"].plain(self.x[0], self.a, stream), self.lin["o"].plain(self.x[1], self.a, stream)]
        x = self.x[2]
        if self.chain:
            ctx.mlp_chain(x.data_ptr(), gu.w.data_ptr(), gu.ws.data_ptr(), dn.w.data_ptr(), dn.ws.data_ptr(), None, self.p.data_ptr(),
                          self.state.data_ptr(), dn.c.data_ptr(), m, HIDDEN, INTER, stream=stream)
        elif self.act:
            ctx.quant(x.data_ptr(), self.a.q.data_ptr(), self.a.s.data_ptr(), m, HIDDEN, stream)
            ctx.gate_up_act(self.a.q.data_ptr(), self.a.s.data_ptr(), gu.w.data_ptr(), gu.ws.data_ptr(), None, self.p.data_ptr(), m, HIDDEN,
                            INTER, stream)
            dn.plain(self.p, a2, stream)
        else:
            c = gu.plain(x, self.a, stream)
            ctx.launch(self.silu, dict(gu=c.data_ptr(), q=a2.q.data_ptr(), scale=a2.s.data_ptr()), stream)
            dn.gemm(a2, stream)
        return out + [dn.c]


class _HadamardLayer:
    def __init__(self, r, m, w8, attention, tables):
        self.m, self.attention, self.tables = m, attention, tables
        # what enters the layer is drawn, not the layer before it: a code that rounds the other way would grow from layer to layer
        self.y, self.res = r.rows(m, HIDDEN), r.rows(m, HIDDEN)
        self.proj = _Linear(r, m, QKV_GATED if attention else QKVZ, HIDDEN, False)
        self.ba = None if attention else _Linear(r, m, BA, HIDDEN, False)
        self.o = _Linear(r, m, HIDDEN, CORE, w8)
        self.gate_up, self.down = _Linear(r, m, 2 * INTER, HIDDEN, False), _Linear(r, m, HIDDEN, INTER, w8)
        self.core = r.rows(m, CORE)
        self.norm1, self.norm2, self.norm_gdn = (r.normal(k).mul_(0.1) for k in (HIDDEN, HIDDEN, 128))
        self.t1, self.t_core, self.t2, self.t3 = (r.signs(k) for k in (HIDDEN, CORE, HIDDEN, INTER))
        self.res1, self.res2 = _bf16(m, HIDDEN), _bf16(m, HIDDEN)
        self.a, self.a_core, self.a_mlp = _Codes(m, HIDDEN), _Codes(m, CORE), _Codes(m, INTER)
        self.pair = self.ba is not None and m <= 32

    def run(self, stream):
        ctx, m, a, ac, am = _ctx(), self.m, self.a, self.a_core, self.a_mlp
        ctx.add_rms_quant_had(self.y.data_ptr(), self.res.data_ptr(), self.norm1.data_ptr(), a.q.data_ptr(), a.s.data_ptr(),
                              self.res1.data_ptr(), m, HIDDEN, EPS, self.t1.data_ptr(), stream)
        p = self.proj
        if self.attention:
            p.gemm(a, stream)
            ctx.attn_gate_quant_had_lut(self.core.data_ptr(), p.c.data_ptr(), ac.q.data_ptr(), ac.s.data_ptr(), m, CORE, HEAD_DIM, QKV_GATED,
                                        self.t_core.data_ptr(), self.tables["sigmoid"].data_ptr(), stream)
        else:
            b = self.ba
            if self.pair:
                ctx.gemm_pair(a.q.data_ptr(), a.s.data_ptr(), p.w.data_ptr(), p.ws.data_ptr(), p.c.data_ptr(), p.n, b.w.data_ptr(), b.ws.data_ptr(),
                              b.c.data_ptr(), b.n, m, HIDDEN, stream)
            else:
                p.gemm(a, stream)
                b.gemm(a, stream)
            ctx.gdn_norm_quant_had(self.core.data_ptr(), p.c.data_ptr() + 2 * Z_OFFSET, QKVZ, self.norm_gdn.data_ptr(), ac.q.data_ptr(),
                                   ac.s.data_ptr(), m, CORE, EPS, self.t_core.data_ptr(), stream)
        self.o.gemm(ac, stream)
        ctx.add_rms_quant_had(self.o.c.data_ptr(), self.res1.data_ptr(), self.norm2.data_ptr(), a.q.data_ptr(), a.s.data_ptr(),
                              self.res2.data_ptr(), m, HIDDEN, EPS, self.t2.data_ptr(), stream)
        self.gate_up.gemm(a, stream)
        ctx.silu_mul_quant_had_lut(self.gate_up.c.data_ptr(), am.q.data_ptr(), am.s.data_ptr(), m, INTER, self.t3.data_ptr(),
                                   self.tables["silu"].data_ptr(), stream)
        self.down.gemm(am, stream)
        return [p.c] + ([] if self.attention else [self.ba.c]) + [self.o.c, self.res2, self.down.c]


def _layers(case, r):
    m, w8 = case["m"], case["w8"]
    if case["basis"] == "plain":
        return [_PlainLayer(r, m, w8) for _ in range(case["layers"])]
    tables = {name: torch.empty(65536, dtype=torch.int16, device="cuda") for name in ("silu", "sigmoid")}
    _ctx().silu_table(tables["silu"].data_ptr())
    _ctx().sigmoid_table(tables["sigmoid"].data_ptr())
    return [_HadamardLayer(r, m, w8, i % 4 == 1, tables) for i in range(case["layers"])]    # one layer in four is attention


def prepare(case, seed):
    r = _Rng(seed)
    st = dict(kind=case["kind"])
    if case["kind"] == "linear":
        m, k = case["m"], case["k"]
        st.update(lin=_Linear(r, m, case["n"], k, case["w8"]), x=r.rows(m, k), a=_Codes(m, k))
    elif case["kind"] == "layers":
        st.update(layers=_layers(case, r), graph=None)
        if case["graph"]:
            torch.cuda.synchronize()
            stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                st["out"] = [layer.run(stream.cuda_stream) for layer in st["layers"]]
            st["graph"] = graph
    else:
        e = EXPERTS + (1 if case["shared"] else 0)
        moe = MoeLayerIU8(_ctx(), case["m"], EXPERTS, TOPK, MOE_HIDDEN, MOE_INTER, shared=case["shared"])
        moe.set_weights(r.bytes(e * MOE_INTER * MOE_HIDDEN).view(e, -1), r.scales(e, 2 * MOE_INTER),
                        r.bytes(e * MOE_HIDDEN * MOE_INTER // 2).view(e, -1), r.scales(e, MOE_HIDDEN))
        if case["shared"]:
            moe.sgate.copy_(r.normal(case["m"]).view(torch.int16))
        st.update(moe=moe, x=r.rows(case["m"], MOE_HIDDEN).view(torch.int16), logits=r.normal(case["m"], EXPERTS).view(torch.int16))
    return st


def run(state):
    stream = torch.cuda.current_stream().cuda_stream
    if state["kind"] == "linear":
        return state["lin"].plain(state["x"], state["a"], stream)
    if state["kind"] == "moe":
        return state["moe"].forward(state["x"], state["logits"], stream).view(torch.bfloat16)
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return [layer.run(stream) for layer in state["layers"]]


def _linear_work(m, n, k, w8):
    """Weights, scales, bf16 rows in and out; multiplications and additions."""
    return n * k // (1 if w8 else 2) + 4 * n + 2 * m * (n + k), 2 * m * n * k


def _touched(m):
    """Experts that m tokens are expected to reach."""
    return EXPERTS * (1.0 - (1.0 - TOPK / EXPERTS) ** m)


def work(case):
    m = case["m"]
    if case["kind"] == "linear":
        b, f = _linear_work(m, case["n"], case["k"], case["w8"])
        return dict(bytes=b, flops=f)
    if case["kind"] == "moe":
        per, rows = 3 * MOE_HIDDEN * MOE_INTER // 2 + 4 * (2 * MOE_INTER + MOE_HIDDEN), m * (TOPK + (1 if case["shared"] else 0))
        experts = _touched(m) + (1 if case["shared"] else 0)
        return dict(bytes=int(experts * per) + 4 * m * MOE_HIDDEN + 2 * m * EXPERTS, flops=2 * rows * 3 * MOE_HIDDEN * MOE_INTER)
    b = f = 0
    for i in range(case["layers"]):
        w8 = case["w8"]
        if case["basis"] == "plain":
            shapes = [(n, k, w8 and name in ("o", "down")) for name, n, k in synth.LAYER_LINEARS]
            inner = 2 * m * (2 * INTER + INTER)            # gate+up's output and down's input stay inside the layer
        else:
            shapes = [(QKV_GATED, HIDDEN, False)] if i % 4 == 1 else [(QKVZ, HIDDEN, False), (BA, HIDDEN, False)]
            shapes += [(HIDDEN, CORE, w8), (2 * INTER, HIDDEN, False), (HIDDEN, INTER, w8)]
            inner = 2 * m * (2 * INTER + INTER)
        for n, k, wide in shapes:
            lb, lf = _linear_work(m, n, k, wide)
            b, f = b + lb, f + lf
        b -= inner
    return dict(bytes=b, flops=f)


def tolerance(case):
    """About four times what the path shows against itself with every product by a weight scale, or the norm's sum, off by
    one unit in the last place of f32: a bf16 value that rounds the other way, and behind a requantisation the int8 codes
    that do. Relative / largest difference seen: linear 2e-5 / 0.0074, plain layers 2.6e-4 / 0.083, routed layer 3.2e-4 /
    0.018, Hadamard layers (three requantisations in a row) 5.7e-3 / 0.26."""
    if case["kind"] == "linear":
        return dict(rel=1e-4, max=0.03)
    if case["kind"] == "moe":
        return dict(rel=1.2e-3, max=0.07)
    return dict(rel=1e-3, max=0.33) if case["basis"] == "plain" else dict(rel=0.02, max=0.99)
