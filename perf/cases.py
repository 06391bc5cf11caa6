"""Performance cases of the quantised linear path: the calls that a program
serving or running a quantised model makes through ``torch.ops.zentorch``.

Every case is one of four kinds:

* ``linear``  one op call on one weight: int4 weight-only (``woq``), dynamic
  int8 (``dyn``, ``dyn_asym``);
* ``layer``   the linears of a decoder layer: QKV, O with the residual, the
  gated MLP (gate, up, silu * mul) and down with the residual, for int4
  (``woq``) or dynamic int8 (``dyn``) weights.  With ``graph`` the calls of
  ``layers`` layers are captured once in a HIP graph and a pass replays it, as
  a decode loop does; otherwise they are issued one by one, as a prefill;
* ``moe``     one int4 mixture-of-experts layer, routing ids given;
* ``static``  a two-layer static int8 MLP (u8 activations with a zero point,
  relu, requantised in between), as a post-training-quantised model runs it.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "zendnn-pytorch-plugin_amd"))
import zentorch  # noqa: E402,F401

DEV = "cuda"
ops = torch.ops.zentorch


def listed():
    return [
        # One projection of a 4-sequence decode step outside a graph: the
        # smallest call, where launch and latency count.
        dict(name="woq_call_m4", kind="linear", op="woq", m=4, n=4096, k=4096, group=128,
             zp=False, bias=False, dtype="bf16"),
        # Single-sequence decode of a Llama-3-8B shaped model, int4 weights.
        dict(name="woq_decode_m1", kind="layer", op="woq", m=1, hidden=4096, qkv=6144, inter=14336,
             group=128, zp=False, graph=True, layers=4),
        # Batched decode with asymmetric int4 weights (zero points) and a QKV
        # bias, Qwen2-7B shapes.
        dict(name="woq_decode_zp_m24", kind="layer", op="woq", m=24, hidden=3584, qkv=4608,
             inter=18944, group=128, zp=True, graph=True, layers=4),
        # A short prompt or a mixed prefill/decode batch on one projection.
        dict(name="woq_mid_m200", kind="linear", op="woq", m=200, n=5120, k=5120, group=128,
             zp=False, bias=True, dtype="bf16"),
        # Prompt chunk of 2048 tokens, Llama-3-8B shapes, int4 weights.
        dict(name="woq_prefill_m2048", kind="layer", op="woq", m=2048, hidden=4096, qkv=6144,
             inter=14336, group=128, zp=False, graph=False, layers=1),
        # Ragged prompt, asymmetric int4 weights in groups of 64, Llama-3.2-3B
        # shapes.
        dict(name="woq_prefill_zp_m777", kind="layer", op="woq", m=777, hidden=3072, qkv=5120,
             inter=8192, group=64, zp=True, graph=False, layers=1),
        # Batched decode with dynamic int8, Llama-3-8B shapes.
        dict(name="dyn_decode_m8", kind="layer", op="dyn", m=8, hidden=4096, qkv=6144, inter=14336,
             graph=True, layers=4),
        # One wide projection at 128 tokens, dynamic int8.
        dict(name="dyn_call_m128", kind="linear", op="dyn", m=128, n=11008, k=4096, bias=True,
             dtype="bf16"),
        # An encoder's feed-forward projection in float32 with a ragged batch.
        dict(name="dyn_fp32_m1000", kind="linear", op="dyn", m=1000, n=4096, k=1024, bias=True,
             dtype="fp32"),
        # The largest: a 4096-token prompt chunk with dynamic int8.
        dict(name="dyn_prefill_m4096", kind="layer", op="dyn", m=4096, hidden=4096, qkv=6144,
             inter=14336, graph=False, layers=1),
        # A Mixtral-shaped int4 MoE layer over a 256-token batch.
        dict(name="moe_m256", kind="moe", m=256, hidden=4096, inter=14336, experts=8, topk=2),
        # Static int8 MLP over a large ragged batch.
        dict(name="static_mlp_m3000", kind="static", m=3000, k=1024, n=4096, n2=1024),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["woq", "woq", "woq_layer", "woq_layer", "dyn", "dyn_layer", "moe", "static"])
    if kind in ("woq", "dyn"):
        k = 128 * _logint(rng, 8, 112)
        n = _logint(rng, 1024, 16384)
        n -= n % rng.choice([1, 8, 16, 64])
        m = _logint(rng, 1, min(4096, 2 * 10 ** 11 // (n * k)))
        c = dict(kind="linear", op=kind, m=m, n=n, k=k, bias=rng.random() < 0.5, dtype="bf16")
        if kind == "woq":
            c.update(group=rng.choice([64, 128, 128, k]), zp=rng.random() < 0.4)
        else:
            if rng.random() < 0.3:
                c["k"] = k - 16 * rng.randrange(1, 8)  # not whole 128-byte steps
            r = rng.random()
            c["op"] = "dyn_asym" if r < 0.25 else "dyn"
            c["dtype"] = "fp32" if r > 0.75 else "bf16"
        return c
    if kind in ("woq_layer", "dyn_layer"):
        graph = rng.random() < 0.5
        hidden = 256 * rng.randrange(8, 21)
        inter = 128 * int(hidden * rng.uniform(2.5, 4) / 128)
        most = min(2048, 4 * 10 ** 11 // (3 * hidden * (hidden + inter)))
        c = dict(kind="layer", op=kind[:3],
                 m=_logint(rng, 1, 64) if graph else _logint(rng, 65, most), hidden=hidden,
                 qkv=hidden + 256 * rng.randrange(1, 9), inter=inter, graph=graph,
                 layers=2 if graph else 1)
        if kind == "woq_layer":
            c.update(group=rng.choice([64, 128, 128]), zp=rng.random() < 0.4)
        return c
    if kind == "moe":
        return dict(kind="moe", m=_logint(rng, 1, 512), hidden=128 * rng.randrange(16, 33),
                    inter=128 * rng.randrange(8, 57), experts=rng.choice([8, 16]), topk=2)
    return dict(kind="static", m=_logint(rng, 64, 4096), k=64 * rng.randrange(8, 33),
                n=64 * rng.randrange(16, 65), n2=64 * rng.randrange(8, 33))


# ------------------------------------------------------------------ inputs
class _Gen:
    """Seeded tensors made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def randn(self, *shape, dtype=torch.bfloat16, scale=1.0):
        return (torch.randn(*shape, generator=self.g, device=DEV) * scale).to(dtype)

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV)

    def ints(self, lo, hi, *shape, dtype=torch.int8):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=dtype)

    def woq(self, n, k, group, zp, bias=False):
        """Packed int4 weight [N, K/8] of uniform nibbles, bf16 scales that
        leave x . W^T at unit variance, int8 zero points around 8."""
        s = (self.rand(k // group, n) * 0.5 + 0.75) / (4.6 * math.sqrt(k))
        return dict(w=self.ints(-2 ** 31, 2 ** 31, n, k // 8, dtype=torch.int32), s=s.bfloat16(),
                    z=self.ints(6, 11, k // group, n) if zp else None,
                    b=self.randn(n, scale=0.1) if bias else None)

    def int8(self, n, k, bias=False):
        return dict(w=self.ints(-127, 128, n, k),
                    s=(self.rand(n) * 0.5 + 0.75) / (73.0 * math.sqrt(k)),
                    b=self.randn(n, dtype=torch.float32, scale=0.1) if bias else None)


_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _inputs(c, seed):
    g = _Gen(seed)
    if c["kind"] == "linear":
        st = dict(x=g.randn(c["m"], c["k"], dtype=_DT[c["dtype"]]))
        st["p"] = (g.woq(c["n"], c["k"], c["group"], c["zp"], c["bias"]) if c["op"] == "woq"
                   else g.int8(c["n"], c["k"], c["bias"]))
        return st
    if c["kind"] == "layer":
        h, i = c["hidden"], c["inter"]

        def lin(n, k, bias=False):
            if c["op"] == "woq":
                return g.woq(n, k, c["group"], c["zp"], bias)
            return g.int8(n, k, bias)

        layers = []
        for _ in range(c["layers"]):
            d = dict(x=g.randn(c["m"], h), ctx=g.randn(c["m"], h),
                     qkv=lin(c["qkv"], h, c["op"] == "woq" and c["zp"]), o=lin(h, h),
                     down=lin(h, i))
            if c["op"] == "woq":
                d["gate_up"] = lin(2 * i, h)
            else:
                d["gate"], d["up"] = lin(i, h), lin(i, h)
            layers.append(d)
        return dict(layers=layers)
    if c["kind"] == "moe":
        e, h, i = c["experts"], c["hidden"], c["inter"]
        p13 = [g.woq(2 * i, h, 128, False) for _ in range(e)]
        p2 = [g.woq(h, i, 128, False) for _ in range(e)]
        top, ids = torch.topk(g.randn(c["m"], e, dtype=torch.float32), c["topk"])
        return dict(x=g.randn(c["m"], h), ids=ids.int(), wts=torch.softmax(top, dim=-1),
                    w13=torch.stack([p["w"] for p in p13]), s13=torch.stack([p["s"] for p in p13]),
                    w2=torch.stack([p["w"] for p in p2]), s2=torch.stack([p["s"] for p in p2]))
    one = lambda v, dt=torch.float32: torch.tensor([v], dtype=dt, device=DEV)  # noqa: E731
    return dict(x=g.randn(c["m"], c["k"]), xs=one(8 / 255), xz=one(128, torch.int32),
                p1=g.int8(c["n"], c["k"], True), hs=one(4 / 255), hz=one(0, torch.int32),
                p2=g.int8(c["n2"], c["n"], True))


# --------------------------------------------------------------- the passes
def _woq_layer(d):
    qkv = ops.zentorch_woq_linear(d["x"], d["qkv"]["w"].t(), d["qkv"]["s"], d["qkv"]["z"],
                                  d["qkv"]["b"])
    x1 = ops.zentorch_woq_linear_add(d["ctx"], d["o"]["w"].t(), d["o"]["s"], d["o"]["z"], d["x"])
    p = d["gate_up"]
    h = ops.zentorch_woq_linear_gate_up_silu_mul(x1, p["w"].t(), p["s"], p["z"])
    p = d["down"]
    return qkv, x1, h, ops.zentorch_woq_linear_add(h, p["w"].t(), p["s"], p["z"], x1)


def _dyn_layer(d):
    qkv = ops.zentorch_dynamic_qlinear(d["x"], d["qkv"]["w"], d["qkv"]["s"])
    x1 = ops.zentorch_dynamic_qlinear_add(d["ctx"], d["o"]["w"], d["o"]["s"], d["x"])
    up = ops.zentorch_dynamic_qlinear(x1, d["up"]["w"], d["up"]["s"])
    h = ops.zentorch_dynamic_qlinear_silu_mul(x1, d["gate"]["w"], d["gate"]["s"], up)
    return qkv, x1, h, ops.zentorch_dynamic_qlinear_add(h, d["down"]["w"], d["down"]["s"], x1)


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    if case["kind"] == "linear" and case["op"] == "dyn_asym":
        st["colsum"] = ops.zentorch_s8_weight_colsum(st["p"]["w"])
    if case["kind"] == "layer":
        st["step"] = _woq_layer if case["op"] == "woq" else _dyn_layer
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for d in st["layers"]:
                    st["step"](d)
            torch.cuda.current_stream().wait_stream(side)
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                st["out"] = [st["step"](d) for d in st["layers"]]
    if case["kind"] == "moe":
        st["out"] = torch.empty_like(st["x"])
    return st


def run(state):
    c = state["case"]
    if c["kind"] == "layer":
        if c["graph"]:
            state["graph"].replay()
            return state["out"]
        return [state["step"](d) for d in state["layers"]]
    if c["kind"] == "moe":
        ops.zentorch_fused_moe(state["out"], state["x"], state["w13"], state["w2"], None, None,
                               state["wts"], state["ids"], False, "silu", state["s13"], state["s2"])
        return state["out"]
    if c["kind"] == "static":
        p, q = state["p1"], state["p2"]
        h = ops.zentorch_qlinear_relu(state["x"], p["w"], state["xs"], state["xz"], p["s"], None,
                                      p["b"], state["hs"], state["hz"], torch.uint8)
        return h, ops.zentorch_qlinear(h, q["w"], state["hs"], state["hz"], q["s"], None, q["b"],
                                       None, None, torch.bfloat16)
    p = state["p"]
    if c["op"] == "woq":
        return ops.zentorch_woq_linear(state["x"], p["w"].t(), p["s"], p["z"], p["b"])
    if c["op"] == "dyn_asym":
        return ops.zentorch_dynamic_qlinear_asym(state["x"], p["w"], p["s"], state["colsum"],
                                                 p["b"])
    return ops.zentorch_dynamic_qlinear(state["x"], p["w"], p["s"], p["b"])


# ------------------------------------------------------------------- work
def _lin_work(c, m, n, k, xb, yb, extra=0):
    """Bytes and operations of one linear: x, weight and its scales read once,
    y written once, `extra` elements of y's size read beside them."""
    if c["op"] == "woq":
        w = n * k // 2 + (k // c["group"]) * n * (3 if c["zp"] else 2)
    else:
        w = n * k + 4 * n
    return w + m * k * xb + m * n * yb + extra * yb, 2 * m * n * k


def work(case):
    c, m = case, case["m"]
    if c["kind"] == "linear":
        e = 4 if c["dtype"] == "fp32" else 2
        parts = [_lin_work(c, m, c["n"], c["k"], e, e)]
    elif c["kind"] == "layer":
        h, i = c["hidden"], c["inter"]
        parts = [_lin_work(c, m, c["qkv"], h, 2, 2), _lin_work(c, m, h, h, 2, 2, m * h),
                 _lin_work(c, m, h, i, 2, 2, m * h)]
        b, f = _lin_work(c, m, 2 * i, h, 2, 2)
        parts.append((b - m * i * 2, f))  # silu(gate) * up: one [m, inter] output
        parts = parts * c["layers"]
    elif c["kind"] == "moe":
        h, i, e = c["hidden"], c["inter"], min(c["experts"], m * c["topk"])
        wb = e * 3 * h * i // 2 + e * (2 * (h // 128) * 2 * i + 2 * (i // 128) * h)
        parts = [(wb + 2 * m * h * 2, 2 * m * c["topk"] * 3 * h * i)]
    else:
        parts = [(m * c["k"] * 2 + c["n"] * c["k"] + m * c["n"], 2 * m * c["n"] * c["k"]),
                 (m * c["n"] + c["n2"] * c["n"] + m * c["n2"] * 2, 2 * m * c["n2"] * c["n"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    if case["kind"] == "static":
        # u8 outputs may differ by a step where the rounded value is a tie;
        # the second product sums 8-bit integers exactly
        return {"rel": 4e-3, "max": 0.1, "differ": 2e-3}
    if case["kind"] == "linear" and case["dtype"] == "fp32":
        # int32 sums are exact: what remains is the fp32 scaling
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "linear":
        return {"rel": 4e-3, "max": 0.05}  # one bf16 rounding of an fp32 sum
    # chains of such products, each rounded to bf16 (and, for int8, quantised
    # again from it)
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------- plain 64-bit results
def _f64_woq(c, p):
    w = p["w"]
    n, kw = w.shape
    u = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], dim=2).reshape(n, kw * 8)
    if p["z"] is None:
        q = torch.where(u > 7, u - 16, u).float()
    else:
        q = u.float() - p["z"].t().float().repeat_interleave(c["group"], dim=1)
    # the ops multiply by the dequantised weight in bf16
    return (q * p["s"].t().float().repeat_interleave(c["group"], dim=1)).bfloat16().double()


def _f64_lin(c, x, p):
    if c["op"] == "woq":
        y = x.double() @ _f64_woq(c, p).t()
    else:
        xf = x.float()
        if c["op"] == "dyn_asym":
            lo, hi = xf.amin(1, True).clamp(max=0), xf.amax(1, True).clamp(min=0)
            s = (hi - lo).clamp(min=1e-12) / 255
            z = torch.round(-lo / s).clamp(0, 255)
            q = (torch.round(xf / s) + z).clamp(0, 255) - z
        else:
            s = xf.abs().amax(1, True).clamp(min=1e-12) / 127
            q = torch.round(xf / s).clamp(-128, 127)
        y = (q.double() @ p["w"].double().t()) * s.double() * p["s"].double()
    return y if p["b"] is None else y + p["b"].double()


def _exact_layer(c, d):
    silu = torch.nn.functional.silu
    qkv = _f64_lin(c, d["x"], d["qkv"])
    x1 = _f64_lin(c, d["ctx"], d["o"]) + d["x"].double()
    x1b = x1.bfloat16()  # each op hands the next one bf16
    if c["op"] == "woq":
        gate, up = _f64_lin(c, x1b, d["gate_up"]).chunk(2, dim=1)
    else:
        gate, up = _f64_lin(c, x1b, d["gate"]), _f64_lin(c, x1b, d["up"])
    h = silu(gate) * up.bfloat16().double()
    return qkv, x1, h, _f64_lin(c, h.bfloat16(), d["down"]) + x1b.double()


def exact(case, seed):
    c, st = case, _inputs(case, seed)
    if c["kind"] == "linear":
        return _f64_lin(c, st["x"], st["p"])
    if c["kind"] == "layer":
        return [_exact_layer(c, d) for d in st["layers"]]
    if c["kind"] == "moe":
        woq = dict(op="woq", group=128, zp=False)
        out = torch.zeros(st["x"].shape, dtype=torch.float64, device=DEV)
        for e in range(c["experts"]):
            t, slot = torch.nonzero(st["ids"] == e, as_tuple=True)
            if not len(t):
                continue
            one = lambda w, s: dict(w=st[w][e], s=st[s][e], z=None, b=None)  # noqa: E731
            gate, up = _f64_lin(woq, st["x"][t], one("w13", "s13")).chunk(2, dim=1)
            h = (torch.nn.functional.silu(gate) * up).bfloat16()
            y = _f64_lin(woq, h, one("w2", "s2")).bfloat16().double()
            out.index_add_(0, t, y * st["wts"][t, slot].double()[:, None])
        return out
    xq = torch.clamp(torch.round(st["x"].float() * (1 / st["xs"])) + 128, 0, 255) - 128
    a = (xq.double() @ st["p1"]["w"].double().t()) * st["xs"].double() * st["p1"]["s"].double()
    a = torch.relu(a + st["p1"]["b"].double())
    hq = torch.clamp(torch.round(a.float() * (1 / st["hs"])), 0, 255)
    y = (hq.double() @ st["p2"]["w"].double().t()) * st["hs"].double() * st["p2"]["s"].double()
    return None, y + st["p2"]["b"].double()
