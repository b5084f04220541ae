"""Performance cases of the MoE layer: the work that callers have it do, each
through a public entry point of ``warp_route``.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges:

  op       "fused": one decode token through ``fused_moe``.  "batched": B
           tokens through ``batched_fused_moe`` (a decode batch, or a chunk of
           a prompt).  "gate": ``gate_topk`` alone.  "stack": one decode step
           of a ``MoEStack`` replayed from its captured graph.
  E, h, I, k, renorm   the layer: experts, hidden and intermediate size,
           experts per token, renormalised weights or not
  w, x     dtypes of the packed expert weights and of x and the output
  B        tokens
  layers   layers of the stack

The shapes are the package's own configurations (``synthetic.CONFIGS``), their
tensor-parallel shards and the reference's test shapes; the ragged one is
generic.  Tokens are x ~ N(0, 1) routed by a router whose logits are N(0, 1),
expert weights N(0, 0.02): an uneven, unclustered load over the experts, as
mixed traffic gives.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "warp-route_amd"))

from warp_route import functional as F  # noqa: E402
from warp_route.stack import MoEStack  # noqa: E402
from warp_route.synthetic import CONFIGS, make_layer  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
          "fp8": torch.float8_e4m3fn, "mxfp4": torch.float4_e2m1fn_x2}
WEIGHT_BITS = {"f32": 32, "f16": 16, "bf16": 16, "fp8": 8, "mxfp4": 4.25}
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _case(op, shape, w, x, B=1, shards=1, layers=1, **named):
    """A case of one of the package's configurations, its intermediate size
    split over ``shards`` GPUs."""
    c = CONFIGS[shape]
    return dict(named, op=op, E=c.num_experts, h=c.hidden_dim, I=c.intermediate_dim // shards,
                k=c.top_k, renorm=c.renormalize, w=w, x=x, B=B, layers=layers)


def listed():
    return [
        # The smallest call: the reference's own test shape in its only weight
        # format, where launches and the host's part count.
        _case("fused", "toy", "f32", "f32", name="toy f32 token"),
        # One decode token through a layer of many small experts.
        _case("fused", "deepseek", "f16", "f16", name="deepseek f16 token"),
        # The headline: one decode token through a layer of large experts.
        _case("fused", "mixtral", "f16", "f32", name="mixtral f16 token"),
        # The same layer in fp8 split over 8 GPUs: one GPU's share of a token.
        _case("fused", "mixtral", "fp8", "f16", shards=8, name="mixtral tp8 fp8 token"),
        # Small decode batch: every expert selected, few tokens each.
        _case("batched", "mixtral", "f16", "f16", B=16, name="mixtral f16 B16"),
        # Decode batches of reduced-precision weights.
        _case("batched", "dbrx", "fp8", "f32", B=32, name="dbrx fp8 B32"),
        _case("batched", "mixtral", "mxfp4", "f16", B=64, name="mixtral mxfp4 B64"),
        # A large serving batch over 64 small experts.
        _case("batched", "deepseek", "bf16", "f16", B=256, name="deepseek bf16 B256"),
        # A prompt chunk through large experts: the largest case.
        _case("batched", "mixtral", "bf16", "f32", B=512, name="mixtral bf16 B512"),
        # Sizes that are multiples of nothing: a layer of a user's own.
        dict(name="ragged f16 B40", op="batched", E=12, h=1500, I=2050, k=3, renorm=True, w="f16",
             x="f32", B=40, layers=1),
        # The router alone, for a caller that dispatches its own experts.
        _case("gate", "deepseek", "f32", "f32", B=256, name="deepseek gate B256"),
        # A whole decode step, as a serving loop replays it: 4 layers, 4 tokens.
        _case("stack", "deepseek", "f16", "f32", B=4, layers=4, name="deepseek f16 stack B4"),
    ]


# The cost bounds of a drawn case: those of the largest listed ones.
MAX_FLOPS = 2.0 * 512 * 2 * 3 * 4096 * 14336
MAX_BYTES = 16 * 3 * 6144 * 10752


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        op = rng.choice(["fused"] * 4 + ["batched"] * 9 + ["gate", "stack"])
        w = rng.choice(sorted(DTYPES))
        x = rng.choice(["f32", "f16"])
        layers = rng.randint(2, 4) if op == "stack" else 1
        B = 1 if op == "fused" else _log_int(rng, 2, 512 if op != "stack" else 16)
        kind = rng.choice(["config", "config", "aligned", "aligned", "ragged"])
        if kind == "config":
            c = _case(op, rng.choice(["mixtral", "dbrx", "deepseek"]), w, x, B=B,
                      shards=rng.choice([1, 1, 2, 4]), layers=layers)
        else:
            # Aligned sizes are multiples of 128, ragged ones (layers of up to
            # 4096 x 4096 and 128 tokens) of anything MXFP4 blocks allow.
            top = 8192 if kind == "aligned" else 4096
            step = 128 if kind == "aligned" else (32 if w == "mxfp4" else rng.choice([1, 2, 8]))
            E = _log_int(rng, 4, 64)
            c = dict(op=op, E=E, h=max(step, _log_int(rng, 256, top) // step * step),
                     I=max(step, _log_int(rng, 256, top) // step * step),
                     k=rng.randint(1, min(6, E)), renorm=rng.random() < 0.5, w=w, x=x,
                     B=min(B, 128) if kind == "ragged" else B, layers=layers)
        total = c["layers"] * c["E"] * 3 * c["h"] * c["I"] * WEIGHT_BITS[w] / 8
        if work(c)["flops"] <= MAX_FLOPS and total <= MAX_BYTES:
            return c


def prepare(case, seed):
    """The layer a serving program holds (router and packed experts) and the
    step's tokens; for a stack, its captured step."""
    dev = torch.device("cuda:0")
    E, h, I = case["E"], case["h"], case["I"]
    state = dict(case)
    batch = None if case["op"] == "fused" else case["B"]
    if case["op"] == "gate":
        gen = torch.Generator(device=dev).manual_seed(seed)
        state["x"] = torch.randn(batch, h, generator=gen, device=dev).to(DTYPES[case["x"]])
        state["gate_w"] = torch.randn(E, h, generator=gen, device=dev) * h ** -0.5
        return state
    made = [make_layer(E, h, I, DTYPES[case["w"]], router_std=h ** -0.5, seed=100 * seed + l,
                       batch=batch, device=dev, gen_device=dev, x_dtype=DTYPES[case["x"]])
            for l in range(case["layers"])]
    state["x"], state["gate_w"], state["buf"] = made[0]
    if case["op"] == "stack":
        state["stacked"] = [(gw, buf) for _, gw, buf in made]
        state["step"] = MoEStack(state["stacked"], E, h, I, case["k"],
                                 case["renorm"]).capture(state["x"])
    return state


def run(state):
    s = state
    if s["op"] == "gate":
        return F.gate_topk(s["x"], s["gate_w"], s["E"], s["h"], s["k"], s["renorm"])
    if s["op"] == "stack":
        return s["step"](s["x"])
    op = F.fused_moe if s["op"] == "fused" else F.batched_fused_moe
    return op(s["x"], s["gate_w"], s["buf"], s["E"], s["h"], s["I"], s["k"], s["renorm"])


def work(case):
    """The router and, per layer, the weights of the experts that B random
    tokens select (their expected number), read once; x read and the output
    written once."""
    E, h, I, k, B, L = (case[n] for n in ("E", "h", "I", "k", "B", "layers"))
    xs = 4 if case["x"] == "f32" else 2
    if case["op"] == "gate":
        return {"bytes": 4.0 * E * h + xs * B * h + 8 * B * k, "flops": 2.0 * B * E * h}
    distinct = E * (1 - (1 - k / E) ** B)
    expert = 3 * h * I * WEIGHT_BITS[case["w"]] / 8
    if case["w"] == "fp8":
        expert += 4 * (2 * I + h)
    return {"bytes": L * (distinct * expert + 4.0 * E * h) + 2.0 * xs * B * h,
            "flops": L * (2.0 * B * k * 3 * h * I + 2.0 * B * E * h)}


def tolerance(case):
    """About four times the error measured against 64 bits: the rounding of an
    fp16 output; else the split of x and act in two bf16 terms (bf16 and MXFP4
    weights), or fp32 sums in another order."""
    if case["op"] == "gate":
        return {"rel": 1e-5, "differ": 0.005}
    if case["x"] == "f16":
        return {"rel": 1e-3, "max": 4e-3}
    if case["w"] in ("bf16", "mxfp4"):
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 1e-5, "max": 1e-4}


def _matrices(buf, e, E, h, I, w):
    """Expert e's gate, up and down matrices in 64 bits, from the packed
    layout: the three matrices row by row, then fp8's row scales (fp32) or
    MXFP4's block scales (E8M0, one per 32 elements)."""
    n = h * I
    raw = buf.view(torch.uint8)
    blk = raw[raw.numel() // E * e:raw.numel() // E * (e + 1)]
    shapes = ((I, h), (I, h), (h, I))
    if w == "mxfp4":
        at = (3 * n // 2 + 15) // 16 * 16
        lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=buf.device)
        out = []
        for j, s in enumerate(shapes):
            q = blk[j * n // 2:(j + 1) * n // 2].to(torch.int64)
            v = torch.stack((lut[q & 15], lut[q >> 4]), dim=-1).reshape(-1, 32)
            sc = blk[at + j * n // 32:at + (j + 1) * n // 32].to(torch.float64)
            out.append((v * torch.exp2(sc - 127).unsqueeze(-1)).reshape(s))
        return out
    es = DTYPES[w].itemsize
    out = [blk[j * n * es:(j + 1) * n * es].view(DTYPES[w]).double().reshape(s)
           for j, s in enumerate(shapes)]
    if w == "fp8":
        at = (3 * n + 15) // 16 * 16
        sc = blk[at:at + 4 * (2 * I + h)].view(torch.float32).double()
        out = [m * r.unsqueeze(-1) for m, r in zip(out, sc.split((I, I, h)))]
    return out


def _route(x, gate_w, k, renorm):
    p = torch.softmax(x @ gate_w.double().t(), dim=-1)
    wt, ids = torch.topk(p, k, dim=-1)
    return ids, wt / wt.sum(-1, keepdim=True) if renorm else wt


def _layer(x, gate_w, buf, case):
    E, h, I = case["E"], case["h"], case["I"]
    ids, wt = _route(x, gate_w, case["k"], case["renorm"])
    out = torch.zeros_like(x)
    for e in range(E):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if len(t):
            g, u, d = _matrices(buf, e, E, h, I, case["w"])
            a = torch.nn.functional.silu(x[t] @ g.t()) * (x[t] @ u.t())
            out[t] += wt[t, slot].unsqueeze(-1) * (a @ d.t())
    return out


def exact(case, seed):
    s = prepare(case, seed)
    x = s["x"].double().reshape(-1, case["h"])
    if case["op"] == "gate":
        ids, wt = _route(x, s["gate_w"], case["k"], case["renorm"])
        return None, wt
    if case["op"] == "stack":
        for gw, buf in s["stacked"]:
            x = x + _layer(x, gw, buf, case)
        return x
    return _layer(x, s["gate_w"], s["buf"], case).reshape(s["x"].shape)
