"""What the speed of this library is measured on: the MoE layer path as its users run it.

A case is one of four kinds of call:
  stack    decode steps through a stack of layers (`Context.stack_decode`), the serving loop's inner step
  layer    one exact layer call (`Context.moe_forward`, or `moe_forward_static` where nothing may be allocated)
  prefill  one layer over a prompt chunk (`Context.moe_prefill`)
  experts  the operators an engine calls itself per expert: gathered gate/up, down, scatter (`gated_linear`, `linear`,
           `scatter_experts`)
at the layer shapes of `workload.config`: S (hidden 2048, intermediate 512), S-mixed (the same with affine Q8 down and
shared projections), F (hidden 3072, intermediate 1024) and ref (hidden 2560, intermediate 640, the reference model's
own), all with 512 experts, top-10 and group 64.

Weights, router offsets and inputs come from the repository's seeded generator, on the GPU.  Decoding takes other hidden
rows at every step, as a serving loop does; prompt rows are standard normal, as after a normalisation."""
import math
import random

import numpy as np
import torch

import zerocool_amd as z
from zerocool_amd import synth, workload

SHAPES = ("S", "S-mixed", "F", "ref")
SKEWS = {"none": None, "normal": ("normal", 0.5), "zipf": ("zipf", 1.1)}


def listed():
    return [
        # one token through one layer without a stack: the smallest call, from a loop that may not allocate
        {"name": "layer-S-1", "kind": "layer", "shape": "S", "tokens": 1, "skew": "normal", "static": True},
        # a short prompt or a verification batch through the exact layer, at the reference model's shape
        {"name": "layer-ref-40", "kind": "layer", "shape": "ref", "tokens": 40, "skew": "normal", "static": False},
        # single-stream decoding through the stand-in model's layers (six of its 48: a state has to fit three times over)
        {"name": "decode-F-1", "kind": "stack", "shape": "F", "tokens": 1, "layers": 6, "steps": 4, "skew": "zipf"},
        # the same stack serving a small and a large batch
        {"name": "decode-F-8", "kind": "stack", "shape": "F", "tokens": 8, "layers": 6, "steps": 2, "skew": "zipf"},
        {"name": "decode-F-64", "kind": "stack", "shape": "F", "tokens": 64, "layers": 6, "steps": 1, "skew": "zipf"},
        # one layer, a batch whose tokens go to many different experts
        {"name": "decode-S-32", "kind": "stack", "shape": "S", "tokens": 32, "layers": 1, "steps": 1, "skew": "normal"},
        # the mixed 4/8-bit artifact, an odd batch
        {"name": "decode-mixed-5", "kind": "stack", "shape": "S-mixed", "tokens": 5, "layers": 4, "steps": 1, "skew": "normal"},
        # single-stream decoding at the reference model's own shape
        {"name": "decode-ref-1", "kind": "stack", "shape": "ref", "tokens": 1, "layers": 4, "steps": 2, "skew": "normal"},
        # an engine that walks the experts itself: eight experts, a ragged number of rows each
        {"name": "experts-ref", "kind": "experts", "shape": "ref", "tokens": 96, "experts": 8, "rows": 21},
        # prompt chunks: the benchmark's, a short one of the mixed artifact, a ragged one of the large shape
        {"name": "prefill-S-2048", "kind": "prefill", "shape": "S", "tokens": 2048, "skew": "none"},
        {"name": "prefill-mixed-300", "kind": "prefill", "shape": "S-mixed", "tokens": 300, "skew": "normal"},
        {"name": "prefill-F-1500", "kind": "prefill", "shape": "F", "tokens": 1500, "skew": "zipf"},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choices(("stack", "layer", "prefill", "experts"), (9, 3, 6, 2))[0]
    shape = rng.choice(SHAPES)
    skew = rng.choice(tuple(SKEWS))
    if kind == "stack":
        return {"kind": kind, "shape": shape, "tokens": _log_int(rng, 1, 64), "layers": rng.randint(1, 4), "steps": 1, "skew": skew}
    if kind == "layer":
        tokens = _log_int(rng, 1, 96)
        return {"kind": kind, "shape": shape, "tokens": tokens, "skew": skew, "static": tokens <= 8 and rng.random() < 0.5}
    if kind == "prefill":
        return {"kind": kind, "shape": shape, "tokens": _log_int(rng, 100, 1400), "skew": skew}
    return {"kind": kind, "shape": shape, "tokens": 64 + rng.randint(0, 64), "experts": rng.randint(2, 8), "rows": rng.randint(1, 64)}


class _Out:
    """Device memory for fp32 results that torch looks at in place: `tensor` keeps it alive, also when the state has gone."""

    def __init__(self, ctx, *shape):
        self.ctx, self.buf = ctx, ctx.zeros(4 * math.prod(shape))
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (self.buf.ptr, False), "version": 3}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        self.ctx.free(self.buf)


_context = None


class _State:
    """What one case keeps between calls.  All states share the process's one context, as the parts of a user's program do:
    calls follow each other on its stream (the static-scratch layer call asks for that).  A state gives its memory back."""

    def __init__(self, case):
        global _context
        if _context is None:
            _context = z.Context(0)
        self.ctx, self.cfg, self.case = _context, workload.config(case["shape"]), case
        self.stack, self.bufs = None, []

    def keep(self, buf):
        self.bufs.append(buf)
        return buf

    def __del__(self):
        if self.stack is not None:
            self.ctx.stack_destroy(self.stack)
        for buf in self.bufs:
            self.ctx.free(buf)


def prepare(case, seed):
    s = _State(case)
    ctx, cfg, T, H = s.ctx, s.cfg, case["tokens"], s.cfg.hidden
    seed = random.Random(seed).getrandbits(30) * 64
    steps = case.get("steps", 1)
    s.xs = [s.keep(workload.hidden_rows(ctx, T, H, seed + 1 + i)) for i in range(steps)]
    if case["kind"] == "experts":
        n, E = case["rows"], case["experts"]
        stride = workload.record_stride(ctx, cfg)
        records = s.keep(ctx.alloc(E * stride))
        ctx.synth_records(cfg, records, stride, E, seed * 4096)
        slots = random.Random(seed).sample(range(T * cfg.topk), n * E)      # the (token, rank) slots of each expert, ascending
        s.rows, s.slots, s.linears = [], [], []
        for e in range(E):
            mine = np.sort(np.array(slots[e * n:(e + 1) * n], np.int32))
            s.rows.append(s.keep(ctx.upload(mine // cfg.topk)))
            s.slots.append(s.keep(ctx.upload(mine)))
            record = records.view(e * stride, stride)
            s.linears.append([ctx.expert_linear(cfg, record, p) for p in range(3)])
        s.act, s.y = s.keep(ctx.alloc(n * cfg.inter * 4)), s.keep(ctx.alloc(n * H * 4))
        s.out = _Out(ctx, T * cfg.topk, H)
        s.result = s.out.tensor()
    else:
        skew = SKEWS[case["skew"]]
        s.layers = [workload.LayerWeights(ctx, cfg, seed + 8 + l, skew) for l in range(case.get("layers", 1))]
        for l in s.layers:
            s.bufs += [b for b in (l.router, l.shared_gate, l.shared_record, l.records, l.offsets) if b is not None]
        s.outs = [_Out(ctx, T, H) for _ in range(steps)]
        s.result = [o.tensor() for o in s.outs]
        if case["kind"] == "stack":
            s.stack = ctx.stack_create(cfg, [l.layer for l in s.layers], T)
        elif case["kind"] == "prefill":
            s.workspace = s.keep(ctx.alloc(ctx.moe_prefill_workspace_bytes(cfg, T)))
        elif not case["static"]:
            s.workspace = s.keep(ctx.alloc(ctx.moe_workspace_bytes(cfg, T)))
    ctx.finish()
    return s


def run(s):
    ctx, cfg, case, T = s.ctx, s.cfg, s.case, s.case["tokens"]
    if case["kind"] == "stack":
        for x, out in zip(s.xs, s.outs):
            ctx.stack_decode(s.stack, x, T, out.buf)
    elif case["kind"] == "prefill":
        ctx.moe_prefill(cfg, s.layers[0].layer, s.xs[0], T, s.outs[0].buf, s.workspace)
    elif case["kind"] == "layer" and case["static"]:
        ctx.moe_forward_static(cfg, s.layers[0].layer, s.xs[0], T, s.outs[0].buf)
    elif case["kind"] == "layer":
        ctx.moe_forward(cfg, s.layers[0].layer, s.xs[0], T, s.outs[0].buf, s.workspace)
    else:
        n = case["rows"]
        for (gate, up, down), rows, slots in zip(s.linears, s.rows, s.slots):
            ctx.gated_linear(gate, up, s.xs[0], T, n, rows, out=s.act)
            ctx.linear(down, s.act, n, out=s.y)
            ctx.scatter_experts(s.y, slots, n, cfg.hidden, s.out.buf)
    return s.result


def _record_bytes(cfg, shared):
    up, down = (cfg.shared_bits_gate_up, cfg.shared_bits_down) if shared else (cfg.bits_gate_up, cfg.bits_down)
    weights = cfg.hidden * cfg.inter
    return 2 * (weights * up // 8 + weights // cfg.group * 4) + weights * down // 8 + weights // cfg.group * 4


def _distinct(cfg, tokens, skew):
    """Experts that a batch of standard normal rows reaches: logits are N(0, 1) plus the router's offsets."""
    offsets = 0.0
    if skew == "normal":
        offsets = synth.normal_offsets(cfg.experts, 5, SKEWS[skew][1])
    elif skew == "zipf":
        offsets = synth.zipf_offsets(cfg.experts, 5, SKEWS[skew][1])
    logits = np.random.RandomState(5).standard_normal((tokens, cfg.experts)) + offsets
    return len(np.unique(np.argpartition(-logits, cfg.topk, axis=1)[:, :cfg.topk]))


def work(case):
    cfg, T = workload.config(case["shape"]), case["tokens"]
    H, I, k = cfg.hidden, cfg.inter, cfg.topk
    routed, shared = _record_bytes(cfg, False), _record_bytes(cfg, True)
    if case["kind"] == "experts":
        n, E = case["rows"], case["experts"]
        return {"bytes": E * routed + T * H * 4 + E * n * (H * 4 + 8), "flops": E * n * 6 * H * I}
    per_token = 6 * H * I * (k + 1) + 2 * H * (cfg.experts + 1)
    fixed = 2 * H * (cfg.experts + 1) + shared + T * H * 8
    first = _distinct(cfg, T, case["skew"])
    # behind the first layer a batch of the synthetic stack agrees on its experts, nearly: at least one token's share
    experts = first + (case.get("layers", 1) - 1) * k
    steps, layers = case.get("steps", 1), case.get("layers", 1)
    return {"bytes": steps * (layers * fixed + experts * routed), "flops": steps * layers * T * per_token}


def tolerance(case):
    # Decoding, the exact layer and the operators are specified bit for bit.  The prefill product is specified by a
    # tolerance on BF16 outputs: a sum that falls on the other side of a rounding boundary moves one activation or one
    # output by 2^-8 of itself.  Sums per scale group in fp32 against sums in 64 bits move the output of ten experts by
    # 2e-4 to 3e-4 and single values by 8e-3.
    if case["kind"] == "prefill":
        return {"rel": 1e-3, "max": 3e-2}
    return "exact"
