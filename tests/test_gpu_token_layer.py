"""One token alone through a layer: its picks, made inside the gate/up launch or by a launch of their own, stand for the job list.
Every output the layer can dump, byte for byte against the CPU oracle, at the smallest and largest numbers of experts and picks
either way takes, in every format, and an input without picks (qwen.metal:742-795, model.cpp:431-557)."""
import numpy as np
import pytest
import oracle
import zerocool_amd as z
from zerocool_amd import workload

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def ctx():
    c = z.Context(0)
    yield c
    c.close()


def run(ctx, cfg, w, x):
    shapes = dict(logits=cfg.experts, ids=cfg.topk, weights=cfg.topk, expert_out=cfg.topk * cfg.hidden, shared=cfg.hidden, gate=1)
    bufs = {k: ctx.alloc(n * 4) for k, n in shapes.items()}
    ws, out = ctx.alloc(ctx.moe_workspace_bytes(cfg, 1)), ctx.alloc(cfg.hidden * 4)
    ctx.fill(ws, 0xff)
    ctx.moe_forward(cfg, w.layer, ctx.upload(x), 1, out, ws, z.Trace(*[b.ptr for b in bufs.values()]))
    return bufs, out


# Up to twenty picks inside the gate/up launch where they are found together (up to 512 experts, as many lanes as picks), up to twelve where they
# are found one by one, and one more by the launch of their own, up to 64 by its first wave's lanes; rows of either width, groups of 32, Q8, a
# shared expert of another format
@pytest.mark.parametrize("hidden,inter,experts,topk,bits,group", [
    (128, 128, 1, 1, (4, 4, 4, 4), 64), (512, 640, 3, 3, (4, 4, 4, 4), 64), (512, 512, 64, 63, (4, 4, 4, 4), 64), (512, 128, 66, 64, (4, 8, 8, 8), 64),
    (512, 128, 66, 65, (4, 8, 8, 8), 64), (512, 128, 512, 20, (4, 4, 4, 4), 64), (512, 128, 153, 20, (4, 4, 4, 4), 64), (512, 128, 152, 20, (4, 8, 8, 8), 64),
    (512, 128, 512, 21, (4, 4, 4, 4), 64), (512, 128, 96, 12, (4, 4, 4, 4), 64), (512, 128, 70, 12, (4, 4, 4, 4), 64), (512, 128, 70, 13, (4, 4, 4, 4), 64),
    (512, 128, 1024, 12, (4, 4, 4, 4), 64), (512, 128, 1024, 13, (4, 4, 4, 4), 64), (640, 128, 512, 10, (8, 8, 4, 4), 64), (256, 128, 513, 10, (8, 4, 4, 8), 32), (128, 64, 1024, 64, (4, 4, 4, 4), 64),
    (32512, 64, 3, 2, (4, 4, 4, 4), 64), (32576, 64, 3, 2, (4, 4, 4, 4), 64)])   # the longest row beside which the selection has room in LDS, and one more
def test_layer(ctx, hidden, inter, experts, topk, bits, group):
    cfg = workload.tiny_config(hidden=hidden, experts=experts, topk=topk, inter=inter, bits=bits, group=group)
    w = workload.LayerWeights(ctx, cfg, 500 + topk, ("normal", 0.5))
    x = oracle.bf(np.random.default_rng(topk).standard_normal((1, hidden)).astype(f32))
    bufs, out = run(ctx, cfg, w, x)
    ctx.moe_check()
    h = w.host()
    want, tr = oracle.moe_layer(oracle.Config(*[getattr(cfg, n) for n, _ in z.Config._fields_]), h["router"], h["shared_gate"], h["shared_record"],
                                h["records"], h["stride"], x, 1, router_offsets=h["offsets"], threads=8, trace=True)
    for k, b in bufs.items():
        assert b.numpy(np.int32 if k == "ids" else f32).tobytes() == tr[k].tobytes(), k
    assert out.numpy(f32).tobytes() == want.tobytes()


@pytest.mark.parametrize("topk", [3, 65])   # (either way of picking)
def test_a_token_without_picks_is_reported(ctx, topk):
    cfg = workload.tiny_config(hidden=512, experts=70, topk=topk, inter=128)
    w = workload.LayerWeights(ctx, cfg, 77, None)
    x = np.full((1, 512), np.nan, f32)
    bufs, _ = run(ctx, cfg, w, x)
    with pytest.raises(z.ZcError):
        ctx.moe_check()
    assert (bufs["ids"].numpy(np.int32) == -1).all()
    run(ctx, cfg, w, oracle.bf(np.ones((1, 512), f32)))
    ctx.moe_check()                              # reported once


# One token: by the one-token kernel, except where a stack has a single layer or Q8 parts; the same bytes and the same reports either way.
@pytest.mark.parametrize("layers,bits,single", [(1, (4, 4, 4, 4), False), (2, (4, 4, 4, 4), True), (2, (4, 8, 8, 8), False), (2, (4, 4, 8, 4), False)])
def test_which_way_a_stack_goes(ctx, layers, bits, single):
    cfg = workload.tiny_config(hidden=1024, experts=64, topk=10, inter=512, bits=bits)
    ws = [workload.LayerWeights(ctx, cfg, 300 + l, ("zipf", 1.1)) for l in range(layers)]
    stack = ctx.stack_create(cfg, [w.layer for w in ws], 1)
    assert ctx.stack_is_persistent(stack, 1) and ctx.stack_single_launch(stack, 1) == single
    x, outs = workload.hidden_rows(ctx, 1, cfg.hidden, 5), []
    for how in ({}, {"single": True}, {"layered": True}):
        out = ctx.alloc(cfg.hidden * 4)
        ctx.stack_decode(stack, x, 1, out, **how)
        ctx.moe_check()
        outs.append(out.numpy(f32).tobytes())
    assert outs[0] == outs[1] == outs[2]
    bad = np.full(cfg.hidden, 0.5, f32); bad[7] = f32(1 + 2.0 ** -20)
    ctx.stack_decode(stack, ctx.upload(bad), 1, ctx.alloc(cfg.hidden * 4))
    with pytest.raises(z.ZcError, match="not BF16-valued"):
        ctx.moe_check()
    ctx.stack_destroy(stack)
