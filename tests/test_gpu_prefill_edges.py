"""The prefill products' first requests: rows of 33 to 64 scale groups, whole and broken pieces of eight groups, tiles of one row to three
blocks, against the exact layer (its outputs byte for byte but for sums on a rounding boundary)."""
import numpy as np
import pytest
import zerocool_amd as z
from zerocool_amd import workload

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def ctx():
    c = z.Context(0)
    yield c
    c.close()


# groups of hidden and intermediate rows: 34 and 36, 40 and 42, 62 and 64, 2 and 6
@pytest.mark.parametrize("hidden,inter,bits", [(2176, 2304, (4, 4, 4, 4)), (2560, 2688, (4, 8, 8, 8)), (3968, 4096, (4, 4, 4, 4)), (128, 384, (8, 4, 4, 8))])
@pytest.mark.parametrize("T", [1, 15, 33, 47])
def test_prefill_matches_the_exact_layer(ctx, hidden, inter, bits, T):
    cfg = workload.tiny_config(hidden, 3, 2, inter, bits=bits)
    weights = workload.LayerWeights(ctx, cfg, 17 + T, ("normal", 0.5))
    x, outs = workload.hidden_rows(ctx, T, hidden, 18), []
    for call, size in ((ctx.moe_forward, ctx.moe_workspace_bytes), (ctx.moe_prefill, ctx.moe_prefill_workspace_bytes)):
        out, ws = ctx.alloc(T * hidden * 4), ctx.alloc(size(cfg, T))
        call(cfg, weights.layer, x, T, out, ws)
        ctx.moe_check()
        outs.append(out.numpy(f32).copy())
        ctx.free(out); ctx.free(ws)
    exact, fast = outs
    assert np.max(np.abs(fast - exact)) <= 2e-3 * np.max(np.abs(exact))
    assert np.mean(fast.view(np.uint32) == exact.view(np.uint32)) > 0.9999
    for b in (weights.router, weights.shared_gate, weights.shared_record, weights.records, x):
        ctx.free(b)


# the dispatch sort in one launch: just enough slots for it, one more step of slots than is in flight, a partly filled last stretch, more
# and fewer experts than a workgroup's wavefronts
@pytest.mark.parametrize("experts,topk,T", [(1024, 10, 103), (1024, 10, 2200), (1021, 7, 2927), (5, 2, 4100), (17, 4, 333)])
def test_prefill_dispatch_of_many_slots(ctx, experts, topk, T):
    cfg = workload.tiny_config(128, experts, topk, 128)
    weights = workload.LayerWeights(ctx, cfg, 19, ("zipf", 1.1))
    x, outs = workload.hidden_rows(ctx, T, 128, 20), []
    for call, size in ((ctx.moe_forward, ctx.moe_workspace_bytes), (ctx.moe_prefill, ctx.moe_prefill_workspace_bytes)):
        out, ws, ids = ctx.alloc(T * 128 * 4), ctx.alloc(size(cfg, T)), ctx.alloc(T * topk * 4)
        call(cfg, weights.layer, x, T, out, ws, z.Trace(None, ids.ptr, None, None, None, None))
        ctx.moe_check()
        outs.append((out.numpy(f32).copy(), ids.numpy(np.int32).tobytes()))
        for b in (out, ws, ids):
            ctx.free(b)
    (exact, exact_ids), (fast, fast_ids) = outs
    assert fast_ids == exact_ids
    assert np.max(np.abs(fast - exact)) <= 2e-3 * np.max(np.abs(exact))
    assert np.mean(fast.view(np.uint32) == exact.view(np.uint32)) > 0.9999
    for b in (weights.router, weights.shared_gate, weights.shared_record, weights.records, x, weights.offsets):
        ctx.free(b)


def down_rows_of_512(ctx, cfg, weights, T):
    x, n, outs = workload.hidden_rows(ctx, T, cfg.hidden, 24), T * cfg.topk, []
    for call, size in ((ctx.moe_forward, ctx.moe_workspace_bytes), (ctx.moe_prefill, ctx.moe_prefill_workspace_bytes)):
        out, ws, eo, sh = ctx.alloc(T * cfg.hidden * 4), ctx.alloc(size(cfg, T)), ctx.alloc(n * cfg.hidden * 4), ctx.alloc(T * cfg.hidden * 4)
        call(cfg, weights.layer, x, T, out, ws, z.Trace(None, None, None, eo.ptr, sh.ptr, None))
        ctx.moe_check()
        outs.append([b.numpy(f32).copy() for b in (out, eo, sh)])
        if call == ctx.moe_prefill:                               # outputs of the slots as bf16
            call(cfg, weights.layer, x, T, out, ws)
            assert out.numpy(f32).tobytes() == outs[1][0].tobytes()
        for b in (out, ws, eo, sh):
            ctx.free(b)
    for exact, fast in zip(*outs):
        assert np.max(np.abs(fast - exact)) <= 2.0 ** -7 * np.max(np.abs(exact))
        assert np.mean(fast.view(np.uint32) == exact.view(np.uint32)) > 0.9999
    assert np.max(np.abs(outs[1][0] - outs[0][0])) <= 2e-3 * np.max(np.abs(outs[0][0]))
    for b in (weights.router, weights.shared_gate, weights.shared_record, weights.records, weights.offsets, x):
        ctx.free(b)


# down rows of 512, a workgroup a block of weight rows: one to three blocks of token rows and several tiles, codes of either width
@pytest.mark.parametrize("hidden,bits", [(640, (4, 4, 4, 4)), (1152, (4, 8, 8, 8)), (128, (8, 8, 4, 4))])
@pytest.mark.parametrize("T", [1, 16, 20, 33, 48, 65, 130])
def test_prefill_down_rows_of_512(ctx, hidden, bits, T):
    cfg = workload.tiny_config(hidden, 2, 2, 512, bits=bits)      # both experts have every token
    down_rows_of_512(ctx, cfg, workload.LayerWeights(ctx, cfg, 23 + T, ("normal", 0.5)), T)


# The same with several blocks a workgroup, the last workgroup with fewer of them: five blocks by two (2 2 1; at 20 tokens) and by four (4 1), nine by four (4 4 1).
# Three experts have every token (tiles of 20 and 33 to 48 rows, and of 32 and 18), the others a few.
@pytest.mark.parametrize("hidden", [640, 1152])
@pytest.mark.parametrize("bits", [(4, 4, 4, 4), (4, 8, 8, 8)])
@pytest.mark.parametrize("T", [20, 33, 48, 50])
def test_prefill_down_rows_of_512_several_blocks_a_workgroup(ctx, hidden, bits, T):
    cfg = workload.tiny_config(hidden, 512, 10, 512, bits=bits)
    weights = workload.LayerWeights(ctx, cfg, 29 + T, ("normal", 0.5))
    offsets = weights.offsets.numpy(f32).copy()
    offsets[[3, 200, 511]] += 40                                   # (logits are N(0, 1) and their offsets)
    ctx.upload(offsets, into=weights.offsets)
    down_rows_of_512(ctx, cfg, weights, T)
