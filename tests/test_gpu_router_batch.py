"""Router logits of 64 tokens and more, whose chains run on the matrix cores sixteen elements of every partition at a time, byte for byte
against the CPU oracle: rows that end in half a piece, token and expert counts that do not fill the last block, every block size; sums
that stay subnormal, that overflow, and that are not numbers; and the same from the bf16 rows of a prefill batch."""
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


@pytest.mark.parametrize("T,K,E,kind", [
    (64, 4096, 40, "normal"), (65, 128, 5, "normal"), (79, 384, 17, "normal"), (96, 640, 512, "normal"), (81, 256, 1021, "normal"),
    (300, 1152, 511, "normal"), (257, 2560, 512, "normal"), (520, 512, 250, "normal"),
    (70, 256, 40, "tiny"), (300, 384, 512, "tiny"), (66, 384, 40, "huge"), (300, 640, 500, "huge"), (67, 1152, 9, "nan"), (290, 512, 512, "nan")])
def test_router_logits(ctx, T, K, E, kind):
    rng = np.random.default_rng(K + T)
    w, x = rng.standard_normal((E, K)), rng.standard_normal((T, K))
    if kind == "tiny":                       # products about 2^-145
        w, x = w * 2.0 ** -70, x * 2.0 ** -75
    elif kind == "huge":                     # some sums leave the range, on the way or at the end
        w, x = np.abs(w) * 2.0 ** 60, x * 2.0 ** rng.integers(55, 67, (T, 1))
        x[1] = np.abs(x[1]); x[1, 3] = np.inf
    w, x = oracle.bf_bits(w.astype(f32)), oracle.bf(x.astype(f32))
    if kind == "nan":
        x[1, 7] = np.nan
    if kind == "normal":
        x[3] = rng.standard_normal(K).astype(f32)   # inputs that are not BF16
    off = rng.standard_normal(E).astype(f32) if kind == "normal" else np.zeros(E, f32)
    got = ctx.router_logits(ctx.upload(w), ctx.upload(x), T, K, E, ctx.upload(off)).numpy(f32).reshape(T, E)
    want = np.asarray(oracle.router_logits(w, x, T, K, E, off)).reshape(T, E)
    assert (np.isnan(got) == np.isnan(want)).all()
    assert np.where(np.isnan(got), f32(0), got).tobytes() == np.where(np.isnan(want), f32(0), want).tobytes()


@pytest.mark.parametrize("T,H,E", [(63, 384, 40), (64, 128, 33), (300, 640, 500), (1030, 384, 512)])
def test_prefill_logits(ctx, T, H, E):
    cfg = workload.tiny_config(H, E, 4, 128)
    weights = workload.LayerWeights(ctx, cfg, 91, ("normal", 0.5))
    x = workload.hidden_rows(ctx, T, H, 92)
    out, ws, logits = ctx.alloc(T * H * 4), ctx.alloc(ctx.moe_prefill_workspace_bytes(cfg, T)), ctx.alloc(T * E * 4)
    ctx.moe_prefill(cfg, weights.layer, x, T, out, ws, z.Trace(logits.ptr, None, None, None, None, None))
    ctx.moe_check()
    want = oracle.router_logits(weights.router.numpy(np.uint16), x.numpy(f32), T, H, E, weights.offsets.numpy(f32))
    assert logits.numpy(f32).tobytes() == np.asarray(want).astype(f32).tobytes()
    for b in (weights.router, weights.shared_gate, weights.shared_record, weights.records, x, out, ws, logits):
        ctx.free(b)


# Exact logits, and from 768 tokens on those that the selection can see.  There: partitions of two, three and four steps of 64 elements, the
# longest rows of the most experts (91 KB of LDS a workgroup), and more picks than the refinement selects itself
@pytest.mark.parametrize("T,H,E,topk", [(767, 1152, 72, 8), (768, 1152, 72, 8), (1025, 1152, 72, 8), (770, 3072, 80, 10), (769, 4096, 1024, 10), (771, 512, 128, 70)])
def test_prefill_selection_of_long_batches(ctx, T, H, E, topk):
    """Rows that tie exactly or nearly, zero, huge, tiny, not finite: ids and softmax weights are the exact layer's bits."""
    cfg = workload.tiny_config(H, E, topk, 128)
    weights = workload.LayerWeights(ctx, cfg, 303, ("normal", 0.5))
    n = T * topk
    router = weights.router.numpy(np.uint16).reshape(E, H).copy()
    router[17] = router[5]; router[61] = router[5]; router[33] = router[64]
    router[70] = router[12]; router[70, 100] ^= 1
    ctx.upload(router.ravel(), into=weights.router)
    x = workload.hidden_rows(ctx, T, H, 304).numpy(f32).reshape(T, H).copy()
    x[7] = 0.0; x[T - 1] = x[11]
    for row, power in ((8, 60), (9, -60), (12, -75), (T - 2, -120)):
        x[row] = oracle.bf(x[row] * f32(2.0 ** power))
    for bad in (False, True):
        if bad:
            x[20, 5] = np.nan; x[T - 3, 9] = np.inf; x[22, 9] = -np.inf; x[22, 10] = np.inf
        dx, got = ctx.upload(x.ravel()), []
        for call, size in ((ctx.moe_forward, ctx.moe_workspace_bytes), (ctx.moe_prefill, ctx.moe_prefill_workspace_bytes)):
            out, ws, ids, w = ctx.alloc(T * H * 4), ctx.alloc(size(cfg, T)), ctx.alloc(n * 4), ctx.alloc(n * 4)
            call(cfg, weights.layer, dx, T, out, ws, z.Trace(None, ids.ptr, w.ptr, None, None, None))
            if bad:
                with pytest.raises(z.ZcError, match="invalid router output"):
                    ctx.moe_check()
            else:
                ctx.moe_check()
            got.append((ids.numpy(np.int32).tobytes(), w.numpy(np.uint32).tobytes()))
            for b in (out, ws, ids, w):
                ctx.free(b)
        assert got[0][0] == got[1][0] and (bad or got[0][1] == got[1][1])
        ctx.free(dx)
    for b in (weights.router, weights.shared_gate, weights.shared_record, weights.records):
        ctx.free(b)
