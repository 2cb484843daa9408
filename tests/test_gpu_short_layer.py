"""The exact layer's short-batch kernels at the edges of their ranges, byte for byte against the CPU oracle: the one-workgroup
selection and dispatch sort with its job list, and the expert kernels' groups of tokens, their two arithmetic
forms (fused products for BF16-valued rows of ordinary magnitude, separate ones for all others) and partial last steps."""
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


def rows(kind, T, hidden, seed):
    x = oracle.bf(np.random.default_rng(seed).standard_normal((T, hidden)))
    if kind == "fp32":                      # not BF16-valued in one row: products round
        x[T // 2, 3] = f32(1.0) + f32(2.0 ** -20)
    elif kind == "large":                   # beyond the fused form's range; sums stay finite
        x[-1] *= f32(2.0 ** 101)
    elif kind == "tiny":                    # subnormal inputs are exact in either form
        x[0] = oracle.bf(x[0] * f32(2.0 ** -128))
    return x


@pytest.mark.parametrize("T,hidden,inter,experts,topk,bits,group,kind", [
    (1, 512, 128, 8, 2, (4, 4, 4, 4), 64, "fp32"),         # one token, both forms
    (1, 544, 96, 8, 8, (8, 8, 8, 8), 32, "large"),         # byte codes, four-element blocks, last step partial
    (5, 512, 128, 4, 2, (4, 4, 4, 4), 64, "bf16"),         # experts with one to five slots: whole groups of tokens and what is left
    (16, 576, 640, 33, 3, (4, 4, 4, 4), 64, "tiny"),       # the most tokens of the joined selection, narrow blocks both ways
    (17, 512, 256, 600, 3, (4, 8, 8, 8), 64, "fp32"),      # one more; sixteen logits a lane; the shared expert in launches of its own
    (9, 512, 160, 96, 70, (8, 4, 8, 4), 32, "bf16"),       # more than 64 picks
    (64, 512, 128, 24, 16, (4, 4, 4, 4), 64, "fp32"),      # 1024 slots: the last size of the one-workgroup sort
    (65, 512, 128, 24, 16, (4, 4, 4, 4), 64, "bf16"),      # 1040: the sort over the device leaves the same job list
    (130, 512, 512, 2, 1, (4, 4, 4, 4), 64, "large"),      # long runs of one expert
])
def test_layer_against_the_oracle(ctx, T, hidden, inter, experts, topk, bits, group, kind):
    cfg = workload.tiny_config(hidden=hidden, experts=experts, topk=topk, inter=inter, group=group, bits=bits)
    w = workload.LayerWeights(ctx, cfg, 700 + T, ("normal", 0.5))
    x = rows(kind, T, hidden, 40 + T)
    dx, ws, out = ctx.upload(x), ctx.alloc(ctx.moe_workspace_bytes(cfg, T)), ctx.alloc(T * hidden * 4)
    ctx.fill(ws, 0xff)                       # what the buffers held before does not matter
    ctx.moe_forward(cfg, w.layer, dx, T, out, ws)
    ctx.moe_check()
    h = w.host()
    want = oracle.moe_layer(oracle.Config(*[getattr(cfg, n) for n, _ in z.Config._fields_]), h["router"], h["shared_gate"],
                            h["shared_record"], h["records"], h["stride"], x, T, router_offsets=h["offsets"], threads=8)
    want = want[0] if isinstance(want, tuple) else want
    assert out.numpy(f32).tobytes() == np.ascontiguousarray(want).tobytes()
    for b in (dx, ws, out, w.router, w.shared_gate, w.shared_record, w.records, w.offsets):
        ctx.free(b)


@pytest.mark.parametrize("tokens,topk,experts", [(1, 1, 1), (1, 64, 64), (13, 5, 7), (64, 1, 1024), (128, 8, 1024), (1023, 1, 3), (1024, 1, 1), (128, 8, 1025), (1025, 1, 9)])
def test_dispatch_sort(ctx, tokens, topk, experts):
    n = tokens * topk
    ids = np.random.default_rng(n + experts).integers(0, experts, n, dtype=np.int64).astype(np.int32)
    if n > 70:
        ids[60:70] = experts - 1             # a run across the border of two waves
    d = ctx.upload(ids)
    off, slots, selected, count, status = ctx.build_dispatch(d, tokens, topk, experts)
    want_off, want_slots, want_selected = oracle.dispatch(ids, tokens, topk, experts)
    assert off.numpy(np.int32).tobytes() == want_off.tobytes() and slots.numpy(np.int32).tobytes() == want_slots.tobytes()
    n_selected = int(count.numpy(np.int32)[0])
    assert n_selected == len(want_selected) and selected.numpy(np.int32)[:n_selected].tobytes() == want_selected.tobytes()
    assert status.numpy(np.int32)[0] == 0


# rows of one weight piece and of several batches, a row too long for LDS (the general kernel), and numbers of tokens and
# experts that leave a group of either partly empty
@pytest.mark.parametrize("T,K,E", [(1, 128, 1), (2, 128, 5), (3, 2560, 17), (4, 1152, 512), (63, 640, 33), (1, 16384, 3), (5, 4224, 20),
                                   (64, 3968, 35), (64, 4096, 35), (64, 4096, 272), (63, 4096, 17)])   # the longest row of the short kernel, and 64 tokens of a longer one on the tiles
def test_router_logits(ctx, T, K, E):
    rng = np.random.default_rng(K + T)
    w, x, off = oracle.bf_bits(rng.standard_normal((E, K))), oracle.bf(rng.standard_normal((T, K))), rng.standard_normal(E).astype(f32)
    got = ctx.router_logits(ctx.upload(w), ctx.upload(x), T, K, E, ctx.upload(off)).numpy(f32)
    assert got.tobytes() == oracle.router_logits(w, x, T, K, E, off).tobytes()


# The single-launch kernels for several tokens, which a call can ask for, against the layer by layer path that it takes
# otherwise: the same bytes, and the same reports for inputs that are not BF16-valued or not routable.
@pytest.mark.parametrize("hidden,bits,tokens", [(1024, (4, 4, 4, 4), (2, 8, 9, 64, 70)), (1024, (4, 8, 8, 8), (2, 9, 64)), (3072, (4, 4, 4, 4), (3, 17))])
def test_stack_paths_agree(ctx, hidden, bits, tokens):
    cfg = workload.tiny_config(hidden=hidden, experts=64, topk=10, inter=512, bits=bits)
    layers = [workload.LayerWeights(ctx, cfg, 800 + l, ("zipf", 1.1)) for l in range(3)]
    stack = ctx.stack_create(cfg, [l.layer for l in layers], max(tokens))
    for T in tokens:
        n = T * cfg.topk
        x, out = workload.hidden_rows(ctx, T, hidden, 60 + T), ctx.alloc(T * hidden * 4)
        ids, w, outs = ctx.alloc(3 * n * 4), ctx.alloc(3 * n * 4), ctx.alloc(3 * T * hidden * 4)
        got = []
        for single in (True, False):
            for trace in (z.StackTrace(ids.ptr, w.ptr, outs.ptr, None), None):
                ctx.fill(out, 0xff)
                ctx.stack_decode(stack, x, T, out, trace, single=single)
                ctx.moe_check()
                got.append(out.numpy(np.uint8).tobytes())
            got[-2:] = [(got[-2], ids.numpy(np.uint8).tobytes(), w.numpy(np.uint8).tobytes(), outs.numpy(np.uint8).tobytes()), got[-1]]
            assert got[-2][0] == got[-1]
        assert got[0] == got[2] and got[1] == got[3]
        for value, text in ((np.float32(1.0000001), "BF16"), (np.float32("nan"), "invalid router output")):
            bad = x.numpy(f32)
            bad[-hidden:] = value           # the last token's row
            dbad = ctx.upload(bad)
            for single in (True, False):
                ctx.stack_decode(stack, dbad, T, out, single=single)
                with pytest.raises(z.ZcError, match=text):
                    ctx.moe_check()
            ctx.free(dbad)
        for b in (x, out, ids, w, outs):
            ctx.free(b)
    ctx.stack_destroy(stack)
    for l in layers:
        for b in (l.router, l.shared_gate, l.shared_record, l.records, l.offsets):
            ctx.free(b)
