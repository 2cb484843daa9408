"""The affine kernels that run four tokens a workgroup on the matrix cores, byte for byte against the CPU oracle: quads that
are exact in any order, quads whose chain has to be run, rows whose products round; rows of one step, of half a step more, and
jobs of one to four tokens; as operators, and in a layer (the reference's lanes: qwen.metal:46-81, 112-144)."""
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


def rows(kind, T, K, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((T, K))
    if kind == "spread":                 # exponents 2^-30 to 1: nearly every quad runs its chain
        x *= 2.0 ** -rng.integers(0, 31, (T, K))
    elif kind == "edge":                 # one element of every other quad about 2^-11 of the others: quads on both sides of the line
        x[:, ::8] *= 2.0 ** -rng.integers(9, 14, (T, (K + 7) // 8))
    elif kind == "powers":               # single-bit significands, zeros of both signs, whole quads of zeros
        x = np.sign(x) * 2.0 ** rng.integers(-20, 20, (T, K)) * (rng.random((T, K)) < 0.6)
        x[:, K // 2:K // 2 + 16] = -0.0
    elif kind == "far":                  # the ends of the range whose products cannot round
        x = np.sign(x) * np.where(rng.random((T, K)) < 0.5, 2.0 ** -99.0, 2.0 ** 60.0)
    x = oracle.bf(x.astype(f32))
    if kind == "strange":                # one row that is not BF16 among rows that are, one beyond the range, one with an infinity
        x[T // 2, 5] = f32(1.0 + 2.0 ** -20)
        x[1] *= f32(2.0 ** 101)
        x[T - 1, K - 1] = np.inf
    return x


@pytest.mark.parametrize("bits,K,N,T,kind", [
    (4, 512, 8, 133, "normal"), (4, 1024, 24, 131, "spread"), (4, 512, 40, 130, "edge"), (4, 1536, 8, 129, "powers"), (4, 512, 16, 132, "far"),
    (4, 512, 8, 130, "strange"), (4, 640, 24, 133, "normal"), (4, 128, 8, 131, "spread"), (4, 384, 12, 130, "edge"), (4, 512, 7, 129, "powers"),
    (4, 640, 8, 130, "strange"), (8, 512, 8, 133, "normal"), (8, 1024, 24, 131, "spread"), (8, 512, 40, 130, "powers"), (8, 512, 16, 129, "strange"),
    # products of fewer outputs and rows than fill the chip's SIMDs stay with the lanes, as those above; from here on not
    (4, 512, 256, 133, "normal"), (4, 1024, 264, 131, "spread"), (4, 512, 296, 130, "edge"), (4, 1536, 256, 129, "powers"), (4, 512, 272, 132, "far"), (4, 512, 256, 130, "strange"),
    (4, 640, 280, 133, "normal"), (4, 128, 264, 131, "spread"), (4, 384, 268, 130, "edge"), (4, 512, 263, 129, "powers"), (4, 640, 264, 130, "strange"), (8, 512, 256, 133, "normal"),
    (8, 1024, 280, 131, "spread"), (8, 512, 296, 130, "powers"), (8, 512, 272, 129, "strange"),
    # either side of the numbers of rows, and of waves, from which the two products go to the matrix cores
    (4, 512, 352, 47, "strange"), (4, 512, 352, 48, "strange"), (4, 640, 264, 127, "edge"), (4, 640, 264, 128, "edge"), (8, 512, 352, 47, "spread"), (8, 512, 352, 48, "spread"),
    (4, 512, 124, 128, "edge"), (4, 512, 128, 128, "edge"), (4, 512, 248, 128, "edge"), (4, 512, 12, 2724, "edge"), (4, 512, 12, 2732, "edge"), (4, 384, 12, 2732, "strange"),
    # the longest rows of each format whose four tokens leave room for two workgroups, and one step more; rows that are not BF16
    # one at a time (5632 and 8704 inputs) and two
    (4, 8704, 256, 129, "strange"), (4, 8704, 320, 50, "edge"), (4, 9216, 256, 129, "strange"), (4, 7936, 256, 129, "strange"), (4, 7936, 320, 51, "edge"), (4, 8064, 256, 129, "strange"),
    (8, 7680, 256, 129, "strange"), (8, 8192, 256, 129, "strange"), (4, 4096, 256, 129, "strange"), (4, 4224, 256, 129, "strange"), (4, 5120, 256, 129, "strange"), (4, 5632, 256, 129, "strange")])
def test_operators(ctx, bits, K, N, T, kind):
    rng = np.random.default_rng(K + N + T)
    mats = []
    for _ in range(2):
        w = rng.integers(0, 2 ** 32, N * K * bits // 32, dtype=np.uint64).astype(np.uint32)
        s, b = oracle.bf_bits(0.02 * rng.random(N * K // 64) + 1e-4), oracle.bf_bits(-0.16 * rng.random(N * K // 64))
        bufs = [ctx.upload(v) for v in (w, s, b)]
        mats.append((oracle.make_linear(w, s, b, K, N, 64, bits), z.Linear(*[v.ptr for v in bufs], K, N, 64, 0, 1, bits), bufs))
    (og, dg, _), (ou, du, _) = mats
    x = rows(kind, T, K, 9 * K + T)
    dx, gather = ctx.upload(x), rng.integers(0, T, T).astype(np.int32)
    got = [ctx.linear(dg, dx, T), ctx.linear(dg, dx, T, float_output=True), ctx.gated_linear(dg, du, dx, T, T), ctx.gated_linear(dg, du, dx, T, T, ctx.upload(gather))]
    want = [oracle.linear(og, x, T), oracle.linear(og, x, T, float_output=True), oracle.gated_linear(og, ou, x, T), oracle.gated_linear(og, ou, x, T, gather)]
    for g, o in zip(got, want):
        assert g.numpy(f32).tobytes() == np.ascontiguousarray(o).tobytes()


# experts with one to four tokens and more, images of the inputs and of the activations; rows whose activations are not
# exact either (inputs of 2^101 times the usual)
@pytest.mark.parametrize("T,hidden,inter,experts,topk,bits,kind", [
    (2, 512, 512, 8, 4, (4, 4, 4, 4), "normal"), (3, 1024, 128, 3, 3, (4, 4, 4, 4), "spread"), (7, 640, 640, 4, 2, (4, 4, 4, 4), "edge"),
    (11, 512, 512, 5, 3, (4, 8, 8, 8), "normal"), (6, 512, 512, 6, 6, (8, 4, 4, 8), "powers"), (9, 512, 640, 3, 1, (4, 4, 4, 4), "strange"),
    (66, 512, 512, 6, 2, (4, 4, 4, 4), "spread"), (520, 512, 128, 3, 2, (4, 4, 4, 4), "normal"),
    # the longest rows and one step more (then both phases are the lanes'), rows of either form's own width, and lists of jobs with one to four tokens
    (7, 8704, 512, 3, 2, (4, 4, 4, 4), "strange"), (7, 9216, 512, 3, 2, (4, 4, 4, 4), "strange"), (9, 512, 8704, 3, 2, (4, 4, 4, 4), "normal"),
    (33, 1024, 640, 24, 3, (4, 4, 4, 4), "strange"), (37, 1536, 512, 40, 4, (4, 8, 8, 8), "strange"), (70, 512, 512, 64, 4, (8, 8, 8, 8), "strange"),
    # either side of the numbers of tokens from which a batch goes to the matrix cores
    (2, 2048, 1024, 6, 3, (4, 4, 4, 4), "edge"), (3, 2048, 1024, 6, 3, (4, 4, 4, 4), "edge"), (8, 512, 512, 9, 4, (4, 4, 4, 4), "normal"), (9, 512, 512, 9, 4, (4, 4, 4, 4), "normal"),
    (2, 512, 512, 6, 4, (4, 8, 8, 8), "edge"), (2, 512, 512, 6, 4, (4, 4, 8, 4), "spread"), (11, 512, 512, 9, 4, (8, 8, 8, 8), "normal"), (12, 512, 512, 9, 4, (8, 8, 8, 8), "normal"),
    (12, 512, 512, 97, 4, (8, 4, 8, 4), "normal"), (12, 512, 512, 96, 4, (8, 4, 8, 4), "normal"), (3, 4096, 2048, 4, 3, (8, 8, 8, 8), "normal"), (4, 4096, 2048, 4, 3, (8, 8, 8, 8), "normal")])
def test_layer(ctx, T, hidden, inter, experts, topk, bits, kind):
    cfg = workload.tiny_config(hidden=hidden, experts=experts, topk=topk, inter=inter, bits=bits)
    w = workload.LayerWeights(ctx, cfg, 900 + T, ("normal", 0.5))
    x = rows(kind, T, hidden, 70 + T)
    if kind == "strange":
        x[T - 1, hidden - 1] = 1         # (an infinity leaves nothing to route)
    dx, ws, out = ctx.upload(x), ctx.alloc(ctx.moe_workspace_bytes(cfg, T)), ctx.alloc(T * hidden * 4)
    ctx.fill(ws, 0xff)
    ctx.moe_forward(cfg, w.layer, dx, T, out, ws)
    ctx.moe_check()
    h = w.host()
    want = oracle.moe_layer(oracle.Config(*[getattr(cfg, n) for n, _ in z.Config._fields_]), h["router"], h["shared_gate"],
                            h["shared_record"], h["records"], h["stride"], x, T, router_offsets=h["offsets"], threads=8)
    want = want[0] if isinstance(want, tuple) else want
    assert out.numpy(f32).tobytes() == np.ascontiguousarray(want).tobytes()
