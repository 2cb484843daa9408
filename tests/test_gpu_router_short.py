"""Router logits of two to 64 tokens, whose chains run on the matrix cores, byte for byte against the CPU oracle: the longest rows of
two, three and four tokens a workgroup and one piece more, workgroups of two waves and of four, partly filled either way, and short rows; sums
that stay subnormal, that overflow, and that are not numbers."""
import numpy as np
import pytest
import oracle
import zerocool_amd as z

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def ctx():
    c = z.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("T,K,E,kind", [
    (2, 8064, 9, "normal"), (2, 8192, 9, "normal"), (3, 5376, 4, "normal"), (3, 5504, 7, "normal"), (4, 3968, 8, "normal"), (7, 2048, 11, "normal"),
    (64, 3968, 247, "normal"), (62, 3968, 273, "normal"), (5, 256, 40, "tiny"), (6, 384, 40, "huge"), (2, 1152, 5, "nan"),
    # one piece of a row a thread and more, in workgroups of two waves and of four (more than the chip holds of two)
    (5, 128, 40, "normal"), (3, 512, 40, "nan"), (5, 640, 40, "normal"), (64, 128, 1024, "tiny"), (64, 1024, 1021, "normal"), (63, 1152, 1024, "huge")])
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
    off = rng.standard_normal(E).astype(f32) if kind == "normal" else np.zeros(E, f32)
    got = ctx.router_logits(ctx.upload(w), ctx.upload(x), T, K, E, ctx.upload(off)).numpy(f32).reshape(T, E)
    want = np.asarray(oracle.router_logits(w, x, T, K, E, off)).reshape(T, E)
    assert (np.isnan(got) == np.isnan(want)).all()
    assert np.where(np.isnan(got), f32(0), got).tobytes() == np.where(np.isnan(want), f32(0), want).tobytes()
