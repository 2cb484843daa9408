"""The gather's row check of the fused gate/up operator: a refused call leaves the output alone, an accepted one is the oracle's.
Lists up to 256 rows are looked at by the product's own kernel (the lanes', or the matrix cores' where the product has a wave for every SIMD: 64 outputs
from 253 rows on, 256 from 61), longer ones in front of it."""
import threading
import numpy as np
import pytest
import oracle
import zerocool_amd as z
from test_gpu_operators import ctx, dev_linear, same_bytes   # noqa: F401  (ctx: the fixture)

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("n", [1, 2, 47, 64, 65, 255, 256, 257, 1030])
@pytest.mark.parametrize("K,N", [(320, 7), (512, 64), (512, 256)])
def test_gathered_rows_are_checked_whichever_kernel_looks(ctx, n, K, N):
    T, rng = 9, np.random.RandomState(n)
    w = rng.randint(0, 2 ** 32, N * K // 8, dtype=np.uint32)
    s, b = np.full(N * K // 64, 0x3c00, np.uint16), np.full(N * K // 64, 0xbd80, np.uint16)
    x = oracle.bf(rng.standard_normal(T * K).astype(f32))
    lin, dx = dev_linear(ctx, w, s, b, K, N), ctx.upload(x)
    rows = rng.randint(0, T, n).astype(np.int32)
    out = ctx.upload(np.full(n * N, 7, f32))
    for at in sorted({0, n // 2, n - 1}):
        for wrong in (T, -1, 2 ** 31 - 1):
            bad = rows.copy(); bad[at] = wrong
            with pytest.raises(z.ZcError, match="row outside input"):
                ctx.gated_linear(lin, lin, dx, T, n, ctx.upload(bad), out=out)
    ctx.finish()
    assert (out.numpy(f32) == 7).all()
    for _ in range(70):   # (more calls than there are words for the answers)
        ctx.gated_linear(lin, lin, dx, T, n, ctx.upload(rows), out=out)
    host = oracle.make_linear(w, s, b, K, N)
    assert same_bytes(out.numpy(f32), oracle.gated_linear(host, host, x, n, rows))


def test_gathers_of_several_threads_are_answered_one_by_one(ctx):
    """Threads that share a context: every call reads its own answer, refused ones beside accepted ones, short lists and long."""
    K, N, T, calls = 320, 7, 9, 60
    rng = np.random.RandomState(5)
    w = rng.randint(0, 2 ** 32, N * K // 8, dtype=np.uint32)
    s, b = np.full(N * K // 64, 0x3c00, np.uint16), np.full(N * K // 64, 0xbd80, np.uint16)
    x = oracle.bf(rng.standard_normal(T * K).astype(f32))
    lin, dx, host = dev_linear(ctx, w, s, b, K, N), ctx.upload(x), oracle.make_linear(w, s, b, K, N)
    jobs, wrong = [], []
    for n in (1, 5, 256, 257, 5, 64, 300, 1, 33, 5, 257, 2):
        rows = rng.randint(0, T, n).astype(np.int32)
        bad = rows.copy(); bad[n // 2] = T
        jobs.append((n, rows, ctx.upload(rows), ctx.upload(bad), ctx.upload(np.full(n * N, 7, f32))))
    ctx.finish()

    def calls_of(job, refused_first):
        n, rows, good, bad, out = job
        for i in range(calls):
            refuse = (i % 3 == 0) == refused_first
            try:
                ctx.gated_linear(lin, lin, dx, T, n, bad if refuse else good, out=out)
                if refuse:
                    wrong.append((n, i, "accepted"))
            except z.ZcError as error:
                if not refuse or "row outside input" not in str(error):
                    wrong.append((n, i, str(error)))

    threads = [threading.Thread(target=calls_of, args=(job, j % 2 == 0)) for j, job in enumerate(jobs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
    ctx.finish()
    for n, rows, _, _, out in jobs:
        assert same_bytes(out.numpy(f32), oracle.gated_linear(host, host, x, n, rows))
