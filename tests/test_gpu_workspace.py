"""The adjoint's kept workspace and reverse lists: calls that follow one
another with other checkpoint spacings, other sizes and other solvers of the
same context give the gradients that each gives in a context of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def gradient(ctx, level, seed, ckpt, pair=None):
    import hom3_amd as H
    from hom3_amd import adjoint as A, cases
    if pair is None:
        _, c, h, _ = cases.channel_cht(H, level=level, seed=seed, ctx=ctx)
        pair = (c, h, A.Snapshot(c, h))
    c, h, snap = pair
    snap.restore()
    _, dts = A.cht_objective(c, h, 0.01, 7)
    snap.restore()
    J, g, _, _ = A.cht_adjoint(c, h, 0.01, dts, ckpt)
    return pair, J, g


def test_interleaved_calls_share_the_workspace():
    import hom3_amd as H
    ref = {k: gradient(H.Context(0), *k)[1:] for k in ((4, 1, 0), (5, 2, 0))}
    ctx = H.Context(0)
    pairs = {}
    for level, seed, ckpt in ((4, 1, 0), (5, 2, 3), (4, 1, -2), (5, 2, 0), (4, 1, 2), (5, 2, -3)):
        pairs[level], J, g = gradient(ctx, level, seed, ckpt, pairs.get(level))
        J0, g0 = ref[(level, seed, 0)]
        assert J == J0
        np.testing.assert_array_equal(g, g0)


def test_memory_kept_between_gradients_is_given_back():
    """release_memory frees what the gradient left on the device, and the next
    gradient has the same bits."""
    import torch
    import hom3_amd as H

    def used():
        ctx.synchronize()
        free, total = torch.cuda.mem_get_info(0)
        return total - free

    ctx = H.Context(0)
    pair, J0, g0 = gradient(ctx, 5, 3, 0)
    kept = used()
    ctx.release_memory()
    released = used()
    # the workspace alone is one chunk of 64 MiB at least
    assert kept - released >= 64 << 20, (kept, released)
    _, J1, g1 = gradient(ctx, 5, 3, 0, pair)
    assert J0 == J1
    np.testing.assert_array_equal(g0, g1)
    assert used() - released >= 64 << 20
    ctx.release_memory()
    ctx.release_memory()
    # (the runtime's own allocations may grow by less than a chunk)
    assert used() - released < 16 << 20
