"""The staged step of a pinned context (one native call: upload, step and
read-back in pieces, host copies beside the link) against the same step of a
context without staging: the same kernels on the same cells, so every output
is bitwise the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGE = 1 << 20                  # bytes of an upload's first piece
DIE = (0.0, 0.0, 1024.0, 1024.0)


def cells(n, dtype, seed):
    rng = np.random.default_rng(seed)
    sx, sy = rng.uniform(1, 9, n), np.full(n, 6.0)
    return [a.astype(dtype) for a in
            (rng.uniform(0, 1, n) * (1024 - sx), rng.uniform(0, 1, n) * (1024 - sy), sx, sy)]


def same(a, b):
    assert list(a) == list(b)
    for k in a:
        assert a[k].shape == b[k].shape and a[k].dtype == b[k].dtype, k
        assert np.array_equal(a[k], b[k]), k


# one cell and none; either side of two pieces' copies (256 KiB each), of the
# split of the first and the last array (two edges), and arrays and maps of
# more than one 8 MiB piece
@pytest.mark.parametrize("n,grid,dtype", [
    (0, 64, np.float32), (1, 64, np.float32), (131071, 128, np.float32),
    (2 * EDGE // 4 - 1, 128, np.float32), (2 * EDGE // 4, 128, np.float32),
    (2 * EDGE // 8 + 1, 128, np.float64), ((8 << 20) // 4 + 3, 2048, np.float32)])
def test_staged_step_is_the_plain_step(n, grid, dtype):
    import dpep
    with dpep.Context(grid, grid, max(n, 5), *DIE, dtype=dtype) as plain, \
            dpep.Context(grid, grid, max(n, 5), *DIE, dtype=dtype, pinned=True) as ctx:
        a, b = cells(n, dtype, 1), cells(n, dtype, 2)
        first = ctx.step(*a)
        kept = {k: v.copy() for k, v in first.items()}
        same(first, plain.step(*a))
        # other positions, sizes kept; forces alone, then one field (both come)
        ref = plain.step(b[0], b[1])
        got = ctx.step(b[0], b[1], outputs=("grad_x", "grad_y"))
        same(got, {k: ref[k] for k in ("grad_x", "grad_y")})
        same(ctx.step(b[0], b[1], outputs=iter(["field_y"])),
             {k: ref[k] for k in ("field_x", "field_y")})
        same(first, kept)                        # copies: later steps leave them
        # cells already in the staging buffers, outputs left in theirs
        host = ctx.host_cells()
        same(ctx.step(host["px"][:n], host["py"][:n], copy=False), ref)
        t = ctx.timings()
        assert t["h2d"] >= 0 and t["d2h_den"] > 0 and t["download"] > 0


def test_staged_step_with_overlapping_or_refused_arguments():
    import dpep
    n = 4096
    with dpep.Context(64, 64, n, *DIE) as plain, \
            dpep.Context(64, 64, n, *DIE, pinned=True, potential=False) as ctx:
        a = cells(n, np.float32, 5)
        with pytest.raises(RuntimeError):
            ctx.step(a[0], a[1])                 # no sizes are resident
        ctx.step(*a)
        host = ctx.host_cells()
        names = ("grad_x", "grad_y")
        # a shifted view of a staging buffer as input
        want = plain.step(a[0][1:], a[1][:-1], a[2][1:], a[3][1:], outputs=names)
        same(ctx.step(host["px"][1:], a[1][:-1], a[2][1:], a[3][1:], outputs=names), want)
        for bad in (("potential",), ("density", "nothing")):
            with pytest.raises((RuntimeError, ValueError)):
                ctx.step(*a, outputs=bad)
        with pytest.raises(ValueError):
            ctx.step(*cells(n + 1, np.float32, 6))
        with pytest.raises(ValueError):
            ctx.step(a[0], a[1], a[2])
        same(ctx.step(*a, outputs=names), plain.step(*a, outputs=names))
