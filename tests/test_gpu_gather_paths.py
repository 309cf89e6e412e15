"""GPU: the direct gather (few cells on small maps: one thread per cell reads
the field bins) and the gather per strip, on either side of the line between
them (cells times bytes per value: 1 MiB up to 2^18 bins, 448 KiB up to 2^20,
none beyond), with cells of one to 40 columns and tall ones, on a moving
placement, against the float64 oracle (the relative error of a field is ~4e-7
at float32 and ~6e-14 at float64, and a force sums ~10 of its values)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,M,N,dtype", [
    (262144, 512, 512, np.float32), (262145, 512, 512, np.float32),
    (131072, 256, 1024, np.float64), (131073, 256, 1024, np.float64),
    (114688, 1024, 1024, np.float32), (114689, 1024, 1024, np.float32),
    (255, 8, 8, np.float32), (257, 8, 32, np.float64), (3000, 4096, 64, np.float32)])
def test_gather_paths_at_their_line(oracle, cells, M, N, dtype):
    import dpep
    rng = np.random.default_rng(cells)
    die = (-50.0, 20.0, 4046.0, 4116.0)
    bx, by = 4096.0 / M, 4096.0 / N
    sx = rng.uniform(0.2, 2.0, cells) * bx
    sy = rng.uniform(0.2, 2.0, cells) * by
    wide, tall = rng.random(cells) < 0.01, rng.random(cells) < 0.003
    sy[wide] = np.minimum(rng.uniform(2, 40, wide.sum()) * by, 2000.0)
    sx[tall] = np.minimum(rng.uniform(3, 30, tall.sum()) * bx, 2000.0)
    with dpep.Context(M, N, cells, *die, dtype=dtype) as ctx:
        for step in range(2):
            # some stretched corners past each edge of the die
            px = rng.uniform(die[0] - 0.2 * bx, die[2] - 0.5 * sx)
            py = rng.uniform(die[1] - 0.2 * by, die[3] - 0.5 * sy)
            c = [a.astype(dtype) for a in (px, py, sx, sy)]
            got = ctx.step(*c)
            ref = oracle.step(*c, M, N, *die)
            tol = 1e-5 if dtype == np.float32 else 1e-11
            for k in ("density", "field_x", "field_y", "grad_x", "grad_y"):
                err = np.linalg.norm(got[k].astype(np.float64) - ref[k]) / np.linalg.norm(ref[k])
                assert err < tol, (k, step, err)
