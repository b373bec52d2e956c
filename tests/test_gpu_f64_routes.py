"""The FP64 integral over the sizes between which its route changes: the register-fed kernel (few cells) with
every number of row blocks per wave, and the LDS-panel kernel in more, shorter passes. Every route adds a result's
products in the same order, so each must equal the LDS-panel kernel with a given tile bit for bit; against the
oracle the bound is that kernel's own (1e-12 relative)."""
import numpy as np
import pytest

from oracle import orc
from relativistic_solver_hllc_amd import _native as N
from relativistic_solver_hllc_amd import device as D
from relativistic_solver_hllc_amd import scatter as rs

pytestmark = pytest.mark.gpu

# (cells, directions, faces, k0, k1): edges of the 16-cell tile, the 4- and 8-direction steps and the 16-row block;
# then larger sizes, and ranges of rows
SIZES = [(1, 1, 4, 0, 1), (15, 3, 4, 0, 3), (16, 4, 1, 0, 4), (17, 8, 4, 0, 8), (63, 9, 1, 0, 9), (65, 16, 4, 0, 16),
         (66, 17, 4, 0, 17), (381, 327, 4, 0, 327), (381, 327, 1, 5, 22), (1003, 302, 4, 0, 302), (2958, 200, 4, 0, 200),
         (2959, 302, 4, 0, 302), (2957, 400, 1, 0, 400), (5001, 302, 4, 0, 302), (5000, 400, 4, 0, 400),
         (9999, 129, 1, 0, 129), (24577, 113, 4, 0, 113), (24577, 302, 1, 7, 301)]


def evaluate(ds, d_in, faces, n, k0, k1, **kw):
    out = D.DeviceArray((k1 - k0, n + 5))
    out.fill(-1.0)
    ds.scatter_f64(d_in, faces, n, k0, k1, out, ld=n + 5, **kw)
    D.synchronize()
    got = out.to_host()
    out.free()
    assert np.all(got[:, n:] == -1.0)  # nothing past the last cell
    return got[:, :n]


@pytest.mark.parametrize("n,m,faces,k0,k1", SIZES)
def test_route_equals_lds_panel_kernel(gpu, n, m, faces, k0, k1):
    rng = np.random.default_rng(n + m)
    illum = rng.lognormal(0.0, 1.5, size=(m, n, faces))
    illum[m // 2, n // 2, :] = np.inf  # stays in its own cell, also where directions are padded
    xyz, w, F = rs.fibonacci_directions(m)
    d_in = D.DeviceArray.from_host(illum if faces == 4 else illum[..., 0])
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.6, normalize=True) as ds:
        got = evaluate(ds, d_in, faces, n, k0, k1)
        want = evaluate(ds, d_in, faces, n, k0, k1, kernel="mfma", tile=(8, 2))
    d_in.free()
    assert np.array_equal(got, want, equal_nan=True)
    cells = [c for c in {0, n - 1, n // 3, n // 2 + 1} if 0 <= c < n and c != n // 2]
    if cells:
        P = orc.phase_matrix(xyz, w, F, 1, 0.6, True)
        ref = orc.scatter_matrix(np.ascontiguousarray(illum[:, cells]), P)[k0:k1]
        assert np.max(np.abs(got[:, cells] - ref) / ref) < 1e-12


def test_tuned_tile_is_for_the_plan_that_was_timed(gpu):
    """rsh_autotune_f64 at 200 directions times thirteen row blocks in one pass. 400 directions of some sizes run as two
    passes of thirteen, in workgroups of eight waves or of four: their route stays, whatever tile the class has. A size
    of the class in one pass takes the tile."""
    def dirset(m):
        xyz, w, F = rs.fibonacci_directions(m)
        return rs.DirectionSet(xyz, w, F)

    with dirset(400) as two, dirset(200) as one:
        def routes():
            return [two.scatter_f64_route(4, n, 0, 400) for n in (14001, 17001)]

        assert routes() == [("panel", 13, 2, 8), ("panel", 13, 2, 4)]
        tile, _ = rs.autotune_f64(200, faces=4, n_cells=4096)
        assert rs.tuned_tile_f64(200) == tile
        assert routes() == [("panel", 13, 2, 8), ("panel", 13, 2, 4)]
        assert one.scatter_f64_route(4, 300000, 0, 200) == ("panel", 13, 1, tile[0])


# One size per kind of route: (cells, directions, faces): row blocks and groups of the register-fed kernel, or row
# blocks per pass, passes and waves of the LDS-panel kernel
ROUTES = {(15, 400, 4): ("register", 1, 25, 0), (13521, 27, 4): ("register", 2, 1, 0),
          (2958, 200, 4): ("register", 3, 5, 0), (2959, 302, 4): ("register", 4, 5, 0),
          (2957, 400, 1): ("register", 5, 5, 0), (5001, 257, 4): ("register", 6, 3, 0),
          (14571, 109, 1): ("register", 7, 1, 0), (5001, 350, 4): ("register", 8, 3, 0),
          (8097, 281, 4): ("register", 10, 2, 0), (40001, 302, 4): ("panel", 19, 1, 4),
          (14001, 400, 4): ("panel", 13, 2, 8), (40001, 400, 4): ("panel", 13, 2, 4),
          (33001, 400, 1): ("panel", 5, 5, 4), (150001, 113, 4): ("panel", 8, 1, 8)}


@pytest.mark.parametrize("size", ROUTES)
def test_every_kind_of_route_equals_the_lds_panel_kernel(gpu, size):
    """The route is the one meant (on 256 CUs; a class that another test has tuned takes its tile's waves), and its
    results are the given tile's bit for bit."""
    n, m, faces = size
    rng = np.random.default_rng(n + m)
    illum = rng.lognormal(0.0, 1.5, size=(m, n) if faces == 1 else (m, n, faces))
    xyz, w, F = rs.fibonacci_directions(m)
    d_in = D.DeviceArray.from_host(illum)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.6, normalize=True) as ds:
        route = ds.scatter_f64_route(faces, n, 0, m)
        kernel, blocks, passes, waves = ROUTES[size]
        if kernel == "panel" and passes == 1 and rs.tuned_tile_f64(m) != (8, 2):
            waves = rs.tuned_tile_f64(m)[0]
        assert route == (kernel, blocks, passes, waves)
        got = evaluate(ds, d_in, faces, n, 0, m)
        want = evaluate(ds, d_in, faces, n, 0, m, kernel="mfma", tile=(8, 2))
    d_in.free()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("faces,m,rows,n", [(4, 22, 22, 42851), (1, 64, 64, 80001), (4, 48, 48, 80001), (4, 302, 61, 40001),
                                            (4, 100, 100, 80003), (1, 200, 200, 250003)])
def test_every_kind_of_store_gives_the_same_results(gpu, faces, m, rows, n):
    """Ragged rows are stored plainly or past the caches by the sizes of faces and results (under 60 MB, between, results
    under an eighth, around the 256 MB cache, far beyond); rows at 64 and 128 bytes past the caches: the same bits, and
    nothing past a row's cells."""
    xyz, w, F = rs.fibonacci_directions(m)
    strides = (n, (n + 7) // 8 * 8, (n + 15) // 16 * 16 + 16)
    d_in, out = D.DeviceArray((m, n, faces)), D.DeviceArray((rows, strides[-1]))
    N.call("rsh_fill_lognormal_dev", d_in.ptr, d_in.size, 0.0, 1.0, 5, None)
    first = None
    with rs.DirectionSet(xyz, w, F) as ds:
        for ld in strides:
            out.fill(-1.0)
            ds.scatter_f64(d_in, faces, n, 0, rows, out, ld=ld)
            D.synchronize()
            got = out.to_host().reshape(-1)[:rows * ld].reshape(rows, ld)
            first = got[:, :n].copy() if first is None else first
            assert np.array_equal(got[:, :n], first)
            assert np.all(got[:, n:] == -1.0)
    for a in (d_in, out):
        a.free()
