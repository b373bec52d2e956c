"""Evaluations under stream capture. Nothing can be allocated there, so a captured call needs a phase panel that an
earlier call has built; a graph is replayed several times, with other work between, and each replay checked."""
import ctypes as C

import numpy as np
import pytest

from relativistic_solver_hllc_amd import _native as N
from relativistic_solver_hllc_amd import device as D
from relativistic_solver_hllc_amd import scatter as rs

pytestmark = pytest.mark.gpu


def hip(name, *args):
    """A call of the HIP runtime that the library has loaded."""
    f = getattr(N.lib, name)
    f.restype = C.c_int
    rc = f(*args)
    assert rc == 0, f"{name}: {rc}"


class Graph:
    """What `record` enqueues on a stream, captured and instantiated."""

    def __init__(self, record):
        self.stream, self.graph, self.exec = D.Stream(), C.c_void_p(), C.c_void_p()
        st = C.c_void_p(self.stream.cuda_stream)
        hip("hipStreamBeginCapture", st, C.c_int(1))  # thread-local
        try:
            record(self.stream)
        finally:
            rc = N.lib.hipStreamEndCapture(st, C.byref(self.graph))
        assert rc == 0
        hip("hipGraphInstantiate", C.byref(self.exec), self.graph, None, None, C.c_size_t(0))

    def replay(self):
        hip("hipGraphLaunch", self.exec, C.c_void_p(self.stream.cuda_stream))
        D.synchronize()

    def close(self):
        hip("hipGraphExecDestroy", self.exec)
        hip("hipGraphDestroy", self.graph)


def dirset(m):
    xyz, w, F = rs.fibonacci_directions(m)
    return rs.DirectionSet(xyz, w, F, phase="hg", g=0.6, normalize=True)


def test_panels_of_40_ranges_in_two_layouts_stay(gpu):
    """The panel cache holds 64 ranges. Sizes that take another layout of a range's panel do not count as ranges: after
    40 of them in two layouts each, the first one is still there for a capture, and the graph's results are those of
    an eager call after further calls."""
    m, few, many = 64, 17, 300000
    with dirset(m) as ds:
        d_in, out, ref = (D.DeviceArray((m, many)), D.DeviceArray((m, many)), D.DeviceArray((m, many)))
        N.call("rsh_fill_lognormal_dev", d_in.ptr, m * many, 0.0, 1.0, 7, None)
        ds.scatter_f64(d_in, 1, few, 0, m, ref)
        for k in range(40):
            for n in (few, many):
                ds.scatter_f64(d_in, 1, n, k, k + 1, out)
        D.synchronize()
        g = Graph(lambda st: ds.scatter_f64(d_in, 1, few, 0, m, out, stream=st))
        want = ref.to_host().reshape(-1)[:m * few]
        for _ in range(3):
            out.fill(-1.0)
            ds.scatter_f64(d_in, 1, many, 3, 4, ref)
            D.synchronize()
            g.replay()
            assert np.array_equal(out.to_host().reshape(-1)[:m * few], want)
        g.close()
        for a in (d_in, out, ref):
            a.free()


@pytest.mark.parametrize("faces", [1, 4])
def test_captured_f64_kernel_does_not_depend_on_the_warm_up_size(gpu, faces):
    """After a call of any one size, a captured call runs its own route if that panel is there and else the plan of
    fewest passes with eight waves (what every size ran before the routes by size); never another size's plan. The
    graph's results are the eager call's."""
    m, sizes = 400, (381, 2957, 24577, 200000)
    d_in, out, ref = (D.DeviceArray((m, sizes[-1], faces)), D.DeviceArray((m, sizes[-1])), D.DeviceArray((m, sizes[-1])))
    N.call("rsh_fill_lognormal_dev", d_in.ptr, d_in.size, 0.0, 1.0, 7, None)
    with dirset(m) as ds:
        eager = {n: ds.scatter_f64_route(faces, n, 0, m) for n in sizes}
    assert eager[381][0] == "register" and eager[200000][:3] == ("panel", 25, 1)
    assert len({r[:3] for r in eager.values()}) >= 3
    fewest = ("panel", 25, 1, rs.tuned_tile_f64(m)[0])  # eight waves unless another test has tuned the class
    for warm in sizes:
        for n in sizes:
            with dirset(m) as ds:
                ds.scatter_f64(d_in, faces, warm, 0, m, out)
                D.synchronize()
                seen = []

                def record(st):
                    seen.append(ds.scatter_f64_route(faces, n, 0, m, stream=st))
                    ds.scatter_f64(d_in, faces, n, 0, m, out, stream=st)

                g = Graph(record)
                there = eager[n][:3] in (eager[warm][:3], fewest[:3])
                assert seen == [eager[n] if there else fewest], (warm, n)
                ds.scatter_f64(d_in, faces, n, 0, m, ref)
                D.synchronize()
                want = ref.to_host().reshape(-1)[:m * n]
                for _ in range(2):
                    out.fill(-1.0)
                    D.synchronize()
                    g.replay()
                    assert np.array_equal(out.to_host().reshape(-1)[:m * n], want), (warm, n)
                g.close()
    for a in (d_in, out, ref):
        a.free()


@pytest.mark.parametrize("m,few,many", [(800, 3000, 30000), (820, 1000, 5000)])
def test_captured_split_kernel_does_not_depend_on_the_warm_up_size(gpu, m, few, many):
    """Where the size decides between the resident and the streaming kernel: after a call of either size a captured large
    call runs the streaming kernel, and a captured small one the resident kernel if its panel is there. The graph's
    results are the eager call's."""
    form = "bf16x2"
    d_in, out, ref = (D.DeviceArray((m, many)) for _ in range(3))
    N.call("rsh_fill_lognormal_dev", d_in.ptr, d_in.size, 0.0, 1.0, 7, None)
    state, scale = {}, {}
    for n in (few, many):
        sb, cb = rs.split_sizes(form, 1, n, m)
        state[n], scale[n] = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_dev(form, d_in, 1, n, m, state[n], scale[n])
    for warm in (few, many):
        for n in (few, many):
            with dirset(m) as ds:
                ds.scatter_split(form, state[warm], scale[warm], 1, warm, 0, m, out)
                D.synchronize()
                seen = []

                def record(st):
                    seen.append(ds.scatter_split_route(form, 1, n, 0, m, stream=st)[0])
                    ds.scatter_split(form, state[n], scale[n], 1, n, 0, m, out, stream=st)

                g = Graph(record)
                assert seen == ["resident" if n == warm == few else "streaming"], (warm, n)
                ds.scatter_split(form, state[n], scale[n], 1, n, 0, m, ref)
                D.synchronize()
                want = ref.to_host().reshape(-1)[:m * n]
                for _ in range(2):
                    out.fill(-1.0)
                    D.synchronize()
                    g.replay()
                    assert np.array_equal(out.to_host().reshape(-1)[:m * n], want), (warm, n)
                g.close()
    for a in (d_in, out, ref, *state.values(), *scale.values()):
        a.free()
