"""GPU parity of the split-precision forms against the FP64 oracle.

The forms differ in how many significand bits their operands keep:
  bf16x2  hi+lo BF16   ~16 bits  -> per-element representation error <= 2^-16
  fp16x2  hi+lo FP16   ~22 bits  (power-of-two scaled per cell and per row)
  bf16x3  hi+mid+lo BF16 ~24 bits
all with FP32 MFMA accumulation (main and cross-term accumulators, combined in
FP64). Tolerances written here, max / mean relative error vs the FP64 oracle:
  fp16x2, bf16x3 : max <= 1e-6
  bf16x2         : max <= 3e-5, mean <= 3e-6  (16-bit operands cannot reach 1e-6 per result;
                   the measured errors are printed and recorded by bench.py)
"""
import numpy as np
import pytest

from oracle import orc
from relativistic_solver_hllc_amd import _native as N
from relativistic_solver_hllc_amd import device as D
from relativistic_solver_hllc_amd import scatter as rs

pytestmark = pytest.mark.gpu

TOL = {"fp16x2": (1e-6, 1e-6), "bf16x3": (1e-6, 1e-6), "bf16x2": (3e-5, 3e-6)}


def errs(got, ref):
    r = np.abs(got - ref) / np.abs(ref)
    return float(r.max()), float(r.mean())


def run_split(ds, form, illum, faces, k0, k1, out_f32=False, ld=None):
    m, n = illum.shape[0], illum.shape[1]
    d_illum = D.DeviceArray.from_host(np.ascontiguousarray(illum, dtype=np.float64))
    sb, cb = rs.split_sizes(form, faces, n, m)
    state = D.DeviceArray((sb,), np.uint8)
    scale = D.DeviceArray((max(cb // 4, 1),), np.float32)
    rs.pack_split_dev(form, d_illum, faces, n, m, state, scale)
    ld = n if ld is None else ld
    out = D.DeviceArray((max(k1 - k0, 1), ld), np.float32 if out_f32 else np.float64)
    ds.scatter_split(form, state, scale, faces, n, k0, k1, out, ld=ld, out_f32=out_f32)
    D.synchronize()
    res = out.to_host()[: k1 - k0, :n].astype(np.float64)
    for a in (d_illum, state, scale, out):
        a.free()
    return res


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
def test_hg08_reduced_n(gpu, form):
    """The HG workload's shape at reduced N: HG g = 0.8, FP64 row normalisation, log-normal(0, 1.5) faces."""
    n, m = 4096, 400
    rng = np.random.default_rng(0x5EED + 3)
    illum = rng.lognormal(0.0, 1.5, size=(m, n, 4))
    xyz, w, F = rs.fibonacci_directions(m)
    ref = orc.scatter_matrix(illum, orc.phase_matrix(xyz, w, F, 1, 0.8, True), threads=16)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.8, normalize=True) as ds:
        got = run_split(ds, form, illum, 4, 0, m)
    mx, mean = errs(got, ref)
    print(f"{form}: max rel err {mx:.3e}, mean {mean:.3e}")
    assert mx <= TOL[form][0] and mean <= TOL[form][1]


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
@pytest.mark.parametrize("n,m,k0,k1,faces", [(1, 1, 0, 1, 4), (37, 26, 3, 21, 4), (1000, 130, 17, 129, 1),
                                             (513, 800, 0, 800, 4), (300, 33, 0, 33, 1)])
def test_split_ragged_thomson(gpu, form, n, m, k0, k1, faces):
    rng = np.random.default_rng(n + 7 * m)
    illum = rng.lognormal(0.0, 1.0, size=(m, n, faces))
    xyz, w, F = rs.fibonacci_directions(m)
    ref = orc.scatter_reference(illum, xyz, w, F, k_disp=k0, k_count=k1 - k0, threads=16)
    with rs.DirectionSet(xyz, w, F) as ds:
        got = run_split(ds, form, illum, faces, k0, k1, ld=n + 5)
    mx, mean = errs(got, ref)
    assert mx <= TOL[form][0] and mean <= TOL[form][1], (mx, mean)


def test_split_fp32_output(gpu):
    n, m = 2000, 200
    rng = np.random.default_rng(3)
    illum = rng.lognormal(0.0, 1.0, size=(m, n, 4))
    xyz, w, F = rs.fibonacci_directions(m)
    ref = orc.scatter_reference(illum, xyz, w, F, threads=16)
    with rs.DirectionSet(xyz, w, F) as ds:
        got = run_split(ds, "fp16x2", illum, 4, 0, m, out_f32=True)
    mx, _ = errs(got, ref)
    assert mx <= 1e-6


def test_split_isotropic_normalised(gpu):
    """I = c everywhere with row-normalised P: S = c up to the split error."""
    n, m = 1000, 400
    illum = np.full((m, n, 4), 3.25)
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.6, normalize=True) as ds:
        for form in ("bf16x2", "fp16x2", "bf16x3"):
            got = run_split(ds, form, illum, 4, 0, m)
            assert np.max(np.abs(got - 3.25) / 3.25) <= TOL[form][0]


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
def test_split_tiles_bit_identical(gpu, form):
    """One wave per tile (waves=4) or two waves splitting the rows (waves=8): same sums, same bits."""
    n, m = 3000, 400
    rng = np.random.default_rng(31)
    illum = rng.lognormal(0.0, 1.5, size=(m, n, 4))
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.8, normalize=True) as ds:
        d_illum = D.DeviceArray.from_host(illum)
        sb, cb = rs.split_sizes(form, 4, n, m)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_dev(form, d_illum, 4, n, m, state, scale)
        outs = []
        for waves in (4, 8):
            out = D.DeviceArray((m, n))
            ds.scatter_split(form, state, scale, 4, n, 0, m, out, waves=waves)
            D.synchronize()
            outs.append(out.to_host())
            out.free()
        for a in (d_illum, state, scale):
            a.free()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
@pytest.mark.parametrize("n,m,k0,k1", [(70001, 400, 0, 400), (5000, 200, 0, 200), (3000, 400, 37, 301),
                                       (17, 26, 0, 26), (9000, 800, 0, 800)])
def test_resident_panel_kernel_bit_identical(gpu, form, n, m, k0, k1):
    """Cell-level state: the resident-panel kernel (waves=1, the default for faces = 1)
    and both streaming kernels sum the same products in the same order."""
    rng = np.random.default_rng(n + m + k0)
    cell = rng.lognormal(0.0, 1.5, size=(m, n, 1))
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.8, normalize=True) as ds:
        d_cell = D.DeviceArray.from_host(cell)
        sb, cb = rs.split_sizes(form, 1, n, m)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_dev(form, d_cell, 1, n, m, state, scale)
        outs = {}
        for waves in (1, 0, 4, 8):
            out = D.DeviceArray((k1 - k0, n + 3))
            out.fill(-1.0)
            ds.scatter_split(form, state, scale, 1, n, k0, k1, out, ld=n + 3, waves=waves)
            D.synchronize()
            outs[waves] = out.to_host()
            out.free()
        for a in (d_cell, state, scale):
            a.free()
    ref = outs[4]
    assert np.all(ref[:, n:] == -1.0)  # padding columns untouched
    for wv, o in outs.items():
        assert np.array_equal(o, ref), wv
    if m <= 400 and n <= 5000:
        P = orc.phase_matrix(xyz, w, F, 1, 0.8, True, k0, k1)
        exact = orc.scatter_matrix(cell, P, threads=16)
        mx, mean = errs(ref[:, :n], exact)
        assert mx <= TOL[form][0] and mean <= TOL[form][1], (mx, mean)


@pytest.mark.parametrize("n", [20480, 20481])
def test_automatic_choice_at_800_directions(gpu, n):
    """17 row groups per XCD: the resident kernel up to 10 chunks of 256 cells for each of its 8 sets, the streaming
    one beyond. Equal bits on both sides of the line."""
    m = 800
    cell = np.resize(np.random.default_rng(n).lognormal(0.0, 1.5, size=1_000_003), (m, n, 1))
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F) as ds:
        d_cell = D.DeviceArray.from_host(cell)
        sb, cb = rs.split_sizes("fp16x2", 1, n, m)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_dev("fp16x2", d_cell, 1, n, m, state, scale)
        outs = []
        for waves in (0, 8):
            out = D.DeviceArray((m, n))
            ds.scatter_split("fp16x2", state, scale, 1, n, 0, m, out, waves=waves)
            D.synchronize()
            outs.append(out.to_host())
            out.free()
        for a in (d_cell, state, scale):
            a.free()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("three", [False, True])
@pytest.mark.parametrize("steps", range(1, 26))
def test_resident_workgroup_forms_bit_identical(gpu, steps, three):
    """Every K-step count's resident plan, with either count of row blocks, in the workgroup forms: one tile per wave
    up to 1 (3 for three parts) rounds of 128 cells per set, then 2 or 4 tiles per wave; FP64 rows with and without
    whole 128-byte lines. The streaming kernel sums the same products in the same order: equal bits."""
    form = "bf16x3" if three else ("bf16x2", "fp16x2")[steps % 2]
    m = 32 * steps - (19 if steps % 3 == 0 else 3)
    need, fit = (m + 15) // 16, min(5, 163840 // (steps * 2048 + 64))
    groups = -(-need // fit)
    rbw = -(-need // groups)
    slots = 8 * (32 // -(-need // rbw))  # sets of the chip's 8 x 32 CUs
    sizes = [3 * 128 * slots, 3 * 128 * slots + 1] if three else [128 * slots, 1024 * slots + 16]
    n_max = max(sizes)
    cell = np.resize(np.random.default_rng(steps).lognormal(0.0, 1.5, size=1_000_003), (m, n_max, 1))
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.8, normalize=True) as ds:
        for n in sizes:
            d_cell = D.DeviceArray.from_host(np.ascontiguousarray(cell[:, :n]))
            sb, cb = rs.split_sizes(form, 1, n, m)
            state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
            rs.pack_split_dev(form, d_cell, 1, n, m, state, scale)
            for f32, ld in ((False, n), (True, n + 3)):
                outs = []
                for waves in (1, 8):
                    out = D.DeviceArray.from_host(np.full((m, ld), -1.0, np.float32 if f32 else np.float64))
                    ds.scatter_split(form, state, scale, 1, n, 0, m, out, ld=ld, out_f32=f32, waves=waves)
                    D.synchronize()
                    outs.append(out.to_host())
                    out.free()
                assert np.array_equal(outs[0], outs[1]), (n, f32)
                assert np.all(outs[0][:, n:] == -1.0)
            for a in (d_cell, state, scale):
                a.free()


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
def test_face_averaged_pack_vs_oracle(gpu, form):
    """rsh_pack_split_avg_dev: 4-face input reduced to a cell-level state in the pack;
    the resident-panel kernel on it matches the FP64 oracle on the 4-face input."""
    n, m = 4096, 400
    rng = np.random.default_rng(0x5EED + 33)
    illum = rng.lognormal(0.0, 1.5, size=(m, n, 4))
    xyz, w, F = rs.fibonacci_directions(m)
    ref = orc.scatter_matrix(illum, orc.phase_matrix(xyz, w, F, 1, 0.8, True), threads=16)
    with rs.DirectionSet(xyz, w, F, phase="hg", g=0.8, normalize=True) as ds:
        d_illum = D.DeviceArray.from_host(illum)
        sb, cb = rs.split_sizes(form, 1, n, m)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_avg_dev(form, d_illum, n, m, state, scale)
        out = D.DeviceArray((m, n))
        ds.scatter_split(form, state, scale, 1, n, 0, m, out)
        D.synchronize()
        got = out.to_host()
        for a in (d_illum, state, scale, out):
            a.free()
    mx, mean = errs(got, ref)
    print(f"{form} face-averaged pack: max rel err {mx:.3e}, mean {mean:.3e}")
    assert mx <= TOL[form][0] and mean <= TOL[form][1]


@pytest.mark.parametrize("n,m", [(1, 16), (17, 17), (32, 128), (33, 129), (257, 257), (4099, 512), (4100, 513),
                                 (515, 800), (64, 896), (65, 897), (131072, 20), (131073, 20)])
def test_face_averaged_pack_exact(gpu, n, m):
    """Every face-averaged pack form (1, 2, 4 and 7 slots of 128 directions, LDS past 896, 64-cell groups for many
    cells with rows inside a line) against the packing computed here: averages in FP64 in the same order, one power
    of two per cell, two FP16 parts with round-to-nearest. Equal bits."""
    rng = np.random.default_rng(n + m)
    illum = rng.lognormal(0.0, 3.0, size=(m, n, 4)) * rng.choice([-1.0, 1.0], size=(m, n, 4))
    d_illum = D.DeviceArray.from_host(illum)
    sb, cb = rs.split_sizes("fp16x2", 1, n, m)
    state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
    rs.pack_split_avg_dev("fp16x2", d_illum, n, m, state, scale)
    D.synchronize()
    got, inv = state.to_host().view(np.float16), scale.to_host()[:n].astype(np.float64)
    for a in (d_illum, state, scale):
        a.free()
    exponent = np.frexp(np.abs(illum).max(axis=(0, 2)))[1]
    assert np.unique(np.ldexp(inv, -exponent)).size == 1  # the same power of two above every cell's maximum
    avg = (((illum[..., 0] + illum[..., 1]) + illum[..., 2]) + illum[..., 3]) * 0.25
    steps, tiles = -(-m // 32), -(-n // 16)
    x64 = np.zeros((steps * 32, tiles * 16))
    x64[:m, :n] = avg / inv
    x = x64.astype(np.float32)
    hi = x64.astype(np.float16)  # FP64 to FP16 in one rounding
    lo = (x - hi.astype(np.float32)).astype(np.float16)
    # [tile][K-step][part][row group of 8][cell of 16][8]
    want = np.stack([hi, lo]).reshape(2, steps, 4, 8, tiles, 16).transpose(4, 1, 0, 2, 5, 3)
    assert np.array_equal(got[:want.size].reshape(want.shape).view(np.uint16), want.astype(np.float16).view(np.uint16))


def test_resident_kernel_rejects_face_state(gpu):
    xyz, w, F = rs.fibonacci_directions(26)
    with rs.DirectionSet(xyz, w, F) as ds:
        sb, cb = rs.split_sizes("bf16x2", 4, 64, 26)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        out = D.DeviceArray((26, 64))
        with pytest.raises(RuntimeError, match="resident-panel"):
            ds.scatter_split("bf16x2", state, scale, 4, 64, 0, 26, out, waves=1)
        for a in (state, scale, out):
            a.free()


def _bf16_rne(x):
    """float32 -> nearest bfloat16 (ties to even), returned as float32 values."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return r.astype(np.uint32).view(np.float32)


def _part_values(bits, form):
    """16-bit part patterns -> their float32 values."""
    if form == "fp16x2":
        return bits.view(np.float16).astype(np.float32)
    return (bits.astype(np.uint32) << 16).view(np.float32)


def _nearest(r, form):
    """The value of the part format nearest to r (ties to even)."""
    return r.astype(np.float16).astype(np.float32) if form == "fp16x2" else _bf16_rne(r)


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
@pytest.mark.parametrize("faces", [4, 1])
def test_cell_pack_matches_layout_definition(gpu, form, faces):
    """The one-pass cell-level pack against a numpy restatement of its definition:
    cell scale 2^-e, e = 11 - ilogb(max_{j,f} |I[j][c][f]|); value (((f0 + f1) + f2) + f3) / 4
    (faces = 4) or I[j][c] (faces = 1), times 2^e, rounded to FP32, split into parts that
    each round what is left to the 16-bit format; stored MFMA-native: the 16-byte vector
    ((tile * steps + s) * parts + part) * 64 + lane holds cells 16 tile + lane % 16,
    directions 32 s + 8 (lane / 16) + e. Ragged cells and directions pad with zeros.
    The device's float -> 16-bit conversions may break an exact tie either way
    (the split stays exact: each remainder is computed in FP32), so a part must
    equal the round-to-nearest-even value or lie at the same distance from the
    remainder."""
    n, m = 1000, 200            # 62.5 cell tiles, 6.25 K-steps
    rng = np.random.default_rng(31 + faces)
    illum = rng.lognormal(0.0, 1.5, size=(m, n, faces))
    illum[:, 17, :] *= 2.0 ** -40      # a cell far from the others' magnitude
    d_illum = D.DeviceArray.from_host(illum)
    sb, cb = rs.split_sizes(form, 1, n, m)
    state = D.DeviceArray((sb,), np.uint8)
    scale = D.DeviceArray((cb // 4,), np.float32)
    if faces == 4:
        rs.pack_split_avg_dev(form, d_illum, n, m, state, scale)
    else:
        rs.pack_split_dev(form, d_illum, 1, n, m, state, scale)
    D.synchronize()
    got_state, got_scale = state.to_host(), scale.to_host()
    for a in (d_illum, state, scale):
        a.free()
    mx = np.max(np.abs(illum), axis=(0, 2))
    e = 11 - (np.frexp(mx)[1] - 1)
    assert np.array_equal(got_scale, np.ldexp(np.float32(1.0), -e).astype(np.float32))
    v = (((illum[..., 0] + illum[..., 1]) + illum[..., 2]) + illum[..., 3]) * 0.25 if faces == 4 else illum[..., 0]
    x = (v * np.ldexp(1.0, e)[None, :]).astype(np.float32)          # [m][n]
    steps, tiles = (m + 31) // 32, (n + 15) // 16
    xp = np.zeros((steps * 32, tiles * 16), np.float32)
    xp[:m, :n] = x
    nt = 3 if form == "bf16x3" else 2
    got = got_state.view(np.uint16).reshape(tiles, steps, nt, 64, 8)
    # [tile][s][part][lane = 16 g + c][e] -> [part][direction 32 s + 8 g + e][cell 16 tile + c]
    vals = got.reshape(tiles, steps, nt, 4, 16, 8).transpose(2, 1, 3, 5, 0, 4).reshape(nt, steps * 32, tiles * 16)
    # Each part is a nearest value of its format to what the parts before it left
    # (the device's conversion may break exact ties either way); what is left after
    # each part is computed exactly in FP32, as the kernel does.
    r = xp.copy()
    for t in range(nt):
        p = _part_values(vals[t], form)
        q = _nearest(r, form)
        tie = np.abs(r.astype(np.float64) - p) == np.abs(r.astype(np.float64) - q)
        bad = np.argwhere(~((p == q) | tie))
        if len(bad):
            j, c = bad[0]
            raise AssertionError(f"part {t}: {len(bad)} of {p.size} parts are not a nearest value, first at "
                                 f"(dir {j}, cell {c}): remainder {r[j, c]!r}, got {p[j, c]!r}, nearest {q[j, c]!r}")
        r = (r - p).astype(np.float32)
    assert np.array_equal(vals[:, m:, :], np.zeros_like(vals[:, m:, :]))    # padding directions
    assert np.array_equal(vals[:, :, n:], np.zeros_like(vals[:, :, n:]))    # padding cells


@pytest.mark.parametrize("form", ["bf16x2", "bf16x3"])
def test_automatic_choice_of_plans_that_leave_cus_idle(gpu, form):
    """Where row groups leave a quarter of an XCD's 32 CUs idle (17 or 18 groups: 769 to 832 directions; 11 groups: some
    ranges of rows) the resident kernel is chosen up to ten 256-cell chunks per set if its K loop is unrolled (800
    directions and fewer), up to one else, where it was measured to be the faster one; with full XCDs always."""
    def kernel(ds, n, k1, faces=1, ld=None):
        return ds.scatter_split_route(form, faces, n, 0, k1, ld=ld)[0]

    def dirset(m):
        xyz, w, F = rs.fibonacci_directions(m)
        return rs.DirectionSet(xyz, w, F)

    for m, k1, line in ((800, 800, 20480), (700, 500, 40960), (820, 820, 2048)):
        with dirset(m) as ds:
            assert [kernel(ds, n, k1) for n in (1, line, line + 1, 10 * line)] == ["resident"] * 2 + ["streaming"] * 2
            assert kernel(ds, 17, k1, faces=4) == "streaming" and kernel(ds, 17, k1, ld=1 << 24) == "streaming"
    for m in (400, 640, 1000):
        with dirset(m) as ds:
            assert [kernel(ds, n, m) for n in (1, 1 << 22)] == ["resident"] * 2


@pytest.mark.parametrize("n", [2048, 2049])
def test_automatic_choice_beyond_800_directions(gpu, n):
    """Both sides of the line at 820 directions (26 K-steps, rolled K loop): the streaming kernel's bits."""
    m = 820
    cell = np.resize(np.random.default_rng(n).lognormal(0.0, 1.5, size=1_000_003), (m, n, 1))
    xyz, w, F = rs.fibonacci_directions(m)
    with rs.DirectionSet(xyz, w, F) as ds:
        d_cell, out = D.DeviceArray.from_host(cell), D.DeviceArray((m, n))
        sb, cb = rs.split_sizes("bf16x3", 1, n, m)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_dev("bf16x3", d_cell, 1, n, m, state, scale)
        outs = []
        for waves in (0, 1, 8):
            out.fill(-1.0)
            ds.scatter_split("bf16x3", state, scale, 1, n, 0, m, out, waves=waves)
            D.synchronize()
            outs.append(out.to_host())
        for a in (d_cell, state, scale, out):
            a.free()
    assert np.array_equal(outs[0], outs[2]) and np.array_equal(outs[1], outs[2])


@pytest.mark.parametrize("form", ["bf16x2", "fp16x2", "bf16x3"])
@pytest.mark.parametrize("n,m", [(33, 100), (4097, 100), (4099, 250), (24577, 257), (16385, 417), (16384, 417), (8193, 450),
                                 (8192, 512), (4097, 513), (4100, 896), (131073, 20)])
def test_face_averaged_pack_instances_agree(gpu, form, n, m):
    """Each instance of the face-averaged pack (1, 2, 4 and 7 slots of lane pairs, 64-cell groups) and the sizes between
    which they are chosen against the one through LDS, which takes the same rows followed by zero rows up to 897
    directions and more: the same scales and the same bits of the first K-steps, for cells without an intensity and
    with infinities and NaN too."""
    rng = np.random.default_rng(n * m)
    illum = rng.lognormal(0.0, 3.0, size=(m, n, 4)) * rng.choice([-1.0, 1.0], size=(m, n, 4))
    illum[:, 3] = 0.0
    illum[m // 2, 5, 1] = np.inf
    illum[m - 1, 7, 2] = np.nan
    illum[0, 9, 0], illum[0, 9, 3] = np.inf, -np.inf
    illum[:, 11] = np.nan
    illum[9, 32, 0] = -np.inf

    def pack(a):
        rows, cells = a.shape[:2]
        d = D.DeviceArray.from_host(np.ascontiguousarray(a))
        sb, cb = rs.split_sizes(form, 1, cells, rows)
        state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
        rs.pack_split_avg_dev(form, d, cells, rows, state, scale)
        D.synchronize()
        got = state.to_host().view(np.uint16), scale.to_host()[:cells]
        for x in (d, state, scale):
            x.free()
        return got

    parts, steps, rows = (3 if form == "bf16x3" else 2), -(-m // 32), 928
    cells = min(n, 256)
    big = np.zeros((rows, cells, 4))
    big[:m] = illum[:, :cells]
    (got, scale), (want, want_scale) = pack(illum), pack(big)
    tile = parts * 64 * 8  # 16-bit values of a tile's K-step
    got = got.reshape(-1, steps, tile)[:-(-cells // 16)]
    want = want.reshape(-1, rows // 32, tile)[:, :steps]
    assert np.array_equal(scale[:cells], want_scale)
    nan = np.isnan(_part_values(got, form))
    assert np.array_equal(nan, np.isnan(_part_values(want, form)))
    assert np.array_equal(got[~nan], want[~nan])
    assert nan.any() and not nan.reshape(nan.shape[0], -1).all(axis=1).any()


@pytest.mark.parametrize("form", ["fp16x2", "bf16x3"])
@pytest.mark.parametrize("faces", [4, 1])
@pytest.mark.parametrize("m", [1248, 1249, 1280, 1281])
def test_cell_pack_around_the_one_pass_limit(gpu, form, faces, m):
    """Up to 1248 directions the cell-level packs read the input once, with a tile's averages in LDS; beyond, in two
    passes. Both against the definition (test_cell_pack_matches_layout_definition): the scales, and each part a value
    of its format nearest to what the parts before it left, a tie broken either way."""
    n = 37
    illum = np.random.default_rng(m).lognormal(0.0, 2.0, size=(m, n, faces))
    d_illum = D.DeviceArray.from_host(illum)
    sb, cb = rs.split_sizes(form, 1, n, m)
    state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
    if faces == 4:
        rs.pack_split_avg_dev(form, d_illum, n, m, state, scale)
    else:
        rs.pack_split_dev(form, d_illum, 1, n, m, state, scale)
    D.synchronize()
    got_state, got_scale = state.to_host(), scale.to_host()[:n]
    for a in (d_illum, state, scale):
        a.free()
    e = 11 - (np.frexp(np.max(illum, axis=(0, 2)))[1] - 1)
    assert np.array_equal(got_scale, np.ldexp(np.float32(1.0), -e).astype(np.float32))
    v = (((illum[..., 0] + illum[..., 1]) + illum[..., 2]) + illum[..., 3]) * 0.25 if faces == 4 else illum[..., 0]
    steps, tiles, nt = -(-m // 32), -(-n // 16), 3 if form == "bf16x3" else 2
    r = np.zeros((steps * 32, tiles * 16), np.float32)
    r[:m, :n] = v * np.ldexp(1.0, e)
    vals = got_state.view(np.uint16).reshape(tiles, steps, nt, 4, 16, 8).transpose(2, 1, 3, 5, 0, 4)
    for part in vals.reshape(nt, steps * 32, tiles * 16):
        p, q = _part_values(part, form), _nearest(r, form)
        x = r.astype(np.float64)
        assert np.all((p == q) | (np.abs(x - p) == np.abs(x - q)))
        r = (r - p).astype(np.float32)


@pytest.mark.parametrize("form,n,m", [("fp16x2", 43477, 854), ("fp16x2", 20001, 854), ("bf16x3", 80001, 640), ("fp16x2", 80001, 640)])
@pytest.mark.parametrize("f32", [False, True])
def test_every_kind_of_store_of_the_resident_kernel(gpu, form, n, m, f32):
    """Long panel slices (20 K-steps and more): results past the caches where the state fits the 256 MB cache and does
    not with the results, plain elsewhere, FP64 rows of whole lines past the caches always. The same bits, those of the
    streaming kernel, and nothing past a row's cells."""
    xyz, w, F = rs.fibonacci_directions(m)
    rows, strides = 300, (n, (n + 15) // 16 * 16 + 16)
    sb, cb = rs.split_sizes(form, 1, n, m)
    state, scale = D.DeviceArray((sb,), np.uint8), D.DeviceArray((cb // 4,), np.float32)
    d_in, out = D.DeviceArray((m, n)), D.DeviceArray((m, strides[-1]), np.float32 if f32 else np.float64)
    N.call("rsh_fill_lognormal_dev", d_in.ptr, d_in.size, 0.0, 1.5, 3, None)
    rs.pack_split_dev(form, d_in, 1, n, m, state, scale)
    mark = np.full(out.shape, -1.0, out.dtype)
    with rs.DirectionSet(xyz, w, F) as ds:
        for k1 in (m, rows):
            first = None
            for waves, ld in ((8, n), (1, n), (1, strides[-1])):
                out.copy_from(mark)
                ds.scatter_split(form, state, scale, 1, n, 0, k1, out, ld=ld, out_f32=f32, waves=waves)
                D.synchronize()
                got = out.to_host().reshape(-1)[:k1 * ld].reshape(k1, ld)
                first = got[:, :n].copy() if first is None else first
                assert np.array_equal(got[:, :n], first)
                assert np.all(got[:, n:] == -1.0)
    for a in (state, scale, d_in, out):
        a.free()
