"""The Z4c tile kernel where its tiles, its store variants and its list rules
can go wrong.

The tile kernel computes 16x4x4 tiles in the bulk and slabs two points thick
along the box faces; a result is stored as the right-hand side, as unew =
upre + c RHS, or as one of the RK4 stage forms.  The right-hand side is
compared with the CPU oracle at 1e-12 of each field's largest value, as in the
other right-hand side tests, or at the rounding floor of its second differences
where that is larger: fields of size max|u|, each rounded by eps and weighted
by at most 64 / 12 per h^2 (the 4th-order row -1 16 -30 16 -1 over 12), leave
5.4 eps max|u| / h^2 a term; some of the small boxes' right-hand sides are no
larger than 1e-3 and their terms are of order one.  The other forms with the sums formed on the host
from the device's own right-hand side: one product and one sum, of which the
device may fuse the product (one rounding of the product, eps |w RHS|).
"""
import ctypes as C

import numpy as np
import pytest

import baum_amd as B
import oracle as O
from spacetimes import flat_z4c, grid, puncture_z4c

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
U, R, A, P, ACC, V, CP = (list(range(25 * k, 25 * k + 25)) for k in range(7))
# one tile and less, one more than a tile in each direction, only shell, slabs longer than a tile
SIZES = [(7, 7, 7), (22, 10, 10), (23, 11, 9), (24, 14, 15), (39, 8, 21), (6, 5, 18)]


def _level(size, seed=0):
    h = 0.2
    ob = O.make_box(*size, -1.9, -0.7, -0.8, h, skip=(1,) * 6)
    X = grid(ob)
    u = puncture_z4c(X, masses=((1.0, (0.05, -0.02, 0.03)),))
    rng = np.random.default_rng(seed)
    u[19:22] = 0.1 * rng.standard_normal((3,) + X.shape[1:])
    u[13] = 0.05 * np.sin(X[0]) * np.cos(X[1])
    u[22:25] = 0.01 * rng.standard_normal((3,) + X.shape[1:])
    lev = B.Level([B.make_box(*size, ob.x0, ob.y0, ob.z0, h)], 175)
    lev.enable(range(175))
    for v in range(175):
        lev.fill(v, 0.0)
    lev.put_state(U, u.reshape(25, -1))
    return lev, ob, u


def _stage(lev, par, src, acc, accout, base, vout, copy, wc, wv):
    L = B.lib()
    ip = C.POINTER(C.c_int)
    L.bamhip_z4c_rhs_rk4_stage.restype = C.c_int
    L.bamhip_z4c_rhs_rk4_stage.argtypes = [C.c_void_p, C.POINTER(B.Z4cParams)] + [ip] * 6 + [C.c_double] * 2 + [ip]
    arr = lambda x: None if x is None else (C.c_int * 25)(*x)  # noqa: E731
    B.check(L.bamhip_z4c_rhs_rk4_stage(lev.h, C.byref(par), arr(src), arr(acc), arr(accout), arr(base), arr(vout),
                                       arr(copy), wc, wv, None), "bamhip_z4c_rhs_rk4_stage")


def _computed(size):
    m = np.zeros(size[::-1], bool)
    m[1:-1, 1:-1, 1:-1] = True
    return m.reshape(-1)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("params", [dict(), dict(z4_shift="withB gamma0 withGadv withBadv withShiftadv",
                                                 z4_shiftalphapower=1.0, z4_kappa1=0.02, z4_lapse="1+log2 withshift")])
def test_rhs_of_partial_tiles_matches_oracle(size, params):
    lev, ob, u = _level(size)
    cpu, _ = O.z4c_rhs(ob, O.z4c_params(**params), u)
    lev.z4c_rhs(B.z4c_params(**params), R, U)
    got = lev.get_state(R).reshape(u.shape)
    floor = 64 / 12 * EPS * np.abs(u).max() / ob.dx ** 2
    for v in range(25):
        assert np.abs(got[v] - cpu[v]).max() <= max(1e-12 * np.abs(cpu[v]).max(), floor), B.VAR_NAMES[v]
    lev.free()


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("has_v,has_cp", [(True, True), (True, False), (False, False), (False, True)])
def test_stage_forms_match_sums_of_the_rhs(size, has_v, has_cp):
    lev, _, u = _level(size)
    par = B.z4c_params()
    lev.z4c_rhs(par, R, U)
    k = lev.get_state(R)
    rng = np.random.default_rng(3)
    acc, base = rng.standard_normal(k.shape), rng.standard_normal(k.shape)
    lev.put_state(ACC, acc)
    lev.put_state(P, base)
    wc, wv = 0.3, 0.7
    _stage(lev, par, U, ACC, A, P, V if has_v else None, CP if has_cp else None, wc, wv)
    on = _computed(size)
    for lst, want, w in ((A, acc + wc * k, wc), (V, base + wv * k, wv), (CP, base, 0.0)):
        got = lev.get_state(lst)
        if (lst is V and not has_v) or (lst is CP and not has_cp):
            assert not got.any()
            continue
        assert not got[:, ~on].any()
        bar = EPS * (np.abs(w * k) + np.abs(want))
        assert (np.abs(got - want)[:, on] <= bar[:, on]).all()
    lev.free()


@pytest.mark.parametrize("size", SIZES)
def test_addlinear_projects_the_sum(size):
    """unew = upre + c RHS with the trace of At removed and det gt = 1"""
    lev, ob, u = _level(size)
    c = 0.05
    par = B.z4c_params()
    lev.put_state(P, u.reshape(25, -1))
    lev.z4c_rhs(par, R, U, upre=P, c=c)
    got = lev.get_state(R)
    lev.z4c_rhs(par, A, U)
    raw = u.reshape(25, -1) + c * lev.get_state(A)
    on = _computed(size)
    g, At = raw[0:6, on], raw[7:13, on]
    det = g[0] * (g[3] * g[5] - g[4] ** 2) - g[1] * (g[1] * g[5] - g[4] * g[2]) + g[2] * (g[1] * g[4] - g[3] * g[2])
    ig = np.array([g[3] * g[5] - g[4] ** 2, g[2] * g[4] - g[1] * g[5], g[1] * g[4] - g[2] * g[3],
                   g[0] * g[5] - g[2] ** 2, g[1] * g[2] - g[0] * g[4], g[0] * g[3] - g[1] ** 2]) / det
    tr = (ig * At * np.array([1, 2, 2, 1, 2, 1])[:, None]).sum(0)
    want = raw[:, on].copy()
    want[7:13] = At - tr / 3 * g
    want[0:6] = g * det ** (-1 / 3)
    for v in range(25):
        assert np.abs(got[v][on] - want[v]).max() <= 1e-13 * max(np.abs(want[v]).max(), np.abs(raw[v]).max(), 1e-30)
    assert not got[:, ~on].any()
    lev.free()


def test_lists_crossed_between_fields():
    """an output that is another field's accumulator or start state: every
    operand is read before any output is written"""
    size = (24, 14, 15)
    par = B.z4c_params()
    rng = np.random.default_rng(5)
    out = []
    for crossed in (False, True):
        lev, _, _ = _level(size)
        acc, base = rng.standard_normal((2, 25, lev.npoints)) if not out else (out[0][2], out[0][3])
        lev.put_state(ACC, acc)
        lev.put_state(P, base)
        # the next state of field v goes where the start state of field v + 1 was
        vout = [P[(v + 1) % 25] for v in range(25)] if crossed else V
        _stage(lev, par, U, ACC, A, P, vout, None, 0.3, 0.7)
        out.append((lev.get_state(A), lev.get_state(vout), acc, base))
        lev.free()
    on = _computed(size)
    for x, y in zip(out[0][:2], out[1][:2]):
        scale = np.abs(x[:, on]).max(axis=1, keepdims=True)
        assert (np.abs(x - y)[:, on] <= 1e-12 * scale).all()


def _bc_stage(lev, par, src, acc, accout, base, vout, copy, wc, wv):
    L = B.lib()
    ip = C.POINTER(C.c_int)
    L.bamhip_z4c_bc_rk4_stage.restype = C.c_int
    L.bamhip_z4c_bc_rk4_stage.argtypes = [C.c_void_p, C.POINTER(B.Z4cParams)] + [ip] * 6 + [C.c_double] * 2 + [C.c_int] * 2
    arr = lambda x: None if x is None else (C.c_int * 25)(*x)  # noqa: E731
    B.check(L.bamhip_z4c_bc_rk4_stage(lev.h, C.byref(par), arr(src), arr(acc), arr(accout), arr(base), arr(vout),
                                      arr(copy), wc, wv, 0, 0), "bamhip_z4c_bc_rk4_stage")


@pytest.mark.parametrize("shift", [0, 1, -1])
def test_radiative_boundary_with_lists_crossed_between_fields(shift):
    """an output that is the operand of the field `shift` places on: the values at the surface are those
    of lists of their own, one product and one sum from the radiative right-hand side"""
    size = (18, 15, 12)
    par = B.z4c_params()
    rng = np.random.default_rng(6)
    ring = lambda lst: [lst[(v + shift) % 25] for v in range(25)]  # noqa: E731
    lev, _, _ = _level(size)
    lev.z4c_set_boundary(par, R, U)
    k = lev.get_state(R)
    on = ~_computed(size)
    assert np.abs(k[:, on]).max() > 0
    base, acc = rng.standard_normal((2,) + k.shape)
    c, wc, wv = 0.4, 0.3, 0.7

    def compare(lst, want, w):
        bar = EPS * (np.abs(w * k) + np.abs(want))
        assert (np.abs(lev.get_state(lst) - want)[:, on] <= bar[:, on]).all()

    lev.put_state(P, base)
    lev.z4c_set_boundary(par, ring(P), U, upre=P, c=c)
    compare(ring(P), base + c * k, c)
    lev.put_state(P, base)
    lev.put_state(ACC, acc)
    _bc_stage(lev, par, U, ACC, ring(ACC), P, ring(P), CP, wc, wv)
    compare(ring(ACC), acc + wc * k, wc)
    compare(ring(P), base + wv * k, wv)
    compare(CP, base, 0.0)
    lev.free()


def test_radiative_boundary_into_one_variable_twice():
    """a list that names a variable twice leaves the later field's value there"""
    size = (9, 8, 10)
    par = B.z4c_params()
    lev, _, _ = _level(size)
    lev.z4c_set_boundary(par, R, U)
    k = lev.get_state(R)
    lev.z4c_set_boundary(par, A[:24] + [A[3]], U)
    got = lev.get_state(A)
    k[3] = k[24]
    k[24] = 0.0
    on = ~_computed(size)
    np.testing.assert_array_equal(got[:, on], k[:, on])
    lev.free()


@pytest.mark.parametrize("front", [((5, 5, 5), (1,) * 6), ((3, 3, 3), (2,) * 6)])
def test_tuned_choice_is_not_taken_over_by_a_misaligned_level(front):
    """a box of even rows admits the 16-byte staging, the same box behind an odd number of points does not:
    the tuner times the second level anew, without it (x4=-1), also where the box in front has no regions"""
    size, (fsize, fskip) = (24, 14, 16), front
    lev, ob, u = _level(size)
    cpu, _ = O.z4c_rhs(ob, O.z4c_params(), u)
    fu = flat_z4c(fsize[::-1])
    box = B.make_box(*size, ob.x0, ob.y0, ob.z0, ob.dx)
    two = B.Level([B.make_box(*fsize, 5.0, 5.0, 5.0, ob.dx, skip=fskip), box], 50)
    two.enable(range(50))
    for v in R:
        two.fill(v, 0.0)
    two.put_state(U, np.concatenate([fu.reshape(25, -1), u.reshape(25, -1)], axis=1))
    B.tune_clear()
    lev.z4c_rhs(B.z4c_params(), R, U)
    assert "x4=-1.0000ms" not in B.tune_report()
    two.z4c_rhs(B.z4c_params(), R, U)
    assert B.tune_report().count("x4=-1.0000ms") >= 1
    got = two.box_view(two.get_state(R), 1)
    floor = 64 / 12 * EPS * np.abs(u).max() / ob.dx ** 2
    for v in range(25):
        assert np.abs(got[v] - cpu[v]).max() <= max(1e-12 * np.abs(cpu[v]).max(), floor), B.VAR_NAMES[v]
    lev.free()
    two.free()


def _flat_level(size, fields=()):
    """flat space with constant fields {index: value}, radiative faces"""
    u = flat_z4c(size[::-1])
    for v, x in fields:
        u[v] = x
    lev = B.Level([B.make_box(*size, 0.0, 0.0, 0.0, 0.1)], 75)
    lev.enable(range(75))
    for v in R + A:
        lev.fill(v, 0.0)
    lev.put_state(U, u.reshape(25, -1))
    return lev, u


def test_lapse_source_with_theta_far_above_khat():
    """d_t alpha = -2 alpha Khat where |Theta| is a million times |Khat|: Khat is used as it is read, so a
    product and its factor round, 2 eps; from K - 2 Theta it would carry eps Theta / Khat.  (The differences of
    a lapse of few bits are 0.)"""
    size, alpha, khat = (24, 14, 15), 0.75, 1.2345e-9
    lev, _ = _flat_level(size, ((18, alpha), (13, khat), (17, 1e-3)))
    lev.z4c_rhs(B.z4c_params(), R, U)
    got = lev.get(R[18])[_computed(size)]
    want = -2.0 * alpha * khat
    assert np.abs(got - want).max() <= 2 * EPS * abs(want)
    lev.free()


@pytest.mark.parametrize("at", [(5, 6, 7), (1, 6, 7)])
@pytest.mark.parametrize("params", [dict(), dict(advection_lopsided=0)])
def test_negative_conformal_factor_is_reported(at, params):
    """psi^-4 = chi^(-4 / chipsipower) of a chi below 0 is not a number, in the bulk and in the shell, in the
    tile kernel and in the per-point kernel; a positive floor under chi makes it one"""
    lev, u = _flat_level((16, 14, 15))
    u[(6,) + at[::-1]] = -1e-3
    lev.put(U[6], u[6])
    with pytest.raises(B.BamhipError, match="non-finite"):
        lev.z4c_rhs(B.z4c_params(**params), R, U)
    lev.z4c_rhs(B.z4c_params(z4_chi_div_floor=1e-4, **params), R, U)
    lev.free()


@pytest.mark.parametrize("params", [dict(), dict(advection_lopsided=0)])
def test_lapse_of_three_is_reported(params):
    """the second slicing's 1 / (3 - alpha) has no value at alpha = 3, whatever its coefficient, in the tile
    kernel as in the per-point kernel"""
    lev, u = _flat_level((16, 14, 15))
    u[18, 7, 6, 5] = 3.0
    lev.put(U[18], u[18])
    with pytest.raises(B.BamhipError, match="non-finite"):
        lev.z4c_rhs(B.z4c_params(**params), R, U)
    lev.free()


@pytest.mark.parametrize("signs", [(1, 1, 1), (-1, -1, -1), (1, -1, 1)])
def test_upwind_row_leaves_out_the_downwind_points(signs):
    """the lop-sided row of a shift component reaches three points upwind and one downwind: a spike anywhere
    else changes nothing, not by rounding either.  B is advected and read at the point, nothing more."""
    size, spike = (24, 14, 15), (11, 7, 7)
    par = dict(z4_shift="withB gamma0 withGadv withBadv withShiftadv", order_dissipation=0)
    rng = np.random.default_rng(8)
    lev, u = _flat_level(size, tuple((19 + a, 0.3 * s) for a, s in enumerate(signs)))
    u[22:25] = rng.standard_normal((3,) + size[::-1])
    ob = O.make_box(*size, 0.0, 0.0, 0.0, 0.1, skip=(1,) * 6)
    out, ref = [], []
    for value in (0.0, 1e10):
        u[(slice(22, 25),) + spike[::-1]] = value
        lev.put_state(U, u.reshape(25, -1))
        lev.z4c_rhs(B.z4c_params(**par), R, U)
        out.append(lev.get_state(R)[22:].reshape((3,) + size[::-1]))
        ref.append(O.z4c_rhs(ob, O.z4c_params(**par), u)[0][22:])
    same = ref[0] == ref[1]
    for a in range(3):  # the points that see the spike two and three points downwind
        for d in (2, 3):
            q = list(spike)
            q[a] += d * signs[a]
            assert same[(slice(None),) + tuple(q[::-1])].all()
    np.testing.assert_array_equal(out[1][same], out[0][same])
    lev.free()


@pytest.mark.parametrize("field", [0, 6, 18, 19])
@pytest.mark.parametrize("off", [(1, 2, 0), (2, 1, 0), (-1, -2, 0), (0, 1, 2), (0, -2, 2), (1, 0, -2)])
def test_order_two_points_do_not_read_the_outer_corners(field, off):
    """one point from a face the mixed derivatives are of order 2 and reach one point: what lies further out
    off the axes does not matter, not even when it is no number"""
    size, at = (16, 14, 15), (1, 7, 6)
    lev, _, u = _level(size)
    lev.set_check(0)
    q = at[0] + size[0] * (at[1] + size[1] * at[2])
    lev.z4c_rhs(B.z4c_params(), R, U)
    want = lev.get_state(R)[:, q]
    u[(field,) + tuple(np.add(at, off))[::-1]] = np.nan
    lev.put(U[field], u[field])
    lev.z4c_rhs(B.z4c_params(), R, U)
    np.testing.assert_array_equal(lev.get_state(R)[:, q], want)
    assert np.isfinite(want).all()
    lev.free()


def test_every_index_of_a_variant_can_be_pinned():
    """nine bulk and six shell indices, several of which share a kernel: each gives bitwise the same"""
    lev, _, _ = _level((24, 14, 16))
    names = [B.variants(k) for k in (B.BULK, B.SHELL)]
    assert [len(n) for n in names] == [9, 6] and [len(set(n)) for n in names] == [3, 3]
    first = None
    try:
        for kind in (B.BULK, B.SHELL):
            for v in range(len(names[kind])):
                B.force_variant(kind, v)
                lev.z4c_rhs(B.z4c_params(), R, U)
                got = lev.get_state(R)
                first = got if first is None else first
                np.testing.assert_array_equal(got, first)
            B.force_variant(kind, -1)
            with pytest.raises(B.BamhipError):
                B.force_variant(kind, len(names[kind]))
    finally:
        B.force_variant(B.BULK, -1)
        B.force_variant(B.SHELL, -1)
    lev.free()


@pytest.fixture(scope="module")
def uneven():
    """three boxes of even rows and offsets with 33 bulk and 44 slab tiles, numbers that 8 does not divide,
    and 25 fields of operands for the update forms"""
    h, rng = 0.2, np.random.default_rng(12)
    boxes, us = [], []
    for (m, n, o), x0 in (((20, 20, 20), (-1.9, -1.8, -2.0)), ((22, 17, 26), (2.3, -1.5, -2.4)),
                          ((8, 13, 7), (-0.4, 2.6, 0.3))):
        ob = O.make_box(m, n, o, *x0, h, skip=(1,) * 6)
        u = puncture_z4c(grid(ob), masses=((1.0, (0.05, -0.02, 0.03)),))
        u[19:22] = 0.1 * rng.standard_normal((3,) + u.shape[1:])
        us.append(u.reshape(25, -1))
        boxes.append(B.make_box(m, n, o, *x0, h, skip=(1,) * 6))
    lev = B.Level(boxes, 175)
    lev.enable(range(175))
    lev.put_state(U, np.concatenate(us, axis=1))
    rng = np.random.default_rng(13)
    for lst in (P, ACC):
        lev.put_state(lst, lev.get_state(U) + 0.01 * rng.standard_normal((25, lev.npoints)))
    yield lev
    lev.free()


@pytest.mark.parametrize("form", ["rhs", "addlinear", (True, True), (True, False), (False, False), (False, True)])
def test_launches_and_stagings_bitwise_equal(uneven, form):
    """every staging, bulk and slabs in one launch or in two, tiles numbered by XCD or not: bitwise one result"""
    lev, par, first = uneven, B.z4c_params(), None
    try:
        for bulk, shell in ((0, 2), (1, 1), (5, 4)):
            B.force_variant(B.BULK, bulk)
            B.force_variant(B.SHELL, shell)
            assert B.variants(B.BULK)[bulk].split()[2:] == B.variants(B.SHELL)[shell].split()[2:]
            for overlap in (True, False):
                for xcd in (True, False):
                    B.set_overlap(overlap)
                    B.set_xcd_map(xcd)
                    for v in R + A + V + CP:
                        lev.fill(v, 0.0)
                    if form == "rhs":
                        lev.z4c_rhs(par, R, U)
                    elif form == "addlinear":
                        lev.z4c_rhs(par, R, U, upre=P, c=0.05)
                    else:
                        _stage(lev, par, U, ACC, A, P, V if form[0] else None, CP if form[1] else None, 0.3, 0.7)
                    got = lev.get_state(R + A + V + CP)
                    first = got if first is None else first
                    np.testing.assert_array_equal(got, first, err_msg=str((bulk, overlap, xcd)))
    finally:
        B.force_variant(B.BULK, -1)
        B.force_variant(B.SHELL, -1)
        B.set_overlap(True)
        B.set_xcd_map(True)
    assert np.abs(first).max() > 0


def test_tuner_times_the_launches_that_run(uneven):
    """a level with bulk and shell: the fastest single launch against the fastest pair, the faster one first"""
    B.tune_clear()
    uneven.z4c_rhs(B.z4c_params(), R, U)
    lines = B.tune_report().splitlines()
    assert len(lines) == 2
    cost, names = [], []
    for line in lines:
        name, times = line.split(" <- ")
        ms = dict(t.rsplit("=", 1) for t in times.split(": ", 1)[1].removesuffix("ms").split("ms "))
        picked = name.split(", ")
        for p in picked:
            same = [float(t) for n, t in ms.items() if n.split()[:2] == p.split()[:2]]
            assert len(same) == 3 and float(ms[p]) == min(same)
        cost.append(sum(float(ms[p]) for p in picked))
        names.append(picked)
    assert cost[0] <= cost[1]
    assert sorted(len(n) for n in names) == [1, 2]


def test_level_of_more_regions_than_a_launch_holds():
    """six boxes are 42 regions, a launch holds 32: the slabs of five boxes and more, then the rest and the
    bulk regions; bitwise each box by itself"""
    size, h = (14, 12, 10), 0.2
    us, boxes = [], []
    for b in range(6):
        ob = O.make_box(*size, 3.0 * b - 8.0, -0.7, -0.8, h, skip=(1,) * 6)
        us.append(puncture_z4c(grid(ob), masses=((1.0, (0.05, -0.02, 0.03)),)).reshape(25, -1))
        boxes.append(B.make_box(*size, ob.x0, ob.y0, ob.z0, h))

    def rhs(bs, u):
        lev = B.Level(bs, 50)
        lev.enable(range(50))
        for v in R:
            lev.fill(v, 0.0)
        lev.put_state(U, u)
        lev.z4c_rhs(B.z4c_params(), R, U)
        got = lev.get_state(R)
        lev.free()
        return got

    apart = np.concatenate([rhs([b], u) for b, u in zip(boxes, us)], axis=1)
    np.testing.assert_array_equal(rhs(boxes, np.concatenate(us, axis=1)), apart)
