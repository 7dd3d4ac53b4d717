"""The GRHD flux divergence on the device (bamhip_grhd_fluxes) against the
CPU oracle of matter_fluxes / grhd_flx1d_fvpr, box by box, on a level of
three boxes whose sizes leave partial tiles in every direction.  The data
hold a shock, smooth variation, a general metric with shift, a point whose
velocity reaches grhd_vmax (its interfaces carry no flux) and a non-finite
point (its interfaces are zeroed).  With the ideal gas every operation is
IEEE-rounded on both sides and FP contraction is off, so the right-hand
sides agree bitwise; the polytrope's pow is not correctly rounded on the
device, so that case is compared at 1e-12 of the largest value."""
import numpy as np
import pytest

import baum_amd as B
import oracle as O

pytestmark = pytest.mark.gpu

RHS = [0, 1, 2, 3, 4]
MET = list(range(5, 15))
PRIM = list(range(15, 20))
NV = 20
SHAPES = [(70, 9, 13, (-3.0, -1.0, -1.0)), (37, 21, 18, (2.0, -1.0, -1.0)), (5, 40, 7, (-3.0, 2.0, 2.0))]
H = 0.1


def _state(box, seed):
    rng = np.random.default_rng(seed)
    shape = (box.o, box.n, box.m)
    x = (box.x0 + H * np.arange(box.m))[None, None, :]
    y = (box.y0 + H * np.arange(box.n))[None, :, None]
    z = (box.z0 + H * np.arange(box.o))[:, None, None]
    met = np.zeros((10,) + shape)
    met[0] = 0.85 + 0.05 * np.sin(x + y) + 0.01 * rng.random(shape)
    met[1] = 0.04 * np.cos(y - z) * np.ones(shape)
    met[2] = -0.03 * np.sin(x * z) * np.ones(shape)
    met[3] = 0.02 * np.ones(shape)
    met[4:10] = np.array([1.1, 0.02, -0.01, 1.05, 0.015, 1.2])[:, None, None, None] + \
        0.01 * rng.standard_normal((6,) + shape)
    prim = np.zeros((5,) + shape)
    shock = np.where(x + 0.3 * y < 0.4, 1.0, 0.125)
    prim[0] = 1e-3 * shock * (1 + 0.1 * np.sin(3 * z)) * np.ones(shape)
    prim[1] = (0.1 + 0.2 * (shock == 1.0)) * (1 + 0.05 * rng.random(shape))
    prim[2] = 0.3 * np.tanh(x) * np.ones(shape)
    prim[3] = -0.2 * np.cos(x + z) * np.ones(shape)
    prim[4] = 0.1 * rng.standard_normal(shape)
    return met, prim


def _level(seed):
    oboxes = [O.make_box(m, n, o, *x0, H) for m, n, o, x0 in SHAPES]
    gboxes = [B.make_box(m, n, o, *x0, H) for m, n, o, x0 in SHAPES]
    lev = B.Level(gboxes, NV)
    lev.enable(range(NV))
    states = [_state(b, seed + k) for k, b in enumerate(oboxes)]
    # a point at grhd_vmax and a non-finite point in the second box
    states[1][1][2][5, 7, 20] = 2.0
    states[1][1][0][9, 3, 11] = np.nan
    rhs0 = [np.random.default_rng(seed + 10 + k).standard_normal((5, b.o, b.n, b.m)) for k, b in enumerate(oboxes)]
    for v in range(10):
        lev.put(MET[v], np.concatenate([s[0][v].reshape(-1) for s in states]))
    for v in range(5):
        lev.put(PRIM[v], np.concatenate([s[1][v].reshape(-1) for s in states]))
        lev.put(RHS[v], np.concatenate([r[v].reshape(-1) for r in rhs0]))
    return lev, oboxes, states, rhs0


def _run(eos, riemann, rec, c, seed=3):
    lev, oboxes, states, rhs0 = _level(seed)
    gp = B.hrsc_params(eos=eos, riemann=riemann, rec=rec)
    op = O.hrsc_params(eos=0 if eos == "ideal" else 1, riemann=riemann, rec=rec)
    lev.grhd_fluxes(gp, RHS, MET, PRIM, c=c)
    got = np.stack([lev.get(v) for v in RHS])
    lev.free()
    want = []
    for b, (met, prim), r in zip(oboxes, states, rhs0):
        want.append(O.grhd_fluxes(b, op, met, prim, r.copy(), c=c).reshape(5, -1))
    return got, np.concatenate(want, axis=1), np.concatenate([r.reshape(5, -1) for r in rhs0], axis=1)


@pytest.mark.parametrize("riemann,rec,c", [("LLF", "WENOZ", 0.0), ("HLL", "WENOZ", 0.0), ("LLF", "WENO5", 0.0),
                                           ("LLF", "WENOZ", 0.0625)])
def test_fluxes_ideal_gas_bitwise(riemann, rec, c):
    got, want, rhs0 = _run("ideal", riemann, rec, c)
    assert np.all(np.isfinite(want))
    np.testing.assert_array_equal(got, want)
    assert np.abs(got - rhs0).max() > 1e-3          # the fluxes did something


def test_fluxes_polytrope():
    got, want, rhs0 = _run("poly", "LLF", "WENOZ", 0.0)
    scale = np.abs(want - rhs0).max()
    assert np.abs(got - want).max() <= 1e-12 * scale
    np.testing.assert_array_equal(got[1], rhs0[1])  # cold EOS: no tau flux


def _one_box(shape, rhs_of, c=0.0625, seed=9):
    ob, gb = O.make_box(*shape, -1.0, -1.0, -1.0, H), B.make_box(*shape, -1.0, -1.0, -1.0, H)
    met, prim = _state(ob, seed)
    rhs0 = np.random.default_rng(seed + 1).standard_normal((5, ob.o, ob.n, ob.m))
    lev = B.Level([gb], NV)
    lev.enable(range(NV))
    for vs, data in ((MET, met), (PRIM, prim), (RHS, rhs0)):
        for v, d in zip(vs, data):
            lev.put(v, d.reshape(-1))
    lev.grhd_fluxes(B.hrsc_params(eos="ideal", riemann="HLL", rec="WENOZ"), rhs_of, MET, PRIM, c=c)
    got = np.stack([lev.get(v) for v in RHS])
    lev.free()
    op = O.hrsc_params(eos=0, riemann="HLL", rec="WENOZ")
    want = O.grhd_fluxes(ob, op, met, prim, rhs0.copy(), c=c).reshape(5, -1)
    add = O.grhd_fluxes(ob, op, met, prim, np.zeros_like(rhs0), c=c).reshape(5, -1)
    return got, want, rhs0.reshape(5, -1), add


@pytest.mark.parametrize("shape", [(62, 14, 17), (63, 15, 15), (64, 16, 16), (127, 5, 31), (16, 31, 4)])
def test_fluxes_at_tile_edges_bitwise(shape):
    """Lines that end just before, at and after the end of a tile of 63 (x) or 15 (y, z) points."""
    got, want, _, _ = _one_box(shape, RHS)
    np.testing.assert_array_equal(got, want)


def test_fluxes_into_one_variable_twice():
    """A list that names a variable twice takes both divergences: six sums, each rounded once."""
    got, _, rhs0, add = _one_box((20, 18, 17), [0, 1, 2, 3, 0])
    want = rhs0.copy()
    want[0] = want[0] + add[0] + add[4]
    want[1:4] = want[1:4] + add[1:4]
    bound = 6 * np.finfo(float).eps * (np.abs(rhs0) + np.abs(add)).max() * 2
    assert np.abs(got[4] - rhs0[4]).max() == 0.
    assert np.abs(got[:4] - want[:4]).max() <= bound
