"""The dense-face forms of the residual kernel at the edges of its
workgroups: whole and part-filled last blocks, elements whose neighbours are
numbered before and after them, every launch variant."""
import numpy as np
import pytest

from pdes_amd import abi, euler, problems
from pdes_amd._lib import check, lib
from helpers import assert_parity, state_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", ["roe", "es"])
@pytest.mark.parametrize("kind,p", [("vortex", 1), ("vortex", 2), ("vortex", 3), ("vortex", 4), ("cube", 1),
                                    ("cube", 2)])
def test_dense_face_residual_at_block_edges(oracle, kind, p, flux):
    """Residual and directional derivative on 2, 32 and 128 triangles (6 and 48
    tets), numbered at random: the oracle's values to 1e-12, the same bits from
    all eight launch variants, and derivatives that the oracle's complex step
    gives to 1e-12."""
    for n in (1, 4, 8) if kind == "vortex" else (1, 2):
        print(f"case {kind} n={n} p={p} {flux}", flush=True)
        m, op, ph = problems.make_problem(kind, n, p, "omega", flux)
        perm = np.random.default_rng(n).permutation(m.numEl)
        place = np.argsort(perm).astype(m.interfaces.dtype)
        for a in ("coords", "dxidx", "jac", "vert_coords"):
            setattr(m, a, np.ascontiguousarray(getattr(m, a)[perm]))
        m.interfaces[:, :2] = place[m.interfaces[:, :2]]
        m.bndryfaces[:, 0] = place[m.bndryfaces[:, 0]]
        if n in (2, 4):   # metric terms of each node of its own
            m.dxidx = m.dxidx * (1.0 + 1e-3 * np.random.default_rng(n).uniform(-1.0, 1.0, m.dxidx.shape))
        b = abi.make_descriptors(m, op, ph)
        q = state_for(kind, m, ph)
        ref, scale = oracle.residual(b, q), oracle.residual_scale(b, q)
        eqn = euler.EulerData(m, op, ph)
        eqn.set_q(q)
        first = None
        for var in range(8):
            check(lib().pdes_set_launch_variant(eqn.ctx, var, var))
            euler.evalResidual(m, op, eqn)
            assert_parity(eqn.res, ref, scale, 1e-12, f"n {n} variant {var}")
            first = eqn.res.copy() if first is None else first
            assert np.array_equal(eqn.res, first), f"n {n}: variant {var} differs from variant 0"
        v = np.random.default_rng(7).standard_normal(q.shape)
        jv = oracle.jv_complex_step(b, q, v)
        assert np.abs(euler.evaldRdqProduct(eqn, v) - jv).max() <= 1e-12 * np.abs(jv).max()
        eqn.free()


@pytest.mark.parametrize("n,p", [(1, 1), (4, 1), (5, 2), (90, 2)])
def test_residual_norm_of_one_and_many_blocks(n, p):
    """calcNorm over 1, 2, 10 and 1,024 reduction blocks (several entries per
    thread in the last), repeated: the same bits each time, and numpy's sum of
    N positive terms to N rounding errors; a state with a negative density
    fails once and not after the state is mended."""
    m, op, ph = problems.make_problem("vortex", n, p, "omega" if p == 1 else "diage", "roe")
    q = problems.vortex_noise_state(m, ph, seed=2)
    eqn = euler.EulerData(m, op, ph)
    eqn.set_q(q)
    euler.evalResidual(m, op, eqn)
    ref = np.sqrt((eqn.res ** 2 * eqn.Minv).sum())
    got = [euler.calcNorm(eqn) for _ in range(4)]
    assert len(set(got)) == 1
    assert abs(got[0] - ref) <= q.size * 2.0 ** -53 * ref
    bad = q.copy()
    bad[-1, 0, 0] = -1.0
    eqn.set_q(bad)
    euler.evalResidual_device(eqn)
    with pytest.raises(Exception):
        euler.calcNorm(eqn)
    eqn.set_q(q)
    euler.evalResidual_device(eqn)
    assert euler.calcNorm(eqn) == got[0]
    eqn.free()


@pytest.mark.parametrize("p", [1, 2, 3, 4])
@pytest.mark.parametrize("where", ["one node", "everywhere"])
def test_split_form_where_logarithms_are_needed(oracle, p, where):
    """Diagonal-E split form with states so far apart (density times 1 to 2) that
    the logarithmic means leave their series: at one node, so that one lane of a
    wave needs the logarithm, and everywhere; the oracle's values to 1e-12."""
    m, op, ph = problems.make_problem("vortex", 5, p, "diage", "ir")
    b = abi.make_descriptors(m, op, ph)
    q = state_for("vortex", m, ph)
    f = 1.0 + np.random.default_rng(p).uniform(0.0, 1.0, q.shape[:2] + (1,))
    if where == "one node":
        q[3, 1] *= 2.0
    else:
        q = q * f
    eqn = euler.EulerData(m, op, ph)
    eqn.set_q(q)
    euler.evalResidual(m, op, eqn)
    assert_parity(eqn.res, oracle.residual(b, q), oracle.residual_scale(b, q), 1e-12, f"p {p} {where}")
    eqn.free()
