"""The adjoint's tape takes each face's state from its upwind cell; faces that
stand still or stay within rel_eps average both sides, and faces on outflow sides
take the inside cell.  Dot-product test against the oracle's forward-mode
derivative under a velocity of such faces, on periodic boxes (mask and compare
indexing) and on the box-list layout with outflow sides."""
import numpy as np
import pytest

import pyoracle
from test_gpu_adjoint import setup_case, stepper_for, to_dev
from test_gpu_step_bc import NN, mac_velocity, scalar_fields, stepper

pytestmark = pytest.mark.gpu

EPS = 1e-3  # so that faces within it still move the solution


def still(rng, shape):
    return rng.choice([-1.0, 1.0], shape) * rng.choice(
        [0.0, 0.5 * EPS, EPS, 0.3, 0.9], shape, p=[0.1, 0.1, 0.1, 0.3, 0.4])


def check(v, jw, sb, ub, ws, wu):
    lhs = float(np.sum(v * jw))
    rhs = float(np.sum(sb * ws) + sum(np.sum(ub[d] * wu[d]) for d in range(3)))
    # some hundred roundings per term on either side
    size = np.sum(np.abs(v * jw)) + np.sum(np.abs(sb * ws)) + sum(
        np.sum(np.abs(ub[d] * wu[d])) for d in range(3))
    assert abs(lhs - rhs) <= 200 * 2.0 ** -53 * size, (lhs, rhs)


@pytest.mark.parametrize("cons", [False, True])
@pytest.mark.parametrize("n,ppm", [(16, 1), (13, 1), (16, 2), (13, 2)])
def test_periodic_still_faces(n, ppm, cons):
    from maestroex_amd.adjoint import ScalStepper
    s, _, dt, _ = setup_case(n=n, seed=5)
    rng = np.random.default_rng(21)
    u = [still(rng, (n, n, n)) for _ in range(3)]
    ws, v = rng.standard_normal(s.shape), rng.standard_normal(s.shape)
    wu = [rng.standard_normal(x.shape) for x in u]
    _, jw = pyoracle.scal_step_bc(s, u, dt, [1.0 / n] * 3, EPS, [1, 1, 1], ws, wu, ppm_type=ppm,
                                  conservative=cons)
    st = ScalStepper(n, s.shape[0], dt, EPS, ppm_type=ppm, conservative=cons)
    sb, ub = st.vjp(to_dev(s), tuple(to_dev(x) for x in u), to_dev(v))
    check(v, jw, sb.cpu().numpy(), [x.cpu().numpy() for x in ub], ws, wu)


@pytest.mark.parametrize("cons", [False, True])
@pytest.mark.parametrize("per", [(1, 1, 0), (0, 0, 0)])
@pytest.mark.parametrize("ppm", [1, 2])
def test_outflow_still_faces(ppm, per, cons):
    dt = 0.02
    s = scalar_fields(NN, 2, seed=6)
    rng = np.random.default_rng(22)
    u = [still(rng, x.shape) for x in mac_velocity(NN, per, seed=7)]
    ws, v = rng.standard_normal(s.shape), rng.standard_normal(s.shape)
    wu = [rng.standard_normal(x.shape) for x in u]
    _, jw = pyoracle.scal_step_bc(s, u, dt, [1.0 / q for q in NN], EPS, per, ws, wu, ppm_type=ppm,
                                  conservative=cons)
    st = stepper(per, ppm, 2, dt, EPS, cons=cons)
    sb, ub = st.vjp(to_dev(s), tuple(to_dev(x) for x in u), to_dev(v))
    check(v, jw, sb.cpu().numpy(), [x.cpu().numpy() for x in ub], ws, wu)
