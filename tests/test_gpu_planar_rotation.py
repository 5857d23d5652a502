"""Planar rotations (about one axis) as real 1D shears, against the FP64 oracle: every line length, every choice
of the axis left alone, one and several steps, and white noise (full Nyquist components along all axes)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import rel

pytestmark = pytest.mark.gpu

AXES = {'z': 0, 'y': 1, 'x': 2}      # angle index (phi, theta, psi) about vec1 = z, vec2 = y, vec3 = x


@pytest.mark.parametrize('shape', [(16, 24, 32), (48, 16, 24), (24, 48, 96), (64, 32, 16), (96, 64, 48), (32, 16, 128),
                                   (16, 256, 24), (128, 24, 256), (256, 16, 16)])
@pytest.mark.parametrize('axis,deg', [('y', 50.0), ('y', -3.0), ('x', 33.0), ('z', -61.0)])
def test_planar_rotation_vs_oracle(shape, axis, deg):
    from mset_amd import lib
    ang = [0.0, 0.0, 0.0]
    ang[AXES[axis]] = deg
    v = np.random.default_rng(sum(shape) + int(abs(deg))).standard_normal(shape).astype(np.float32)
    print('case: planar rotation', shape, axis, deg, flush=True)
    R, _ = O.rot_matrix(ang)
    with lib.Context(0) as ctx:
        out = ctx.rotate(v, R)
    ref = O.rotate(v, R)
    assert rel(out, ref) < 1e-5              # as for the general routine
