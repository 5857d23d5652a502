"""TV_method on volumes whose rows are and are not whole float4s, with sides down to one voxel (every neighbour
periodic), and odd and even iteration counts (the dual field alternates between two buffers)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape,iters', [((1, 1, 4), 3), ((2, 1, 1), 4), ((1, 5, 3), 7), ((3, 2, 8), 6), ((9, 17, 33), 11),
                                         ((16, 24, 20), 12), ((7, 64, 260), 5), ((5, 6, 4), 0)])
def test_tv_shapes_vs_oracle(shape, iters):
    from mset_amd import lib
    v = np.random.default_rng(sum(shape) + iters).uniform(0, 3, shape).astype(np.float32)
    print('case: tv', shape, iters, flush=True)
    with lib.Context(0) as ctx:
        out, err = ctx.tv(v, 0.25, iters)
    ref, rerr = O.tv(v, 0.25, iters)
    # FP32 iteration, each step a contraction of the previous error: a few ulps
    assert rel(out, ref) < 1e-5
    assert abs(err - rerr) <= 1e-4 * abs(rerr) + 1e-5
