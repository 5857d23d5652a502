"""Mini-batches of more positions than the device keeps resident, so that gradient slabs are added to: every size of the
on-chip separable routine, against the FP64 oracle and bit for bit under a capped grid."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.test_gpu_parity import LOSS_TOL, assert_update_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,nz', [(16, 3), (24, 2), (32, 3), (48, 2), (64, 1), (96, 1)])
def test_slabs_of_several_positions(n, nz):
    from mset_amd import lib
    npos = lib.batch_slots(n) + 37               # at least every workgroup that any routine keeps resident
    c = small_case(n=n, nz=nz, binning=1, npos=npos, seed=n + 1, spread=n / 6)
    steps = (30.0, 2e-4, 2e-2)
    print('case: slab reuse', n, nz, npos, flush=True)
    out = []
    for slots in (0, 60):
        with lib.Context(0) as ctx:
            ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=1,
                       step_size=steps, n_scan=(npos, 1))
            ctx.set_slot_limit(slots)
            err = ctx.run_batched(npos)
            out.append(ctx.download() + (err,))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    V, pr, xl, yl, err = out[0]
    G, P, D, ep = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], 1, c['sig'], c['dx'])
    assert abs(err / (ep.sum() / npos) - 1) < LOSS_TOL
    assert_update_close(V, c['V'] + steps[0] * G, c['V'], npos)
    assert_update_close(pr, c['probe'] - steps[1] * P, c['probe'], npos)
    assert_update_close(xl, c['xl'] + steps[2] * D[:, 0], c['xl'], 2)
    assert_update_close(yl, c['yl'] + steps[2] * D[:, 1], c['yl'], 2)
