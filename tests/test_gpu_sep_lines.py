"""On-chip separable routine (sep_lines.hpp): mini-batch updates, sequential updates and the error pass against the
FP64 oracle at every plane size, for one plane, odd and even plane counts and partial last bins, with more positions
than one, and each gradient term alone."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.test_gpu_parity import GRAD_TOL, LOSS_TOL, assert_update_close

pytestmark = pytest.mark.gpu

SIZES = [16, 24, 32, 48, 64, 96, 128]


def _upload(ctx, c, steps):
    ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
               step_size=steps, n_scan=(c['npos'], 1))


@pytest.mark.parametrize('n', SIZES)
@pytest.mark.parametrize('nz,binning,steps', [(1, 1, (30.0, 2e-3, 2e-2)), (5, 2, (30.0, 2e-3, 2e-2)),
                                              (4, 1, (30.0, 0.0, 0.0)), (2, 2, (0.0, 2e-3, 0.0)), (3, 1, (0.0, 0.0, 2e-2))])
def test_batched_update_vs_oracle(n, nz, binning, steps):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=binning, npos=5, seed=5 * n + nz, spread=n / 8)
    print('case: separable batch', n, nz, binning, steps, flush=True)
    with lib.Context(0) as ctx:
        _upload(ctx, c, steps)
        e0 = ctx.error_resident()
        err = ctx.run_batched(5)
        V, pr, xl, yl = ctx.download()
    G, P, D, ep = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], c['bin'], c['sig'],
                               c['dx'])
    oerr = ep.sum() / c['npos']
    assert abs(err / oerr - 1) < LOSS_TOL and abs(e0 / oerr - 1) < LOSS_TOL
    oV = c['V'] + steps[0] * np.repeat(G, c['bin'], axis=0)[:nz]
    assert_update_close(V, oV, c['V'], 2)
    assert_update_close(pr, c['probe'] - steps[1] * P, c['probe'], 2)
    assert_update_close(xl, c['xl'] + steps[2] * D[:, 0], c['xl'], 2)
    assert_update_close(yl, c['yl'] + steps[2] * D[:, 1], c['yl'], 2)


@pytest.mark.parametrize('n', SIZES)
def test_sequential_update_vs_oracle(n):
    from mset_amd import lib
    c = small_case(n=n, nz=5, binning=2, npos=4, seed=11 * n, spread=n / 8)
    steps = (30.0, 2e-3, 2e-2)
    print('case: separable sequential', n, flush=True)
    with lib.Context(0) as ctx:
        _upload(ctx, c, steps)
        V, pr, xl, yl, err = ctx.run()
    oV, opr, oxl, oyl, oerr, _ = O.run_tilt(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'],
                                            c['npos'], 1, c['bin'], c['sig'], c['dx'], steps)
    assert abs(err / oerr - 1) < LOSS_TOL
    for new, onew, old in ((V, oV, c['V']), (pr, opr, c['probe']), (xl, oxl, c['xl']), (yl, oyl, c['yl'])):
        assert_update_close(new, onew, old, c['npos'])


@pytest.mark.parametrize('n,npos', [(24, 700), (64, 600), (96, 300)])
def test_slabs_reused_and_grid_capped(n, npos):
    """More positions than resident workgroups: a capped grid gives the same state bit for bit."""
    from mset_amd import lib
    c = small_case(n=n, nz=2, binning=1, npos=npos, seed=n, spread=n / 6)
    print('case: separable slabs', n, npos, flush=True)
    out = []
    for slots in (0, 64):
        with lib.Context(0) as ctx:
            _upload(ctx, c, (30.0, 2e-4, 2e-2))
            ctx.set_slot_limit(slots)
            err = ctx.run_batched(npos)
            out.append(ctx.download() + (err,))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    G, P, D, ep = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], c['bin'], c['sig'],
                               c['dx'])
    assert abs(out[0][4] / (ep.sum() / npos) - 1) < LOSS_TOL
    assert_update_close(out[0][0], c['V'] + 30.0 * G, c['V'], npos)
    assert_update_close(out[0][1], c['probe'] - 2e-4 * P, c['probe'], npos)
