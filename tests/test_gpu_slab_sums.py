"""Sum of the positions' gradient slabs: remainders of the loads in flight (groups of 32 or 8 slabs and single
ones) and both sides of the size from which a thread sums four floats."""
import numpy as np
import pytest

from tests.cases import small_case

pytestmark = pytest.mark.gpu


# L n^2 = 2^16 (one float per thread) and one plane more (four)
@pytest.mark.parametrize('npos', [1, 7, 9, 45])
@pytest.mark.parametrize('n,nz', [(16, 3), (64, 16), (64, 17)])
def test_slab_sum_matches_positions(n, nz, npos):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=1, npos=npos, seed=n + nz, spread=n / 6)
    print('case: slab sum', n, nz, npos, flush=True)
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=1,
                   n_scan=(npos, 1))
        whole = ctx.grad()[0]
        single = np.stack([ctx.grad(k, 1)[0] for k in range(npos)]).astype(np.float64)
    # npos - 1 roundings of partial sums, each at most the sum of the magnitudes
    bound = npos * 2.0 ** -24 * np.abs(single).sum(0)
    assert (np.abs(whole - single.sum(0)) <= bound).all()
