"""Launches of the host logic, on the CPU with a stand-in HIP runtime: grids and routes that a result does not show."""
import pytest

from tests import fake_hip


@pytest.fixture(scope='session')
def tmp(tmp_path_factory):
    return tmp_path_factory.mktemp('fake_hip')


@pytest.mark.parametrize('n,nz,binning,method', [(24, 24, 1, 'SSET'), (64, 48, 48, 'MSET'), (24, 20, 6, 'MSET')])
def test_object_step_has_a_thread_per_4_voxels(tmp, n, nz, binning, method):
    fake_hip.run(tmp, '''
        ctx = lib.Context(0)
        upload(ctx, %d, %d, 3, binning=%d)
        fake.fake_reset()
        ctx.run_batched(3, method=lib.METHOD_%s)
        (name, gx, gy, threads, _), = launches('update_volume') or launches('k_volume<true')
        assert 4 * gx * gy * threads >= %d, (name, gx, gy, threads)
    ''' % (n, nz, binning, method, n * n * nz))
