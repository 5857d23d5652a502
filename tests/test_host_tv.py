"""Scratch of the TV regulariser, on the CPU with a stand-in HIP runtime: less of it where the device is nearly full."""
import pytest

from tests import fake_hip


@pytest.fixture(scope='session')
def tmp(tmp_path_factory):
    return tmp_path_factory.mktemp('fake_hip')


def test_runs_on_four_volumes_where_seven_do_not_fit(tmp):
    fake_hip.run(tmp, '''
        ctx = lib.Context(0)
        v = np.ones((6, 8, 12), np.float32)
        ctx.tv(v, 0.5, 3)
        assert len(launches('k_tv_iterate')) == 3 and not launches('k_tv_project')
        big = np.ones((12, 8, 12), np.float32)
        fake.fake_reset()
        fake.fake_fail_malloc(7 * big.size * 4)
        for _ in range(2):
            ctx.tv(big, 0.5, 3)
        assert len(launches('k_tv_dual_residual')) == len(launches('k_tv_project')) == 6 and not launches('k_tv_iterate')
        fake.fake_reset()
        fake.fake_fail_malloc(0)
        ctx.tv(big, 0.5, 3)
        assert len(launches('k_tv_iterate')) == 3
    ''')
