"""Scratch of the TV regulariser, on the CPU with a stand-in HIP runtime: less of it where the device is nearly full,
and given back where something else needs the room."""
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


# what comes after the TV call on a device that its kept scratch fills
@pytest.mark.parametrize('what', ['upload', 'run_batched', 'rotate_resident', 'rotate', 'tv'])
def test_kept_scratch_makes_room(tmp, what):
    fake_hip.run(tmp, '''
        def call(ctx):
            return dict(upload=lambda: upload(ctx, 64, 24, 40), run_batched=lambda: ctx.run_batched(40),
                        rotate_resident=lambda: ctx.rotate_resident((10., 20., 30.), False),
                        rotate=lambda: ctx.rotate(np.ones((64, 64, 64), np.float32), physics_R, 11.0),
                        tv=lambda: ctx.tv(np.ones((16, 64, 64), np.float32), 0.5, 1))[%r]()

        a, b = np.cos(0.5), np.sin(0.5)
        physics_R = np.array([[a, 0, b], [0, 1, 0], [-b, 0, a]]) @ np.array([[1, 0, 0], [0, a, b], [0, -b, a]])
        need = []
        for with_tv in (False, True):
            ctx = lib.Context(0)
            upload(ctx, 64, 24, 4)
            if %r != 'upload':
                upload(ctx, 64, 24, 40)
            if with_tv:
                ctx.tv(np.ones((24, 64, 64), np.float32), 0.5, 1)
                kept = fake.fake_bytes()
                # room for the call without the scratch, and for nothing beside it
                fake.fake_device_memory(max(need[0], kept))
            else:
                fake.fake_reset()
            call(ctx)
            need.append(fake.fake_peak())
            ctx.close()
    ''' % (what, what))


def test_allocations_that_never_fit_are_refused_and_leave_the_context_usable(tmp):
    fake_hip.run(tmp, '''
        ctx = lib.Context(0)
        upload(ctx, 64, 24, 4)
        ctx.tv(np.ones((24, 64, 64), np.float32), 0.5, 1)
        fake.fake_device_memory(fake.fake_bytes())
        try:
            upload(ctx, 64, 24, 4000)
            raise SystemExit('fitted')
        except lib.MsetError as e:
            assert e.code == lib.MSET_ENOMEM
        fake.fake_device_memory(288 << 30)
        upload(ctx, 64, 24, 4)
        ctx.run_batched(4)
        ctx.tv(np.ones((24, 64, 64), np.float32), 0.5, 1)
    ''')


@pytest.mark.parametrize('what', ['recon', 'context'])
def test_scratch_of_another_context_is_left_alone(tmp, what):
    """it may be in use on another thread: what this thread called last says nothing about it"""
    fake_hip.run(tmp, '''
        a = lib.Context(0)
        b = lib.Context(0)
        a.tv(np.ones((24, 64, 64), np.float32), 0.5, 1)
        kept = fake.fake_bytes()
        fake.fake_device_memory(kept + 1000)
        try:
            if %r == 'recon':
                recon(64, 16, 4)
            else:
                upload(b, 64, 24, 4)
            raise SystemExit('fitted')
        except lib.MsetError as e:
            assert e.code == lib.MSET_ENOMEM
        assert fake.fake_bytes() >= kept, (fake.fake_bytes(), kept)
    ''' % what)
