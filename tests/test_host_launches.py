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


@pytest.mark.parametrize('engine', ['AUTO', 'ALT_SHAPE', 'GENERAL'])
def test_forward_grid_does_not_depend_on_earlier_calls(tmp, engine):
    """the error pass of one position size after batched calls of another, and after another engine's"""
    fake_hip.run(tmp, '''
        fake.fake_occupancy(b'k_batch<256, 1', 3)
        def grid(before):
            ctx = lib.Context(0)
            for n, e in before:
                upload(ctx, n, 2, 5)
                ctx.set_engine(e)
                ctx.run_batched(5)
            upload(ctx, 256, 2, 700)
            ctx.set_engine(lib.ENGINE_%s)
            fake.fake_reset()
            ctx.error_resident()
            (name, gx, _, threads, _), = launches('k_fwd<256')
            planes = fake.fake_bytes()
            ctx.close()
            return name, gx, threads
        fresh = grid(())
        assert fresh[1] == 512                   # two workgroups on each of 256 CUs
        for before in (((64, 0),), ((24, 0),), ((64, 2),), ((256, 2),), ((256, 1), (48, 0)), ((256, 0),)):
            assert grid(before) == fresh, before
    ''' % engine)


# the general routine keeping fewer workgroups than the separable one, and more
@pytest.mark.parametrize('n,general,separable', [(24, 5, 6), (16, 16, 19), (64, 3, 2), (96, 1, 1), (128, 1, 9)])
def test_batch_slots_covers_the_kernels_of_a_batched_call(tmp, n, general, separable):
    fake_hip.run(tmp, '''
        n, g, s = %d, %d, %d
        fake.fake_occupancy(b'k_batch<%%d, 0' %% n, g)
        fake.fake_occupancy(b'k_batch<%%d, 4' %% n, g)      # the small workgroup for many positions
        fake.fake_occupancy(b'k_sep_batch<%%d' %% n, s)
        slots = lib.batch_slots(n)
        per_cu = max(g, s) if n < 128 else g
        assert slots == 256 * per_cu, slots
        ctx = lib.Context(0)
        npos = 256 * max(g, s) + 3 if n < 32 else 600
        for separable in (True, False):
            upload(ctx, n, 2, npos, separable=separable)
            fake.fake_reset()
            ctx.run_batched(npos)
            (name, gx, _, _, _), = launches('k_sep_batch') + launches('k_batch')
            assert gx <= slots, (name, gx, slots)
            if npos > slots:
                assert gx == 256 * (s if 'sep' in name else g), (name, gx)
    ''' % (n, general, separable))


@pytest.mark.parametrize('P,vol', [(32, 16), (64, 32), (128, 32), (256, 16)])
def test_serving_footprint_covers_what_a_job_allocates(tmp, P, vol):
    fake_hip.run(tmp, '''
        from mset_amd import serve
        fake.fake_occupancy(b'k_batch<', 2)
        fake.fake_occupancy(b'k_sep_batch<', 5)
        spec = serve.JobSpec(job_id=0, vol=%d, P=%d, tilts=[0.0, 10.0], scan=16, seed=1)
        fake.fake_reset()
        r = serve.make_recon(spec)
        for _ in range(2):
            r.iterate(1, 128, True, True)
        r.snapshot()
        assert fake.fake_peak() <= serve.footprint_bytes(spec, lib.batch_slots(spec.P)), (fake.fake_peak(), serve.footprint_bytes(spec, lib.batch_slots(spec.P)))
    ''' % (vol, P))


@pytest.mark.parametrize('n,npos,threads', [(16, 8, 64), (24, 8, 128), (32, 8, 128), (48, 8, 384), (64, 256, 512), (64, 257, 256),
                                            (96, 8, 1024), (128, 8, 512), (256, 8, 256)])
def test_alternative_shape(tmp, n, npos, threads):
    fake_hip.run(tmp, '''
        ctx = lib.Context(0)
        upload(ctx, %d, 2, %d)
        ctx.set_engine(lib.ENGINE_ALT_SHAPE)
        fake.fake_reset()
        ctx.run_batched(%d)
        (name, _, _, threads, _), = launches('k_batch')
        assert threads == %d, (name, threads)
    ''' % (n, npos, npos, threads))


def test_many_positions_at_24_take_the_small_workgroup(tmp):
    """one position more than the default shape keeps resident; the grid is that of the shape that is launched"""
    fake_hip.run(tmp, '''
        fake.fake_occupancy(b'k_batch<24, 0', 3)
        fake.fake_occupancy(b'k_batch<24, 4', 7)
        for npos, shape, threads in ((3 * 256, 0, 192), (3 * 256 + 1, 4, 64)):
            ctx = lib.Context(0)
            upload(ctx, 24, 2, npos, separable=False)
            for wv in (lib.EXIT_WAVES_STORE, lib.EXIT_WAVES_CHECKPOINT):
                ctx.set_exit_waves(wv)
                fake.fake_reset()
                ctx.run_batched(npos)
                ctx.grad()
                for name, gx, _, nt, _ in launches('k_batch<'):
                    assert 'k_batch<24, %%d' %% shape in name and nt == threads and gx == npos, (name, gx, nt)
            fake.fake_reset()
            ctx.error_resident()
            (name, gx, _, nt, _), = launches('k_fwd<')
            assert 'k_fwd<24, %%d' %% shape in name and nt == threads and gx == npos, (name, gx, nt)
            ctx.run_batched(700)                     # the launches of a pass decide, not the positions of the tilt
            fake.fake_reset()
            ctx.run_batched(700)
            assert all(nt == 192 for _, _, _, nt, _ in launches('k_batch<'))
            ctx.close()
        r = recon(24, 16, (500, 600), angles=(0., 10.))
        r.set_engine(lib.ENGINE_GENERAL)
        fake.fake_reset()
        r.error_pass()
        (name, gx, _, nt, _), = launches('k_fwd<')
        assert 'k_fwd<24, 4' in name and nt == 64 and gx == 1100, (name, gx, nt)
    '''.replace('%%', '%'))


def test_sequential_kernels_are_the_ones_that_are_reached(tmp):
    """the one-position separable kernel is built where the sequential path launches it, and nowhere else"""
    fake_hip.run(tmp, '''
        ctx = lib.Context(0)
        reached = set()
        for n in (16, 24, 32, 48, 64, 96, 128, 256):
            upload(ctx, n, 3, 2)
            fake.fake_reset()
            ctx.run_resident()
            reached |= {name for name, *_ in launches('k_sep_plain')}
            assert bool(launches('k_line_pass')) == (n >= 96)
        built = {l for l in fake.fake_kernels().decode().splitlines() if 'k_sep_plain' in l}
        assert built == reached and len(built) == 5, built ^ reached
    ''')
