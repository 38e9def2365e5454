"""What a run says that it launched."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu

LANES = 65_536   # one wave per SIMD of 256 CUs: up to here runs need no throughput launch


def params(model, n, **over):
    kw = dict(N=n, seed=9, dt=500.0, r_inj=95.0, T_min=1.0)
    kw.update(over)
    return abi.make_params(model, **kw)


@pytest.mark.parametrize("model", (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE))
def test_stats_name_the_launch_that_was_made(engine, model):
    def launched(f, *a):
        f(*a)
        st = engine.last_stats()
        return st.grid_blocks, st.block_threads
    assert launched(engine.run_plain, params(model, LANES)) == (0, 0)
    grid, block = launched(engine.run_plain, params(model, LANES + 1))
    assert grid > 0 and block in (128, 256, 512)
    assert launched(engine.run_plain_noalloc, params(model, 100)) > (0, 0)
    half = [params(model, LANES // 2, first=LANES // 2 * i) for i in range(3)]
    assert launched(engine.run_batch, half[:2]) == (0, 0)
    grid, block = launched(engine.run_batch, half)
    assert grid > 0 and block in (128, 256, 512)


@pytest.mark.parametrize("model", (abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP))
def test_autotuner_times_the_kernel_it_tunes(model):
    """Pilots that fit the tail launches are timed in the throughput kernel all the
    same, and the shape found is a default again afterwards."""
    from geliosphere_amd.engine import Engine
    with Engine(0) as e:
        for kernel, pilots in ((abi.KERNEL_PLAIN, [params(model, 3000)]), (abi.KERNEL_BATCH, [params(model, 500, seed=i) for i in (1, 2)])):
            shape, rate = e.autotune_shape(pilots, kernel)
            assert rate > 0 and e.last_stats().grid_blocks > 0 and e.last_stats().block_threads > 0
            assert e.launch_shape(model, kernel)[:2] == shape[:2]
            e.run_plain(pilots[0]) if kernel == abi.KERNEL_PLAIN else e.run_batch(pilots)
            assert e.last_stats().grid_blocks == 0
