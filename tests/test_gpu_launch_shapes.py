"""Launch shapes: what a caller sets is what runs, for few particles too; shapes from
the autotuner's cache are defaults."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu

MODELS = (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE)


def params(model, n, **over):
    kw = dict(N=n, seed=9, dt=500.0, r_inj=95.0, T_min=1.0)
    kw.update(over)
    return abi.make_params(model, **kw)


@pytest.mark.parametrize("model", MODELS)
def test_a_shape_that_is_set_is_the_one_that_runs(engine, model):
    p = params(model, 100_000)
    want = engine.run_plain(p)[0]
    cus = {}
    try:
        for shape in ((256, 1, 64), (128, 6, 16), (512, 1, 0), (0, 3, 0)):
            engine.set_launch_shape(model, abi.KERNEL_PLAIN, *shape)
            used = engine.launch_shape(model, abi.KERNEL_PLAIN)
            assert bytes(engine.run_plain(p)[0]) == bytes(want)
            st = engine.last_stats()
            assert st.block_threads == used[0] and st.grid_blocks % used[1] == 0
            cus[shape] = st.grid_blocks // used[1]
        assert len(set(cus.values())) == 1   # always blocks per CU times the CUs
    finally:
        engine.set_launch_shape(model, abi.KERNEL_PLAIN)


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("counts", ((1, 0, 63, 2000), (40_000, 1, 33_000)))
def test_batches_in_a_shape_that_is_set(engine, model, counts):
    """Few particles through the throughput kernel, by simulations: lanes that move on
    to the next one, and its hand-on to tail launches."""
    sims = [params(model, n, seed=20 + i, r_inj=60.0 + 5 * i, T_min=0.3) for i, n in enumerate(counts)]
    want = [bytes(engine.run_plain_noalloc(p)) for p in sims]
    assert [bytes(o) for o in engine.run_batch(sims)] == want
    for shape in ((256, 1, 16), (128, 2, 64), (512, 1, 256)):
        engine.set_launch_shape(model, abi.KERNEL_BATCH, *shape)
        try:
            outs = engine.run_batch(sims)
            assert engine.last_stats().block_threads == shape[0]
        finally:
            engine.set_launch_shape(model, abi.KERNEL_BATCH)
        assert [bytes(o) for o in outs] == want, shape
    assert [bytes(o) for o in engine.run_batch(sims)] == want
