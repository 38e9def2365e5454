"""Runs under a step cap, where lifetimes hardly differ: launches of the shape's size,
and no tail launches for caps of less than 512 steps."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE))
@pytest.mark.parametrize("max_steps", (510, 511, 512, 513, 16_383, 16_384))
def test_capped_run_equals_throughput_kernel(engine, model, max_steps):
    p = abi.make_params(model, N=70_001, seed=31, first=5, dt=500.0, r_inj=30.0, T_min=0.3, max_steps=max_steps)
    s = engine.run_plain(p)[0]
    assert s.n_particles == 70_001 and bytes(s) == bytes(engine.run_plain_noalloc(p))


def test_small_caps_do_not_wait_for_tail_launches():
    """A quarter of the steps in 0.39 of the time with the shipped launch shapes (0.49
    with two waves a SIMD and tail launches)."""
    import os

    import geliosphere_amd
    from geliosphere_amd.engine import Engine
    with Engine(0) as engine:
        engine.autotune_load(os.path.join(os.path.dirname(geliosphere_amd.__file__), "data", "autotune.txt"))

        def best(cap):
            ms = []
            for k in range(6):
                engine.run_plain(abi.make_params(abi.MODEL_1D_BP, N=3_000_000, seed=k, max_steps=cap))
                ms.append(engine.last_stats().kernel_ms)
            return min(ms)
        short, longer = best(500), best(2000)
        assert short < 0.44 * longer, (short, longer)
