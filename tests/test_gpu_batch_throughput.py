"""The batch's throughput kernels with several simulations to a launch (groups of more
particles than tail launches take alone): lanes that move from one simulation to the
next, hand-on by simulation, and the order in which the queue hands particles out."""
import pytest

from geliosphere_amd import abi
from geliosphere_amd import engine as E

pytestmark = pytest.mark.gpu

MODELS = (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE)
COUNTS = (30_000, 1, 45_000, 0, 17_001, 2)   # 92,004 > 65,536


def sims_of(model, counts, seed=60):
    return [abi.make_params(model, N=n, seed=seed + i, first=3 * i, dt=500.0 if i % 2 else 300.0, r_inj=70.0 + 5 * i,
                            T_min=0.3, K0_cm2s=5e22 * (1 + i / 10), tilt_deg=10.0 + 9 * i, theta_deg=60.0 + 15 * i,
                            polarity=1.0 if i % 3 else -1.0, max_steps=0 if i != 4 else 4001)
            for i, n in enumerate(counts)]


@pytest.mark.parametrize("model", MODELS)
def test_several_simulations_of_a_model(engine, model):
    sims = sims_of(model, COUNTS)
    outs = engine.run_batch(sims)
    assert engine.last_stats().grid_blocks > 0   # the throughput kernel ran
    for p, o in zip(sims, outs):
        assert o.n_particles == p.n_particles and bytes(o) == bytes(engine.run_plain_noalloc(p)), p.n_particles


def test_several_simulations_of_every_model(engine):
    sims = [s for four in zip(*(sims_of(m, COUNTS, seed=80 + m) for m in MODELS)) for s in four]
    want = [bytes(engine.run_plain_noalloc(p)) for p in sims]
    for mode in (E.ORDER_ENERGY, E.ORDER_ID):
        engine.set_order(mode)
        try:
            outs = engine.run_batch(sims)
        finally:
            engine.set_order(E.ORDER_ENERGY)
        assert [bytes(o) for o in outs] == want


def test_more_simulations_than_one_launch_holds(engine):
    sims = [abi.make_params(abi.MODEL_1D_BP, N=68 + (i % 9), seed=50_000 + i, r_inj=60.0 + i % 30,
                            K0_cm2s=5e22 * (1 + (i % 5) / 10.0)) for i in range(1100)]
    outs = engine.run_batch(sims)
    assert engine.last_stats().grid_blocks > 0
    assert all(o.n_particles == p.n_particles for p, o in zip(sims, outs))
    for i in (*range(0, 1024, 31), *range(1020, 1100, 7)):
        assert bytes(outs[i]) == bytes(engine.run_plain_noalloc(sims[i])), i


@pytest.mark.parametrize("model", MODELS[1:])
def test_queue_order_does_not_change_results(engine, model):
    p = abi.make_params(model, N=90_001, seed=7, first=11, dt=500.0, r_inj=80.0, T_min=0.1)
    want = bytes(engine.run_plain(p)[0])
    assert engine.last_stats().grid_blocks > 0
    engine.set_order(E.ORDER_ID)
    try:
        assert bytes(engine.run_plain(p)[0]) == want
    finally:
        engine.set_order(E.ORDER_ENERGY)
