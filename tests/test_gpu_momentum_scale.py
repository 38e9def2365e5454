"""The 1D models carry momenta times 2 K0 dt T0 where that is a number of
ordinary size, and plain momenta (full steps only) where it is not: both against
the oracle, particle by particle, and the kernels against each other."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", (abi.MODEL_1D_BP, abi.MODEL_1D_FP))
# ordinary; 2 K0 dt T0 near 1e-13 and 1e10 (scaled, momenta growing out of the range
# of the single-precision seeds in the first), and beyond both ends
@pytest.mark.parametrize("k0,steps", ((5e22, 0), (5e10, 30_000), (5e32, 3000), (5e-60, 3000), (5e110, 3000)))
def test_scales_against_the_oracle(engine, oracle, model, k0, steps):
    n = 1500 if model == abi.MODEL_1D_BP else 40_000
    p = abi.make_params(model, N=n, seed=19, K0_cm2s=k0, max_steps=steps, T_min=0.05, r_inj=70.0)
    s, recs, nev = engine.run_plain(p, records=True, rec_cap=4 * n)
    rc, o, orecs, on = oracle.run(p, n_threads=0, records=True, rec_cap=4 * n)
    assert rc == 0 and nev == on and s.total_steps == o.total_steps
    assert s.n_step_cap == o.n_step_cap and s.n_nan == o.n_nan and list(s.count) == list(o.count)
    for g, r in zip(recs, orecs):
        assert g.id == r.id and g.t_inj == pytest.approx(r.t_inj, rel=1e-12)
        assert g.t_exit == pytest.approx(r.t_exit, rel=1e-9) and g.r == pytest.approx(r.r, rel=1e-9)
    assert bytes(s) == bytes(engine.run_plain_noalloc(p))
    b = engine.run_batch([p, abi.make_params(model, N=500, seed=20)])
    assert bytes(b[0]) == bytes(s)
