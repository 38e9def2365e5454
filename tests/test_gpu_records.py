"""Exit records ordered on the device against the same run in launches of so few
particles that the host orders them: the same bytes."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu

CASES = [
    ("1D B-p, 513 records and an odd shard", abi.MODEL_1D_BP, 513, 400, dict(first=7, dt=500.0)),
    ("1D B-p, a tile of the sums and one more", abi.MODEL_1D_BP, 4097, 500, dict(dt=500.0, r_inj=60.0)),
    ("1D F-p, several crossings of some particles", abi.MODEL_1D_FP, 2_000_001, 400_000,
     dict(first=11, dt=500.0, V_kms=10.0, K0_cm2s=1e24)),
    ("SolarProp, ids beyond 2^32", abi.MODEL_2D_SOLARPROP, 1500, 500, dict(first=(1 << 33) + 5, dt=500.0, r_inj=30.0)),
]


@pytest.mark.parametrize("label,model,n,chunk,extra", CASES, ids=[c[0] for c in CASES])
def test_device_order_equals_host_order(engine, label, model, n, chunk, extra):
    p = abi.make_params(model, N=n, seed=23, **extra)
    cap = 200_000
    s, recs, nev = engine.run_plain(p, records=True, rec_cap=cap)
    got = [bytes(r) for r in recs]
    assert nev == len(got) > 512
    engine.set_plain_limits(max_chunk=chunk)
    try:
        s2, recs2, nev2 = engine.run_plain(p, records=True, rec_cap=cap)
    finally:
        engine.set_plain_limits()
    assert nev2 == nev and nev * chunk / n < 512 and [bytes(r) for r in recs2] == got
    ids = [r.id for r in recs]
    assert ids == sorted(ids)
    if model == abi.MODEL_1D_FP:
        assert len(set(ids)) < len(ids)
        assert all(a.id < b.id or a.sumac <= b.sumac for a, b in zip(recs, recs[1:]))
    # a capacity below the number of events: its first records
    for k in (1, 512, nev - 1):
        _, r, m = engine.run_plain(p, records=True, rec_cap=k)
        assert m == nev and [bytes(x) for x in r] == got[:k]
