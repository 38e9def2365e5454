"""Device predictions go to the network kernel in launches of up to 65,536 rows, of
which it takes tiles of 16, 32, 64 or 128 (host predictions, in blocks of 8,192 rows,
reach the largest with more than 16 members only): every query's bits at each switch,
remainder and launch, whatever the tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members,layers,n_in", [(4, 4, 8), (1, 1, 5), (3, 2, 17), (5, 7, 32)])
def test_every_tile_and_launch_gives_the_same_bits(members, layers, n_in):
    from types import SimpleNamespace

    from geliosphere_amd.devmem import DeviceArray
    from geliosphere_amd.surrogate import Surrogate
    s = Surrogate(0, seed=3, n_members=members, n_hidden_layers=layers, n_inputs=n_in, std_limit=0.02)
    s.set_normalization(np.linspace(-0.2, 0.3, n_in), np.linspace(0.8, 1.7, n_in), np.full(n_in, -1.5), np.full(n_in, 1.5))
    # rows at which the tile changes to 32, 64 and 128, the launch's 65,536, two launches
    edges = [r // members for r in (16 * 256, 32 * 256, 64 * 2048)] + [65_536, 131_072]
    sizes = sorted({1, 17, *(e + d for e in edges for d in (-1, 0, 1, 65, 127)), 65_536 + 128})
    most = max(sizes)
    x = np.random.default_rng(8).normal(0, 1, (most, n_in)).astype(np.float32)
    xd = DeviceArray.from_host(x)
    sd, mean = DeviceArray((most, 30), np.float32), None
    m_d, _, f_d = s.predict_device(xd, mean, sd)
    mean, spread, flags = m_d.to_host(), sd.to_host(), f_d.to_host()
    assert np.all(np.isfinite(mean)) and 0 < np.count_nonzero(flags & 2) < most
    for n in sizes:
        at = most - n   # other rows than the first
        view = SimpleNamespace(shape=(n, n_in), dtype=x.dtype, ptr=type(xd.ptr)(xd.ptr.value + 4 * n_in * at))
        sd_n = DeviceArray((n, 30), np.float32)
        m, _, f = s.predict_device(view, None, sd_n)
        assert np.array_equal(m.to_host(), mean[at:]) and np.array_equal(sd_n.to_host(), spread[at:]), n
        assert np.array_equal(f.to_host(), flags[at:]), n
    # the smallest tile on the same rows, a few at a time
    for at in (0, 777, most - 16):
        assert np.array_equal(s.predict(x[at:at + 16])[0], mean[at:at + 16])
