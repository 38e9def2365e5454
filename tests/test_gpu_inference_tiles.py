"""Inference picks its row tile by the number of rows: every tile, at its edges
and across the switches between tiles, must give each query the same bits, and
the inputs may share memory with the outputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(members, layers, n_in):
    from geliosphere_amd.surrogate import Surrogate
    s = Surrogate(0, seed=3, n_members=members, n_hidden_layers=layers, n_inputs=n_in, std_limit=0.02)
    s.set_normalization(np.linspace(-0.2, 0.3, n_in), np.linspace(0.8, 1.7, n_in), np.full(n_in, -1.5), np.full(n_in, 1.5))
    return s


@pytest.mark.parametrize("members,layers,n_in", [(4, 4, 8), (1, 1, 5), (3, 2, 17), (5, 7, 32)])
def test_every_tile_gives_the_same_bits(members, layers, n_in):
    s = make(members, layers, n_in)
    # rows at which the tile changes (16 to 32, to 64, to 128), and one chunk and a bit
    edges = [r // members for r in (16 * 256, 32 * 256, 64 * 2048)]
    sizes = sorted({1, 15, 16, 17, 33, 129, 65_537, *(e + d for e in edges for d in (0, 1, 127))})
    x = np.random.default_rng(8).normal(0, 1, (max(sizes), n_in)).astype(np.float32)
    mean, sd, fb = s.predict(x)
    assert np.all(np.isfinite(mean)) and 0 < np.count_nonzero(fb & 0x2) < len(x)
    for n in sizes:
        at = len(x) - n                    # other rows than the first
        m, d, f = s.predict(x[at:])
        assert np.array_equal(m, mean[at:]) and np.array_equal(d, sd[at:]) and np.array_equal(f, fb[at:]), n
    # the training forward pass (a kernel of its own) on the same rows: zero loss on
    # its own prediction
    if members == 1:
        _, loss = s.gradients(x[:700], mean[:700], np.ones_like(mean[:700]))
        assert loss[0] == 0.0


def test_flags_follow_the_rule_on_special_values():
    s = make(3, 2, 8)
    x = np.zeros((9, 8), np.float32)
    x[0, 3], x[1, 0], x[2, 7], x[3, 1], x[4, 2], x[5, 5] = np.nan, np.inf, -np.inf, 1.5, np.nextafter(np.float32(1.5), np.float32(2)), -1.6
    mean, sd, fb = s.predict(x)
    assert [int(f) & 2 for f in fb] == [2, 2, 2, 0, 2, 2, 0, 0, 0]
    sel = [c for c in range(30) if (s.cfg.std_outputs >> c) & 1]
    assert [int(f) & 1 for f in fb] == [int(np.any(~(sd[r, sel] <= np.float32(s.cfg.std_limit)))) for r in range(9)]
    assert np.all(np.isnan(mean[0]))


def test_device_inputs_may_share_memory_with_the_outputs():
    from types import SimpleNamespace

    from geliosphere_amd.devmem import DeviceArray
    s = make(4, 4, 8)
    x = np.random.default_rng(9).normal(0, 1, (300, 8)).astype(np.float32)
    mean, sd, fb = s.predict(x)
    block = np.zeros((300, 30), np.float32)
    block.reshape(-1)[:x.size] = x.reshape(-1)
    b = DeviceArray.from_host(block)
    view = SimpleNamespace(shape=x.shape, dtype=x.dtype, ptr=b.ptr)
    sd_d = DeviceArray((300, 30), np.float32)
    m_d, _, fb_d = s.predict_device(view, b, sd_d)
    assert np.array_equal(m_d.to_host(), mean) and np.array_equal(sd_d.to_host(), sd) and np.array_equal(fb_d.to_host(), fb)


@pytest.mark.parametrize("n", (1, 4096, 4097, 8192, 8193, 16_385, 24_577))
def test_host_blocks_equal_device_call(n):
    """Host calls go in blocks of 8,192 rows through two halves of pinned memory
    (inputs read there up to 4,096 rows of a block, copied beyond); outputs that
    share memory with the inputs take the copies."""
    import ctypes

    from geliosphere_amd.devmem import DeviceArray
    from geliosphere_amd.surrogate import lib
    s = make(4, 4, 8)
    x = np.random.default_rng(n).normal(0, 1, (n, 8)).astype(np.float32)
    sd_d = DeviceArray((n, 30), np.float32)
    m_d, _, f_d = s.predict_device(DeviceArray.from_host(x), None, sd_d)
    want = m_d.to_host(), sd_d.to_host(), f_d.to_host()
    for a, b in zip(s.predict(x), want):
        assert np.array_equal(a, b)
    m, none, f = s.predict(x, want_sd=False)
    assert none is None and np.array_equal(m, want[0]) and np.array_equal(f, want[2])
    shared = np.zeros((n, 30), np.float32)
    shared.reshape(-1)[-x.size:] = x.reshape(-1)
    pf = ctypes.POINTER(ctypes.c_float)
    px = ctypes.cast(shared.ctypes.data + 4 * (shared.size - x.size), pf)
    assert lib().gs_surrogate_predict(s._h, px, n, shared.ctypes.data_as(pf), None, None) == 0
    assert np.array_equal(shared, want[0])
