"""The device memory that ordering exit records takes is given back after a large run,
and later runs with records go on as before."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu


def test_large_runs_give_their_record_buffers_back():
    import ctypes
    import time

    from geliosphere_amd.devmem import hip
    from geliosphere_amd.engine import Engine, lib

    def free_memory():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def run(e, p, buf):
        s, n = abi.GsSpectrum(), ctypes.c_uint64(0)
        assert lib().gs_run_plain(e._ctx, ctypes.byref(p), ctypes.byref(s), buf, len(buf) if buf else 0, ctypes.byref(n)) == 0
        return n.value, free_memory()
    with Engine(0) as e:
        p = abi.make_params(abi.MODEL_1D_BP, N=6_000_000, seed=3, r_inj=99.5, T_min=1.0)
        small = abi.make_params(abi.MODEL_1D_BP, N=20_000, seed=4, r_inj=99.5, T_min=1.0)
        _, before = run(e, p, None)   # grows what a run without records needs
        buf = (abi.GsExitRecord * 6_000_000)()
        n, after = run(e, p, buf)
        assert n > 5_600_000          # 48 bytes each, and 4 per particle
        until = time.monotonic() + 5.0   # (the runtime may give the memory back a moment later)
        while before - after >= 64 << 20 and time.monotonic() < until:
            time.sleep(0.05)
            after = free_memory()
        assert before - after < 64 << 20
        first = [bytes(buf[i]) for i in range(0, n, 100_003)]
        few = (abi.GsExitRecord * 20_000)()
        k, _ = run(e, small, few)
        ids = [r.id for r in few[:k]]
        assert k > 512 and ids == sorted(ids)
        assert run(e, p, buf)[0] == n and [bytes(buf[i]) for i in range(0, n, 100_003)] == first
