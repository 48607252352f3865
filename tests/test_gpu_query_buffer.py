"""The buffer that a context keeps between batches of queries: large ones go back, and a count
whose bytes do not fit 64 bits is refused as any that cannot be allocated."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free():
    import torch
    return torch.cuda.mem_get_info()[0]


def test_gpu_query_buffer_goes_back(gpu):
    cm = gpu
    cl = cm.make_plummer(20000, seed=2)
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        x = np.linspace(0.05, 3.0, 1000)
        first = ctx.potential_at(x)
        before = _free()
        many = ctx.potential_at(np.tile(x, 20000))                # 320 MB of inputs and outputs
        assert _free() > before - (64 << 20)
        assert np.array_equal(many.reshape(20000, 1000)[[0, 9999, 19999]], np.tile(first, (3, 1)))
        assert np.array_equal(ctx.potential_at(x), first)
        d = ctx.download(fields=["E", "J"])
        a = ctx.apsides(1, d["E"][1:101], d["J"][1:101])
        assert np.all(a["rp"] <= a["ra"])


@pytest.mark.parametrize("count", [2 ** 59, 2 ** 60, 2 ** 62, 2 ** 63 - 1])
def test_gpu_query_count_beyond_64_bits_is_refused(gpu, count):
    cm = gpu
    cl = cm.make_plummer(1000, seed=2)
    x = np.linspace(0.05, 3.0, 8)
    y = np.zeros(8)
    p = C.POINTER(C.c_double)
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        rc = cm.lib.cmcg_potential_at(ctx.h, C.c_int64(count), x.ctypes.data_as(p), y.ctypes.data_as(p))
        assert rc == -13                                            # CMCG_E_NOMEM
        assert np.all(ctx.potential_at(x) < 0.0)
