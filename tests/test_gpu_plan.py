"""What sadmc_plan_move hands back when the wall refuses the move."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")


@pytest.mark.parametrize("n,lanes", [(13, 4), (31, 8)])
def test_a_refused_move_has_no_energy(gpu_ctx_factory, n, lanes):
    print("case refused plan", n, lanes, flush=True)
    ctx = gpu_ctx_factory()
    s = ctx.add_set(S.make_params(system=S.LJ, n=n, lanes=lanes, method=S.SAD, method_param=0.05, move_param=0.1,
                                  energy_bin=0.01, has_max_e=1, max_e=0.0), np.array([3], np.uint64), geom=3.0)
    ctx.init()
    made = refused = 0
    for _ in range(120):
        e, some = C.c_double(np.nan), C.c_int32(-1)
        assert S.lib().sadmc_plan_move(ctx.h, s, 0, 2.0, C.byref(e), C.byref(some)) == 0
        if some.value:
            made += 1
            assert e.value != 0.0
        else:
            refused += 1
            assert np.float64(e.value).tobytes() == np.float64(0.0).tobytes()
    assert made and refused
