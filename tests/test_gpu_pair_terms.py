"""Lennard-Jones pair sums where 1/r^2 leaves the range in which the kernels'
reciprocal and the division agree on their own: coincident atoms, r^2 that
underflows or overflows, atoms at an infinite distance.  The sums must be the
division's in every case, NaN where it gives NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")


def _pair(a, b):
    d = a - b
    s = np.float64(1.0) / ((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2])
    s2 = s * s
    return 4.0 * (s2 * (s2 * s2) - s * s2)


def _same(got, want):
    return got == want or (np.isnan(got) and np.isnan(want))


@pytest.mark.parametrize("n,lanes", [(5, 2), (13, 4), (31, 8)])
@pytest.mark.parametrize("shift", [0.0, 1e-162, 1e-155, 1e-120, 1e-110, 1e110, 1e116, 1e130, 1e160, 1e200])
def test_pair_sums_at_the_ends_of_the_range(gpu_ctx_factory, n, lanes, shift):
    import oracle as O
    print("case", n, lanes, shift, flush=True)
    ctx = gpu_ctx_factory()
    s = ctx.add_set(S.make_params(system=S.LJ, n=n, lanes=lanes, method=S.SAD, method_param=0.05, move_param=0.1,
                                  energy_bin=0.01, has_max_e=1, max_e=0.0), np.array([7], np.uint64), geom=3.0)
    ctx.init()
    st, bins = ctx.download_raw(s)
    x = ctx.coords(s, 0).reshape(3, n).copy()
    x[:, 2] = 0.0
    x[:, n - 1] = (shift, 0.0, 0.0)  # atom 2 at the origin, the last one `shift` from it
    ctx.upload_raw(s, st, bins, coords=x.reshape(-1))
    rng = O.RNG(state=tuple(int(v) for v in st[0]["rng"]))
    E = float(st[0]["E"])

    def total(part):
        while len(part) > 1:
            part = part[0::2] + part[1::2]
        return float(part[0])

    with np.errstate(all="ignore"):
        part = np.zeros(lanes)
        for i in range(n):
            for j in range(i):
                part[i % lanes] += _pair(x[:, i], x[:, j])
        assert _same(ctx.compute_energy(s, 0), total(part))
        for _ in range(4 * n):
            e = ctx.plan_move(s, 0, 0.3)
            w = rng.uniform_index(n)
            f = x[:, w].copy()
            t = f + np.array([rng.uniform_f64(-0.3, 0.3) for _ in range(3)])
            tt, ff = ((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2] for v in (t, f))
            if tt > 9.0 and tt > ff:
                assert e is None
                continue
            part = np.zeros(lanes)
            for j in range(n):
                if j != w:
                    part[j % lanes] += _pair(x[:, j], t) - _pair(x[:, j], f)
            assert _same(e, E + total(part)), (w, e)
