"""How walkers share wavefronts must not show in them: the number of walkers
per wave (set by the size of the set), idle lane groups, energies recomputed
by the whole wave, and walkers of one wave standing at different move numbers.
Every comparison is bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")

LJ13 = dict(system=S.LJ, n=13, lanes=4, method=S.SAD, method_param=0.05, move_param=0.1, energy_bin=0.01,
            has_max_e=1, max_e=0.0)
WCA32 = dict(system=S.WCA, n=32, lanes=8, method=S.SAMC, method_param=1e4, move_param=0.05, energy_bin=0.05,
             has_max_e=1, max_e=80.0)
ISING = dict(system=S.ISING, n=8, ising_init=1, method=S.SAD, method_param=1.0)


def _run(factory, kw, walkers, geom, moves):
    ctx = factory()
    s = ctx.add_set(S.make_params(**kw), np.arange(walkers, dtype=np.uint64) + 11, geom=geom)
    ctx.init()
    ctx.run(moves)
    return ctx, s


@pytest.mark.parametrize("kw,geom,sizes", [
    # 64 / lanes walkers a wave from 1024 (Ising 2048) waves on, fewer below
    pytest.param(LJ13, 2.5, (5, 2049, 17000), id="lj13"),
    pytest.param(dict(LJ13, n=45, lanes=8), 3.5, (3, 1500, 8200), id="lj45-clamped-slots"),
    pytest.param(WCA32, 4.2, (3, 2100, 8195), id="wca32"),
    pytest.param(ISING, None, (3, 5000, 131100), id="ising"),
])
def test_walkers_do_not_depend_on_their_wave(gpu_ctx_factory, kw, geom, sizes):
    ref = None
    for walkers in sizes:
        ctx, s = _run(gpu_ctx_factory, kw, walkers, geom, 1500)
        st, _ = ctx.download_raw(s, with_bins=False)
        got = (st[:sizes[0]].tobytes(), [ctx.bins(s, w)["lnw"].tobytes() for w in range(sizes[0])])
        ctx.close()
        ref = ref or got
        assert got == ref, f"{walkers} walkers"


@pytest.mark.parametrize("kw,geom", [pytest.param(LJ13, 2.5, id="lj13"), pytest.param(ISING, None, id="ising")])
def test_walkers_at_different_move_numbers(gpu_ctx_factory, kw, geom):
    W = 64
    early, s = _run(gpu_ctx_factory, kw, W, geom, 700)
    late, _ = _run(gpu_ctx_factory, kw, W, geom, 1000)
    mixed, _ = _run(gpu_ctx_factory, kw, W, geom, 1)
    (sa, ba), (sb, bb) = early.download_raw(s), late.download_raw(s)
    odd = (np.arange(W) % 2).astype(bool)
    st, bins = np.where(odd, sb, sa), np.where(odd[:, None], bb, ba)
    key = "spins" if kw["system"] == S.ISING else "coords"
    read = [getattr(c, key) for c in (early, late)]
    system = np.concatenate([read[int(o)](s, w) for w, o in enumerate(odd)])
    mixed.upload_raw(s, st, bins, **{key: system})
    for c in (early, late, mixed):
        c.run(900)
    want = np.where(odd, late.download_raw(s, False)[0], early.download_raw(s, False)[0])
    assert mixed.download_raw(s, False)[0].tobytes() == want.tobytes()


@pytest.mark.parametrize("kw,geom", [
    pytest.param(dict(LJ13, n=31, lanes=8), 3.0, id="lj31"),
    pytest.param(dict(LJ13, n=38, lanes=64), 3.2, id="lj38-64-lanes"),
    pytest.param(dict(WCA32, n=45), 5.0, id="wca45"),
    pytest.param(ISING, None, id="ising"),
])
def test_energy_query_is_the_lane_group_sum(gpu_ctx_factory, kw, geom):
    """compute_energy against the lanes' sums added up in the documented order."""
    ctx, s = _run(gpu_ctx_factory, kw, 3, geom, 400)
    for w in range(3):
        if kw["system"] == S.ISING:
            x = ctx.spins(s, w).reshape(8, 8).astype(float)
            want = float((x * (np.roll(x, 1, 0) + np.roll(x, 1, 1))).sum())
        else:
            n, G = kw["n"], kw["lanes"]
            x = ctx.coords(s, w).reshape(3, n)
            part = np.zeros(G)
            for i in range(n):
                for j in range(i):
                    d = x[:, i] - x[:, j]
                    if kw["system"] == S.WCA:
                        d = np.where(d > 0.5 * geom, d - geom, np.where(d < -0.5 * geom, d + geom, d))
                    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
                    if kw["system"] == S.WCA and not r2 < S.WCA_RC2:
                        continue
                    q = 1.0 / r2
                    q2 = q * q
                    v = 4.0 * (q2 * (q2 * q2) - q * q2)
                    part[i % G] += v + 1.0 if kw["system"] == S.WCA else v
            while len(part) > 1:
                part = part[0::2] + part[1::2]
            want = float(part[0])
        assert ctx.compute_energy(s, w) == want


@pytest.mark.parametrize("binning", [S.BIN_HISTOGRAM, S.BIN_LINEAR])
@pytest.mark.parametrize("kw,geom,sizes", [
    pytest.param(LJ13, 2.5, (3, 2049, 17000), id="lj13"),
    pytest.param(dict(WCA32, method=S.WL, method_param=1e-6), 4.2, (3, 8195), id="wca32-wl"),
    pytest.param(ISING, None, (3, 5000, 131100), id="ising"),
])
def test_binning_walkers_do_not_depend_on_their_wave(gpu_ctx_factory, kw, geom, sizes, binning):
    ref = None
    for walkers in sizes:
        ctx = gpu_ctx_factory()
        s = ctx.bin_add_set(S.make_params(binning=binning, **kw), np.arange(walkers, dtype=np.uint64) + 11, geom=geom)
        ctx.bin_run(s, 700)
        ctx.bin_run(s, 500)
        got = [(ctx.bin_state(s, w).tobytes(), ctx.bin_bins(s, w).tobytes()) for w in range(sizes[0])]
        ctx.close()
        ref = ref or got
        assert got == ref, f"{walkers} walkers"
