"""Counters of uploaded walkers beyond 2^53, where doubles are no longer whole:
they are kept and counted as integers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")

BIG = 2 ** 53 + 1  # not a double


@pytest.mark.parametrize("kw,geom", [
    pytest.param(dict(system=S.ISING, n=8, ising_init=1, method_param=1.0), None, id="ising"),
    pytest.param(dict(system=S.LJ, n=13, lanes=4, method_param=0.05, move_param=0.1, energy_bin=0.2, has_max_e=1,
                      max_e=0.0), 2.5, id="lj13"),
    pytest.param(dict(system=S.WCA, n=8, lanes=8, method_param=0.1, move_param=0.05, energy_bin=0.2, has_max_e=1,
                      max_e=40.0, collect_pressure=1), 2.6, id="wca8-pressure"),
])
@pytest.mark.parametrize("walkers", [3, 2100])
def test_counters_stay_whole(gpu_ctx_factory, kw, geom, walkers):
    print("case counters", kw["system"], walkers, flush=True)
    ctx = gpu_ctx_factory()
    s = ctx.add_set(S.make_params(method=S.SAD, **kw), np.arange(walkers, dtype=np.uint64), geom=geom)
    ctx.init()
    ctx.run(300)
    st, bins = ctx.download_raw(s)
    st, bins = st.copy(), bins.copy()
    for k, name in enumerate(("moves", "tF", "num_states", "tmax")):
        st[name] = BIG + 2 * k
    st["tL"] = BIG - 2
    found = bins["t_found"] > 0
    bins["t_found"][found] = BIG - 2
    ctx.upload_raw(s, st, bins)
    ctx.run(0)
    same, _ = ctx.download_raw(s)
    for name in ("moves", "tF", "num_states", "tmax", "tL"):
        assert np.array_equal(same[name], st[name]), name
    n, before = 130, ctx.bins(s, 0)["pressure_count"].sum()
    ctx.run(n)
    after, rows = ctx.download_raw(s)
    end = BIG + n
    assert np.all(after["moves"] == end)
    grown = after["num_states"].astype(np.int64) - st["num_states"].astype(np.int64)
    assert np.all((grown >= 0) & (grown <= rows.shape[1]))
    for name in ("tL", "tF", "tmax"):
        kept = after[name] == st[name]
        assert np.all(kept | (after[name] > BIG) & (after[name] <= end)), name
    t = rows["t_found"][rows["t_found"] > 0]
    assert np.all((t == BIG - 2) | ((t > BIG) & (t <= end)))
    assert np.any(t % 2 == 0) and np.any((t > BIG) & (t % 2 == 1))
    if kw["system"] == S.WCA:
        every = kw["n"] ** 2
        assert ctx.bins(s, 0)["pressure_count"].sum() - before == end // every - BIG // every
