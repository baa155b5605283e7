"""Wavefronts that hold several walkers, of which some have stopped or stand
at another move number. Set sizes are chosen by how many walkers a wave then
holds: 64 / lanes of them in sets that fill the chip's 1024 SIMDs (Ising: twice
that) with such waves, fewer in smaller sets; the sizes that this file calls
full have every wave full under any rule that fills the chip first."""
import numpy as np
import pytest

from conftest import compare_walker, oracle_params, run_oracles

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")

LJ13 = dict(system=S.LJ, n=13, lanes=4, method=S.SAD, method_param=0.05, move_plan=S.ACCEPTANCE_RATE, move_param=0.3,
            energy_bin=0.2, has_max_e=1, max_e=0.0)
LJ13_FULL, ISING_FULL = 16 * 1024 + 20, 64 * 2048 + 70


@pytest.mark.parametrize("kw,geom,walkers,code,moves", [
    # odd lattice: an initial energy on the edge of its bin stops the walker
    pytest.param(dict(system=S.ISING, n=5, ising_init=1, method=S.SAD, method_param=1.0), None, 4200, -8, (200, 301),
                 id="ising5-2-a-wave"),
    pytest.param(dict(system=S.ISING, n=5, ising_init=1, method=S.SAD, method_param=1.0), None, ISING_FULL, -8,
                 (200, 301), id="ising5-full"),
    # a window that ends above the energies the walk reaches
    pytest.param(dict(LJ13, e_lo_bound=-20.0, e_hi_bound=0.0), 2.5, 2100, -3, (1500, 2001), id="lj13-2-a-wave"),
    pytest.param(dict(LJ13, e_lo_bound=-20.0, e_hi_bound=0.0), 2.5, LJ13_FULL, -3, (1500, 2001), id="lj13-full"),
])
def test_running_walkers_beside_stopped_ones(gpu_ctx_factory, kw, geom, walkers, code, moves):
    """The stopped walkers stop where the oracle's do; the others go on, bit
    for bit, in this launch and the next."""
    print("case", kw["system"], walkers, flush=True)
    sp = S.make_params(**kw)
    ctx = gpu_ctx_factory()
    s = ctx.add_set(sp, np.arange(walkers, dtype=np.uint64), geom=geom)
    ctx.init()
    for m in moves:
        with pytest.raises(S.SadmcError) as e:
            ctx.run(m)
        assert e.value.code == code
    look = 192  # the first walkers: three full Ising waves, twelve of LJ13
    st, _ = ctx.download_raw(s, with_bins=False)
    stopped = st["status"][:look] != 0
    mixed = stopped[0::2] != stopped[1::2]  # neighbours share a wave in all of these sets
    assert mixed.any() and (~stopped).any()
    total = sum(moves)
    orcs = run_oracles([oracle_params(sp, w, geom or 0.0) for w in range(look)], total)
    for w in np.flatnonzero(~stopped):
        compare_walker(ctx.state(s, w), ctx.bins(s, w), orcs[w], sp.method, label=f"walker {w}")
    for w in np.flatnonzero(stopped):
        if code == -8:  # the oracle stops there too; a window's end it does not have
            o = orcs[w].scalars()
            assert int(st[w]["status"]) == o["status"] and int(st[w]["moves"]) == o["moves"], w
        else:
            assert int(st[w]["moves"]) <= total, w


@pytest.mark.parametrize("kw,geom,walkers", [
    pytest.param(LJ13, 2.5, 5000, id="lj13-4-a-wave"),
    pytest.param(LJ13, 2.5, LJ13_FULL, id="lj13-full"),
    pytest.param(dict(system=S.ISING, n=8, ising_init=1, method=S.SAD, method_param=1.0), None, 4200,
                 id="ising-2-a-wave"),
    pytest.param(dict(system=S.ISING, n=8, ising_init=1, method=S.SAD, method_param=1.0), None, ISING_FULL,
                 id="ising-full"),
])
def test_neighbours_at_different_move_numbers(gpu_ctx_factory, kw, geom, walkers):
    """Every other walker uploaded 300 moves ahead of its neighbours."""
    print("case", kw["system"], walkers, flush=True)

    def start(moves):
        ctx = gpu_ctx_factory()
        s = ctx.add_set(S.make_params(**kw), np.arange(walkers, dtype=np.uint64) + 11, geom=geom)
        ctx.init()
        ctx.run(moves)
        return ctx, s

    (early, s), (late, _), (mixed, _) = start(700), start(1000), start(1)
    (sa, ba), (sb, bb) = early.download_raw(s), late.download_raw(s)
    odd = (np.arange(walkers) % 2).astype(bool)
    st, bins = np.where(odd, sb, sa), np.where(odd[:, None], bb, ba)
    assert len(np.unique(st["moves"][:2])) == 2
    key = "spins" if kw["system"] == S.ISING else "coords"
    read = [getattr(c, key) for c in (early, late)]
    system = np.concatenate([read[int(o)](s, w) for w, o in enumerate(odd)])
    mixed.upload_raw(s, st, bins, **{key: system})
    for c in (early, late, mixed):
        c.run(500)
    (sa, ba), (sb, bb), (sm, bm) = (c.download_raw(s) for c in (early, late, mixed))
    for c in (early, late, mixed):
        c.close()
    assert sm.tobytes() == np.where(odd, sb, sa).tobytes()
    assert bm.tobytes() == np.where(odd[:, None], bb, ba).tobytes()


@pytest.mark.parametrize("kw,geom,sizes", [
    pytest.param(dict(LJ13, method=S.WL, method_param=0.0, has_min_e=1, min_e=-44.0), 2.5, (3, 2100, LJ13_FULL),
                 id="lj13-wl"),
    pytest.param(dict(LJ13, method=S.INV_T_WL, method_param=0.0, has_min_e=1, min_e=-44.0), 2.5, (3, 2100, LJ13_FULL),
                 id="lj13-inv-t-wl"),
    pytest.param(dict(LJ13, method=S.CANONICAL, method_param=0.3), 2.5, (3, 2100, LJ13_FULL), id="lj13-canonical"),
    pytest.param(dict(LJ13, method=S.CANONICAL, method_param=0.2, precision=S.FP32_PAIRS, refresh=256), 2.5,
                 (3, 2100, LJ13_FULL), id="lj13-fp32-canonical"),
    pytest.param(dict(LJ13, precision=S.FP32_PAIRS, refresh=256), 2.5, (3, 2100, LJ13_FULL), id="lj13-fp32-sad"),
    pytest.param(dict(system=S.WCA, n=32, lanes=8, method=S.CANONICAL, method_param=1.0, move_param=0.05,
                      energy_bin=0.2, has_max_e=1, max_e=80.0, collect_pressure=1), 3.6, (3, 1100, 8 * 1024 + 10),
                 id="wca32-canonical"),
    pytest.param(dict(system=S.ISING, n=8, ising_init=1, method=S.INV_T_WL, has_min_e=1, min_e=-116.0, has_max_e=1,
                      max_e=116.0), None, (3, 4200, ISING_FULL), id="ising-inv-t-wl"),
])
def test_methods_do_not_depend_on_the_wave(gpu_ctx_factory, kw, geom, sizes):
    """The first walkers of small and full sets, and the small set's against the oracle."""
    print("case", kw["system"], kw["method"], flush=True)
    sp = S.make_params(**kw)
    moves, ref = (700, 600), None
    for walkers in sizes:
        ctx = gpu_ctx_factory()
        s = ctx.add_set(sp, np.arange(walkers, dtype=np.uint64) + 300, geom=geom)
        ctx.init()
        for m in moves:
            ctx.run(m)
        st, _ = ctx.download_raw(s, with_bins=False)
        bins = [ctx.bins(s, w) for w in range(3)]
        got = (st[:3].tobytes(), [{k: v.tobytes() for k, v in b.items()} for b in bins])
        if ref is None:
            ref = got
            orcs = run_oracles([oracle_params(sp, w + 300, geom or 0.0) for w in range(3)], sum(moves))
            for w in range(3):
                compare_walker(ctx.state(s, w), bins[w], orcs[w], sp.method, label=f"walker {w}")
        ctx.close()
        assert got == ref, f"{walkers} walkers"
