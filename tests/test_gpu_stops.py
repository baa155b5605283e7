"""The state a walker is left in by the move that stops it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")


@pytest.mark.parametrize("n,lanes,walkers", [(13, 4, 96), (31, 8, 96)])
def test_bins_of_a_walker_whose_energy_check_fails(gpu_ctx_factory, n, lanes, walkers):
    """The move whose energy check fails still proposes, and the bins grow to
    the proposed energy, before the walker stops: generator, move count and bins
    as planned on a second context."""
    print("case failed check", n, lanes, walkers, flush=True)
    kw = dict(system=S.LJ, n=n, lanes=lanes, method=S.SAD, method_param=0.05, move_param=0.1, energy_bin=0.05,
              has_max_e=1, max_e=0.0)
    made = []
    for _ in range(2):
        ctx = gpu_ctx_factory()
        s = ctx.add_set(S.make_params(**kw), np.arange(walkers, dtype=np.uint64), geom=2.5 if n == 13 else 3.0)
        ctx.init()
        ctx.run(3)
        made.append(ctx)
    run, plan = made
    st, bins = run.download_raw(s)
    st = st.copy()
    st["moves"] = st["len"].astype(np.uint64) ** 2 * 1000 - 1  # the check is due at the next move
    st["E"] += 1e-3
    for c in made:
        c.upload_raw(s, st, bins)
    with pytest.raises(S.SadmcError) as e:
        run.run(1)
    assert e.value.code == -4
    got, after = run.download_raw(s)
    up = down = 0
    for w in range(walkers):
        e2 = plan.plan_move(s, w, float(st[w]["translation_scale"]))
        length, base, lo = int(st[w]["len"]), int(st[w]["base"]), float(st[w]["bins_min"])
        if e2 is not None and not (e2 > 0.0 and e2 > st[w]["E"]):
            while e2 < lo:
                length, base, lo, down = length + 1, base - 1, lo - 0.05, down + 1
            while e2 >= lo + 0.05 * length:
                length, up = length + 1, up + 1
        assert (int(got[w]["len"]), int(got[w]["base"]), float(got[w]["bins_min"])) == (length, base, lo), w
        assert int(got[w]["moves"]) == int(st[w]["moves"]) + 1
        assert list(got[w]["rng"]) == list(plan.state(s, w)["rng"])
        new = after[w][base:base + length]
        assert (new["round_trips"] >= 1).all()
        assert new["histogram"].sum() == bins[w]["histogram"].sum()
    assert up and down
