"""The device S(E) reduction against the host's over the same downloaded bins,
at walker counts around the walkers a lane has in flight (4) and the chunks
(one walker each up to 64 chunks), and with windows inside every walker's range, reaching past it
(the window mean then needs the extension) and outside some walkers' bins."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

S = pytest.importorskip("sadmc_amd")
A = pytest.importorskip("analysis")


@pytest.mark.parametrize("walkers", [1, 3, 5, 70, 261])
@pytest.mark.parametrize("system", ["lj13", "ising"])
def test_entropy_windows_and_sizes(gpu_ctx_factory, walkers, system):
    if system == "lj13":
        p = S.make_params(system=S.LJ, n=13, lanes=4, method=S.SAD, method_param=0.05, move_param=0.1, energy_bin=0.02,
                          has_max_e=1, max_e=0.0)
        geom, moves = 2.5, 20000
    else:
        p = S.make_params(system=S.ISING, n=6, ising_init=1, method=S.SAD, method_param=1.0)
        geom, moves = None, 20000
    ctx = gpu_ctx_factory()
    s = ctx.add_set(p, np.arange(walkers, dtype=np.uint64) + 5, geom=geom)
    ctx.init()
    ctx.run(moves)
    st, rows = ctx.download_raw(s)
    pairs = [(st[w], S.logical_bins(st[w], rows[w])) for w in range(walkers)]
    lo, hi = st["too_lo"].max(), st["too_hi"].min()
    width = st["bins_width"][0]
    assert hi > lo
    for window in (None, (lo + width, hi - width), (lo - 3 * width, hi), (lo, hi + 4 * width), (lo - 400 * width, hi)):
        if window and not window[0] + width < window[1]:
            continue
        Eh, Sh, ch = A.mean_entropy(pairs, window)
        Ed, Sd, cd = ctx.mean_entropy(s, window)
        assert np.array_equal(ch, cd), window
        if len(Eh):
            assert np.allclose(Eh, Ed, rtol=0, atol=1e-9)
            # sums of at most 261 terms of size |S| <~ 1e2, each rounded a few times
            assert np.allclose(Sh, Sd, rtol=1e-11, atol=1e-10), window
