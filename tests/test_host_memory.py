"""The library's host code against a stand-in for the HIP runtime
(standin_runtime.c), without a GPU: what it allocates, copies and waits for.
Each test runs in a process of its own, where the stand-in is loaded first."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "sad-monte-carlo_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    out = tmp_path_factory.mktemp("standin") / "libstandin.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-o", str(out), os.path.join(HERE, "standin_runtime.c")], check=True)
    return str(out)


def _run(standin, body):
    head = f"""
import ctypes, sys
R = ctypes.CDLL({standin!r}, mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, {PKG!r})
import numpy as np
import sadmc_amd as S
"""
    r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(body)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("kind", ["ising", "wca"])
def test_a_failed_start_can_be_repeated_with_more_sets(standin, kind):
    """sadmc_init with each of its allocations failing once: the start is
    refused, more sets may be added, and the next start holds memory for all of
    them and no memory of the failed one."""
    out = _run(standin, f"""
    ising = S.make_params(system=S.ISING, n=4, ising_init=1, method=S.WL, method_param=1e-6)
    wca = S.make_params(system=S.WCA, n=8, lanes=4, method=S.SAD, method_param=0.1, energy_bin=0.5, has_max_e=1,
                        max_e=20.0, collect_pressure=1)
    params, geom = (ising, None) if {kind!r} == "ising" else (wca, 4.0)
    failed = 0
    for k in range(100):
        ctx = S.Context(0)
        ctx.add_set(params, np.arange(3, dtype=np.uint64), geom=geom)
        R.standin_fail_allocation(k)
        try:
            ctx.init()
        except S.SadmcError as e:
            assert e.code == -2 and "error" in str(e), e
            failed += 1
            for _ in range(3):
                ctx.add_set(ising, np.arange(5, dtype=np.uint64))
            ctx.init()
        unused = R.standin_fail_allocation(-1) >= 0
        ctx.run(10)
        ctx.run_set(len(ctx.sets) - 1, 10)
        assert R.standin_overruns() == 0, k
        ctx.close()
        assert R.standin_live() == 0, k
        if unused:
            break
    print(failed)
    """)
    assert int(out) >= 5  # every allocation of a start was the failing one once


def test_training_has_ended_when_the_call_returns(standin):
    """sadmc_prop_train waits for its steps whether or not the losses are asked for."""
    _run(standin, """
    ctx = S.Context(0)
    ctx.prop_load_records(np.zeros((64, S.PROP_REC), np.float32))
    for losses in (np.zeros(3, np.float32), None):
        ctx._check(S.lib().sadmc_prop_train(ctx.h, 3, 64, 1e-3, S._p(losses)), "prop_train")
        assert R.standin_queued() == 0, losses
    """)
