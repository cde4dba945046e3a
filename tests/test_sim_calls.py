"""Device calls of several blocks on the CPU simulation build of the library
(tests/cpu_sim): buffers, shapes and orders of calls at which the call path
and the paths for single blocks have to agree."""
import os
import subprocess
import sys

import pytest

from test_sim_replay import SIM, sim_built  # noqa: F401 (fixture)


def _run(name, guard="start", fill="0xff", timeout=600, **kw):
    env = dict(os.environ, SIM_GUARD=guard, SIM_FILL=fill)
    p = subprocess.run([sys.executable, os.path.join(SIM, "call_scenarios.py"), name] +
                       [f"{k}={v}" for k, v in kw.items()], env=env, capture_output=True, text=True, timeout=timeout)
    assert p.returncode == 0, (p.returncode, p.stdout[-2000:], p.stderr[-2000:])


@pytest.mark.parametrize("method", [0, 1, 2], ids=["uniform", "nonuniform", "time"])
def test_in_place(sim_built, method):  # noqa: F811
    _run("in_place", method=method)


@pytest.mark.parametrize("P,kp,B", [(1, 4, 64), (2, 4, 64), (4, 16, 64), (8, 4, 64), (4, 4, 1024), (8, 12, 512)])
def test_few_partitions(sim_built, P, kp, B):  # noqa: F811
    _run("few_partitions", P=P, kp=kp, B=B)


@pytest.mark.parametrize("method", [0, 1], ids=["uniform", "nonuniform"])
def test_chunk_changes(sim_built, method):  # noqa: F811
    _run("chunk_changes", method=method)


@pytest.mark.parametrize("kp,precision", [(0, 0), (2, 0), (4, 0), (4, 1), (7, 0), (8, 2), (12, 0), (16, 0)])
def test_mixed_uniform(sim_built, kp, precision):  # noqa: F811
    for seed in (1, 2):
        _run("mixed", seed=seed, kp=kp, precision=precision)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_mixed_nonuniform(sim_built, seed):  # noqa: F811
    _run("mixed", seed=seed, method=1)


@pytest.mark.parametrize("method,kp", [(0, 0), (0, 8), (0, 12), (1, 0)])
def test_next_block(sim_built, method, kp):  # noqa: F811
    _run("next_block", method=method, kp=kp)
