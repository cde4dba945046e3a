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
