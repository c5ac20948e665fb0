"""The kernels behind the environment switches.  The library reads its switches once per process, so each setting runs the
same parity case (tests/two_valued_case.py) in one child process: the default (lookup kernels for two-valued inputs,
packed backward pass) and the polynomial kernels for the same inputs."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("env", [{}, {"BBHIP_CORNER": "2", "BBHIP_PACK": "2"}, {"BBHIP_PACK": "2"}, {"BBHIP_CORNER": "0", "BBHIP_PACK": "0"},
                                 {"BBHIP_CORNER": "0"}, {"BBHIP_FWD_NODES": "1", "BBHIP_BWD_SLAB": "256"},
                                 {"BBHIP_DX_STEPS": "1", "BBHIP_DX_CHUNK": "64", "BBHIP_BIN_NODES": "1", "BBHIP_BIN_CHUNK": "64"},
                                 {"BBHIP_DX_STEPS": "4", "BBHIP_DX_CHUNK": "512", "BBHIP_FWD_CHUNK": "512", "BBHIP_BIN_NODES": "2", "BBHIP_BIN_CHUNK": "256"},
                                 {"BBHIP_DX_SPLIT": "1"}, {"BBHIP_DX_SPLIT": "0", "BBHIP_BIN_NODES": "4"},
                                 {"BBHIP_INLINE_TABLES": "0"}, {"BBHIP_FWD_CHUNK": "2048"}, {"BBHIP_DX_QUADS": "1"}, {"BBHIP_DX_QUADS": "2"},
                                 {"BBHIP_DX_QUADS": "4"}, {"BBHIP_DX_QUADS": "4", "BBHIP_DX_SPLIT": "1"}])
def test_two_valued_inputs_under_switches(env):
    child_env = dict(os.environ)
    child_env.update(env)
    child_env["PYTHONPATH"] = os.pathsep.join([os.path.dirname(HERE), HERE, child_env.get("PYTHONPATH", "")])
    p = subprocess.run([sys.executable, os.path.join(HERE, "two_valued_case.py")], env=child_env, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and "two-valued case ok" in p.stdout, (env, p.stdout[-2000:], p.stderr[-2000:])
    # the switches took effect: 0 and 2 turn a path off, unset leaves it on
    want = {name: 0 if env.get(var) in ("0", "2") else 1 for name, var in (("corner", "BBHIP_CORNER"), ("pack", "BBHIP_PACK"))}
    assert "switches corner=%d pack=%d inline_tables=%d dx_quads=%d\n" % (want["corner"], want["pack"], 0 if env.get("BBHIP_INLINE_TABLES") == "0" else 1,
                                                                         int(env.get("BBHIP_DX_QUADS", "0"))) in p.stdout, (env, p.stdout[-500:])


@pytest.mark.parametrize("env, units", [({}, 1), ({"BBHIP_FWD_CHUNK": "512"}, 2), ({"BBHIP_FWD_CHUNK": "64"}, 16), ({"BBHIP_FWD_CHUNK": "320", "BBHIP_INLINE_TABLES": "0"}, 4),
                                        ({"BBHIP_FWD_CHUNK": "2048", "BBHIP_PACK": "0"}, 1)])
def test_forward_units_of_up_to_1024_frames_under_the_switch(env, units):
    """BBHIP_FWD_CHUNK holds for short passes too: the frames of a unit, and no training pass in one unit per node because of its size"""
    child_env = dict(os.environ)
    child_env.update(env)
    child_env["PYTHONPATH"] = os.pathsep.join([os.path.dirname(HERE), HERE, child_env.get("PYTHONPATH", "")])
    p = subprocess.run([sys.executable, os.path.join(HERE, "two_valued_case.py"), "small"], env=child_env, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and "small passes ok, units of a training pass: [%d]" % units in p.stdout, (env, p.stdout[-2000:], p.stderr[-2000:])
