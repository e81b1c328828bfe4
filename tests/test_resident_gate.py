"""The gate of the resident decode steps (csrc/resident_gate.hip) on a model of the runtime's streams, events and captures
(gate_model/): which launches may run together, and what a turn may touch.  No GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mamba_rs_amd", "csrc")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("gate") / "model")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(HERE, "gate_model"), "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "gate_model", "model.cpp"), "-lpthread"], check=True)

    def run(*args, bus="0"):
        return subprocess.run([exe, *map(str, args)], env={**os.environ, "MODEL_BUS": f"model{os.getpid()}.{bus}"}, capture_output=True, text=True)
    return run


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("fail_every", [0, 7])
def test_launches_that_do_not_fit_together_are_ordered(model, seed, fail_every):
    """Random engines, steps, waits and captures: no two launches that need more places than there are run unordered, no turn
    records or waits on a stream but its own or on one that is in a capture, a caller's capture gets no launch, and neither does a
    failing event let one through."""
    r = model(seed, fail_every)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
    in_turns, refused = map(int, r.stdout.split()[1:])
    assert in_turns > 500 and refused > 50     # both ways were taken
