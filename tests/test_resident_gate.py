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

    def run(*args, bus="0", wait=True, **env):
        cmd, env = [exe, *map(str, args)], {**os.environ, "MODEL_BUS": f"model{os.getpid()}.{bus}", **env}
        if wait:
            return subprocess.run(cmd, env=env, stdin=subprocess.DEVNULL, capture_output=True, text=True)
        return subprocess.Popen(cmd, env=env, stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    return run


def test_one_process_per_gpu_on_the_whole_gpu(model):
    """The route belongs to the first process that asks for a GPU until it ends; an engine that may not use every compute unit
    does not get it."""
    assert model("claim").stdout == "1\n"                        # (and gave it back by ending)
    holder = model("claim", wait=False)
    assert holder.stdout.readline() == "1\n"
    assert model("claim").stdout == "0\n"
    assert model("claim", bus="1").stdout == "1\n"               # another GPU
    holder.kill()                                                # whatever way it ends
    holder.wait()
    assert model("claim").stdout == "1\n"
    assert model("claim", MODEL_CU_MASK="fffffffe").stdout == "0\n"
    assert model("claim", HSA_CU_MASK="0:0-127").stdout == "0\n"
    assert model("claim", MODEL_CU_MASK="ffffffff", HSA_CU_MASK="").stdout == "1\n"


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


@pytest.mark.parametrize("answers", [(1, 1), (0, 1), (1, 1, 1), (0, 1, 1), (0, 0, 0)])
def test_roll_call_has_one_outcome(answers):
    """The steps of csrc/resident.hpp's RollCall, every word read and written on its own, over all interleavings of two and three
    workgroups that may lose patience at any poll (0: one that does not answer): all of them go on, or none does."""
    N = len(answers)
    seen, stack, ends = set(), [(0, (0,) * N, 0, (("begin",),) * N)], set()
    NONE, DOUBT, GO, OFF = range(4)
    while stack:
        lost, got, ruling, at = state = stack.pop()
        if state in seen:
            continue
        seen.add(state)
        if all(a[0] == "end" for a in at):
            ends.add(frozenset(a[1] for a in at))

        def to(i, nxt, lost=lost, got=got, ruling=ruling):
            stack.append((lost, got, ruling, at[:i] + (nxt,) + at[i + 1:]))
        for i, a in enumerate(at):
            if a[0] == "begin":
                to(i, ("end", OFF) if lost else ("answer",))
            elif a[0] == "answer":
                to(i, ("read", 0, True), got=got[:i] + (answers[i],) + got[i + 1:])
            elif a[0] in ("read", "read again"):
                k, all_there = a[1] + 1, a[2] and got[a[1]] == 1
                after = ("ruling", all_there) if a[0] == "read" else ("resolve", all_there)
                to(i, (a[0], k, all_there) if k < N else after)
            elif a[0] == "ruling":
                if ruling == OFF:
                    to(i, ("end", OFF))
                elif a[1] and ruling != DOUBT:
                    to(i, ("end", GO))
                else:
                    to(i, ("read", 0, True))
                    if ruling == NONE:
                        to(i, ("doubt",))
            elif a[0] == "doubt":
                to(i, ("read again", 0, True), ruling=DOUBT) if ruling == NONE else to(i, ("read", 0, True))
            elif a[0] == "resolve":
                to(i, ("end", GO), ruling=GO) if a[1] else to(i, ("called off",), lost=1)
            elif a[0] == "called off":
                to(i, ("end", OFF), ruling=OFF)
    assert ends == ({frozenset([GO]), frozenset([OFF])} if all(answers) else {frozenset([OFF])})
