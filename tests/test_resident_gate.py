"""The gate of the resident decode steps (csrc/resident_gate.hip) on a model of the runtime's streams, events and captures
(gate_model/): which launches may run together, and what a turn may touch.  No GPU."""
import os
import re
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


def _first_layer(tile):
    """What the roll-call wave and the first computing wave of a workgroup of csrc/resident_rows.hip do in layer 0 up to barrier C, as
    the source has it: barriers (capitals), `outcome`, and the waits for u ("see u") and for the x_proj rows ("see x") with what
    goes out before them.  tile: the workgroup forms an x_proj tile."""
    text = open(os.path.join(CSRC, "resident_rows.hip")).read()
    feed, kernel = (text[text.index(at):] for at in ("void bring_rows_weights", "void resident_rows_kernel"))

    def walk(text, marks):
        text = text[text.index("for (int l ="):]
        text = text[:text.index("// C") + 4]
        found = [(m.start(), m.group(1)) for m in re.finditer(r"lds_barrier\(\);\s*// ([A-Z])", text)]
        for pattern, what in marks:
            at = [m.start() for m in re.finditer(pattern, text)]
            assert len(at) <= 1, pattern
            found += [(a, what) for a in at]
        return [what for _, what in sorted(found)]
    roll = walk(feed, [(r"l == 0 && f\.hurry\) take_outcome\(\)", "outcome" if tile else None),
                       (r"l == 0 && !f\.hurry\) take_outcome\(\)", None if tile else "outcome"),
                       (r"call\.outcome\(\)", "outcome")])
    compute = walk(kernel, [(r"say\(xb \+ S::e2f", "put u"), (r"return find\(S::e2f", "see u" if tile else None),
                            (r"xch_put_word\(xb \+ S::e2", "put x" if tile else None), (r"xch_poll<XW>", "see x")])
    return tuple(w for w in roll if w), tuple(w for w in compute if w)


def _run_to_the_end(tiles, places, programs):
    """Every interleaving of workgroups with the programs of _first_layer (tiles[i]: which kind), at most `places` of them on the chip
    at once.  Returns the outcomes, and the states from which nobody comes to an end any more."""
    N = len(tiles)
    NONE, GO, OFF, CALL = "none", "go", "off", "call"
    # per workgroup: place in the roll-call wave's program, in the computing wave's, its state; then lost, answers, ruling, u, x
    begin = ((None,) * N, False, frozenset(), NONE, frozenset(), frozenset())
    after, stack, ends = {}, [begin], set()

    def moves(s):
        wgs, lost, got, ruling, u, x = s
        running = sum(w not in (None, GO, OFF) for w in wgs)
        for i, w in enumerate(wgs):
            def to(w2, lost=lost, got=got, ruling=ruling, u=u, x=x, i=i):
                return (wgs[:i] + (w2,) + wgs[i + 1:], lost, got, ruling, u, x)
            if w is None:
                if running < places:    # the answer: one that is already too late leaves without a word
                    yield to(OFF) if lost else to((0, 0, CALL), got=got | {i})
                continue
            if w in (GO, OFF):
                continue
            roll, comp = programs[tiles[i]]
            r, c, state = w
            if r < len(roll) and c < len(comp) and roll[r] == comp[c]:          # a barrier both have come to
                if roll[r] == "C":
                    yield to(state if state in (GO, OFF) else "no ruling")
                else:
                    yield to((r + 1, c + 1, state))
                continue
            if roll[r] == "outcome":
                if ruling == OFF:
                    yield to((r + 1, c, OFF))
                elif len(got) == N:
                    yield to((r + 1, c, GO))
                else:                                                            # out of patience (or not yet: no change)
                    yield to((r + 1, c, OFF), lost=True, ruling=OFF)
            if comp[c] == "put u":
                yield to((r, c + 1, state), u=u | {i})
            elif comp[c] == "put x":
                yield to((r, c + 1, state), x=x | {i})
            elif comp[c] in ("see u", "see x"):
                there = len(u) == N if comp[c] == "see u" else x >= {k for k in range(N) if tiles[k]}
                if there or state == OFF:
                    yield to((r, c + 1, state))
    while stack:
        s = stack.pop()
        if s in after:
            continue
        after[s] = list(moves(s))
        stack += after[s]
        if all(isinstance(w, str) for w in s[0]):
            ends.add(frozenset(s[0]))
    can_end, grown = {s for s in after if all(isinstance(w, str) for w in s[0])}, True
    while grown:
        more = {s for s, t in after.items() if s not in can_end and any(n in can_end for n in t)}
        can_end |= more
        grown = bool(more)
    return ends, set(after) - can_end


@pytest.mark.parametrize("tiles", [(True, False, False), (True, True, False), (True, False, False, False)])
@pytest.mark.parametrize("short_of", [0, 1, 2])
def test_a_step_of_many_rows_that_lacks_places_ends(tiles, short_of):
    """Layer 0 of csrc/resident_rows.hip, barriers and waits where the source has them: whatever places are missing and whoever
    loses patience first, every workgroup comes to an end, and all of them the same way.  (With the outcome behind the barrier that the
    first wait stands in front of, they do not: the model sees that.)"""
    programs = {t: _first_layer(t) for t in (True, False)}
    assert programs[False] == (("A", "B", "X", "outcome", "C"), ("A", "put u", "B", "X", "see x", "C"))
    assert programs[True][1] == ("A", "put u", "see u", "B", "X", "put x", "see x", "C")
    ends, stuck = _run_to_the_end(tiles, len(tiles) - short_of, programs)
    assert not stuck
    assert ends == ({frozenset(["off"])} if short_of else {frozenset(["go"]), frozenset(["off"])})
    late = {**programs, True: (("A", "B", "X", "outcome", "C"), programs[True][1])}
    assert _run_to_the_end(tiles, len(tiles) - short_of, late)[1]
