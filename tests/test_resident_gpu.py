"""GPU: the resident decode step (a whole 16-bit Mamba-1 step in one launch whose workgroups exchange through memory) against
the CPU route, and against itself: eager and replayed, alone, beside other engines, threads and processes, in captures, called off."""
import numpy as np
import pytest

import orc
from util import cosine, scaled_err
from test_engine_gpu import oracle_params

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMambaBackbone, MambaConfig, MambaWeights, WeightDtype  # noqa: E402


@pytest.mark.parametrize("dm,L,B", [(1024, 20, 1), (1024, 20, 3), (2560, 4, 3), (1024, 20, 40), (1024, 20, 65)])
def test_weights_past_the_last_cache(dm, L, B):
    """Models whose weights are more than the last cache holds, so that some layers' (resident steps of a row and of several) or all layers' in_proj (a launch per product) are read past it,
    and there the states as well (three forms of the step kernel): outputs against the CPU route, as below.  Every layer has weights of its own (one layer's with their columns moved
    along), so that a block of another layer's shows."""
    import copy
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 11)
    w.input_proj_w = np.zeros((0, dm), np.float32)
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=L)
    w.layers = [copy.copy(w.layers[0]) for _ in range(L)]
    for l, lw in enumerate(w.layers):
        for n in ("in_proj_w", "x_proj_w", "dt_proj_w", "out_proj_w"):
            setattr(lw, n, np.roll(getattr(lw, n), 37 * l, axis=1))
    P = oracle_params(w, cfg, dm, round_to=orc.BF16)
    print(f"case past the cache {dm} {L} {B}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.BF16)
    st = {b: orc.m1_zero_state(P) for b in {0, B - 1}}
    for t in range(2):
        x = np.random.default_rng(t).standard_normal((B, dm)).astype(np.float32)
        got = eng.step(x)
        for b in st:
            want = orc.m1_backbone_step(P, x[b], *st[b], identity_proj=True)
            assert cosine(got[b], want) >= 0.999, (t, b, cosine(got[b], want))
    eng.close()


@pytest.mark.parametrize("shape", [
    (32, 2, 32, 1),       # one k-step, four workgroups; an x_proj row of 34: a last tile of two entries
    (64, 3, 20, 16),      # input projection; dt_rank 4; a group of workgroups per row, sixteen of them
    (192, 2, 192, 5),     # 24 channels per workgroup, dt_rank 12
    (256, 2, 256, 8),     # eight rows of 32 workgroups: every compute unit
    (768, 2, 768, 1),     # 24 channels and 12 out_proj columns per workgroup
    (768, 2, 768, 4),
    (1024, 2, 1024, 1),   # the widest: 128 workgroups, four and eight k-steps per wave
    (896, 2, 896, 2),     # 112 workgroups per row, a width the groups of several rows do not take
    (640, 2, 640, 3),     # 80 per row, the same
    # several rows per group of workgroups (resident_rows.hip)
    (256, 2, 20, 9),      # input projection; groups of five and four rows
    (256, 2, 256, 128),   # eight full groups; dt_rank 16: a k-step of dt_proj with zeros behind it
    (512, 2, 512, 37),    # groups of ten and nine rows: the second wave that writes operands has two or one
    (768, 2, 768, 5),     # one group; 24 channels: a channel tile that is half empty
    (768, 2, 768, 17),    # three groups, of six, six and five rows
    (768, 2, 768, 64),    # full groups, three k-steps per wave
    (1024, 2, 1024, 2),   # the smallest group
    (1024, 2, 1024, 3),
    (1024, 2, 1024, 31),  # two groups of 128 workgroups, sixteen and fifteen rows
])
@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
def test_resident_step_follows_the_cpu_route(shape, dtype):
    """Six steps (three eager, three replayed): every row within the 16-bit engines' tolerance of the CPU route on
    storage-rounded weights (cosine >= 0.999 as for the kernel chains: the same rounding points, sums in another order), states
    as well.  A second engine steps behind the first -- each call returns with its rows, so nothing overlaps here; the queued steps
    below do -- and ends on the same bits: all sums are in a fixed order."""
    dm, L, idim, B = shape
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=L)
    w = MambaWeights.init(cfg, idim, 11)
    if idim == dm:
        w.input_proj_w = np.zeros((0, dm), np.float32)
    identity = w.input_proj_w.size == 0
    code = orc.BF16 if dtype == WeightDtype.BF16 else orc.F16
    P = oracle_params(w, cfg, idim, round_to=code)
    print(f"case resident step {shape} {dtype.name}", flush=True)
    a = GpuMambaBackbone.new_with_dtype(0, w, cfg, idim, B, dtype)
    b = GpuMambaBackbone.new_with_dtype(0, w, cfg, idim, B, dtype)
    assert a.decode_route() == 2 and b.decode_route() == 2      # one launch
    rng = np.random.default_rng(dm + B)
    x = rng.standard_normal((6, B, idim)).astype(np.float32)
    # the ends of every group: eight rows wanted, at most 256 workgroups
    groups = min(-(-B // 8), 256 // (dm // (12 if dm == 768 else 8)))
    first = [g * (B // groups) + min(g, B % groups) for g in range(groups + 1)]
    rows = sorted({0, B // 2, B - 1} | {r for a, b in zip(first, first[1:]) for r in (a, b - 1)})
    st = {r: orc.m1_zero_state(P) for r in rows}
    for t in range(6):
        if t == 3:
            a.capture_graph()
        got = a.step(x[t])
        assert np.array_equal(b.step(x[t]), got), t
        for r in rows:
            want = orc.m1_backbone_step(P, x[t, r], *st[r], identity_proj=identity)
            assert cosine(got[r], want) >= 0.999, (t, r, cosine(got[r], want))
    di = cfg.d_inner()
    for l in range(L):
        conv, ssm = a.download_state(l)
        for r in rows:
            assert cosine(conv[r][:, 1:], st[r][0][l].reshape(di, 3)) >= 0.999, (l, r)
            want = st[r][1][l].reshape(di, 16)
            assert cosine(ssm[r], want) >= 0.999 and scaled_err(ssm[r], want) < 5e-2, (l, r, cosine(ssm[r], want), scaled_err(ssm[r], want))
    a.reset()
    b.reset()
    assert np.array_equal(a.step(x[0]), b.step(x[0]))
    a.close()
    b.close()


def _engines(shape, n, dtype=WeightDtype.BF16):
    dm, L, B = shape
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=L)
    w = MambaWeights.init(cfg, dm, 5)
    w.input_proj_w = np.zeros((0, dm), np.float32)
    return [GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype) for _ in range(n)]


def test_queued_steps_of_engines_that_do_not_fit_together():
    """Two engines of 256 workgroups (and a third of 128): their steps are queued in turns with nothing waited for in between, so
    each launch meets the one before still running.  Every engine ends on the bits of one that was alone."""
    a, b = _engines((768, 6, 4), 2)
    c, = _engines((768, 4, 2), 1)
    rng = np.random.default_rng(2)
    x = {e: rng.standard_normal((e.batch, 768)).astype(np.float32) for e in (a, b, c)}

    def run(engines, n):
        for e in engines:
            e.reset()
            e.step(x[e])
        for _ in range(n):
            for e in engines:
                e.step_gpu_only()
        return [e.download_temporal() for e in engines]
    print("case queued steps of three engines", flush=True)
    assert [e.decode_route() for e in (a, b, c)] == [2, 2, 2]
    alone = [run([e], 24)[0] for e in (a, b, c)]
    for got, want in zip(run([a, b, c], 24), alone):
        assert np.array_equal(got, want)
    for e in (a, b, c):
        e.close()


def test_an_engine_captures_while_another_one_steps():
    """Two threads, two engines that do not fit together: one builds language models and captures their step over and over, the
    other queues steps.  Nothing of one engine ends in the other's graph: tokens and rows are those of each one alone."""
    import threading
    from mamba_rs_amd import GpuMambaLM
    a, b = _engines((768, 4, 4), 2)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((4, 768)).astype(np.float32)
    embed = rng.standard_normal((256, 768)).astype(np.float32)
    first = np.arange(4, dtype=np.int32)

    def captured():
        lm = GpuMambaLM(a, embed)
        a.reset()
        lm.set_tokens(first)
        lm.capture_graph()
        got = []
        for _ in range(6):
            lm.decode_step()
            got.append(lm.get_tokens().tolist())
        lm.close()
        return got

    def stepped():
        b.reset()
        b.step(x)
        for _ in range(40):
            b.step_gpu_only()
        return b.download_temporal()
    print("case capture beside steps", flush=True)
    want, row = captured(), stepped()
    res = {"a": [], "b": []}

    def loop(key, fn, n):
        try:
            for _ in range(n):
                res[key].append(fn())
        except Exception as e:      # into the main thread
            res[key].append(e)
    ts = [threading.Thread(target=loop, args=("a", captured, 12)), threading.Thread(target=loop, args=("b", stepped, 24))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(res["a"]) == 12 and all(r == want for r in res["a"])
    assert len(res["b"]) == 24 and all(isinstance(r, np.ndarray) and np.array_equal(r, row) for r in res["b"])
    a.close()
    b.close()


def _family(family, rows=4):
    """(a constructor of engines of so many rows on the same weights, d_model, the language model class) of either network."""
    from mamba_rs_amd import GpuMamba3Backbone, GpuMamba3LM, GpuMambaLM
    if family == "m1":
        return lambda: _engines((768, 3, rows), 1)[0], 768, GpuMambaLM
    if family == "m1rows":      # rows on one group of 128 workgroups (resident_rows.hip)
        return lambda: _engines((1024, 3, rows), 1)[0], 1024, GpuMambaLM
    from test_m3_engine_gpu import perturbed
    from test_resident_m3_gpu import cfg_
    cfg = cfg_(256, 16, 16, 1, 3)
    w = perturbed(cfg, 256, 11)
    w.input_proj_w = np.zeros(0, np.float32)
    return lambda: GpuMamba3Backbone.new_with_dtype(0, w, cfg, 256, rows, WeightDtype.BF16), 256, GpuMamba3LM


@pytest.mark.parametrize("family", ["m1", "m3", "m1rows"])
def test_a_caller_s_capture_gets_the_kernel_chain(family, monkeypatch):
    """step_gpu_only and a language model's decode_step captured by the caller on the engine's stream: the graph holds the kernel
    chain (its replays take no turns), so every replay, with eager work in between, leaves the bits of an engine that has only the
    chain; the engine's own steps are resident before and after."""
    import torch
    make, dm, lm_of = _family(family)
    a = make()
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = make()
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((4, dm)).astype(np.float32)
    embed = rng.standard_normal((128, dm)).astype(np.float32)
    print(f"case capture by the caller {family}", flush=True)
    resident = a.step(x)
    chain.step(x)
    lms = []
    for e in (a, chain):
        lm = lm_of(e, embed)
        lm.set_tokens(np.arange(4, dtype=np.int32))
        lm.decode_step()          # (the head's GEMM library settles its choice outside the captures)
        e.sync()
        lms.append(lm)
    lms[0].capture_graph()
    graphs = []
    for e, lm in zip((a, chain), lms):
        for call in (e.step_gpu_only, lm.decode_step):
            side = torch.cuda.ExternalStream(e.stream())
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side, capture_error_mode="thread_local"):
                call()
            graphs.append((e, side, g))

    def replay(i):
        e, side, g = graphs[i]
        with torch.cuda.stream(side):
            g.replay()
    for e, lm in zip((a, chain), lms):
        e.reset()
        lm.set_tokens(np.arange(4, dtype=np.int32))
    for n in range(4):
        rows, toks = [], []
        for i, (e, lm) in enumerate(zip((a, chain), lms)):
            replay(2 * i + n % 2)
            replay(2 * i + 1)
            rows.append(lm.last_logits())
            toks.append(lm.get_tokens())
            _ = torch.ones(1 << 16, device="cuda").sum().item()
        assert np.array_equal(rows[0], rows[1]) and np.array_equal(toks[0], toks[1]), n
        assert np.isfinite(rows[0]).all()
    a.reset()
    assert np.array_equal(a.step(x), resident) and a.decode_route() == 2
    del graphs
    for e in (*lms, a, chain):
        e.close()


@pytest.mark.parametrize("dm,B", [(32, 4), (64, 16), (256, 8)])
def test_conv_windows_move_by_one_step(dm, B):
    """Narrow models, where a workgroup's waves read a conv window at nearly the time its first wave stores the next one: after every
    step each window holds the last three entries of the one before, and a second engine has the same bits."""
    a, b = _engines((dm, 2, B), 2)
    rng = np.random.default_rng(dm)
    print(f"case conv windows {dm} x {B}", flush=True)
    assert a.decode_route() == 2
    old = [a.download_state(l)[0] for l in range(2)]
    for t in range(60):
        x = rng.standard_normal((B, dm)).astype(np.float32)
        assert np.array_equal(a.step(x), b.step(x)), t
        for l in range(2):
            new = a.download_state(l)[0]
            assert np.array_equal(new[..., :3], old[l][..., 1:]), (t, l)
            old[l] = new
    a.close()
    b.close()


def _states(e):
    """All recurrent states, whatever the engine's check says."""
    from mamba_rs_amd import backbone, mamba3
    out = []
    for l in range(e.cfg.n_layers):
        if isinstance(e, GpuMambaBackbone):
            parts = [np.empty((e.batch, e.cfg.d_inner(), n), np.float32) for n in (e.cfg.d_conv, e.cfg.d_state)]
            backbone._bind().mrs_backbone_download_state(e._h, l, *map(backbone._fp, parts))
        else:
            nh, hd, ds = e.cfg.nheads(), e.cfg.headdim, e.cfg.d_state
            na = max(1, e.cfg.num_rope_angles())
            parts = [np.empty((e.batch, *n), np.float32) for n in ((nh, hd, ds), (nh, ds), (nh, hd), (nh, na))]
            mamba3._bind().mrs_m3_backbone_download_state(e._h, l, *map(backbone._fp, parts))
        out += parts
    return out


@pytest.mark.parametrize("family", ["m1", "m3", "m1rows"])
def test_a_step_that_finds_no_places(family, monkeypatch):
    """A wait of 0 calls every resident launch off.  step() then has the kernel chain's bits, from whatever state it started in; queued
    steps leave the state alone and raise at the next call that waits for them, however many there are; after a reset the engine
    steps as before."""
    from mamba_rs_amd import MambaHipError
    make, dm, lm_of = _family(family)
    a = make()
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = make()
    rng = np.random.default_rng(6)
    x = rng.standard_normal((4, 4, dm)).astype(np.float32)
    print(f"case called off {family}", flush=True)
    lm = lm_of(a, rng.standard_normal((128, dm)).astype(np.float32))
    resident = [a.step(r) for r in x]
    before = _states(a)

    a.set_resident_wait(0)
    for _ in range(50):
        a.step_gpu_only()
    for _ in range(2):                      # it stays an error
        with pytest.raises(MambaHipError, match="did not come free"):
            a.sync()
    with pytest.raises(MambaHipError, match="did not come free"):
        a.step(x[0])
    assert all(np.array_equal(p, q) for p, q in zip(before, _states(a)))

    a.reset()
    for r in x:                             # called off each time the engine was reset, else on the chain at once
        assert np.array_equal(a.step(r), chain.step(r))
    assert all(np.array_equal(p, q) for p, q in zip(_states(a), _states(chain)))
    a.step_gpu_only()
    a.sync()
    a.reset()
    lm.set_tokens(np.arange(4, dtype=np.int32))
    lm.capture_graph()                      # its warm-up step is called off: the replays are kernel chains until a reset
    lm.decode_step()
    assert np.isfinite(lm.last_logits()).all()
    a.reset()
    lm.decode_step()
    with pytest.raises(MambaHipError, match="did not come free"):
        lm.get_tokens()

    a.reset()
    a.set_resident_wait(1 << 23)
    for r, want in zip(x, resident):
        assert np.array_equal(a.step(r), want)
    for e in (lm, a, chain):
        e.close()


@pytest.mark.parametrize("family", ["m1", "m3", "m1rows"])
def test_a_reset_waits_for_the_steps_before_it(family):
    """Steps that are called off while a reset is already asked for: the reset waits for them, says once that they were lost, and the
    engine steps as a fresh one; a second reset has nothing to say."""
    from mamba_rs_amd import MambaHipError
    make, dm, _ = _family(family)
    a = make()
    x = np.random.default_rng(7).standard_normal((4, dm)).astype(np.float32)
    print(f"case reset behind lost steps {family}", flush=True)
    want = a.step(x)
    a.reset()
    for _ in range(3):
        a.set_resident_wait(0)
        for _ in range(20):
            a.step_gpu_only()
        with pytest.raises(MambaHipError, match="not carried out"):
            a.reset()
        a.set_resident_wait(1 << 23)
        assert np.array_equal(a.step(x), want)
        a.reset()
        assert np.array_equal(a.step(x), want)
        a.reset()
    a.close()


@pytest.mark.parametrize("family", ["m1", "m3"])
def test_generation_hands_out_no_token_of_a_lost_step(family, monkeypatch):
    """Streaming and batched generation whose steps are called off: from the start, the kernel chain generates instead (its own
    engine's tokens); behind the third token, the caller has exactly the three it was given, and an error."""
    from mamba_rs_amd import MambaHipError, SampleParams
    make, dm, lm_of = _family(family, 1)
    a = make()
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = make()
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    embed = np.random.default_rng(8).standard_normal((128, dm)).astype(np.float32)
    prompt, params = [5, 9, 2], SampleParams(temperature=0.9, top_k=20, max_tokens=8, seed=3)
    print(f"case generation behind lost steps {family}", flush=True)
    lm, lm_chain = lm_of(a, embed), lm_of(chain, embed)

    def stream(m, at=lambda n: None):
        got = []

        def take(tok):
            got.append(tok)
            at(len(got))
        try:
            m.generate_streaming(prompt, params, take)
        except MambaHipError as e:
            return got, e
        return got, None
    whole, err = stream(lm)
    assert err is None and len(whole) == 8
    got, err = stream(lm, lambda n: a.set_resident_wait(0) if n == 3 else None)
    assert got == whole[:3] and "did not come free" in str(err)
    assert stream(lm) == stream(lm_chain)                  # (the wait is still 0)
    assert lm.generate_batch([prompt], [params]) == lm_chain.generate_batch([prompt], [params])
    a.set_resident_wait(1 << 23)
    assert stream(lm) == (whole, None)
    for e in (lm, lm_chain, a, chain):
        e.close()


@pytest.mark.parametrize("family", ["m1", "m1rows"])
def test_prompts_in_pieces_before_lost_steps(family, monkeypatch):
    """Prompts that go through the prefill kernels in front of steps that are called off: the generation starts over on the kernel chain,
    prompts and all, with that engine's tokens and states; behind a streamed token the caller has what it was given, and an error; the
    next generation, with places, is the first one again."""
    from mamba_rs_amd import MambaHipError, SampleParams
    rows = 1 if family == "m1" else 3
    make, dm, lm_of = _family(family, rows)
    a = make()
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = make()
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    rng = np.random.default_rng(13)
    embed = rng.standard_normal((128, dm)).astype(np.float32)
    prompts = [rng.integers(0, 128, n).tolist() for n in (41, 37, 44)[:rows]]      # two pieces
    params = [SampleParams(temperature=0.9, top_k=20, max_tokens=6, seed=i) for i in range(rows)]
    print(f"case prompts in pieces before lost steps {family}", flush=True)
    lm, lm_chain = lm_of(a, embed), lm_of(chain, embed)
    want, want_chain = lm.generate_batch(prompts, params), lm_chain.generate_batch(prompts, params)
    a.set_resident_wait(0)
    for _ in range(2):
        assert lm.generate_batch(prompts, params) == want_chain
        assert all(np.array_equal(p, q) for p, q in zip(_states(a), _states(chain)))
    a.set_resident_wait(1 << 23)
    assert lm.generate_batch(prompts, params) == want
    if rows == 1:
        got = []

        def take(tok):
            got.append(tok)
            if len(got) == 2:
                a.set_resident_wait(0)
        with pytest.raises(MambaHipError, match="did not come free"):
            lm.generate_streaming(prompts[0], params[0], take)
        assert got == want[0][:2]
        a.set_resident_wait(1 << 23)
        assert lm.generate_batch(prompts, params) == want
    for e in (lm, lm_chain, a, chain):
        e.close()


def test_a_second_process_keeps_the_kernel_chain(monkeypatch, tmp_path):
    """While this process has resident engines on the GPU, another process's engine has the kernel chain, with the chain's bits."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    a, = _engines((256, 2, 2), 1)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain, = _engines((256, 2, 2), 1)
    monkeypatch.delenv("MRS_DECODE_NO_RESIDENT")
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    x = np.random.default_rng(9).standard_normal((2, 256)).astype(np.float32)
    np.save(tmp_path / "x.npy", x)
    program = ("import sys; sys.path[:0] = sys.argv[1:3]; import numpy as np; from test_resident_gpu import _engines\n"
               "e, = _engines((256, 2, 2), 1); np.save(sys.argv[3] + '/y.npy', e.step(np.load(sys.argv[3] + '/x.npy'))); print(e.decode_route())")
    print("case a second process", flush=True)
    r = subprocess.run([sys.executable, "-c", program, os.path.dirname(here), here, str(tmp_path)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1] == "1", r.stdout + r.stderr
    assert np.array_equal(np.load(tmp_path / "y.npy"), chain.step(x))
    a.step(x)
    for e in (a, chain):
        e.close()


@pytest.mark.parametrize("layer", [0, 1])
def test_an_infinite_share_stays_infinite(layer, monkeypatch):
    """One entry of a layer's x_proj row overflows to -inf in one workgroup's share (a dt entry whose weights are positive, so the step
    size becomes 0 and every output is finite): the exchange hands it on as -inf, and the rows are the kernel chain's."""
    cfg = MambaConfig(d_model=64, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.init(cfg, 64, 5)
    w.input_proj_w = np.zeros((0, 64), np.float32)
    lw = w.layers[layer]
    lw.conv1d_bias[3] = 8.0
    lw.x_proj_w.reshape(cfg.d_inner(), -1)[:, 0] = 0.0
    lw.x_proj_w.reshape(cfg.d_inner(), -1)[3, 0] = -3e38
    lw.dt_proj_w.reshape(-1, cfg.d_inner())[0, :] = 0.5
    a = GpuMambaBackbone.new_with_dtype(0, w, cfg, 64, 2, WeightDtype.BF16)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = GpuMambaBackbone.new_with_dtype(0, w, cfg, 64, 2, WeightDtype.BF16)
    print(f"case infinite share in layer {layer}", flush=True)
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    for x in np.random.default_rng(10).standard_normal((5, 2, 64)).astype(np.float32):
        got, want = a.step(x), chain.step(x)
        assert np.isfinite(want).all() and np.isfinite(got).all()
        assert min(cosine(g, c) for g, c in zip(got, want)) >= 0.999
    a.close()
    chain.close()


@pytest.mark.parametrize("family", ["m1", "m3"])
def test_a_replayed_step_that_finds_no_places(family, monkeypatch):
    """With an input projection the engine's graph holds the resident launch: called off, its step is the kernel chain's, eager, until
    a reset; then the graph is replayed again."""
    if family == "m1":
        cfg = MambaConfig(d_model=64, d_state=16, d_conv=4, expand=2, n_layers=2)
        w = MambaWeights.init(cfg, 20, 3)

        def make():
            return GpuMambaBackbone.new_with_dtype(0, w, cfg, 20, 4, WeightDtype.F16)
    else:
        from mamba_rs_amd import GpuMamba3Backbone
        from test_m3_engine_gpu import perturbed
        from test_resident_m3_gpu import cfg_
        cfg = cfg_(64, 16, 16, 1, 2)
        w = perturbed(cfg, 20, 3)

        def make():
            return GpuMamba3Backbone.new_with_dtype(0, w, cfg, 20, 4, WeightDtype.F16)
    a = make()
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = make()
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    x = np.random.default_rng(11).standard_normal((3, 4, 20)).astype(np.float32)
    print(f"case replay called off {family}", flush=True)
    a.capture_graph()
    resident = [a.step(r) for r in x]
    a.reset()
    a.set_resident_wait(0)
    for r in x:
        assert np.array_equal(a.step(r), chain.step(r))
    a.reset()
    a.set_resident_wait(1 << 23)
    for r, want in zip(x, resident):
        assert np.array_equal(a.step(r), want)
    a.close()
    chain.close()


def test_steps_queued_before_an_engine_was_there(monkeypatch):
    """Steps that were queued while an engine had the chip to itself carry no event: an engine that does not fit beside it steps on the
    kernel chain until somebody has waited for them, or the first engine has launched again."""
    a, = _engines((768, 2, 4), 1)
    x = np.random.default_rng(12).standard_normal((4, 768)).astype(np.float32)
    want = a.step(x)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain, = _engines((768, 2, 4), 1)
    monkeypatch.delenv("MRS_DECODE_NO_RESIDENT")
    want_chain = chain.step(x)
    assert not np.array_equal(want, want_chain)     # (the two routes can be told apart here)
    print("case steps from before", flush=True)
    for settle in (a.sync, a.step_gpu_only):
        a.step_gpu_only()
        b, = _engines((768, 2, 4), 1)
        assert np.array_equal(b.step(x), want_chain)
        settle()
        b.reset()
        assert np.array_equal(b.step(x), want)
        b.close()
        a.sync()
    a.close()
    chain.close()
