"""GPU: the resident Mamba-3 decode step (a whole 16-bit step in one launch whose workgroups exchange through memory) against the
CPU route, against the kernel chain it replaces, and against itself: eager and replayed, beside a second engine (queued steps, threads and
captures of both networks: test_resident_gpu.py)."""
import numpy as np
import pytest

import orc
from util import cosine, scaled_err
from test_m3_engine_gpu import oracle_params, perturbed

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMamba3Backbone, Mamba3Config, Mamba3Weights, WeightDtype  # noqa: E402


def cfg_(dm, ds, hd, ng, L, rope=0.5):
    return Mamba3Config(d_model=dm, d_state=ds, expand=2, headdim=hd, ngroups=ng, n_layers=L, rope_fraction=rope)


@pytest.mark.parametrize("cfg,idim,B", [
    (cfg_(64, 16, 16, 1, 3), 20, 16),          # input projection; 4 lanes per state row; sixteen groups of eight workgroups
    (cfg_(64, 32, 32, 2, 2), 64, 3),           # two B/C groups, 8 lanes per row, eight channels per workgroup: four workgroups per head
    (cfg_(64, 64, 64, 1, 2, 1.0), 64, 5),      # every coordinate rotated, 11 shared columns per workgroup, the last one's share cut short
    (cfg_(256, 16, 16, 1, 2), 256, 8),         # 32 workgroups per row: every compute unit
    (cfg_(768, 64, 64, 1, 2), 768, 1),         # 96 workgroups, some without a share of the shared columns
    (cfg_(768, 64, 64, 1, 2), 768, 2),
    (cfg_(1024, 64, 64, 1, 2), 1024, 1),       # the widest: 128 workgroups, four and eight k-steps per wave
])
@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
def test_resident_step_follows_the_cpu_route(cfg, idim, B, dtype, monkeypatch):
    """Six steps (three eager, three replayed): every row within the 16-bit engines' tolerance of the CPU route on
    storage-rounded weights (cosine >= 0.999, as for the kernel chain), all four states as well; the kernel chain on the same
    weights agrees as closely.  A second engine steps behind the first and ends on the same bits: all sums are in a fixed
    order."""
    w = perturbed(cfg, idim, 11)
    if idim == cfg.d_model:
        w.input_proj_w = np.zeros(0, np.float32)
    identity = w.input_proj_w.size == 0
    code = orc.BF16 if dtype == WeightDtype.BF16 else orc.F16
    wo = Mamba3Weights(np.eye(idim, dtype=np.float32), np.zeros(idim, np.float32), w.layers, w.norm_f_weight) if identity else w
    P = oracle_params(wo, cfg, idim, round_to=code)
    print(f"case resident Mamba-3 step d_model={cfg.d_model} d_state={cfg.d_state} groups={cfg.ngroups} batch={B} {dtype.name}", flush=True)
    a = GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, B, dtype)
    b = GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, B, dtype)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, B, dtype)
    assert (a.decode_route(), b.decode_route(), chain.decode_route()) == (2, 2, 1)      # one launch, one launch, own chain
    rng = np.random.default_rng(cfg.d_model + B)
    x = rng.standard_normal((6, B, idim)).astype(np.float32)
    rows = sorted({0, B // 2, B - 1})
    st = {r: P.zero_state() for r in rows}
    for t in range(6):
        if t == 3:
            a.capture_graph()
        got = a.step(x[t])
        assert np.array_equal(b.step(x[t]), got), t
        assert min(cosine(g, c) for g, c in zip(got, chain.step(x[t]))) >= 0.999, t
        for r in rows:
            want = orc.m3_backbone_step(P, x[t, r], st[r])
            assert cosine(got[r], want) >= 0.999, (t, r, cosine(got[r], want))
    for l in range(cfg.n_layers):
        ssm, k, v, ang = a.download_state(l)
        for r in rows:
            for g, s in ((ssm, 0), (k, 1), (v, 2)):
                assert cosine(g[r], st[r][s][l]) >= 0.999 and scaled_err(g[r], st[r][s][l]) < 5e-2, (l, r, s, cosine(g[r], st[r][s][l]))
            # angles live on a circle; six steps of sums of 16-bit-rounded inputs through at most three layers
            assert np.max(np.abs(np.sin(ang[r]) - np.sin(st[r][3][l]))) < 0.1 and np.max(np.abs(np.cos(ang[r]) - np.cos(st[r][3][l]))) < 0.1, (l, r)
    a.reset()
    b.reset()
    assert np.array_equal(a.step(x[0]), b.step(x[0]))
    for e in (a, b, chain):
        e.close()


@pytest.mark.parametrize("layers,route", [(4, 2), (5, 1)])
def test_deep_models_keep_the_kernel_chain(layers, route, monkeypatch):
    """Five layers and more step on the chain, with its bits; up to four the resident step stays within twice the 0.2 % of the output by
    which two orders of the chain's own sums differ there (measured, 32 steps)."""
    cfg = cfg_(256, 16, 16, 1, layers)
    w = perturbed(cfg, 256, 3)
    w.input_proj_w = np.zeros(0, np.float32)
    a = GpuMamba3Backbone.new_with_dtype(0, w, cfg, 256, 2, WeightDtype.BF16)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = GpuMamba3Backbone.new_with_dtype(0, w, cfg, 256, 2, WeightDtype.BF16)
    assert (a.decode_route(), chain.decode_route()) == (route, 1)
    x = np.random.default_rng(layers).standard_normal((32, 2, 256)).astype(np.float32)
    got, want = np.stack([a.step(r) for r in x]), np.stack([chain.step(r) for r in x])
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"case {layers} layers: resident against chain {rel:.2e}", flush=True)
    assert rel == 0 if route == 1 else rel < 4e-3
    a.close()
    chain.close()


@pytest.mark.parametrize("cfg,idim,dtype", [
    (cfg_(256, 16, 16, 1, 6), 256, WeightDtype.BF16),              # 32 lanes per row of in_proj, 4 lanes per state row
    (cfg_(256, 64, 64, 4, 5, 1.0), 20, WeightDtype.F16),           # input projection, every coordinate rotated, 16 shared columns cut short
    (cfg_(512, 32, 32, 2, 5, 1.0), 512, WeightDtype.BF16),         # 64 lanes per row, one piece each; 8 lanes per state row
    (cfg_(512, 32, 8, 1, 5), 512, WeightDtype.F16),                # eight channels and four columns of out_proj per workgroup: idle waves
    (cfg_(768, 64, 64, 1, 3), 768, WeightDtype.F16),
    (cfg_(1024, 64, 64, 1, 2), 1024, WeightDtype.BF16),
    (cfg_(1024, 64, 64, 1, 20), 1024, WeightDtype.BF16),           # more weights than the last cache holds: some layers' are read past it
])
def test_one_row_keeps_the_chain_s_bits(cfg, idim, dtype, monkeypatch):
    """One row at any depth: one launch, and output and states are the kernel chain's bit for bit -- eager, replayed, in steps that
    are called off and run on the chain in between, and with infinities in the input (where the chain has NaN, NaN)."""
    w = perturbed(cfg, idim, 13)
    if idim == cfg.d_model:
        w.input_proj_w = np.zeros(0, np.float32)
    print(f"case one row d_model={cfg.d_model} d_state={cfg.d_state} headdim={cfg.headdim} groups={cfg.ngroups} {dtype.name}", flush=True)
    a = GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, 1, dtype)
    monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    chain = GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, 1, dtype)
    assert (a.decode_route(), chain.decode_route()) == (2, 1)
    same = lambda p, q: np.array_equal(p, q, equal_nan=True)
    x = np.random.default_rng(idim).standard_normal((12, 1, idim)).astype(np.float32)
    x[11, 0, 3] = np.inf
    for t, r in enumerate(x):
        if t == 4:
            a.capture_graph()
        if t == 8:      # (the state is not touched by a launch that is called off)
            a.set_resident_wait(0)
        assert same(a.step(r), chain.step(r)), t
        if t >= 10:
            continue
        for l in range(cfg.n_layers):
            assert all(same(p, q) for p, q in zip(a.download_state(l), chain.download_state(l))), (t, l)
    a.reset()
    chain.reset()
    a.set_resident_wait(1 << 23)
    for r in x:
        assert same(a.step(r), chain.step(r))
    for e in (a, chain):
        e.close()
