"""GPU parity: the Mamba-1 backbone / LM engines vs the oracle's restatement of the reference CPU path.

The test bodies follow the reference's own engine tests (tests/m1_test_correctness.rs:17-146, 732-860;
tests/prefill.rs:173-232; tests/mixed_prefill_parity.rs:116-153).
"""
import numpy as np
import pytest

import orc
from util import cosine, det, max_rel, scaled_err

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMambaBackbone, GpuMambaLM, MambaConfig, MambaWeights, ScanMode, WeightDtype  # noqa: E402


def oracle_params(w: MambaWeights, cfg: MambaConfig, input_dim: int, round_to=None) -> orc.M1Params:
    """Copy product-side weights into the oracle's flat block (optionally with the bulk matrices rounded to a storage dtype)."""
    P = orc.M1Params(cfg.d_model, cfg.d_state, cfg.d_conv, cfg.expand, cfg.n_layers, max(input_dim, 1), seed=0)
    rq = (lambda a: orc.round_to(a, round_to)) if round_to is not None else (lambda a: a)
    if w.input_proj_w.size:
        P.input_proj_w[:] = w.input_proj_w; P.input_proj_b[:] = w.input_proj_b
    for l, lw in enumerate(w.layers):
        d = P.layers[l]
        d["norm_weight"][:] = lw.norm_weight
        d["in_proj_w"][:] = rq(lw.in_proj_w); d["x_proj_w"][:] = rq(lw.x_proj_w)
        d["dt_proj_w"][:] = rq(lw.dt_proj_w); d["out_proj_w"][:] = rq(lw.out_proj_w)
        d["conv1d_weight"][:] = lw.conv1d_weight; d["conv1d_bias"][:] = lw.conv1d_bias
        d["dt_proj_b"][:] = lw.dt_proj_b; d["a_log"][:] = lw.a_log; d["a_neg"][:] = -np.exp(lw.a_log); d["d_param"][:] = lw.d_param
    P.norm_f_weight[:] = w.norm_f_weight
    return P


TINY = MambaConfig(d_model=128, d_state=16, d_conv=4, expand=2, n_layers=2)   # the tiny CPU configuration


def test_weights_init_matches_oracle_init():
    w = MambaWeights.init(TINY, 128, 42)
    P = orc.M1Params(128, 16, 4, 2, 2, 128, seed=42)
    assert np.array_equal(w.input_proj_w, P.input_proj_w)
    for l in range(2):
        for k in ("in_proj_w", "conv1d_weight", "x_proj_w", "dt_proj_w", "out_proj_w"):
            assert np.array_equal(getattr(w.layers[l], k), P.layers[l][k]), k
        assert np.allclose(w.layers[l].dt_proj_b, P.layers[l]["dt_proj_b"], atol=2e-6)
        assert np.allclose(w.layers[l].a_log, P.layers[l]["a_log"], atol=2e-7)


def test_f32_engine_step_sequence_matches_cpu_reference_path():
    """Tiny config, f32, batch 1, 256 steps: every step output and the final states against the CPU route
    (tests/m1_test_correctness.rs:732-779 does this with max_diff < 5.0; here rel 1e-4 of the output scale)."""
    w = MambaWeights.init(TINY, 128, 42)
    P = oracle_params(w, TINY, 128)
    eng = GpuMambaBackbone.new(0, w, TINY, 128, 1)
    conv, ssm = orc.m1_zero_state(P)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((256, 128)).astype(np.float32)
    worst = 0.0
    for t in range(256):
        got = eng.step(x[t])
        want = orc.m1_backbone_step(P, x[t], conv, ssm)
        worst = max(worst, scaled_err(got[0], want))
    assert worst < 1e-4, worst
    for l in range(2):
        c, s = eng.download_state(l)
        assert scaled_err(s[0], ssm[l].reshape(256, 16)) < 1e-4
        assert np.allclose(c[0][:, 1:], conv[l].reshape(256, 3), atol=1e-5)       # GPU keeps d_conv slots, CPU d_conv-1
    # reset reproduces; state carries
    eng.reset()
    a = eng.step(x[0]); b = eng.step(x[0])
    assert np.max(np.abs(a - b)) > 1e-6
    eng.reset()
    assert np.array_equal(eng.step(x[0]), a)
    eng.close()


def test_f32_prefill_matches_cpu_prefill_and_hands_over_to_step():
    # tests/prefill.rs:173-232: prefill T then one step == T+1 steps (cos > 0.9999, max_rel < 1e-2)
    w = MambaWeights.init(TINY, 128, 42)
    P = oracle_params(w, TINY, 128)
    T = 256
    rng = np.random.default_rng(2)
    x = rng.standard_normal((T + 1, 128)).astype(np.float32)
    for mode in (ScanMode.SEQUENTIAL, ScanMode.PARALLEL):
        cfg = MambaConfig(d_model=128, d_state=16, d_conv=4, expand=2, n_layers=2, scan_mode=mode)
        eng = GpuMambaBackbone.new(0, w, cfg, 128, 1)
        last = eng.prefill_sequence(x[None, :T])
        conv, ssm = orc.m1_zero_state(P)
        ref = orc.m1_backbone_prefill(P, x[:T], conv, ssm)
        assert scaled_err(last[0], ref[-1]) < 1e-4, mode
        for l in range(2):
            assert scaled_err(eng.download_state(l)[1][0], ssm[l].reshape(256, 16)) < 1e-4
        nxt = eng.step(x[T])
        want = orc.m1_backbone_step(P, x[T], conv, ssm)
        assert cosine(nxt[0], want) > 0.9999 and max_rel(nxt[0], want, floor=1e-3) < 1e-2
        eng.close()


def test_batch_equals_individual_and_graph_equals_eager():
    # tests/m1_test_correctness.rs:100-146 (batch == individual) and :781-860 (graph == eager, 1e-5)
    cfg = MambaConfig(d_model=64, d_state=16, d_conv=4, expand=2, n_layers=3)
    w = MambaWeights.init(cfg, 20, 7)
    B = 4
    x = det(6 * B * 20, 9, 2.0).reshape(6, B, 20)
    eng = GpuMambaBackbone.new(0, w, cfg, 20, B)
    outs = [eng.step(x[t]) for t in range(6)]
    for b in range(B):
        one = GpuMambaBackbone.new(0, w, cfg, 20, 1)
        for t in range(6):
            assert np.allclose(one.step(x[t, b]), outs[t][b], atol=1e-5)
        one.close()
    eng.reset()
    eng.capture_graph()
    for t in range(6):
        assert np.allclose(eng.step(x[t]), outs[t], atol=1e-5), t      # replays stay equal to eager, step after step
    eng.reset()
    assert np.allclose(eng.step(x[0]), outs[0], atol=1e-5)
    eng.close()


@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
def test_16bit_engine_tracks_f32_reference(dtype):
    """bf16/f16 storage engine vs the CPU route run on weights rounded to the storage type.  Activations are
    rounded between kernels, so this is a tolerance test: cosine >= 0.999 per step, as the reference's
    mixed-precision parity tests (tests/mixed_prefill_parity.rs:125-134)."""
    w = MambaWeights.init(TINY, 128, 42)
    code = orc.BF16 if dtype == WeightDtype.BF16 else orc.F16
    P = oracle_params(w, TINY, 128, round_to=code)
    eng = GpuMambaBackbone.new_with_dtype(0, w, TINY, 128, 2, dtype)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((40, 2, 128)).astype(np.float32)
    st = [orc.m1_zero_state(P) for _ in range(2)]
    for t in range(40):
        got = eng.step(x[t])
        for b in range(2):
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (t, b)
    # parallel-scan prefill route vs sequential route on the same engine type (mixed_prefill_parity.rs)
    T = 300
    xs = rng.standard_normal((2, T, 128)).astype(np.float32)
    outs = []
    for mode in (ScanMode.SEQUENTIAL, ScanMode.PARALLEL):
        cfg = MambaConfig(d_model=128, d_state=16, d_conv=4, expand=2, n_layers=2, scan_mode=mode)
        e2 = GpuMambaBackbone.new_with_dtype(0, w, cfg, 128, 2, dtype)
        outs.append((e2.prefill_sequence(xs), e2.download_state(1)[1]))
        e2.close()
    assert cosine(outs[0][0], outs[1][0]) >= 0.999 and cosine(outs[0][1], outs[1][1]) >= 0.999
    conv, ssm = orc.m1_zero_state(P)
    ref = orc.m1_backbone_prefill(P, xs[0], conv, ssm)
    assert cosine(outs[1][0][0], ref[-1]) >= 0.999
    eng.close()


def test_lm_greedy_decode_and_prefill():
    """Greedy LM loop with a tied head on a small random LM: every generated token must be the (last) argmax of
    the oracle's logits, for the step-by-step path and for prefill + decode."""
    cfg = MambaConfig(d_model=64, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.random_lm(cfg, seed=5, std=0.1)
    vocab = 300
    rng = np.random.default_rng(6)
    embed = (rng.standard_normal((vocab, 64)) * 0.5).astype(np.float32)
    P = oracle_params(w, cfg, 64)
    eng = GpuMambaBackbone.new(0, w, cfg, 64, 1)
    lm = GpuMambaLM(eng, embed)
    prompt = [int(v) for v in rng.integers(0, vocab, 12)]

    def oracle_generate(n):
        conv, ssm = orc.m1_zero_state(P)
        h = None
        for tok in prompt:
            h = orc.m1_backbone_step(P, embed[tok], conv, ssm, identity_proj=True)
        out = []
        for _ in range(n):
            logits = embed @ h
            tok = int(np.flatnonzero(logits == logits.max())[-1])
            margin = np.sort(logits)[-1] - np.sort(logits)[-2]
            out.append((tok, margin))
            h = orc.m1_backbone_step(P, embed[tok], conv, ssm, identity_proj=True)
        return out

    want = oracle_generate(8)
    got = lm.generate(prompt, 8)                          # prefill path
    for (tok, margin), g in zip(want, got):
        if margin < 1e-3:
            break                                          # a near-tie may legitimately flip across routes
        assert g == tok
    logits = lm.last_logits()
    assert logits.shape == (1, vocab) and np.isfinite(logits).all()
    # step-by-step path with a captured graph gives the same tokens as eager prefill path
    eng.reset()
    for tok in prompt[:-1]:
        lm.set_tokens([tok]); lm.decode_step()
    lm.set_tokens([prompt[-1]])
    lm.capture_graph()
    seq = []
    for _ in range(8):
        lm.decode_step(); seq.append(int(lm.get_tokens()[0]))
    assert seq[:3] == got[:3]
    lm.close(); eng.close()


def test_engine_rejects_bad_config():
    from mamba_rs_amd import MambaHipError
    cfg = MambaConfig(d_model=64, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, 10, 1)
    with pytest.raises(ValueError):
        GpuMambaBackbone.new(0, w, MambaConfig(d_model=64, d_state=300, n_layers=1), 10, 1)
    with pytest.raises(ValueError):
        GpuMambaBackbone.new(0, w, cfg, 11, 1)            # weight / input_dim mismatch
    eng = GpuMambaBackbone.new(0, w, cfg, 10, 1)
    with pytest.raises(ValueError):
        eng.step(np.zeros(3, np.float32))
    with pytest.raises(MambaHipError):
        eng.alloc_prefill_scratch(1)                      # one token is a step, not a prefill
    eng.alloc_prefill_scratch(16)
    eng.alloc_prefill_scratch(32)                         # the scratch follows the sequence length
    eng.close()


def test_16bit_engine_batch_above_64_takes_the_library_gemm_chain():
    """The own skinny GEMM serves batch <= 64; a batch of 65 runs add+RMSNorm, vendor GEMMs, conv step and the fused
    scan step instead.  Same bar as the small-batch chain: cosine >= 0.999 per step against the CPU route on rounded
    weights, and rows 0 and 64 (first row of the fifth 16-row tile, were it tiled) behave alike."""
    w = MambaWeights.init(TINY, 128, 43)
    P = oracle_params(w, TINY, 128, round_to=orc.BF16)
    B = 65
    eng = GpuMambaBackbone.new_with_dtype(0, w, TINY, 128, B, WeightDtype.BF16)
    rng = np.random.default_rng(8)
    x = rng.standard_normal((12, B, 128)).astype(np.float32)
    rows = (0, 31, 64)
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(12):
        got = eng.step(x[t])
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (t, b)
    eng.close()


def test_wide_dt_rank_at_large_batch_runs_dt_proj_as_its_own_gemm():
    """batch x dt_rank above the fusion limit (4096): the decode step takes delta from a GEMM instead of forming it
    inside the step kernel -- own-GEMM chain at batch 40, the last row count it takes for a wide model (d_model 2048 ->
    dt_rank 128, 40 x 128 = 5120), and library chain at batch 41 and 65."""
    cfg = MambaConfig(d_model=2048, d_state=16, d_conv=4, expand=1, n_layers=1)
    w = MambaWeights.init(cfg, 2048, 44)
    w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    P = oracle_params(w, cfg, 2048, round_to=orc.BF16)
    P.input_proj_w[:] = np.eye(2048, dtype=np.float32); P.input_proj_b[:] = 0
    rng = np.random.default_rng(4)
    for B in (40, 41, 65):
        eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 2048, B, WeightDtype.BF16)
        x = rng.standard_normal((4, B, 2048)).astype(np.float32)
        rows = (0, B - 1)
        st = {b: orc.m1_zero_state(P) for b in rows}
        for t in range(4):
            got = eng.step(x[t])
            for b in rows:
                want = orc.m1_backbone_step(P, x[t, b], *st[b])
                assert cosine(got[b], want) >= 0.999, (B, t, b)
        eng.close()


@pytest.mark.parametrize("B", [100, 128])
def test_narrow_model_keeps_the_own_chain_up_to_128_rows(B):
    """Above 64 rows (up to 128 for narrow models) the decode chain still runs on the library's own GEMM, with dt_proj as
    a launch of its own (batch x dt_rank above the fusion limit).  First, middle and last row against the CPU route."""
    cfg = MambaConfig(d_model=768, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.random_lm(cfg, seed=B, std=0.05)
    P = oracle_params(w, cfg, 768, round_to=orc.BF16)
    P.input_proj_w[:] = np.eye(768, dtype=np.float32); P.input_proj_b[:] = 0
    rng = np.random.default_rng(B)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 768, B, WeightDtype.BF16)
    x = rng.standard_normal((4, B, 768)).astype(np.float32)
    rows = (0, B // 2, B - 1)
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(4):
        if t == 2:
            eng.capture_graph()
        got = eng.step(x[t])
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (B, t, b)
    eng.close()


@pytest.mark.parametrize("dm,B", [(1024, 41), (1024, 65), (1280, 128), (1536, 97)])
def test_models_of_middle_width_keep_the_own_chain_up_to_128_rows(dm, B):
    """Widths between those of the narrow models and of the column-tile kernel's, at rows that were the library's: as above."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.random_lm(cfg, seed=B, std=0.05)
    P = oracle_params(w, cfg, dm, round_to=orc.BF16)
    P.input_proj_w[:] = np.eye(dm, dtype=np.float32); P.input_proj_b[:] = 0
    rng = np.random.default_rng(B)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.BF16)
    x = rng.standard_normal((3, B, dm)).astype(np.float32)
    rows = (0, B // 2, B - 1)
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(3):
        got = eng.step(x[t])
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (B, t, b)
    eng.close()


@pytest.mark.parametrize("B", [1, 3, 20])
def test_wide_model_runs_x_proj_as_a_split_k_launch(B):
    """d_inner 2048 x xdbl 96: a row's per-tile shares would be 48 KB, so x_proj does not ride in the in_proj launch; it
    runs as its own launch with K cut into slices whose shares the step kernel sums -- on the matrix cores also at one to
    four rows.  Checked against the CPU route on storage-rounded weights, step after step."""
    cfg = MambaConfig(d_model=1024, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.init(cfg, 1024, 45)
    w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    P = oracle_params(w, cfg, 1024, round_to=orc.BF16)
    P.input_proj_w[:] = np.eye(1024, dtype=np.float32); P.input_proj_b[:] = 0
    rng = np.random.default_rng(B)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 1024, B, WeightDtype.BF16)
    x = rng.standard_normal((5, B, 1024)).astype(np.float32)
    rows = sorted({0, B - 1})
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(5):
        if t == 2:
            eng.capture_graph()
        got = eng.step(x[t])
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (B, t, b)
    eng.close()


@pytest.mark.parametrize("dm,batch", [(256, 1), (256, 3), (512, 4), (768, 2), (768, 7), (256, 16), (512, 13)])
def test_few_row_decode_chain_with_folded_x_proj_equals_the_many_row_chain(dm, batch):
    """Up to 16 rows x_proj rides in the in_proj launch (per-tile shares, summed by the step kernel), and at one to four
    rows the projections take the lanes-along-the-row route; an engine of 24 rows runs x_proj as its own launch on the
    matrix cores.  Same weights, same inputs: the rows must agree to 16-bit rounding, step after step, eager and replayed."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=3)
    w = MambaWeights.random_lm(cfg, seed=dm + batch, std=0.05)
    few = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, batch, WeightDtype.BF16)
    many = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, 24, WeightDtype.BF16)
    rng = np.random.default_rng(dm)
    for t in range(24):
        if t == 8:
            few.capture_graph()
        x = rng.standard_normal((24, dm)).astype(np.float32)
        a, b = few.step(x[:batch]), many.step(x)[:batch]
        assert np.isfinite(a).all()
        assert cosine(a, b) >= 0.9995 and scaled_err(a, b) < 3e-2, (t, cosine(a, b), scaled_err(a, b))
    for layer in range(3):
        (ca, sa), (cb, sb) = few.download_state(layer), many.download_state(layer)
        assert cosine(sa, sb[:batch]) >= 0.9995 and cosine(ca, cb[:batch]) >= 0.9995
    few.close(); many.close()


def test_prefill_with_tuned_vendor_gemms_matches_the_default_choice_and_the_cpu_route():
    """set_gemm_tuning: the first prefill of 1024 rows or more times the GEMM library's kernels for each projection
    shape and later prefills run the fastest.  Another kernel sums in another order, so the tuned prefill is held to
    the untuned one by cosine and, like it, to the CPU route; tuned runs repeat bit for bit."""
    cfg = MambaConfig(d_model=256, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.init(cfg, 256, 77)
    P = oracle_params(w, cfg, 256, round_to=orc.BF16)
    B, T = 2, 512
    xs = (np.random.default_rng(5).standard_normal((B, T, 256)) * 0.5).astype(np.float32)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 256, B, WeightDtype.BF16)
    print("case prefill, default vendor kernels", flush=True)
    base = eng.prefill_sequence(xs).copy()
    base_ssm = [eng.download_state(l)[1].copy() for l in range(2)]
    eng.set_gemm_tuning(True)
    runs = []
    for i in range(3):
        print(f"case prefill, tuned vendor kernels, run {i}", flush=True)
        eng.reset()
        runs.append((eng.prefill_sequence(xs).copy(), [eng.download_state(l)[1].copy() for l in range(2)]))
    for last, ssm in runs[1:]:
        assert np.array_equal(last, runs[0][0]) and all(np.array_equal(a, b) for a, b in zip(ssm, runs[0][1]))
    assert cosine(runs[0][0], base) >= 0.9999
    for l in range(2):
        assert cosine(runs[0][1][l], base_ssm[l]) >= 0.9999
    conv, ssm = orc.m1_zero_state(P)
    want = orc.m1_backbone_prefill(P, xs[1], conv, ssm)
    assert cosine(runs[0][0][1], want[-1]) >= 0.999
    eng.close()


def test_generation_times_no_vendor_kernels():
    """With set_gemm_tuning a generation whose prompts have a new length is no slower than a quarter of a first prefill of the same
    rows, which does time the library's kernels, and it has the bits of an engine without tuning, also behind that prefill."""
    import time
    from mamba_rs_amd import SampleParams
    B, T = 64, 24      # 1536 rows: in_proj and out_proj of a prompt's piece go to the library
    cfg = MambaConfig(d_model=768, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.random_lm(cfg, seed=3, std=0.05)
    rng = np.random.default_rng(8)
    embed = rng.standard_normal((500, 768)).astype(np.float32)
    prompts = rng.integers(0, 500, (B, T + 1)).tolist()
    params = [SampleParams(temperature=0.8, top_k=20, max_tokens=2, seed=i) for i in range(B)]
    print("case generation with tuning", flush=True)
    out = []
    for tuned in (False, True):
        eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 768, B, WeightDtype.BF16)
        lm = GpuMambaLM(eng, embed)
        eng.set_gemm_tuning(tuned)
        lm.generate_batch([p[:9] for p in prompts], params)
        t0 = time.perf_counter()
        first = lm.generate_batch(prompts, params)
        new_length = time.perf_counter() - t0
        if tuned:
            x = rng.standard_normal((B, T, 768)).astype(np.float32)
            t0 = time.perf_counter()
            eng.prefill_sequence(x)
            assert new_length < 0.25 * (time.perf_counter() - t0), new_length
        assert lm.generate_batch(prompts, params) == first
        out.append((first, [p for l in range(2) for p in eng.download_state(l)]))
        lm.close()
        eng.close()
    assert out[0][0] == out[1][0] and all(np.array_equal(p, q) for p, q in zip(out[0][1], out[1][1]))


@pytest.mark.parametrize("tuned", [False, True])
def test_decode_above_the_own_chain_limit_runs_the_projections_from_the_transposed_copies(tuned):
    """130 rows at d_model 768: past the own chain's limit, so in_proj and out_proj go to the GEMM library reading the
    transposed weight copies, x_proj and dt_proj reading the originals.  Eager steps, then replays of the captured step;
    with set_gemm_tuning the step that precedes the capture times the library's kernels for the four shapes and the
    graph holds the chosen ones.  First, middle and last row against the CPU route on storage-rounded weights."""
    B = 130
    cfg = MambaConfig(d_model=768, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.random_lm(cfg, seed=B, std=0.05)
    P = oracle_params(w, cfg, 768, round_to=orc.BF16)
    P.input_proj_w[:] = np.eye(768, dtype=np.float32); P.input_proj_b[:] = 0
    rng = np.random.default_rng(B)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, 768, B, WeightDtype.BF16)
    if tuned:
        eng.set_gemm_tuning(True)
    x = rng.standard_normal((5, B, 768)).astype(np.float32)
    rows = (0, B // 2, B - 1)
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(5):
        print(f"case library-chain decode, tuned={tuned}, step {t}", flush=True)
        if t == 2:
            eng.capture_graph()
        got = eng.step(x[t])
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert cosine(got[b], want) >= 0.999, (t, b)
    eng.close()


@pytest.mark.parametrize("shape", [
    # d_model, d_state, d_conv, expand, layers, input_dim, batch
    (128, 16, 4, 2, 3, 128, 1),      # the reference's default configuration
    (128, 16, 4, 2, 2, 128, 128),    # ... at the published batch size
    (64, 8, 2, 2, 2, 24, 5),         # input projection, short window, d_state 8
    (128, 64, 4, 2, 2, 128, 3),      # d_state 64: eight passes of the scan step
    (192, 16, 4, 1, 2, 192, 2),      # dt_rank 12: a second round of dt weights
    (128, 4, 3, 1, 4, 40, 7),        # expand 1, d_state 4 (one pass of 512 rows), dt_rank 8, x_proj row of 16
    (128, 16, 4, 2, 2, 130, 3),      # input row wider than d_model and not a multiple of four floats
    (64, 8, 4, 3, 2, 64, 2),         # expand 3
    (36, 16, 2, 3, 2, 36, 2),        # dt_rank 3: an x_proj row of 35 floats is outside the route, kernel chains on both sides
])
def test_small_f32_models_step_in_one_launch(shape, monkeypatch):
    """Small f32 engines (every product at most three rounds of sixteen weight rows per lane) run a backbone step as one kernel (one workgroup per batch row walks input
    projection, every layer and the final norm).  Held to the CPU route step after step (outputs 1e-4 of their scale, conv window
    and SSM state of every layer at the end), to the kernel chains it replaces (MRS_DECODE_NO_TINY=1 at creation), and
    to itself: graph replays and a second engine give the same bits."""
    dm, ds, dc, ex, L, idim, B = shape
    cfg = MambaConfig(d_model=dm, d_state=ds, d_conv=dc, expand=ex, n_layers=L)
    w = MambaWeights.init(cfg, idim, 7)
    P = oracle_params(w, cfg, idim)
    rng = np.random.default_rng(dm + B)
    steps = 6
    x = rng.standard_normal((steps, B, idim)).astype(np.float32)
    rows = sorted({0, B // 2, B - 1})
    st = {b: orc.m1_zero_state(P) for b in rows}
    print(f"case one-launch step {shape}", flush=True)
    eng = GpuMambaBackbone.new(0, w, cfg, idim, B)
    xd = cfg.dt_rank() + 2 * ds
    assert (eng.decode_route() == 2) == (xd % 4 == 0), (shape, eng.decode_route())   # 2 = the whole step in one launch
    assert eng.temporal_dtype() == WeightDtype.F32
    outs = []
    for t in range(steps):
        if t == 3:
            eng.capture_graph()
        got = eng.step(x[t])
        outs.append(got.copy())
        for b in rows:
            want = orc.m1_backbone_step(P, x[t, b], *st[b])
            assert scaled_err(got[b], want) < 1e-4, (t, b)
    for l in range(L):
        conv, ssm = eng.download_state(l)
        di = cfg.d_inner()
        for b in rows:
            # (the GPU keeps d_conv window slots, the CPU route d_conv - 1)
            assert np.allclose(conv[b][:, 1:], st[b][0][l].reshape(di, dc - 1), atol=1e-5), (l, b)
            assert scaled_err(ssm[b], st[b][1][l].reshape(di, ds)) < 1e-4, (l, b)
    eng.close()
    eng2 = GpuMambaBackbone.new(0, w, cfg, idim, B)
    for t in range(steps):
        assert np.array_equal(eng2.step(x[t]), outs[t]), t
    eng2.close()
    monkeypatch.setenv("MRS_DECODE_NO_TINY", "1")
    print(f"case kernel chains {shape}", flush=True)
    ref = GpuMambaBackbone.new(0, w, cfg, idim, B)
    assert ref.decode_route() != 2
    for t in range(steps):
        assert scaled_err(ref.step(x[t]), outs[t]) < 1e-4, t
    ref.close()


@pytest.mark.parametrize("dm,L,idim,B", [
    (128, 1, 128, 1),      # one layer: nothing is asked for ahead
    (128, 2, 1, 3),        # narrowest input row: slices of its projection without rows
    (128, 3, 512, 2),      # widest input row of the streamed kernel
    (128, 2, 513, 2),      # one more: the other kernel
    (128, 5, 0, 300),      # identity input projection, more rows than compute units
    (64, 1, 64, 1),
    (64, 4, 0, 5),
    (64, 2, 131, 7),       # rows of the projection's last slice missing
])
def test_small_f32_step_with_streamed_weights_follows_the_cpu_route(dm, L, idim, B):
    """Single-launch step of f32 models of the default expand, d_state, d_conv and dt_rank: the weights of a layer are requested during the one
    before.  Outputs and states of every layer against the CPU route over several steps; f32 sums of at most 513 terms in another order,
    1e-4 of the scale as for the other single-launch steps."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=L)
    w = MambaWeights.init(cfg, idim or dm, 5)
    if not idim:
        w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    rng = np.random.default_rng(L + B)
    for lw in w.layers:   # vectors that are constant in a fresh model
        for n in ("norm_weight", "conv1d_bias", "d_param"):
            getattr(lw, n)[:] = 1.0 + 0.2 * rng.standard_normal(getattr(lw, n).shape)
    w.norm_f_weight[:] = 1.0 + 0.2 * rng.standard_normal(dm)
    P = oracle_params(w, cfg, idim or dm)
    if not idim:
        P.input_proj_w[:] = np.eye(dm, dtype=np.float32).reshape(P.input_proj_w.shape); P.input_proj_b[:] = 0
    print(f"case streamed step {dm} {L} {idim} {B}", flush=True)
    eng = GpuMambaBackbone.new(0, w, cfg, idim or dm, B)
    assert eng.decode_route() == 2
    rows = sorted({0, B // 2, B - 1})
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(4):
        x = rng.standard_normal((B, idim or dm)).astype(np.float32)
        if t == 2:
            eng.capture_graph()
        got = eng.step(x)
        for b in rows:
            assert scaled_err(got[b], orc.m1_backbone_step(P, x[b], *st[b])) < 1e-4, (t, b)
    for l in range(L):
        conv, ssm = eng.download_state(l)
        for b in rows:
            assert scaled_err(conv[b][:, 1:], st[b][0][l].reshape(2 * dm, 3)) < 1e-4 and scaled_err(ssm[b], st[b][1][l].reshape(2 * dm, 16)) < 1e-4, (l, b)
    eng.close()


@pytest.mark.parametrize("dm,B,dtype", [(64, 1, WeightDtype.F32), (64, 7, WeightDtype.F32), (64, 8, WeightDtype.F32), (64, 9, WeightDtype.F32), (128, 130, WeightDtype.F32),
                                        (128, 17, WeightDtype.BF16)])
def test_rows_a_step_hands_to_the_host_are_the_rows_it_leaves_on_the_device(dm, B, dtype):
    """The host waits for one flag per row, eight at a time (single-launch steps and the kernel behind the others): every row of every step, bit for bit."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    eng = GpuMambaBackbone.new_with_dtype(0, MambaWeights.init(cfg, dm, 5), cfg, dm, B, dtype)
    rng = np.random.default_rng(B)
    for _ in range(20):
        got = eng.step(rng.standard_normal((B, dm)).astype(np.float32))
        assert np.isfinite(got).all() and np.array_equal(got, eng.download_temporal())
    eng.close()


@pytest.mark.parametrize("family,dm,ds,B", [("m1", 64, 16, 1), ("m1", 128, 16, 128), ("m1", 64, 8, 3), ("m3", 64, 16, 5), ("m3", 128, 16, 48), ("m3", 96, 16, 3), ("m1", 96, 16, 3)])
def test_rows_of_a_step_are_on_the_device_when_it_returns(family, dm, ds, B):
    """step() returns on the rows' flags, before its launch has ended: the final rows behind temporal_ptr(), read by another stream with no wait in between, are those of the host, bit
    for bit (row-streaming and general forms of the single-launch steps, and a step of several launches)."""
    import torch
    from mamba_rs_amd import GpuMamba3Backbone, Mamba3Config, Mamba3Weights
    if family == "m1":
        cfg = MambaConfig(d_model=dm, d_state=ds, d_conv=4, expand=2, n_layers=2)
        eng = GpuMambaBackbone.new(0, MambaWeights.init(cfg, 24, 5), cfg, 24, B)
    else:
        cfg = Mamba3Config(d_model=dm, d_state=ds, expand=2, headdim=16, ngroups=1, n_layers=2, rope_fraction=0.5)
        eng = GpuMamba3Backbone.new(0, Mamba3Weights.init(cfg, 24, 5), cfg, 24, B)

    assert eng.decode_route() == (1 if (family, dm) == ("m1", 96) else 2)

    class Rows:
        __cuda_array_interface__ = {"shape": (B, dm), "typestr": "<f4", "version": 3, "data": (eng.temporal_ptr(), False), "strides": None}
    rows, side = torch.as_tensor(Rows(), device="cuda:0"), torch.cuda.Stream()
    kept = torch.empty_like(rows)
    rng = np.random.default_rng(B)
    with torch.cuda.stream(side):
        for t in range(20):
            got = eng.step(rng.standard_normal((B, 24)).astype(np.float32))
            kept.copy_(rows)
            assert np.isfinite(got).all() and np.array_equal(got, kept.cpu().numpy()), t
    eng.close()


@pytest.mark.parametrize("family,dm,ds,B", [("m1", 64, 16, 1), ("m1", 128, 16, 128), ("m1", 64, 8, 3), ("m3", 64, 16, 5), ("m3", 128, 16, 48), ("m3", 96, 16, 3)])
def test_input_rows_of_a_step_are_on_the_device_when_it_returns(family, dm, ds, B):
    """The same of the input rows behind input_ptr(): another stream reads those of the step that has just returned, and what it puts there is what a step on the device starts from."""
    import torch
    from mamba_rs_amd import GpuMamba3Backbone, Mamba3Config, Mamba3Weights
    if family == "m1":
        cfg = MambaConfig(d_model=dm, d_state=ds, d_conv=4, expand=2, n_layers=2)
        w = MambaWeights.init(cfg, 24, 5)
        make = lambda: GpuMambaBackbone.new(0, w, cfg, 24, B)  # noqa: E731
    else:
        cfg = Mamba3Config(d_model=dm, d_state=ds, expand=2, headdim=16, ngroups=1, n_layers=2, rope_fraction=0.5)
        w = Mamba3Weights.init(cfg, 24, 5)
        make = lambda: GpuMamba3Backbone.new(0, w, cfg, 24, B)  # noqa: E731
    eng, plain = make(), make()
    assert eng.decode_route() == 2

    def view(ptr, width):
        return torch.as_tensor(type("View", (), {"__cuda_array_interface__": {"shape": (B, width), "typestr": "<f4", "version": 3, "data": (ptr, False), "strides": None}})(), device="cuda:0")
    rows, final, side = view(eng.input_ptr(), 24), view(eng.temporal_ptr(), dm), torch.cuda.Stream()
    kept = torch.empty_like(rows)
    rng = np.random.default_rng(B)
    with torch.cuda.stream(side):
        for t in range(20):
            x, follow = (rng.standard_normal((B, 24)).astype(np.float32) for _ in range(2))
            put = torch.from_numpy(follow).cuda()
            side.synchronize()
            eng.step(x)
            kept.copy_(rows)
            rows.copy_(put)
            side.synchronize()
            assert np.array_equal(kept.cpu().numpy(), x), t
            eng.step_gpu_only()
            eng.sync()
            plain.step(x)
            assert np.array_equal(final.cpu().numpy(), plain.step(follow)), t
    eng.close()
    plain.close()


@pytest.mark.parametrize("dm,dc,ds,B", [(64, 4, 16, 1), (128, 4, 16, 64), (96, 3, 16, 3), (64, 3, 8, 3), (128, 2, 16, 5)])
def test_states_of_a_step_are_on_the_device_when_it_returns(dm, dc, ds, B):
    """The same of the states behind state_ptrs(): another stream reads those that a later download gives, and a step goes on from what another stream put there."""
    import ctypes
    import torch
    from mamba_rs_amd import backbone
    cfg = MambaConfig(d_model=dm, d_state=ds, d_conv=dc, expand=2, n_layers=2)
    eng = GpuMambaBackbone.new(0, MambaWeights.init(cfg, 24, 5), cfg, 24, B)
    assert eng.decode_route() == (1 if dm == 96 else 2)
    bind, di, last = backbone._bind(), 2 * dm, cfg.n_layers - 1
    conv, ssm = ctypes.c_void_p(), ctypes.c_void_p()
    assert bind.mrs_backbone_state_ptrs(eng._h, last, ctypes.byref(conv), ctypes.byref(ssm)) == 0

    def view(ptr, *shape):
        return torch.as_tensor(type("View", (), {"__cuda_array_interface__": {"shape": shape, "typestr": "<f4", "version": 3, "data": (ptr.value, False), "strides": None}})(), device="cuda:0")
    views, side = [view(conv, B, di, dc), view(ssm, B, di, ds)], torch.cuda.Stream()
    kept = [torch.empty_like(v) for v in views]
    rng = np.random.default_rng(B)
    with torch.cuda.stream(side):
        for t in range(20):
            eng.step(rng.standard_normal((B, 24)).astype(np.float32))
            for k, v in zip(kept, views):
                k.copy_(v)
            side.synchronize()
            for k, d in zip(kept, eng.download_state(last)):
                assert np.array_equal(k.cpu().numpy().ravel(), np.asarray(d).ravel()), t
            if t == 10:   # both states back to nothing, behind the step that has just returned
                eng.step(rng.standard_normal((B, 24)).astype(np.float32))
                for v in views:
                    v.zero_()
                side.synchronize()
                assert not any(np.asarray(d).any() for d in eng.download_state(last))
    eng.close()


@pytest.mark.parametrize("dm,L,B", [(96, 2, 1), (160, 2, 17), (192, 2, 4), (192, 1, 128), (256, 2, 5), (256, 2, 16), (768, 1, 33), (1088, 1, 7), (800, 1, 64), (192, 1, 129)])
def test_f32_rows_on_the_own_chain_follow_the_cpu_route(dm, L, B):
    """f32 models past the single-launch step: the own chain with its products on the matrix cores' f32 instructions (k-steps fewer than the waves, row tiles partly filled, more rows
    than x_proj rides in in_proj for), and the library's past 128 rows.  f32 sums of at most 2176 terms in another order, 1e-4 of the scale as for the other f32 steps."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=L)
    w = MambaWeights.init(cfg, 40, 5)
    P = oracle_params(w, cfg, 40)
    rng = np.random.default_rng(dm + B)
    print(f"case f32 rows {dm} {L} {B}", flush=True)
    eng = GpuMambaBackbone.new(0, w, cfg, 40, B)
    assert eng.decode_route() == (1 if B <= 128 else 0)
    rows = sorted({0, B // 2, B - 1})
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(4):
        x = rng.standard_normal((B, 40)).astype(np.float32)
        if t == 2:
            eng.capture_graph()
        got = eng.step(x)
        for b in rows:
            assert scaled_err(got[b], orc.m1_backbone_step(P, x[b], *st[b])) < 1e-4, (t, b)
    for l in range(L):
        conv, ssm = eng.download_state(l)
        for b in rows:
            assert scaled_err(conv[b][:, 1:], st[b][0][l].reshape(2 * dm, 3)) < 1e-4 and scaled_err(ssm[b], st[b][1][l].reshape(2 * dm, 16)) < 1e-4, (l, b)
    eng.close()


@pytest.mark.parametrize("dm,idim,B", [(192, 1, 1), (192, 9, 3), (160, 513, 2), (320, 88, 128), (320, 88, 129), (36, 4096, 2), (36, 4097, 2)])
def test_input_rows_through_the_projection_kernel(dm, idim, B):
    """One row's product per workgroup, from host memory (step) and from the device (step_gpu_only), eager and in front of a recorded step; past 128 rows or 4096 inputs the library's.
    f32: sums of at most 4097 terms in another order, 1e-4 of the scale as above."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, idim, 5)
    rng = np.random.default_rng(idim)
    w.input_proj_b[:] = rng.standard_normal(dm)
    P = oracle_params(w, cfg, idim)
    print(f"case projected rows {dm} {idim} {B}", flush=True)
    eng = GpuMambaBackbone.new(0, w, cfg, idim, B)
    rows = sorted({0, B // 2, B - 1})
    st = {b: orc.m1_zero_state(P) for b in rows}
    for t in range(6):
        x = rng.standard_normal((B, idim)).astype(np.float32)
        if t == 2:
            eng.capture_graph()
        got = eng.step(x)
        for b in rows:
            assert scaled_err(got[b], orc.m1_backbone_step(P, x[b], *st[b])) < 1e-4, (t, b)
        if t % 2:   # the same rows once more: they are on the device
            eng.step_gpu_only()
            got = eng.download_temporal()
            for b in rows:
                assert scaled_err(got[b], orc.m1_backbone_step(P, x[b], *st[b])) < 1e-4, (t, b)
    eng.close()


@pytest.mark.parametrize("family,dm,idim,B,in_front", [("m1", 320, 88, 128, True), ("m1", 320, 88, 129, False), ("m3", 192, 40, 129, False), ("m1", 36, 4097, 2, False), ("m3", 192, 40, 3, True)])
def test_what_stands_in_front_of_a_recorded_step(family, dm, idim, B, in_front):
    """The library's products of a projection are part of the recorded step (more than 128 rows, more than 4096 inputs), the projection's kernel stands in front of it, as step() has it take
    the rows from host memory: the calls of a step on the device, and the rows of steps with the host, bit for bit those of an engine that replays nothing."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    from mamba_rs_amd import GpuMamba3Backbone, Mamba3Config, Mamba3Weights
    if family == "m1":
        cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=2)
        w = MambaWeights.init(cfg, idim, 5)
        make = lambda: GpuMambaBackbone.new(0, w, cfg, idim, B)  # noqa: E731
    else:
        cfg = Mamba3Config(d_model=dm, d_state=16, expand=2, headdim=16, ngroups=1, n_layers=2, rope_fraction=0.5)
        w = Mamba3Weights.init(cfg, idim, 5)
        make = lambda: GpuMamba3Backbone.new_with_dtype(0, w, cfg, idim, B, WeightDtype.F32)  # noqa: E731
    eager, recorded = make(), make()
    rng = np.random.default_rng(B)
    recorded.capture_graph()
    for _ in range(3):
        x = rng.standard_normal((B, idim)).astype(np.float32)
        assert np.array_equal(eager.step(x), recorded.step(x))
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        recorded.step_gpu_only()
        recorded.sync()
    calls = [e.name for e in prof.events() if "Launch" in e.name]
    assert calls == ["hipLaunchKernel"] * in_front + ["hipGraphLaunch"]
    eager.close()
    recorded.close()


@pytest.mark.parametrize("dm,lens,dtype", [
    (128, (9, 5), WeightDtype.F16),              # four tokens; dt_rank 8: a quarter of a k-step of dt_proj
    (256, (6, 40, 18), WeightDtype.BF16),        # five
    (256, (70, 33, 81), WeightDtype.BF16),       # 32: one whole piece
    (768, (34, 36), WeightDtype.F16),            # 33: two pieces of 16 and 17, a last tile of one step; dt_rank 48
    (1024, (100,), WeightDtype.BF16),            # 99: four pieces
    (2560, (9, 40), WeightDtype.BF16),           # dt_rank 160: five k-steps of dt_proj, rows of x_proj 192 apart
])
def test_prompts_of_a_generation_in_pieces(dm, lens, dtype):
    """What all prompts have in front of their last token goes through the prefill's kernels, up to 32 steps at a time, with dt_proj inside
    the scan: tokens are those of an engine that takes every token as a step (scan_mode SEQUENTIAL keeps the prompt out of the
    prefill kernels), all states and the last rows within the tolerance between two routes that round at the same 16-bit points
    (1 % in norm: three layers, each rounding its projections, u and y once), and not the same bits: two routes there were."""
    from mamba_rs_amd import SampleParams
    rng = np.random.default_rng(sum(lens))
    embed = rng.standard_normal((500, dm)).astype(np.float32)
    prompts = [rng.integers(0, 500, n).tolist() for n in lens]
    params = [SampleParams(temperature=0.8, top_k=20, max_tokens=4, seed=i) for i in range(len(lens))]
    out = []
    print(f"case prompts in pieces {dm} {lens} {dtype.name}", flush=True)
    for mode in (ScanMode.AUTO, ScanMode.SEQUENTIAL):
        cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=3, scan_mode=mode)
        w = MambaWeights.init(cfg, dm, 9)
        w.input_proj_w = np.zeros((0, dm), np.float32)
        e = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, len(lens), dtype)
        lm = GpuMambaLM(e, embed)
        first = lm.generate_batch(prompts, params)
        lm.generate_batch([p[:3] for p in prompts], params)     # too short for it
        assert lm.generate_batch(prompts, params) == first      # again, on what the others left behind
        out.append((first, [e.download_temporal()] + [p for l in range(3) for p in e.download_state(l)]))
        lm.close()
        e.close()
    assert out[0][0] == out[1][0]
    assert not all(np.array_equal(p, q) for p, q in zip(out[0][1], out[1][1]))
    for p, q in zip(out[0][1], out[1][1]):
        assert np.linalg.norm(p - q) <= 1e-2 * np.linalg.norm(q), np.linalg.norm(p - q) / np.linalg.norm(q)


@pytest.mark.parametrize("dm,B,T,dtype", [
    (128, 1, 16, WeightDtype.BF16),     # the shortest prompt; one row, lanes along the weight row
    (256, 4, 33, WeightDtype.F16),      # the most rows of that route
    (128, 5, 17, WeightDtype.BF16),     # matrix cores, part of a row tile
    (64, 3, 16, WeightDtype.F16),       # matrix cores at few rows: a weight row of no whole 32 lanes
    (64, 17, 40, WeightDtype.F16),      # a second row tile, of one row
    (128, 128, 16, WeightDtype.BF16),   # the most rows
])
def test_prefill_projects_the_last_steps_alone_in_its_last_layer(dm, B, T, dtype):
    """Behind the last layer's scan only the last step of each sequence goes on.  Against the same prompt in two calls, the second of eight
    steps, whose out_proj runs over all rows: states as two calls leave them, last rows within the tolerance between two routes that
    round at the same 16-bit points (1 % in norm: three layers, each rounding its projections, u and y once)."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=3)
    w = MambaWeights.init(cfg, dm, 5)
    w.input_proj_w = np.zeros((0, dm), np.float32)
    x = np.random.default_rng(B + T).standard_normal((B, T, dm)).astype(np.float32)
    print(f"case last steps {dm} {B}x{T} {dtype.name}", flush=True)
    e = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    got = [e.prefill_sequence(x).copy()] + [p for l in range(3) for p in e.download_state(l)]
    e.reset()
    e.prefill_sequence(x[:, :T - 8].copy())
    want = [e.prefill_sequence(x[:, T - 8:].copy()).copy()] + [p for l in range(3) for p in e.download_state(l)]
    e.close()
    for p, q in zip(got, want):
        assert np.linalg.norm(p - q) <= 1e-2 * np.linalg.norm(q), np.linalg.norm(p - q) / np.linalg.norm(q)


@pytest.mark.parametrize("dm,B,T,trained,dtype", [
    (256, 1, 72, False, WeightDtype.BF16),     # a first call of 64 steps: the longest single pass
    (512, 1, 105, True, WeightDtype.F16),      # two chunks and more, four lanes per channel; a last chunk of one step
    (1024, 1, 777, True, WeightDtype.BF16),
    (768, 2, 1033, False, WeightDtype.BF16),   # one lane per channel, one launch where all outputs are wanted
    (768, 8, 1040, True, WeightDtype.F16),     # general A, two launches
    (768, 4, 2056, False, WeightDtype.BF16),   # in_proj on the large tiles
])
def test_prefill_forms_gate_and_outputs_of_the_last_steps_alone_in_its_last_layer(dm, B, T, trained, dtype):
    """The same over the routes of the scan and of in_proj, where the last layer has half an in_proj and outputs of its last chunk: against two calls, the second of
    eight steps, which form everything.  Tolerance as above."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.init(cfg, dm, 5)
    w.input_proj_w = np.zeros((0, dm), np.float32)
    rng = np.random.default_rng(B + T)
    if trained:
        for lw in w.layers:
            lw.a_log = lw.a_log + 0.15 * rng.standard_normal(lw.a_log.shape).astype(np.float32)
    x = rng.standard_normal((B, T, dm)).astype(np.float32)
    print(f"case last layer {dm} {B}x{T} {trained} {dtype.name}", flush=True)
    e = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    got = [e.prefill_sequence(x).copy()] + [p for l in range(2) for p in e.download_state(l)]
    e.reset()
    e.prefill_sequence(x[:, :T - 8].copy())
    want = [e.prefill_sequence(x[:, T - 8:].copy()).copy()] + [p for l in range(2) for p in e.download_state(l)]
    e.close()
    for p, q in zip(got, want):
        assert np.linalg.norm(p - q) <= 1e-2 * np.linalg.norm(q), np.linalg.norm(p - q) / np.linalg.norm(q)
