"""GPU: the prefill projections of few rows (the 64 x 64-tile kernel, and x_proj on the decode chain's 16 x 16 tiles) through one
layer of the engine, against the CPU route on storage-rounded weights."""
import numpy as np
import pytest

import orc
from util import cosine, scaled_err
from test_engine_gpu import oracle_params

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMambaBackbone, MambaConfig, MambaWeights, WeightDtype  # noqa: E402


@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
@pytest.mark.parametrize("dm,B,T", [
    (64, 1, 2),      # one k-step of in_proj, two of out_proj: fewer than the buffers; two rows of a tile
    (64, 1, 63),     # a row tile short of its last row
    (64, 2, 32),     # a whole row tile
    (128, 1, 65),    # one row past it
    (192, 3, 43),    # three, then six k-steps; 129 rows: the third row tile holds one
    (320, 1, 200),   # five k-steps and ten: one more than the buffers; workgroups not a multiple of eight
    (96, 1, 70),     # K not a multiple of the k-step: in_proj (96) stays with the library, out_proj (192) does not
])
def test_prefill_of_few_rows_follows_the_cpu_route(dm, B, T, dtype):
    """Every sequence's last row and the states behind it.  16-bit storage: cosine >= 0.999 per row as for the decode chains, and 5e-2 of
    the largest element -- a tile row or column gone wrong shows in the states, which hold every channel's history."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 5)
    P = oracle_params(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    x = (np.random.default_rng(dm + T).standard_normal((B, T, dm)) * 0.5).astype(np.float32)
    print(f"case prefill projections d_model={dm} rows={B * T} {dtype.name}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    last = eng.prefill_sequence(x)
    conv, ssm = eng.download_state(0)
    eng.close()
    di = cfg.d_inner()
    for b in range(B):
        c, s = orc.m1_zero_state(P)
        want = orc.m1_backbone_prefill(P, x[b], c, s)[-1]
        assert cosine(last[b], want) >= 0.999 and scaled_err(last[b], want) < 5e-2, (b, cosine(last[b], want), scaled_err(last[b], want))
        hs, cs = s[0].reshape(di, 16), c[0].reshape(di, 3)
        assert cosine(ssm[b], hs) >= 0.999 and scaled_err(ssm[b], hs) < 5e-2, (b, cosine(ssm[b], hs), scaled_err(ssm[b], hs))
        assert cosine(conv[b][:, 1:], cs) >= 0.999 and scaled_err(conv[b][:, 1:], cs) < 5e-2, (b, cosine(conv[b][:, 1:], cs))


@pytest.mark.parametrize("dm,B,T,dtype", [
    (192, 3, 43, WeightDtype.BF16),     # six k-steps in two slices; 129 rows
    (320, 1, 63, WeightDtype.F16),      # ten in three, the last of two; a row tile short of its last row
    (448, 1, 130, WeightDtype.BF16),    # fourteen in four, the last of two
    (384, 2, 8, WeightDtype.F16),       # sixteen rows, four slices of three
    (1088, 1, 40, WeightDtype.BF16),    # rows of more than one piece a lane
    (768, 1, 700, WeightDtype.BF16),    # one slice: tiles for half of the units
])
def test_out_proj_in_slices_of_k(dm, B, T, dtype):
    """Two layers: the first one's out_proj leaves products over slices of K, which the second one's norm sums.  Bounds as above."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=2)
    w = MambaWeights.init(cfg, dm, 7)
    P = oracle_params(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    x = (np.random.default_rng(dm + T).standard_normal((B, T, dm)) * 0.5).astype(np.float32)
    print(f"case out_proj in slices d_model={dm} rows={B * T} {dtype.name}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    last = eng.prefill_sequence(x)
    state = [eng.download_state(l) for l in range(2)]
    eng.close()
    for b in range(B):
        c, s = orc.m1_zero_state(P)
        want = orc.m1_backbone_prefill(P, x[b], c, s)[-1]
        assert cosine(last[b], want) >= 0.999 and scaled_err(last[b], want) < 5e-2, (b, cosine(last[b], want), scaled_err(last[b], want))
        for l in range(2):
            hs = s[l].reshape(2 * dm, 16)
            assert cosine(state[l][1][b], hs) >= 0.999 and scaled_err(state[l][1][b], hs) < 5e-2, (b, l, cosine(state[l][1][b], hs), scaled_err(state[l][1][b], hs))


@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
@pytest.mark.parametrize("dm,B,T", [
    (128, 33, 1000),   # tiles of 192 columns, the last a third empty; two k-steps, one pair of buffers
    (320, 11, 1187),   # tiles of 320 columns; five k-steps; the last row tile holds one row
    (320, 13, 1024),   # whole tiles both ways
    (448, 10, 946),    # the last column tile holds 192 of its 320; seven k-steps; workgroups not a multiple of eight
])
def test_long_prefill_on_the_large_tiles_follows_the_cpu_route(dm, B, T, dtype):
    """in_proj on the 256-row tiles (row counts at which the library's would leave a round partly empty): sequences from both ends and
    the middle of the rows, bounds as above."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 6)
    P = oracle_params(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    x = (np.random.default_rng(dm + T).standard_normal((B, T, dm)) * 0.5).astype(np.float32)
    print(f"case large prefill projections d_model={dm} rows={B * T} {dtype.name}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    last = eng.prefill_sequence(x)
    conv, ssm = eng.download_state(0)
    eng.close()
    di = cfg.d_inner()
    for b in (0, 1, B // 2, B - 2, B - 1):
        c, s = orc.m1_zero_state(P)
        want = orc.m1_backbone_prefill(P, x[b], c, s)[-1]
        assert cosine(last[b], want) >= 0.999 and scaled_err(last[b], want) < 5e-2, (b, cosine(last[b], want), scaled_err(last[b], want))
        hs, cs = s[0].reshape(di, 16), c[0].reshape(di, 3)
        assert cosine(ssm[b], hs) >= 0.999 and scaled_err(ssm[b], hs) < 5e-2, (b, cosine(ssm[b], hs), scaled_err(ssm[b], hs))
        assert cosine(conv[b][:, 1:], cs) >= 0.999 and scaled_err(conv[b][:, 1:], cs) < 5e-2, (b, cosine(conv[b][:, 1:], cs))


@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
@pytest.mark.parametrize("dm,B,T", [
    (128, 3, 867),    # 512 + 156 columns in three column tiles, the line between storage type and f32 inside the second; two k-steps; 41 rows in the last row tile
    (256, 2, 1409),   # 1024 + 168, the line inside the fourth; the last row tile holds two rows
])
def test_long_mamba3_prefill_with_all_columns_of_in_proj_at_once_follows_the_cpu_route(dm, B, T, dtype):
    """z and x in the storage type and the shared columns in f32 out of one launch; bounds as above."""
    from mamba_rs_amd import GpuMamba3Backbone, Mamba3Config
    from test_m3_engine_gpu import oracle_params as oracle_params3, perturbed
    cfg = Mamba3Config(d_model=dm, d_state=64, expand=2, headdim=64, ngroups=1, n_layers=1, rope_fraction=0.5)
    w = perturbed(cfg, dm, 3)
    P = oracle_params3(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    x = (np.random.default_rng(T).standard_normal((B, T, dm)) * 0.5).astype(np.float32)
    print(f"case m3 in_proj at once d_model={dm} rows={B * T} {dtype.name}", flush=True)
    eng = GpuMamba3Backbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    last = eng.prefill_sequence(x)
    ssm = eng.download_state(0)[0]
    eng.close()
    for b in (0, B - 1):
        st = P.zero_state()
        for t in range(T):
            want = orc.m3_backbone_step(P, x[b, t], st)
        assert cosine(last[b], want) >= 0.999 and scaled_err(last[b], want) < 5e-2, (b, cosine(last[b], want), scaled_err(last[b], want))
        assert cosine(ssm[b], st[0][0].reshape(ssm[b].shape)) >= 0.999, (b, cosine(ssm[b], st[0][0].reshape(ssm[b].shape)))
