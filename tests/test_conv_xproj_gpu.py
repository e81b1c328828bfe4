"""GPU: conv1d + SiLU and x_proj as one launch (long prefills), through one layer of the engine with a carried window, against the CPU route
on storage-rounded weights."""
import numpy as np
import pytest

import orc
from util import cosine, scaled_err
from test_engine_gpu import oracle_params

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMambaBackbone, MambaConfig, MambaWeights, WeightDtype  # noqa: E402


@pytest.mark.parametrize("dm,B,T,dtype", [
    (768, 3, 600, WeightDtype.BF16),     # 32 steps a workgroup, five column tiles; the last workgroup of a sequence has 24
    (768, 3, 609, WeightDtype.F16),      # ... one step
    (768, 6, 1801, WeightDtype.BF16),    # 64 steps a workgroup, the last has nine
    (1024, 4, 421, WeightDtype.F16),     # six column tiles
    (1024, 11, 961, WeightDtype.BF16),   # ... of 64 steps, the last one step
    (2560, 32, 112, WeightDtype.BF16),   # twelve column tiles, four pieces in LDS
    (2560, 84, 100, WeightDtype.F16),    # ... of 64 steps, the second workgroup of a sequence half full
])
def test_long_prefill_behind_a_short_one_follows_the_cpu_route(dm, B, T, dtype):
    """Five steps first, whose window the long prompt starts from, so that a workgroup's first rows see it; then every last row and the states, which hold
    every channel's history.  16-bit storage: cosine >= 0.999 per row and 5e-2 of the largest element, as for the other prefills."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.random_lm(cfg, seed=dm, std=0.05)
    P = oracle_params(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    x = np.random.default_rng(dm + T).standard_normal((B, 5 + T, dm)).astype(np.float32)
    print(f"case conv + x_proj d_model={dm} {B} x {T} {dtype.name}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    eng.prefill_sequence(x[:, :5])
    last = eng.prefill_sequence(x[:, 5:])
    conv, ssm = eng.download_state(0)
    eng.close()
    di = cfg.d_inner()
    for b in (0, B - 1):
        c, s = orc.m1_zero_state(P)
        orc.m1_backbone_prefill(P, x[b, :5], c, s, identity_proj=True)
        want = orc.m1_backbone_prefill(P, x[b, 5:], c, s, identity_proj=True)[-1]
        assert cosine(last[b], want) >= 0.999 and scaled_err(last[b], want) < 5e-2, (b, cosine(last[b], want), scaled_err(last[b], want))
        hs, cs = s[0].reshape(di, 16), c[0].reshape(di, 3)
        assert cosine(ssm[b], hs) >= 0.999 and scaled_err(ssm[b], hs) < 5e-2, (b, cosine(ssm[b], hs), scaled_err(ssm[b], hs))
        assert cosine(conv[b][:, 1:], cs) >= 0.999 and scaled_err(conv[b][:, 1:], cs) < 5e-2, (b, cosine(conv[b][:, 1:], cs))


@pytest.mark.parametrize("dm,B,T,dtype", [
    (768, 1, 737, WeightDtype.BF16),     # the fewest rows: eight slices of three pieces; the last tile has one step
    (768, 12, 61, WeightDtype.F16),      # two tiles a sequence
    (768, 25, 4, WeightDtype.BF16),      # sequences of a window's length
    (1024, 1, 777, WeightDtype.BF16),    # eight slices of four pieces
    (1024, 3, 530, WeightDtype.F16),     # five of seven pieces, the last of four
    (2560, 1, 768, WeightDtype.BF16),    # twelve column tiles, ten slices of eight
    (2560, 3, 1130, WeightDtype.F16),    # two of 40
])
def test_prefill_in_slices_of_the_channels_follows_the_cpu_route(dm, B, T, dtype):
    """Fewer rows: the workgroups share out the channels too.  As above."""
    test_long_prefill_behind_a_short_one_follows_the_cpu_route(dm, B, T, dtype)


@pytest.mark.parametrize("dm,B,T", [(768, 3, 600), (768, 6, 1801), (1024, 4, 421), (2560, 32, 112), (768, 25, 4), (1024, 3, 530)])
def test_rows_do_not_depend_on_the_sequences_beside_them(dm, B, T):
    """The same sequence in every place of the batch, in front of it a window of its own: all of them end with the same bits."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.random_lm(cfg, seed=1, std=0.05)
    x = np.repeat(np.random.default_rng(T).standard_normal((1, 5 + T, dm)).astype(np.float32), B, 0)
    print(f"case conv + x_proj, equal sequences d_model={dm} {B} x {T}", flush=True)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.BF16)
    for _ in range(3):
        eng.reset()
        eng.prefill_sequence(x[:, :5])
        last = eng.prefill_sequence(x[:, 5:])
        conv, ssm = eng.download_state(0)
        assert (last == last[:1]).all() and (conv == conv[:1]).all() and (ssm == ssm[:1]).all()
    eng.close()
