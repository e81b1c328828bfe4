"""GPU: the resident decode step (a whole 16-bit Mamba-1 step in one launch whose workgroups exchange through memory) against
the CPU route, and against itself: eager and replayed, alone and taking turns with a second engine."""
import numpy as np
import pytest

import orc
from util import cosine, scaled_err
from test_engine_gpu import oracle_params

pytestmark = pytest.mark.gpu

from mamba_rs_amd import GpuMambaBackbone, MambaConfig, MambaWeights, WeightDtype  # noqa: E402


@pytest.mark.parametrize("shape", [
    (32, 2, 32, 1),       # one k-step, four workgroups; an x_proj row of 34: a last tile of two entries
    (64, 3, 20, 16),      # input projection; dt_rank 4; a group of workgroups per row, sixteen of them
    (192, 2, 192, 5),     # 24 channels per workgroup, dt_rank 12
    (256, 2, 256, 8),     # eight rows of 32 workgroups: every compute unit
    (768, 2, 768, 1),     # 24 channels and 12 out_proj columns per workgroup
    (768, 2, 768, 4),
    (1024, 2, 1024, 2),   # the widest: 128 workgroups per row, four and eight k-steps per wave
])
@pytest.mark.parametrize("dtype", [WeightDtype.BF16, WeightDtype.F16])
def test_resident_step_follows_the_cpu_route(shape, dtype):
    """Six steps (three eager, three replayed): every row within the 16-bit engines' tolerance of the CPU route on
    storage-rounded weights (cosine >= 0.999 as for the kernel chains: the same rounding points, sums in another order), states
    as well.  A second engine steps in turns with the first -- together they have more workgroups than the chip has places
    from 129 up -- and ends on the same bits: all sums are in a fixed order."""
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
    rows = sorted({0, B // 2, B - 1})
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
