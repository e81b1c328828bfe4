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
    (768, 3, 600, WeightDtype.BF16),     # five column tiles; 57 tiles of 32 steps, in slices of the channels; the last has 24 steps
    (768, 3, 609, WeightDtype.F16),      # ... one step
    (768, 6, 1801, WeightDtype.BF16),    # 64 steps a workgroup, the last has nine
    (1024, 4, 421, WeightDtype.F16),     # six column tiles; slices
    (1024, 11, 961, WeightDtype.BF16),   # ... of 64 steps, the last one step
    (2560, 32, 112, WeightDtype.BF16),   # twelve column tiles, four pieces in LDS; two slices
    (2560, 84, 100, WeightDtype.F16),    # ... of 64 steps, the second workgroup of a sequence half full
])
def test_long_prefill_behind_a_short_one_follows_the_cpu_route(dm, B, T, dtype):
    """Five steps first, whose window the long prompt starts from; then the last rows and the states.  What the first rows of a sequence and of a tile see is looked
    at by the tests of short prompts below: these steps lie too far back here.  16-bit storage: cosine >= 0.999 per row and 5e-2 of the largest element, as for the other prefills."""
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


# d_model by columns of x_proj: 48 .. 192 in tiles of 16, three to twelve of them, the last one full but for 68, 84, 100, 132 and 184
WIDTHS = [256, 512, 576, 768, 832, 1024, 1088, 1280, 1536, 1600, 1792, 2048, 2304, 2432, 2560]


def _prompts(width_index):
    """Prompts that end right behind a window and a tile boundary, many sequences of them, in every form that the width takes: (batch, steps)."""
    i = width_index % 3
    forms = [(330, 4 + i), (110, 65 + i), (70, 33 + i)]   # 64 steps a workgroup: the first of a sequence, the first of the second; 32 steps
    return forms + ([(25, 33 + i), (40, 5)] if WIDTHS[width_index] >= 512 else [(40, 34)])   # in slices of the channels; narrow models have none


@pytest.mark.parametrize("width", range(len(WIDTHS)), ids=[str(dm) for dm in WIDTHS])
def test_u_is_the_conv_kernels(width):
    """A layer that hands u through: in_proj and out_proj pick single features, x_proj is zero (so B, C and the state are), and silu of the gate is the gate.  Inputs
    are small integers, whose squares any kernel sums exactly.  A few sequences alone take the conv kernel; the same sequences among many, at both ends of the
    batch, have the same window and the same u: a last place of it is 2^-11 of an output at least, the final norm's f32 sum in another order 1e-6.  In f16 the
    compiler rounds silu's last product to f16 at once in one kernel and by way of f32 in the other, which differ where the product lies within 2^-13 of a last
    place of the middle between two values, 2^-12 of all: eight times that many are let through, by a last place."""
    dm = WIDTHS[width]
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    di, dtype = 2 * dm, (WeightDtype.BF16, WeightDtype.F16)[width % 2]
    rng = np.random.default_rng(dm)
    w = MambaWeights.zeros(cfg, 0)
    w.input_proj_w = np.zeros((0, dm), np.float32)
    lw = w.layers[0]
    lw.in_proj_w[1 + np.arange(di) % (dm - 1), np.arange(di)] = 1
    lw.in_proj_w[0, di:] = 32
    lw.conv1d_weight = rng.uniform(-0.87, 0.87, (di, 4)).astype(np.float32)
    lw.conv1d_bias = (0.1 * rng.standard_normal(di)).astype(np.float32)
    lw.out_proj_w[rng.permutation(di)[:dm], np.arange(dm)] = 1
    few = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, 5, dtype)
    for B, T in _prompts(width):
        x = rng.integers(-4, 5, (B, 5 + T, dm)).astype(np.float32)
        x[:, :, 0] = 4   # (the gate's feature: 32 times its normed value is above 32, and 1 + exp(-32) is 1)
        print(f"case conv + x_proj, u d_model={dm} {B} x {T} {dtype.name}", flush=True)
        eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
        eng.prefill_sequence(x[:, :5])
        got = eng.prefill_sequence(x[:, 5:])
        conv = eng.download_state(0)[0]
        eng.close()
        for part in (slice(0, 5), slice(B - 5, B)):
            few.reset()
            few.prefill_sequence(x[part, :5])
            want = few.prefill_sequence(x[part, 5:])
            assert np.isfinite(want).all() and len(np.unique(want)) > dm // 2
            off = np.abs(got[part] - want)
            other = (off > 1e-5 * np.abs(want) + 2e-6).sum()
            assert other <= (want.size / 512 + 1 if dtype == WeightDtype.F16 else 0) and off.max() <= 2.0 ** -10 * np.abs(want).max(), (other, off.max())
            assert (conv[part] == few.download_state(0)[0]).all()
    few.close()


@pytest.mark.parametrize("width", range(len(WIDTHS)), ids=[str(dm) for dm in WIDTHS])
def test_every_row_of_a_short_prompt_counts(width):
    """States that forget nothing (A near zero), so that every x_proj row of the prompt, its first three and those behind a tile boundary among them, has its share
    in them.  An oracle without the carried window, and one without the rows in front of the last tile, are further off than the bound: by three times at least.
    The bound on the 2-norm: a term of the state is a product of three rounded factors (delta, u, B), u and B of values rounded twice in front, in all about
    seven independent roundings of at most half a unit in the last place, 2^-9 (bf16) or 2^-12 (f16) of the value: sqrt(7) of them; twice that."""
    dm = WIDTHS[width]
    dtype = (WeightDtype.F16, WeightDtype.BF16)[width % 2]
    bound = 2 * 7 ** 0.5 * (2.0 ** -9 if dtype == WeightDtype.BF16 else 2.0 ** -12)
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.random_lm(cfg, seed=dm, std=dm ** -0.5)
    w.layers[0].a_log[:] = -7
    P = oracle_params(w, cfg, dm, round_to=orc.BF16 if dtype == WeightDtype.BF16 else orc.F16)
    rng = np.random.default_rng(dm + 1)
    di = cfg.d_inner()

    def states(x, cuts):
        """The CPU route's state behind x, its window cleared in front of the steps `cuts`; and the last row."""
        c, s = orc.m1_zero_state(P)
        for a, b, clear in zip((0, *cuts), (*cuts, len(x)), (False, *[True] * len(cuts))):
            if clear:
                c[:] = 0
            last = orc.m1_backbone_prefill(P, x[a:b], c, s, identity_proj=True)[-1]
        return s[0].reshape(di, 16).copy(), last
    far = lambda a, b: float(np.linalg.norm(np.float64(a) - b) / np.linalg.norm(np.float64(b)))  # noqa: E731
    for B, T in _prompts(width):
        x = rng.standard_normal((B, 5 + T, dm)).astype(np.float32)
        print(f"case conv + x_proj, rows d_model={dm} {B} x {T} {dtype.name}", flush=True)
        eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype)
        eng.prefill_sequence(x[:, :5])
        got = eng.prefill_sequence(x[:, 5:])
        ssm = eng.download_state(0)[1]
        eng.close()
        for b in (0, B // 2, B - 1):
            want, last = states(x[b], ())
            print(f"  row {b}: state {far(ssm[b], want):.2e}, output {far(got[b], last):.2e} of {bound:.2e}", flush=True)
            assert far(ssm[b], want) < bound and far(got[b], last) < bound
        assert far(states(x[b], (5,))[0], want) > 3 * bound
        edge = 64 if T > 64 else 32
        if T > edge:
            assert far(states(x[b], (5 + edge,))[1], last) > 3 * bound
