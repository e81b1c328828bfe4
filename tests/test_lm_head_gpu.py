"""The language model head (csrc/lm_head.hip): logits of every row against the product in 64 bits, and the greedy pick against numpy."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mamba_rs_amd import backbone, GpuMambaBackbone, GpuMambaLM, MambaConfig, MambaWeights, WeightDtype  # noqa: E402


@pytest.mark.parametrize("dm,B,vocab,dtype,untied", [
    (64, 1, 5, WeightDtype.BF16, False),         # fewer columns than one workgroup, fewer k-steps than are asked for ahead
    (64, 16, 64, WeightDtype.F16, False),
    (64, 17, 1090, WeightDtype.BF16, True),      # one row more than a row tile; a last workgroup with one tile; a head of its own
    (288, 33, 2100, WeightDtype.BF16, False),    # k-steps that are no multiple of those ahead
    (768, 49, 700, WeightDtype.BF16, False),     # workgroups of sixteen waves
    (1024, 64, 1500, WeightDtype.F16, False),    # the most rows of the widest model they go to
    (1088, 64, 300, WeightDtype.BF16, False),    # one step wider: the library's
    (64, 65, 300, WeightDtype.BF16, False),      # one row more: the library's
    (768, 3, 170000, WeightDtype.BF16, False),   # a table past the cache's size: read past it
])
def test_logits_and_pick(dm, B, vocab, dtype, untied):
    """f32 sums of K products of 16-bit values: 2 K eps of the sum of the products' magnitudes bounds them."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 3)
    w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    g = torch.Generator().manual_seed(B)
    embed = torch.randn(vocab, dm, generator=g)
    embed[vocab // 2:vocab // 2 + 2] = embed[:2] if vocab > 4 else embed[vocab // 2:vocab // 2 + 2]   # equal columns: the last of them is the pick
    head = torch.randn(dm, vocab, generator=g) if untied else embed.T
    lm = GpuMambaLM(GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype), embed.numpy(), head.contiguous().numpy() if untied else None)
    tt = dtype.torch_dtype()
    for step in range(2):
        lm.set_tokens(((np.arange(B) * 7 + step) % vocab).astype(np.int32))
        lm.decode_step()
        got = torch.from_numpy(lm.last_logits()).reshape(B, -1)[:, :vocab]
        hid = torch.from_numpy(lm.backbone.download_temporal()).to(tt).double()
        table = head.to(tt).double()
        bound = 2 * dm * 2.0 ** -24 * (hid.abs() @ table.abs()) + 1e-30
        assert ((got.double() - hid @ table).abs() <= bound).all(), step
        last = vocab - 1 - np.argmax(got.numpy()[:, ::-1], axis=1)
        assert np.array_equal(lm.get_tokens(), last), step


@pytest.mark.parametrize("untied", [False, True])
def test_what_a_table_takes(untied):
    """The rows that tokens are looked up in and the head's tiles, 82 MB each; the f32 rows go through a part of them.  Two uploads of a head of its own take no more, and the second is the
    one that the logits come from."""
    dm, vocab = 1024, 40000
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 3)
    w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    rng = np.random.default_rng(1)
    embed = rng.standard_normal((vocab, dm), np.float32)
    eng = GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, 1, WeightDtype.F16)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    lm = GpuMambaLM(eng, embed, rng.standard_normal((dm, vocab), np.float32) if untied else None)
    head = embed.T
    if untied:
        head = rng.standard_normal((dm, vocab), np.float32)
        backbone._call("mrs_lm_set_untied_head", lm._h, backbone._fp(head))
    assert free - torch.cuda.mem_get_info()[0] <= 2 * vocab * dm * 2 + (16 << 20)
    lm.set_tokens(np.zeros(1, np.int32))
    lm.decode_step()
    got, hid = lm.last_logits().reshape(-1)[:vocab], eng.download_temporal().astype(np.float16).astype(np.float64)
    want = (hid @ head.astype(np.float16).astype(np.float64)).reshape(-1)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
    lm.close()
    eng.close()


@pytest.mark.parametrize("dm,B,dtype", [(768, 1, WeightDtype.BF16), (768, 64, WeightDtype.F16), (1024, 33, WeightDtype.BF16), (2560, 16, WeightDtype.BF16), (2560, 3, WeightDtype.F16)])
def test_logits_are_sums_of_short_sums(dm, B, dtype):
    """A rounding is 2^-24 / sqrt(3) of what is summed so far, so sums of four k-steps, added up over K / 128 of them, are off by that times sqrt(2 + K / 256) of their norm and one chain by
    sqrt(K / 64): 0.8 and 1.2e-7 at 768, 1.2 and 2.2e-7 at 2560.  The matrix cores' sums within a k-step make it up to 1.1 and 1.4 times as much (measured); 1.25 times lies between."""
    cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=1)
    w = MambaWeights.init(cfg, dm, 3)
    w.input_proj_w = np.zeros(0, np.float32); w.input_proj_b = np.zeros(0, np.float32)
    embed = torch.randn(2000, dm, generator=torch.Generator().manual_seed(B))
    lm = GpuMambaLM(GpuMambaBackbone.new_with_dtype(0, w, cfg, dm, B, dtype), embed.numpy(), None)
    lm.set_tokens((np.arange(B) * 7).astype(np.int32))
    lm.decode_step()
    got = torch.from_numpy(lm.last_logits()).reshape(B, -1)[:, :2000].double()
    want = torch.from_numpy(lm.backbone.download_temporal()).to(dtype.torch_dtype()).double() @ embed.to(dtype.torch_dtype()).double().T
    off, unit = float((got - want).norm() / want.norm()), 2.0 ** -24 / 3 ** 0.5
    print(f"logits {dm} {B} {dtype.name} {off:.3e} of {unit * (2 + dm / 256) ** 0.5:.3e}", flush=True)
    assert off <= 1.25 * unit * (2 + dm / 256) ** 0.5
