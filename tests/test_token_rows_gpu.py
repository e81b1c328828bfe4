"""GPU: what a decode step takes its rows from (the embedding table, inside the step's first kernel) and what picks the next token."""
import numpy as np
import pytest
import torch

from util import cosine

pytestmark = pytest.mark.gpu

from mamba_rs_amd import (GpuMamba3Backbone, GpuMamba3LM, GpuMambaBackbone, GpuMambaLM, Mamba3Config, Mamba3Weights, MambaConfig, MambaWeights,  # noqa: E402
                          WeightDtype)


class _Device:
    """Device memory of an engine as a tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "version": 3, "data": (ptr, False), "strides": None}


def _model(family, dm, layers):
    if family == "m1":
        cfg = MambaConfig(d_model=dm, d_state=16, d_conv=4, expand=2, n_layers=layers)
        return cfg, MambaWeights.random_lm(cfg, seed=3, std=0.05), GpuMambaBackbone, GpuMambaLM
    cfg = Mamba3Config(d_model=dm, d_state=64, expand=2, headdim=64, ngroups=1, n_layers=layers, rope_fraction=0.5)
    return cfg, Mamba3Weights.random_lm(cfg, seed=3, std=0.05), GpuMamba3Backbone, GpuMamba3LM


@pytest.mark.parametrize("family,dm,layers,B,dtype,resident", [
    ("m1", 256, 2, 1, WeightDtype.BF16, True),     # resident_step.hip
    ("m1", 256, 2, 1, WeightDtype.BF16, False),    # the kernel chain, row-wise
    ("m1", 256, 2, 40, WeightDtype.F16, True),     # resident_rows.hip, rows over several groups
    ("m1", 256, 2, 40, WeightDtype.F16, False),    # the kernel chain on tiles
    ("m1", 256, 2, 130, WeightDtype.BF16, True),   # the library chain: rows gathered by a launch
    ("m1", 64, 2, 3, WeightDtype.F32, True),       # one launch per step, f32
    ("m1", 256, 1, 2, WeightDtype.F32, True),      # f32 chain
    ("m3", 256, 2, 1, WeightDtype.BF16, True),     # resident_m3_row.hip
    ("m3", 256, 2, 4, WeightDtype.F16, True),      # resident_m3_step.hip
    ("m3", 256, 2, 4, WeightDtype.F16, False),     # its kernel chain
])
def test_a_step_on_tokens_is_the_step_on_their_embedding_rows(family, dm, layers, B, dtype, resident, monkeypatch):
    """The same kernels on the same values: the final rows are equal to the bit, and the input buffer holds the embedding rows
    (tokens outside the vocabulary are clamped to it)."""
    if not resident:
        monkeypatch.setenv("MRS_DECODE_NO_RESIDENT", "1")
    cfg, w, backbone, lm_kind = _model(family, dm, layers)
    rng = np.random.default_rng(B)
    V = 777
    embed = rng.standard_normal((V, dm)).astype(np.float32)
    stored = torch.from_numpy(embed).to(dtype.torch_dtype()).float().numpy()
    tokens = rng.integers(0, V, B).astype(np.int32)
    tokens[0] = V + 5
    if B > 2:
        tokens[1] = -3
    want_in = stored[np.clip(tokens, 0, V - 1)]
    print(f"case token rows {family} d_model={dm} rows={B} {dtype.name} resident={resident}", flush=True)
    plain = backbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    want = plain.step(want_in)
    plain.close()
    bb = backbone.new_with_dtype(0, w, cfg, dm, B, dtype)
    lm = lm_kind(bb, embed)
    lm.set_tokens(tokens)
    lm.decode_step()
    got_tokens = lm.get_tokens()
    logits = lm.last_logits()
    rows = torch.as_tensor(_Device(bb.temporal_ptr(), (B, dm)), device="cuda:0").cpu().numpy()
    took = torch.as_tensor(_Device(bb.input_ptr(), (B, dm)), device="cuda:0").cpu().numpy()
    assert (took == want_in).all()
    assert (rows == want).all()
    assert (got_tokens == logits.argmax(1)).all()
    head = torch.from_numpy(rows).to(dtype.torch_dtype()).float().numpy() @ stored.T
    assert min(cosine(logits[b], head[b]) for b in range(B)) > 0.99999
    bb.close()


@pytest.mark.parametrize("V,B", [(1, 3), (7, 3), (64, 3), (2047, 3), (2048, 3), (2049, 3), (5000, 7), (5000, 8), (8191, 9), (8192, 9), (8193, 9), (20001, 8)])
def test_the_greedy_token_is_the_last_of_the_largest(V, B):
    """Every column of the head occurs several times, in all slices of a row and at its ends, and rows of equal logits throughout: the last
    index of the maximum, step after step (the words the slices meet in are cleared by the last of them)."""
    dm = 64
    cfg, w, backbone, lm_kind = _model("m1", dm, 1)
    rng = np.random.default_rng(V)
    head = rng.standard_normal((dm, 1 + V // 5)).astype(np.float32)[:, rng.integers(0, 1 + V // 5, V)]
    embed = rng.standard_normal((V, dm)).astype(np.float32)
    for lm_head in (head, np.zeros((dm, V), np.float32)):
        print(f"case greedy ties vocab={V}", flush=True)
        bb = backbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.F32)
        lm = lm_kind(bb, embed, lm_head)
        lm.set_tokens(np.arange(B, dtype=np.int32) % V)
        for _ in range(4):
            lm.decode_step()
            got, logits = lm.get_tokens(), lm.last_logits()
            assert (got == V - 1 - logits[:, ::-1].argmax(1)).all()
        bb.close()


@pytest.mark.parametrize("V,B", [(1, 3), (7, 3), (2049, 3), (5000, 8), (8193, 8), (20001, 8)])
def test_the_greedy_token_of_rows_with_masks_infinities_and_nan(V, B):
    """Head columns that make a logit -inf, inf or NaN in every row: the last of the largest numbers, NaN passed over, and the vocabulary's last entry where
    nothing is above -inf (Iterator::max_by keeps the later of two that do not compare).  Masked columns take a row's positive entry times -inf,
    all other terms of the sum being zero."""
    dm = 64
    cfg, w, backbone, lm_kind = _model("m1", dm, 1)
    rng = np.random.default_rng(V)
    embed = rng.standard_normal((V, dm)).astype(np.float32)
    tokens = np.arange(B, dtype=np.int32) % min(V, 3)
    plain = backbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.F32)
    rows = plain.step(embed[tokens])
    plain.close()
    k = int(rows.min(0).argmax())
    assert rows[:, k].min() > 0
    head = rng.standard_normal((dm, V)).astype(np.float32)
    low, high, nan = np.zeros(dm, np.float32), np.zeros(dm, np.float32), np.full(dm, np.nan, np.float32)
    low[k], high[k] = -np.inf, np.inf

    def some(*columns):   # most columns of the first kind, a few numbers or other kinds among them
        h = np.tile(columns[0][:, None], (1, V))
        for i, c in enumerate(columns[1:]):
            at = rng.integers(0, V, 1 + V // 50)
            h[:, at] = head[:, at] if c is None else c[:, None]
        return h
    for what, lm_head in (("-inf", some(low)), ("nan", some(nan)), ("-inf and nan", some(low, nan)), ("nan and -inf", some(nan, low)), ("-inf, numbers", some(low, None)),
                          ("nan, numbers", some(nan, None)), ("nan, numbers, -inf", some(nan, None, low)), ("-inf, inf, nan", some(low, high, nan))):
        print(f"case greedy vocab={V} rows={B}: {what}", flush=True)
        bb = backbone.new_with_dtype(0, w, cfg, dm, B, WeightDtype.F32)
        lm = lm_kind(bb, embed, lm_head)
        for _ in range(3):
            bb.reset()
            lm.set_tokens(tokens)
            lm.decode_step()
            got, logits = lm.get_tokens(), lm.last_logits()
            assert (np.isnan(logits) == np.isnan(lm_head).any(0)).all() and (np.isneginf(logits) == np.isneginf(lm_head).any(0)).all()
            v = np.where(np.isnan(logits), -np.inf, logits)
            assert (got == V - 1 - v[:, ::-1].argmax(1)).all(), (what, got)
        bb.close()
