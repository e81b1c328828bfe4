"""The calls whose speed this package answers for, as a user's program makes them.

A case is a dict of plain values; `kind` says which entry point it goes through:

  step      one control step of a small backbone: GpuMambaBackbone.step / GpuMamba3Backbone.step, host row in, host row out
            (the reference's default configurations: policies and time series models in f32, called once per tick)
  greedy    greedy decoding with a language model: GpuMambaLM.decode_step over a captured graph, the tokens read at the end
  generate  GpuMambaLM.generate_batch: ragged prompts, the sampler in the loop, one list of tokens per slot
  prefill   GpuMambaLM.prefill of whole prompts, the first token read, one decode step on the state it leaves, the second read
  scan      ops.ssm_scan_fwd on tensors that a model of one's own has in hand

Widths are those of the configurations used throughout this repository: the two small default configurations, the 130m,
370m and 2.8b shapes of Mamba-1 and the 768-wide Mamba-3 backbone (the last two Mamba-1 shapes with fewer layers, as the
layers are alike).  Weights are random: projections N(0, 0.02), dt bias inv-softplus(loguniform[1e-3, 1e-1]), A the
S4D-real initialisation or, with `trained_a`, a matrix that has moved away from it as a trained checkpoint's has.
Embedding rows are N(0, 1), so that the token's own identity carries the residual stream and the next token stands out
from the others by far more than rounding, as with a trained model.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mamba_rs_amd import (GpuMamba3Backbone, GpuMamba3LM, GpuMambaBackbone, GpuMambaLM, Mamba3Config, Mamba3LayerWeights,
                          Mamba3Weights, MambaConfig, MambaLayerWeights, MambaWeights, SampleParams, WeightDtype, ops)

DTYPES = {"f32": WeightDtype.F32, "f16": WeightDtype.F16, "bf16": WeightDtype.BF16}


def listed():
    return [
        # an RL policy's tick: the reference's default Mamba-1 configuration, one environment
        {"name": "m1_step_f32_b1", "kind": "step", "family": "m1", "d_model": 128, "n_layers": 3, "input_dim": 128, "batch": 1,
         "dtype": "f32", "trained_a": False},
        # the same for the default Mamba-3 configuration with a vector of environments
        {"name": "m3_step_f32_b48", "kind": "step", "family": "m3", "d_model": 128, "n_layers": 4, "input_dim": 128, "batch": 48,
         "dtype": "f32", "trained_a": False},
        # one user chatting with a 130m-shape model: latency per token is all that counts
        {"name": "greedy_130m_bf16_b1", "kind": "greedy", "family": "m1", "d_model": 768, "n_layers": 24, "batch": 1, "dtype": "bf16",
         "trained_a": False, "vocab": 50280, "steps": 32},
        # a server's full batch on the same model
        {"name": "greedy_130m_bf16_b64", "kind": "greedy", "family": "m1", "d_model": 768, "n_layers": 24, "batch": 64, "dtype": "bf16",
         "trained_a": False, "vocab": 50280, "steps": 16},
        # a wide model at a server's small batch: the weights' bytes begin to count
        {"name": "greedy_2.8b_bf16_b16", "kind": "greedy", "family": "m1", "d_model": 2560, "n_layers": 8, "batch": 16, "dtype": "bf16",
         "trained_a": True, "vocab": 50280, "steps": 16},
        # one user on the Mamba-3 backbone
        {"name": "greedy_m3_768_bf16_b1", "kind": "greedy", "family": "m3", "d_model": 768, "n_layers": 24, "batch": 1, "dtype": "bf16",
         "trained_a": False, "vocab": 50280, "steps": 32},
        # an odd number of requests with prompts of different lengths, sampled, f16 storage
        {"name": "generate_370m_f16_b13", "kind": "generate", "family": "m1", "d_model": 1024, "n_layers": 24, "batch": 13, "dtype": "f16",
         "trained_a": True, "vocab": 50280, "prompt": 12, "steps": 20},
        # a batch of long prompts
        {"name": "prefill_130m_bf16_8x2048", "kind": "prefill", "family": "m1", "d_model": 768, "n_layers": 24, "batch": 8, "T": 2048,
         "dtype": "bf16", "trained_a": False, "vocab": 50280},
        # one prompt of a length that fits no tile, on a trained checkpoint
        {"name": "prefill_370m_bf16_1x777", "kind": "prefill", "family": "m1", "d_model": 1024, "n_layers": 24, "batch": 1, "T": 777,
         "dtype": "bf16", "trained_a": True, "vocab": 50280},
        # the largest: long prompts on a wide model
        {"name": "prefill_2.8b_bf16_4x4096", "kind": "prefill", "family": "m1", "d_model": 2560, "n_layers": 8, "batch": 4, "T": 4096,
         "dtype": "bf16", "trained_a": False, "vocab": 50280},
        # long prompts on the Mamba-3 backbone
        {"name": "prefill_m3_768_bf16_4x4096", "kind": "prefill", "family": "m3", "d_model": 768, "n_layers": 24, "batch": 4, "T": 4096,
         "dtype": "bf16", "trained_a": False, "vocab": 50280},
        # the scan alone, on a trained model's A
        {"name": "scan_bf16_8x2048x1536", "kind": "scan", "batch": 8, "T": 2048, "d_inner": 1536, "dtype": "bf16", "trained_a": True,
         "gated": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, kind):
    """(family, d_model, n_layers): a shape the repository measures, by how often it is met."""
    shapes = [("m1", 768, 24), ("m1", 768, 24), ("m1", 1024, 24), ("m1", 2560, 8), ("m3", 768, 24)]
    return rng.choice(shapes[:-1] if kind == "generate" else shapes)


def draw(rng):
    kind = rng.choice(["step", "greedy", "greedy", "generate", "prefill", "prefill", "scan"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    trained = rng.random() < 0.5
    if kind == "step":
        family = rng.choice(["m1", "m3"])
        return {"kind": kind, "family": family, "d_model": rng.choice([64, 128, 128, 192, 256]), "n_layers": rng.randint(2, 5),
                "input_dim": rng.randint(8, 192), "batch": _log(rng, 1, 128), "dtype": rng.choice(["f32", "f32", "f32", "bf16"]),
                "trained_a": trained and family == "m1"}
    if kind == "scan":
        return {"kind": kind, "batch": rng.randint(1, 8), "T": _log(rng, 64, 4096), "d_inner": 8 * _log(rng, 64, 320),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "trained_a": trained, "gated": rng.random() < 0.8}
    family, d_model, n_layers = _shape(rng, kind)
    trained = trained and family == "m1"
    case = {"kind": kind, "family": family, "d_model": d_model, "n_layers": n_layers, "dtype": dtype, "trained_a": trained, "vocab": 50280}
    if kind == "greedy":
        # one to four rows also in f32, the default storage of the engines
        case["batch"] = _log(rng, 1, 128)
        if case["batch"] <= 4 and d_model < 2560 and rng.random() < 0.3:
            case["dtype"] = "f32"
        case["steps"] = 16
    elif kind == "generate":
        case.update(batch=_log(rng, 1, 64), prompt=rng.randint(4, 24), steps=16)
    else:
        case["batch"] = rng.choice([1, 1, 2, 3, 4, 8])
        case["T"] = max(24, _log(rng, 64, 16384) // case["batch"])
    return case


def _cfg(case):
    if case["family"] == "m1":
        return MambaConfig(d_model=case["d_model"], d_state=16, d_conv=4, expand=2, n_layers=case["n_layers"])
    small = case["d_model"] <= 256
    return Mamba3Config(d_model=case["d_model"], d_state=16 if small else 64, expand=2, headdim=16 if small else 64, ngroups=1,
                        n_layers=case["n_layers"], rope_fraction=0.5)


class _Host:
    """Seeded random host arrays (drawn on the GPU, which is quicker for a hundred million of them)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda:0")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device="cuda:0", generator=self.g).mul_(std).cpu().numpy()

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device="cuda:0", generator=self.g).mul_(hi - lo).add_(lo).cpu().numpy()

    def ints(self, n, *shape):
        return torch.randint(0, n, shape, device="cuda:0", generator=self.g, dtype=torch.int32).cpu().numpy()


def _dt_bias(host, n):
    dt = np.exp(host.uniform(n, lo=math.log(1e-3), hi=math.log(1e-1)))
    return np.log(np.expm1(dt)).astype(np.float32)


def _a_log(host, di, ds, trained):
    a = np.tile(np.log(np.arange(1, ds + 1, dtype=np.float32)), (di, 1))
    return a + host.normal(di, ds, std=0.15) if trained else a


def _weights(case, cfg, host, input_dim):
    """input_dim None: the embedding goes straight in (language models)."""
    L, dm, di, ds = cfg.n_layers, cfg.d_model, cfg.d_inner(), cfg.d_state
    ipw = np.zeros((0, dm), np.float32) if input_dim is None else host.normal(input_dim, dm, std=1 / math.sqrt(input_dim))
    std = 0.02 if dm >= 512 else 1 / math.sqrt(dm)
    near_one = lambda *s: 1 + host.normal(*s, std=0.1)  # noqa: E731
    layers = []
    for _ in range(L):
        if case["family"] == "m1":
            dr = cfg.dt_rank()
            layers.append(MambaLayerWeights(near_one(dm), host.normal(dm, 2 * di, std=std), host.uniform(di, cfg.d_conv, lo=-0.87, hi=0.87),
                                            host.normal(di, std=0.1), host.normal(di, dr + 2 * ds, std=std), host.normal(dr, di, std=std),
                                            _dt_bias(host, di), _a_log(host, di, ds, case["trained_a"]), near_one(di),
                                            host.normal(di, dm, std=std)))
        else:
            nh = cfg.nheads()
            layers.append(Mamba3LayerWeights(near_one(dm), host.normal(dm, cfg.in_proj_out_dim(), std=std), _dt_bias(host, nh), near_one(ds),
                                             near_one(ds), near_one(nh, ds), near_one(nh, ds), near_one(nh), near_one(di),
                                             host.normal(di, dm, std=std)))
    kind = MambaWeights if case["family"] == "m1" else Mamba3Weights
    return kind(ipw, np.zeros(dm, np.float32), layers, near_one(dm))


def _backbone(case, host, input_dim, batch):
    cfg = _cfg(case)
    w = _weights(case, cfg, host, input_dim)
    make = GpuMambaBackbone if case["family"] == "m1" else GpuMamba3Backbone
    return make.new_with_dtype(0, w, cfg, cfg.d_model if input_dim is None else input_dim, batch, DTYPES[case["dtype"]])


class _Rows:
    """The engine's final-norm rows as a tensor on its own memory."""

    def __init__(self, backbone):
        self.owner = backbone
        self.__cuda_array_interface__ = {"shape": (backbone.batch, backbone.cfg.d_model), "typestr": "<f4", "version": 3,
                                         "data": (backbone.temporal_ptr(), False), "strides": None}


def _prepare_scan(case, host_seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(host_seed)
    B, T, di, ds = case["batch"], case["T"], case["d_inner"], 16
    dt = DTYPES[case["dtype"]].torch_dtype()
    n = lambda *s: torch.randn(*s, device="cuda:0", generator=g)  # noqa: E731
    bias = torch.log(torch.expm1(torch.exp(torch.rand(di, device="cuda:0", generator=g) * math.log(100.0) + math.log(1e-3))))
    delta = torch.nn.functional.softplus(n(B, T, di) * 0.5 + bias).to(dt)
    a_log = torch.log(torch.arange(1, ds + 1, device="cuda:0", dtype=torch.float32)).repeat(di, 1)
    if case["trained_a"]:
        a_log = a_log + 0.15 * n(di, ds)
    a_neg = ops.exp_negate(a_log.contiguous())
    flags = (ops.GATE_SILU if case["gated"] else 0) | ops.SCAN_FLAGS_ZERO | (ops.A_S4D_REAL if ops.a_neg_is_s4d_real(a_neg) else 0)
    return {"case": case, "h": torch.zeros(B, di, ds, device="cuda:0"), "y": torch.empty_like(delta), "delta": delta,
            "u": n(B, T, di).to(dt), "B": n(B, T, ds).to(dt), "C": n(B, T, ds).to(dt), "a_neg": a_neg,
            "D": torch.rand(di, device="cuda:0", generator=g) + 0.5, "gate": n(B, T, di).to(dt) if case["gated"] else None, "flags": flags,
            "ws": torch.zeros(max(256, ops.ssm_scan_workspace_bytes(B, T, di, ds)), dtype=torch.uint8, device="cuda:0")}


def prepare(case, seed):
    if case["kind"] == "scan":
        return _prepare_scan(case, seed)
    host = _Host(seed)
    if case["kind"] == "step":
        bb = _backbone(case, host, case["input_dim"], case["batch"])
        x = host.normal(case["batch"], case["input_dim"])
        bb.capture_graph()
        return {"case": case, "backbone": bb, "x": x}
    bb = _backbone(case, host, None, case["batch"])
    make = GpuMambaLM if case["family"] == "m1" else GpuMamba3LM
    lm = make(bb, host.normal(case["vocab"], case["d_model"]))
    state = {"case": case, "backbone": bb, "lm": lm, "rows": torch.as_tensor(_Rows(bb), device="cuda:0")}
    if case["kind"] == "generate":
        lens = [case["prompt"] + i % 5 for i in range(case["batch"])]
        state["prompts"] = [host.ints(case["vocab"], n).tolist() for n in lens]
        state["params"] = [SampleParams(temperature=0.8, top_k=50, top_p=0.95, max_tokens=case["steps"], seed=seed + i)
                           for i in range(case["batch"])]
        return state
    if case["kind"] == "prefill":
        state["tokens"] = host.ints(case["vocab"], case["batch"], case["T"])
        bb.alloc_prefill_scratch(case["T"])
    else:
        state["tokens"] = host.ints(case["vocab"], case["batch"])
    lm.set_tokens(np.zeros(case["batch"], np.int32))
    lm.capture_graph()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        return state["backbone"].step(state["x"])
    if kind == "scan":
        state["h"].zero_()
        y = ops.ssm_scan_fwd(state["h"], state["y"], state["delta"], state["u"], state["B"], state["C"], state["a_neg"], state["D"],
                             gate=state["gate"], flags=state["flags"], workspace=state["ws"])
        return {"y": y, "h": state["h"]}
    lm = state["lm"]
    if kind == "generate":
        return {"tokens": np.asarray(lm.generate_batch(state["prompts"], state["params"]), np.int32), "rows": state["rows"]}
    state["backbone"].reset()
    if kind == "prefill":
        lm.prefill(state["tokens"])
        first = lm.get_tokens()
        lm.decode_step()
        return {"first": first, "second": lm.get_tokens(), "rows": state["rows"]}
    lm.set_tokens(state["tokens"])
    for _ in range(case["steps"]):
        lm.decode_step()
    return {"tokens": lm.get_tokens(), "rows": state["rows"]}


def _layer(case):
    """(weight elements, recurrent state floats of a row) of one layer."""
    cfg = _cfg(case)
    dm, di = cfg.d_model, cfg.d_inner()
    if case["family"] == "m1":
        xd = cfg.xdbl_dim()
        return dm * 2 * di + di * xd + cfg.dt_rank() * di + di * dm, di * (cfg.d_state + cfg.d_conv)
    return dm * cfg.in_proj_out_dim() + di * dm, cfg.nheads() * (cfg.headdim * cfg.d_state + cfg.d_state + cfg.headdim + cfg.num_rope_angles())


def work(case):
    es = DTYPES[case["dtype"]].size_bytes()
    B = case["batch"]
    if case["kind"] == "scan":
        T, di, ds = case["T"], case["d_inner"], 16
        return {"bytes": es * B * T * (di * (3 + case["gated"]) + 2 * ds) + 8 * B * di * ds + 4 * di * (ds + 1), "flops": 6 * B * T * di * ds}
    weights, state = _layer(case)
    L, dm = case["n_layers"], case["d_model"]
    if case["kind"] == "step":
        weights_all = L * weights + case["input_dim"] * dm
        return {"bytes": es * weights_all + 8 * L * B * state + 4 * B * (case["input_dim"] + dm), "flops": 2 * B * weights_all}
    head = case["vocab"] * dm
    one = {"bytes": es * (L * weights + head) + 8 * L * B * state, "flops": 2 * B * (L * weights + head)}
    if case["kind"] == "prefill":
        rows = B * case["T"]
        cfg = _cfg(case)
        # Mamba-3 from 64 steps up: the four contractions of a chunk of 64
        chunks = 0 if case["family"] == "m1" else 4 * 2 * 64 * cfg.headdim * cfg.d_state * math.ceil(case["T"] / 64) * B * cfg.nheads()
        return {"bytes": 2 * one["bytes"] + rows * (4 + es * dm), "flops": one["flops"] + L * (2 * rows * weights + chunks) + 2 * B * head}
    n = case["steps"] + (case["prompt"] + min(B - 1, 4) if case["kind"] == "generate" else 0)
    return {"bytes": n * one["bytes"], "flops": n * one["flops"]}


def tolerance(case):
    if case["kind"] == "scan":
        return {"rel": 2e-5} if case["dtype"] == "f32" else {"rel": 1e-2}
    # f32: the layers' sums in another order, and the exponentials of the scan; 16 bits: every layer rounds its projections,
    # its gate and its output once each, and the layers' roundings add up along the residual stream
    if case["dtype"] == "f32":
        return {"rel": 5e-5, "differ": 0.01}
    return {"rel": 2e-2, "differ": 0.01}
