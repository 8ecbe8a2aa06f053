"""A tile's columns cut over several workgroups (launch_gateup_raw + launch_down_act, what `auto` runs with few tiles) at the edges
of its tiles: 1 to 129 rows per expert, idle experts, one and several column blocks, I = 256, 384, 512; against the fp32 oracle and
against the uncut kernels, and the state-keeping training pair through the same launches."""
import numpy as np
import pytest
import torch

import bibo_amd
from bibo_amd import ops
from oracle import bibo_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _rel(a, ref):
    return float((a.double().cpu() - ref.double()).abs().max() / ref.double().abs().max().clamp_min(1e-30))


def _with_idle_experts(rows):
    """So many that `auto` cuts these rows at every size here: past streaming's rows per expert, within split_columns."""
    return rows + (0,) * ((8 if sum(rows) < 300 else 16) - len(rows))


@pytest.mark.parametrize("H,I", [(768, 256), (640, 384), (768, 384), (1024, 512), (1024, 256)])
@pytest.mark.parametrize("rows", [(40, 1, 0, 200), (31, 32, 33, 64), (65, 128, 129, 127), (300, 0, 0, 96)])
def test_cut_tiles(H, I, rows):
    rows = _with_idle_experts(rows)
    E, k = len(rows), 1
    T = sum(rows)
    p = O.make_inputs(T=T, H=H, E=E, k=k, I=I, theta="normal", seed=T + H)
    idx = np.repeat(np.arange(E, dtype=np.int32), rows)
    np.random.default_rng(T).shuffle(idx)
    idx = idx.reshape(T, 1)
    w = np.random.default_rng(1).random((T, 1)).astype(np.float32)
    args = [torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))]
    ref = O.experts_forward(p["x"], idx, w, p["w_gate_up"], p["w_down"], p["theta"])
    for act in ("radial", "silu"):
        got, counts = ops.experts_fwd(p["x"].to(DEV), *args, act=act, want_counts=True)
        whole, _ = ops.experts_fwd(p["x"].to(DEV), *args, act=act, algo="mfma" if I == 512 else "fused")
        torch.cuda.synchronize()
        assert counts.tolist() == list(rows)
        assert _rel(got, whole.cpu()) <= 1e-2
        if act == "radial":
            assert _rel(got, ref) <= 2e-2


@pytest.mark.parametrize("H,I", [(768, 384), (1024, 256), (640, 384)])
def test_cut_tiles_lose_no_precision(H, I):
    """Pre-activations cross memory in fp32: the same sums as the uncut kernel's registers hold, activated in the same order but
    for the sum of squares, so results differ only where that tips a rounding.  (Rounded to bf16 on the way, their 2^-9 shows up
    as 4e-3 here.)"""
    rows = _with_idle_experts((65, 128, 129, 127))
    T, E = sum(rows), len(rows)
    p = O.make_inputs(T=T, H=H, E=E, k=1, I=I, theta="normal", seed=T + H)
    args = [torch.from_numpy(np.repeat(np.arange(E, dtype=np.int32), rows).reshape(T, 1)).to(DEV), torch.ones(T, 1, device=DEV),
            *(p[n].to(DEV) for n in ("w_gate_up", "w_down", "theta"))]
    cut = ops.experts_fwd(p["x"].to(DEV), *args)[0].double()
    whole = ops.experts_fwd(p["x"].to(DEV), *args, algo="fused")[0].double()
    assert float((cut - whole).norm() / whole.norm()) <= 5e-4


def test_training_on_cut_tiles():
    """The module's training forward takes the cut kernels too: its output is the inference forward's, its gradients those of
    a layer that keeps nothing, bit for bit."""
    torch.manual_seed(0)
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=768, moe_intermediate_size=384, num_routed_experts=16, num_experts_per_tok=3,
                                 special_expert_pairs=1, bias_update_factor=0.0)
    layer = bibo_amd.BiBoMoELayer(cfg).to(DEV).bfloat16()
    x = torch.randn(1, 500, 768, device=DEV).bfloat16()
    d = torch.randn(1, 500, 768, device=DEV).bfloat16()
    with torch.no_grad():
        plain = layer(x)
    grads = []
    for layer.keep_activations in (True, False):
        layer.zero_grad(set_to_none=True)
        xg = x.clone().requires_grad_()
        out = layer(xg)
        assert torch.equal(out, plain)
        out.backward(d)
        grads.append([xg.grad] + [p.grad for p in layer.parameters() if p.requires_grad])
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("algo", ["fused", "mfma"])
def test_a_named_family_runs_in_training_too(algo):
    """A layer asked for a family by name runs it in training as in inference: the same bits, also where `auto` cuts the tiles."""
    torch.manual_seed(0)
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=768, moe_intermediate_size=384, num_routed_experts=16, num_experts_per_tok=3,
                                 special_expert_pairs=0, bias_update_factor=0.0)
    layer = bibo_amd.BiBoMoELayer(cfg).to(DEV).bfloat16()
    x = torch.randn(1, 500, 768, device=DEV).bfloat16()
    with torch.no_grad():
        auto = layer(x)
        layer.experts.algo = algo
        plain = layer(x)
    assert not torch.equal(plain, auto)                 # `auto` does cut here
    assert torch.equal(layer(x.clone().requires_grad_()), plain)
