"""The balancing step that a training forward takes along in its combine kernel (or behind the few-token kernels) against the step as a launch
of its own: the same counts and biases, bit for bit, with updates in between, through every combine kernel."""
import pytest
import torch
import torch.utils.checkpoint

import bibo_amd

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("dtype,T,H,I,E,k,pairs", [
    (torch.bfloat16, 300, 256, 128, 64, 6, 0),     # bf16 slot rows, 8 columns a thread
    (torch.bfloat16, 40, 256, 512, 9, 2, 1),       # fp32 slot rows, 4 columns a thread
    (torch.float32, 777, 64, 32, 63, 3, 0),
    (torch.float32, 60, 50, 30, 5, 2, 1),          # one column a thread
    (torch.bfloat16, 60, 50, 30, 5, 2, 1),
    (torch.bfloat16, 300, 1024, 512, 8, 2, 0),     # counts from workgroups that find their rows themselves
    (torch.float32, 4, 64, 32, 8, 3, 0),           # few tokens: no combine
    (torch.bfloat16, 1, 256, 128, 8, 2, 0),
])
def test_balance_in_the_combine(dtype, T, H, I, E, k, pairs):
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=H, moe_intermediate_size=I, num_routed_experts=E, num_experts_per_tok=k,
                                 special_expert_pairs=pairs, bias_update_threshold=2 * T)
    layers = []
    for keep in (True, False):                     # without kept activations the step is a launch of its own
        torch.manual_seed(3)
        layer = bibo_amd.BiBoMoELayer(cfg).to(DEV).train()
        for p in (layer.gate.gate_proj.weight, layer.experts.gate_up_proj, layer.experts.down_proj):
            p.data = p.data.to(dtype)
        layer.keep_activations = keep
        layers.append(layer)
    a, b = layers
    for step in range(5):
        x = torch.randn(1, T, H, device=DEV).to(dtype)
        versions = a.gate.bias._version, a.accumulated_tpe._version
        a(x), b(x)
        assert torch.equal(a.gate.bias, b.gate.bias) and torch.equal(a.accumulated_tpe, b.accumulated_tpe)
        assert (a.gate.bias._version > versions[0]) == (step % 2 == 1) and a.accumulated_tpe._version > versions[1]
        assert a._fwd_step == b._fwd_step and a._update_every == b._update_every == 2
    assert float(a.gate.bias.abs().max()) > 0 and float(a.accumulated_tpe.sum()) == T * k


def test_replaced_balance_is_called():
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=128, moe_intermediate_size=128, num_routed_experts=16, num_experts_per_tok=4, special_expert_pairs=0)
    layer, seen = bibo_amd.BiBoMoELayer(cfg).to(DEV).train(), []
    layer._balance = lambda counts, n: seen.append((int(counts.sum()), n))
    layer(torch.randn(1, 60, 128, device=DEV))
    assert seen == [(240, 60)] and float(layer.accumulated_tpe.abs().max()) == 0


def _small(**kw):
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=128, moe_intermediate_size=128, num_routed_experts=16, num_experts_per_tok=4, special_expert_pairs=0, **kw)
    layer = bibo_amd.BiBoMoELayer(cfg).to(DEV).train()
    for p in (layer.gate.gate_proj.weight, layer.experts.gate_up_proj, layer.experts.down_proj):
        p.data = p.data.bfloat16()
    return layer, torch.randn(1, 60, 128, device=DEV, dtype=torch.bfloat16, requires_grad=True)


def test_a_recomputation_takes_no_step_of_its_own():
    """Checkpointing ends the recomputation with the last tensor it needs, in front of the balancing step: with a cadence of two forwards the
    bias moves with every second one, from the counts of two."""
    layer, x = _small(bias_update_threshold=120)
    plain, _ = _small(bias_update_threshold=120)
    plain.load_state_dict(layer.state_dict())
    for step in range(4):
        torch.utils.checkpoint.checkpoint(layer, x, use_reentrant=False).sum().backward()
        plain(x)
        assert layer._fwd_step == plain._fwd_step == step + 1
        assert torch.equal(layer.accumulated_tpe, plain.accumulated_tpe) and torch.equal(layer.gate.bias, plain.gate.bias)
    assert float(layer.gate.bias.abs().max()) > 0


def test_a_forward_that_a_hook_ends_takes_no_step():
    layer, x = _small(bias_update_threshold=1)
    def refuse(t):
        raise RuntimeError("refused")
    with pytest.raises(RuntimeError, match="refused"), torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t):
        layer(x)
    assert layer._fwd_step == 0 and float(layer.gate.bias.abs().max()) == 0 and float(layer.accumulated_tpe.abs().max()) == 0


def test_the_step_follows_the_shared_expert():
    layer, x = _small(bias_update_threshold=1, use_shared_expert=True)
    layer.shared_experts_list[0].bfloat16()
    seen = []
    def refuse(module, args):
        seen.append((layer._fwd_step, float(layer.gate.bias.abs().max())))
        if len(seen) == 1:
            raise RuntimeError("refused")
    layer.shared_experts_list[0].register_forward_pre_hook(refuse)
    with pytest.raises(RuntimeError, match="refused"):
        layer(x)
    layer(x)
    assert seen == [(0, 0.0), (0, 0.0)] and layer._fwd_step == 1 and float(layer.gate.bias.abs().max()) > 0
