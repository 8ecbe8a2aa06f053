"""bibo_moe_balance_step against the tensor operations of BiBoMoELayer._balance_step / update_bias (moe.py:131-155), and the
layer's own use of it: counts accumulate between updates, the bias moves on the update, versions advance."""
import pytest
import torch

import bibo_amd
from bibo_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("E", [1, 9, 63, 64])
def test_balance_step_kernel(E):
    g = torch.Generator(device=DEV).manual_seed(E)
    counts = torch.randint(0, 1000, (E,), generator=g, device=DEV, dtype=torch.int32)
    acc = torch.randint(0, 1000, (E,), generator=g, device=DEV).float()
    bias = torch.rand(E, generator=g, device=DEV) * 0.02
    for c in (counts, torch.zeros_like(counts)):
        a, b = acc.clone(), bias.clone()
        L.native().balance_step(c, a, b, 0.4, False)
        assert torch.equal(a, acc + c) and torch.equal(b, bias)
        L.native().balance_step(c, a, b, 0.4, True)
        load = (acc + 2 * c) / (acc + 2 * c).sum().clamp_min(1.0)
        assert torch.allclose(b, bias + 0.4 * (load.mean() - load), rtol=0, atol=1e-8)
        assert float(a.abs().max()) == 0.0


def test_training_forwards_move_the_bias_as_the_tensor_operations_do():
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=128, moe_intermediate_size=128, num_routed_experts=16, num_experts_per_tok=4,
                                 special_expert_pairs=1, bias_update_threshold=120)
    layer = bibo_amd.BiBoMoELayer(cfg).to(DEV)
    plain = bibo_amd.BiBoMoELayer(cfg).to(DEV)
    plain.load_state_dict(layer.state_dict())
    plain.update_bias = lambda tpe: bibo_amd.BiBoMoELayer.update_bias(plain, tpe)      # overridden: the tensor operations
    for step in range(5):
        x = torch.randn(1, 60, 128, device=DEV)
        version = layer.gate.bias._version
        assert torch.equal(layer(x), plain(x))
        assert (layer.gate.bias._version > version) == (step % 2 == 1)
        assert torch.equal(layer.accumulated_tpe, plain.accumulated_tpe)
        assert torch.allclose(layer.gate.bias, plain.gate.bias, rtol=0, atol=1e-8)


@pytest.mark.parametrize("method", ["update_bias", "_balance_step"])
def test_balancing_methods_replaced_on_the_class_are_called(method, monkeypatch):
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=128, moe_intermediate_size=128, num_routed_experts=16, num_experts_per_tok=4,
                                 special_expert_pairs=0, bias_update_threshold=60)
    layer, seen = bibo_amd.BiBoMoELayer(cfg).to(DEV), []
    plain = getattr(bibo_amd.BiBoMoELayer, method)
    monkeypatch.setattr(bibo_amd.BiBoMoELayer, method, lambda self, *a, **kw: seen.append(1) or plain(self, *a, **kw))
    layer(torch.randn(1, 60, 128, device=DEV))
    assert seen == [1]
