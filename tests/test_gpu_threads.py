"""Forward passes of one thread beside training steps of another on the same stream: each call keeps the stream's workspace
until its launches are queued, so every result is the one the call gives alone."""
import threading

import pytest
import torch

import bibo_amd

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _layer(seed, H=256, I=128, E=16, k=4):
    torch.manual_seed(seed)
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=H, moe_intermediate_size=I, num_routed_experts=E, num_experts_per_tok=k,
                                 special_expert_pairs=0, bias_update_factor=0.0)
    return bibo_amd.BiBoMoELayer(cfg).to(DEV).bfloat16()


def test_two_threads_on_one_stream():
    infer, train = _layer(0).eval(), _layer(1)
    train.keep_activations = False                  # the backward pass recomputes: the longest use of the workspace
    x, y = torch.randn(1, 700, 256, device=DEV).bfloat16(), torch.randn(1, 900, 256, device=DEV).bfloat16()
    d = torch.randn_like(y)

    def forward():
        with torch.no_grad():
            return [infer(x)]

    def step():
        yg = y.clone().requires_grad_()
        train.zero_grad(set_to_none=True)
        out = train(yg)
        out.backward(d)
        return [out.detach(), yg.grad] + [p.grad for p in train.parameters() if p.requires_grad]

    want = {f: f() for f in (forward, step)}
    torch.cuda.synchronize()
    wrong = []

    def loop(f, n):
        for _ in range(n):
            got = f()
            torch.cuda.current_stream().synchronize()
            if not all(torch.equal(a, b) for a, b in zip(got, want[f])):
                wrong.append(f.__name__)

    threads = [threading.Thread(target=loop, args=a) for a in ((forward, 300), (step, 100))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
