"""Forward passes of one thread beside training steps of another on the same stream: each call keeps the stream's workspace
until its launches are queued, so every result is the one the call gives alone."""
import threading
import time

import pytest
import torch

import bibo_amd
from bibo_amd import ops

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


def _together(*loops):
    threads = [threading.Thread(target=f) for f in loops]
    for t in threads:
        t.start()
    for t in threads:
        t.join()


def test_buffer_that_grows_and_goes_while_threads_use_it():
    """The buffer is allocated anew in a backward pass and in forwards, after Python has had it in hand (its last reference then
    takes the interpreter lock) and while allocations ask for Python's stack (they take it too)."""
    infer, train = _layer(0).eval(), _layer(1)
    train.keep_activations = False
    sizes = [64 + 97 * i for i in range(12)]
    g = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(1, sizes[-1], 256, generator=g, device=DEV).bfloat16()
    d = torch.randn_like(x)

    def forward(n):
        with torch.no_grad():
            return infer(x[:, :n])

    def step(n):
        xg = x[:, :n].clone().requires_grad_()
        train(xg).backward(d[:, :n])
        return xg.grad

    want = {(f, n): f(n) for f in (forward, step) for n in sizes}
    wrong = []

    def loop(f, order):
        def run():
            for n in order:
                got = f(n)
                torch.cuda.current_stream().synchronize()
                if not torch.equal(got, want[f, n]):
                    wrong.append((f.__name__, n))
        return run

    def clear():
        for _ in range(100):
            ops.workspace(DEV, 1)                   # seen by Python
            ops._workspaces.clear()
            time.sleep(0.002)

    torch.cuda.memory._record_memory_history(max_entries=1000)
    try:
        for _ in range(5):
            _together(loop(forward, sizes), loop(step, sizes), loop(forward, sizes[::-1]), clear)
    finally:
        torch.cuda.memory._record_memory_history(enabled=None)
    assert not wrong, wrong[:5]


def test_tensor_level_calls_keep_the_buffer_too():
    infer, other = _layer(0).eval(), _layer(2)
    x, y = torch.randn(1, 700, 256, device=DEV).bfloat16(), torch.randn(900, 256, device=DEV).bfloat16()
    p = [t.detach() for t in (other.gate.gate_proj.weight, other.gate.bias.float(), other.experts.gate_up_proj, other.experts.down_proj,
                              other.experts.radial_theta.float())]

    def forward():
        with torch.no_grad():
            return [infer(x)]

    def tensors():
        return [ops.moe_forward(y, *p, 4)[0], *ops.moe_backward(y, y, *p, 4)[:5]]

    want = {f: f() for f in (forward, tensors)}
    wrong = []

    def loop(f, n):
        def run():
            for _ in range(n):
                got = f()
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[f])):
                    wrong.append(f.__name__)
        return run

    _together(loop(forward, 200), loop(tensors, 100))
    assert not wrong, wrong[:5]


def test_a_waiting_call_leaves_the_interpreter_to_others():
    layer, x, done = _layer(0).eval(), torch.randn(1, 64, 256, device=DEV).bfloat16(), []
    with torch.no_grad():
        want = layer(x)

    def call():
        with torch.no_grad():
            done.append(layer(x))

    thread = threading.Thread(target=call)
    with ops._held(DEV, 1):
        thread.start()
        for _ in range(10):                         # each needs the interpreter back while the call waits for the buffer
            time.sleep(0.02)
        assert not done
        with ops._held(DEV, 1 << 22) as (_, size):  # the same thread may take it again, and larger
            assert size >= 1 << 22
    thread.join()
    assert torch.equal(done[0], want)
