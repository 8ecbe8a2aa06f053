"""Expert kernels that find a tile's rows in the routing itself (no permutation launch; a call that asks for counts has one): the same
bits either way, at the ends of 8, 16 and 32 slots a thread and of the range, cut and uncut tiles, with experts that every token picks,
with +/-Identity experts, and with nothing but those."""
import pytest
import torch

from bibo_amd import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _same(T, H, I, Eg, k, pairs=0, hot=(), algo="auto"):
    g = torch.Generator().manual_seed(T + I)
    E = Eg + 2 * pairs
    x = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    wr = (torch.randn(E, H, generator=g) * 0.1).bfloat16().to(DEV)
    bias = torch.rand(E, generator=g) * 0.02 - 0.01
    bias[list(hot)] += 2.0
    gu = (torch.randn(Eg, 2 * I, H, generator=g) * 0.05).bfloat16().to(DEV)
    dn = (torch.randn(Eg, H, I, generator=g) * 0.05).bfloat16().to(DEV)
    th = torch.randn(Eg, generator=g).to(DEV)
    args = (x, wr, bias.to(DEV), gu, dn, th, k)
    kw = dict(n_pos=pairs, n_neg=pairs, algo=algo)
    ref, _, _, counts, _ = ops.moe_forward(*args, want_counts=True, **kw)
    for _ in range(2):                                    # the second pass finds the first one's scratch memory
        got, idx, _, _, _ = ops.moe_forward(*args, want_routing=True, **kw)
        assert torch.equal(got, ref)
    assert torch.equal(torch.bincount(idx.flatten().long(), minlength=E).int(), counts)
    assert float(ref.float().abs().max()) > 0
    return counts


@pytest.mark.parametrize("T", [1, 17, 511, 512, 513, 4095, 4096, 4097, 8191])
@pytest.mark.parametrize("H,I", [(128, 128), (256, 256), (384, 384), (512, 512)])
def test_one_expert_per_token(H, I, T):
    _same(T, H, I, 7, 1, algo="fused" if I < 512 else "auto")


@pytest.mark.parametrize("T,k", [(64, 8), (682, 6), (683, 6), (1024, 8), (1366, 6), (2048, 8), (2049, 8), (2730, 6), (2731, 6)])
@pytest.mark.parametrize("H,I", [(256, 256), (384, 384), (512, 512)])
def test_ends_of_the_range(H, I, T, k):
    _same(T, H, I, 64, k)


@pytest.mark.parametrize("T", [100, 256, 400])
@pytest.mark.parametrize("H,I,E,k", [(768, 384, 64, 6), (1024, 512, 64, 8), (1024, 256, 32, 4)])
def test_cut_tiles(H, I, E, k, T):
    _same(T, H, I, E, k)


@pytest.mark.parametrize("T", [130, 300, 1111])
@pytest.mark.parametrize("H,I", [(768, 384), (512, 256)])
def test_skew_and_identity(H, I, T):
    counts = _same(T, H, I, 62, 6, pairs=1, hot=(0, 7, 61, 62))
    assert int(counts[0]) == T and int(counts[62]) == T
    counts = _same(T, H, I, 30, 2, pairs=1, hot=(30, 31))
    assert int(counts[:30].sum()) == 0


def test_nothing_but_identity_after_a_full_call():
    """The scratch memory of a call with rows must not pass for a permutation of one without."""
    _same(300, 768, 384, 62, 6)
    _same(300, 768, 384, 62, 2, pairs=1, hot=(62, 63))


@pytest.mark.parametrize("T,k,E", [(1, 1, 5), (100, 8, 64), (513, 8, 64), (1024, 8, 64), (1025, 8, 64), (1111, 2, 9), (2730, 6, 64),
                                   (2731, 6, 64)])
@pytest.mark.parametrize("H,I", [(128, 128), (256, 256), (768, 384)])
def test_training_state(H, I, T, k, E):
    """The state that a training forward leaves serves the backward pass as a permutation does (moe_backward makes its own)."""
    g = torch.Generator().manual_seed(T + I)
    x, d_out = (torch.randn(T, H, generator=g).bfloat16().to(DEV) for _ in range(2))
    wr = (torch.randn(E, H, generator=g) * 0.1).bfloat16().to(DEV)
    bias = (torch.rand(E, generator=g) * 0.02 - 0.01).to(DEV)
    gu = (torch.randn(E, 2 * I, H, generator=g) * 0.05).bfloat16().to(DEV)
    dn = (torch.randn(E, H, I, generator=g) * 0.05).bfloat16().to(DEV)
    th = torch.randn(E, generator=g).to(DEV)
    _, idx, _, _, _ = ops.moe_forward(x, wr, bias, gu, dn, th, k, want_routing=True)
    out, counts, state = ops.moe_forward_train(x, wr, bias, gu, dn, th, k, want_counts=True)
    assert torch.equal(torch.bincount(idx.flatten().long(), minlength=E).int(), counts)
    assert torch.equal(out, ops.moe_forward(x, wr, bias, gu, dn, th, k, algo="fused")[0])
    saved = ops.moe_backward_saved(x, d_out, wr, gu, dn, th, k, state, want_dw=True)
    again = ops.moe_backward(x, d_out, wr, bias, gu, dn, th, k, want_dw=True)
    for a, b in zip(saved, again):
        assert torch.equal(a, b)
