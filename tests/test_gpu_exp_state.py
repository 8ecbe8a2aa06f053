"""The 10-layer forward keeps nothing between calls: parameters written through `.data`, another sequence length, inference
mode, autocast and graph replays all see the values of their own call; vectors in bf16 give the bits of their fp32 copies."""
import pytest
import torch

from bibo_amd import _lib as L
from bibo_amd import exp_model as X
from test_exp_model import randomize

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _model(seed=0):
    cfg = X.BiBoExpConfig(vocab_size=97, hidden_size=256, num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2,
                          intermediate_size=256, moe_intermediate_size=128, num_routed_experts=8, num_experts_per_tok=2,
                          sliding_window=16, mlp_only_layers=(0, 3))
    model = randomize(X.BiBoExpForCausalLM(cfg), seed).to(DEV, torch.bfloat16).eval()
    return model


def _ids(B, S, seed):
    return torch.randint(0, 97, (B, S), generator=torch.Generator().manual_seed(seed)).to(DEV)


@torch.no_grad()
def test_writes_through_data_are_seen():
    model, ids = _model(), _ids(2, 40, 1)
    before = model(ids)
    new = _model(seed=5)
    for p, q in zip(model.parameters(), new.parameters()):
        p.data.copy_(q)
    for m in model.modules():                       # what the layers keep in kernel dtype, and row norms, are told of it
        if hasattr(m, "refresh_weights"):
            m.refresh_weights()
        if isinstance(m, X.RMSNorm):
            m.__dict__.pop("_fp32_weight", None)
    after = model(ids)
    assert not torch.equal(before, after) and torch.equal(after, new(ids))


def test_inference_mode_sequence_lengths_and_autocast():
    model = _model()
    want = {}
    with torch.no_grad():
        for S in (40, 17):
            want[S] = model(_ids(2, S, S))
    with torch.inference_mode():
        for S in (40, 17, 40):
            assert torch.equal(model(_ids(2, S, S)), want[S])
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(model(_ids(2, 40, 40)), want[40])


@torch.no_grad()
def test_replays_after_calls_of_another_length():
    model, ids, other = _model(), _ids(2, 40, 1), _ids(1, 65, 2)
    side = torch.cuda.Stream(device=DEV)
    side.wait_stream(torch.cuda.current_stream(DEV))
    with torch.cuda.stream(side):
        model(ids)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = model(ids)
    for seed in (3, 4, 3):
        ids.copy_(_ids(2, 40, seed))
        model(other)                                # tables of another length in between
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, model(ids))


@torch.no_grad()
@pytest.mark.parametrize("name", ["self_attn.q_proj", "self_attn.o_proj", "self_attn.k_norm", "input_layernorm", "mlp.up_proj"])
@pytest.mark.parametrize("how", ["forward", "subclass", "hook"])
def test_replaced_and_observed_modules_are_called(name, how):
    model, ids, seen = _model(), _ids(2, 20, 1), []
    layer = model.model.layers[3 if "mlp" in name else 1]
    module = layer.get_submodule(name)
    model(ids)
    if how == "forward":
        plain = module.forward
        module.forward = lambda x: seen.append(1) or plain(x)
    elif how == "subclass":
        base = type(module)
        module.__class__ = type("Wrapped", (base,), {"forward": lambda self, x: seen.append(1) or base.forward(self, x)})
    else:
        module.register_forward_hook(lambda *a: seen.append(1))
    model(ids)
    assert seen == [1]


@torch.no_grad()
@pytest.mark.parametrize("cls,method", [(X.RMSNorm, "forward"), (X.RMSNorm, "__call__"), (torch.nn.Linear, "forward"), (X.BiBoExpMLP, "forward")])
def test_methods_replaced_on_the_class_are_called(cls, method, monkeypatch):
    model, ids, seen = _model(), _ids(2, 20, 1), set()
    want = model(ids)
    plain = getattr(cls, method)
    monkeypatch.setattr(cls, method, lambda self, x: seen.add(self) or plain(self, x))
    got = model(ids)
    layers, dense = model.model.layers, [l for l in model.model.layers if not l.is_moe_layer]
    if cls is X.RMSNorm:
        expected = {model.model.norm, *(l.post_attention_layernorm for l in dense)}
        for l in layers:
            expected |= {l.input_layernorm, l.self_attn.q_norm, l.self_attn.k_norm}
    elif cls is torch.nn.Linear:
        expected = {model.lm_head, *(m for l in layers for m in (l.self_attn.q_proj, l.self_attn.k_proj, l.self_attn.v_proj, l.self_attn.o_proj)),
                    *(m for l in dense for m in (l.mlp.gate_proj, l.mlp.up_proj, l.mlp.down_proj))}
    else:
        expected = {l.mlp for l in dense}
    assert expected <= seen
    monkeypatch.undo()
    assert torch.equal(model(ids), want)
    for m in model.modules():                        # observed modules run by themselves too: the same route, the same bits
        if type(m) is cls:
            m.register_forward_hook(lambda *a: None)
    assert torch.equal(model(ids), got)


@torch.no_grad()
@pytest.mark.parametrize("H,S", [(256, 33), (768, 5)])
def test_bf16_vectors_give_the_bits_of_their_fp32_copies(H, S):
    g = torch.Generator().manual_seed(H + S)
    r = lambda *s: torch.randn(*s, generator=g).to(DEV, torch.bfloat16)
    nat, d, nh, nkv = L.native(), H // 4, 4, 2
    cands, a, b, w = [r(1, S, H) for _ in range(3)], r(H), r(1, H), r(H)
    odd = r(H + 1)[1:]                              # a view no 16-byte load may read
    full = lambda t: None if t is None else t.float()
    for x, y, z in ((a, b, w), (a, None, w), (odd, b, w), (a, b, None)):
        for got, ref in zip(nat.exp_attn_res_norm(cands, x, y, 1e-6, z, 1e-6),
                            nat.exp_attn_res_norm(cands, full(x), full(y), 1e-6, full(z), 1e-6)):
            assert got is ref or torch.equal(got, ref)
    product = (a.float() * b.float().view(-1)).contiguous()
    assert torch.equal(nat.exp_attn_res_norm(cands, a, b, 1e-6, None, 0.0)[0], nat.exp_attn_res_norm(cands, product, None, 1e-6, None, 0.0)[0])
    for th in (a, odd):
        assert all(torch.equal(p, q) for p, q in zip(nat.exp_carry(cands[0], cands[1], th, cands[2]),
                                                     nat.exp_carry(cands[0], cands[1], th.float(), cands[2])))
    x, wq, wk, wv, wo = r(2, S, H), r(nh * d, H), r(nkv * d, H), r(nkv * d, H), r(H, nh * d)
    qw, kw, alpha = r(d), r(d), r(nh)
    cos, sin = r(S, d), r(S, d)
    vecs = (qw, kw, 1e-6, cos, sin, alpha)
    one = nat.exp_attention(x, wq, wk, wv, wo, *vecs, nh, nkv, d, 0, d ** -0.5)
    two = nat.exp_attention(x, wq, wk, wv, wo, *(v.float() if torch.is_tensor(v) else v for v in vecs), nh, nkv, d, 0, d ** -0.5)
    assert torch.equal(one, two)


@torch.no_grad()
def test_weights_lie_in_one_block_until_one_is_replaced():
    import copy
    model, ids = _model(), _ids(2, 20, 1)
    attn, mlp = model.model.layers[1].self_attn, model.model.layers[3].mlp
    for group in ((attn.q_proj, attn.k_proj, attn.v_proj), (mlp.gate_proj, mlp.up_proj)):
        assert len({m.weight.untyped_storage().data_ptr() for m in group}) == 1
    want = model(ids)
    assert torch.equal(copy.deepcopy(model)(ids), want)                            # copies lie apart
    other = _model(seed=3)
    other.load_state_dict(model.state_dict())
    for m in other.modules():
        m.__dict__.pop("_fp32_weight", None)
    assert torch.equal(other(ids), want)
    for m in (attn.k_proj, mlp.up_proj):
        m.weight = torch.nn.Parameter(m.weight.clone())
    assert torch.equal(model(ids), want)
    attn.v_proj.weight.data.mul_(2.0)                # (a factor on q would vanish in its norm)
    assert not torch.equal(model(ids), want)
    attn.v_proj.weight.data.mul_(0.5)
    assert torch.equal(model.float().to(torch.bfloat16)(ids), want)


@torch.no_grad()
def test_weights_changed_before_a_capture_are_seen_outside_it():
    """Copies in kernel dtype that a captured call makes are the graph's; a call outside makes its own."""
    model, ids, new = _model(), _ids(2, 20, 1), _model(seed=5)
    want = new(ids)
    side = torch.cuda.Stream(device=DEV)
    side.wait_stream(torch.cuda.current_stream(DEV))
    with torch.cuda.stream(side):
        model(ids)
        for p, q in zip(model.parameters(), new.parameters()):
            p.copy_(q)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = model(ids)
    assert torch.equal(model(ids), want)             # before any replay
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(model(ids), want)


@torch.no_grad()
@pytest.mark.parametrize("source", ["built", "assigned", "flat"])
def test_a_move_that_moves_nothing_leaves_the_weights_where_they_are(source):
    model, ids = _model(), _ids(2, 20, 1)
    want = model(ids)
    tensors = {n: p.detach().clone() for n, p in model.named_parameters()}
    if source == "built":                            # on the device and in the type of every later move
        for m in model.modules():
            if isinstance(m, torch.nn.Linear):
                m.weight = torch.nn.Parameter(m.weight.clone())
    elif source == "assigned":
        model.load_state_dict(tensors, strict=False, assign=True)
    else:                                            # views of a flat buffer with gaps between them
        flat = torch.zeros(sum(t.numel() + 128 for t in tensors.values()), dtype=torch.bfloat16, device=DEV)
        at = 0
        for n, p in model.named_parameters():
            p.data = flat[at:at + p.numel()].view_as(p).copy_(tensors[n])
            tensors[n] = p.data
            at += (p.numel() + 127) // 64 * 64
    where = {n: p.data_ptr() for n, p in model.named_parameters()}
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream(device=DEV)
    side.wait_stream(torch.cuda.current_stream(DEV))
    with torch.cuda.stream(side):
        model(ids)
    side.synchronize()
    with torch.cuda.graph(graph, stream=side):
        out = model(ids)
    for move in (lambda: model.cuda(), lambda: model.to(DEV), lambda: model.to(torch.bfloat16), lambda: model.bfloat16()):
        move()
        assert {n: p.data_ptr() for n, p in model.named_parameters()} == where
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(model(ids), want)
    if source != "built":                            # a write through the other name of a weight is seen
        tensors["model.layers.1.self_attn.v_proj.weight"].mul_(2.0)
        changed = model(ids)
        graph.replay()
        torch.cuda.synchronize()
        assert not torch.equal(changed, want) and torch.equal(out, changed)


@pytest.mark.parametrize("S,half,dtype", [(1, 32, torch.float32), (77, 96, torch.float32), (2048, 64, torch.bfloat16)])
def test_rope_tables_give_the_bits_of_the_tensor_operations(S, half, dtype):
    inv = (10000.0 ** (-torch.arange(0, half, dtype=torch.float32) / half)).to(DEV, dtype)
    ang = torch.arange(S, device=DEV, dtype=torch.float32)[:, None] * inv.float()[None, :]
    ang = torch.cat((ang, ang), -1)
    cos, sin = L.native().exp_rope_tables(inv, S)
    assert torch.equal(cos, ang.cos().bfloat16()) and torch.equal(sin, ang.sin().bfloat16())


@torch.no_grad()
@pytest.mark.parametrize("T,H", [(5, 256), (40, 96), (70, 2304)])
def test_seam_reads_a_bf16_norm_weight_in_place(T, H):
    import bibo_amd
    cfg = bibo_amd.BiBoMoEConfig(hidden_size=H, moe_intermediate_size=32, num_routed_experts=8, num_experts_per_tok=2, special_expert_pairs=0)
    with torch.device(DEV):
        layer = bibo_amd.BiBoMoELayer(cfg).to(torch.bfloat16).eval()
    g = torch.Generator().manual_seed(T)
    h = torch.randn(1, T, H, generator=g).to(DEV, torch.bfloat16)
    w = torch.randn(H + 1, generator=g).to(DEV, torch.bfloat16)
    for nw in (w[:H], w[1:]):                       # the second on no 16-byte boundary
        assert torch.equal(layer.ffn_forward(h, nw, 1e-6), layer.ffn_forward(h, nw.float(), 1e-6))
