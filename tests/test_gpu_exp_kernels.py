"""The launches around the MoE block in the 10-layer forward, through the C ABI, against plain fp32 PyTorch on the CPU: QK-norm
and RoPE in place, causal / banded attention with XSA at the edges of its 32-key blocks and query blocks, the depth mix with
its norm, the carry sums and SwiGLU's product."""
import ctypes

import pytest
import torch

from bibo_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _call(name, *args):
    L.check(getattr(L.lib(), name)(*args, ctypes.c_void_p(torch.cuda.current_stream(DEV).cuda_stream)), name)
    torch.cuda.synchronize()


def _rel(a, ref):
    return float((a.float().cpu() - ref).abs().max() / ref.abs().max().clamp_min(1e-30))


@pytest.mark.parametrize("D,nq,nkv", [(64, 2, 2), (64, 4, 1), (128, 2, 1), (192, 4, 2)])
@pytest.mark.parametrize("S,window", [(1, 0), (31, 0), (33, 16), (64, 64), (65, 0), (129, 32), (200, 128), (300, 0), (390, 33)])
def test_attention(D, nq, nkv, S, window):
    B, ld = 2, (nq + 2 * nkv) * D + 8
    g = torch.Generator().manual_seed(S + D)
    qkv = torch.randn(B, S, ld, generator=g).bfloat16()
    qkv[0, S // 2, :nq * D] *= 30                                  # a row whose maximum jumps late
    qw, kw = torch.rand(D, generator=g) + 0.5, torch.rand(D, generator=g) + 0.5
    ang = torch.arange(S)[:, None] * (10000.0 ** (-torch.arange(0, D, 2) / D))[None]
    cos, sin = ang.cos(), ang.sin()
    alpha = torch.randn(nq, generator=g)
    scale = D ** -0.5
    d = qkv.to(DEV)
    dev = [t.to(DEV).contiguous() for t in (qw, kw, cos, sin, alpha)]
    _call("bibo_moe_exp_qk_norm_rope", _ptr(d), ld, B, S, nq, nkv, D, _ptr(dev[0]), _ptr(dev[1]), 1, ctypes.c_float(1e-6), _ptr(dev[2]), _ptr(dev[3]), 1, D // 2)
    x = qkv.float()

    def heads(lo, n):
        return x[..., lo * D:(lo + n) * D].reshape(B, S, n, D)

    def norm_rope(t, w):
        t = (t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6)).bfloat16().float() * w
        a, b = t[..., :D // 2], t[..., D // 2:]
        c, s = cos[None, :, None], sin[None, :, None]
        return torch.cat((a * c - b * s, b * c + a * s), -1)

    q, k, v = norm_rope(heads(0, nq), qw), norm_rope(heads(nq, nkv), kw), heads(nq + nkv, nkv)
    got = d.cpu().float()
    assert _rel(got[..., :nq * D].reshape(q.shape), q) <= 8e-3 and _rel(got[..., nq * D:(nq + nkv) * D].reshape(k.shape), k) <= 8e-3
    assert torch.equal(got[..., (nq + nkv) * D:], x[..., (nq + nkv) * D:])          # v and the padding stay as they are
    q, k = got[..., :nq * D].reshape(q.shape), got[..., nq * D:(nq + nkv) * D].reshape(k.shape)
    rep = nq // nkv
    kx, vx = k.repeat_interleave(rep, 2), v.repeat_interleave(rep, 2)
    i = torch.arange(S)
    allow = (i[None] <= i[:, None]) & ((i[:, None] - i[None] < window) if window else True)
    for xsa in (None, dev[4]):
        out = torch.full((B, S, nq * D), float("nan"), dtype=torch.bfloat16, device=DEV)
        _call("bibo_moe_exp_attention_fwd", _ptr(d), ld, B, S, nq, nkv, D, window, ctypes.c_float(scale), _ptr(xsa), 1, _ptr(out))
        y = torch.empty(B, S, nq, D)
        for h in range(nq):
            p = (q[:, :, h] @ k[:, :, h // rep].transpose(1, 2).contiguous() * scale).masked_fill(~allow, -torch.inf).softmax(-1)
            y[:, :, h] = p @ vx[:, :, h]
        if xsa is not None:
            vn = torch.nn.functional.normalize(vx, dim=-1)
            y = y - (y * vn).sum(-1, keepdim=True) * torch.tanh(alpha)[None, None, :, None] * vn
        assert _rel(out, y.reshape(B, S, nq * D)) <= 1e-2, (xsa is not None)


@pytest.mark.parametrize("B,S,nq,nkv,D,window,spread", [(1, 48, 4, 2, 192, 128, 1), (1, 700, 4, 2, 192, 128, 1), (1, 700, 4, 2, 192, 128, 3),
                                                        (2, 333, 4, 1, 64, 128, 1), (1, 257, 2, 2, 128, 64, 3)])
def test_banded_attention_is_as_exact_as_its_output_type(B, S, nq, nkv, D, window, spread):
    """The probabilities' 16 bits of mantissa do not show: the result is as far from float64 as the float64 result rounded to bf16
    is (2^-17 beside 2^-9, in quadrature: 1e-5 of it)."""
    g = torch.Generator().manual_seed(S)
    qkv = torch.randn(B, S, (nq + 2 * nkv) * D, generator=g)
    qkv[..., :nq * D] *= spread
    qkv = qkv.bfloat16()
    out = torch.empty(B, S, nq * D, dtype=torch.bfloat16, device=DEV)
    d = qkv.to(DEV)
    _call("bibo_moe_exp_attention_fwd", _ptr(d), qkv.shape[-1], B, S, nq, nkv, D, window, ctypes.c_float(D ** -0.5), None, 1, _ptr(out))
    q, k, v = (t.double().view(B, S, -1, D).transpose(1, 2) for t in qkv.split([nq * D, nkv * D, nkv * D], -1))
    i = torch.arange(S)
    allow = (i[None] <= i[:, None]) & (i[:, None] - i[None] < window)
    rep = nq // nkv
    p = (q @ k.repeat_interleave(rep, 1).transpose(-1, -2).contiguous() * D ** -0.5).masked_fill(~allow, -torch.inf).softmax(-1)
    ref = (p @ v.repeat_interleave(rep, 1)).transpose(1, 2).reshape(B, S, nq * D)
    assert float((out.cpu().double() - ref).norm()) <= 1.001 * float((ref.bfloat16().double() - ref).norm())


@pytest.mark.parametrize("D,nq,nkv", [(64, 2, 2), (128, 4, 2), (192, 4, 2)])
@pytest.mark.parametrize("S,window,many", [(1, 0, True), (33, 16, True), (97, 0, True), (200, 64, True), (97, 64, False)])
@pytest.mark.parametrize("normed,rope,bf16", [(True, True, True), (True, False, False), (False, True, False), (False, False, True)])
def test_attention_takes_the_queries_as_the_norm_kernel_does(D, nq, nkv, S, window, many, normed, rope, bf16):
    """One call and two leave the same bits: the queries' norm and rotation inside the attention add in the norm kernel's order.  Rows
    wider than their heads, tables wider than D / 2; from 3 << 20 elements of queries on the one call leaves the queries alone."""
    B = -(-(3 << 20) // (S * nq * D)) if many else 2
    ld, ldr = (nq + 2 * nkv) * D + 8, D
    g = torch.Generator(device=DEV).manual_seed(S + D)
    dt = torch.bfloat16 if bf16 else torch.float32
    rows = torch.randn(B * S, ld, generator=g, device=DEV).bfloat16()
    qw, kw = ((torch.rand(D, generator=g, device=DEV) + 0.5).to(dt) for _ in range(2)) if normed else (None, None)
    ang = torch.rand(S, ldr, generator=g, device=DEV) * 6
    cos, sin = (ang.cos().to(dt), ang.sin().to(dt)) if rope else (None, None)
    xsa = torch.randn(nq, generator=g, device=DEV)
    pp = lambda t: None if t is None else _ptr(t)
    code = 0 if bf16 else 1                                        # BIBO_DTYPE_BF16, BIBO_DTYPE_F32
    norm = (pp(qw), pp(kw), code, ctypes.c_float(1e-6), pp(cos), pp(sin), code, ldr)
    one, two = rows.clone(), rows.clone()
    out = [torch.empty(B * S, nq * D, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    _call("bibo_moe_exp_norm_attention_fwd", _ptr(one), ld, B, S, nq, nkv, D, *norm, window, ctypes.c_float(D ** -0.5), _ptr(xsa), 1, _ptr(out[0]))
    _call("bibo_moe_exp_qk_norm_rope", _ptr(two), ld, B, S, nq, nkv, D, *norm)
    _call("bibo_moe_exp_attention_fwd", _ptr(two), ld, B, S, nq, nkv, D, window, ctypes.c_float(D ** -0.5), _ptr(xsa), 1, _ptr(out[1]))
    assert torch.equal(out[0], out[1])
    assert torch.equal(one[:, :nq * D], (rows if many else two)[:, :nq * D]) and torch.equal(one[:, nq * D:], two[:, nq * D:])


@pytest.mark.parametrize("far", [1 << 26, (1 << 26) + 8])
@pytest.mark.parametrize("D,nq,nkv,S,window", [(64, 2, 1, 33, 0), (192, 2, 2, 31, 16)])
def test_attention_of_rows_far_apart(D, nq, nkv, S, window, far):
    """Rows so far apart that the last row of a 32-key block is just in reach of 32-bit offsets, and just out of it, leave the bits of packed rows."""
    w = (nq + 2 * nkv) * D
    packed = torch.randn(S, w, generator=torch.Generator(device=DEV).manual_seed(S), device=DEV).bfloat16()
    apart = torch.empty((S - 1) * far + w, dtype=torch.bfloat16, device=DEV)
    apart.as_strided((S, w), (far, 1)).copy_(packed)
    out = [torch.empty(S, nq * D, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for rows, ld, o in ((packed, w, out[0]), (apart, far, out[1])):
        _call("bibo_moe_exp_attention_fwd", _ptr(rows), ld, 1, S, nq, nkv, D, window, ctypes.c_float(D ** -0.5), None, 1, _ptr(o))
    assert torch.isfinite(out[0]).all() and torch.equal(*out)


def test_attention_refuses_what_it_does_not_take():
    args = lambda nq, nkv, D: (None, 4096, 1, 4, nq, nkv, D, 0, ctypes.c_float(1.0), None, 1, None, None)
    for nq, nkv, D in ((4, 2, 96), (3, 2, 64), (3, 1, 64), (4, 0, 64)):
        assert L.lib().bibo_moe_exp_attention_fwd(*args(nq, nkv, D)) == -6
    assert L.lib().bibo_moe_exp_attention_fwd(*args(4, 2, 64)) == -1


@pytest.mark.parametrize("T,H", [(1, 8), (3, 520), (7, 768), (65, 1024)])
def test_depth_mix_carry_and_swiglu(T, H):
    g = torch.Generator().manual_seed(T + H)
    rows = lambda: torch.randn(T, H, generator=g).bfloat16()
    sw, nw, theta = torch.randn(H, generator=g) * 0.1, torch.rand(H, generator=g) + 0.5, torch.rand(H, generator=g)
    for n in (1, 2, 5, 8):
        cands = [rows() for _ in range(n)]
        dc = [c.to(DEV) for c in cands]
        mixed, normed = L.native().exp_attn_res_norm(dc, sw.to(DEV), None, 1e-6, nw.to(DEV), 1e-6)
        v = torch.stack([c.float() for c in cands], 1)
        ref = (((v @ sw) * torch.rsqrt(v.pow(2).mean(-1) + 1e-6)).softmax(-1)[..., None] * v).sum(1)
        assert _rel(mixed, ref) <= 8e-3
        m = mixed.cpu().float()
        assert _rel(normed, (m * torch.rsqrt(m.pow(2).mean(-1, keepdim=True) + 1e-6)) * nw) <= 1.2e-2
        assert torch.equal(L.native().exp_attn_res_norm(dc, sw.to(DEV), None, 1e-6, None, 0.0)[0], mixed)
    r, a, p = rows(), rows(), rows()
    hs, prefix = L.native().exp_carry(r.to(DEV), a.to(DEV), theta.to(DEV), p.to(DEV))
    assert _rel(hs, r.float() + theta * a.float()) <= 8e-3 and torch.equal(prefix.cpu(), p + a)
    hs, prefix = L.native().exp_carry(r.to(DEV), a.to(DEV), None, None)
    assert torch.equal(hs.cpu(), r + a) and torch.equal(prefix.cpu(), a)
    gu = torch.randn(T, 2 * H, generator=g).bfloat16().to(DEV)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=DEV)
    _call("bibo_moe_exp_silu_mul_fwd", _ptr(gu), T, H, _ptr(out))
    f = gu.cpu().float()
    assert _rel(out, torch.nn.functional.silu(f[:, :H]) * f[:, H:]) <= 8e-3
