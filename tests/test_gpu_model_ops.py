"""The decoder layer's operations around the attention (csrc/model_ops.hip): rotations, the SiLU
gate and the slots against the torch expressions they stand for, bit for bit; the weight
products of few tokens against float64 within their roundings."""
import pytest
import torch
import torch.nn.functional as F

from starkv_serve.kernels import model_ops as mo
from starkv_serve.kernels.stock_decode import write_kv_full

pytestmark = pytest.mark.gpu


def _rotated(positions, x, table):
    cos, sin = table[positions].float().chunk(2, dim=-1)
    cos, sin = cos[:, None, :], sin[:, None, :]
    x1, x2 = x.float().chunk(2, dim=-1)
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1).to(x.dtype)


@pytest.mark.parametrize("T,H,Hkv,dt,tdt,pdt", [(1, 32, 32, torch.bfloat16, torch.bfloat16, torch.int64),
                                               (37, 6, 2, torch.float16, torch.float32, torch.int32),
                                               (300, 8, 1, torch.bfloat16, torch.float16, torch.int64),
                                               (5, 3, 3, torch.float32, torch.float32, torch.int64)])
def test_rope_write(cuda, T, H, Hkv, dt, tdt, pdt):
    g = torch.Generator().manual_seed(T)
    qkv = torch.randn(T, (H + 2 * Hkv) * 128, generator=g).to(dt).to(cuda)
    q, k, v = (t.view(T, -1, 128) for t in qkv.split([H * 128, Hkv * 128, Hkv * 128], dim=-1))
    table = torch.randn(50, 128, generator=g).clamp(-1, 1).to(tdt).to(cuda)
    pos = torch.randint(-3, 50, (T,), generator=g).to(pdt).to(cuda)
    nb = (T + 15) // 16 + 1
    slots = torch.randperm(nb * 16, generator=g)[:T].to(cuda)
    if T > 4:
        slots[2], slots[3] = -1, nb * 16 + 5  # neither is written
    kc, vc = (torch.randn(nb, 16, Hkv, 128, generator=g).to(dt).to(cuda) for _ in range(2))
    kw, vw = kc.clone(), vc.clone()
    assert mo.rope_fits(table, pos, q, k, v)
    qo, ko, k16, v16 = mo.rope_write(pos, q, k, v, table, kc, vc, slots, True, True)
    qw, kr = _rotated(pos.long(), q, table), _rotated(pos.long(), k, table)
    assert torch.equal(qo, qw) and torch.equal(ko, kr) and torch.equal(mo.rope(pos, q, table), qw)
    assert torch.equal(k16, kr.to(torch.float16)) and torch.equal(v16, v.to(torch.float16))
    if dt != torch.float32:
        write_kv_full(kr, v, kw, vw, slots)
        assert torch.equal(kc, kw) and torch.equal(vc, vw)


@pytest.mark.parametrize("T,width,dt", [(1, 8, torch.bfloat16), (5, 11008, torch.bfloat16), (3, 2056, torch.float16)])
def test_silu_mul(cuda, T, width, dt):
    g = torch.Generator().manual_seed(width)
    x = (torch.randn(T, 2 * width, generator=g) * 8).to(dt)
    x[0, :8] = torch.tensor([0.0, -0.0, 80.0, -80.0, 2.0 ** -20, float("inf"), -100.0, 1.0])
    x = x.to(cuda)
    a, b = x.chunk(2, dim=-1)
    assert torch.equal(mo.silu_mul(x), F.silu(a) * b)


@pytest.mark.parametrize("n,bs,dt", [(1, 16, torch.int32), (300, 32, torch.int64)])
def test_decode_slots(cuda, n, bs, dt):
    g = torch.Generator().manual_seed(n)
    bt = torch.randint(0, 1000, (n, 14), generator=g).to(dt).to(cuda)[:, ::2]
    pos = torch.randint(0, 7 * bs, (n,), generator=g).to(cuda)
    slots, lens = mo.decode_slots(bt, pos, bs)
    rows = torch.arange(n, device=cuda)
    assert torch.equal(slots, bt[rows, pos // bs].long() * bs + pos % bs) and torch.equal(lens, (pos + 1).int())


@pytest.mark.parametrize("n,width,dt", [(1, 32000, torch.bfloat16), (3, 7, torch.float32), (70, 8200, torch.float16)])
def test_greedy_step(cuda, n, width, dt):
    """Equal maxima (coarse values), rows of -inf, a NaN: the first largest, as argmax."""
    g = torch.Generator().manual_seed(width)
    buf = torch.randn(n, (width + 7) // 8 * 8, generator=g).mul_(2).round().to(dt)
    x = buf[:, :width]
    x[-1] = float("-inf")
    if n > 2:
        x[1, width // 2:] = float("nan")
        x[0, -1] = 50.0
    x = buf.to(cuda)[:, :width]
    tokens, pos = torch.full((n,), -5, device=cuda), torch.arange(n, device=cuda)
    mo.greedy_step(x, tokens, pos)
    assert tokens.tolist() == [int(r.argmax()) for r in x.float().cpu()]
    assert torch.equal(pos, torch.arange(n, device=cuda) + 1)


@pytest.mark.parametrize("n,N,K,dt", [(1, 4096, 4096, torch.bfloat16), (8, 40, 11008, torch.bfloat16),
                                     (16, 16, 32, torch.bfloat16), (3, 1, 96, torch.bfloat16),
                                     (5, 72, 544, torch.float16), (2, 4096, 288, torch.float16), (4, 16402, 64, torch.bfloat16), (2, 16384, 32, torch.float16)])
def test_few_linear(cuda, n, N, K, dt):
    """Roundings, with u the largest relative rounding of the dtype (8 and 11 significant bits): the operand x times
    the norm's weight (once), the fp32 sums (K + 16 operations of 2^-24) and the result (once)."""
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(n, K, generator=g).to(dt).to(cuda)
    w = (torch.randn(2 * N, K, generator=g) * K ** -0.5).to(dt).to(cuda)
    nw = (1 + 0.2 * torch.randn(K, generator=g)).to(dt).to(cuda)
    res = torch.randn(n, N, generator=g).to(dt).to(cuda)
    u = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11

    def check(got, want, err):
        assert got.shape == want.shape and ((got.double() - want).abs() <= want.abs() * u + err * (1 + u) + 2.0 ** -24).all()

    X, W = x.double(), w.double()
    mag = X.abs() @ W.abs().T * (K + 16) * 2.0 ** -24
    check(mo.few_linear(x, w[:N]), X @ W[:N].T, mag[:, :N])
    check(mo.few_linear(x, w[:N], residual=res), res.double() + X @ W[:N].T, mag[:, :N] + (res.double().abs() + 1) * 2.0 ** -22)
    if dt != torch.bfloat16:
        with pytest.raises(RuntimeError, match="norm"):
            mo.few_linear(x, w, nw, 1e-5)
        return
    h = X * torch.rsqrt(X.square().mean(-1, keepdim=True) + 1e-5) * nw.double()
    err = h.abs() @ W.abs().T * (u + (2 * K + 32) * 2.0 ** -24)
    h_out = torch.empty_like(x)
    y = h @ W.T
    check(mo.few_linear(x, w, nw, 1e-5, h_out), y, err)
    check(h_out, h, h.abs() * (K + 16) * 2.0 ** -24)
    a, b = y[:, :N], y[:, N:]
    s = F.silu(a)
    check(mo.few_linear(x, w, nw, 1e-5, gate=True), s * b,
          1.1 * err[:, :N] * (b.abs() + err[:, N:]) + s.abs() * err[:, N:] + (s * b).abs() * 2.0 ** -20)


def test_rotary_under_transforms(cuda):
    """vmap, jvp, dual tensors and gradients through Rotary.apply take torch's operations: the plain
    call's values, and the rotation of the tangent (it is linear in x)."""
    from starkv_serve.model import Rotary
    g = torch.Generator().manual_seed(3)
    rot = Rotary(50, torch.float32, cuda, 10000.0)
    pos = torch.tensor([0, 49, 7], device=cuda)
    x, dx = (torch.randn(2, 3, 4, 128, generator=g).to(cuda) for _ in range(2))
    want, dwant = ([rot.apply(pos, t[i]) for i in range(2)] for t in (x, dx))
    near = lambda a, b: torch.testing.assert_close(a, b, rtol=0, atol=8 * 8 * 2 ** -24)  # |x| < 8, up to 8 fp32 roundings
    near(torch.vmap(lambda t: rot.apply(pos, t))(x), torch.stack(want))
    out, tan = torch.func.jvp(lambda t: rot.apply(pos, t), (x[0],), (dx[0],))
    near(out, want[0])
    near(tan, dwant[0])
    with torch.autograd.forward_ad.dual_level():
        dual = rot.apply(pos, torch.autograd.forward_ad.make_dual(x[0], dx[0]))
        near(torch.autograd.forward_ad.unpack_dual(dual).tangent, dwant[0])
    leaf = x[0].clone().requires_grad_()
    (rot.apply(pos, leaf) * want[0]).sum().backward()  # the rotation's transpose undoes it
    near(leaf.grad, x[0])


def test_rotary_and_slots_compile_and_trace(cuda):
    """torch.compile (one graph), jit.trace and make_fx of Rotary.apply and torch.compile of decode_metadata see torch's
    operations only, and give the plain calls' values."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from starkv_serve.model import Rotary, decode_metadata
    g = torch.Generator().manual_seed(3)
    rot = Rotary(50, torch.float32, cuda, 10000.0)
    pos = torch.tensor([0, 49, 7], device=cuda)
    x = torch.randn(3, 4, 128, generator=g).to(cuda)
    want = rot.apply(pos, x)
    near = lambda a, b: torch.testing.assert_close(a, b, rtol=0, atol=8 * 8 * 2 ** -24)  # as above
    near(torch.compile(rot.apply, fullgraph=True, backend="eager")(pos, x), want)
    traced = torch.jit.trace(rot.apply, (pos, x), check_trace=False)
    assert "starkv::" not in str(traced.graph)
    near(traced(pos[:2], x[:2]), want[:2])
    bt = torch.arange(12, dtype=torch.int32, device=cuda).view(3, 4)
    graph = make_fx(lambda p, t: rot.apply(p, t))(pos, x)
    assert "starkv." not in graph.code
    near(graph(pos, x), want)
    md, got = (f(bt, pos, 16, 64) for f in (decode_metadata, torch.compile(decode_metadata, fullgraph=True,
                                                                          backend="eager")))
    assert torch.equal(md.slot_mapping, got.slot_mapping) and torch.equal(md.seq_lens, got.seq_lens)
