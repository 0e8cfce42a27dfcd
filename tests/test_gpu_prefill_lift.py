"""The prompt lift kernel (starkv_prefill_lift) against float64: K = RoPE(codes @ U) rounded
once to fp16 and the V codes in fp16 rows.

Bound per value: the fp16 rounding (2^-11 of it, 2^-25 below fp16's normal range) plus the
fp32 sum of at most 2 R products and the rotation's, each within 2^-24 of the sum of their
magnitudes (2 R + 4 operations). V rows equal torch's
conversion."""
import pytest
import torch

from starkv_serve.kernels.prefill import prefill_lift, prompt_tables

pytestmark = pytest.mark.gpu

CASES = {
    # name: (prompt lengths, head widths, v_rank, codes dtype, cos/sin dtype)
    "one_token": ([1], [16], 1, torch.bfloat16, torch.bfloat16),
    "tile_edges": ([31, 33, 0, 32], [16, 48, 128, 32, 16, 16, 32, 64, 16], 37, torch.bfloat16, torch.bfloat16),
    "empty_ends": ([0, 70, 0], [32, 16, 48], 64, torch.bfloat16, torch.float32),
    "odd_row": ([5, 100], [16] * 17, 1291, torch.bfloat16, torch.float16),
    "fp16_codes": ([65, 2], [32, 128, 16, 16, 64], 40, torch.float16, torch.float16),
    "fp32_codes": ([33, 4], [32, 80, 16], 11, torch.float32, torch.float32),
    "odd_widths": ([40], [17, 1, 50], 9, torch.bfloat16, torch.bfloat16),
}


@pytest.mark.parametrize("name", list(CASES))
def test_lift_vs_float64(cuda, name):
    lens, widths, rv, dt, cdt = CASES[name]
    g = torch.Generator().manual_seed(len(name))
    T, W, H = sum(lens), sum(widths), len(widths)
    offs = [sum(widths[:h]) for h in range(H)]
    codes = torch.randn(T, W + rv + 1, generator=g).to(dt).to(cuda)
    k_codes, v_codes = codes[:, :W], codes[:, W:W + rv]
    u = (torch.randn(W, 128, generator=g) * 0.2).to(cuda)
    ang = torch.arange(max(lens) + 3, dtype=torch.float64)[:, None] * torch.logspace(0, -4, 64, dtype=torch.float64)
    cs = torch.cat([ang.cos(), ang.sin()], 1).to(cdt).to(cuda)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda)  # noqa: E731
    key, v16 = prefill_lift(k_codes, v_codes, prompt_tables(lens, cuda)[0], u, i32(offs), i32(widths), cs)
    torch.cuda.synchronize()
    c, s = cs[torch.cat([torch.arange(L) for L in lens]).to(cuda)].double().chunk(2, 1)
    for h in range(H):
        a = codes[:, offs[h]:offs[h] + widths[h]].double()
        b = u[offs[h]:offs[h] + widths[h]].double()
        x1, x2 = (a @ b).chunk(2, 1)
        m1, m2 = (a.abs() @ b.abs()).chunk(2, 1)
        want = torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], 1)
        mag = torch.cat([m1 * c.abs() + m2 * s.abs(), m2 * c.abs() + m1 * s.abs()], 1)
        bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + (2 * widths[h] + 4) * 2.0 ** -24 * mag
        assert ((key[:, h].double() - want).abs() <= bound).all(), f"{name}: head {h}"
    assert torch.equal(v16, v_codes.to(torch.float16))
    if dt == torch.float16:
        assert v16.data_ptr() == v_codes.data_ptr()


@pytest.mark.parametrize("name", list(CASES))
def test_lift_bit_for_bit(cuda, name):
    """The keys' bits: per value one fp32 chain of fused multiply-adds over the ranks, by eights in the order
    0 2 4 6 1 3 5 7, the rotation's products and sums rounded one by one, one rounding to fp16. (A fused
    multiply-add is formed here in float64, which holds the product, and rounded once.)"""
    lens, widths, rv, dt, cdt = CASES[name]
    g = torch.Generator().manual_seed(100 + len(name))
    T, W, H = sum(lens), sum(widths), len(widths)
    offs = [sum(widths[:h]) for h in range(H)]
    codes = torch.randn(T, W + rv, generator=g).to(dt)
    u = torch.randn(W, 128, generator=g) * 0.2
    ang = torch.arange(max(lens) + 3, dtype=torch.float64)[:, None] * torch.logspace(0, -4, 64, dtype=torch.float64)
    cs = torch.cat([ang.cos(), ang.sin()], 1).to(cdt)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda)  # noqa: E731
    dev = codes.to(cuda)
    key = prefill_lift(dev[:, :W], dev[:, W:], prompt_tables(lens, cuda)[0], u.to(cuda), i32(offs), i32(widths), cs.to(cuda))[0]
    c, s = cs[torch.cat([torch.arange(L) for L in lens])].float().chunk(2, 1)
    for h in range(H):
        x = torch.zeros(T, 128)
        for r0 in range(0, widths[h], 8):
            for r in (r0 + i for i in (0, 2, 4, 6, 1, 3, 5, 7)):
                if r < widths[h]:
                    x = (x.double() + codes[:, offs[h] + r, None].double() * u[offs[h] + r].double()).float()
        x1, x2 = x.chunk(2, 1)
        want = torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], 1).to(torch.float16)
        assert torch.equal(key[:, h].cpu().view(torch.int16), want.view(torch.int16)), f"{name}: head {h}"
