"""Channel mixing on the library's batched products (``_irreps_gemm``): the layouts they are handed."""
import pytest
import torch


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shared", [True, False])
def test_no_transposed_right_operand_in_16_bits(monkeypatch, dtype, shared):
    """The gradient of the input reads the weight transposed; the library's 16-bit products fault on such a view."""
    from equitorch_amd.nn import IrrepsLinear
    from equitorch_amd.nn.functional import _irreps_gemm as G
    plan = G.plan_of_linear_info(IrrepsLinear("0e+1o+2e", "2e+0e+1o+0e", 8, 12).forward_info)
    gen = torch.Generator().manual_seed(0)
    g = torch.randn(5, plan.out_size, 12, generator=gen)
    w = torch.randn(*(() if shared else (5,)), plan.n_paths, 8, 12, generator=gen)
    back, rows, product = G.transposed(plan, 9), [], torch.baddbmm

    def spy(inp, a, b, **kw):
        rows.append(b.is_contiguous())
        return product(inp, a, b, **kw)
    monkeypatch.setattr(torch, "baddbmm", spy)
    low = G._mix_raw(g.to(dtype), w.to(dtype), back, True)
    assert rows and all(rows)
    want = G._mix_raw(g.to(dtype).double(), w.to(dtype).double(), back, True)
    # 12 products summed in fp32 (or, path by path, rounded): four roundings of the result at most
    assert float((low.double() - want).norm()) <= 4 * torch.finfo(dtype).eps * float(want.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("n,c", [(40, 64), (1000, 256)])
def test_bf16_input_gradient(device, n, c):
    from equitorch_amd.nn import IrrepsLinear
    from equitorch_amd.nn.functional import _irreps_gemm as G
    plan = G.plan_of_linear_info(IrrepsLinear("0e+1o+2e", "2e+0e+1o+0e", 8, 12).forward_info)
    gen = torch.Generator().manual_seed(1)
    x, g, w = (torch.randn(*s, generator=gen).bfloat16() for s in ((n, 9, c), (n, plan.out_size, c), (plan.n_paths, c, c)))
    xd = x.to(device).requires_grad_(True)
    got, = torch.autograd.grad(G._Mix.apply(xd, w.to(device), plan, False, 9), [xd], g.to(device))
    want = G._mix_raw(g.double(), w.double(), G.transposed(plan, 9), True)
    assert float((got.double().cpu() - want).norm()) <= 4 * 2.0 ** -8 * float(want.norm())
