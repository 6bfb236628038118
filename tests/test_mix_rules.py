"""Which layers too large for the fp32 kernels of channel mixing leave the library's products (host side)."""
import pytest
import torch


@pytest.mark.parametrize("kind,l,c,n,widened,fits", [
    ("so2", 6, 64, 16000, False, True), ("so2", 6, 64, 4000, True, True), ("so2", 6, 256, 4000, False, True), ("so2", 6, 256, 4000, True, False),
    ("so2", 6, 288, 100, False, False),                   # 108 units in a row
    ("lin", 4, 128, 1000, False, True), ("lin", 4, 128, 1000, True, False), ("lin", 4, 128, 16000, False, False), ("lin", 4, 320, 50, False, False),
    ("copies", 4, 64, 100, False, True), ("copies", 5, 64, 100, False, False)])
def test_by_rows_work_and_type(kind, l, c, n, widened, fits):
    from test_uv_mix import _module

    from equitorch_amd.nn.functional import _irreps_gemm as G
    from equitorch_amd.nn.functional import _uv_native as N
    mod = _module(kind, l, 4, 4, "cpu")
    if kind == "so2":
        plan = G.plan_of_product_info(mod.info_forward, mod.irreps_in.dim, mod.num_weights)
    else:
        plan = G.plan_of_linear_info(mod.forward_info)
    from test_uv_mix import _table
    table = _table([(p.o0 + j, p.i0 + j, p.w, p.scale) for p in plan.paths for j in range(p.k)], mod.irreps_in.dim, plan.out_size, plan.n_paths)
    x, w = torch.empty(1).expand(n, mod.irreps_in.dim, c), torch.empty(1).expand(plan.n_paths, c, c)
    if x.data_ptr() % 16:
        pytest.skip("the allocation is not on a 16-byte boundary")
    assert N.mix_fits(x, w, table, kind == "so2", widened) == fits
