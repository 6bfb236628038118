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


def _mix(kind, irreps):
    from test_uv_mix import _table

    from equitorch_amd import nn as enn
    from equitorch_amd.nn.functional import _irreps_gemm as G
    from equitorch_amd.nn.functional import _uv_native as N
    if kind == "so2":
        mod = enn.SO2Linear(irreps, irreps, 4, 4, feature_mode="uv")
        plan = G.plan_of_product_info(mod.info_forward, mod.irreps_in.dim, mod.num_weights)
    else:
        mod = enn.IrrepsLinear(irreps, irreps, 4, 4)
        plan = G.plan_of_linear_info(mod.forward_info)
    return N._MixTable(_table([(p.o0 + j, p.i0 + j, p.w, p.scale) for p in plan.paths for j in range(p.k)], mod.irreps_in.dim, plan.out_size,
                              plan.n_paths).coo, False)


@pytest.mark.parametrize("kind,irreps,cin,cout,n,fp32", [
    ("so2", "0e+1o", 64, 64, 4096, True), ("so2", "0e+1o", 64, 64, 5000, False), ("so2", "0e+1o", 64, 68, 4096, False),
    ("so2", "0e+1o", 64, 32, 4096, False), ("so2", "0e+1o", 96, 32, 4096, True), ("so2", "0e+1o", 32, 64, 4096, False),
    ("so2", "0e+1o+2e", 64, 16, 4096, True), ("so2", "0e+1o+2e", 128, 16, 9999, True), ("so2", "0e+1o+2e", 128, 16, 10000, False),
    ("so2", "0e+1o+2e", 128, 20, 4096, False), ("so2", "0e+1o+2e+3o", 128, 16, 500, False),
    ("lin", "0e+0e", 128, 128, 500, True), ("lin", "0e+0e+0e", 128, 64, 500, False), ("lin", "0e+1o", 128, 64, 500, False),
    ("lin", "0e+1o", 256, 256, 2047, True), ("lin", "0e+1o", 256, 256, 2048, False)])
def test_small_results_of_two_rows_stay_on_the_fp32_kernels(kind, irreps, cin, cout, n, fp32):
    from equitorch_amd.nn.functional import _uv_native as N
    assert N._few_and_long(_mix(kind, irreps), n, cin, cout) == fp32


@pytest.mark.parametrize("n", [1, 500, 4097, 32768, 1 << 20])
@pytest.mark.parametrize("cin,cout,paths", [(64, 64, 3), (128, 128, 2), (128, 128, 16), (96, 68, 85), (64, 128, 4), (16, 100, 1)])
def test_the_weight_gradient_takes_no_more_memory(n, cin, cout, paths):
    """Partial results of the weight gradient: as many as the fp32 kernels have, twice as many with 64 channels on one side only."""
    import ctypes as C

    from equitorch_amd import _lib
    a = _lib.UvlGwArgs(4096, 4096, 4096, 4096, 4096, 4096, n, paths, 3, 16, 16, cin, cout)
    one_side = (cin > 64) != (cout > 64)
    most = 512 if max(cin, cout) <= 64 else 256 if one_side else 128
    size = _lib.lib.cgtp_uvl_grad_w_workspace_bytes(C.byref(a))
    assert 0 < size <= most * paths * cin * cout * 4
    if n >= 4097:
        assert size <= (2 if one_side else 1) * _lib.lib.cgtp_uvt_grad_w_workspace_bytes(n, paths, cin, cout, _lib.dtype_code(torch.float32))
