"""The weight gradient of the fully connected products in fp32 on the half-precision matrix cores (``cgtp_uvg_apply``): no less
precise than fp32 matrix instructions and of their range."""
import numpy as np
import pytest
import torch

from helpers import stable_seed

SH = {1: "0e+1o", 2: "0e+1o+2e", 3: "0e+1o+2e+3o"}


@pytest.mark.parametrize("cost,n_wgs", [([1.0], 64), ([1.3, 4.1, 0.2], 2), ([1.0] * 100, 64), ([7.0, 1.0, 9.5, 3.0], 64), ([2.0, 2.0], 1)])
def test_the_shares_are_dealt_once_and_evenly(cost, n_wgs):
    """Every share of every path to one workgroup, the costs equal to within one share of the dearest path."""
    from equitorch_amd.nn.functional._uv_native import _GradWWalk as W
    jobs = W.deal(cost, n_wgs)
    assert len(jobs) == n_wgs
    seen = [0] * len(cost)
    for mine in jobs:
        assert len({p for p, _ in mine}) == len(mine)          # a path's shares of a workgroup are one job
        for p, mask in mine:
            assert mask and not seen[p] & mask
            seen[p] |= mask
    assert all(s == 2 ** 64 - 1 for s in seen)
    load = [sum(cost[p] * bin(mask).count("1") for p, mask in mine) for mine in jobs]
    assert max(load) <= sum(cost) * 64 / n_wgs + 1.01 * max(cost)
    # a path's job of half its shares or more has one of any two steps in a row
    for mine in jobs:
        for p, mask in mine:
            if bin(mask).count("1") >= 32:
                assert all(mask >> b & 3 for b in range(63))


def test_the_tables_name_every_job_once():
    from equitorch_amd.nn import SO3Linear
    from equitorch_amd.nn.functional import _uv_native as N
    for l in SH:
        coo = N._coo(SO3Linear(SH[l], SH[l], SH[l], 4, 4, internal_weights=False, feature_mode="uv").tp_info_forward)
        walk = N._GradWWalk(coo, 64, "cpu")
        words = walk.words.numpy()
        jobs = words[:walk.at[1] // 4].reshape(-1, 4)
        job_ptr, slot_ptr = words[walk.at[1] // 4:walk.at[2] // 4], words[walk.at[2] // 4:]
        assert len(jobs) == walk.n_slots == job_ptr[-1] == slot_ptr[-1] and len(job_ptr) == 65 and len(slot_ptr) == coo.P + 1
        assert sorted(jobs[:, 1]) == list(range(walk.n_slots)) and (jobs[:, 2:] != 0).any(axis=1).all()
        for p, slot in jobs[:, :2]:
            assert slot_ptr[p] <= slot < slot_ptr[p + 1]
        assert (np.diff(slot_ptr) > 0).all()


@pytest.mark.parametrize("l", [1, 2, 3])
def test_the_workspace_does_not_grow_with_the_batch(l):
    """As many slots as the fp32 kernel has partial results, or eight ranges' where that is more."""
    from equitorch_amd.nn import SO3Linear
    from equitorch_amd.nn.functional import _uv_native as N
    coo = N._coo(SO3Linear(SH[l], SH[l], SH[l], 4, 4, internal_weights=False, feature_mode="uv").tp_info_forward)
    walk = N._GradWWalk(coo, 64, "cpu")
    for n in (2048, 8192, 32768, 1 << 17, 1 << 20, 1 << 26):
        ranges = walk.ranges(-(-n // 16))
        assert ranges % 8 == 0 and 8 <= ranges and ranges * walk.n_slots <= max(128 * coo.P, 8 * walk.n_slots)


# ---- on the GPU ------------------------------------------------------------------------------------------------------
def _operands(l, c, cy, n, seed):
    d, gen = (l + 1) ** 2, torch.Generator().manual_seed(seed)
    y = torch.randn(n, d, cy, generator=gen) if cy else torch.randn(n, d, generator=gen)
    return [torch.randn(n, d, c, generator=gen), y, torch.randn(n, d, c, generator=gen)]


def _routes(device, monkeypatch, l, ops):
    from equitorch_amd.nn import SO3Linear
    from equitorch_amd.nn.functional import _uv_native as N
    info = SO3Linear(SH[l], SH[l], SH[l], 4, 4, internal_weights=False, feature_mode="uv").to(device).tp_info_forward
    x, y, g = (t.to(device) for t in ops)
    new = N._split_grad_w(x, y, g, info)
    assert new is not None
    monkeypatch.setattr(N, "_split_grad_w", lambda *args: None)
    return new, N.grad_w(x, y, g, info), N.grad_w(x.double(), y.double(), g.double(), info)


SIZES = [(2, 128, 0, 2048), (2, 68, 0, 2500), (3, 128, 0, 5003), (3, 96, 0, 20001), (2, 100, 0, 17000), (2, 32, 32, 2049), (1, 24, 28, 8200),
         (2, 32, 24, 16400)]


@pytest.mark.gpu
@pytest.mark.parametrize("l,c,cy,n", SIZES)
@pytest.mark.parametrize("values", ["normal", "wide"])
def test_no_less_precise_than_fp32_matrix_instructions(device, monkeypatch, l, c, cy, n, values):
    """Ragged batches and channels; ``wide``: samples spread over twenty binary orders of magnitude, with exact zeros."""
    ops = _operands(l, c, cy, n, stable_seed("gw", l, c, cy, n))
    if values == "wide":
        gen = torch.Generator().manual_seed(3)
        for t in ops:
            t.mul_(torch.exp2(torch.randint(-10, 11, (n,) + (1,) * (t.ndim - 1), generator=gen).float()))
        ops[0][5:40] = 0.0
    new, old, ref = _routes(device, monkeypatch, l, ops)
    for p in range(ref.shape[0]):
        e_new, e_old = (float((t[p].double() - ref[p]).norm() / ref[p].norm()) for t in (new, old))
        print(f"lmax={l} c={c} cy={cy} n={n} {values} path {p}: split {e_new:.2e} fp32 {e_old:.2e}")
    e_new, e_old = (float((t.double() - ref).norm() / ref.norm()) for t in (new, old))
    print(f"all paths: split {e_new:.2e} fp32 {e_old:.2e}")
    # with samples of very different size a few of them make the result: the order they are added in decides
    assert e_new <= (1.1 if values == "normal" else 2.0) * e_old


@pytest.mark.gpu
@pytest.mark.parametrize("where", [0, 1, 2])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.39e38])
@pytest.mark.parametrize("cy", [0, 24])
def test_values_that_are_not_finite_stay_where_they_couple(device, monkeypatch, where, value, cy):
    ops = _operands(2, 24 if cy else 80, cy, 2100, 5)
    if value == 3.39e38:             # no bf16 is as large; with the other operands small no product overflows on either route
        ops = [t if k == where else t * 2.0 ** -8 for k, t in enumerate(ops)]
    ops[where].view(-1)[4321] = value
    new, old, _ = _routes(device, monkeypatch, 2, ops)
    fin = torch.isfinite(old)        # the fp32 kernel pads terms with zero coefficients: NaN where an infinity is left here
    assert torch.equal(fin, torch.isfinite(new)) and (fin.all() or value != 3.39e38)
    assert torch.equal(new[~fin & ~old.isnan()], old[~fin & ~old.isnan()])
    assert float((new[fin].double() - old[fin].double()).norm()) <= 2e-6 * float(old[fin].double().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("exponents", [(0, 0, 0), (-105, 0, 0), (-115, 0, 40), (0, -60, -60), (40, 0, 60), (-118, 20, 100), (70, 0, 30)])
@pytest.mark.parametrize("cy", [0, 24])
def test_the_range_of_operands_is_that_of_fp32(device, monkeypatch, exponents, cy):
    ops = [t * 2.0 ** e for t, e in zip(_operands(2, 24 if cy else 80, cy, 2100, 6), exponents)]
    new, old, ref = _routes(device, monkeypatch, 2, ops)
    assert torch.equal(torch.isfinite(new), torch.isfinite(old))
    if ref.abs().max() > 2.0 ** -110 and torch.isfinite(old).all():
        e_new, e_old = (float((t.double() - ref).norm() / ref.norm()) for t in (new, old))
        print(f"{exponents} cy={cy}: split {e_new:.2e} fp32 {e_old:.2e}")
        assert e_new <= 1.5 * e_old + 3e-8


@pytest.mark.gpu
@pytest.mark.parametrize("l,c,cy", [(2, 32, 32), (3, 96, 0)])
def test_a_large_batch_in_little_memory(device, monkeypatch, l, c, cy):
    from equitorch_amd.nn import SO3Linear
    from equitorch_amd.nn.functional import _uv_native as N
    info = SO3Linear(SH[l], SH[l], SH[l], 4, 4, internal_weights=False, feature_mode="uv").to(device).tp_info_forward
    x, y, g = (t.to(device) for t in _operands(l, c, cy, 150001, 11))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    new = N._split_grad_w(x, y, g, info)
    used = torch.cuda.max_memory_allocated() - before
    assert used <= 130 * new.numel() * 4 + (1 << 22)        # 128 partial results, the gradient, the tables
    monkeypatch.setattr(N, "_split_grad_w", lambda *args: None)
    old = N.grad_w(x, y, g, info)
    ref = N.grad_w(x.double(), y.double(), g.double(), info)
    e_new, e_old = (float((t.double() - ref).norm() / ref.norm()) for t in (new, old))
    print(f"lmax={l} c={c} cy={cy}: {used / 1e6:.0f} MB, split {e_new:.2e} fp32 {e_old:.2e}")
    assert e_new <= 1.1 * e_old


@pytest.mark.gpu
@pytest.mark.parametrize("cy", [0, 24])
@pytest.mark.parametrize("scaled", ["all", "some samples", "some channels"])
def test_products_that_only_vanish_in_one_order(device, monkeypatch, cy, scaled):
    """y and grad_out whose product is below the smallest number, next to an x that makes up for it: zero where grad_out is
    mixed with y first, and no small matter where y meets x first, as in the fp32 kernel."""
    ops = _operands(2, 24 if cy else 80, cy, 2100, 9)
    at = {"all": slice(None), "some samples": slice(700, 703), "some channels": (slice(None), slice(None), slice(3, 5))}[scaled]
    for t, e in zip(ops, (100, -80, -80)):
        if t.ndim == 3 or scaled != "some channels":
            t[at] *= 2.0 ** e
        else:
            t *= 2.0 ** e
    if scaled == "some samples":       # the others are zero: what the result is made of is theirs alone
        for t in ops:
            t[:700], t[703:] = 0.0, 0.0
    new, old, ref = _routes(device, monkeypatch, 2, ops)
    assert float(ref.abs().max()) > 2.0 ** -70
    for p in range(ref.shape[0]):
        e_new, e_old = (float((t[p].double() - ref[p]).norm() / ref[p].norm()) for t in (new, old))
        print(f"cy={cy} {scaled} path {p}: split {e_new:.2e} fp32 {e_old:.2e}")
        assert e_new <= 2.0 * e_old + 3e-8


@pytest.mark.gpu
@pytest.mark.parametrize("cy", [0, 32])
def test_recorded_in_a_graph(device, cy):
    from equitorch_amd.nn import SO3Linear
    from equitorch_amd.nn.functional import _uv_native as N
    info = SO3Linear(SH[2], SH[2], SH[2], 4, 4, internal_weights=False, feature_mode="uv").to(device).tp_info_forward
    x, y, g = (t.to(device) for t in _operands(2, 32 if cy else 96, cy, 2300, 7))
    N.grad_w(x, y, g, info)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        N.grad_w(x, y, g, info)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = N._split_grad_w(x, y, g, info)
    for replay in range(3):
        x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(replay)) * 2.0 ** (4 * replay))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, N.grad_w(x, y, g, info)), replay
