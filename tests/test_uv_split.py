"""The fully connected product of the compiled tables in fp32 on the half-precision matrix cores (``cgtp_uvs_apply``): every
operand carried as three bf16 parts, no less precise than fp32 matrix instructions and of their range."""
import pytest
import torch

from helpers import stable_seed
from oracle import ref_ops

pytestmark = pytest.mark.gpu
SH = {1: "0e+1o", 2: "0e+1o+2e", 3: "0e+1o+2e+3o"}


def _operands(device, lmax, cin, cout, n, seed):
    from equitorch_amd.nn import SO3Linear
    mod = SO3Linear(SH[lmax], SH[lmax], SH[lmax], cin, cout, internal_weights=False, feature_mode="uv").to(device)
    d = (lmax + 1) ** 2
    gen = torch.Generator().manual_seed(seed)
    return mod, [torch.randn(n, d, cin, generator=gen), torch.randn(n, d, generator=gen),
                 torch.randn(mod.num_paths, cin, cout, generator=gen) * (cin * mod.num_paths) ** -0.5,
                 torch.randn(n, d, cout, generator=gen)]


def _step(mod, device, x, y, w, ct):
    wrt = [t.to(device).requires_grad_(True) for t in (x, y, w)]
    out = mod(*wrt)
    return [t.detach() for t in (out, *torch.autograd.grad(out, wrt, ct.to(device)))]


def _both_routes(monkeypatch, mod, device, operands):
    """Results on both routes; the split one takes all three products but those with 128 contracted and 32 produced channels."""
    from equitorch_amd.nn.functional import _uv_native
    results, kinds, split = {}, [], _uv_native._split

    def spy(kind, *args):
        out = split(kind, *args)
        kinds.append((kind, out is not None))
        return out
    monkeypatch.setattr(_uv_native, "_split", spy)
    results["split"] = _step(mod, device, *operands)
    cin, cout = operands[2].shape[1:]
    assert sorted(kinds) == [(0, (cin, cout) != (128, 32)), (1, (cout, cin) != (128, 32)), (2, (cin, cout) != (128, 32))], kinds
    monkeypatch.setattr(_uv_native, "_split", lambda *args: None)
    results["fp32"] = _step(mod, device, *operands)
    return results["split"], results["fp32"]


@pytest.mark.parametrize("lmax,cin,cout,n", [(1, 32, 32, 1), (1, 128, 64, 17), (2, 64, 32, 33), (2, 128, 128, 300),
                                             (3, 32, 128, 47), (3, 64, 64, 1000), (3, 128, 128, 555)])
@pytest.mark.parametrize("values", ["normal", "wide"])
def test_no_less_precise_than_fp32_matrix_instructions(device, monkeypatch, lmax, cin, cout, n, values):
    """Both routes against the dense float64 oracle, ragged batches and every tile width; ``wide``: rows of x, paths of W
    and single elements spread over twenty binary orders of magnitude."""
    mod, ops = _operands(device, lmax, cin, cout, n, stable_seed("split", lmax, cin, cout, n))
    if values == "wide":
        gen = torch.Generator().manual_seed(3)
        for t in ops:
            lead = (t.shape[0],) + (1,) * (t.ndim - 1)
            t.mul_(torch.exp2(torch.randint(-20, 21, lead, generator=gen).float()))
        ops[0].mul_(torch.exp2(torch.randint(-10, 11, ops[0].shape, generator=gen).float()))
    split, fp32 = _both_routes(monkeypatch, mod, device, ops)
    T = ref_ops.dense_coupling(SH[lmax], SH[lmax], SH[lmax]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_u1v, T, ops[:3], ops[3])
    for k, (name, want) in enumerate(zip(("out", "grad x", "grad y"), (ref_out, *ref_grads[:2]))):
        # row by row: a row's error against its own size
        def err(a):
            d, w = (a.cpu().double() - want).flatten(1).norm(dim=1), want.flatten(1).norm(dim=1)
            return float((d / w.clamp_min(1e-30)).square().mean().sqrt())
        e_split, e_fp32 = err(split[k]), err(fp32[k])
        print(f"{name} lmax={lmax} {cin}->{cout} n={n} {values}: split {e_split:.2e} fp32 {e_fp32:.2e}")
        # one sample's rounding errors are a handful of draws: a factor of two between two orders of summation
        assert e_split <= (1.1 if n >= 300 else 2.0) * e_fp32 + 3e-8, name


@pytest.mark.parametrize("where,value", [(0, float("inf")), (0, float("nan")), (2, float("inf")), (2, float("nan")), (3, float("-inf")),
                                         (0, 3e38), (2, 1e25), (1, float("inf"))])
def test_values_that_are_not_finite_stay_where_they_couple(device, monkeypatch, where, value):
    mod, ops = _operands(device, 2, 64, 64, 100, 5)
    ops[where].view(-1)[567] = value
    split, fp32 = _both_routes(monkeypatch, mod, device, ops)
    for a, b in zip(split, fp32):
        fin = torch.isfinite(b)
        assert torch.equal(fin, torch.isfinite(a)) and torch.equal(a[~fin].nan_to_num(), b[~fin].nan_to_num())
        assert float((a[fin] - b[fin]).norm()) <= 1e-6 * float(b[fin].norm())


def _per_channel(got, want):
    """Error of every (row, channel) over the samples against its own size (rows alone for a result without channels)."""
    d = (got.cpu().double() - want).norm(dim=0) / want.norm(dim=0)
    return float(d.square().mean().sqrt()), float(d.max())


def _no_worse(name, split, fp32, want, slack):
    for which, new, old in zip(("mean", "largest"), _per_channel(split, want), _per_channel(fp32, want)):
        print(f"{name}: {which} error over the channels: split {new:.2e} fp32 {old:.2e}")
        # each channel's error is that of a few hundred draws: the largest of them scatters more than the mean
        assert new <= slack[which == "largest"] * old + 3e-8, (name, which)


@pytest.mark.parametrize("lmax,cin,cout", [(1, 128, 64), (2, 64, 64), (3, 64, 32), (3, 128, 128)])
def test_every_channel_keeps_its_precision(device, monkeypatch, lmax, cin, cout):
    """Channels of x, of grad_out and of the weight (on either axis) that are up to 2^-30 of the largest, with the products
    of x, W and grad_out balanced, so that every channel counts; errors per row and channel against its own size."""
    mod, ops = _operands(device, lmax, cin, cout, 200, stable_seed("channels", lmax, cin, cout))
    gen = torch.Generator().manual_seed(11)
    a, b = (torch.exp2(torch.randint(0, 31, (c,), generator=gen).float()) for c in (cin, cout))
    ops[0] /= a
    ops[2] *= a[:, None] / b
    ops[3] *= b
    split, fp32 = _both_routes(monkeypatch, mod, device, ops)
    T = ref_ops.dense_coupling(SH[lmax], SH[lmax], SH[lmax]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_u1v, T, ops[:3], ops[3])
    for name, new, old, want in zip(("out", "grad x", "grad y"), split, fp32, (ref_out, *ref_grads[:2])):
        _no_worse(f"{name} lmax={lmax} {cin}->{cout}", new, old, want, (1.1, 1.5))


# exponents of x, y, W and grad_out: results that are ordinary fp32 numbers, of operands or products that are far from 1
RANGES = [(0, 0, 0, 100), (0, 0, -5, 115), (-70, 0, -40, 0), (-40, 0, -40, -30), (-60, 60, -60, 30), (-90, 80, -60, 100),
          (-105, 0, 0, 0), (0, 0, -105, 0), (-107, 0, 1, 0), (2, 2, -106, 0), (-115, 0, 2, -100), (59, -40, 59, 0), (70, -30, 55, -50), (63, 20, 40, 0), (10, 90, 10, 10)]


def _scaled(ops, exponents):
    return [t * 2.0 ** e for t, e in zip(ops, exponents)]


def _check_range(names, split, fp32, refs, exponents):
    for name, new, old, want in zip(names, split, fp32, refs):
        if not torch.isfinite(old).all():
            continue
        assert torch.isfinite(new).all(), (name, exponents)
        if want.abs().max() > 2.0 ** -110:         # below, the terms of the sums are subnormal numbers on either route
            _no_worse(f"{name} of {exponents}", new, old, want, (1.5, 2.5))


@pytest.mark.parametrize("exponents", RANGES)
def test_the_range_of_operands_is_that_of_fp32(device, monkeypatch, exponents):
    mod, ops = _operands(device, 2, 64, 32, 70, 21)
    ops = _scaled(ops, exponents)
    ops[0][3, 2, 5] = 0.0              # an exact zero has no exponent
    split, fp32 = _both_routes(monkeypatch, mod, device, ops)
    T = ref_ops.dense_coupling(SH[2], SH[2], SH[2]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_u1v, T, ops[:3], ops[3])
    _check_range(("out", "grad x", "grad y"), split, fp32, (ref_out, *ref_grads[:2]), exponents)


# ---- channels on both operands ("uvw"): cgtp_uvsw_apply -----------------------------------------------------------
def _uvw_routes(monkeypatch, device, lmax, u, v, c, operands):
    from equitorch_amd.nn import TensorProduct
    from equitorch_amd.nn.functional import _uv_native
    mod = TensorProduct(SH[lmax], SH[lmax], SH[lmax], u, v, c, feature_mode="uvw", internal_weights=False).to(device)
    kinds, split = [], _uv_native._split_uvw

    def spy(kind, *args):
        out = split(kind, *args)
        kinds.append((kind, out is not None))
        return out
    monkeypatch.setattr(_uv_native, "_split_uvw", spy)
    new = _step(mod, device, *operands)
    monkeypatch.setattr(_uv_native, "_split_uvw", lambda *args: None)
    return new, _step(mod, device, *operands), sorted(kinds)


def _uvw_operands(lmax, u, v, c, n, seed):
    d, gen = (lmax + 1) ** 2, torch.Generator().manual_seed(seed)
    paths = {1: 4, 2: 11}[lmax]
    return [torch.randn(n, d, u, generator=gen), torch.randn(n, d, v, generator=gen),
            torch.randn(paths, u, v, c, generator=gen) / u, torch.randn(n, d, c, generator=gen)]


@pytest.mark.parametrize("lmax,u,v,c,n,taken", [(1, 32, 32, 32, 1, (1, 1, 1)), (2, 32, 32, 32, 333, (1, 1, 1)),
                                                (2, 32, 20, 64, 50, (1, 0, 0)), (2, 64, 32, 32, 17, (0, 1, 1)),
                                                (1, 32, 4, 32, 40, (1, 1, 0)), (2, 32, 64, 32, 31, (1, 1, 1))])
@pytest.mark.parametrize("values", ["normal", "wide"])
def test_uvw_no_less_precise_than_fp32_matrix_instructions(device, monkeypatch, lmax, u, v, c, n, taken, values):
    ops = _uvw_operands(lmax, u, v, c, n, stable_seed("uvw split", lmax, u, v, c, n))
    if values == "wide":
        gen = torch.Generator().manual_seed(3)
        for t in ops:
            t.mul_(torch.exp2(torch.randint(-20, 21, (t.shape[0],) + (1,) * (t.ndim - 1), generator=gen).float()))
        ops[0].mul_(torch.exp2(torch.randint(-10, 11, ops[0].shape, generator=gen).float()))
    new, old, kinds = _uvw_routes(monkeypatch, device, lmax, u, v, c, ops)
    assert kinds == [(k, bool(t)) for k, t in enumerate(taken)]
    T = ref_ops.dense_coupling(SH[lmax], SH[lmax], SH[lmax]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_uvw, T, ops[:3], ops[3])
    for k, (name, want) in enumerate(zip(("out", "grad x", "grad y"), (ref_out, *ref_grads[:2]))):
        def err(a):
            d, w = (a.cpu().double() - want).flatten(1).norm(dim=1), want.flatten(1).norm(dim=1)
            return float((d / w.clamp_min(1e-30)).square().mean().sqrt())
        e_new, e_old = err(new[k]), err(old[k])
        print(f"uvw {name} lmax={lmax} {u},{v}->{c} n={n} {values}: split {e_new:.2e} fp32 {e_old:.2e}")
        assert e_new <= (1.1 if n >= 300 else 2.0) * e_old + 3e-8, name


@pytest.mark.parametrize("where,value", [(0, float("inf")), (1, float("nan")), (1, float("inf")), (2, float("inf")),
                                         (3, float("-inf")), (0, 3e38), (2, 1e25)])
def test_uvw_values_that_are_not_finite_stay_where_they_couple(device, monkeypatch, where, value):
    ops = _uvw_operands(2, 32, 32, 32, 50, 6)
    ops[where].view(-1)[567] = value
    new, old, kinds = _uvw_routes(monkeypatch, device, 2, 32, 32, 32, ops)
    for a, b in zip(new, old):
        fin = torch.isfinite(b)
        assert torch.equal(fin, torch.isfinite(a))
        # the fp32 route sums chains of 1024 products times the rows of a path: rounding 6e-8 each at random, 6e-8 * sqrt(1024)
        # = 2e-6 of the result (0.6e-6 to 1.5e-6 measured against 64 bits in the test above)
        assert float((a[fin] - b[fin]).norm()) <= 2e-6 * float(b[fin].norm())


def test_uvw_every_channel_keeps_its_precision(device, monkeypatch):
    u, v, c = 32, 32, 32
    ops = _uvw_operands(2, u, v, c, 150, stable_seed("uvw channels"))
    gen = torch.Generator().manual_seed(12)
    a, z, b = (torch.exp2(torch.randint(0, 21, (k,), generator=gen).float()) for k in (u, v, c))
    ops[0] /= a
    ops[1] /= z
    ops[2] *= a[:, None, None] * z[:, None] / b
    ops[3] *= b
    new, old, _ = _uvw_routes(monkeypatch, device, 2, u, v, c, ops)
    T = ref_ops.dense_coupling(SH[2], SH[2], SH[2]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_uvw, T, ops[:3], ops[3])
    for name, a, b, want in zip(("out", "grad x", "grad y"), new, old, (ref_out, *ref_grads[:2])):
        _no_worse(f"uvw {name}", a, b, want, (1.1, 1.5))


@pytest.mark.parametrize("exponents", RANGES)
def test_uvw_the_range_of_operands_is_that_of_fp32(device, monkeypatch, exponents):
    ops = _scaled(_uvw_operands(2, 32, 32, 32, 40, 22), exponents)
    new, old, _ = _uvw_routes(monkeypatch, device, 2, 32, 32, 32, ops)
    T = ref_ops.dense_coupling(SH[2], SH[2], SH[2]).float().double()
    ref_out, ref_grads = ref_ops.dense_grads(ref_ops.dense_uvw, T, ops[:3], ops[3])
    _check_range(("out", "grad x", "grad y"), new, old, (ref_out, *ref_grads[:2]), exponents)


@pytest.mark.parametrize("mode", ["uv", "uvw"])
def test_recorded_in_a_graph(device, mode):
    """Forward and gradients recorded into a HIP graph and replayed on new inputs and weights: the weights are packed anew by
    every replay."""
    if mode == "uv":
        mod, ops = _operands(device, 2, 64, 64, 50, 4)
    else:
        from equitorch_amd.nn import TensorProduct
        ops = _uvw_operands(2, 32, 32, 32, 50, 4)
        mod = TensorProduct(SH[2], SH[2], SH[2], 32, 32, 32, feature_mode="uvw", internal_weights=False).to(device)
    inputs, ct = [t.to(device).requires_grad_(True) for t in ops[:3]], ops[3].to(device)

    def step():
        out = mod(*inputs)
        return (out, *torch.autograd.grad(out, inputs, ct))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = step()
    for replay in range(3):
        with torch.no_grad():
            for t in inputs:
                t.copy_(torch.randn(t.shape, generator=torch.Generator().manual_seed(replay)) * 2.0 ** (5 * replay))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(recorded, step()):
            assert torch.equal(a, b), replay
