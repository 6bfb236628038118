"""Channel mixing in fp32 on the half-precision matrix cores (``cgtp_uvl_apply``, ``cgtp_uvl_grad_w``; IrrepsLinear and SO2Linear('uv') with a shared
weight): every operand carried as three bf16 parts, no less precise than fp32 matrix instructions and of their range."""
import numpy as np
import pytest
import torch

from helpers import stable_seed

SH = {l: "+".join(f"{k}{'eo'[k % 2]}" for k in range(l + 1)) for l in range(7)}


def _coo(kind, l):
    """Table of a layer as entries (row of the result, row of the input, weight, coefficient)."""
    from equitorch_amd import nn as enn
    from equitorch_amd.nn.functional import _irreps_gemm as G
    if kind == "so2":
        mod = enn.SO2Linear(SH[l], SH[l], 4, 4, feature_mode="uv")
        plan = G.plan_of_product_info(mod.info_forward, mod.irreps_in.dim, mod.num_weights)
    else:
        mod = enn.IrrepsLinear(SH[l], "2e+0e+1o+0e", 4, 4)
        plan = G.plan_of_linear_info(mod.forward_info)
    return [(p.o0 + j, p.i0 + j, p.w, p.scale) for p in plan.paths for j in range(p.k)], plan, (l + 1) ** 2


def _table(entries, n_in, n_out, n_w):
    from equitorch_amd._tables import TpCoo
    from equitorch_amd.nn.functional import _uv_native as N
    m, m1, p, c = (np.asarray(v) for v in zip(*entries))
    z = np.zeros(len(m), dtype=np.int32)
    coo = TpCoo(c.astype(np.float64), m.astype(np.int32), m1.astype(np.int32), z, p.astype(np.int32), z, n_in, 1, n_out, n_w)
    return N.CooTable(coo, torch.zeros(1), None, mixing=True)


@pytest.mark.parametrize("kind,l", [("so2", 2), ("so2", 6), ("lin", 2), ("own", 0), ("any", 1), ("any", 2), ("any", 3)])
@pytest.mark.parametrize("transposed", [False, True])
def test_the_steps_are_the_table(kind, l, transposed):
    """Tasks, steps and groups for every number of groups against the table's entries; ``own``: several weights and coefficients
    for one pair of rows, and rows of either side that no entry reaches; ``any``: entries at random."""
    from equitorch_amd.nn.functional import _uv_native as N
    if kind == "own":
        entries, n_in, n_out, n_w = [(0, 2, 1, 0.5), (0, 2, 0, -2.0), (3, 2, 1, 0.5), (3, 0, 1, 1.5), (0, 0, 2, 3.0), (1, 4, 2, 1.0)], 6, 5, 3
    elif kind == "any":
        rng = np.random.default_rng(l)
        n_in, n_out, n_w = 11 * l, 7 * l, 3
        entries = [(int(a), int(b), int(c), float(s)) for a, b, c, s in zip(*(rng.integers(0, k, 40 * l) for k in (n_out, n_in, n_w)),
                                                                            rng.choice([1.0, 0.5], 40 * l))]
    else:
        entries, plan, n_in = _coo(kind, l)
        n_out, n_w = plan.out_size, plan.n_paths
    table = N._MixTable(_table(entries, n_in, n_out, n_w).coo, transposed)
    want = sorted(((i, m) if transposed else (m, i)) + (p, np.float32(c)) for m, i, p, c in entries)
    walk = N._MixWalk(table, "cpu")
    words = walk.words.numpy()
    n_steps = sum(map(len, table.steps))
    for g, (at_steps, at_groups, at_tasks, at_blocks) in walk.at.items():
        assert at_steps % 16 == 0 and at_groups % 8 == 0 and at_tasks % 8 == 0 and at_blocks % 8 == 0
        steps = words[at_steps // 4:].reshape(-1)[:4 * n_steps].reshape(-1, 4)
        groups = words[at_groups // 4:][:2 * g].reshape(-1, 2)
        tasks = words[at_tasks // 4:][:2 * len(table.tasks)].reshape(-1, 2)
        blocks = words[at_blocks // 4:][:2 * table.n_blocks].reshape(-1, 2)
        assert groups[0, 0] == 0 and groups[-1, 1] == len(steps) and (groups[1:, 0] == groups[:-1, 1]).all()
        assert (groups[:, 1] > groups[:, 0]).all() and (groups[:, 1] - groups[:, 0]).max() == walk.max_steps[g]
        assert all(steps[e - 1, 3] >= 0 for _, e in groups)                 # whole tasks
        got, rows, begin = [], [], 0
        for s, (row, b0, b1, task) in enumerate(steps):
            if task < 0:
                continue
            for i, x0, x1, _ in steps[begin:s + 1]:
                for row_out, b in zip(tasks[task], (x0, x1)):
                    if b >= 0:
                        assert row_out >= 0
                        got.append((int(row_out), int(i), int(blocks[b, 0]), blocks[b, 1:].view(np.float32)[0]))
            rows += [int(r) for r in tasks[task] if r >= 0]
            begin = s + 1
        assert sorted(got) == want and sorted(rows) == list(range(table.n_out))
    if kind == "so2":
        assert table.rows_per_task == 2
    assert table.groups_for(10 ** 6, 1) >= 1 and max(len(s) for s in table.steps) == table.longest


def test_rows_that_the_same_rows_reach_are_paired():
    """Copies of irreps mixed with copies: two rows at a time, also where an odd row is left over or reached by nearly the same."""
    from equitorch_amd.nn.functional import _uv_native as N
    full = [(m, i, 0, 1.0) for m in range(5) for i in range(6)]
    assert N._MixTable(_table(full, 6, 5, 1).coo, False).tasks == [(0, 1), (2, 3), (4, -1)]
    most = [e for e in full if e[:2] != (4, 0)] + [(5, i, 0, 1.0) for i in range(6)]       # 4 has five of the six of 5
    assert N._MixTable(_table(most, 6, 6, 1).coo, False).tasks == [(0, 1), (2, 3), (4, 5)]
    apart = [(m, i, 0, 1.0) for m in range(4) for i in range(6) if i % 4 == m]
    assert N._MixTable(_table(apart, 6, 4, 1).coo, False).tasks == [(m, -1) for m in range(4)]


def test_layers_of_one_table_share_its_steps():
    """A second layer over the same irreps repeats no host work; another table or direction has steps of its own."""
    from equitorch_amd.nn.functional import _uv_native as N
    tables = [_table(entries, n_in, plan.out_size, plan.n_paths) for entries, plan, n_in in (_coo("so2", 2), _coo("so2", 2), _coo("lin", 2))]
    first, second, other = (N._mix_table(t, False) for t in tables)
    assert first is second and first is not other and N._mix_table(tables[0], True) is not first
    assert first.words[0] is second.words[0]


# ---- on the GPU ------------------------------------------------------------------------------------------------------
def _module(kind, l, cin, cout, device):
    from equitorch_amd import nn as enn
    torch.manual_seed(stable_seed("mix", kind, l, cin, cout))
    if kind == "so2":
        return enn.SO2Linear(SH[l], SH[l], cin, cout, feature_mode="uv").to(device)
    if kind == "copies":               # a result's row of l inputs, and an input's of l results; the others are many
        return enn.IrrepsLinear(f"{l}x0e+8o+9o", f"8o+{l}x0e+9o", cin, cout).to(device)
    return enn.IrrepsLinear(SH[l], SH[l] if kind == "lin" else "2e+0e+1o+0e", cin, cout).to(device)


def _run(mod, x, g):
    x = x.detach().requires_grad_(True)
    out = mod(x)
    return [t.detach() for t in (out, torch.autograd.grad(out, [x], g)[0])]


def _routes(monkeypatch, kind, l, cin, cout, x, g, device, scale=1.0, sign=False):
    """Results of the split kernels, of the route without them and of float64."""
    from equitorch_amd.nn.functional import _uv_native as N
    mod = _module(kind, l, cin, cout, device)
    with torch.no_grad():
        mod.weight.mul_(scale)
        if sign:
            mod.weight.abs_()
    taken, split = [], N._mix_split

    def spy(*args):
        out = split(*args)
        taken.append(out is not None)
        return out
    monkeypatch.setattr(N, "_mix_split", spy)
    new = _run(mod, x.to(device), g.to(device))
    assert taken == [True, True]
    monkeypatch.setattr(N, "_mix_split", lambda *args: None)
    monkeypatch.setattr(N, "mix_fits", lambda *args: False)
    old = _run(mod, x.to(device), g.to(device))
    ref = _run(mod.double(), x.double().to(device), g.double().to(device))
    return new, old, ref


def _operands(kind, l, cin, cout, n, seed):
    gen = torch.Generator().manual_seed(seed)
    rows_out = (l + 1) ** 2 if kind != "own" else 10
    return torch.randn(n, (l + 1) ** 2, cin, generator=gen), torch.randn(n, rows_out, cout, generator=gen)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n", [
    ("lin", 1, 4, 4, 1), ("lin", 2, 12, 20, 65), ("own", 3, 36, 100, 129), ("lin", 2, 64, 64, 3000), ("lin", 3, 128, 96, 700),
    ("lin", 1, 160, 32, 2500), ("so2", 2, 32, 32, 63), ("so2", 4, 64, 64, 1000), ("so2", 6, 48, 48, 257), ("so2", 3, 40, 132, 31)])
@pytest.mark.parametrize("values", ["normal", "wide"])
def test_no_less_precise_than_fp32_matrix_instructions(device, monkeypatch, kind, l, cin, cout, n, values):
    """Ragged batches, channels that fill no tile, rows no entry reaches; ``wide``: samples and elements spread over twenty
    binary orders of magnitude."""
    x, g = _operands(kind, l, cin, cout, n, stable_seed("mix operands", kind, l, cin, cout, n))
    if values == "wide":
        gen = torch.Generator().manual_seed(3)
        for t in (x, g):
            t.mul_(torch.exp2(torch.randint(-20, 21, (n, 1, 1), generator=gen).float()))
            t.mul_(torch.exp2(torch.randint(-10, 11, t.shape, generator=gen).float()))
    new, old, ref = _routes(monkeypatch, kind, l, cin, cout, x, g, device)
    for name, a, b, want in zip(("out", "grad x"), new, old, ref):
        def err(t):
            d, w = (t.double() - want).flatten(1).norm(dim=1), want.flatten(1).norm(dim=1)
            return float((d / w.clamp_min(1e-30)).square().mean().sqrt())
        print(f"{name} {kind} lmax={l} {cin}->{cout} n={n} {values}: split {err(a):.2e} fp32 {err(b):.2e}")
        # one sample's rounding errors are a handful of draws: a factor of two between two orders of summation
        assert err(a) <= (1.1 if n >= 300 else 2.0) * err(b) + 3e-8, name


def _tile(mod, kind, transposed, n):
    """What a launch of ``n`` samples is made of: 16 channels and 64 samples so many times, rows of the result at a time; and
    whether a group has several tasks."""
    from equitorch_amd.nn.functional import _irreps_gemm as G
    from equitorch_amd.nn.functional import _uv_native as N
    plan = G.plan_of_product_info(mod.info_forward, mod.irreps_in.dim, mod.num_weights) if kind == "so2" else G.plan_of_linear_info(mod.forward_info)
    mix = N._MixTable(_table([(p.o0 + j, p.i0 + j, p.w, p.scale) for p in plan.paths for j in range(p.k)], mod.irreps_in.dim, plan.out_size,
                             plan.n_paths).coo, transposed)
    cout = mod.weight.shape[1 if transposed else 2]
    tw = 4 if cout % 64 == 0 or cout % 64 > 32 else 2
    groups, nt = mix.groups_for(n, -(-cout // 64)), 4 // mix.rows_per_task
    while nt > 1 and -(-n // (64 * nt)) * groups * -(-cout // (16 * tw)) < 512:
        nt //= 2
    return tw, nt, mix.rows_per_task, groups < len(mix.tasks)


LARGE = [("so2", 4, 64, 64, 33001, (4, 2, 2, True), (4, 2, 2, True)), ("so2", 4, 36, 32, 33001, (2, 2, 2, True), (4, 2, 2, True)),
         ("so2", 6, 48, 32, 4001, (2, 2, 2, True), (4, 2, 2, True)), ("lin", 2, 64, 32, 20003, (2, 2, 1, True), (4, 2, 1, True)),
         ("lin", 2, 32, 64, 70001, (4, 4, 1, True), (2, 4, 1, True)), ("lin", 3, 64, 32, 8001, (2, 4, 1, False), (4, 4, 1, False)),
         ("so2", 2, 64, 64, 20003, (4, 1, 2, True), (4, 1, 2, True)), ("so2", 6, 32, 64, 1500, (4, 1, 2, True), (2, 1, 2, True)),
         ("lin", 4, 128, 32, 3601, (2, 2, 1, False), (4, 2, 1, True)), ("lin", 6, 96, 32, 9001, (2, 2, 1, True), (2, 4, 1, True)),
         ("lin", 4, 128, 128, 1001, (4, 1, 1, False), (4, 1, 1, False))]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n,tile,tile_back", LARGE)
def test_every_tile_is_no_less_precise(device, monkeypatch, kind, l, cin, cout, n, tile, tile_back):
    """Sizes that take two and four times 64 samples of either width, several tasks in a group, ragged at the end."""
    mod = _module(kind, l, cin, cout, "cpu")
    assert (_tile(mod, kind, False, n), _tile(mod, kind, True, n)) == (tile, tile_back)
    x, g = _operands(kind, l, cin, cout, n, stable_seed("mix tiles", kind, l, cin, cout, n))
    new, old, ref = _routes(monkeypatch, kind, l, cin, cout, x, g, device)
    for name, a, b, want in zip(("out", "grad x"), new, old, ref):
        def err(t):        # row by row of the result: each against its own size, the last of the samples by themselves too
            d = t.double() - want
            return torch.stack([d[s].norm(dim=(0, 2)) / want[s].norm(dim=(0, 2)).clamp_min(1e-30) for s in (slice(None), slice(-41, None))])
        e_new, e_old = err(a), err(b)
        print(f"{name} {kind} lmax={l} {cin}->{cout} n={n}: split {e_new.amax(1).tolist()} fp32 {e_old.amax(1).tolist()}")
        # 41 samples are some thousand draws, a tenth of the error either way at most; 3e-8: half a rounding of the result
        assert bool((e_new <= 1.1 * e_old + 3e-8).all()), name


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n", [case[:5] for case in LARGE])
def test_what_is_not_split_in_every_tile(device, monkeypatch, kind, l, cin, cout, n):
    """A sample with an infinity and one with a tiny element in every row, spread over the batch: first, middle and last tasks
    of a group form their results anew, and no other result changes."""
    from equitorch_amd.nn.functional import _uv_native as N
    x, g = _operands(kind, l, cin, cout, n, 17)
    for t in (x, g):
        rows = t.shape[1]
        for k in range(rows):
            t[(k + 1) * n // (rows + 2), k, 3 * k % t.shape[2]] = float("inf")
            t[n - 1 - k, k, 5 * k % t.shape[2]] = 2.0 ** -120
    mod = _module(kind, l, cin, cout, device)
    new = _run(mod, x.to(device), g.to(device))
    monkeypatch.setattr(N, "_mix_split", lambda *args: None)
    monkeypatch.setattr(N, "mix_fits", lambda *args: False)
    for a, b in zip(new, _run(mod, x.to(device), g.to(device))):
        fin = torch.isfinite(b)
        assert not fin.all() and torch.equal(fin, torch.isfinite(a)) and torch.equal(a[~fin].nan_to_num(), b[~fin].nan_to_num())
        a, b = (t.nan_to_num(0.0, 0.0, 0.0).double() for t in (a, b))
        assert float(((a - b).norm(dim=(0, 2)) / b.norm(dim=(0, 2)).clamp_min(1e-30)).max()) <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n", [("so2", 6, 48, 48, 700), ("so2", 5, 64, 96, 500), ("lin", 4, 256, 64, 900), ("so2", 6, 256, 32, 300),
                                               ("copies", 4, 64, 36, 400), ("copies", 2, 128, 128, 600)])
@pytest.mark.parametrize("sign", [False, True])
def test_long_rows_are_no_less_precise_than_the_library(device, monkeypatch, kind, l, cin, cout, n, sign):
    """Rows past the fp32 kernels' sizes were products of the library, which sums in blocks; ``sign``: inputs and weights of one
    sign, where a rounding to one side does not average out.  Both are random errors of a few hundred sums each: a tenth."""
    mod = _module(kind, l, cin, cout, "cpu")
    gen = torch.Generator().manual_seed(stable_seed("long", kind, l, cin, cout))
    x, g = torch.randn(n, mod.irreps_in.dim, cin, generator=gen), torch.randn(n, mod.irreps_out.dim, cout, generator=gen)
    if sign:
        x, g = x.abs(), g.abs()
    new, old, ref = _routes(monkeypatch, kind, l, cin, cout, x, g, device, sign=sign)
    for name, a, b, want in zip(("out", "grad x"), new, old, ref):
        e_new, e_old = (float((t.double() - want).norm() / want.norm()) for t in (a, b))
        print(f"{name} {kind} {l} {cin}->{cout} sign={sign}: split {e_new:.2e} library {e_old:.2e}")
        assert e_new <= 1.1 * e_old, name


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n", [("so2", 6, 48, 48, 300), ("so2", 6, 256, 256, 40), ("so2", 6, 256, 256, 300), ("so2", 6, 256, 256, 511),
                                               ("so2", 6, 256, 256, 512), ("so2", 6, 132, 96, 300), ("lin", 4, 256, 64, 40), ("lin", 4, 256, 64, 512)])
@pytest.mark.parametrize("sign", [False, True])
def test_their_weight_gradient_is_no_less_precise_than_the_library(device, monkeypatch, kind, l, cin, cout, n, sign):
    """Of the same layers; thousands of sums each, so that the errors are known to a few parts in a hundred."""
    from equitorch_amd.nn.functional import _uv_native as N
    mod = _module(kind, l, cin, cout, device)
    gen = torch.Generator().manual_seed(stable_seed("long gw", kind, l, cin, cout, n))
    x, g = (torch.randn(n, irreps.dim, c, generator=gen).to(device) for irreps, c in ((mod.irreps_in, cin), (mod.irreps_out, cout)))
    if sign:
        x, g = x.abs(), g.abs()
    taken, fits = [], N.mix_fits

    def spy(*args):
        taken.append(fits(*args))
        return taken[-1]
    monkeypatch.setattr(N, "mix_fits", spy)
    new, = torch.autograd.grad(mod(x), [mod.weight], g)
    assert taken == [True]
    monkeypatch.setattr(N, "mix_fits", lambda *args: False)
    old, = torch.autograd.grad(mod(x), [mod.weight], g)
    mod.double()
    want, = torch.autograd.grad(mod(x.double()), [mod.weight], g.double())
    e_new, e_old = (float((t.double() - want).norm() / want.norm()) for t in (new, old))
    print(f"grad W {kind} {l} {cin}->{cout} n={n} sign={sign}: kernel {e_new:.2e} library {e_old:.2e}")
    assert e_new <= 1.1 * e_old


@pytest.mark.gpu
def test_what_stays_on_the_library(device, monkeypatch):
    """Rows whose sums the library forms more precisely, and products it forms as quickly."""
    from equitorch_amd.nn.functional import _uv_native as N
    monkeypatch.setattr(N, "_mix_split", lambda *args: pytest.fail("a kernel was called"))
    for kind, l, c, n in (("copies", 24, 128, 70), ("copies", 60, 256, 70), ("so2", 6, 288, 70), ("lin", 4, 320, 70), ("lin", 4, 128, 4000)):
        mod = _module(kind, l, c, c, device)
        x = torch.randn(n, mod.irreps_in.dim, c, generator=torch.Generator().manual_seed(1)).to(device)
        want = _module(kind, l, c, c, device).double()(x.double())
        assert float((mod(x).double() - want).detach().norm()) <= 1e-6 * float(want.detach().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("where,value", [("x", float("inf")), ("x", float("nan")), ("g", float("-inf")), ("x", 3.4e38), ("w", float("inf"))])
@pytest.mark.parametrize("kind", ["lin", "so2"])
def test_values_that_are_not_finite_stay_where_they_couple(device, monkeypatch, kind, where, value):
    from equitorch_amd.nn.functional import _uv_native as N
    x, g = _operands(kind, 2, 32, 64, 150, 7)
    mod = _module(kind, 2, 32, 64, device)
    {"x": x, "g": g, "w": mod.weight.data}[where].view(-1)[567] = value
    new = _run(mod, x.to(device), g.to(device))
    monkeypatch.setattr(N, "_mix_split", lambda *args: None)
    for a, b in zip(new, _run(mod, x.to(device), g.to(device))):
        fin = torch.isfinite(b)
        assert torch.equal(fin, torch.isfinite(a)) and torch.equal(a[~fin].nan_to_num(), b[~fin].nan_to_num())
        assert float((a[fin] - b[fin]).norm()) <= 1e-6 * float(b[fin].norm())


@pytest.mark.gpu
@pytest.mark.parametrize("exponent,scale", [(0, 0), (-70, -40), (-105, 0), (-115, 0), (-118, 30), (0, -112), (-60, -50), (60, 60), (100, -20), (-113, 100)])
def test_the_range_of_operands_is_that_of_fp32(device, monkeypatch, exponent, scale):
    x, g = _operands("so2", 2, 64, 32, 70, 8)
    x[3, 2, 5] = 0.0                   # an exact zero has no exponent
    x, g = x * 2.0 ** exponent, g * 2.0 ** exponent
    new, old, ref = _routes(monkeypatch, "so2", 2, 64, 32, x, g, device, 2.0 ** scale)
    for name, a, b, want in zip(("out", "grad x"), new, old, ref):
        assert torch.isfinite(a).all() == torch.isfinite(b).all()
        if want.abs().max() > 2.0 ** -110 and torch.isfinite(b).all():    # below, the products are subnormal numbers on either route
            def err(t):
                d = (t.double() - want).norm(dim=0) / want.norm(dim=0)
                return float(d.square().mean().sqrt())
            print(f"{name} of 2^{exponent}, 2^{scale}: split {err(a):.2e} fp32 {err(b):.2e}")
            assert err(a) <= 1.5 * err(b) + 3e-8, name


@pytest.mark.gpu
def test_weights_that_a_coefficient_takes_to_zero(device, monkeypatch):
    """The smallest subnormal weights next to large inputs: a coefficient below one half (rows of order 0) may meet x, not them."""
    from equitorch_amd.nn.functional import _uv_native as N
    x, g = (t * 2.0 ** 100 for t in _operands("so2", 4, 32, 32, 70, 13))
    mod = _module("so2", 4, 32, 32, device)
    with torch.no_grad():
        mod.weight.copy_(mod.weight.sign() * 2.0 ** -149)
    new = _run(mod, x.to(device), g.to(device))
    monkeypatch.setattr(N, "_mix_split", lambda *args: None)
    old = _run(mod, x.to(device), g.to(device))
    ref = _run(mod.double(), x.double().to(device), g.double().to(device))
    for name, a, b, want in zip(("out", "grad x"), new, old, ref):
        e_new, e_old = ((t.double() - want).norm(dim=(0, 2)) / want.norm(dim=(0, 2)) for t in (a, b))
        print(f"{name}: split {float(e_new.max()):.2e} fp32 {float(e_old.max()):.2e}")
        assert bool((e_new <= 2.0 * e_old + 3e-8).all()), name


# ---- gradient of the weight --------------------------------------------------------------------------------------------
def _weight_gradients(monkeypatch, kind, l, cin, cout, x, g, device):
    from equitorch_amd.nn.functional import _uv_native as N
    mod = _module(kind, l, cin, cout, device)
    taken, split = [], N._mix_grad_w

    def spy(*args):
        taken.append(args)
        return split(*args)
    monkeypatch.setattr(N, "_mix_grad_w", spy)
    new, = torch.autograd.grad(mod(x.to(device)), [mod.weight], g.to(device))
    (xs, gs, table), = taken
    ones = torch.ones(xs.shape[0], 1, device=device)
    monkeypatch.setattr(N, "_mix_grad_w", lambda *args: None)
    return new, N.grad_w(xs, ones, gs, table), N.grad_w(xs.double(), ones.double(), gs.double(), table)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,l,cin,cout,n", [("lin", 1, 4, 4, 1), ("lin", 2, 12, 20, 65), ("own", 3, 36, 100, 129), ("lin", 2, 64, 64, 70001),
                                               ("lin", 3, 128, 96, 700), ("so2", 2, 32, 64, 31), ("so2", 4, 64, 32, 2077), ("so2", 6, 48, 48, 257), ("lin", 1, 96, 128, 40001),
                                               ("own", 2, 128, 64, 33000)])
@pytest.mark.parametrize("values", ["normal", "wide"])
def test_the_weight_gradient_is_no_less_precise(device, monkeypatch, kind, l, cin, cout, n, values):
    x, g = _operands(kind, l, cin, cout, n, stable_seed("mix gw", kind, l, cin, cout, n))
    if values == "wide":
        gen = torch.Generator().manual_seed(3)
        for t in (x, g):
            t.mul_(torch.exp2(torch.randint(-10, 11, (n, 1, 1), generator=gen).float()))
        x[n // 2 + 1:n // 2 + 9] = 0.0
    new, old, ref = _weight_gradients(monkeypatch, kind, l, cin, cout, x, g, device)
    e_new, e_old = (float((t.double() - ref).norm() / ref.norm()) for t in (new, old))
    print(f"grad W {kind} lmax={l} {cin}->{cout} n={n} {values}: split {e_new:.2e} fp32 {e_old:.2e}")
    assert e_new <= e_old + 3e-8


@pytest.mark.gpu
@pytest.mark.parametrize("where,value", [(0, float("inf")), (1, float("nan")), (1, float("-inf")), (0, 3.39e38)])
def test_the_weight_gradient_of_values_that_are_not_finite(device, monkeypatch, where, value):
    ops = list(_operands("so2", 2, 32, 64, 150, 7))
    ops[1 - where] *= 2.0 ** -8
    ops[where].view(-1)[567] = value
    new, old, _ = _weight_gradients(monkeypatch, "so2", 2, 32, 64, *ops, device)
    fin = torch.isfinite(old)
    assert torch.equal(fin, torch.isfinite(new)) and torch.equal(new[~fin & ~old.isnan()], old[~fin & ~old.isnan()])
    assert float((new[fin].double() - old[fin].double()).norm()) <= 1e-6 * float(old[fin].double().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("exponents", [(0, 0), (-105, 0), (-118, 100), (0, -113), (-60, -48), (60, 60)])
def test_the_weight_gradient_has_the_range_of_fp32(device, monkeypatch, exponents):
    ops = [t * 2.0 ** e for t, e in zip(_operands("lin", 2, 64, 32, 300, 8), exponents)]
    new, old, ref = _weight_gradients(monkeypatch, "lin", 2, 64, 32, *ops, device)
    assert torch.equal(torch.isfinite(new), torch.isfinite(old))
    if ref.abs().max() > 2.0 ** -100:
        e_new, e_old = (float((t.double() - ref).norm() / ref.norm()) for t in (new, old))
        print(f"{exponents}: split {e_new:.2e} fp32 {e_old:.2e}")
        assert e_new <= 1.5 * e_old + 3e-8


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["lin", "so2"])
def test_recorded_in_a_graph(device, kind):
    """Forward and gradients recorded and replayed on new inputs and weights: the weight is packed anew by every replay."""
    mod = _module(kind, 2, 32, 64, device)
    x, g = (t.to(device) for t in _operands(kind, 2, 32, 64, 100, 9))
    x.requires_grad_(True)

    def step():
        out = mod(x)
        return (out, *torch.autograd.grad(out, [x, mod.weight], g))
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
            gen = torch.Generator().manual_seed(replay)
            for t in (x, mod.weight):
                t.copy_(torch.randn(t.shape, generator=gen) * 2.0 ** (5 * replay))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(recorded, step()):
            assert torch.equal(a, b), replay


@pytest.mark.gpu
def test_transforms_of_the_library_route_stay(device):
    """An SO(2) layer too large for the fp32 kernels was tensor algebra: forward mode and vmap still take it."""
    mod = _module("so2", 6, 64, 64, device)
    x, t = (v.to(device) for v in _operands("so2", 6, 64, 64, 20, 10))
    want = mod(t).detach()             # the layer's plan is made by a plain call
    out, tangent = torch.func.jvp(mod, (x,), (t,))
    assert float((out - mod(x)).detach().norm()) <= 2e-6 * float(out.detach().norm())
    assert float((tangent - want).detach().norm()) <= 2e-6 * float(want.norm())
    batched = torch.func.vmap(lambda v: mod(v))(x.view(2, 10, *x.shape[1:]))
    assert float((batched.flatten(0, 1) - out).detach().norm()) <= 2e-6 * float(out.detach().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("first", ["jvp", "vmap"])
def test_a_first_call_inside_a_transform(device, first):
    """The tables that a layer's first call makes from its plan are data, also where that call is inside a transform."""
    from equitorch_amd.nn.functional import _irreps_gemm as G
    mod, other = (_module("so2", 6, 64, 64, device) for _ in range(2))
    G.plan_of_product_info(mod.info_forward, mod.irreps_in.dim, mod.num_weights)     # which no transform lets be read off
    x, t = (v.to(device) for v in _operands("so2", 6, 64, 64, 20, 10))
    if first == "jvp":
        got, tangent = torch.func.jvp(mod, (x,), (t,))
        assert float((tangent - other(t)).detach().norm()) <= 2e-6 * float(tangent.detach().norm())
    else:
        got = torch.func.vmap(lambda v: mod(v))(x.view(2, 10, *x.shape[1:])).flatten(0, 1)
    want = other(x)
    for a in (got, mod(x), torch.func.jvp(mod, (x,), (t,))[0]):
        assert float((a - want).detach().norm()) <= 2e-6 * float(want.detach().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["batched gradients", "vmap of the gradient", "second order", "operators seen", "autocast"])
def test_what_tensor_algebra_takes_is_taken(device, monkeypatch, what):
    """A layer that was tensor algebra, in all that sees its operations one by one: as on the library route."""
    from torch.utils.flop_counter import FlopCounterMode

    from equitorch_amd.nn.functional import _uv_native as N
    x, t = (v.to(device) for v in _operands("so2", 6, 64, 64, 6, 11))
    gs = torch.randn(3, *t.shape, generator=torch.Generator().manual_seed(12)).to(device)

    def results():
        mod = _module("so2", 6, 64, 64, device)
        leaf = x.clone().requires_grad_(True)
        if what == "batched gradients":
            return torch.autograd.grad(mod(leaf), [leaf, mod.weight], gs, is_grads_batched=True)
        if what == "vmap of the gradient":
            out = mod(leaf)
            return torch.func.vmap(lambda g: torch.autograd.grad(out, [leaf, mod.weight], g, retain_graph=True))(gs)
        if what == "second order":
            first = torch.autograd.grad(mod(leaf), [leaf, mod.weight], t, create_graph=True)
            return torch.autograd.grad(sum((f * f).sum() for f in first), [leaf, mod.weight])
        if what == "operators seen":
            with FlopCounterMode(display=False) as count:
                out = mod(x)
            assert count.get_total_flops() > 0
            return [out]
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return [mod(x)]
    got = results()
    monkeypatch.setattr(N, "mix_fits", lambda *args: False)
    for a, b in zip(got, results()):
        assert a.dtype == b.dtype
        assert float((a.double() - b.double()).detach().norm()) <= 4e-6 * float(b.detach().double().norm())
