"""The matrix-core segment kernels of small tables that are not compiled in (``cgtp_uvu_mx_fwd`` / ``_bwd``): the walk
the host builds for them, read back word by word on the CPU, and the kernels at the edges of their range."""
import numpy as np
import pytest
import torch

from helpers import assert_close, stable_seed
from oracle import ref_ops

# (out, in1, in2): several multiplicities, one row only, 16 rows on either side, 32 rows of y, an uncoupled middle,
# output irreps of more than seven rows (two or more items of the four-row walk per path)
TABLES = [
    ("1o+2e+1e", "0e+1o+2e", "0e+1o"),
    ("0e+1o+2e+3o", "1o+2e+3o", "0e+1o+2e"),
    ("2x0e+1o+1e", "0e+2x1o", "0e+1o+1e"),
    ("0e", "0e", "0e+0e"),
    ("0e+1e+2e+3e", "0e+1o+2e+3o", "0e+1o"),
    ("1o+3o", "0e+3o", "0e+1o+2e+3o+4e"),
    ("0e+4e", "0e+1o+2e", "0e+1o+2e+3o+4e"),
    ("1o+5o", "0e+1o+2e", "0e+1o+2e+3o+4e"),
    ("4e", "4e", "0e+2e"),
    ("7o", "0e+4e", "3o+4e"),
]


def _info(irreps):
    from equitorch_amd.nn import SO3Linear
    io, i1, i2 = irreps
    return SO3Linear(i1, i2, io, 4, 4, internal_weights=False, feature_mode="uu").tp_info_forward


@pytest.mark.parametrize("irreps", TABLES)
def test_the_walk_covers_the_table(irreps):
    """Forward and the three gradients of one edge, computed from the words alone with the kernels' index arithmetic,
    against the table's entries."""
    from equitorch_amd.ops import kernels
    coo = kernels.coo_of(_info(irreps))
    m = kernels.uvu_mx_words(coo)
    assert m is not None
    rng = np.random.default_rng(stable_seed("mx walk", irreps))
    D1, D2, DO, P, C = coo.D1, coo.D2, coo.DO, coo.P, 3
    x, y, w, g = (rng.standard_normal(s) for s in ((D1, C), (D2,), (P, C), (DO, C)))
    want = {"out": np.zeros((DO, C)), "gx": np.zeros((D1, C)), "gy": np.zeros(D2), "gw": np.zeros((P, C))}
    for c, M, a, b, p in zip(coo.coef, coo.M, coo.M1, coo.M2, coo.p):
        c = float(np.float32(c))
        want["out"][M] += c * x[a] * y[b] * w[p]
        want["gx"][a] += c * g[M] * y[b] * w[p]
        want["gy"][b] += c * (g[M] * x[a] * w[p]).sum()
        want["gw"][p] += c * g[M] * x[a] * y[b]

    def f32(v):
        return float(np.uint32(v).view(np.float32))

    def couple(words, n_rec, n_ent):
        A = np.zeros(64 * n_ent + 4)
        for c0, c1, k in words[:3 * n_rec].reshape(-1, 3):
            A[k >> 16] = f32(c0) * y[k & 255] + f32(c1) * y[(k >> 8) & 255]
        return A, words[3 * n_rec:3 * n_rec + n_ent]

    def contract(A, entries, rows):
        rows = np.concatenate([rows, np.zeros((3, C))])
        acc = np.zeros((16, C))
        for e, k in enumerate(entries):
            b = w[k & 255] * rows[(k >> 8):(k >> 8) + 4]
            acc += A[64 * e:64 * e + 64].reshape(4, 16).T @ b
        return acc
    A, entries = couple(m["fwd"], m["fwd_records"], m["fwd_entries"])
    got = {"out": contract(A, entries, x)[:DO]}
    A, entries = couple(m["bwd"], m["bwd_records"], m["bwd_entries"])
    got["gx"] = contract(A, entries, g)[:D1]
    at = 3 * m["bwd_records"] + m["bwd_entries"]
    rows = m["bwd"][at:at + 16 * m["row_tiles"]]
    at += 16 * m["row_tiles"]
    xz = np.concatenate([x, np.zeros((16 - D1, C))])
    G = np.concatenate([(w[k & 255] * g[k >> 8]) @ xz.T for k in rows])
    terms = m["bwd"][at:at + 128 * m["rounds"]].reshape(-1, 64, 2)
    at += 128 * m["rounds"]
    lanes = np.array([sum(f32(t[lane, 0]) * G[t[lane, 1]] for t in terms) for lane in range(64)])
    assert D2 << m["lanes_log2"] <= 64
    got["gy"] = lanes.reshape(-1, 1 << m["lanes_log2"]).sum(1)[:D2]
    gw = np.full((P, C), np.nan)
    gz = np.concatenate([g, np.zeros((3, C))])
    for tile in m["bwd"][at:at + 5 * m["tiles"]].reshape(-1, 5):
        seen = set()
        for k in tile[1:]:
            n, p = int(k >> 25), int((k >> 16) & 255)
            if n == 0:
                continue
            assert p not in seen
            seen.add(p)
            v = np.zeros(C)
            for i in range(n):
                r0 = int(tile[0] & 255)
                D = sum(A[(k & 0xffff) + 64 * s + 16 * q + i] * gz[r0 + 4 * s + q]
                        for s in range(int(tile[0] >> 8)) for q in range(4))
                v += x[(k & 15) + i] * D
            gw[p] = v + gw[p] if k & (1 << 24) else v
    got["gw"] = gw
    for name in want:
        np.testing.assert_allclose(got[name], want[name], rtol=0, atol=1e-12 * max(1, np.abs(want[name]).max()), err_msg=name)


def test_tables_that_do_not_fit_are_left_to_the_general_walk():
    from equitorch_amd.ops import kernels
    assert kernels.uvu_mx_words(kernels.coo_of(_info(("0e+1e+2e+4e", "0e+1o+2e", "0e+1o+2e")))) is None      # 18 rows
    assert kernels.uvu_mx_words(kernels.coo_of(_info(("0e+2e", "0e+4e+2e+3o", "0e+2e")))) is None             # 22 rows


def test_struct_layout():
    import ctypes as C
    from equitorch_amd import _lib
    n = _lib.lib.cgtp_abi_layout(12, None, 0)
    buf = (C.c_int64 * n)()
    assert _lib.lib.cgtp_abi_layout(12, buf, n) == n == 1 + len(_lib.UvuMx._fields_)
    assert buf[0] == C.sizeof(_lib.UvuMx)
    assert list(buf)[1:] == [getattr(_lib.UvuMx, name).offset for name, _ in _lib.UvuMx._fields_]


def _edge_case(irreps, channels, n_nodes, n_edges, hub, seed):
    from equitorch_amd.irreps import Irreps
    io, i1, i2 = irreps
    gen = torch.Generator().manual_seed(seed)
    src = torch.randint(0, n_nodes, (n_edges,), generator=gen)
    dst = torch.randint(0, n_nodes, (n_edges,), generator=gen)
    if hub:
        dst[torch.rand(n_edges, generator=gen) < 0.4] = 1
        src[src == 2], dst[dst == 2] = 0, 0
    P = len(set(_paths(irreps)))
    return (src, dst, torch.randn(n_nodes, Irreps(i1).dim, channels, generator=gen),
            torch.randn(n_edges, Irreps(i2).dim, generator=gen), torch.randn(n_edges, P, channels, generator=gen),
            torch.randn(n_nodes, Irreps(io).dim, channels, generator=gen))


def _paths(irreps):
    from equitorch_amd.ops import kernels
    return kernels.coo_of(_info(irreps)).p.tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("irreps", TABLES)
@pytest.mark.parametrize("channels,n_nodes,n_edges,hub", [(64, 5, 1, False), (60, 40, 700, True), (48, 3, 9000, False),
                                                          (32, 300, 2049, True), (18, 50, 600, False), (16, 70, 900, False),
                                                          (5, 30, 400, True), (36, 3000, 2500, False)])
def test_product_and_gradients(device, monkeypatch, irreps, channels, n_nodes, n_edges, hub):
    """One, two and four channels per lane with and without idle lanes; one edge, ranges of more than 64 positions,
    nodes without edges, a node whose edges span many ranges; every subset of gradients the kernels tell apart."""
    from equitorch_amd.nn.functional import EdgePlan, edge_tensor_product_uu
    from equitorch_amd.ops import kernels
    monkeypatch.setattr(kernels, "_mx_pays", lambda *args: True)          # the kernels, also where the walk is quicker
    info = _info(irreps).to(device)
    src, dst, x, y, w, ct = _edge_case(irreps, channels, n_nodes, n_edges, hub, stable_seed("mx", irreps, channels))
    plan = EdgePlan(src.to(device), dst.to(device), n_nodes)
    T = ref_ops.dense_coupling(*irreps).float().double()

    def ref_fn(T, x, sh, w):
        return ref_ops.scatter_sum(ref_ops.dense_u1u(T, x.index_select(0, src), sh, w), dst, n_nodes)
    ref_out, ref_grads = ref_ops.dense_grads(ref_fn, T, (x, y, w), ct)
    for need in ((True, True, True), (False, True, False), (True, False, False), (False, False, True)):
        wrt = [t.to(device).requires_grad_(n) for t, n in zip((x, y, w), need)]
        out = edge_tensor_product_uu(*wrt, plan, info)
        grads = torch.autograd.grad(out, [t for t, n in zip(wrt, need) if n], ct.to(device))
        assert_close(out, ref_out, 1e-5, f"{irreps} C={channels} out", norm="max")
        for name, got, want in zip([k for k, n in zip("xyw", need) if n], grads, [r for r, n in zip(ref_grads, need) if n]):
            assert_close(got, want, 1e-5, f"{irreps} C={channels} grad {name} of {need}", norm="max")


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["x", "y", "w", "ct"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e38])
@pytest.mark.parametrize("channels", [32, 60, 64])
def test_values_that_are_not_finite_stay_where_they_couple(device, monkeypatch, channels, where, value):
    """An infinity, a NaN or a product that overflows: the results are those of the entry-by-entry kernels, in which a row
    reaches only the rows it couples to.  32 channels, and the one-channel-per-lane backward with and without idle lanes."""
    from equitorch_amd.nn.functional import EdgePlan, edge_tensor_product_uu
    from equitorch_amd.ops import kernels
    irreps = TABLES[1]
    src, dst, x, y, w, ct = _edge_case(irreps, channels, 40, 500, False, 7)
    {"x": x, "y": y, "w": w, "ct": ct}[where].view(-1)[123] = value
    if value == 1e38:
        {"x": x, "y": y, "w": w, "ct": ct}[where].mul_(10)
    plan = EdgePlan(src.to(device), dst.to(device), 40)
    results = {}
    for route in ("matrix", "entries"):
        info = _info(irreps).to(device)
        if route == "entries":
            monkeypatch.setattr(kernels, "_mx_words_of_content", lambda *content: None)
        wrt = [t.to(device).requires_grad_(True) for t in (x, y, w)]
        out = edge_tensor_product_uu(*wrt, plan, info)
        assert (kernels.uvu_table_of(info, wrt[0].device).mx is None) == (route == "entries")
        results[route] = (out, *torch.autograd.grad(out, wrt, ct.to(device)))
    for a, b in zip(results["matrix"], results["entries"]):
        fin = torch.isfinite(b)
        assert torch.equal(fin, torch.isfinite(a)) and torch.equal(a[~fin].nan_to_num(), b[~fin].nan_to_num())
        # in a range without a value that is not finite the sums run in another order: norm-wise
        assert float((a[fin] - b[fin]).detach().abs().max()) <= 1e-5 * float(b[fin].detach().abs().max())


@pytest.mark.parametrize("irreps", TABLES)
def test_the_wide_walk_covers_the_table(irreps):
    """The walk of the kernels with one channel per lane: the coupling matrix of every item, put back in its place, is the
    table's, every path and produced row is visited once, and the gradients of one edge formed as the kernel forms them
    (the weight gradient's rows hold another edge's values at first) are those of the table's entries."""
    from equitorch_amd.ops import kernels
    coo = kernels.coo_of(_info(irreps))
    m = kernels.uvu_mx_words(coo)
    rng = np.random.default_rng(3)
    y, C = rng.standard_normal(coo.D2), 3
    x, w, g = (rng.standard_normal(s) for s in ((coo.D1, C), (coo.P, C), (coo.DO, C)))
    gz = np.concatenate([g, np.zeros((6, C))])
    gx, gw = np.zeros((coo.D1, C)), rng.standard_normal((coo.P, C))
    f32 = lambda v: float(np.uint32(v).view(np.float32))     # noqa: E731
    for which, produced, contracted, n_prod, n_con in (("bwd", coo.M1, coo.M, coo.D1, coo.DO),):
        words, n_items, n_chunks = m[which + "4"], m[which + "4_items"], m[which + "4_chunks"]
        n_rec = m[which + "_records"]
        assert n_items % 2 == 0 and n_items <= 64 and n_chunks <= 8
        want, got = np.zeros((coo.P, n_prod, n_con)), np.zeros((coo.P, n_prod + 4, n_con + 7))
        for c, r, k, b, p in zip(coo.coef, produced, contracted, coo.M2, coo.p):
            want[p, r, k] += float(np.float32(c)) * y[b]
        A = np.zeros(32 * n_items)
        for c0, c1, k in words[:3 * n_rec].reshape(-1, 3):
            A[k >> 16] = f32(c0) * y[k & 255] + f32(c1) * y[(k >> 8) & 255]
        items = words[3 * n_rec:3 * n_rec + n_items]
        chunks = words[3 * n_rec + n_items:3 * n_rec + n_items + 8][:n_chunks]
        pair, rows_seen, paths = 0, [], set()
        for chunk in chunks:
            r0, n = int(chunk & 255), int((chunk >> 8) & 255)
            rows_seen += range(r0, r0 + n)
            while pair < (chunk >> 16):
                for h in (0, 1):
                    k = int(items[2 * pair + h])
                    p, row, rows = k & 255, (k >> 8) & 255, (k >> 16) & 15
                    assert rows in (1, 3, 5, 7) and row + rows <= n_con + 6
                    slots = A[pair * 64 + 32 * h:pair * 64 + 32 * h + 32].reshape(8, 4)
                    assert not slots[rows:].any() and not slots[:, n:].any()
                    got[p, r0:r0 + 4, row:row + rows] += slots[:rows].T
                    D = slots[:7].T[:n] @ gz[row:row + 7]
                    gx[r0:r0 + n] += w[p] * D
                    gw[p] = (gw[p] if k >> 20 & 1 else 0) + (x[r0:r0 + n] * D).sum(0)
                    if slots.any() or not k >> 20 & 1:             # all but an item that only fills a pair
                        assert bool(k >> 20 & 1) == (p in paths)        # sets the path's gradient, then adds to it
                        paths.add(p)
                pair += 1
        assert pair * 2 == n_items and sorted(rows_seen) == list(range(n_prod))
        assert paths == set(range(coo.P))
        np.testing.assert_allclose(got[:, :n_prod, :n_con], want, rtol=0, atol=1e-12)
        np.testing.assert_allclose(gx, np.einsum("prk,kc,pc->rc", want, g, w), rtol=0, atol=1e-12)
        np.testing.assert_allclose(gw, np.einsum("prk,kc,rc->pc", want, g, x), rtol=0, atol=1e-12)


# tables with some of a compiled table's paths (own paths of all): lmax 1 (2 of 4), 2 (8 of 11, 9 of 15), 3 (17, 28 of 34)
SUBSETS = [("0o+1e", "0e+1o", "0e+1e"), ("0o+1e+2o", "0e+1e+2o", "0e+1o+2e"), ("0e+1e+2e", "0e+1o+2e", "0e+1o+2e"),
           ("0e+1e+2e+3e", "0e+1e+2e+3o", "0e+1e+2o+3o"), ("0e+1e+2e+3e", "0e+1o+2o+3o", "0e+1o+2o+3o")]


def _subset_taken(irreps, channels, n_edges):
    from equitorch_amd.irreps import Irreps
    from equitorch_amd.ops import kernels
    info = _info(irreps)
    cfg = kernels.uvu_config_of(info)
    assert int(cfg) >= 0 and cfg.w_rows is not None
    x, y, w = torch.empty(16, Irreps(irreps[1]).dim, channels), torch.empty(n_edges, Irreps(irreps[2]).dim), None
    w = torch.empty(n_edges, kernels.coo_of(info).P, channels)
    return kernels.uvu_subset_table(cfg, info, x, y, w) is not None


def test_where_a_table_with_some_paths_runs_as_it_is():
    """At 64 channels and for short lists always; otherwise by the share of the compiled table's paths, by the width the
    channels are padded to.  Never where the kernels do not take the table or the channels."""
    from equitorch_amd.ops.kernels import _subset_pays
    small, p8, p9, p17, p28 = SUBSETS
    for irreps in (p8, p9, p17, p28):
        assert _subset_taken(irreps, 64, 50000) and all(_subset_taken(irreps, c, 3000) for c in (8, 16, 32, 48))
        assert not _subset_taken(irreps, 68, 1000) and not _subset_taken(irreps, 63, 1000)
    assert not _subset_taken(small, 32, 1000) and _subset_taken(small, 64, 1000)
    tables = (p8, p9, p17, p28)                                      # 0.73, 0.6, 0.5, 0.82 of the paths
    for channels, taken in ((8, (0, 0, 0, 0)), (16, (0, 0, 0, 0)), (32, (0, 1, 1, 0)), (36, (1, 1, 1, 0)), (48, (1, 1, 1, 1))):
        assert [_subset_taken(t, channels, 50000) for t in tables] == [bool(v) for v in taken], channels
    assert [_subset_taken(p9, 16, n) for n in (27777, 27778)] == [True, False]
    # a compiled table's paths in another order, or but one
    assert [_subset_pays(c, 65536, 23, 23) for c in (32, 36, 60, 64)] == [False, False, False, True]
    assert [_subset_pays(c, 65536, 10, 11) for c in (36, 48, 64)] == [False, True, True]
    assert [_subset_pays(c, 8000, 23, 23) for c in (16, 32, 36, 60)] == [True, True, False, False]


def test_where_the_walk_entry_by_entry_is_quicker():
    from equitorch_amd.ops.kernels import _mx_pays
    takes = lambda backward, nnz, n, shared=False, degree=16: [_mx_pays(backward, c, n, n // degree, nnz, shared)  # noqa: E731
                                                               for c in (1, 4, 16, 32, 48, 64)]
    for backward in (0, 1):
        assert takes(backward, 2, 1000) == takes(backward, 2, 200000) == [False] * 6
        assert takes(backward, 39, 1000) == takes(backward, 206, 16384) == [True] * 6
    assert takes(0, 39, 200000) == [False] * 5 + [True] and takes(0, 105, 200000) == [False] * 3 + [True] * 3
    assert takes(0, 206, 100000) == [False] + [True] * 5 and takes(0, 206, 200000) == [False] * 3 + [True] * 3
    assert takes(0, 351, 200000) == [False] + [True] * 5
    assert takes(1, 39, 200000) == [False] * 4 + [True] * 2 and takes(1, 70, 200000) == [False] * 3 + [True] * 3
    assert takes(1, 147, 500000) == [False] + [True] * 5
    assert takes(0, 147, 65536, degree=1) == [False] * 3 + [True] * 3 and takes(1, 147, 65536, degree=1) == [False] * 2 + [True] * 4
    assert takes(1, 39, 65536, degree=1) == [False] * 5 + [True]
    assert takes(0, 50, 200000, True) == [False] * 6 and takes(1, 50, 200000, True) == [False] * 4 + [True] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("channels,n_edges,want", [(16, 20000, [False, False]), (64, 20000, [True, True]), (48, 20000, [False, True]),
                                                   (16, 2000, [True, False])])
def test_long_lists_take_the_quicker_kernels(device, monkeypatch, channels, n_edges, want):
    """Which kernels run for 39 coefficients (forward, backward), and that the results are the oracle's."""
    from equitorch_amd import _lib
    from equitorch_amd.nn.functional import EdgePlan, edge_tensor_product_uu
    irreps = TABLES[0]
    info = _info(irreps).to(device)
    src, dst, x, y, w, ct = _edge_case(irreps, channels, 500, n_edges, False, stable_seed("quicker", channels, n_edges))
    plan = EdgePlan(src.to(device), dst.to(device), 500)
    ran = []
    for name, mx in (("cgtp_uvu_mx_fwd", True), ("cgtp_uvu_mx_bwd", True), ("cgtp_uvu_tab_fwd", False), ("cgtp_uvu_tab_bwd", False)):
        entry = getattr(_lib.lib, name)
        monkeypatch.setattr(_lib.lib, name, lambda *args, entry=entry, mx=mx: (ran.append(mx), entry(*args))[1])
    wrt = [t.to(device).requires_grad_(True) for t in (x, y, w)]
    out = edge_tensor_product_uu(*wrt, plan, info)
    grads = torch.autograd.grad(out, wrt, ct.to(device))
    assert ran == want
    T = ref_ops.dense_coupling(*irreps).float().double()

    def ref_fn(T, x, sh, w):
        return ref_ops.scatter_sum(ref_ops.dense_u1u(T, x.index_select(0, src), sh, w), dst, 500)
    ref_out, ref_grads = ref_ops.dense_grads(ref_fn, T, (x, y, w), ct)
    for name, got, ref in zip(("out", "grad x", "grad y", "grad w"), (out, *grads), (ref_out, *ref_grads)):
        assert_close(got, ref, 1e-5, f"C={channels} {name}", norm="max")


@pytest.mark.gpu
@pytest.mark.parametrize("irreps", SUBSETS)
@pytest.mark.parametrize("channels,n_nodes,n_edges", [(64, 40, 700), (36, 3, 2000), (24, 300, 900), (8, 30, 400)])
def test_a_table_with_some_paths_on_both_routes(device, monkeypatch, irreps, channels, n_nodes, n_edges):
    """As it is and on the compiled table with expanded weights, both against the oracle."""
    from equitorch_amd.nn.functional import EdgePlan, edge_tensor_product_uu
    from equitorch_amd.ops import kernels
    info = _info(irreps).to(device)
    src, dst, x, y, w, ct = _edge_case(irreps, channels, n_nodes, n_edges, False, stable_seed("subset", irreps, channels))
    plan = EdgePlan(src.to(device), dst.to(device), n_nodes)
    T = ref_ops.dense_coupling(*irreps).float().double()

    def ref_fn(T, x, sh, w):
        return ref_ops.scatter_sum(ref_ops.dense_u1u(T, x.index_select(0, src), sh, w), dst, n_nodes)
    ref_out, ref_grads = ref_ops.dense_grads(ref_fn, T, (x, y, w), ct)
    launches = []
    launch = kernels._uvu_tab_launch
    monkeypatch.setattr(kernels, "_uvu_tab_launch", lambda *args: (launches.append(1), launch(*args)))
    for route in ("as it is", "expanded"):
        if route == "expanded":
            monkeypatch.setattr(kernels, "uvu_subset_table", lambda *args: None)
        wrt = [t.to(device).requires_grad_(True) for t in (x, y, w)]
        out = edge_tensor_product_uu(*wrt, plan, info)
        grads = torch.autograd.grad(out, wrt, ct.to(device))
        for name, got, want in zip(("out", "grad x", "grad y", "grad w"), (out, *grads), (ref_out, *ref_grads)):
            assert_close(got, want, 1e-5, f"{irreps} C={channels} {route}: {name}", norm="max")
        assert len(launches) == (2 if route == "as it is" and (channels > 32 or irreps != SUBSETS[0]) else 0)
        launches.clear()


@pytest.mark.gpu
def test_recorded_in_a_graph(device, monkeypatch):
    """Forward and gradients recorded into a HIP graph and replayed on new inputs, eager work in between: the flags of the
    ranges are written anew by every replay (the second one sees a value that is not finite, the third none again)."""
    from equitorch_amd.nn.functional import EdgePlan, edge_tensor_product_uu
    from equitorch_amd.ops import kernels
    info = _info(TABLES[1]).to(device)
    src, dst, x, y, w, ct = _edge_case(TABLES[1], 64, 40, 700, False, 9)
    plan = EdgePlan(src.to(device), dst.to(device), 40)
    inputs = [t.to(device).requires_grad_(True) for t in (x, y, w)]
    ct = ct.to(device)

    def step():
        out = edge_tensor_product_uu(*inputs, plan, info)
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
                t.copy_(torch.randn(t.shape, generator=torch.Generator().manual_seed(replay)))
            if replay == 1:
                inputs[0][3, 2, 5] = float("inf")
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(recorded, step()):
            assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num()), replay
        # the walk entry by entry: values that are not finite at the same places
        with monkeypatch.context() as m:
            m.setattr(kernels, "_mx_pays", lambda *args: False)
            for a, b in zip(recorded, step()):
                fin = torch.isfinite(b)
                assert torch.equal(fin, torch.isfinite(a)), replay
                assert float((a[fin] - b[fin]).detach().abs().max()) <= 1e-5 * float(b[fin].detach().abs().max()), replay
