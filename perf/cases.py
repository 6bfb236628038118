"""The work this library is timed on: what a user's program has it do through its public entry points.

``listed()`` gives twelve fixed cases, ``draw(rng)`` one more of the same ranges; ``prepare`` makes what the program
holds before the call, ``run`` is one pass, ``work`` the bytes and operations it cannot do without, and ``tolerance``
how far two correct implementations at the same precision may be apart.

Kinds of case:

* ``edge``       message passing: gather at the source, channel-wise product with the edge harmonics and a weight per
                 edge, sum to the destination.  ``step`` is forward and all gradients (training), ``forward`` inference.
* ``batch``      the channel-wise product on a plain batch of rows with a shared weight, forward and all gradients.
* ``layer``      a whole message-passing layer built from the modules, forward and backward, launched eagerly.
* ``uv``         the fully connected product, channels of the first operand only, a shared weight or one per sample.
* ``uvw``        the fully connected product of two channelled operands, shared weight.
* ``so2``        features of an edge turned into the edge's frame, mixed by an SO(2) layer and turned back.
"""
import functools
import math

import torch

from equitorch_amd import nn as enn
from equitorch_amd.irreps import Irreps
from equitorch_amd.nn.functional import (EdgePlan, edge_tensor_product_uu, edge_tensor_product_uu_radial,
                                         edge_tensor_product_uu_vectors, sincos, spherical_harmonics)

# Irreps triples (out, in1, in2) that no compiled table covers: a user's own choice of features.
OWN_IRREPS = ("0e+1o+2e+3o < 1o+2e+3o < 0e+1o+2e", "0e+1o+2e < 0e+1o < 0e+1o+2e+3o", "0e+1e+2e < 0e+1o+2e < 0e+1o+2e")

LAYER_BASIS, LAYER_HIDDEN, LAYER_CUTOFF = 8, 16, 3.0


def _sh_irreps(lmax):
    return "+".join(f"{l}{'e' if l % 2 == 0 else 'o'}" for l in range(lmax + 1))


def listed():
    return [
        # One small molecule at inference: a call of a few microseconds, bound by launches and host work.
        {"name": "edge_molecule_forward", "kind": "edge", "lmax": 2, "channels": 64, "nodes": 30, "edges": 420,
         "graph": "uniform", "operand": "vectors", "pass": "forward"},
        # A small batch of rows through a module with its own weight (a readout head, a unit-test sized model).
        {"name": "batch_small_step", "kind": "batch", "lmax": 2, "channels": 16, "rows": 1024},
        # The ordinary training step of a message-passing model: the benchmark's headline workload.
        {"name": "edge_l2_step", "kind": "edge", "lmax": 2, "channels": 64, "nodes": 4096, "edges": 65536,
         "graph": "uniform", "operand": "harmonics", "pass": "step"},
        # A bulk structure whose atoms are ordered in space, ragged sizes, harmonics evaluated inside the kernels.
        {"name": "edge_l3_ragged_step", "kind": "edge", "lmax": 3, "channels": 64, "nodes": 3001, "edges": 47917,
         "graph": "local", "operand": "vectors", "pass": "step"},
        # High degrees: large coupling tables, few channels.
        {"name": "edge_l6_step", "kind": "edge", "lmax": 6, "channels": 32, "nodes": 20000, "edges": 200000,
         "graph": "uniform", "operand": "harmonics", "pass": "step"},
        # Irreps of the user's own choice, for which no table is compiled in.
        {"name": "edge_own_irreps_step", "kind": "edge", "irreps": OWN_IRREPS[0], "channels": 64, "nodes": 4096,
         "edges": 65536, "graph": "uniform", "operand": "harmonics", "pass": "step"},
        # A layer as a model stacks it: radial basis and network, edge product, channel mixing, gate, norm.
        {"name": "layer_step", "kind": "layer", "channels": 64, "nodes": 4096, "edges": 65536, "graph": "uniform"},
        # Fully connected product with a shared weight in mixed-precision training.
        {"name": "uv_bf16_step", "kind": "uv", "lmax": 3, "channels": 128, "rows": 32768, "dtype": "bf16",
         "weight": "shared"},
        # The same module in single precision.
        {"name": "uv_f32_step", "kind": "uv", "lmax": 3, "channels": 128, "rows": 32768, "dtype": "f32",
         "weight": "shared"},
        # A weight per sample from a radial network: a stream over the weights.
        {"name": "uv_per_sample_step", "kind": "uv", "lmax": 2, "channels": 16, "rows": 65536, "dtype": "f32",
         "weight": "per_sample"},
        # Product of two channelled features (self-interaction of node features).
        {"name": "uvw_f32_step", "kind": "uvw", "lmax": 2, "channels": 32, "rows": 32768},
        # Convolution in the edge frame.
        {"name": "so2_edge_step", "kind": "so2", "lmax": 4, "channels": 64, "rows": 32768},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["edge", "edge", "edge", "edge_high", "edge_own", "batch", "layer", "uv", "uv", "per_sample",
                       "uvw", "so2"])
    if kind in ("edge", "edge_high", "edge_own"):
        case = {"kind": "edge", "graph": rng.choice(["uniform", "local"]), "operand": "harmonics",
                "pass": rng.choice(["step", "step", "forward"])}
        if kind == "edge":
            case["lmax"], case["channels"] = rng.randint(1, 4), rng.choice([16, 32, 48, 64, 96, 128])
            case["operand"] = rng.choice(["harmonics", "vectors"])
            most = 5e8 / (4 * _table(case)["paths"] * case["channels"])       # the weights of all edges: 500 MB
            case["edges"] = _log(rng, 300, min(200000, most))
        elif kind == "edge_high":
            case["lmax"], case["channels"] = rng.randint(5, 6), rng.choice([16, 24, 32])
            case["edges"] = _log(rng, 5000, 100000)
        else:
            case["irreps"], case["channels"] = rng.choice(OWN_IRREPS), rng.choice([16, 32, 48, 64])
            case["edges"] = _log(rng, 3000, 65536)
        case["nodes"] = max(16, int(case["edges"] / rng.uniform(8, 40)))
        return case
    if kind == "batch":
        return {"kind": "batch", "lmax": rng.randint(1, 3), "channels": rng.choice([8, 16, 32, 64]),
                "rows": _log(rng, 64, 65536)}
    if kind == "layer":
        edges = _log(rng, 2000, 65536)
        return {"kind": "layer", "channels": rng.choice([32, 64, 64]), "edges": edges,
                "nodes": max(16, int(edges / rng.uniform(8, 40))), "graph": rng.choice(["uniform", "local"])}
    if kind == "uv":
        return {"kind": "uv", "lmax": rng.randint(1, 3), "channels": rng.choice([32, 48, 64, 96, 128]),
                "rows": _log(rng, 500, 32768), "dtype": rng.choice(["bf16", "f32"]), "weight": "shared"}
    if kind == "per_sample":
        case = {"kind": "uv", "lmax": rng.randint(1, 2), "channels": rng.choice([8, 16, 24, 32]), "dtype": "f32",
                "weight": "per_sample"}
        most = 7e8 / (4 * _table(case)["paths"] * case["channels"] ** 2)
        case["rows"] = _log(rng, 1000, min(65536, most))
        return case
    if kind == "uvw":
        return {"kind": "uvw", "lmax": rng.randint(1, 2), "channels": rng.choice([8, 16, 24, 32]),
                "rows": _log(rng, 500, 32768)}
    return {"kind": "so2", "lmax": rng.randint(2, 6), "channels": rng.choice([32, 48, 64]),
            "rows": _log(rng, 1000, 16384)}


# ---- the products' tables: sizes for `work` and `draw`, modules for `prepare` ------------------------------------------
def _triple(case):
    if "irreps" in case:
        return tuple(s.strip() for s in case["irreps"].split("<"))
    return (_sh_irreps(case["lmax"]),) * 3


@functools.lru_cache(maxsize=None)
def _table_sizes(out, in1, in2):
    mod = enn.SO3Linear(in1, in2, out, internal_weights=False, feature_mode="uu")
    coupling = mod.tp_info_forward.info_Mij_fwd       # its segments are the (path, output row) pairs
    return {"out": Irreps(out).dim, "in1": Irreps(in1).dim, "in2": Irreps(in2).dim, "paths": mod.num_paths,
            "coefficients": int(coupling.scale.shape[0]), "rows": int(coupling.out_size)}


def _table(case):
    return _table_sizes(*_triple(case))


def _edges(case, gen, dev):
    n, e = case["nodes"], case["edges"]
    dst = torch.randint(0, n, (e,), generator=gen, device=dev)
    if case["graph"] == "local":       # atoms ordered in space: an edge starts within 64 ids of where it ends
        src = (dst + torch.randint(-64, 65, (e,), generator=gen, device=dev)) % n
    else:
        src = torch.randint(0, n, (e,), generator=gen, device=dev)
    return EdgePlan(src, dst, n)


def _unit(n, gen, dev):
    v = torch.randn(n, 3, generator=gen, device=dev)
    return v / v.norm(dim=-1, keepdim=True).clamp_min(1e-6)


class _Layer(torch.nn.Module):
    """Radial basis and cutoff, radial network (its last linear inside the edge kernels), edge product with the
    harmonics evaluated in place, channel mixing, gate, norm."""

    def __init__(self, c):
        super().__init__()
        irr = _sh_irreps(2)
        self.c = c
        self.basis = enn.BesselBasis(LAYER_CUTOFF, LAYER_BASIS, trainable=False)
        self.cutoff = enn.PolynomialCutoff(LAYER_CUTOFF)
        self.tp = enn.SO3Linear(irr, irr, irr, c, c, internal_weights=False, feature_mode="uu")
        self.hidden = torch.nn.Sequential(torch.nn.Linear(LAYER_BASIS, LAYER_HIDDEN), torch.nn.SiLU())
        self.last = torch.nn.Linear(LAYER_HIDDEN, self.tp.num_paths * c, bias=False)
        self.mix = enn.IrrepsLinear(irr, irr, c, c)
        self.gate_lin = enn.IrrepsLinear(irr, "0e+0e+0e", c, c)
        self.gate = enn.Gate(irr, activation=torch.nn.Sigmoid())
        self.norm = enn.LayerRMSNorm(irr, c)

    def forward(self, x, edge_vec, plan):
        r = edge_vec.norm(dim=-1)
        feat = self.hidden(self.basis(r) * self.cutoff(r)[:, None])
        w_last = self.last.weight.t().reshape(LAYER_HIDDEN, self.tp.num_paths, self.c)
        msg = edge_tensor_product_uu_radial(x, edge_vec, feat, w_last, plan, self.tp.tp_info_forward, edge_vectors=True)
        h = self.mix(msg)
        return self.norm(self.gate(h, self.gate_lin(h)))


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    torch.manual_seed(seed)            # the modules' own initialisation

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    kind, c = case["kind"], case["channels"]
    s = {"case": case}
    if kind == "edge":
        t = _table(case)
        out, in1, in2 = _triple(case)
        s["mod"] = enn.SO3Linear(in1, in2, out, c, c, internal_weights=False, feature_mode="uu").to(dev)
        s["plan"] = _edges(case, gen, dev)
        vec = _unit(case["edges"], gen, dev)
        if case["operand"] == "vectors":
            y = vec * (0.5 + torch.rand(case["edges"], 1, generator=gen, device=dev))
        else:
            degrees = [ir.l for ir in Irreps(in2)]
            y = spherical_harmonics(vec, max(degrees))[:, :t["in2"]].contiguous()
        s["wrt"] = [randn(case["nodes"], t["in1"], c), y, randn(case["edges"], t["paths"], c)]
        s["ct"] = randn(case["nodes"], t["out"], c)
    elif kind == "batch":
        irr = _sh_irreps(case["lmax"])
        s["mod"] = enn.SO3Linear(irr, irr, irr, c, c, feature_mode="uu").to(dev)
        y = spherical_harmonics(_unit(case["rows"], gen, dev), case["lmax"])
        s["wrt"] = [randn(case["rows"], y.shape[1], c), y]
        s["ct"] = randn(case["rows"], y.shape[1], c)
    elif kind == "layer":
        s["mod"] = _Layer(c).to(dev)
        s["plan"] = _edges(case, gen, dev)
        s["wrt"] = [randn(case["nodes"], 9, c), randn(case["edges"], 3) * 1.2]
        s["ct"] = randn(case["nodes"], 9, c)
    elif kind == "uv":
        irr, n = _sh_irreps(case["lmax"]), case["rows"]
        dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        mod = enn.SO3Linear(irr, irr, irr, c, c, internal_weights=False, feature_mode="uv").to(dev)
        y = spherical_harmonics(_unit(n, gen, dev), case["lmax"])
        lead = (n,) if case["weight"] == "per_sample" else ()
        w = randn(*lead, mod.num_paths, c, c).mul_((c * mod.num_paths) ** -0.5)
        s["mod"] = mod
        s["wrt"] = [randn(n, y.shape[1], c).to(dtype), y.to(dtype), w.to(dtype)]
        s["ct"] = randn(n, y.shape[1], c).to(dtype)
    elif kind == "uvw":
        irr, n = _sh_irreps(case["lmax"]), case["rows"]
        d = Irreps(irr).dim
        s["mod"] = enn.TensorProduct(irr, irr, irr, c, c, c, feature_mode="uvw", internal_weights=False).to(dev)
        s["wrt"] = [randn(n, d, c), randn(n, d, c), randn(s["mod"].num_paths, c, c, c) / c]
        s["ct"] = randn(n, d, c)
    else:
        irr, n, lmax = _sh_irreps(case["lmax"]), case["rows"], case["lmax"]
        d = Irreps(irr).dim
        s["rotation"] = enn.SparseWignerRotation(irr).to(dev)
        s["mod"] = enn.SO2Linear(irr, irr, c, c, feature_mode="uv").to(dev)
        v = _unit(n, gen, dev)
        theta, phi = torch.acos(v[:, 2].clamp(-1, 1)), torch.atan2(v[:, 1], v[:, 0])
        s["to_edge"] = (None, sincos(-theta, lmax), sincos(-phi, lmax))
        s["from_edge"] = (sincos(phi, lmax), sincos(theta, lmax), None)
        s["wrt"] = [randn(n, d, c)]
        s["ct"] = randn(n, d, c)
    if case.get("pass") != "forward":
        s["wrt"] = [t.requires_grad_(True) for t in s["wrt"]]
        s["parameters"] = list(s["mod"].parameters())
    return s


def _forward(s):
    case, mod, wrt = s["case"], s["mod"], s["wrt"]
    kind = case["kind"]
    if kind == "edge":
        product = edge_tensor_product_uu_vectors if case["operand"] == "vectors" else edge_tensor_product_uu
        return product(*wrt, s["plan"], mod.tp_info_forward)
    if kind == "layer":
        return mod(*wrt, s["plan"])
    if kind == "so2":
        return s["rotation"](mod(s["rotation"](wrt[0], *s["to_edge"])), *s["from_edge"])
    return mod(*wrt)


def run(s):
    if s["case"].get("pass") == "forward":
        with torch.no_grad():
            return _forward(s)
    out = _forward(s)
    return (out, *torch.autograd.grad(out, s["wrt"] + s["parameters"], s["ct"]))


def work(case):
    kind, c = case["kind"], case["channels"]
    f = 4
    if kind == "edge":
        t, e, n = _table(case), case["edges"], case["nodes"]
        y = 3 if case["operand"] == "vectors" else t["in2"]
        w, nx, no, ys, idx = e * t["paths"] * c * f, n * t["in1"] * c * f, n * t["out"] * c * f, e * y * f, 16 * e
        nbytes, flops = w + nx + no + ys + idx, 2.0 * e * c * (t["coefficients"] + t["rows"])
        if case["pass"] == "step":
            nbytes += (w + nx + no + ys + idx) + (w + nx + ys)
            flops *= 4
        return {"bytes": nbytes, "flops": flops}
    if kind == "batch":
        t, n = _table(case), case["rows"]
        rows = n * c * f
        nbytes = rows * (t["in1"] + t["out"]) + rows * (2 * t["in1"] + t["out"]) + 3 * n * t["in2"] * f
        return {"bytes": nbytes + 3 * t["paths"] * c * f, "flops": 8.0 * n * c * (t["coefficients"] + t["rows"])}
    if kind == "layer":
        t, e, n = _table_sizes(*(_sh_irreps(2),) * 3), case["edges"], case["nodes"]
        node = n * 9 * c * f
        per_edge = (3 + 1 + LAYER_BASIS + LAYER_HIDDEN) * f + 16
        # the weights of an edge never need to be in memory: they are formed from its radial features, and so are
        # their gradients contracted; node tensors: product, mixing, gate, norm, each once in each direction
        flops = 8.0 * e * c * (t["coefficients"] + t["rows"]) + 6.0 * e * t["paths"] * c * LAYER_HIDDEN \
            + 6.0 * n * c * c * 12
        return {"bytes": 3 * e * per_edge + node * (2 + 3 * 2 + 3 * 3), "flops": flops}
    if kind == "uv":
        t, n = _table(case), case["rows"]
        b = 2 if case["dtype"] == "bf16" else 4
        w = t["paths"] * c * c * b * (n if case["weight"] == "per_sample" else 1)
        x, o, y = n * t["in1"] * c * b, n * t["out"] * c * b, n * t["in2"] * b
        return {"bytes": (x + y + w + o) + (x + y + w + o) + (x + y + w), "flops": 4 * 2.0 * n * t["rows"] * c * c}
    if kind == "uvw":
        t, n = _table(case), case["rows"]
        w, x, y, o = t["paths"] * c ** 3 * f, n * t["in1"] * c * f, n * t["in2"] * c * f, n * t["out"] * c * f
        return {"bytes": (x + y + w + o) + (x + y + w + o) + (x + y + w), "flops": 4 * 2.0 * n * t["rows"] * c ** 3}
    lmax, n = case["lmax"], case["rows"]
    d = (lmax + 1) ** 2
    row = n * d * c * f
    # components of order m: one for m = 0, a pair for m > 0, of every degree l >= m
    entries = (lmax + 1) ** 2 + sum(4 * (lmax + 1 - m) ** 2 for m in range(1, lmax + 1))
    turn = sum(2.0 * (2 * l + 1) ** 2 for l in range(lmax + 1)) * n * c
    # the input is read and the output written once each way, the SO(2) layer's input is kept for its weight gradient
    return {"bytes": 6 * row, "flops": 3 * 2.0 * n * entries * c * c + 4 * turn}


def tolerance(case):
    """About four times what the path differs by from itself in float64 (from float64 arithmetic on the same rounded
    operands for bf16), over outputs and gradients: 2.3e-3 and 1.2e-2 at most in bf16; in fp32 2.1e-7 and 2.6e-6 for
    sums over a table and the edges of a node, 1.3e-6 and 1.1e-5 where channels, rows or a chain of modules are summed."""
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 5e-2}
    if case["kind"] == "edge" or case.get("weight") == "per_sample":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 5e-6, "max": 5e-5}
