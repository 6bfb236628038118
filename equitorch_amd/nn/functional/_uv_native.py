"""Fully connected products in fp32 with a shared weight on the table-driven matrix-core kernels (``cgtp_uvt_*``):
``tensor_product_u1v`` (``SO3Linear('uv')``) and ``tensor_product_uvw`` (``TensorProduct('uvw')``) for any irreps and
normalisation, forward and first-order gradients, without the reference's ``(N, segments, C)`` intermediate
(``equitorch/nn/functional/linears.py:257-336``, ``tensor_products.py:92-172``).

The kernels walk a flat list of items (segment = (weight path, output row), chunk of the contracted channel axis)
ordered by output row; this module cuts that list from the table for each of the roles a product is used in:

    forward      out[M]   <- first operand rows M1, second operand rows M2, weight as stored
    grad first   g1[M1]   <- rows M of grad_out,   second operand rows M2, weight transposed
    ('uvw' only) g2[M2]   <- rows M of grad_out,   first operand rows M1,  weight permuted
"""
import ctypes as C
import functools
import heapq
from typing import NamedTuple, Optional

import numpy as np
import torch
from torch import Tensor
from torch.autograd import Function

from ... import _lib
from ..._tables import TpCoo
from ...ops import kernels

FIRST, LAST = 1, 2


class CooTable:
    """A product table given directly by its coordinates (``coo``: ``TpCoo`` fields M, M1, M2, p, coef and the extents)
    instead of a ``TensorProductInfo`` — the tables of the channel-mixing layers, whose second operand is the scalar 1.
    ``anchor``: a tensor that lives as long as the table (cache key); ``fallback(x, y, w)``: a differentiable
    evaluation of the same product for gradients of higher order.  ``mixing``: the second operand is the scalar 1 in every
    sample (channel mixing).  ``algebra``: the fallback is tensor algebra, which takes gradients that are batched or traced."""

    def __init__(self, coo, anchor: Tensor, fallback, mixing: bool = False, algebra: bool = False):
        self.coo, self.anchor, self.fallback, self.mixing, self.algebra = coo, anchor, fallback, mixing, algebra


def _anchor(table) -> Tensor:
    return table.anchor if isinstance(table, CooTable) else table.info_Mij_fwd.scale
MAX_TERMS = 8      # terms of a segment the weight-gradient kernel holds in registers (kUvtTerms)


class _Coefficients:
    """The coefficients of a walk's terms as a device tensor of the launch's dtype (made on first use)."""

    def term_c(self, dtype: torch.dtype) -> Tensor:
        if dtype not in self._term_c:
            self._term_c[dtype] = torch.from_numpy(np.ascontiguousarray(self._coef, dtype=np.float64)).to(
                device=self._device, dtype=dtype)
        return self._term_c[dtype]


class _Walk(_Coefficients):
    """Item list of one role of one table: one item per segment (weight path, output row), the items of a row
    consecutive, the rows dealt to ``n_groups`` groups of about equal numbers of items (the wavefronts of a workgroup
    take one group each)."""

    def __init__(self, out_idx, a_idx, b_idx, p_idx, coef, n_out: int, n_groups: int, device):
        order = np.lexsort([b_idx, a_idx, p_idx, out_idx])
        out_idx, a_idx, b_idx, p_idx = (np.asarray(v)[order] for v in (out_idx, a_idx, b_idx, p_idx))
        coef = np.asarray(coef, dtype=np.float64)[order]
        rows = []
        t, n_terms = 0, out_idx.shape[0]
        for row in range(n_out):
            items = []
            while t < n_terms and out_idx[t] == row:
                t1 = t
                while t1 < n_terms and out_idx[t1] == row and p_idx[t1] == p_idx[t]:
                    t1 += 1
                items.append([int(p_idx[t]), 0, 0, t, t1, row, 0, 0])
                t = t1
            if not items:                                  # a row without terms is written as zeros
                items.append([0, 0, 0, 0, 0, row, 0, 0])
            items[0][6] |= FIRST
            items[-1][6] |= LAST
            rows.append(items)
        # longest rows first, each to the group with the fewest items so far
        groups = [[] for _ in range(n_groups)]
        for items in sorted(rows, key=len, reverse=True):
            min(groups, key=len).extend(items)
        flat = [it for grp in groups for it in grp]
        self.n_items = len(flat)
        self.group_ptr = np.cumsum([0] + [len(grp) for grp in groups]).tolist()
        self.items = torch.tensor(flat, dtype=torch.int32).reshape(-1, 8).to(device)
        self.term_a = torch.from_numpy(a_idx.astype(np.int32)).to(device)
        self.term_b = torch.from_numpy(b_idx.astype(np.int32)).to(device)
        self._coef, self._device, self._term_c = coef, device, {}


def _walk(tp_info, role: str, n_groups: int, device) -> _Walk:
    def build():
        c = _coo(tp_info)
        if role == "out":        # rows of the first operand, rows of the second operand
            return _Walk(c.M, c.M1, c.M2, c.p, c.coef, c.DO, n_groups, device)
        if role == "in1":        # first operand of the launch = grad_out, second = input2
            return _Walk(c.M1, c.M, c.M2, c.p, c.coef, c.D1, n_groups, device)
        if role == "in1_uvw":    # first operand of the launch = input2, second = grad_out
            return _Walk(c.M1, c.M2, c.M, c.p, c.coef, c.D1, n_groups, device)
        if role == "in2_uvw":    # first operand of the launch = grad_out, second = input1
            return _Walk(c.M2, c.M, c.M1, c.p, c.coef, c.D2, n_groups, device)
        raise ValueError(role)
    return kernels.cached(_anchor(tp_info), ("uvt_walk", role, n_groups, str(device)), build)


class _PathWalk(_Coefficients):
    """Segments (weight path, output row) of a table sorted by path, with their terms: the walk of the weight-gradient
    kernel, which owns one path per workgroup."""

    def __init__(self, coo, device):
        order = np.lexsort([coo.M2, coo.M1, coo.M, coo.p])
        p_idx, m_idx, a_idx, b_idx = (np.asarray(v)[order] for v in (coo.p, coo.M, coo.M1, coo.M2))
        coef = np.asarray(coo.coef, dtype=np.float64)[order]
        items, path_ptr = [], [0]
        t, n_terms = 0, p_idx.shape[0]
        for p in range(coo.P):
            while t < n_terms and p_idx[t] == p:
                t1 = t
                while t1 < n_terms and p_idx[t1] == p and m_idx[t1] == m_idx[t]:
                    t1 += 1
                for tb in range(t, t1, MAX_TERMS):       # the kernel keeps at most MAX_TERMS terms of an item
                    items.append([p, 0, 0, tb, min(tb + MAX_TERMS, t1), int(m_idx[t]), 0, 0])
                t = t1
            path_ptr.append(len(items))
        self.n_items, self.n_terms, self.n_paths = len(items), n_terms, coo.P
        self.items = torch.tensor(items, dtype=torch.int32).reshape(-1, 8).to(device)
        self.path_ptr = torch.tensor(path_ptr, dtype=torch.int32).to(device)
        self.term_a = torch.from_numpy(a_idx.astype(np.int32)).to(device)
        self.term_b = torch.from_numpy(b_idx.astype(np.int32)).to(device)
        self._coef, self._device, self._term_c = coef, device, {}


class _MixPairs:
    """The (row of the input, row of the result, coefficient) of every weight of a channel-mixing table."""

    def __init__(self, coo, device):
        order = np.lexsort([coo.M, coo.M1, coo.p])
        pairs = np.zeros((len(order), 4), dtype=np.int32)
        pairs[:, 0], pairs[:, 1] = np.asarray(coo.M1)[order], np.asarray(coo.M)[order]
        pairs[:, 2] = np.asarray(coo.coef)[order].astype(np.float32).view(np.int32)
        ptr = np.searchsorted(np.asarray(coo.p)[order], np.arange(coo.P + 1)).astype(np.int32)
        self.words, self.ptr_at = torch.from_numpy(np.concatenate([pairs.ravel(), ptr])).to(device), 4 * pairs.size
        self.max_pairs = int(np.diff(ptr).max())


def _mix_grad_w(x: Tensor, g: Tensor, table) -> Optional[Tensor]:
    """:func:`grad_w` of channel mixing in fp32 on the half-precision matrix cores (``cgtp_uvl_grad_w``), or None where the fp32
    matrix instructions serve: past 128 channels, where their blocks of 128 x 128 read the rows less often (256 -> 256, 4096
    samples: 69 us against 78), and for the same reason past 64 with the few single pairs of SO2Linear of lmax 1 (six paths, eight
    pairs; 128 channels, 4096 samples 32.5 us against 29.4, 65536 203 against 180; lmax 2, 19 and 29: 54.9 against 64.6 and 539 against
    620).  IrrepsLinear and SO2Linear, 8 to 128 channels, 500 to 65536 samples: 0.5 to 1.0 of their time (SO2Linear of lmax 2, 64 channels, 2000
    samples 1.05).  Tables that were products of the library stay here past 128 channels below 512 samples: its sums are more precise there
    than those of the fp32 instructions (SO2Linear, lmax 6, 256 channels, 300 samples: library 3.1e-7, fp32 instructions 3.8e-7, here 0.9e-7;
    IrrepsLinear, lmax 4, 256 -> 64, 40 samples 1.2e-7, 2.4e-7, 0.7e-7; from 512 samples on 4.05e-7 and 4.03e-7), for 708 us against 327 in the first and 31
    against 49 in the second layer, whose steps still take less than the library's."""
    if not (isinstance(table, CooTable) and table.mixing) or x.dtype != torch.float32 or x.shape[0] == 0:
        return None
    (n, dx, cx), (_, dg, cout), n_paths = x.shape, g.shape, table.coo.P
    if max(cx, cout) > 128 and (n >= 512 or not _was_the_library(n, cx, cout, table)):
        return None
    if min(cx, cout) > 64 and n_paths <= 8 and len(table.coo.p) < 2 * n_paths and n > 2000:
        return None
    pairs = kernels.cached(_anchor(table), ("uvl_pairs", str(x.device)), lambda: _MixPairs(table.coo, x.device))
    gw = torch.empty((n_paths, cx, cout), dtype=x.dtype, device=x.device)
    a = _lib.UvlGwArgs(x.data_ptr(), g.data_ptr(), gw.data_ptr(), 0, pairs.words.data_ptr(), pairs.words.data_ptr() + pairs.ptr_at, n,
                       n_paths, pairs.max_pairs, dx, dg, cx, cout)
    size = int(_lib.lib.cgtp_uvl_grad_w_workspace_bytes(C.byref(a)))
    if size <= 0:
        return None
    ws = torch.empty(size, dtype=torch.uint8, device=x.device)
    a.workspace = ws.data_ptr()
    _lib.check(_lib.lib.cgtp_uvl_grad_w(C.byref(a), _lib.stream_ptr(x.device)), "cgtp_uvl_grad_w")
    return gw


class _GradWWalk:
    """The work of ``cgtp_uvg_apply`` for a table, dealt to ``n_wgs`` workgroups."""
    SHARES = 64

    def __init__(self, coo, n_wgs: int, device):
        words, self.at, self.n_slots = _grad_w_words(n_wgs, int(coo.P), *(np.ascontiguousarray(v, dtype=np.int32).tobytes()
                                                                          for v in (coo.M, coo.M1, coo.p)))
        self.words, self.n_paths = torch.tensor(words, device=device), coo.P

    def ranges(self, steps: int) -> int:
        """Ranges the steps are cut into, each with slots of its own: 128 steps or more in each, and no more than the fp32 kernel has
        partial results (128 of every path) where the eight of the XCDs leave room for it: 155 MB for "uvw", lmax 2, 32 channels,
        past 32768 samples.  (With ranges of 128 steps throughout 1.24 GB at 262144 samples, 5946 us against 6823; lmax 1 1478
        against 1424, without channels on y the same; fp32 instructions 1310 at 32768 samples, here 820.)"""
        return 8 * max(1, min(steps // 1024, 16 * self.n_paths // self.n_slots))

    @classmethod
    def deal(cls, cost, n_wgs: int):
        """Per workgroup its ``(path, mask)``: the 64 shares of every path, dealt in the order of the paths so that all
        workgroups carry the same cost, the shares of a path spread over its steps."""
        room = sum(cost) * cls.SHARES / n_wgs
        portions_of, w, left = [], 0, room
        for c in cost:
            todo, portions = cls.SHARES, []
            while todo:
                take = min(todo, max(0, int(left / c + 0.5))) if w < n_wgs - 1 else todo
                if take:
                    portions.append((w, take))
                    todo -= take
                    left -= take * c
                if todo:
                    w, left = w + 1, left + room           # what was taken too much or too little carries over
            portions_of.append(portions)
        most = max(map(len, portions_of))
        takes = np.array([[take for _, take in portions] + [0] * (most - len(portions)) for portions in portions_of])
        jobs = [[] for _ in range(n_wgs)]
        for p, masks in enumerate(cls.masks(takes)):
            for (g, _), mask in zip(portions_of[p], masks):
                jobs[g].append((p, mask))
        return jobs

    @classmethod
    def masks(cls, takes):
        """``takes``: a row of portions for each path, filled up with zeros.  A bit for each of a path's shares to the portion
        that is most behind its part of them."""
        behind, at, owner = np.zeros_like(takes), np.arange(len(takes)), np.zeros((len(takes), cls.SHARES), dtype=np.int64)
        for bit in range(cls.SHARES):
            behind += takes
            owner[:, bit] = k = behind.argmax(axis=1)
            behind[at, k] -= cls.SHARES
        bits = owner[:, None, :] == np.arange(takes.shape[1])[:, None]
        return np.packbits(bits, axis=-1, bitorder="little").view("<u8")[..., 0].tolist()


@functools.lru_cache(maxsize=32)
def _grad_w_words(n_wgs: int, n_paths: int, *indices: bytes):
    """The arrays of a :class:`_GradWWalk` by the table's content (host work that a second module of the table does not
    repeat): jobs, their places by workgroup and the slots by path in one array, where each begins in bytes, slots."""
    M, M1, path = (np.frombuffer(v, dtype=np.int32).astype(np.int64) for v in indices)

    def rows(idx):
        return np.bincount(np.unique(path << 32 | idx) >> 32, minlength=n_paths)
    # of a step: its products (as many as the side with fewer rows has), and the rows that are read
    cost = (np.minimum(rows(M1), rows(M)) + 0.15 * (rows(M1) + rows(M))).tolist()
    jobs = _GradWWalk.deal(cost, n_wgs)
    by_path = sorted((p, w) for w, mine in enumerate(jobs) for p, _ in mine)
    slots = {job: k for k, job in enumerate(by_path)}
    flat = [(p, slots[p, w], mask & 0xffffffff, mask >> 32) for w, mine in enumerate(jobs) for p, mask in mine]
    parts = [np.array(flat, dtype=np.uint32).view(np.int32), np.cumsum([0] + [len(mine) for mine in jobs]).astype(np.int32),
             np.searchsorted([p for p, _ in by_path], np.arange(n_paths + 1)).astype(np.int32)]
    return np.concatenate([v.ravel() for v in parts]), [4 * sum(v.size for v in parts[:k]) for k in range(len(parts))], len(slots)



def _split_grad_w(x: Tensor, y: Tensor, g: Tensor, tp_info) -> Optional[Tensor]:
    """:func:`grad_w` in fp32 on the half-precision matrix cores (``cgtp_uvg_apply``), or None where the fp32 matrix
    instructions serve: tables that are not compiled in as they are, different numbers of channels, and where they are
    quicker or more precise.  Without channels on ``y`` that is up to 64 channels (8192 samples, lmax 3: 91 us against 148, but
    errors of 3.7e-7 against 2.8e-7), lmax 1 (4000 samples, 128 channels: 38 us against 28) and small batches (lmax 3, 1000
    samples, 128 channels 77 us against 67; up to 4096 samples equal errors); with channels, below 24 of them (16: 128 us against 110; 20: 417 and 405) and
    small batches (lmax 2, 1000 samples 107 us against 77; lmax 1, 2100 samples 50 and 44)."""
    if isinstance(tp_info, CooTable) or x.dtype != torch.float32 or x.shape[0] == 0 or x.shape[2] != g.shape[2]:
        return None
    cfg = kernels.uv_config_of(tp_info)
    if int(cfg) < 0 or cfg.path_scale is not None or cfg.w_rows is not None:
        return None
    (n, _, c), cy = x.shape, y.shape[2] if y.ndim == 3 else 0
    coo = _coo(tp_info)
    if (min(c, cy) < 24 or n < (2048 if coo.P > 4 else 8192)) if cy else (c <= 64 or n < (2048 if coo.P <= 11 else 5000)):
        return None
    steps, n_wgs = -(-n // 16), 64                       # of a range: 32 compute units, two wavefronts per SIMD
    walk = kernels.cached(_anchor(tp_info), ("uvg_walk", n_wgs, str(x.device)), lambda: _GradWWalk(coo, n_wgs, x.device))
    n_ranges = walk.ranges(steps)
    gw = torch.empty((coo.P, c * max(cy, 1), c), dtype=x.dtype, device=x.device)
    jobs, job_ptr, slot_ptr = (walk.words.data_ptr() + v for v in walk.at)
    a = _lib.UvgArgs(x.data_ptr(), y.data_ptr(), g.data_ptr(), gw.data_ptr(), 256, jobs, job_ptr, slot_ptr, n, int(cfg), n_ranges, n_wgs,
                     walk.n_slots, c, cy)
    if _lib.lib.cgtp_uvg_validate(C.byref(a)) != 0:
        return None
    ws = torch.empty(n_ranges * walk.n_slots * gw[0].numel(), dtype=x.dtype, device=x.device)
    a.workspace = ws.data_ptr()
    _lib.check(_lib.lib.cgtp_uvg_apply(C.byref(a), _lib.stream_ptr(x.device)), "cgtp_uvg_apply")
    return gw


def grad_w(x: Tensor, y: Tensor, g: Tensor, tp_info) -> Tensor:
    """``gw[p, k, w] = sum_n sum_{(p, M)} inter[n, (p, M), k] g[n, M, w]`` (``cgtp_uvt_grad_w``, in fp32 ``cgtp_uvg_apply``):
    ``(P, K, C_out)`` with ``K = C_x`` or ``C_x * C_y``; the caller reshapes."""
    gw = _split_grad_w(x, y, g, tp_info)
    if gw is None:
        gw = _mix_grad_w(x, g, tp_info)
    if gw is not None:
        return gw
    walk = kernels.cached(_anchor(tp_info), ("uvt_path_walk", str(x.device)),
                          lambda: _PathWalk(_coo(tp_info), x.device))
    n, dx, cx = x.shape
    dy = y.shape[1]
    cy = y.shape[2] if y.ndim == 3 else 0
    k = cx * cy if cy else cx
    cout = g.shape[-1]
    gw = torch.empty((walk.n_paths, k, cout), dtype=x.dtype, device=x.device)
    ws = torch.empty(max(int(_lib.lib.cgtp_uvt_grad_w_workspace_bytes(n, walk.n_paths, k, cout, _lib.dtype_code(x.dtype))), 16), dtype=torch.uint8,
                     device=x.device)
    a = _lib.UvtGwArgs()
    a.x, a.y, a.g, a.gw, a.workspace = x.data_ptr(), y.data_ptr(), g.data_ptr(), gw.data_ptr(), ws.data_ptr()
    a.items, a.path_ptr = walk.items.data_ptr(), walk.path_ptr.data_ptr()
    a.term_a, a.term_b, a.term_c = walk.term_a.data_ptr(), walk.term_b.data_ptr(), walk.term_c(x.dtype).data_ptr()
    a.n_rows, a.n_items, a.n_terms, a.n_paths = n, walk.n_items, walk.n_terms, walk.n_paths
    a.dx, a.dy, a.dg, a.cx, a.cy, a.cout, a.dtype = dx, dy, g.shape[1], cx, cy, cout, _lib.dtype_code(x.dtype)
    _lib.check(_lib.lib.cgtp_uvt_grad_w(C.byref(a), _lib.stream_ptr(x.device)), "cgtp_uvt_grad_w")
    return gw


class _SegWalk(_Coefficients):
    """Segments (weight path, row of the first operand) with their terms (row of grad_out, row of the second operand):
    the walk of ``cgtp_uvt_grad_y``.  Segments are not split: the kernel forms one matrix product per segment."""

    def __init__(self, coo, device):
        order = np.lexsort([coo.M, coo.M2, coo.M1, coo.p])
        p_idx, a_idx, b_idx, m_idx = (np.asarray(v)[order] for v in (coo.p, coo.M1, coo.M2, coo.M))
        coef = np.asarray(coo.coef, dtype=np.float64)[order]
        items = []
        t, n_terms = 0, p_idx.shape[0]
        while t < n_terms:
            t1 = t
            while t1 < n_terms and p_idx[t1] == p_idx[t] and a_idx[t1] == a_idx[t]:
                t1 += 1
            items.append([int(p_idx[t]), 0, 0, t, t1, int(a_idx[t]), 0, 0])
            t = t1
        # longest segments first: the wavefront groups take segments round robin
        items.sort(key=lambda it: it[3] - it[4])
        self.n_items, self.n_terms = len(items), n_terms
        self.items = torch.tensor(items, dtype=torch.int32).reshape(-1, 8).to(device)
        self.term_m = torch.from_numpy(m_idx.astype(np.int32)).to(device)
        self.term_b = torch.from_numpy(b_idx.astype(np.int32)).to(device)
        self._coef, self._device, self._term_c = coef, device, {}


def grad_y_supported(n: int, dx: int, dy: int, cx: int, cout: int, tp_info, itemsize: int = 4) -> bool:
    """Whether the 16 staged samples of a ``cgtp_uvt_grad_y`` workgroup and its tables fit the LDS."""
    c = _coo(tp_info)
    kx = ((cx + 15) // 16 + 3) // 4 * 4 * 16
    # one 32-byte item per (weight path, row of the first operand) segment, 8 bytes + a coefficient per term
    n_items = kernels.cached(_anchor(tp_info), "uvt_seg_count",
                             lambda: len(set(zip(np.asarray(c.p).tolist(), np.asarray(c.M1).tolist()))))
    lds = (16 * (dx * kx + 4) + 8 * 16 * dy) * itemsize + n_items * 32 + len(c.coef) * (8 + itemsize) + 16
    return cx % 4 == 0 and cout % 4 == 0 and lds <= 160 * 1024


def grad_y(x: Tensor, g: Tensor, wp: Tensor, tp_info, dy: int) -> Tensor:
    """``gy[n, b] = sum_t c_t <g[n, M_t, :], x[n, a_t, :] @ W[p_t]>`` (``cgtp_uvt_grad_y``); ``wp``: the weight as packed
    for the forward."""
    walk = kernels.cached(_anchor(tp_info), ("uvt_seg_walk", str(x.device)),
                          lambda: _SegWalk(_coo(tp_info), x.device))
    n, dx, cx = x.shape
    gy = torch.empty((n, dy), dtype=x.dtype, device=x.device)
    a = _lib.UvtGyArgs()
    a.x, a.g, a.wp, a.gy = x.data_ptr(), g.data_ptr(), wp.data_ptr(), gy.data_ptr()
    a.items, a.term_m, a.term_b, a.term_c = (walk.items.data_ptr(), walk.term_m.data_ptr(), walk.term_b.data_ptr(),
                                             walk.term_c(x.dtype).data_ptr())
    a.n_rows, a.n_items, a.n_terms = n, walk.n_items, walk.n_terms
    a.dx, a.dy, a.dg, a.cx, a.cout, a.dtype = dx, dy, g.shape[1], cx, g.shape[2], _lib.dtype_code(x.dtype)
    _lib.check(_lib.lib.cgtp_uvt_grad_y(C.byref(a), _lib.stream_ptr(x.device)), "cgtp_uvt_grad_y")
    return gy


def chunk_of(n_rows: int, dx: int, dy: int, dout: int, cx: int, cy: int, cout: int, dtype=torch.float32) -> int:
    """Blocks of 16 contracted channels a launch with these extents pads to; <= 0: the kernels do not take them
    (channel counts not multiples of 4, rows of 16 samples beyond the LDS)."""
    return int(_lib.lib.cgtp_uvt_chunk(n_rows, dx, dy, dout, cx, cy, cout, _lib.dtype_code(dtype)))


def pack(w: Tensor, n_paths: int, k: int, cout: int, stride_p: int, stride_k: int, stride_c: int) -> Tensor:
    """The weight viewed as ``(n_paths, k, cout)`` through element strides, in matrix-core fragment order."""
    packed = torch.empty(int(_lib.lib.cgtp_uvt_packed_elems(n_paths, k, cout)), dtype=w.dtype, device=w.device)
    _lib.check(_lib.lib.cgtp_uvt_pack_weights(w.data_ptr(), packed.data_ptr(), n_paths, k, cout, stride_p, stride_k,
                                              stride_c, _lib.dtype_code(w.dtype), _lib.stream_ptr(w.device)), "cgtp_uvt_pack_weights")
    return packed


class StoredWeight(NamedTuple):
    """A weight ``(P, U, W)`` as the caller holds it, packed by :func:`apply` for the kernel that serves."""
    w: Tensor
    transposed: bool


def apply(x: Tensor, y: Tensor, wp, tp_info, role: str, dout: int, cout: int) -> Tensor:
    """``x (N, dx, cx)``, ``y (N, dy)`` or ``(N, dy, cy)`` -> ``(N, dout, cout)``: one launch of ``cgtp_uvt_apply``, with
    ``wp`` a weight packed for it, or (a :class:`StoredWeight`) of ``cgtp_uvl_apply`` for channel mixing in fp32."""
    if isinstance(wp, StoredWeight):
        out = _mix_split(x, wp.w, tp_info, wp.transposed)
        if out is not None:
            return out
        p, u, wc = wp.w.shape
        wp = pack(wp.w, p, wc, u, u * wc, 1, wc) if wp.transposed else pack(wp.w, p, u, wc, u * wc, wc, 1)
    n, dx, cx = x.shape
    dy = y.shape[1]
    cy = y.shape[2] if y.ndim == 3 else 0
    k = cx * cy if cy else cx
    kbi = chunk_of(n, dx, dy, dout, cx, cy, cout, x.dtype)
    if kbi <= 0:
        raise _lib.CgtpError(f"cgtp_uvt_apply does not take these extents (status {-kbi})")
    n_groups = int(_lib.lib.cgtp_uvt_item_groups(n, dx, dy, dout, cx, cy, cout, _lib.dtype_code(x.dtype)))
    walk = _walk(tp_info, role, n_groups, x.device)
    out = torch.empty((n, dout, cout), dtype=x.dtype, device=x.device)
    if n == 0:
        return out
    a = _lib.UvtArgs()
    a.x, a.y, a.wp, a.out = x.data_ptr(), y.data_ptr(), wp.data_ptr(), out.data_ptr()
    a.items, a.term_a, a.term_b, a.term_c = (walk.items.data_ptr(), walk.term_a.data_ptr(), walk.term_b.data_ptr(),
                                             walk.term_c(x.dtype).data_ptr())
    a.n_rows, a.n_items, a.n_terms = n, walk.n_items, walk.term_a.shape[0]
    a.dx, a.dy, a.dout, a.cx, a.cy, a.cout = dx, dy, dout, cx, cy, cout
    a.kbi, a.dtype = kbi, _lib.dtype_code(x.dtype)
    a.n_groups = n_groups
    for i, v in enumerate(walk.group_ptr):
        a.group_ptr[i] = v
    _lib.check(_lib.lib.cgtp_uvt_apply(C.byref(a), _lib.stream_ptr(x.device)), "cgtp_uvt_apply")
    return out


def _split(kind: int, x: Tensor, y: Tensor, w: Tensor, tp_info, rows_out: int) -> Optional[Tensor]:
    """The product of a compiled table in fp32 on the half-precision matrix cores (``cgtp_uvs_apply``; ``kind`` 0: forward, 1:
    gradient of the first operand, 2: gradient of the second), or None where the fp32 matrix instructions serve: tables
    that are not compiled in as they are, contracted channels other than 32, 64, 128, and 128 -> 32.  From 100 to 32768 samples, lmax 1
    to 3, equal channels it takes 0.3 to 0.9 of their time (100 samples, lmax = 1, 32 channels: 14 to 18 us on both,
    launches alone)."""
    if isinstance(tp_info, CooTable) or x.dtype != torch.float32:
        return None
    cfg = kernels.uv_config_of(tp_info)
    if int(cfg) < 0 or cfg.path_scale is not None or cfg.w_rows is not None:
        return None
    n, p, u, wc = x.shape[0], *w.shape
    cin, cout = (wc, u) if kind == 1 else (u, wc)
    aligned = 256
    if _lib.lib.cgtp_uvs_validate(int(cfg), kind, x.data_ptr(), y.data_ptr(), aligned, w.data_ptr(), aligned,
                                                    n, cin, cout) != 0:
        return None
    packed = torch.empty(int(_lib.lib.cgtp_uvs_packed_bytes(p, cin, cout)), dtype=torch.uint8, device=x.device)
    out = torch.empty((n, rows_out) if kind == 2 else (n, rows_out, cout), dtype=x.dtype, device=x.device)
    stream = _lib.stream_ptr(x.device)
    _lib.check(_lib.lib.cgtp_uvs_pack_weights(w.data_ptr(), packed.data_ptr(), p, cin, cout, int(kind == 1), stream),
               "cgtp_uvs_pack_weights")
    _lib.check(_lib.lib.cgtp_uvs_apply(int(cfg), kind, x.data_ptr(), y.data_ptr(), packed.data_ptr(), w.data_ptr(),
                                       out.data_ptr(), n, cin, cout, stream), "cgtp_uvs_apply")
    return out


def _split_uvw(kind: int, x: Tensor, z: Tensor, w: Tensor, tp_info, rows_out: int) -> Optional[Tensor]:
    """The same for channels on both operands (``cgtp_uvsw_apply``), ``w (P, U, V, W)``; ``kind`` 0: forward, 1: gradient of the
    first operand (``x`` = grad_out, ``z`` = the second operand), 2: gradient of the second (``x`` = grad_out, ``z`` = the
    first).  32 contracted channels, which one matrix instruction takes whole, a multiple of 32 produced ones, up to nine
    produced rows (lmax = 2: the registers hold them all).  Takes 0.3 to 0.7 of the time of the fp32 matrix instructions from 100 to 32768
    samples."""
    if isinstance(tp_info, CooTable) or x.dtype != torch.float32:
        return None
    cfg = kernels.uv_config_of(tp_info)
    if int(cfg) < 0 or cfg.path_scale is not None or cfg.w_rows is not None:
        return None
    n, (p, u, v, c) = x.shape[0], w.shape
    aligned = 256
    if _lib.lib.cgtp_uvsw_validate(int(cfg), kind, x.data_ptr(), z.data_ptr(), aligned, w.data_ptr(), aligned, n, u, v, c) != 0:
        return None
    packed = torch.empty(int(_lib.lib.cgtp_uvsw_packed_bytes(p, u, v, c)), dtype=torch.uint8, device=x.device)
    out = torch.empty((n, rows_out, (c, u, v)[kind]), dtype=x.dtype, device=x.device)
    _lib.check(_lib.lib.cgtp_uvsw_apply(int(cfg), kind, x.data_ptr(), z.data_ptr(), packed.data_ptr(), w.data_ptr(),
                                        out.data_ptr(), n, u, v, c, _lib.stream_ptr(x.device)), "cgtp_uvsw_apply")
    return out


_MIX_STEPS = 64          # of a group, one lane each


class _MixTable:
    """A channel-mixing table for ``cgtp_uvl_apply`` (``transposed``: the gradient of its input): the rows of the result by two
    where most of the rows of the input that reach one reach both (the ``+m`` and ``-m`` rows of an SO(2) layer, which then
    load and split them once), else one by one, and their steps."""

    def __init__(self, coo, transposed: bool):
        rows_out, rows_in, n_out = (coo.M1, coo.M, coo.D1) if transposed else (coo.M, coo.M1, coo.DO)
        o, i, p = (np.asarray(v, dtype=np.int64) for v in (rows_out, rows_in, coo.p))
        coef = np.asarray(coo.coef, dtype=np.float64).astype(np.float32)
        # (path, coefficient) has a place in the packed weight
        keys, block = np.unique(p << 32 | coef.view(np.uint32), return_inverse=True)
        self.blocks = np.stack([(keys >> 32), (keys & 0xffffffff)], axis=1).astype(np.uint32).view(np.int32)
        if not len(keys):
            self.blocks = np.zeros((1, 2), dtype=np.int32)
        self.n_out, self.n_blocks = n_out, len(self.blocks)
        pairs, alone, shared = self._pairs(o, i, n_out)
        if 4 * shared < len(np.unique(o * (1 << 32) + i)):
            pairs, alone = [], list(range(n_out))
        self.rows_per_task = 2 if pairs else 1
        self.tasks = sorted(pairs + [(m, -1) for m in alone])
        # a step: a row of the input and a block for each row of the task; entries of one row and input row one after the other
        tasks = np.array(self.tasks, dtype=np.int64).reshape(-1, 2)
        task_of, side_of = np.zeros(n_out, dtype=np.int64), np.zeros(n_out, dtype=np.int64)
        for side in (0, 1):
            real = tasks[:, side] >= 0
            task_of[tasks[real, side]], side_of[tasks[real, side]] = np.nonzero(real)[0], side
        order = np.lexsort([i, o])
        o, i, block = o[order], i[order], block.ravel()[order]
        at = np.arange(len(o))
        new = np.ones(len(o), dtype=bool)
        new[1:] = (o[1:] != o[:-1]) | (i[1:] != i[:-1])
        turn = at - np.maximum.accumulate(np.where(new, at, 0))
        empty = np.nonzero(np.bincount(task_of[o], minlength=len(tasks)) == 0)[0]       # written as zeros: a step without blocks
        n_in, most = int(i.max(initial=0)) + 1, int(turn.max(initial=0)) + 1
        keys, step = np.unique(np.concatenate([(task_of[o] * n_in + i) * most + turn, empty * n_in * most]), return_inverse=True)
        steps = np.full((len(keys), 4), -1, dtype=np.int32)
        steps[:, 0] = keys // most % n_in
        steps[step.ravel()[:len(o)], 1 + side_of[o]] = block
        task = keys // most // n_in
        last = np.ones(len(task), dtype=bool)
        last[:-1] = task[1:] != task[:-1]
        steps[last, 3] = task[last]
        ends = (np.nonzero(last)[0] + 1).tolist()
        self.steps = [steps[b:e] for b, e in zip([0] + ends, ends)]
        self._sizes = list(map(len, self.steps))
        self._longest_first = sorted(range(len(ends)), key=lambda t: -self._sizes[t])
        self.longest = max(self._sizes)
        # whether the fp32 kernel, which deals the rows to a power of two of wavefronts, has no longer chains
        row_entries = sorted(np.bincount(o, minlength=n_out).tolist(), reverse=True)
        chains = [0] * (1 << min(n_out.bit_length() - 1, 4))
        for k in row_entries:
            heapq.heapreplace(chains, chains[0] + k)
        self.even = max(chains) <= self.longest
        # the numbers of groups to choose from, with the most steps of a group and their cost: a group's steps are a lane each
        dealt = {g: self.dealt(g) for g in (1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, len(self.tasks)) if g <= len(self.tasks)}
        self.choices = {g: most for g, (_, most) in dealt.items()}
        self.costs = [(g, most + 2) for g, most in self.choices.items() if most <= _MIX_STEPS]
        self._dealt = {g: dealt[g][0] for g, _ in self.costs}

    @staticmethod
    def _pairs(o, i, n_out: int):
        """Pairs of rows of the result, the rows left, and the rows of the input that both rows of a pair share, added up: of
        rows that the same rows of the input reach two by two, and of the rest as many as share most of them."""
        reach = np.unique(o * (1 << 32) + i)
        row, at = reach >> 32, reach & 0xffffffff
        ends = np.searchsorted(row, np.arange(n_out + 1))
        rows_in = [at[ends[m]:ends[m + 1]] for m in range(n_out)]
        pairs, shared, waiting = [], 0, {}
        for m, mine in enumerate(rows_in):
            if len(mine):
                first = waiting.pop(key := mine.tobytes(), None)
                if first is None:
                    waiting[key] = m
                else:
                    pairs.append((first, m))
                    shared += len(mine)
        alone = np.ones(n_out, dtype=bool)
        alone[[m for pair in pairs for m in pair]] = False
        if len(waiting) > 1:
            by_in = np.argsort(at, kind="stable")
            in_ends = np.searchsorted(at[by_in], np.arange(int(at.max()) + 2))
            reached = row[by_in]
            for m in sorted(waiting.values()):
                if alone[m]:
                    both = np.bincount(np.concatenate([reached[in_ends[k]:in_ends[k + 1]] for k in rows_in[m]]), minlength=n_out)
                    both = np.where(alone, both, 0)
                    both[m] = 0
                    most = int(both.argmax())
                    if 2 * both[most] > max(len(rows_in[m]), len(rows_in[most])):
                        pairs.append((m, most))
                        alone[[m, most]] = False
                        shared += int(both[most])
        return pairs, np.nonzero(alone)[0].tolist(), shared

    def dealt(self, n_groups: int):
        """The tasks in ``n_groups`` groups: the longest first, each to the group with the fewest steps so far."""
        groups, count = [[] for _ in range(n_groups)], [(0, g) for g in range(n_groups)]
        for t in self._longest_first:
            steps, g = count[0]
            groups[g].append(t)
            heapq.heapreplace(count, (steps + self._sizes[t], g))
        return groups, max(count)[0]

    @functools.cached_property
    def words(self):
        """What the kernel reads, dealt to every number of groups there is to choose from, in one array, and where the steps, the
        groups and the tasks and blocks they share begin, in bytes, for each."""
        parts = [np.array(v, dtype=np.int32).ravel() for v in (self.tasks, self.blocks)]
        parts = [np.resize(v, -(-v.size // 4) * 4) for v in parts]          # steps are read 16 bytes at a time
        end, at = sum(v.size for v in parts), {}
        for n_groups, groups in self._dealt.items():
            ptr, begin = [], 0
            for group in groups:
                ptr += [begin, begin := begin + sum(self._sizes[t] for t in group)]
            ptr += [0] * (len(ptr) % 4)
            parts += [np.concatenate([self.steps[t] for group in groups for t in group]).ravel(), np.array(ptr, dtype=np.int32)]
            at[n_groups] = tuple(4 * v for v in (end, end + parts[-2].size, 0, parts[0].size))
            end += parts[-2].size + parts[-1].size
        return np.concatenate(parts), at

    def groups_for(self, n: int, column_blocks: int) -> int:
        """Groups (workgroups a block of samples is cut into): what lets whole rounds of two workgroups per compute unit end
        soonest, a workgroup costing its steps and about two more to start."""
        blocks = -(-n * self.rows_per_task // 256) * column_blocks
        least, best = None, 0
        for g, cost in self.costs:
            time = -(-blocks * g // 512) * cost
            if least is None or time < least:
                least, best = time, g
        return best


class _MixWalk:
    """The words of a :class:`_MixTable` on the device, copied in one piece: a batch of another size copies nothing."""

    def __init__(self, table: _MixTable, device):
        words, self.at = table.words
        self.max_steps = table.choices
        self.words = torch.tensor(words, device=device)
        self.address = {g: tuple(self.words.data_ptr() + v for v in at) for g, at in self.at.items()}


@functools.lru_cache(maxsize=64)
def _mix_table_of_content(transposed: bool, D1: int, DO: int, coef: bytes, *indices: bytes) -> _MixTable:
    """:class:`_MixTable` by the table's content: host work that a second layer over the same irreps does not repeat.  Host arrays
    only, read by every caller and written by none."""
    M, M1, p = (np.frombuffer(v, dtype=np.int32) for v in indices)
    return _MixTable(TpCoo(np.frombuffer(coef, dtype=np.float64), M, M1, None, p, None, D1, 1, DO, 0), transposed)


def _mix_table(table, transposed: bool) -> _MixTable:
    c = table.coo
    return kernels.cached(_anchor(table), ("uvl_table", transposed), lambda: _mix_table_of_content(
        transposed, int(c.D1), int(c.DO), np.ascontiguousarray(c.coef, dtype=np.float64).tobytes(),
        *(np.ascontiguousarray(v, dtype=np.int32).tobytes() for v in (c.M, c.M1, c.p))))


def _observed(*tensors: Tensor) -> bool:
    """Whether something looks at the operations on these tensors one by one (a transform, forward mode, tracing, a dispatch
    mode, a tensor subclass, autocast): tensor algebra serves it, an autograd function over raw pointers does not."""
    functorch = torch._C._functorch
    return (functorch.peek_interpreter_stack() is not None or torch.autograd.forward_ad._current_level >= 0
            or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0 or torch.is_autocast_enabled("cuda")
            or any(type(t) not in (Tensor, torch.nn.Parameter) or functorch.is_legacy_batchedtensor(t) for t in tensors))


def mix_fits(x: Tensor, w: Tensor, table, one_product: bool, widened: bool) -> bool:
    """Whether channel mixing with this table, too large for the fp32 kernels, runs on the half-precision matrix cores in
    both directions.  ``one_product``: the library has all entries of a row in one product (SO(2) layers, forward and gradients of
    50 to 16000 samples, 48 to 256 channels 0.1 to 0.8 of its time), else one for each entry, which wins where the launches do
    not count: past 1.5e9 multiplications (lmax 6, 96 channels, 16000 samples 692 us against 677, lmax 3, 64 -> 256 453 against 353,
    below 0.4 to 0.9) and past 256 channels (lmax 6, 384, 300 samples 314 against 250).  ``widened`` from 16 bits, in which the library
    is quicker: SO(2) layers up to 1.7e10 multiplications (lmax 6, 64 channels, 4000 samples 399 us against 1387, lmax 5, 256, 1000 897
    against 1384; past it lmax 4, 192, 4000 1545 against 1225, lmax 6, 256, 4000 4598 against 2543).
    Long rows stay on the library, which sums in blocks and entries of their own.  Relative to 64 bits, operands of one sign,
    kernel and library: one product of 12 entries of 256 channels (96 units of 32) 1.4e-7 and 2.0e-7; entries of their own, one of 384
    channels 0.6e-7 and 3.1e-7, 3 of 640 1.0e-7 and 0.8e-7, 24 of 128 1.5e-7 and 0.9e-7."""
    c = table.coo
    if _observed(x, w):
        return False
    if x.shape[0] * len(c.p) * w.shape[1] * w.shape[2] > {(False, False): 1.5e9, (False, True): 0, (True, True): 1.7e10}.get(
            (one_product, widened), float("inf")):
        return False

    def short(transposed: bool) -> bool:
        steps = _mix_table(table, transposed).longest
        return steps <= _MIX_STEPS and steps * -(-w.shape[1 + transposed] // 32) <= (96 if one_product else 8)
    return (x.dtype == w.dtype == torch.float32 and x.shape[0] > 0 and x.data_ptr() % 16 == 0 and w.shape[1] % 4 == 0
            and w.shape[2] % 4 == 0 and w.shape[0] == c.P and tuple(x.shape[1:]) == (c.D1, w.shape[1])
            and max(c.D1 * w.shape[1], c.DO * w.shape[2]) <= 1 << 22
            and short(False) and short(True))


def _few_and_long(mix: _MixTable, n: int, cx: int, cout: int) -> bool:
    """Whether the workgroups of ``cgtp_uvl_apply`` are so few and long that the fp32 kernel, of 16 samples each, ends sooner: past 128
    contracted channels and below 2048 samples (256 -> 256, lmax 4, 700 samples: 43 us against 38), and small results made two
    rows at a time where that kernel has no longer chains either, the pack included: SO2Linear of lmax 1, 128 -> 48 channels, 1500
    samples 18.1 us against 14.3, 8000 20.5 against 22.1; 64 -> 64, 1500 12.6 against 11.9; of lmax 2, 128 -> 16, 4096 24.0 against 18.6, 64 ->
    16 15.2 against 14.2, 128 -> 20 24.4 and 24.1; two scalars, 128 -> 128, 4096 19.0 against 15.5."""
    if cx > 128 and n < 2048:
        return True
    return (mix.rows_per_task == 2 and mix.even and cx > (64 if 16 < cout <= 32 else 32)
            and n < (10000 if cx > 64 and cout <= 16 else 5000) and mix.n_out * cout <= (256 if mix.n_out <= 4 else 144))


def _was_the_library(n: int, u: int, wc: int, table) -> bool:
    """Whether the fp32 kernels do not take channel mixing with this table, ``u -> wc`` channels: the products of the library, whose
    sums are more precise than theirs, served it."""
    return kernels.cached(_anchor(table), ("uvl_was_library", u, wc), lambda: not u1v_fits(n, u, wc, table, torch.float32))


def _mix_split(x: Tensor, w: Tensor, table, transposed: bool) -> Optional[Tensor]:
    """Channel mixing in fp32 on the half-precision matrix cores (``cgtp_uvl_apply``), or None where the fp32 matrix
    instructions serve.  Over 1000 launches (IrrepsLinear of lmax 1 to 4 and of copies of an irrep, SO2Linear of lmax 1 to 6, 8 to
    256 channels on either side, 100 to 65000 samples) it takes 0.4 to 1.0 of their time, apart from those of
    :func:`_few_and_long` and, up to 1.05, SO2Linear of lmax 1 and 2 with 96 and more to 16 channels about 12000 samples."""
    if not (isinstance(table, CooTable) and table.mixing) or x.dtype != torch.float32:
        return None
    n, dx, cx = x.shape
    cout = w.shape[1] if transposed else w.shape[2]
    mix = _mix_table(table, transposed)
    if mix.longest > _MIX_STEPS or (_few_and_long(mix, n, cx, cout) and chunk_of(n, dx, 1, mix.n_out, cx, 0, cout) > 0):
        return None
    n_groups = mix.groups_for(n, -(-cout // 64))
    walk = kernels.cached(_anchor(table), ("uvl_walk", transposed, str(x.device)), lambda: _MixWalk(mix, x.device))
    by_unit = int(_was_the_library(n, w.shape[1], w.shape[2], table))
    packed = torch.empty(int(_lib.lib.cgtp_uvl_packed_bytes(mix.n_blocks, cx, cout)), dtype=torch.uint8, device=x.device)
    out = torch.empty((n, mix.n_out, cout), dtype=x.dtype, device=x.device)
    steps, groups, tasks, blocks = walk.address[n_groups]
    a = _lib.UvlArgs(x.data_ptr(), packed.data_ptr(), w.data_ptr(), out.data_ptr(), steps, tasks, groups, blocks,
                     n, w.stride(0), w.stride(2 if transposed else 1), w.stride(1 if transposed else 2),
                     mix.n_blocks, n_groups, mix.rows_per_task, walk.max_steps[n_groups], dx, mix.n_out, cx, cout, by_unit)
    status = _lib.lib.cgtp_uvl_apply(C.byref(a), _lib.stream_ptr(x.device))
    if status in (2, 3):               # extents or an alignment it does not take: nothing was launched
        return None
    _lib.check(status, "cgtp_uvl_apply")
    return out


def _coo(tp_info):
    return tp_info.coo if isinstance(tp_info, CooTable) else kernels.coo_of(tp_info)


def _aligned(g: Tensor) -> Tensor:
    """The incoming gradient as the kernels want it: contiguous and on a 16-byte boundary.  Autograd may hand over a
    view into a larger buffer (the gradient of a ``cat`` or of a slice), contiguous but at any element offset."""
    g = g.contiguous()
    return g.clone() if g.data_ptr() % 16 else g


class _U1vNative(Function):
    """u1v, shared fp32 weight ``(P, U, W)``.  The gradient of the first operand is the forward kernel with the rows'
    roles exchanged and the weight read transposed; the gradients of the weight and of the second operand have
    kernels of their own (``cgtp_uvt_grad_w``, ``cgtp_uvt_grad_y``).  Under ``create_graph`` the backward is the
    differentiable two-stage route of ``_uv_gemm``."""

    @staticmethod
    def forward(ctx, x: Tensor, y: Tensor, w: Tensor, tp_info):
        c = _coo(tp_info)
        p, u, wc = w.shape
        out = _split(0, x, y, w, tp_info, c.DO)
        if out is None:
            out = apply(x, y, StoredWeight(w, False), tp_info, "out", c.DO, wc)
        ctx.save_for_backward(x, y, w)
        ctx.tp_info = tp_info
        return out

    @staticmethod
    def backward(ctx, g):
        from . import _uv_gemm
        x, y, w = ctx.saved_tensors
        need = ctx.needs_input_grad[:3]
        tp_info = ctx.tp_info
        higher = torch.is_grad_enabled()  # higher-order derivative: the differentiable route throughout
        if higher or (isinstance(tp_info, CooTable) and tp_info.algebra and _observed(g)):
            with torch.enable_grad():
                out = tp_info.fallback(x, y, w) if isinstance(tp_info, CooTable) else _uv_gemm.u1v(x, y, w, tp_info)
                wanted = [t for t, n in zip((x, y, w), need) if n]
                got = iter(torch.autograd.grad(out, wanted, g, create_graph=higher, allow_unused=True))
            return tuple(next(got) if n else None for n in need) + (None,)
        c = _coo(tp_info)
        p, u, wc = w.shape
        gx = gy = gw = None
        g = _aligned(g)
        if need[0]:
            gx = _split(1, g, y, w, tp_info, c.D1)
            if gx is None:
                gx = apply(g, y, StoredWeight(w, True), tp_info, "in1", c.D1, u)
        if need[2]:
            gw = grad_w(x, y, g, tp_info)
        if need[1]:
            gy = _split(2, x, g, w, tp_info, c.D2)
            if gy is None:
                gy = grad_y(x, g, pack(w, p, u, wc, u * wc, wc, 1), tp_info, c.D2)
        return gx, gy, gw, None


def u1v_supported(x: Tensor, y: Tensor, w: Tensor, tp_info) -> bool:
    if not (x.dtype == y.dtype == w.dtype and x.dtype in (torch.float32, torch.float64) and x.ndim == 3 and y.ndim == 2
            and w.ndim == 3):
        return False
    if x.shape[0] == 0:
        return False
    c = _coo(tp_info)
    _, u, wc = w.shape
    n = x.shape[0]
    dt = x.dtype
    if tuple(x.shape) != (n, c.D1, u) or tuple(y.shape) != (n, c.D2) or w.shape[0] != c.P:
        raise _lib.CgtpError(f"operands {tuple(x.shape)}, {tuple(y.shape)}, {tuple(w.shape)} do not fit the table: "
                             f"expected (N, {c.D1}, U), (N, {c.D2}), ({c.P}, U, W)")
    return u1v_fits(n, u, wc, tp_info, dt) and x.data_ptr() % 16 == 0


def u1v_fits(n: int, u: int, wc: int, tp_info, dtype: torch.dtype) -> bool:
    """Whether the forward, the gradient of the channelled operand and the gradient of the second operand have a launch
    shape for ``n`` samples, ``u -> wc`` channels in ``dtype`` (float32 | float64): extents only, no tensors."""
    c = _coo(tp_info)
    size = torch.empty(0, dtype=dtype).element_size()
    return (n > 0 and chunk_of(n, c.D1, c.D2, c.DO, u, 0, wc, dtype) > 0
            and chunk_of(n, c.DO, c.D2, c.D1, wc, 0, u, dtype) > 0
            and grad_y_supported(n, c.D1, c.D2, u, wc, tp_info, size))


def u1v(x: Tensor, y: Tensor, w: Tensor, tp_info) -> Tensor:
    return _U1vNative.apply(x.contiguous(), y.contiguous(), w.contiguous(), tp_info)


# ---- 1vu: the channels on the second operand — u1v on the table with the operands' rows exchanged -------------------
def operands_exchanged(tp_info) -> CooTable:
    def build():
        from . import _uv_gemm
        c = _coo(tp_info)
        return CooTable(c._replace(M1=c.M2, M2=c.M1, D1=c.D2, D2=c.D1), torch.zeros(1),
                        lambda xx, yy, ww: _uv_gemm.one_vu(yy, xx, ww, tp_info))
    return kernels.cached(_anchor(tp_info), "1vu_table", build)


# ---- vu1: out[n, M] = sum_t c_t <y[n, b_t, :], x[n, a_t, :] @ W[p_t]> ---------------------------------------------
# With the table's output rows and second-operand rows exchanged (T'), this is the gradient of u1v_T' with respect to
# its channel-less operand for the cotangent y — the kernel cgtp_uvt_grad_y — and its own gradients are the forward
# (grad y), the input gradient (grad x) and the weight gradient of u1v_T' with the cotangent of vu1 as the channel-less
# operand.  The reference computes it in three stages, weight first (equitorch/nn/functional/linears.py:414-492).
def _swapped(tp_info) -> CooTable:
    def build():
        c = _coo(tp_info)
        return CooTable(c._replace(M=c.M2, M2=c.M, D2=c.DO, DO=c.D2), torch.zeros(1), None)
    return kernels.cached(_anchor(tp_info), "vu1_table", build)


class _Vu1Native(Function):
    @staticmethod
    def forward(ctx, x: Tensor, y: Tensor, w: Tensor, tp_info):
        t = _swapped(tp_info)
        p, u, wc = w.shape
        out = grad_y(x, y, pack(w, p, u, wc, u * wc, wc, 1), t, t.coo.D2)
        ctx.save_for_backward(x, y, w)
        ctx.tp_info = tp_info
        return out

    @staticmethod
    def backward(ctx, g):
        from . import _uv_gemm
        x, y, w = ctx.saved_tensors
        need = ctx.needs_input_grad[:3]
        if torch.is_grad_enabled():       # higher-order derivative: the differentiable route throughout
            with torch.enable_grad():
                out = _uv_gemm.vu1(x, y, w, ctx.tp_info)
                wanted = [v for v, n in zip((x, y, w), need) if n]
                got = iter(torch.autograd.grad(out, wanted, g, create_graph=True, allow_unused=True))
            return tuple(next(got) if n else None for n in need) + (None,)
        t = _swapped(ctx.tp_info)
        c = t.coo
        p, u, wc = w.shape
        g = _aligned(g)
        gx = apply(y, g, pack(w, p, wc, u, u * wc, 1, wc), t, "in1", c.D1, u) if need[0] else None
        gy = apply(x, g, pack(w, p, u, wc, u * wc, wc, 1), t, "out", c.DO, wc) if need[1] else None
        gw = grad_w(x, g, y, t) if need[2] else None
        return gx, gy, gw, None


def vu1_supported(x: Tensor, y: Tensor, w: Tensor, tp_info) -> bool:
    if not (x.dtype == y.dtype == w.dtype and x.dtype in (torch.float32, torch.float64) and x.ndim == 3 and y.ndim == 3
            and w.ndim == 3 and x.shape[0] > 0):
        return False
    c = _coo(tp_info)
    n, (_, u, wc) = x.shape[0], w.shape
    if tuple(x.shape) != (n, c.D1, u) or tuple(y.shape) != (n, c.D2, wc) or w.shape[0] != c.P:
        raise _lib.CgtpError(f"operands {tuple(x.shape)}, {tuple(y.shape)}, {tuple(w.shape)} do not fit the table: "
                             f"expected (N, {c.D1}, C1), (N, {c.D2}, C2), ({c.P}, C1, C2)")
    return u1v_fits(n, u, wc, _swapped(tp_info), x.dtype) and x.data_ptr() % 16 == 0 and y.data_ptr() % 16 == 0


def vu1(x: Tensor, y: Tensor, w: Tensor, tp_info) -> Tensor:
    return _Vu1Native.apply(x.contiguous(), y.contiguous(), w.contiguous(), tp_info)


class _UvwNative(Function):
    """uvw, shared fp32 weight ``(P, U, V, W)``: forward and the gradients of both operands on ``cgtp_uvt_apply``
    (with the weight permuted as the reference permutes it, ``tensor_products.py:126-150``); the weight gradient and
    higher orders from the two-stage route of ``_uvw_gemm``."""

    @staticmethod
    def forward(ctx, x: Tensor, y: Tensor, w: Tensor, tp_info):
        c = _coo(tp_info)
        p, u, v, wc = w.shape
        out = _split_uvw(0, x, y, w, tp_info, c.DO)
        if out is None:
            out = apply(x, y, pack(w, p, u * v, wc, u * v * wc, wc, 1), tp_info, "out", c.DO, wc)
        ctx.save_for_backward(x, y, w)
        ctx.tp_info = tp_info
        return out

    @staticmethod
    def backward(ctx, g):
        from . import _uvw_gemm
        x, y, w = ctx.saved_tensors
        need = ctx.needs_input_grad[:3]
        tp_info = ctx.tp_info
        if torch.is_grad_enabled():
            with torch.enable_grad():
                out = _uvw_gemm.uvw(x, y, w, tp_info)
                wanted = [t for t, n in zip((x, y, w), need) if n]
                got = iter(torch.autograd.grad(out, wanted, g, create_graph=True, allow_unused=True))
            return tuple(next(got) if n else None for n in need) + (None,)
        c = _coo(tp_info)
        p, u, v, wc = w.shape
        g = _aligned(g)
        gx = gy = gw = None
        if need[0]:
            gx = _split_uvw(1, g, y, w, tp_info, c.D1)
        if need[1]:
            gy = _split_uvw(2, g, x, w, tp_info, c.D2)
        if need[0] and gx is None:     # first operand of the launch: y (channels v), second: grad_out (channels w); weight (P, V, W, U)
            wt = w.permute(0, 2, 3, 1).contiguous()
            gx = apply(y, g, pack(wt, p, v * wc, u, v * wc * u, u, 1), tp_info, "in1_uvw", c.D1, u)
        if need[1] and gy is None:     # first: grad_out (channels w), second: x (channels u); weight (P, W, U, V)
            wt = w.permute(0, 3, 1, 2).contiguous()
            gy = apply(g, x, pack(wt, p, wc * u, v, wc * u * v, v, 1), tp_info, "in2_uvw", c.D2, v)
        if need[2]:
            gw = grad_w(x, y, g, tp_info).view(p, u, v, wc)
        return gx, gy, gw, None


def uvw_supported(x: Tensor, y: Tensor, w: Tensor, tp_info) -> bool:
    if not (x.dtype == y.dtype == w.dtype and x.dtype in (torch.float32, torch.float64) and x.ndim == 3 and y.ndim == 3
            and w.ndim == 4):
        return False
    if x.shape[0] == 0:
        return False
    c = _coo(tp_info)
    _, u, v, wc = w.shape
    n = x.shape[0]
    dt = x.dtype
    if tuple(x.shape) != (n, c.D1, u) or tuple(y.shape) != (n, c.D2, v) or w.shape[0] != c.P:
        raise _lib.CgtpError(f"operands {tuple(x.shape)}, {tuple(y.shape)}, {tuple(w.shape)} do not fit the table: "
                             f"expected (N, {c.D1}, U), (N, {c.D2}, V), ({c.P}, U, V, W)")
    return uvw_fits(n, u, v, wc, tp_info, dt) and x.data_ptr() % 16 == 0 and y.data_ptr() % 16 == 0


def uvw_fits(n: int, u: int, v: int, wc: int, tp_info, dtype: torch.dtype) -> bool:
    """The same for the product with channels on both operands."""
    c = _coo(tp_info)
    return (n > 0 and chunk_of(n, c.D1, c.D2, c.DO, u, v, wc, dtype) > 0
            and chunk_of(n, c.D2, c.DO, c.D1, v, wc, u, dtype) > 0 and chunk_of(n, c.DO, c.D1, c.D2, wc, u, v, dtype) > 0)


def uvw(x: Tensor, y: Tensor, w: Tensor, tp_info) -> Tensor:
    return _UvwNative.apply(x.contiguous(), y.contiguous(), w.contiguous(), tp_info)
