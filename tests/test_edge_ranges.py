"""How a sorted edge list is cut into one range per wavefront (``SegIndex``): host arithmetic only."""
import pytest
import torch

COEFFICIENTS = {1: 10, 2: 83, 3: 353}


def _index(degrees):
    from equitorch_amd.ops.kernels import SegIndex
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), torch.tensor(degrees).cumsum(0)])
    n = int(ptr[-1])
    return SegIndex(ptr, None, torch.repeat_interleave(torch.arange(len(degrees)), torch.tensor(degrees)), torch.zeros(n, dtype=torch.int64))


@pytest.mark.parametrize("degree,n_edges,lmax,slots,aligned", [
    (64, 60000, 1, 64, True), (64, 60000, 2, 16, True), (64, 60000, 3, 32, True),      # few channels, a node in a few steps
    (30, 8192, 2, 4, False), (30, 8192, 3, 2, False),                                  # short list: cut finer than a node
    (30, 65536, 2, 4, True), (30, 65536, 3, 2, False), (4, 60000, 1, 2, True),         # the chip is full either way
    (100, 100, 1, 4, True), (200, 400, 3, 16, False)])
def test_forward_ranges(degree, n_edges, lmax, slots, aligned):
    seg = _index([degree] * (n_edges // degree))
    assert seg.prefers_aligned(slots, False, COEFFICIENTS[lmax]) == aligned
    assert not seg.prefers_aligned(slots, True, COEFFICIENTS[lmax])


def test_a_hub_node_has_no_aligned_ranges():
    assert not _index([257] + [8] * 5000).prefers_aligned(64, False, 10)
    assert _index([256] + [8] * 5000).prefers_aligned(64, False, 10)


@pytest.mark.parametrize("degrees", [[1], [3, 0, 0, 5], [0, 64, 65, 1, 0], [300] + [2] * 900, [17] * 9000])
def test_ranges_cover_the_list_in_whole_steps(degrees):
    seg = _index(degrees)
    n = sum(degrees)
    starts = set((seg.ptr[:-1]).tolist()) | {n}
    if seg.wave_seg is not None:
        cuts = seg.wave_seg.tolist()
        assert cuts[0] == 0 and cuts[-1] == len(degrees) and cuts == sorted(cuts)
    for slots in seg.SLOT_COUNTS:
        cuts = seg.balanced_positions(slots).tolist()
        assert cuts[0] == 0 and cuts[-1] == n and cuts == sorted(cuts)
        for c in cuts[1:-1]:                                 # a multiple of the slots past the start of its segment
            first = max(s for s in starts if s <= c)
            assert (c - first) % slots == 0
