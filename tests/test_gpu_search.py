"""The drop-in list's grid search at its edges: bins with more atoms than the waves of a bin take
in one turn, empty bins, grids of one, two, three and four bins along an axis, atoms on the faces.
The pair index [2, C] is compared bit for bit with the oracle's and the full rows with the same
pairs in both orientations; whole numbers, so no tolerance."""

import numpy as np
import pytest
import torch

from nabladyn_amd.neighbors import NeighborList
from oracle import neighbors as on

pytestmark = pytest.mark.gpu

CELLS = [
    (4.9, 4.9, 4.9),   # four bins an axis: most bins touch a face
    (3.7, 6.1, 8.5),   # three bins along x
    (2.5, 6.1, 3.7),   # two along x: minimum image per pair
    (8.5, 2.5, 2.5),   # two along y and z
]


def _frame(kind, cell, rng):
    cell = np.array(cell)
    if kind == "sparse":  # under two atoms a bin: a lane per center
        return rng.uniform(0, 1, (40, 3)) * cell
    if kind == "dense":  # more atoms a bin than 16 waves of 4 or 8 centers take at once
        return rng.uniform(0, 1, (6000, 3)) * cell
    if kind == "clustered":  # most atoms in one corner, most bins empty
        x = rng.normal(0, 0.15, (900, 3))
        return np.concatenate([x, rng.uniform(0, 1, (60, 3)) * cell])
    x = rng.uniform(0, 1, (700, 3)) * cell  # "faces": a third of the atoms on a face
    x[::3, 0] = 0.0
    x[1::6, 1] = cell[1]
    return x


@pytest.mark.parametrize("dtype,npdt", [(torch.float32, np.float32), (torch.float64, np.float64)])
@pytest.mark.parametrize("kind", ["sparse", "dense", "clustered", "faces"])
@pytest.mark.parametrize("cell", CELLS)
def test_search_at_its_edges(device, dtype, npdt, kind, cell):
    x = _frame(kind, cell, np.random.default_rng(17))
    L = np.array(cell).astype(npdt)
    wrapped, _ = on.wrap(x.astype(npdt), L)
    ref = on.build(wrapped, L, npdt(1.2), capacity_multiplier=1.25)
    for full in (True, False):
        nl = NeighborList(1.0, skin=0.2, full=full)
        nl.allocate(torch.tensor(x, dtype=dtype, device=device),
                    torch.tensor(L, dtype=dtype, device=device))
        assert not nl.all_pairs
        index = nl.tensors().index.cpu().numpy()
        np.testing.assert_array_equal(index, ref.pairs)
        if full:
            half = on.pair_set(index, nl.num_pairs)
            rows = nl.tensors().full
            counts, slices, entries, ids = (v.cpu().numpy() for v in (
                rows.counts, rows.slices, rows.index, rows.rows))
            got = np.concatenate([
                np.stack([np.full(c, ids[r]), entries[slices[r // 64] + r % 64 + 64 * np.arange(c)]],
                         axis=1) for r, c in enumerate(counts)])
            both = np.concatenate([half, half[:, ::-1]])
            key = lambda a: a[np.lexsort((a[:, 1], a[:, 0]))]  # noqa: E731
            np.testing.assert_array_equal(key(got), key(both))


@pytest.mark.parametrize("dims", [161, 162])
def test_scan_of_many_bins(device, dims):
    """The bins' scan with each block adding up the tile sums before it (161^3 bins, 4,076 tiles)
    and with a launch that scans them (162^3 bins, 4,152 tiles)."""
    cell = np.full(3, dims * 0.1 + 0.01, dtype=np.float32)
    rng = np.random.default_rng(3)
    x = (rng.uniform(0, 1, (4000, 3)) * cell).astype(np.float32)
    x[::2] = x[1::2] + rng.normal(0, 0.02, (2000, 3))  # a neighbor for most atoms
    wrapped, _ = on.wrap(x, cell)
    ref = on.build(wrapped, cell, np.float32(0.1), capacity_multiplier=1.25)
    nl = NeighborList(0.1)
    nl.allocate(torch.tensor(x, device=device), torch.tensor(cell, device=device))
    assert nl._device.buffers["bin_counts"].numel() == dims**3 + 1
    assert ref.pair_total > 1000
    np.testing.assert_array_equal(nl.tensors().index.cpu().numpy(), ref.pairs)


@pytest.mark.parametrize("n", [65472, 65473, 70000])
def test_scan_of_many_slices(device, n):
    """The slices' scan, in the columns' launches, over one tile and over two: 1,024 entries, one
    more, and some more. Each slice is 64 times as long as its longest row, the last the total."""
    rng = np.random.default_rng(n)
    cell = np.full(3, (n / 21.0) ** (1 / 3), dtype=np.float32)
    x = (rng.uniform(0, 1, (n, 3)) * cell).astype(np.float32)
    nl = NeighborList(0.5)
    nl.allocate(torch.tensor(x, device=device), torch.tensor(cell, device=device))
    wrapped, _ = on.wrap(x, cell)
    ref = on.build(wrapped, cell, np.float32(0.5), capacity_multiplier=1.25)
    np.testing.assert_array_equal(nl.tensors().index.cpu().numpy(), ref.pairs)
    rows = nl.tensors().full
    counts, slices = rows.counts.cpu().numpy(), rows.slices.cpu().numpy()
    padded = np.zeros(-(-n // 64) * 64, np.int64)
    padded[:n] = counts
    np.testing.assert_array_equal(np.diff(slices), 64 * padded.reshape(-1, 64).max(axis=1))
    assert slices[0] == 0 and counts.sum() == 2 * ref.pair_total


@pytest.mark.parametrize("dtype,npdt", [(torch.float32, np.float32), (torch.float64, np.float64)])
@pytest.mark.parametrize("shift", [0, 1, 37])
def test_bins_of_more_atoms_than_a_block_takes(device, dtype, npdt, shift):
    """Bins that hold around one, two and three blocks' share of centers (64), and one that holds
    many tiles of candidates, at slots before and after a multiple of the share."""
    rng = np.random.default_rng(shift)
    width, per = 1.0, 6
    cell = np.full(3, per * width * 1.001).astype(npdt)
    crowded = {(1, 1, 1): 63, (3, 1, 1): 64, (5, 1, 2): 65, (0, 3, 0): 127, (2, 3, 5): 128,
               (4, 4, 3): 129, (5, 5, 5): 192, (3, 3, 2): 193, (0, 0, 3): 2500}
    x = [(np.array(bin) + rng.uniform(0.05, 0.95, (count, 3))) * width
         for bin, count in crowded.items()]
    x.append(np.full((shift, 3), 0.5) + rng.uniform(-0.3, 0.3, (shift, 3)))  # in the first bin
    x.append(rng.uniform(0, per * width, (700, 3)))
    x = rng.permutation(np.concatenate(x))
    wrapped, _ = on.wrap(x.astype(npdt), cell)
    ref = on.build(wrapped, cell, npdt(width), capacity_multiplier=1.25)
    for full in (True, False):
        nl = NeighborList(width, full=full)
        nl.allocate(torch.tensor(x, dtype=dtype, device=device),
                    torch.tensor(cell, dtype=dtype, device=device))
        buffers = nl._device.buffers
        assert buffers["bin_counts"].numel() == per**3 + 1
        occupied = np.diff(buffers["bin_offsets"].cpu().numpy())
        assert np.sum(occupied > 64) >= 6 and occupied.max() > 2048
        np.testing.assert_array_equal(nl.tensors().index.cpu().numpy(), ref.pairs)
        if full:
            rows = nl.tensors().full
            assert int(rows.counts.sum()) == 2 * nl.num_pairs
