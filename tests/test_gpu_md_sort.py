"""The MD build's one-block sort at the edges of its sizes: everything but the fill in one block
(to 1,024 atoms), the sort alone (to 65,536 atoms), and the separate launches past it. After a run
with rebuilds the resident list holds exactly the pairs within its radius of the frame it was
built on, in both orientations, and the frame read out in atom order is a permutation's inverse:
whole numbers, so no tolerance (the pairs by the oracle's cell list)."""

import numpy as np
import pytest
import torch

from nabladyn_amd import md, potential, workloads
from oracle import neighbors as on

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [343, 1023, 1024, 1025, 3000, 65536, 65537])
def test_builds_of_every_size(device, dtype, n):
    per = int(np.ceil(n ** (1 / 3)))
    length = per * 0.3625
    x = workloads.lattice((per,) * 3, (length,) * 3, 0.02, np.random.default_rng(n), n=n)
    x = np.random.default_rng(7).permutation(x)
    masses = torch.full((n,), workloads.ARGON_MASS, dtype=dtype, device=device)
    model = potential.lennard_jones(
        atom_types=torch.zeros(n, dtype=torch.int64, device=device),
        sigma=torch.tensor([0.34], dtype=dtype, device=device),
        epsilon=torch.tensor([0.996], dtype=dtype, device=device), cutoff=1.0)
    sim = md.nve(model, torch.tensor(x, dtype=dtype, device=device),
                 md.maxwell_boltzmann(masses, 120.0, 1), masses,
                 torch.full((3,), length, dtype=dtype, device=device), timestep=0.004, skin=0.1)
    sim.run(60)
    nb = sim._neighbors
    assert nb._rebuild_count > 1
    ids = nb.buffers["ids"].cpu().numpy()
    np.testing.assert_array_equal(np.sort(ids), np.arange(n))
    # sorted by sub-bin, then by atom id
    offsets = nb.buffers["bin_offsets"].cpu().numpy()
    assert offsets[0] == 0 and offsets[-1] == n
    starts = np.zeros(n, bool)
    starts[offsets[:-1][offsets[:-1] < n]] = True
    assert np.all((np.diff(ids) > 0) | starts[1:])
    # the frame of the last build, in atom order
    slots = nb.reference_positions.cpu().numpy()
    built = np.empty_like(slots)
    built[ids] = slots
    cell = sim.cell.cpu().numpy()
    ref = on.build(built, cell, built.dtype.type(nb.radius))
    half = on.pair_set(ref.pairs, ref.pair_total)
    both = np.concatenate([half, half[:, ::-1]])
    got = nb.atom_pairs().numpy()
    key = lambda a: a[np.lexsort((a[:, 1], a[:, 0]))]  # noqa: E731
    np.testing.assert_array_equal(key(got), key(both))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [500, 1500])
@pytest.mark.parametrize("dims", [(27, 35, 39), (32, 32, 36), (34, 35, 36)])
def test_builds_of_dilute_boxes(device, dtype, n, dims):
    """The other bound of the one-block sort, the 36,863 sub-bins whose counts its LDS holds: a drop
    in a large box, with a few sub-bins less (27 x 35 x 39 = 36,855, the sort at its largest), one
    more and more, which take the separate launches."""
    length = np.array(dims) * 0.5505
    per = int(np.ceil(n ** (1 / 3)))
    x = workloads.lattice((per,) * 3, (per * 0.38,) * 3, 0.02, np.random.default_rng(n), n=n)
    x = np.random.default_rng(7).permutation(x) - 0.7  # over three faces
    masses = torch.full((n,), workloads.ARGON_MASS, dtype=dtype, device=device)
    model = potential.lennard_jones(
        atom_types=torch.zeros(n, dtype=torch.int64, device=device),
        sigma=torch.tensor([0.34], dtype=dtype, device=device),
        epsilon=torch.tensor([0.996], dtype=dtype, device=device), cutoff=1.0)
    sim = md.nve(model, torch.tensor(x, dtype=dtype, device=device),
                 md.maxwell_boltzmann(masses, 60.0, 1), masses,
                 torch.tensor(length, dtype=dtype, device=device), timestep=0.004, skin=0.1)
    assert tuple(sim._neighbors.dims) == dims
    sim.run(100)
    nb = sim._neighbors
    assert nb._rebuild_count > 1
    ids = nb.buffers["ids"].cpu().numpy()
    np.testing.assert_array_equal(np.sort(ids), np.arange(n))
    offsets = nb.buffers["bin_offsets"].cpu().numpy()
    assert offsets[0] == 0 and offsets[-1] == n and np.all(np.diff(offsets) >= 0)
    built = np.empty((n, 3), nb.reference_positions.cpu().numpy().dtype)
    built[ids] = nb.reference_positions.cpu().numpy()
    cell = sim.cell.cpu().numpy()
    pairs = on.brute_pairs(built, cell, built.dtype.type(nb.radius))
    both = np.concatenate([pairs, pairs[:, ::-1]])
    key = lambda a: a[np.lexsort((a[:, 1], a[:, 0]))]  # noqa: E731
    np.testing.assert_array_equal(key(nb.atom_pairs().numpy()), key(both))
