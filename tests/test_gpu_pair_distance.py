"""The fp64 root and reciprocals of the pair kernels: isolated pairs over the whole range of
distances, each pair's force against numpy's correctly rounded root and division.

The table is linear between knots of a power-of-two spacing, so a pair's force is its slope times
the unit vector, in a handful of roundings: 8 of 2^-53 relative. An atom pair is along x, so the
force's x is the slope itself to within those. (A linear table's slope is the same wherever the
knot coordinate falls: test_gpu_knot_coordinate.py has the quotient that gives it.)"""

import numpy as np
import pytest
import torch

from nabladyn_amd import potential, quantity
from nabladyn_amd.neighbors import NeighborList

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_types", [1, 2])
def test_forces_over_the_range_of_distances(device, num_types):
    pairs, knots, spacing = 512, 129, 2.0 ** -7
    r = np.linspace(1e-3, 0.999, pairs)
    x = np.zeros((2 * pairs, 3))
    grid = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3) * 4.0
    x[0::2] = grid + 1.0
    x[1::2] = grid + 1.0
    x[1::2, 0] += r
    rows = num_types * (num_types + 1) // 2
    table = np.stack([(knots - 1 - np.arange(knots)) * spacing * (k + 1) for k in range(rows)])
    types = np.repeat(np.arange(pairs) % num_types, 2)
    row = np.array([0, 2])[types[0::2]] if num_types == 2 else np.zeros(pairs, np.int64)
    f64 = dict(dtype=torch.float64, device=device)
    model = potential.tabulated(
        atom_types=torch.tensor(types, dtype=torch.int64, device=device),
        table=torch.tensor(table, **f64), start=torch.zeros(rows, **f64), cutoff=1.0)
    xd, cell = torch.tensor(x, **f64), torch.full((3,), 32.0, **f64)
    nl = NeighborList(1.0)
    nl.allocate(xd, cell)
    energy, forces = quantity.energy_and_force(model)(xd, cell, nl.tensors())
    forces = forces.cpu().numpy()
    slope = row + 1.0
    np.testing.assert_allclose(forces[1::2, 0], slope, rtol=8 * 2.0 ** -53, atol=0)
    np.testing.assert_allclose(forces[0::2, 0], -slope, rtol=8 * 2.0 ** -53, atol=0)
    np.testing.assert_allclose(float(energy), (slope * (1.0 - (x[1::2, 0] - x[0::2, 0]))).sum(),
                               rtol=1e-12)
