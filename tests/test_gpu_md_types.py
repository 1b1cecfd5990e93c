"""The MD force kernel over Lennard-Jones models of several types: up to 8 types' coefficients are
staged in LDS as a square, those of more are read from the triangle of unordered pairs. Forces,
virial and energy against the oracle's closed form in fp64 on the frame the simulation holds.

Tolerances: fp64 3e-12 of the largest value (sums of some hundred terms of 1e-15 each, with room
for their cancellation). fp32 3e-5: a displacement of placed positions is off by up to 2.4e-7 of
4 nm, 1.5e-6 of the shortest distances, which a force takes to the 14th power."""

import numpy as np
import pytest
import torch

from nabladyn_amd import md, potential
from oracle import neighbors as on
from oracle import potentials as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tolerance", [(torch.float32, 3e-5), (torch.float64, 3e-12)])
@pytest.mark.parametrize("num_types", [2, 3, 8, 9, 20])
def test_typed_lj_forces(device, dtype, tolerance, num_types):
    n, length = 1331, 4.0
    rng = np.random.default_rng(num_types)
    x = on.jittered_lattice(11, length, 0.03, seed=num_types)
    rows = num_types * (num_types + 1) // 2
    sigma, epsilon = rng.uniform(0.26, 0.36, rows), rng.uniform(0.4, 1.4, rows)
    types = rng.integers(0, num_types, n)
    model = potential.lennard_jones(
        atom_types=torch.tensor(types, dtype=torch.int64, device=device),
        sigma=torch.tensor(sigma, dtype=dtype, device=device),
        epsilon=torch.tensor(epsilon, dtype=dtype, device=device), cutoff=0.9)
    sigma = model.sigma.cpu().double().numpy()
    epsilon = model.epsilon.cpu().double().numpy()
    xd = torch.tensor(x, dtype=dtype, device=device)
    cell = torch.full((3,), length, dtype=dtype, device=device)
    masses = torch.full((n,), 39.948, dtype=dtype, device=device)
    sim = md.nve(model, xd, torch.zeros_like(xd), masses, cell, timestep=0.002, skin=0.1)
    xw = on.wrap(xd.cpu().numpy(), cell.cpu().numpy())[0].astype(np.float64)
    box = np.full(3, length)
    pairs = on.brute_pairs(xw, box, 0.9).T.copy()
    E0, F0, W0 = op.lj_efw(xw, box, pairs, types, sigma, epsilon, 0.9)
    F = sim._to_atoms(sim.forces).cpu().numpy()
    W = sim.virial.cpu().numpy()
    assert np.abs(F - F0).max() <= tolerance * np.abs(F0).max()
    assert np.abs(W - W0).max() <= tolerance * np.abs(W0).max()
    assert abs(float(sim.energy) - E0) <= tolerance * max(1.0, abs(E0))
