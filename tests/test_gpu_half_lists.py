"""Energies and forces over half lists of any order: columns that are not a multiple of a wave, runs
of one first atom and none, padding and ids out of range between them, at no strain and at one, fp64
against the oracle's autograd on the CPU. Tolerance 1e-12 of the largest value, as the force
tests' (sums of some hundred terms of 1e-16 each)."""

import numpy as np
import pytest
import torch

from nabladyn_amd import potential
from nabladyn_amd.potential._energy import evaluate
from oracle import neighbors as on
from oracle import potentials as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strained", [False, True])
@pytest.mark.parametrize("order", ["runs", "shuffled"])
@pytest.mark.parametrize("columns", [1, 63, 64, 65, 700, 3001])
def test_columns_of_any_order(device, columns, order, strained):
    n, length = 343, 2.6
    rng = np.random.default_rng(columns)
    x = on.wrap(on.jittered_lattice(7, length, 0.02, seed=1), np.full(3, length))[0]
    pairs = on.brute_pairs(x, np.full(3, length), 0.9)[:columns]
    if order == "shuffled":
        pairs = rng.permutation(pairs)
        pairs = np.where(rng.random(len(pairs))[:, None] < 0.5, pairs, pairs[:, ::-1])
    listed = np.ascontiguousarray(pairs.T).astype(np.int32)
    if columns > 64:  # columns that are not pairs, anywhere
        holes = rng.integers(0, columns, 20)
        listed[:, holes[:10]] = 5
        listed[1, holes[10:15]] = n
        listed[0, holes[15:]] = -1
    kept = listed[:, (listed[0] != listed[1]) & (listed >= 0).all(0) & (listed < n).all(0)]
    f64 = dict(dtype=torch.float64)
    types = torch.tensor(rng.integers(0, 2, n))
    sigma, epsilon = torch.tensor([0.34, 0.33, 0.31], **f64), torch.tensor([0.9, 1.1, 0.7], **f64)
    strain = torch.tensor([[0.01, 0.003, -0.002], [0.004, -0.02, 0.001], [0.0, 0.005, 0.015]], **f64)
    strain = strain if strained else torch.zeros(3, 3, **f64)
    xt, cell = torch.tensor(x, **f64).requires_grad_(), torch.full((3,), length, **f64)
    e0 = op.t_lj_energy(xt, strain.requires_grad_(), cell, torch.tensor(kept).long(), types, sigma,
                        epsilon, 0.9)
    f0, w0 = (-g for g in torch.autograd.grad(e0, (xt, strain)))
    model = potential.lennard_jones(atom_types=types.to(device), sigma=sigma.to(device),
                                    epsilon=epsilon.to(device), cutoff=0.9)
    e, f, w = evaluate(model, xt.detach().to(device), cell.to(device),
                       torch.tensor(listed, device=device),
                       strain.detach().to(device) if strained else None)
    for got, want in ((e, e0.detach()), (f, f0), (w, w0)):
        assert float((got.cpu() - want).abs().max()) <= 1e-12 * max(1.0, float(want.abs().max()))
