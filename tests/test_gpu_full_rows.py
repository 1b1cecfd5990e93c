"""E, F and W over full rows at the edges of their launch: one, four and sixteen waves to a slice
of 64 rows (the counts on both sides of each line, a last slice of one row), and a one-type table
staged in LDS against the largest that is and the first that is not. Tolerance as in the force
tests: fp64 1e-12 (tables 3e-12) against the oracle's closed forms; fp32 LJ 1e-5, and a table
1e-5 of the reference's own fp32 route."""

import numpy as np
import pytest
import torch

from nabladyn_amd import potential, quantity, workloads
from nabladyn_amd.neighbors import NeighborList
from oracle import neighbors as on
from oracle import potentials as op
from _parity import check_against_route, rel, table_route

pytestmark = pytest.mark.gpu


def _evaluate(n, dtype, device, build):
    per = int(np.ceil(n ** (1 / 3)))
    length = per * 0.3625
    x = workloads.lattice((per,) * 3, (length,) * 3, 0.02, np.random.default_rng(n), n=n)
    x = np.random.default_rng(5).permutation(x)
    xd = torch.tensor(x, dtype=dtype, device=device)
    cell = torch.full((3,), length, dtype=dtype, device=device)
    model = build(torch.zeros(n, dtype=torch.int64, device=device))
    nl = NeighborList(model.cutoff)
    nl.allocate(xd, cell)
    e, f, w = quantity.energy_force_virial(model)(xd, cell, nl.tensors())
    xw = on.wrap(xd.cpu().numpy(), cell.cpu().numpy())[0]
    b = on.build(xw, cell.cpu().numpy(), xw.dtype.type(model.cutoff))
    return model, (float(e), f.cpu().numpy(), w.cpu().numpy()), xw, cell.cpu().numpy(), \
        b.pairs[:, :b.pair_total]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [400, 8128, 8129, 262081])
def test_waves_of_a_slice(device, dtype, n):
    def build(types):
        return potential.lennard_jones(
            atom_types=types, sigma=torch.tensor([0.34], dtype=dtype, device=device),
            epsilon=torch.tensor([0.996], dtype=dtype, device=device), cutoff=1.0)

    model, (e, f, w), xw, cell, pairs = _evaluate(n, dtype, device, build)
    e0, f0, w0 = op.lj_efw(xw.astype(np.float64), cell.astype(np.float64), pairs,
                           np.zeros(n, np.int64), model.sigma.detach().cpu().numpy(),
                           model.epsilon.detach().cpu().numpy(), 1.0)
    bar = 1e-5 if dtype == torch.float32 else 1e-12
    assert rel(f, f0) <= bar
    assert rel(w, w0) <= bar
    assert abs(e - e0) <= bar * max(1.0, abs(e0))


@pytest.mark.parametrize("dtype,knots", [(torch.float32, 4), (torch.float32, 1025),
                                         (torch.float32, 1026), (torch.float64, 513),
                                         (torch.float64, 514)])
def test_staged_tables(device, dtype, knots):
    r = 0.36 + np.arange(knots) * (1.2 - 0.36) / (knots - 1)  # some pairs below the first knot
    u = 4 * 0.996 * ((0.34 / r) ** 12 - (0.34 / r) ** 6)
    u[-1] = 0.0

    def build(types):
        return potential.tabulated(
            atom_types=types, table=torch.tensor(u[None], dtype=dtype, device=device),
            start=torch.tensor([0.36], dtype=dtype, device=device), cutoff=1.2)

    model, got, xw, cell, pairs = _evaluate(2000, dtype, device, build)
    args = (model.table.detach().cpu().numpy(), model.start.cpu().numpy())
    spacing = model.spacing.cpu().numpy()
    types = np.zeros(2000, np.int64)
    fp64 = op.table_efw(xw.astype(np.float64), cell.astype(np.float64), pairs, types, *args, 1.2,
                        spacing=spacing)
    if dtype == torch.float32:
        route = table_route(xw, cell, pairs, types, *args, spacing, 1.2)
        check_against_route(f"{knots} knots", got, route, fp64)
    else:
        assert rel(got[1], fp64[1]) <= 3e-12
        assert rel(got[2], fp64[2]) <= 3e-12
        assert abs(got[0] - fp64[0]) <= 3e-12 * max(1.0, abs(fp64[0]))
