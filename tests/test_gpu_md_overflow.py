"""Lists whose atoms crowd together after the first build. Free atoms (a negligible potential) fly
toward the middle of the box, so every later frame is known: x0 + v t. Positions to 2e-4 nm: some
100 steps, each of a rounding of some 5 nm in fp32 (2^-22) and a drift by the potential below
1e-6."""

import numpy as np
import pytest
import torch

from nabladyn_amd import md, potential
from nabladyn_amd.md._simulation import halo_limit

pytestmark = pytest.mark.gpu


def _gathering(device, dtype, n, length, shrink, steps):
    """A simulation of n atoms that draw together by the factor `shrink` over `steps` steps."""
    rng = np.random.default_rng(n)
    per = int(np.ceil(n ** (1 / 3)))
    grid = np.stack(np.meshgrid(*[np.arange(per)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (grid + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * length / per
    rate = (1.0 - shrink) / (steps * 0.004)
    mass = rng.permutation(np.arange(1.0, n + 1.0))
    v = -rate * (x - 0.5 * length)
    v -= (mass[:, None] * v).sum(0) / mass.sum()  # as a simulation does
    as_t = lambda a: torch.tensor(a, dtype=dtype, device=device)  # noqa: E731
    masses = as_t(mass)
    model = potential.lennard_jones(atom_types=torch.zeros(n, dtype=torch.int64, device=device),
                                    sigma=as_t([0.02]), epsilon=as_t([1e-9]), cutoff=1.0)
    sim = md.nve(model, as_t(x), as_t(v), masses, as_t([length] * 3), timestep=0.004, skin=0.1)
    return sim, x, v, masses


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_a_box_that_halos_span_may_gather(device, dtype):
    """64 atoms of a box seven sub-bins across end in one corner of a brick's halo: every row (64
    entries at least) and every halo has room for all of them."""
    sim, x, v, _ = _gathering(device, dtype, 64, 4.3, 0.3, 100)
    sim.run(100)
    expected = x + v * 0.4
    got = sim.state().positions.cpu().numpy()
    np.testing.assert_allclose(got, expected, rtol=0, atol=2e-4)
    assert sim._neighbors._rebuild_count > 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [1000, 1500, 5000])
def test_a_row_overflow_moves_the_whole_frame(device, dtype, n):
    """Rows that outgrow their entries stop a run with its error; the build that met them has still
    put every atom home: each slot's mass and place are those of the atom it names. (1,000 atoms
    take the build of one block and a fill, the others the launches that unpack beside the fill.)"""
    length = 0.62 * np.ceil(n ** (1 / 3))
    sim, x, v, masses = _gathering(device, dtype, n, length, 0.5, 100)
    with pytest.raises(ValueError, match="a neighbor row needs"):
        sim.run(100)
    ids = sim._neighbors.buffers["ids"].cpu().numpy()
    np.testing.assert_array_equal(np.sort(ids), np.arange(n))
    np.testing.assert_array_equal(sim.slot_masses.cpu().numpy(), masses.cpu().numpy()[ids])
    got = sim.positions.cpu().numpy()
    np.testing.assert_allclose(got, (x + v * 0.4)[ids], rtol=0, atol=2e-4)


@pytest.mark.parametrize("dtype,point", [(torch.float32, 16), (torch.float64, 32)])
def test_a_halo_may_take_half_a_units_lds(device, dtype, point):
    """The largest halo: half of a compute unit's 160 KB, less 656 bytes of a block's own. 6,000 atoms
    of some 200 bricks take all of it, and run."""
    limit = halo_limit(dtype)
    assert limit >= (160 * 1024 // 2 - 656) // point - 1
    sim, x, v, _ = _gathering(device, dtype, 6000, 0.4 * 19, 0.95, 20)
    assert sim._neighbors.halo_capacity == min(limit, 6000)
    sim.run(20)
    got = sim.state().positions.cpu().numpy()
    np.testing.assert_allclose(got, x + v * 0.08, rtol=0, atol=2e-4)
