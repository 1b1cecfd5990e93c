"""The knot coordinate of a table's pairs, (r - start) / h, at knots and next to them: the
reference's square root, subtraction and division, each correctly rounded, through the table in
LDS (one type) and the rows in memory (two types), in the list's kernels and the MD step's.

Isolated pairs along x, from x = 0, so a pair's r is its second atom's x. The tables are random
between -1 and 1 over 1,024 segments, and numpy forms the coordinate in the dtype, which its
operations round correctly; the cubic there in fp64. With a, b, c its terms the kernel's slope
rounds some 16 times by 2^-24 (2^-53 in fp64) of |a| + 2 |b| + 3 |c|; a coordinate that is off by
an ulp moves it by 2^-15 of |b| at the 256th knot, 30 times that.

h = 2^-10 (2 - k ulp) with a small odd k has a reciprocal that Newton's steps from the hardware's
estimate do not round correctly in fp64 (k = 3, 5, .., 13), and offsets of powers of two have
quotients next to halfway between two numbers, which a reciprocal an ulp too large gets wrong."""

import numpy as np
import pytest
import torch

from nabladyn_amd import md, potential, quantity
from nabladyn_amd.neighbors import NeighborList

pytestmark = pytest.mark.gpu

KNOTS = 1025


def _distances(start, h, cutoff, kind, rng):
    one = kind(1)
    ulp = np.spacing(one)
    powers = start + kind(2.0) ** np.arange(-9, 1).astype(kind)
    at = (start + np.arange(1, KNOTS - 1).astype(kind) * h)[rng.permutation(KNOTS - 2)[:300]]
    r = np.concatenate([powers, at, np.nextafter(at, one), np.nextafter(at, kind(0)),
                        rng.uniform(0.2, float(cutoff) * 0.999, 300).astype(kind)])
    assert r.dtype == kind and ulp > 0
    return r[(r > 0.01) & (r < cutoff)]


def _slopes(table, row, r, start, h, kind):
    """(du/dr in fp64, the scale of its rounding) at the coordinate the dtype gives."""
    x = (r - start).astype(kind) / h
    assert x.dtype == kind
    segment = np.clip(np.floor(x), 0, KNOTS - 2).astype(int)
    t = (x - segment.astype(kind)).astype(np.float64)
    padded = np.empty((len(table), KNOTS + 2))
    padded[:, 1:-1] = table
    padded[:, 0] = 3 * table[:, 0] - 3 * table[:, 1] + table[:, 2]
    padded[:, -1] = 3 * table[:, -1] - 3 * table[:, -2] + table[:, -3]
    u0, u1, u2, u3 = (padded[row, segment + k] for k in range(4))
    a, b, c = u2 - u0, 2 * u0 - 5 * u1 + 4 * u2 - u3, 3 * (u1 - u2) + u3 - u0
    slope = 0.5 * (a + t * (2 * b + 3 * c * t)) / float(h)
    return slope, (abs(a) + 2 * abs(b) + 3 * abs(c)) / float(h)


@pytest.mark.parametrize("route", ["list", "md"])
@pytest.mark.parametrize("num_types", [1, 2])
@pytest.mark.parametrize("ulps", [1, 3, 5, None])
@pytest.mark.parametrize("dtype,kind", [(torch.float32, np.float32), (torch.float64, np.float64)])
def test_slopes_at_knots(device, dtype, kind, ulps, num_types, route):
    rng = np.random.default_rng(41)
    cutoff = kind(2.0)
    start = kind(0.1) if ulps is None else kind(ulps) * np.spacing(kind(1))
    h = kind(cutoff - start) / kind(KNOTS - 1)
    r = _distances(start, h, cutoff, kind, rng)
    count = len(r)
    per = int(np.ceil(np.sqrt(count)))
    length = 5.0 * per
    x = np.zeros((2 * count, 3), kind)
    x[0::2, 1] = x[1::2, 1] = 5.0 * (np.arange(count) % per) + 1
    x[0::2, 2] = x[1::2, 2] = 5.0 * (np.arange(count) // per) + 1
    x[1::2, 0] = r
    rows = num_types * (num_types + 1) // 2
    table = rng.uniform(-1, 1, (rows, KNOTS)).astype(kind)
    table[:, -1] = 0
    types = np.repeat(np.arange(count) % num_types, 2)
    row = np.array([0, 2])[types[0::2]] if num_types == 2 else np.zeros(count, int)
    as_t = lambda v: torch.tensor(v, dtype=dtype, device=device)  # noqa: E731
    model = potential.tabulated(
        atom_types=torch.tensor(types, dtype=torch.int64, device=device), table=as_t(table),
        start=as_t(np.full(rows, start)), cutoff=2.0)
    assert np.all(model.spacing.cpu().numpy() == h)
    cell = as_t([length] * 3)
    if route == "list":
        nl = NeighborList(2.0)
        nl.allocate(as_t(x), cell)
        forces = quantity.force(model)(as_t(x), cell, nl.tensors())
    else:
        masses = torch.ones(2 * count, dtype=dtype, device=device)
        sim = md.nve(model, as_t(x), torch.zeros_like(as_t(x)), masses, cell, timestep=0.001)
        forces = sim.state().forces
    forces = forces.double().cpu().numpy()
    slope, scale = _slopes(table.astype(np.float64), row, r, start, h, kind)
    bound = 16 * (2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53) * scale
    assert np.all(np.abs(forces[1::2, 0] + slope) <= bound)
    assert np.all(np.abs(forces[0::2, 0] - slope) <= bound)
