"""What a first frame's host code reads back, and the wraps with no crossings: the same bits as
``space.wrap``, frame by frame; a coordinate that is not finite is found wherever it lies; strided
and transposed inputs; a list's own tensors do not share memory that another writes."""

import numpy as np
import pytest
import torch

from nabladyn_amd import space
from nabladyn_amd.neighbors import NeighborList
from oracle import neighbors as on

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_wraps_are_the_wrap(device, dtype):
    rng = np.random.default_rng(1)
    x = torch.tensor(rng.normal(0, 9, (5, 301, 3)), dtype=dtype, device=device)
    cells = torch.tensor(rng.uniform(1, 6, (7, 3)), dtype=dtype, device=device)
    frames = space.wrapped_frames(x, cells)
    for f in range(5):
        expected, _ = space.wrap(x[f], cells[f])
        assert torch.equal(frames[f], expected)
        assert torch.equal(space.wrapped(x[f], cells[f]), expected)
    turned = x.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    assert torch.equal(space.wrapped_frames(turned, cells), frames)
    with pytest.raises(ValueError):
        space.wrapped_frames(x, cells[:4])
    with pytest.raises(TypeError):
        space.wrapped_frames(x.cpu(), cells)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("atom", [0, 1333, 2743])
def test_a_coordinate_that_is_not_finite(device, dtype, value, atom):
    x = torch.tensor(on.jittered_lattice(14, 5.1, 0.02, seed=2), dtype=dtype, device=device)
    cell = torch.full((3,), 5.1, dtype=dtype, device=device)
    x[atom, atom % 3] = value
    with pytest.raises(ValueError, match="finite"):
        NeighborList(1.0).allocate(x, cell)


@pytest.mark.parametrize("n,full", [(1, True), (2, False), (343, True), (5000, True)])
def test_a_lists_tensors_are_apart(device, n, full):
    per = max(1, int(np.ceil(n ** (1 / 3))))
    length = max(2.2, 0.3625 * per)
    x = torch.tensor(on.jittered_lattice(per, length, 0.02, seed=2)[:n], dtype=torch.float32,
                     device=device)
    nl = NeighborList(1.0, full=full)
    strided = x.t().contiguous().t()
    nl.allocate(strided, torch.full((3,), length, device=device))
    dev = nl._device
    tensors = [*dev.buffers.values(), *dev.reuse.values(), *(dev.full or {}).values()]
    spans = sorted((t.data_ptr(), t.data_ptr() + t.numel() * t.element_size())
                   for t in tensors if t.numel())
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    assert all(t.data_ptr() % 8 == 0 for t in tensors)
    ref = on.build(on.wrap(x.cpu().numpy(), np.full(3, length, np.float32))[0],
                   np.full(3, length, np.float32), np.float32(1.0))
    np.testing.assert_array_equal(nl.tensors().index.cpu().numpy(), ref.pairs)
    assert nl._rebuild_count == 1 and nl.num_pairs == ref.pair_total
