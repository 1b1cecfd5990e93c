"""The batch gradient of a fit from the kernels alone (channels, loss and VJP over a choice of the
stored frames) against the same through autograd, which a fit takes for parameters that are not
the model's own: a permuted, a repeated and a partial choice of frames, each subset of the
channels, one type, two types and a sum, force components on both sides of a loss block (1,365 and
1,366 atoms).

Tolerance. Both routes evaluate the same channels in the model's dtype and add the parameters'
pair sums in fp64; they differ by the rounding of the upstream gradients, some 3 ulp each and
independent over the components. fp64 1e-11 of max |g|, fp32 1e-5; the loss and its terms, sums of
squares in another order, 1e-12 and 1e-5 of themselves."""

import numpy as np
import pytest
import torch

from nabladyn_amd import potential, training, workloads
from nabladyn_amd.training import _fit

pytestmark = pytest.mark.gpu


def _model(kind, n, dtype, device):
    as_t = lambda v: torch.tensor(v, dtype=dtype, device=device)  # noqa: E731
    zeros = torch.zeros(n, dtype=torch.int64, device=device)
    table = lambda: potential.tabulated(  # noqa: E731
        atom_types=zeros, table=as_t(workloads.lj_table(40, noise=0.0, sigma=0.45)[None]),
        start=as_t([0.3]), cutoff=1.2, trainable=("table",))
    if kind == "table":
        return table()
    if kind == "mixture":
        types = torch.arange(n, device=device) % 2
        return potential.lennard_jones(atom_types=types, sigma=as_t([0.47, 0.46, 0.45]),
                                       epsilon=as_t([3.0, 3.1, 3.2]), cutoff=1.2,
                                       trainable=("sigma", "epsilon"))
    lj = potential.lennard_jones(atom_types=zeros, sigma=as_t([0.46]), epsilon=as_t([2.0]),
                                 cutoff=1.0, trainable=("epsilon",))
    return potential.sum(lj, table())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("kind,n,channels", [
    ("table", 1365, ("energy", "forces", "virial")), ("table", 1366, ("forces",)),
    ("mixture", 500, ("energy", "virial")), ("mixture", 500, ("forces", "virial")),
    ("sum", 500, ("energy", "forces", "virial")),
])
def test_kernel_gradient_equals_autograd(device, dtype, kind, n, channels):
    rng = np.random.default_rng(n)
    frames, length = 6, (n / 8.0) ** (1 / 3)
    per = int(np.ceil(n ** (1 / 3)))
    x = np.stack([workloads.lattice((per,) * 3, (length,) * 3, 0.04, rng, n=n)
                  for _ in range(frames)])
    labels = {"energy": rng.normal(0, 50, frames), "forces": rng.normal(0, 30, (frames, n, 3)),
              "virial": rng.normal(0, 80, (frames, 3, 3))}
    as_np = lambda v: np.asarray(v).astype(np.float32 if dtype == torch.float32 else np.float64)  # noqa: E731
    data = training.Dataset(as_np(x), as_np(np.full((frames, 3), length)),
                            **{k: as_np(labels[k]) for k in channels})
    model = _model(kind, n, dtype, device)
    prepared = _fit._prepare(model, data, channels)
    scales = training.scales(**prepared.labels)
    weights = {name: 0.5 + k for k, name in enumerate(channels)}
    own = {name: p for name, p in model.named_parameters() if p.requires_grad}
    copies = {name: p.detach().clone() for name, p in own.items()}
    assert _fit._kernel_parts(model, own, prepared) is not None
    assert _fit._kernel_parts(model, copies, prepared) is None
    loose, tight = (1e-5, 1e-5) if dtype == torch.float32 else (1e-11, 1e-12)
    for chosen, size in (([3, 0, 5, 1, 4, 2], 6), ([2, 2, 0], 3), ([4, 1, 3], 2), ([5], 1)):
        chosen = torch.tensor(chosen)
        g, loss, terms = _fit.batch_gradient(model, own, prepared, chosen, size, weights, scales)
        g0, loss0, terms0 = _fit.batch_gradient(model, copies, prepared, chosen, size, weights,
                                                scales)
        assert set(g) == set(g0) and set(terms) == set(terms0) == set(channels)
        for name in g:
            assert g[name].dtype == g0[name].dtype and g[name].shape == g0[name].shape
            assert float((g[name] - g0[name]).abs().max()) <= loose * float(g0[name].abs().max())
        assert abs(float(loss) - float(loss0)) <= tight * abs(float(loss0))
        for name in terms:
            assert abs(float(terms[name]) - float(terms0[name])) <= tight * abs(float(terms0[name]))


def _shared(kind, n, dtype, device, tied):
    """A model in which one tensor trains under more than one name; untied, the same model with a
    tensor of its own for each name."""
    as_t = lambda v: torch.tensor(v, dtype=dtype, device=device)  # noqa: E731
    zeros = torch.zeros(n, dtype=torch.int64, device=device)
    lj = lambda sigma, epsilon, cutoff: potential.lennard_jones(  # noqa: E731
        atom_types=zeros, sigma=as_t([sigma]), epsilon=as_t([epsilon]), cutoff=cutoff,
        trainable=("sigma", "epsilon"))
    if kind == "one tensor in one part":
        only = lj(0.46, 0.46, 1.0)
        if tied:
            only.epsilon = only.sigma
        return only
    first, second = lj(0.46, 2.0, 1.0), lj(0.44, 2.0, 1.2)
    again = first if tied else lj(0.46, 2.0, 1.0)
    if kind == "one part twice":
        return potential.sum(first, again)
    if tied:
        second.epsilon = first.epsilon
    return potential.sum(first, potential.sum(second, again))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("kind", ["one part twice", "one tensor in one part",
                                  "one tensor in two parts"])
def test_shared_parameters_get_every_use(device, dtype, kind):
    n, frames = 300, 4
    rng = np.random.default_rng(5)
    length = (n / 8.0) ** (1 / 3)
    x = np.stack([workloads.lattice((7,) * 3, (length,) * 3, 0.04, rng, n=n)
                  for _ in range(frames)])
    as_np = lambda v: np.asarray(v).astype(np.float32 if dtype == torch.float32 else np.float64)  # noqa: E731
    channels = ("energy", "forces", "virial")
    data = training.Dataset(as_np(x), as_np(np.full((frames, 3), length)),
                            energy=as_np(rng.normal(0, 50, frames)),
                            forces=as_np(rng.normal(0, 30, (frames, n, 3))),
                            virial=as_np(rng.normal(0, 80, (frames, 3, 3))))
    model = _shared(kind, n, dtype, device, True)
    twin = _shared(kind, n, dtype, device, False)
    prepared = _fit._prepare(model, data, channels)
    scales = training.scales(**prepared.labels)
    weights = {name: 1.0 for name in channels}
    own = dict(model.named_parameters())
    chosen = torch.arange(frames)
    g, loss, _ = _fit.batch_gradient(model, own, prepared, chosen, 3, weights, scales)
    # through autograd, a tensor for each use, then the uses of one tensor added
    copies = {name: p.detach().clone() for name, p in twin.named_parameters()}
    uses, loss0, _ = _fit.batch_gradient(twin, copies, prepared, chosen, 3, weights, scales)
    names = {id(p): name for name, p in own.items()}
    g0 = {name: torch.zeros_like(p) for name, p in own.items()}
    for name, p in model.named_parameters(remove_duplicate=False):
        g0[names[id(p)]] += uses[name]
    assert set(g) == set(g0)
    # the parts' sums in fp64, each rounded and then added: an ulp a use beside the bounds above
    loose = 1e-5 if dtype == torch.float32 else 1e-11
    for name in g:
        assert float((g[name] - g0[name]).abs().max()) <= loose * float(g0[name].abs().max()), name
    assert abs(float(loss) - float(loss0)) <= loose * abs(float(loss0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_labels_of_any_strides(device, dtype):
    n, frames = 300, 5
    rng = np.random.default_rng(6)
    kind = np.float32 if dtype == torch.float32 else np.float64
    length = (n / 8.0) ** (1 / 3)
    x = np.stack([workloads.lattice((7,) * 3, (length,) * 3, 0.04, rng, n=n)
                  for _ in range(frames)]).astype(kind)
    cells = np.full((frames, 3), length, kind)
    labels = {"energy": rng.normal(0, 50, frames).astype(kind),
              "forces": rng.normal(0, 30, (frames, n, 3)).astype(kind),
              "virial": rng.normal(0, 80, (frames, 3, 3)).astype(kind)}
    strided = {"energy": torch.tensor(np.repeat(labels["energy"], 2))[::2],
               "forces": torch.tensor(labels["forces"].transpose(0, 2, 1).copy()).transpose(1, 2),
               "virial": np.asfortranarray(labels["virial"])}
    model = _model("table", n, dtype, device)
    own = dict(model.named_parameters())
    out = []
    for given in (labels, strided):
        data = training.Dataset(x, cells, **given)
        prepared = _fit._prepare(model, data, tuple(labels))
        out.append(_fit.batch_gradient(model, own, prepared, torch.tensor([3, 0, 4]), 2,
                                       {name: 1.0 for name in labels},
                                       training.scales(**prepared.labels)))
    # the same numbers in the same order; the scales and the VJP's sums (atomics) in another order
    loose = 1e-5 if dtype == torch.float32 else 1e-11
    for name in out[0][0]:
        a, b = out[0][0][name], out[1][0][name]
        assert float((a - b).abs().max()) <= loose * float(a.abs().max())
    for name in labels:
        assert abs(float(out[0][2][name]) - float(out[1][2][name])) <= loose * abs(float(out[0][2][name]))
