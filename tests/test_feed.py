"""What the feeder puts on the GPU for molecules held in different forms, against the data set's own batches; and energies and
gradients from one pass against those from two."""
import numpy as np
import pytest
import torch

from khan_amd import batching, model, ops

pytestmark = pytest.mark.gpu

FORMS = {"rows": lambda m: m, "columns": np.asfortranarray, "single": lambda m: m.astype(np.float32), "lists": lambda m: m.tolist()}


def _molecules(sizes, seed=5):
    rng = np.random.default_rng(seed)
    return [np.concatenate([rng.integers(0, 4, (n, 1)).astype(np.float64), rng.uniform(0.0, 1.4 * max(n, 1) ** (1 / 3), (n, 3))], axis=1)
            for n in sizes]


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("labelled", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_feeder_takes_molecules_in_any_form(form, labelled, dtype):
    sizes = [3, 1, 63, 64, 65, 257, 13, 32, 33, 5, 2]          # the size classes' edges, and the padding of the buffer
    mols = [FORMS[form](m) for m in _molecules(sizes)]
    raw = batching.RawDataset(mols, list(range(len(mols))) if labelled else None)
    for batch_size in (4, 11):
        feeder = batching.DeviceFeeder(raw, batch_size, dtype=dtype)
        for b, (rows, ids, labels, _) in zip(feeder, raw.iterate(batch_size, False)):
            b.wait()
            want = batching.split_columns(rows, ids, dtype)
            for got, ref in zip((b.xs, b.ys, b.zs, b.atom_types, b.mol_idxs), want):
                assert got.cpu().numpy().dtype == ref.dtype and np.array_equal(got.cpu().numpy(), ref)
            macs, mos = ops.mol_offsets(b.mol_idxs, b.n_mols)
            assert torch.equal(macs, b.mol_atom_counts) and torch.equal(mos, b.mol_offsets)
            assert b.labels == labels and b.host_sizes() == macs.tolist()
            acs, _, classes = b.host_counts()
            assert acs == np.bincount(want[3], minlength=4).tolist()
            assert isinstance(classes, torch.Tensor) and classes.dtype == torch.int32
            assert classes.tolist() == np.histogram(macs.cpu().numpy(), [0, 33, 65, 257, 10 ** 9])[0].tolist()


@pytest.mark.parametrize("fit_charges", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_energies_and_gradients_from_one_pass(fit_charges, dtype):
    m = model.AniModel(dtype=dtype, fit_charges=fit_charges, seed=2)
    raw = batching.RawDataset(_molecules([9, 1, 13, 40, 70, 3]))
    energies, gradients = m.predict(raw), list(m.coordinate_gradients(raw, 4))
    both = list(m.energies_and_gradients(raw, 4))
    assert len(both) == len(energies) == len(gradients) == 6
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    for (e, g), e_ref, g_ref in zip(both, energies, gradients):
        assert isinstance(e, float) and abs(e - e_ref) <= tol * (1.0 + abs(e_ref))
        assert g.shape == g_ref.shape and g.dtype == g_ref.dtype and np.abs(g - g_ref).max() <= tol * (1.0 + np.abs(g_ref).max())


@pytest.mark.parametrize("of", [float, np.float32, np.int64, lambda v: torch.tensor(v), lambda v: torch.tensor(float(v))])
def test_counts_of_any_kind_of_number(of):
    """Atom counts and class totals as int() takes them: Python and numpy floats, zero-dimensional tensors, and whole tensors of
    another type."""
    m = _molecules([9, 40, 70])
    b = next(iter(batching.DeviceFeeder(batching.RawDataset(m, [0.0] * 3), 3))).wait()
    acs, order, classes = b.host_counts()
    args = (b.xs, b.ys, b.zs, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs)
    want = ops.featurize(*args, list(acs), order=order, size_classes=classes)
    for counts, totals in (([of(v) for v in acs], [of(v) for v in classes.tolist()]), (torch.tensor(acs, dtype=torch.float64), np.array(classes.tolist(), dtype=np.float32))):
        got = ops.featurize(*args, counts, order=order, size_classes=totals)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    with pytest.raises(ValueError):
        ops.featurize(*args, [float(v) for v in acs] + [0.0], order=order)
    with pytest.raises(Exception):
        ops.featurize(*args, [float("nan")] * 4, order=order)


def test_errors_of_the_backward_pass_keep_their_type():
    """What an autograd node refuses in the engine's own thread arrives as the exception it is; here coordinates swapped for
    fewer between the passes (past the version counter: the node sees them)."""
    from khan_amd import autograd
    m = _molecules([9, 12])
    b = next(iter(batching.DeviceFeeder(batching.RawDataset(m, [0.0] * 2), 2))).wait()
    acs, order, classes = b.host_counts()
    xyz = [v.detach().clone().requires_grad_(True) for v in (b.xs, b.ys, b.zs)]
    rows = autograd.featurize(*xyz, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs, acs, order=order, size_classes=classes)
    loss = sum(r.sum() for r in rows)
    kept, xyz[1].data = xyz[1].data, xyz[1].data[:5].clone()
    with pytest.raises(ValueError, match="same length"):
        torch.autograd.grad(loss, xyz[0], retain_graph=True)
    xyz[1].data = kept
    assert torch.isfinite(torch.autograd.grad(loss, xyz[0])[0]).all()
