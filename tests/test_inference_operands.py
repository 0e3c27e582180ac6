"""Inference takes the parameters as they are when it runs: written to past the version counter, replaced by other tensors, or held
in another order of memory."""
import numpy as np
import pytest
import torch

from khan_amd import datagen, model
from khan_amd.batching import DeviceBatch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _batch(n_mols, dtype, kind="organic", first=0):
    b = datagen.make_batch(kind, n_mols, first_mol=first)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    return DeviceBatch.from_device_arrays(*(d(v).to(dtype) for v in (b.X, b.Y, b.Z)), d(b.A), d(b.mol_idxs), b.n_mols)


def _like(m, layers, dtype, charges):
    """A model of its own with the parameters that m has now."""
    other = model.AniModel(layers, model.celu, dtype, DEV, fit_charges=charges, seed=99)
    with torch.no_grad():
        for k, p in other.named_parameters().items():
            p.copy_(m.named_parameters()[k])
    return other


# every way a network runs in inference: one launch, layer by layer in both precisions, with a charge network
@pytest.mark.parametrize("layers,dtype,charges,only", [
    (model.DEFAULT_LAYERS, torch.float32, False, ""), (model.DEFAULT_LAYERS, torch.float64, False, ""),
    ((100, 1), torch.float32, False, ""), (model.DEFAULT_LAYERS, torch.float64, True, "")])
def test_parameters_written_past_the_version_counter(layers, dtype, charges, only):
    m = model.AniModel(layers, model.celu, dtype, DEV, fit_charges=charges, seed=1)
    b = _batch(50, dtype)
    before, _ = m.batch_energies(b, need_grad=True)
    for k, p in m.named_parameters().items():
        if only in k:
            version = p._version
            p.data.add_(0.01)
            assert p._version == version
    got, got_g = m.batch_energies(b, need_grad=True)
    want, want_g = _like(m, layers, dtype, charges).batch_energies(b, need_grad=True)
    assert torch.equal(got, want) and torch.equal(got_g, want_g) and not torch.equal(got, before)


@pytest.mark.parametrize("layers,dtype", [(model.DEFAULT_LAYERS, torch.float64), ((100, 1), torch.float32), (model.DEFAULT_LAYERS, torch.float32)])
def test_parameters_replaced_and_strided(layers, dtype):
    """New tensors in `params`, weights in column order and biases with a stride; a parameter of another type is refused."""
    m = model.AniModel(layers, model.celu, dtype, DEV, seed=1)
    b = _batch(50, dtype)
    m.batch_energies(b)
    for k, p in list(m.near.params.items()):
        v = p.detach() + 0.01
        m.near.params[k] = (v.t().contiguous().t() if v.dim() == 2 else torch.stack([v, v], dim=1)[:, 0]).requires_grad_(True)
    got, got_g = m.batch_energies(b, need_grad=True)
    want, want_g = _like(m, layers, dtype, False).batch_energies(b, need_grad=True)
    assert torch.equal(got, want) and torch.equal(got_g, want_g)
    k = m.near.names["C"][0][0]
    m.near.params[k] = m.near.params[k].detach().to(torch.float32 if dtype == torch.float64 else torch.float64)
    with pytest.raises((TypeError, ValueError)):
        m.batch_energies(b)


def test_weights_packed_from_the_stored_matrices():
    """The same bytes as from the transposed copies, and a stream's own: nothing is kept between calls that another stream would
    have to wait for."""
    from khan_amd import ops
    net = model.AniModel(seed=4).near
    stored = [[net.params[net.names[t][k][0]].detach() for t in model.TYPE_MAP] for k in range(3)]
    want = ops.pack_network_weights([net.layer_transposed(k) for k in range(3)], stored)
    assert torch.equal(ops.pack_stored_network_weights(stored), want)
    assert torch.equal(ops.pack_stored_network_weights([[w.t().contiguous().t() for w in layer] for layer in stored]), want)
    torch.cuda.synchronize()
    first = net.one_launch_operands()[0]
    with torch.cuda.stream(torch.cuda.Stream()):
        second = net.one_launch_operands()[0]
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want) and first.data_ptr() != second.data_ptr()


@pytest.mark.parametrize("exponent", [0, 24, -30])
def test_float32_networks_beside_a_charge_network(exponent):
    """Default networks in float32 with a charge network: products of all 24 bits over float32's range.  Layer 1 (kept clear
    of CELU's knee by its biases) scaled by 2^exponent and layer 2 by the inverse leave the result what it is, and carry
    activations and weights past half precision's range (65,504; 6e-5).  Bound: the roundings of four layers' sums and the
    way back, 2e-6 of sum |x| |w| each as for one layer, whose terms are some times the largest result here."""
    models = [model.AniModel(model.DEFAULT_LAYERS, model.celu, dt, DEV, fit_charges=True, seed=6) for dt in (torch.float32, torch.float64)]
    single, double = (m.named_parameters() for m in models)
    with torch.no_grad():
        for k, p in single.items():
            if "_l1:" in k:
                if "b_" in k:
                    p.fill_(8.0)
                p.mul_(2.0 ** exponent)
            if "_l2:" in k and "W_" in k:
                p.mul_(2.0 ** -exponent)
            double[k].copy_(p)
    got, want = (m.batch_energies(_batch(400, dt), need_grad=True) for m, dt in zip(models, (torch.float32, torch.float64)))
    for g, w in zip(got, want):
        assert torch.isfinite(g).all()
        assert float((g.double() - w).abs().max()) <= 2e-5 * float(w.abs().max())


@pytest.mark.parametrize("layers,dtype", [(model.DEFAULT_LAYERS, torch.float32), (model.DEFAULT_LAYERS, torch.float64), ((100, 1), torch.float32)])
def test_captured_inference_reads_the_parameters_when_it_is_replayed(layers, dtype):
    """batch_energies of a batch made on another stream, recorded into a graph: every replay, with eager work and parameter
    writes in between, gives what an eager pass gives then."""
    m = model.AniModel(layers, model.celu, dtype, DEV, seed=1)
    b = _batch(300, dtype)
    m.batch_energies(b, need_grad=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m.batch_energies(b, need_grad=True)
    for k in range(3):
        for o in out:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        want = m.batch_energies(b, need_grad=True)
        assert all(torch.equal(a, w) for a, w in zip(out, want)), k
        for p in m.near.parameters():
            p.data.add_(0.01)
        torch.cuda.synchronize()
