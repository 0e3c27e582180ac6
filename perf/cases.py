"""What this package's users have it do, as cases that can be timed and compared.

A case names one of seven jobs and its size; each runs through the package's public entry points on synthetic
molecules (`khan_amd.datagen`), which a seed puts in an order of its own and moves out of their equilibrium:

    request  one molecule's energy and gradient from the energy server (JSON text in, JSON text out)
    dataset  energies and coordinate gradients of a data set in host memory
    step     one batch of the featurizer: offsets, type sort, feature rows, gradient of given upstream rows;
             with `charges` also the charge energy and its gradients
    infer    energies and coordinate gradients of one batch that is on the GPU
    train    one step of plain gradient descent on the squared error of the energies
    forces   the same with the squared error of the forces added (a second derivative)
    charges  charge energies with their gradients alone
"""
import functools
import json
import math

import numpy as np
import torch

from khan_amd import autograd, datagen, model, ops, server
from khan_amd.batching import DeviceBatch, PackedDataset, RawDataset

DEVICE = "cuda:0"
DTYPES = {"f32": (torch.float32, np.float32), "f64": (torch.float64, np.float64)}
LAYERS = {"default": model.DEFAULT_LAYERS, "deep": model.DEEP_LAYERS}
# A training step moves the weights by so little that any number of passes sees the same network
LEARNING_RATE = 1e-7


def listed():
    return [
        # the energy server as it ships: float64, one molecule of about a dozen atoms per request
        {"name": "request_organic_f64", "job": "request", "kind": "organic", "dtype": "f64", "layers": "default", "charge": False},
        # predict + coordinate_gradients of a data set of organic molecules at their default batch sizes
        {"name": "dataset_organic4096_f32", "job": "dataset", "kind": "organic", "mols": 4096, "dtype": "f32", "packed": False},
        # featurizer batches: the reference trainer's batch size, the configuration the headline figure is quoted on, ...
        {"name": "step_organic1024_f32", "job": "step", "kind": "organic", "mols": 1024, "dtype": "f32", "charges": False},
        {"name": "step_organic65536_f32", "job": "step", "kind": "organic", "mols": 65536, "dtype": "f32", "charges": False},
        # ... dense boxes of 64-256 atoms, systems of 1,024-4,096 atoms, and double precision with the charge energy
        {"name": "step_boxes4096_f32", "job": "step", "kind": "boxes", "mols": 4096, "dtype": "f32", "charges": False},
        {"name": "step_bigboxes64_f32", "job": "step", "kind": "bigboxes", "mols": 64, "dtype": "f32", "charges": False},
        {"name": "step_organic16384_f64", "job": "step", "kind": "organic", "mols": 16384, "dtype": "f64", "charges": True},
        # batched inference on the GPU: the default networks on a large batch, the deep ones with a charge network on a ragged one
        {"name": "infer_organic65536_f32", "job": "infer", "kind": "organic", "mols": 65536, "dtype": "f32", "layers": "default",
         "charge": False, "gradients": True},
        {"name": "infer_deep_organic4001_f32", "job": "infer", "kind": "organic", "mols": 4001, "dtype": "f32", "layers": "deep",
         "charge": True, "gradients": True},
        # training: the reference's batch size on energies, a larger odd one on energies and forces
        {"name": "train_organic1024_f32", "job": "train", "kind": "organic", "mols": 1024, "dtype": "f32"},
        {"name": "forces_organic3001_f32", "job": "forces", "kind": "organic", "mols": 3001, "dtype": "f32"},
        # charge energies and their gradients of dense boxes in double precision
        {"name": "charges_boxes4096_f64", "job": "charges", "kind": "boxes", "mols": 4096, "dtype": "f64"},
    ]


# The largest batch of each kind of molecule that the package's own benchmark runs, by precision
MOST_MOLS = {("organic", "f32"): 65536, ("organic", "f64"): 16384, ("boxes", "f32"): 4096, ("boxes", "f64"): 1024,
             ("bigboxes", "f32"): 64, ("bigboxes", "f64"): 16}


def draw(rng):
    def size(least, most):
        return int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))

    job = rng.choice(("request", "dataset", "step", "step", "infer", "infer", "train", "forces", "charges"))
    case = {"job": job, "kind": rng.choice(("organic", "organic", "boxes")), "dtype": "f32"}
    if job == "request":
        # `first`: which molecule of the generator's sequence, so that requests differ in size
        case.update(dtype="f64", layers=rng.choice(("default", "default", "deep")), charge=rng.random() < 0.25, first=rng.randrange(1 << 20))
    elif job == "dataset":
        case.update(mols=size(64, 8192 if case["kind"] == "organic" else 512), packed=rng.random() < 0.5)
    elif job == "step":
        case["kind"] = rng.choice(("organic", "organic", "boxes", "bigboxes"))
        case["dtype"] = rng.choice(("f32", "f32", "f64"))
        case.update(mols=size(1, MOST_MOLS[case["kind"], case["dtype"]]), charges=rng.random() < 0.5)
    elif job == "infer":
        layers = rng.choice(("default", "default", "deep"))
        most = MOST_MOLS[case["kind"], "f32"]
        case.update(layers=layers, charge=rng.random() < 0.25, gradients=rng.random() < 0.75, mols=size(1, most // 16 if layers == "deep" else most))
    elif job in ("train", "forces"):
        case.update(mols=size(128, 4096 if case["kind"] == "organic" else 256))
    else:
        case["dtype"] = rng.choice(("f32", "f64"))
        case.update(mols=size(1, 16384 if case["kind"] == "organic" else 4096))
    return case


@functools.lru_cache(maxsize=1)
def _base(kind, mols, first):
    return datagen.make_batch(kind, mols, first_mol=first)


def _batch_of(case, seed):
    """-> (types [n] int32, coordinates [n, 3] float64, molecule sizes): the case's molecules in an order that the seed
    gives, every atom displaced by 0.03 Angstrom per component, about what it vibrates by."""
    base = _base(case["kind"], case.get("mols", 1), case.get("first", 0))
    rng = np.random.default_rng(seed)
    order = rng.permutation(base.n_mols)
    sizes = base.MACs[order]
    at = np.repeat(base.MOs[order] - (np.cumsum(sizes) - sizes), sizes) + np.arange(base.n_atoms)
    xyz = np.stack([base.X[at], base.Y[at], base.Z[at]], axis=1) + rng.normal(0.0, 0.03, (base.n_atoms, 3))
    return base.A[at], xyz, sizes


def _molecules(types, xyz, sizes):
    """As the reference's data sets hold them: one float64 array of (type, x, y, z) rows per molecule."""
    return np.split(np.concatenate([types[:, None], xyz], axis=1), np.cumsum(sizes)[:-1])


def prepare(case, seed):
    job = case["job"]
    tdt, ndt = DTYPES[case["dtype"]]
    mols = 1 if job == "request" else case["mols"]
    types, xyz, sizes = _batch_of(case, seed)
    n = types.size
    s = {"case": case, "n_mols": mols}
    if job in ("request", "dataset", "infer", "train", "forces"):
        s["model"] = model.AniModel(LAYERS[case.get("layers", "default")], model.celu, tdt, DEVICE,
                                    fit_charges=case.get("charge", False), seed=seed)
    if job == "request":
        s["text"] = json.dumps({"X": _molecules(types, xyz, sizes)[0].tolist()})
        return s
    if job == "dataset":
        s["data"] = RawDataset(_molecules(types, xyz, sizes), np.zeros(mols))
        if case["packed"]:
            s["data"] = PackedDataset.from_raw(s["data"], ndt)
        return s
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    s["xs"], s["ys"], s["zs"] = torch.from_numpy(xyz).to(DEVICE).t().to(tdt).contiguous()
    s["types"], s["mol_idxs"] = (torch.from_numpy(v).to(DEVICE) for v in (types, np.repeat(np.arange(mols, dtype=np.int32), sizes)))
    if job == "step":
        s["upstream"] = torch.randn(n * ops.FEATURE_SIZE, dtype=tdt, device=DEVICE, generator=gen)
    if job == "charges" or case.get("charges"):
        # partial charges of a third of an electron, and the derivative of some loss by each molecule's energy
        s["qs"] = 0.3 * torch.randn(n, dtype=tdt, device=DEVICE, generator=gen)
        s["energy_grads"] = torch.randn(mols, dtype=tdt, device=DEVICE, generator=gen)
    if job == "charges":
        s["macs"], s["mos"] = ops.mol_offsets(s["mol_idxs"], mols)
    if job in ("train", "forces"):
        s["model"].near.weights_need_grad = True
        s["labels"] = torch.randn(mols, dtype=tdt, device=DEVICE, generator=gen)
        s["labelled_forces"] = torch.randn(3, n, dtype=tdt, device=DEVICE, generator=gen)
    return s


def run(s):
    return _RUN[s["case"]["job"]](s)


def _run_request(s):
    answer = json.loads(server.handle_request(s["model"], s["text"]))
    return {"energy": answer["energy"], "gradient": np.array(answer["gradient"])}


def _run_dataset(s):
    energies = s["model"].predict(s["data"])
    gradients = list(s["model"].coordinate_gradients(s["data"]))
    return {"energies": np.array(energies), "gradients": np.concatenate(gradients)}


def _batch(s):
    return DeviceBatch.from_device_arrays(s["xs"], s["ys"], s["zs"], s["types"], s["mol_idxs"], s["n_mols"])


def _run_step(s):
    b = _batch(s)
    acs, order, classes = b.host_counts()
    args = (b.xs, b.ys, b.zs, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs, acs)
    rows = ops.featurize(*args, order=order, size_classes=classes)
    upstream = torch.split(s["upstream"], [c * ops.FEATURE_SIZE for c in acs])
    grads = ops.featurize_grad(*args, *upstream, order=order, size_classes=classes)
    out = {"rows": rows, "grads": grads, "sort": (b.mol_atom_counts, b.mol_offsets, b.scatter_idxs, b.gather_idxs, b.atom_counts)}
    if s["case"]["charges"]:
        out["charges"] = ops.ani_charge_all(b.xs, b.ys, b.zs, s["qs"], b.mol_offsets, b.mol_atom_counts, s["energy_grads"])
    return out


def _run_infer(s):
    return s["model"].batch_energies(_batch(s), need_grad=s["case"]["gradients"])


def _energies(s, b, xyz):
    acs, order, classes = b.host_counts()
    rows = autograd.featurize(*xyz, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs, acs, order=order, size_classes=classes)
    return autograd.mol_energy(s["model"].near.type_outputs(rows), b.atom_types, b.scatter_idxs, b.mol_offsets, b.mol_atom_counts)


def _descend(s, loss):
    params = s["model"].near.parameters()
    grads = torch.autograd.grad(loss, params)
    with torch.no_grad():
        torch._foreach_add_(params, grads, alpha=-LEARNING_RATE)
    return grads


def _run_train(s):
    b = _batch(s)
    energies = _energies(s, b, (b.xs, b.ys, b.zs))
    loss = ((energies - s["labels"]) ** 2).mean()
    return {"energies": energies.detach(), "grads": _descend(s, loss)}


def _run_forces(s):
    b = _batch(s)
    xyz = [v.detach().requires_grad_(True) for v in (b.xs, b.ys, b.zs)]
    energies = _energies(s, b, xyz)
    forces = torch.stack(torch.autograd.grad(energies.sum(), xyz, create_graph=True))
    loss = ((energies - s["labels"]) ** 2).mean() + ((forces - s["labelled_forces"]) ** 2).mean()
    return {"energies": energies.detach(), "forces": forces.detach(), "grads": _descend(s, loss)}


def _run_charges(s):
    return ops.ani_charge_all(s["xs"], s["ys"], s["zs"], s["qs"], s["mos"], s["macs"], s["energy_grads"])


_RUN = {"request": _run_request, "dataset": _run_dataset, "step": _run_step, "infer": _run_infer, "train": _run_train,
        "forces": _run_forces, "charges": _run_charges}


def work(case):
    """Bytes: every input read once, every output written once.  Operations: the pair and triple terms of the batch
    (a sample's counts, scaled up) and the multiply-adds of the networks."""
    mols, w = case.get("mols", 1), 4 if case["dtype"] == "f32" else 8
    sample = datagen.make_batch(case["kind"], min(mols, 4 if case["kind"] == "bigboxes" else 64), first_mol=case.get("first", 0))
    per_mol = {k: v / sample.n_mols for k, v in dict(sample.work_counts(), N=sample.n_atoms).items()}
    N, D, PR, PA, T, C = (per_mol[k] * mols for k in ("N", "D", "P_R", "P_A", "T", "C"))
    rows_flops = 9 * D + 100 * PR + 5 * PA + 150 * T
    grad_flops = 9 * D + 220 * PR + 8 * PA + 390 * T
    widths = (ops.FEATURE_SIZE,) + tuple(LAYERS[case.get("layers", "default")])
    weights = sum(x * y for x, y in zip(widths, widths[1:]))          # of one atom type
    networks = 2 if case.get("charge") else 1
    atoms_in = N * (3 * w + 8)
    job = case["job"]
    if job == "charges":
        return {"bytes": N * 8 * w + mols * (2 * w + 8), "flops": 45 * C}
    if job == "step":
        nbytes = atoms_in + N * (2 * ops.FEATURE_SIZE * w + 3 * w + 8) + 8 * mols
        charges = case["charges"]
        return {"bytes": nbytes + (N * 5 * w + mols * 2 * w if charges else 0), "flops": rows_flops + grad_flops + (45 * C if charges else 0)}
    with_grad = job != "infer" or case["gradients"]
    # products with the weights: forward 1, data gradient 1, weight gradient 1, and twice as many for a loss on forces
    products = {"train": 3, "forces": 6}.get(job, 2 if with_grad else 1)
    flops = rows_flops * (2 if job == "forces" else 1) + (0 if job == "train" or not with_grad else grad_flops)
    flops += 2 * weights * N * products * networks + (45 * C if case.get("charge") else 0)
    nbytes = atoms_in + mols * w + (N * 3 * w if with_grad and job != "train" else 0) + 4 * weights * w * networks
    if job in ("train", "forces"):
        nbytes += 2 * 4 * weights * w + mols * w + (N * 3 * w if job == "forces" else 0)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Float32: sums of up to a few hundred rounded terms, and through the networks and their gradients a few such sums
    in a row (5e-7 to 2e-6 from float64 results at these sizes, single values ten times that).  Float64 the same, with
    the server's text keeping every digit.  Indices and counts are exact."""
    return {"rel": 1e-5, "max": 2e-4} if case["dtype"] == "f32" else {"rel": 1e-11}
