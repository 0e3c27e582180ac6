"""The per-type atomic networks behind the featurizer, their npz checkpoint format, and batched inference.

Mirror of khan/model/nn.py (AtomNN 3-88, MoleculeNN 122-201), of the activation functions in
khan/model/activations.py:63-77, and of the inference half of khan/training/trainer_multi_tower.py:
save_numpy / load_numpy (451-499), predict (655-678), coordinate_gradients (580-615), and the tower wiring
features -> per-type networks -> gather -> segment_sum (+ ani_charge) of lines 306-385.

The featurizer, its gradient and the charge energy are the HIP kernels of this package (through
`khan_amd.autograd`).  On the GPU, networks with CELU run in this package's matrix-core kernels: the reference's default
widths in float32 with constant weights in one launch (`ops.atomic_networks`), inference of other widths and of models with
charges in float32 in a launch each way (csrc/net_chain.hip), everything else layer by layer, forward, gradient, second order
and weight gradients (csrc/net_layers.hip).  Other activations, and the CPU, take PyTorch's
operations.  Parameter
names are the reference's TensorFlow variable names, `<prefix>W_<type>_<in>x<out>_l<k>:0` and
`<prefix>b_...` (nn.py:41-60), so a checkpoint written by the reference's `save_numpy` loads unchanged;
whatever else such a file holds (optimizer slots, learning rate, moving averages) is ignored.
"""
import os

import numpy as np
import torch
from torch.autograd import forward_ad

from . import _native

TYPE_MAP = ("H", "C", "N", "O")
DEFAULT_LAYERS = (128, 128, 64, 1)                       # energy_server.py:121
DEEP_LAYERS = (256, 256, 256, 256, 256, 256, 256, 128, 64, 8, 1)   # energy_server.py:123
FEATURE_SIZE = 384


# ------------------------------------------------------------------ activation functions (activations.py:63-77)
def celu(a, alpha=0.1):
    # a for a >= 0, alpha (exp(a / alpha) - 1) below.  float32: PyTorch's celu, one elementwise kernel forward and
    # one backward.  float64: spelled out, because that kernel's backward rounds alpha to float (1e-8 off).
    if a.dtype == torch.float32:
        return torch.nn.functional.celu(a, alpha)
    return torch.where(a >= 0, a, alpha * torch.expm1(torch.clamp(a, max=0.0) / alpha))


def normal(a, mean=0.0, std=1.0):
    return torch.exp(-((a - mean) / std) ** 2 / 2.0)


def gaussian(a):
    return torch.exp(-a * a)


def softplus(a, shift=0.69314718056):
    return torch.nn.functional.softplus(a) - shift


ACTIVATIONS = {"celu": celu, "normal": normal, "gaussian": gaussian, "softplus": softplus}


def get_fn_by_name(name, *args):
    """activations.get_fn_by_name: the function with its leading extra arguments bound."""
    if name not in ACTIVATIONS:
        raise KeyError("unknown activation function %r (have %s)" % (name, sorted(ACTIVATIONS)))
    fn = ACTIVATIONS[name]
    return (lambda a: fn(a, *args)) if args else fn


def parameter_names(prefix, layer_sizes):
    """[(W name, b name, in, out)] per type and layer, in the reference's order (nn.py:38-60)."""
    out = {}
    for t in TYPE_MAP:
        rows = []
        for idx in range(1, len(layer_sizes)):
            x, y = layer_sizes[idx - 1], layer_sizes[idx]
            name = "_%s_%dx%d_l%d" % (t, x, y, idx)
            rows.append((prefix + "W" + name + ":0", prefix + "b" + name + ":0", x, y))
        out[t] = rows
    return out


def _transformed(tensors):
    """True where the tensors stand for something else than their elements: under a tracer or compiler, torch.func's
    transforms, forward-mode differentiation, a dispatch mode, or as a subclass.  Launches would see none of that;
    library operations do."""
    return (torch._C._get_tracing_state() is not None or torch.compiler.is_compiling()
            or torch._C._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0
            or torch._C._len_torch_dispatch_stack() > 0
            or any(type(t) not in (torch.Tensor, torch.nn.Parameter) for t in tensors))


class MoleculeNN:
    """Four atomic networks (H, C, N, O) mapping feature rows to one number per atom."""

    def __init__(self, layer_sizes=DEFAULT_LAYERS, activation_fn=celu, dtype=torch.float32, device="cpu",
                 prefix="near_", seed=None, first_layer_kernel=True):
        self.first_layer_kernel = bool(first_layer_kernel)
        self.whole_network_kernel = True    # the one-launch network where it applies (`one_launch`); False: layer by layer
        self.weights_need_grad = False      # set it to differentiate through the kernel layers' weights (training)
        layer_sizes = tuple(int(v) for v in layer_sizes)
        if layer_sizes[-1] != 1:
            raise ValueError("the last layer must have size 1")
        self.layer_sizes = (FEATURE_SIZE,) + layer_sizes
        self.activation_fn = activation_fn
        self.dtype, self.device, self.prefix = dtype, torch.device(device), prefix
        self.names = parameter_names(prefix, self.layer_sizes)
        gen = torch.Generator().manual_seed(0 if seed is None else int(seed))
        self.params = {}
        for t in TYPE_MAP:
            for wn, bn, x, y in self.names[t]:
                # random normal with standard deviation sqrt(2 / (in + out)), zero biases (nn.py:49-58)
                w = torch.randn((x, y), generator=gen, dtype=torch.float64) * (2.0 / (x + y)) ** 0.5
                self.params[wn] = w.to(dtype).to(self.device).requires_grad_(True)
                self.params[bn] = torch.zeros((y,), dtype=dtype, device=self.device).requires_grad_(True)

    def parameters(self):
        return [self.params[k] for k in self.params]

    def atom_type_outputs(self, type_idx, feats, layers_done=0):
        """[n_t, 384] feature rows of one type -> [n_t] network outputs (`layers_done`: `feats` are the activations of
        that many leading layers already)."""
        rows = self.names[TYPE_MAP[type_idx]]
        a = feats
        for k, (wn, bn, _, _) in enumerate(rows):
            if k < layers_done:
                continue
            a = torch.addmm(self.params[bn], a, self.params[wn])
            if k != len(rows) - 1:
                a = self.activation_fn(a)
        return a.reshape(-1)

    def layer_transposed(self, k):
        """The four weights of layer k transposed ([out, in], the summed index contiguous), as `ops.dense` takes them."""
        return [self.params[self.names[t][k][0]].detach().t().contiguous() for t in TYPE_MAP]

    def kernel_layers(self):
        """How many leading layers have the widths of the split-operand matrix-core kernels (`ops.dense`,
        `ops.atomic_networks`): float32 on the GPU, CELU with its default alpha, input width a multiple of 32 and output
        width a multiple of 64 -- for the reference's default network 384-128-128-64-1 all but the last."""
        if not (self.first_layer_kernel and self.dtype == torch.float32 and self.device.type == "cuda"
                and self.activation_fn is celu):
            return 0
        n = 0
        for x, y in zip(self.layer_sizes[:-2], self.layer_sizes[1:-1]):      # the last layer has no activation
            if x % 32 or y % 64:
                break
            n += 1
        return n

    def one_launch(self):
        """True if the whole network runs in `ops.atomic_networks` (one launch for the three CELU layers and the output
        layer of the four types, and for the gradient back to the feature rows): the reference's default widths
        384-128-128-64-1 in float32 on the GPU with CELU, the weights taken as constants (inference)."""
        from . import ops
        return (self.whole_network_kernel and self.kernel_layers() == 3 and self.layer_sizes == ops.NETWORK_WIDTHS + (1,)
                and not self.weights_need_grad)

    def one_launch_operands(self):
        """-> (packed weights, biases, head_weights, head_biases) as `ops.atomic_networks` takes them; the weights are
        split into their half-precision parts by one launch on the current stream, as they are when it runs."""
        from . import ops
        rows = [[self.params[self.names[t][k][j]].detach() for t in TYPE_MAP] for j in (0, 1) for k in range(4)]
        return ops.pack_stored_network_weights(rows[:3]), rows[4:7], rows[3], rows[7]

    def atom_outputs(self, atom_type_features, gather_idxs):
        """Per-type flat feature buckets -> one number per atom in the batch's atom order (nn.py:176-177)."""
        # gather_idxs is a permutation: index_select's backward is a scatter-add, where indexing with [] sorts the
        # indices first (a merge sort of n atoms in every backward pass)
        return torch.index_select(torch.cat(self.type_outputs(atom_type_features)), 0, gather_idxs.long())

    def layer_launches(self):
        """True if the layers run in this package's own launches for any widths, precision and order of derivative
        (csrc/net_layers.hip): on the GPU with CELU, two to twelve layers."""
        return (self.first_layer_kernel and self.device.type == "cuda" and self.activation_fn is celu
                and self.dtype in (torch.float32, torch.float64) and 3 <= len(self.layer_sizes) <= 13)

    def _in_flat_order(self):
        """The parameters as the layer launches take them end to end: for every layer the four types' weights, then for every
        layer the four types' biases."""
        if "_flat_names" not in self.__dict__:
            self._flat_names = [self.names[t][k][j] for j in (0, 1) for k in range(len(self.layer_sizes) - 1) for t in TYPE_MAP]
        return [self.params[name] for name in self._flat_names]

    def constants(self, one_launch=True):
        """-> (the parameters in flat order, True if the one-launch kernel takes them (never without `one_launch`), the
        widths): what inference takes.  The passes read the parameters where they lie, and the one-launch kernel's packed
        form is made of them in every pass: nothing is kept that a write to them could leave behind."""
        return self._in_flat_order(), one_launch and self.one_launch(), list(self.layer_sizes)

    def type_outputs(self, atom_type_features):
        """Per-type flat feature buckets -> the four per-type output vectors [acs[t]] (nn.py:165-175)."""
        if not self.layer_launches() or _transformed(atom_type_features):
            return [self.atom_type_outputs(t, f.reshape(-1, FEATURE_SIZE)) for t, f in enumerate(atom_type_features)]
        native, ps, live = _native.load(), self._in_flat_order(), self._live_from()
        if live > 0:
            layers = len(self.layer_sizes) - 1
            ps = [p if k // 4 % layers >= live else p.detach() for k, p in enumerate(ps)]
        return native.network_autograd(native.flatten(ps), list(atom_type_features), self.layer_sizes, 0.1, live)

    def _live_from(self):
        """The first layer whose parameters are differentiated by.  In single precision inference is the default: unless
        `weights_need_grad` the leading `kernel_layers` are constants, and with them an output layer right behind the last
        of them where that has width 64 (it rides in that layer's launch in `ops.dense_head`)."""
        layers = len(self.layer_sizes) - 1
        if not torch.is_grad_enabled():
            return layers
        if self.weights_need_grad:
            return 0
        constant = self.kernel_layers()
        return layers if constant == layers - 1 and self.layer_sizes[-2] == 64 else constant


class AniModel:
    """Near-field network, optional charge network with the pairwise charge energy, and their checkpoint."""

    def __init__(self, layer_sizes=DEFAULT_LAYERS, activation_fn=celu, dtype=torch.float32, device="cuda:0",
                 fit_charges=False, seed=None, first_layer_kernel=True):
        self.dtype, self.device = dtype, torch.device(device)
        self.near = MoleculeNN(layer_sizes, activation_fn, dtype, device, "near_", seed, first_layer_kernel)
        self.charge = None
        if fit_charges:
            self.charge = MoleculeNN(layer_sizes, activation_fn, dtype, device, "charge_",
                                     None if seed is None else seed + 1, first_layer_kernel)

    # -------------------------------------------------------------------------------------- checkpoint
    def named_parameters(self):
        out = dict(self.near.params)
        if self.charge is not None:
            out.update(self.charge.params)
        return out

    def save_numpy(self, npz_file):
        """trainer_multi_tower.py:451-470: one array per variable, keyed by the variable's name."""
        if os.path.splitext(npz_file)[1] != ".npz":
            raise ValueError("the checkpoint file name must end in .npz")
        np.savez(npz_file, **{k: v.detach().cpu().numpy() for k, v in self.named_parameters().items()})

    def load_numpy(self, npz_file, strict=False):
        """trainer_multi_tower.py:472-499.  `strict` refuses a checkpoint of another precision; arrays the model
        has no parameter for are ignored; a parameter missing from the file is an error."""
        objs = np.load(npz_file, allow_pickle=False)
        mine = self.named_parameters()
        missing = [k for k in mine if k not in objs.files]
        if missing:
            raise KeyError("checkpoint %s lacks %d parameters, e.g. %s" % (npz_file, len(missing), missing[0]))
        np_dtype = np.float32 if self.dtype == torch.float32 else np.float64
        for k, p in mine.items():
            arr = objs[k]
            if arr.dtype != np_dtype and strict:
                raise TypeError("Cannot deserialize %s into %s. You may want to set strict=False."
                                % (arr.dtype, np.dtype(np_dtype)))
            if tuple(arr.shape) != tuple(p.shape):
                raise ValueError("%s has shape %s in the checkpoint, %s in the model" % (k, arr.shape, tuple(p.shape)))
            with torch.no_grad():
                p.copy_(torch.from_numpy(np.ascontiguousarray(arr.astype(np_dtype))).to(self.device))

    # --------------------------------------------------------------------------------------- inference
    def batch_energies(self, b, need_grad=False):
        """DeviceBatch -> per-molecule energies [n_mols] (and d energy / d xyz when need_grad)."""
        energies, *parts = self._energies(b, need_grad)
        return energies, torch.stack(parts, dim=1) if need_grad else None

    def _energies(self, b, need_grad, joined=False, waited=False):
        """DeviceBatch -> [energies [n_mols]] and, with need_grad, the energy's gradient by x, y and z; with `joined` also the
        one array all of them are parts of: the energies, padded to 64 elements, then the gradient's three parts.  `waited`:
        the caller has had the current stream wait for the batch."""
        if not self.near.layer_launches():
            energies, *parts = self._energies_through_autograd(b, need_grad)
            if joined:
                parts.append(torch.cat([energies, energies.new_empty(-b.n_mols % 64)] + parts))
            return [energies] + parts
        acs, order, classes = b._counts(waited)
        # Networks beside a charge network have products of all 24 bits over float32's range (net_chain.hip, or layer by
        # layer), where the one-launch kernel's operands are off by up to 2^-23 of their size between 6e-5 and 65,504.
        alone = self.charge is None
        return _native.load().infer(
            b.xs, b.ys, b.zs, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs, b.gather_idxs, acs, order, classes,
            self.near.constants(alone), None if alone else self.charge.constants(False), 0.1, need_grad, joined)

    def _energies_through_autograd(self, b, need_grad):
        """_energies for networks of library operations (other activations than CELU)."""
        from . import autograd
        xs, ys, zs = b.xs, b.ys, b.zs
        acs, order, classes = b._counts()
        if need_grad:
            xs, ys, zs = (t.detach().clone().requires_grad_(True) for t in (xs, ys, zs))
        feats = autograd.featurize(xs, ys, zs, b.atom_types, b.mol_offsets, b.mol_atom_counts, b.scatter_idxs, acs,
                                   order=order, size_classes=classes)
        # the networks' outputs summed by molecule straight from the four per-type vectors (nn.py:165-177 in one launch)
        energies = autograd.mol_energy(self.near.type_outputs(feats), b.atom_types, b.scatter_idxs, b.mol_offsets,
                                       b.mol_atom_counts)
        if self.charge is not None:
            qs = self.charge.atom_outputs(feats, b.gather_idxs)
            energies = energies + autograd.ani_charge(xs, ys, zs, qs.contiguous(), b.mol_offsets, b.mol_atom_counts)
        if not need_grad:
            return [energies.detach()]
        return [energies.detach(), *torch.autograd.grad(energies, (xs, ys, zs), grad_outputs=torch.ones_like(energies))]

    def _feeder(self, dataset, batch_size):
        from .batching import DeviceFeeder
        np_dtype = np.float32 if self.dtype == torch.float32 else np.float64
        return DeviceFeeder(dataset, batch_size, shuffle=False, dtype=np_dtype, device=self.device)

    def _results(self, dataset, batch_size, of_batch):
        """For every batch of the data set (of_batch(batch) on the host, the batch), copied out asynchronously: the GPU
        works on the next batch while the caller handles this one.  The array is good until the next one is asked for."""
        ahead = None
        for b in self._feeder(dataset, batch_size):
            stream = torch.cuda.current_stream(self.device)
            b.wait(stream)
            out = of_batch(b)
            host = torch.empty(out.shape, dtype=out.dtype, pin_memory=True)
            host.copy_(out, non_blocking=True)
            done = torch.cuda.Event()
            done.record(stream)
            if ahead is not None:
                ahead[1].synchronize()
                yield ahead[0].numpy(), ahead[2]
            ahead = host, done, b
        if ahead is not None:
            ahead[1].synchronize()
            yield ahead[0].numpy(), ahead[2]

    def predict(self, dataset, batch_size=2048):
        """-> [y0, y1, ...] in the order of the dataset's molecules (trainer_multi_tower.py:655-678)."""
        ys = []
        for e, _ in self._results(dataset, batch_size, lambda b: self._energies(b, False, waited=True)[0]):
            ys.extend(e.tolist())
        return ys

    def coordinate_gradients(self, dataset, batch_size=1024):
        """Yields one [n_atoms, 3] array of d energy / d (x, y, z) per molecule (trainer_multi_tower.py:580-615)."""
        of_batch = lambda b: self._energies(b, True, joined=True, waited=True)[-1][-3 * b.xs.numel():] if b.xs.numel() else b.xs
        for g, b in self._results(dataset, batch_size, of_batch):
            yield from _native.load().molecule_rows(g.reshape(3, -1), b.host_sizes())

    def energies_and_gradients(self, dataset, batch_size=1024):
        """Yields (energy, [n_atoms, 3] gradient) per molecule from one pass over the data set."""
        for v, b in self._results(dataset, batch_size, lambda b: self._energies(b, True, joined=True, waited=True)[-1]):
            gradient = v[v.size - 3 * b.xs.numel():].reshape(3, -1)
            yield from zip(v[:b.n_mols].tolist(), _native.load().molecule_rows(gradient, b.host_sizes()))
