"""Host batch assembly and device feeding for the featurizer.

`RawDataset` mirrors khan/data/dataset.py:7-183: molecules are ragged arrays of rows (type, x, y, z), a
batch is their concatenation plus, per atom, the index of its molecule inside the batch; the last
batch is not padded (dataset.py:118-183).

`PackedDataset` holds the same data packed once into flat arrays and assembles a batch with a native,
multi-threaded gather (csrc/host_batch.c) instead of one numpy operation per molecule.

`DeviceFeeder` is what the reference does with a feed dict and a staging queue
(khan/training/trainer_multi_tower.py:767-792, 291-303), done for one GPU with PyTorch as the memory
and stream plumbing: it splits a batch into the flat arrays the ops take (xs, ys, zs, atom types,
molecule indices) in one pinned host buffer (csrc/torch_feed.cpp), copies it asynchronously on a side stream,
runs the batch's preparation (`mol_offsets`, `ani_sort`, `size_order`) on the device, and keeps one batch in flight while the
caller works on the previous one.
"""
import ctypes
import math
import os

import numpy as np

from . import _native

_HERE = os.path.dirname(os.path.abspath(__file__))
HOST_LIB_PATH = os.path.join(_HERE, "csrc", "libkhan_host.so")
_host_lib = None


def _host():
    """The native batch assembler (csrc/host_batch.c); no GPU code in it."""
    global _host_lib
    if _host_lib is None:
        if not os.path.exists(HOST_LIB_PATH):
            raise RuntimeError("%s is missing: run `python -m khan_amd.build`" % HOST_LIB_PATH)
        lib = ctypes.CDLL(HOST_LIB_PATH)
        vp, i64 = ctypes.c_void_p, ctypes.c_int64
        lib.khan_host_batch_offsets.restype = i64
        lib.khan_host_batch_offsets.argtypes = [vp, i64, vp, i64, vp]
        for name in ("khan_host_gather_f32", "khan_host_gather_f64"):
            fn = getattr(lib, name)
            fn.restype = None
            fn.argtypes = [vp, vp, vp, vp, vp, vp, i64, vp, vp, vp, vp, vp, vp, ctypes.c_int]
        lib.khan_host_gather_rows3_f64.restype = None
        lib.khan_host_gather_rows3_f64.argtypes = [vp, vp, vp, i64, vp, vp, ctypes.c_int]
        _host_lib = lib
    return _host_lib


def _np_ptr(a):
    return ctypes.c_void_p(a.ctypes.data)


def _selections(dataset, batch_size, shuffle, rng):
    perm = np.arange(dataset.num_mols(), dtype=np.int64)
    if shuffle:
        (np.random.default_rng() if rng is None else rng).shuffle(perm)
    for batch_idx in range(dataset.num_batches(batch_size)):
        yield perm[batch_idx * batch_size:min((batch_idx + 1) * batch_size, dataset.num_mols())]


class RawDataset:
    """Ragged molecules [(n_i, 4) arrays of (type, x, y, z)], optional labels and per-atom gradients."""

    def __init__(self, all_Xs, all_ys=None, all_grads=None):
        self.all_Xs = list(all_Xs)
        self.all_ys = None if all_ys is None else list(all_ys)
        self.all_grads = None if all_grads is None else list(all_grads)
        if self.all_ys is not None and len(self.all_ys) != len(self.all_Xs):
            raise ValueError("all_ys must have one entry per molecule")
        if self.all_grads is not None and len(self.all_grads) != len(self.all_Xs):
            raise ValueError("all_grads must have one entry per molecule")

    def num_mols(self):
        return len(self.all_Xs)

    def num_batches(self, batch_size):
        return math.ceil(self.num_mols() / batch_size)

    def iterate(self, batch_size, shuffle, fuzz=None, rng=None):
        """Yields (mol_Xs [N,4], mol_ids [N], mol_yts or None, mol_grads [N,3] or None) per batch.

        mol_ids[a] is the position of atom a's molecule inside the batch.  `fuzz` adds uniform noise in
        [-fuzz, fuzz] to the coordinates (dataset.py:166-169).  `rng` is a numpy Generator (the reference
        draws from numpy's global state)."""
        rng = np.random.default_rng() if rng is None else rng
        for sel in self.selections(batch_size, shuffle, rng):
            yield self.batch(sel, fuzz, rng)

    def selections(self, batch_size, shuffle, rng=None):
        """The molecule indices of every batch, in order (the last batch is not padded)."""
        return _selections(self, batch_size, shuffle, rng)

    def batch(self, sel, fuzz=None, rng=None):
        """The tuple of `iterate` for the molecules `sel`."""
        mols = [np.asarray(self.all_Xs[p]) for p in sel]
        mol_ids = np.repeat(np.arange(len(sel), dtype=np.int32), [len(m) for m in mols])
        mol_Xs = np.concatenate(mols, axis=0) if mols else np.zeros((0, 4))
        if fuzz is not None:
            mol_Xs = mol_Xs.copy()
            mol_Xs[:, 1:4] += rng.uniform(-fuzz, fuzz, (mol_Xs.shape[0], 3))
        mol_yts = None if self.all_ys is None else [self.all_ys[p] for p in sel]
        mol_grads = None
        if self.all_grads is not None:
            mol_grads = np.concatenate([np.asarray(self.all_grads[p]) for p in sel], axis=0)
        return mol_Xs, mol_ids, mol_yts, mol_grads


class PackedDataset:
    """The same data set packed once into flat arrays: every atom's type and coordinates end to end plus the
    molecule offsets.  A batch is then gathered by a native routine (parallel over molecules) straight into the
    flat arrays the ops take, instead of one numpy operation per molecule; `iterate` still yields the
    reference's tuples.  Coordinates are kept in `dtype`, the precision the featurizer will run in."""

    def __init__(self, all_Xs, all_ys=None, all_grads=None, dtype=np.float32, n_threads=None):
        counts = np.array([len(m) for m in all_Xs], dtype=np.int64)
        self.offsets = np.zeros(len(counts) + 1, dtype=np.int64)
        np.cumsum(counts, out=self.offsets[1:])
        flat = np.concatenate([np.asarray(m, dtype=np.float64).reshape(-1, 4) for m in all_Xs], axis=0) \
            if len(counts) else np.zeros((0, 4))
        self.dtype = np.dtype(dtype)
        self.types = np.ascontiguousarray(flat[:, 0]).astype(np.int32)
        self.x, self.y, self.z = (np.ascontiguousarray(flat[:, k], dtype=self.dtype) for k in (1, 2, 3))
        self.ys = None if all_ys is None else np.asarray(all_ys)
        if self.ys is not None and len(self.ys) != len(counts):
            raise ValueError("all_ys must have one entry per molecule")
        self.grads = None
        if all_grads is not None:
            if len(all_grads) != len(counts):
                raise ValueError("all_grads must have one entry per molecule")
            self.grads = np.ascontiguousarray(np.concatenate([np.asarray(g, dtype=np.float64).reshape(-1, 3)
                                                              for g in all_grads], axis=0)) if len(counts) else np.zeros((0, 3))
        self.n_threads = int(n_threads) if n_threads else min(16, os.cpu_count() or 1)

    @classmethod
    def from_raw(cls, raw, dtype=np.float32, n_threads=None):
        return cls(raw.all_Xs, raw.all_ys, raw.all_grads, dtype, n_threads)

    def num_mols(self):
        return self.offsets.size - 1

    def num_batches(self, batch_size):
        return math.ceil(self.num_mols() / batch_size)

    def batch_atoms(self, sel):
        """-> (per-molecule offsets inside the batch [len(sel) + 1], number of atoms) for molecules `sel`."""
        sel = np.ascontiguousarray(sel, dtype=np.int64)
        out_off = np.empty(sel.size + 1, dtype=np.int64)
        n = _host().khan_host_batch_offsets(_np_ptr(self.offsets), self.num_mols(), _np_ptr(sel), sel.size, _np_ptr(out_off))
        if n < 0:
            raise IndexError("molecule index out of range")
        return sel, out_off, int(n)

    def gather_into(self, sel, out_off, xs, ys, zs, types, mol_ids):
        """Fills the first out_off[-1] elements of the given flat arrays (numpy views, e.g. of pinned tensors)."""
        for a, dt in ((xs, self.dtype), (ys, self.dtype), (zs, self.dtype), (types, np.int32), (mol_ids, np.int32)):
            if a.dtype != dt or not a.flags["C_CONTIGUOUS"] or a.size < out_off[-1]:
                raise ValueError("destination arrays must be contiguous, of the data set's types, and large enough")
        fn = _host().khan_host_gather_f32 if self.dtype == np.float32 else _host().khan_host_gather_f64
        fn(_np_ptr(self.offsets), _np_ptr(self.types), _np_ptr(self.x), _np_ptr(self.y), _np_ptr(self.z), _np_ptr(sel),
           sel.size, _np_ptr(out_off), _np_ptr(xs), _np_ptr(ys), _np_ptr(zs), _np_ptr(types), _np_ptr(mol_ids), self.n_threads)

    def gather(self, sel):
        """-> (xs, ys, zs, atom types, molecule index per atom) of the batch made of molecules `sel`."""
        sel, out_off, n = self.batch_atoms(sel)
        xs, ys, zs = (np.empty(n, dtype=self.dtype) for _ in range(3))
        types, mol_ids = np.empty(n, dtype=np.int32), np.empty(n, dtype=np.int32)
        self.gather_into(sel, out_off, xs, ys, zs, types, mol_ids)
        return xs, ys, zs, types, mol_ids

    def gather_grads(self, sel, out_off):
        out = np.empty((int(out_off[-1]), 3), dtype=np.float64)
        _host().khan_host_gather_rows3_f64(_np_ptr(self.offsets), _np_ptr(self.grads), _np_ptr(sel), sel.size,
                                           _np_ptr(out_off), _np_ptr(out), self.n_threads)
        return out

    def selections(self, batch_size, shuffle, rng=None):
        """The molecule indices of every batch, in order (the last batch is not padded)."""
        return _selections(self, batch_size, shuffle, rng)

    def iterate(self, batch_size, shuffle, fuzz=None, rng=None):
        """Same tuples as RawDataset.iterate: (mol_Xs [N,4] float64, mol_ids, mol_yts or None, mol_grads or None)."""
        rng = np.random.default_rng() if rng is None else rng
        for sel in self.selections(batch_size, shuffle, rng):
            sel, out_off, n = self.batch_atoms(sel)
            xs, ys, zs, types, mol_ids = self.gather(sel)
            mol_Xs = np.stack([types.astype(np.float64), xs.astype(np.float64), ys.astype(np.float64), zs.astype(np.float64)], axis=1)
            if fuzz is not None:
                mol_Xs[:, 1:4] += rng.uniform(-fuzz, fuzz, (n, 3))
            mol_yts = None if self.ys is None else list(self.ys[sel])
            mol_grads = None if self.grads is None else self.gather_grads(sel, out_off)
            yield mol_Xs, mol_ids, mol_yts, mol_grads


def split_columns(mol_Xs, mol_ids, dtype=np.float32):
    """(type, x, y, z) rows -> the flat arrays the ops take: xs, ys, zs [N] dtype; atom types, mol ids int32
    (trainer_multi_tower.py:769-779)."""
    mol_Xs = np.asarray(mol_Xs)
    return (np.ascontiguousarray(mol_Xs[:, 1], dtype=dtype), np.ascontiguousarray(mol_Xs[:, 2], dtype=dtype),
            np.ascontiguousarray(mol_Xs[:, 3], dtype=dtype), np.ascontiguousarray(mol_Xs[:, 0]).astype(np.int32),
            np.ascontiguousarray(mol_ids, dtype=np.int32))


class DeviceBatch:
    """One batch resident on the GPU, with everything `featurize` needs."""

    __slots__ = ("xs", "ys", "zs", "atom_types", "mol_idxs", "n_mols", "mol_atom_counts", "mol_offsets",
                 "scatter_idxs", "gather_idxs", "atom_counts", "size_order", "counts_pinned", "labels", "grads", "ready",
                 "memory", "sizes", "totals", "made_on")

    def __init__(self):
        self.labels = self.grads = self.counts_pinned = None
        self.made_on = None       # the stream that `ready` was recorded on (its address, on the arrays' device)
        self.memory = self.sizes = self.totals = None    # of a batch from the host: its one buffer, molecule sizes, counts

    def host_counts(self):
        """-> (atoms per type, a list of 4; the size order on the device; molecules per size class, int32[4] on the host): what
        the host has to know before it can launch the passes.  A batch from the host brings them along; otherwise the sort
        writes them to pinned memory, and this waits for it.  The numbers may be there before the batch's arrays are, so
        the current stream is made to wait for those: what it is given from here on finds them (work for a further stream:
        `wait()` there).  Waiting for them on the host instead costs 8 us: 74 -> 83 us for the featurizer's step on 1,024
        organic molecules."""
        acs, order, classes = self._counts()
        if isinstance(classes, tuple):
            import torch
            classes = torch.tensor(classes, dtype=torch.int32)
        return acs, order, classes

    def _counts(self, waited=False):
        """`host_counts()`, with the class totals of a batch from the host as they are held (a tuple; a tensor costs 10 us).
        `waited`: the current stream has done so already."""
        if not waited:
            self._join()
        if self.totals is not None:
            return list(self.totals[0]), self.size_order, self.totals[1]
        counts = _native.load().wait_for_counts(self.counts_pinned)
        if counts is None:
            self.ready.synchronize()
            counts = self.counts_pinned[0:4].tolist(), self.counts_pinned[4:8].clone()
        return counts[0], self.size_order, counts[1]

    def host_sizes(self):
        """The molecules' sizes, a list on the host."""
        if self.sizes is None:
            self._join()
        return self.mol_atom_counts.tolist() if self.sizes is None else self.sizes

    @classmethod
    def from_device_arrays(cls, xs, ys, zs, atom_types, mol_idxs, n_mols):
        """A batch from arrays that are on the GPU already: runs `mol_offsets`, `ani_sort` and `size_order` on the
        current stream and enqueues the copy of the counts."""
        import torch
        from . import ops
        b = cls()
        b.xs, b.ys, b.zs, b.atom_types, b.mol_idxs, b.n_mols = xs, ys, zs, atom_types, mol_idxs, n_mols
        b.finish_on_current_stream()
        return b

    def finish_on_current_stream(self):
        """Offsets, type sort, size order and the copy of the counts for the arrays already in place; records `ready`."""
        import torch
        from . import ops
        self.counts_pinned = torch.empty(8, dtype=torch.int32, pin_memory=True)     # from the pinned-memory cache; the sort writes it
        (self.mol_atom_counts, self.mol_offsets, self.scatter_idxs, self.gather_idxs, self.atom_counts,
         self.size_order) = ops.prepare_batch(self.mol_idxs, self.atom_types, self.n_mols, self.counts_pinned)
        self.ready = torch.cuda.Event()
        self.ready.record()
        self.made_on = self._current()

    def _current(self):
        import torch
        return torch._C._cuda_getCurrentRawStream(self.xs.device.index)

    def _join(self):
        """`wait()`, where the current stream is not the one the batch was made on."""
        if self._current() != self.made_on:
            self.wait()

    def wait(self, stream=None):
        """Makes the current stream (`stream`, if the caller has it at hand) wait for the copies and the sort of this batch."""
        import torch
        cur = torch.cuda.current_stream() if stream is None else stream
        cur.wait_event(self.ready)
        if self.memory is not None:        # the memory was allocated on the feeder's stream
            self.memory.record_stream(cur)
            if self.grads is not None:
                self.grads.record_stream(cur)
            return self
        for name in ("xs", "ys", "zs", "atom_types", "mol_idxs", "mol_atom_counts", "mol_offsets", "scatter_idxs",
                     "gather_idxs", "atom_counts", "size_order", "grads"):
            t = getattr(self, name)
            if t is not None:
                t.record_stream(cur)
        return self


class DeviceFeeder:
    """Iterates a RawDataset as DeviceBatch objects, one batch ahead of the consumer.

    Pinned staging buffers are allocated once (for the largest batch seen so far, two sets), a batch goes over in one
    copy on a side stream of default priority (a single batch, which nothing can overlap with, on the current stream),
    and its preparation is enqueued behind the copy.  The consumer calls `batch.wait()` before using the tensors on
    its own stream."""

    def __init__(self, dataset, batch_size, shuffle=False, fuzz=None, dtype=np.float32, device="cuda:0", rng=None):
        import torch
        self.dataset, self.batch_size, self.shuffle, self.fuzz = dataset, batch_size, shuffle, fuzz
        self.dtype, self.device, self.rng = dtype, torch.device(device), rng
        self.f64 = np.dtype(dtype) == np.float64
        alone = isinstance(dataset, (RawDataset, PackedDataset)) and dataset.num_batches(batch_size) <= 1
        self.stream = torch.cuda.current_stream(self.device) if alone else torch.cuda.Stream(device=self.device)
        self._stream_id = (self.stream.stream_id, self.stream.device_index, self.stream.device_type)
        self._pinned = [None, None]
        self._events = [None, None]       # the last copy out of a staging set

    def _staging(self, slot, n_bytes):
        import torch
        if self._pinned[slot] is None or self._pinned[slot].numel() < n_bytes:
            self._pinned[slot] = torch.empty(max(n_bytes, 1 << 16), dtype=torch.uint8, pin_memory=True)
        return self._pinned[slot]

    def _parts(self, slot, n):
        """The staging set's arrays for n atoms: xs, ys, zs, types, molecule indices (host tensors)."""
        native = _native.load()
        return native.staging_parts(self._staging(slot, native.staging_bytes(n, self.f64)), n, self.f64)

    def _fill_from_raw(self, slot, sel):
        """Molecule selection of a RawDataset -> staging set, read natively from the molecules' arrays.  None if they are
        not all contiguous float64 rows: numpy has to make those."""
        ds, native = self.dataset, _native.load()
        staged = native.stage_molecules(ds.all_Xs, sel, self._staging(slot, 0), self.f64)
        if isinstance(staged, int):
            staged = native.stage_molecules(ds.all_Xs, sel, self._staging(slot, staged), self.f64)
        if staged is None:
            return None
        n, sizes, totals = staged
        labels = grads = None
        if ds.all_ys is not None:
            labels = native.picked(ds.all_ys, sel) if type(ds.all_ys) is list else [ds.all_ys[p] for p in sel.tolist()]
        else:
            while sizes and sizes[-1] == 0:         # without labels the last molecule is the last that has atoms
                sizes.pop()
                totals = (totals[0], (totals[1][0] - 1,) + totals[1][1:])
        if ds.all_grads is not None:
            grads = np.concatenate([np.asarray(ds.all_grads[p]) for p in sel.tolist()], axis=0)
        return n, len(sizes), labels, grads, sizes, totals

    def _fill_from_tuple(self, slot, item):
        """Reference-style tuple -> staging set; returns (n atoms, n molecules, labels, gradients)."""
        import torch
        mol_Xs, mol_ids, mol_yts, mol_grads = item
        xs, ys, zs, types, mids = split_columns(mol_Xs, mol_ids, self.dtype)
        n = xs.size
        # one molecule per label: trailing molecules without atoms still count (mol_ids alone would drop them)
        n_mols = len(mol_yts) if mol_yts is not None else (int(mids[-1]) + 1 if n else 0)
        if n and int(mids[-1]) >= n_mols:
            raise ValueError("mol_ids names molecule %d but the batch has %d labels" % (int(mids[-1]), n_mols))
        for part, values in zip(self._parts(slot, n), (xs, ys, zs, types, mids)):
            part.copy_(torch.from_numpy(values))
        return n, n_mols, mol_yts, mol_grads, None, None

    def _fill_from_packed(self, slot, sel):
        """Molecule selection of a PackedDataset -> staging set, gathered natively into the pinned buffers."""
        ds = self.dataset
        sel, out_off, n = ds.batch_atoms(sel)
        xs, ys, zs, types, mids = (part.numpy() for part in self._parts(slot, n))
        ds.gather_into(sel, out_off, xs, ys, zs, types, mids)
        if self.fuzz is not None:
            rng = np.random.default_rng() if self.rng is None else self.rng
            for part, noise in zip((xs, ys, zs), rng.uniform(-self.fuzz, self.fuzz, (3, n)).astype(xs.dtype)):
                part += noise
        labels = None if ds.ys is None else ds.ys[sel]            # an array here (a list from a RawDataset)
        grads = None if ds.grads is None else ds.gather_grads(sel, out_off)
        totals = _native.load().staged_totals(self._pinned[slot], n, out_off, self.f64)
        return n, sel.size, labels, grads, np.diff(out_off).tolist(), totals

    def _enqueue(self, slot, item):
        import torch
        if self._events[slot] is not None:
            self._events[slot].synchronize()          # the previous copy out of this staging set has finished
        if isinstance(self.dataset, PackedDataset):
            filled = self._fill_from_packed(slot, item)
        elif isinstance(item, np.ndarray):
            filled = self._fill_from_raw(slot, item)
            if filled is None:
                filled = self._fill_from_tuple(slot, self.dataset.batch(item))
        else:
            filled = self._fill_from_tuple(slot, item)
        b = DeviceBatch()
        n, b.n_mols, b.labels, mol_grads, b.sizes, b.totals = filled
        if b.totals is None:
            b.counts_pinned = torch.empty(8, dtype=torch.int32, pin_memory=True)
        (b.memory, b.xs, b.ys, b.zs, b.atom_types, b.mol_idxs, b.mol_atom_counts, b.mol_offsets, b.scatter_idxs, b.gather_idxs,
         b.atom_counts, b.size_order) = _native.load().feed_batch(self._staging(slot, 0), n, b.n_mols, self.f64, self.device,
                                                                  b.counts_pinned, self._stream_id)
        if mol_grads is not None:
            with torch.cuda.stream(self.stream):
                b.grads = torch.from_numpy(np.ascontiguousarray(mol_grads, dtype=self.dtype)).to(self.device)
        b.ready = self._events[slot] = torch.cuda.Event()
        b.made_on = self.stream.cuda_stream
        b.ready.record(self.stream)
        return b

    def __iter__(self):
        if isinstance(self.dataset, PackedDataset):
            if self.dataset.dtype != np.dtype(self.dtype):
                raise TypeError("the packed data set holds %s coordinates, the feeder was asked for %s"
                                % (self.dataset.dtype, np.dtype(self.dtype)))
            it = self.dataset.selections(self.batch_size, self.shuffle, self.rng)
        elif type(self.dataset) is RawDataset and self.fuzz is None:
            it = self.dataset.selections(self.batch_size, self.shuffle, self.rng)
        else:
            it = self.dataset.iterate(self.batch_size, self.shuffle, self.fuzz, self.rng)
        slot, ahead = 0, None
        for item in it:
            nxt = self._enqueue(slot, item)
            slot ^= 1
            if ahead is not None:
                yield ahead
            ahead = nxt
        if ahead is not None:
            yield ahead
