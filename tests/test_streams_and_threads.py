"""A batch that is still on its way is waited for by whatever stream its passes are given on; one model on several streams and
from several threads."""
import threading

import numpy as np
import pytest
import torch

from khan_amd import batching, datagen, model


class _Stream:
    def __init__(self):
        self.waited = []

    def wait_event(self, event):
        self.waited.append(event)


class _Tensor:
    def __init__(self):
        self.used_on = []

    def record_stream(self, stream):
        self.used_on.append(stream)


def test_the_counts_bring_the_batch_with_them(monkeypatch):
    """The counts can be on the host before the batch's arrays are complete: asking for them orders the current stream behind the
    batch and tells the allocator, on another stream than the batch's own."""
    own, other = _Stream(), _Stream()
    b = batching.DeviceBatch()
    b.xs, b.ready, b.made_on, b.memory, b.size_order, b.totals = torch.zeros(1), object(), id(own), _Tensor(), None, ((1, 2, 3, 4), (1, 0, 0, 0))
    for current, waited in ((own, []), (other, [b.ready])):
        monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: current)
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda *a: id(current), raising=False)
        assert b.host_counts()[0] == [1, 2, 3, 4]
        assert current.waited == waited
    assert b.memory.used_on == [other]


def _data(n_mols, first):
    b = datagen.make_batch("organic", n_mols, first_mol=first)
    rows = np.concatenate([b.A[:, None].astype(np.float64), np.stack([b.X, b.Y, b.Z], axis=1)], axis=1)
    return batching.RawDataset(np.split(rows, np.cumsum(b.MACs)[:-1]), [0.0] * n_mols)


DELAY = 20_000_000           # cycles that a batch's stream is held up for: about ten milliseconds


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("side", [False, True])
def test_a_feeder_batch_in_flight(dtype, side):
    """Energies and gradients of batches nobody called wait() for, on the default stream and on another one."""
    m = model.AniModel(dtype=dtype, seed=3)
    data = _data(120, 5)
    energies, gradients = np.array(m.predict(data)), np.concatenate(list(m.coordinate_gradients(data)))
    feeder = m._feeder(data, 40)
    got = []
    batches = iter(feeder)
    with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.current_stream()):
        for _ in range(3):
            with torch.cuda.stream(feeder.stream):
                torch.cuda._sleep(DELAY)
            b = next(batches)
            got.append(m.batch_energies(b, need_grad=True))
            del b
        torch.cuda.current_stream().synchronize()
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    for part, want in zip((torch.cat([e for e, _ in got]), torch.cat([g for _, g in got])), (energies, gradients)):
        part = part.cpu().numpy()
        assert part.shape == want.shape and np.abs(part - want).max() <= tol * np.abs(want).max()


@pytest.mark.gpu
def test_a_batch_made_on_another_stream():
    m = model.AniModel(seed=3)
    b = datagen.make_batch("organic", 3000)
    arrays = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (b.X, b.Y, b.Z, b.A, b.mol_idxs)]
    want = m.batch_energies(batching.DeviceBatch.from_device_arrays(*arrays, b.n_mols), need_grad=True)
    torch.cuda.synchronize()
    maker, user = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(maker):
            torch.cuda._sleep(DELAY)
            made = batching.DeviceBatch.from_device_arrays(*arrays, b.n_mols)
        with torch.cuda.stream(user):
            got = m.batch_energies(made, need_grad=True)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_one_model_in_several_threads(dtype):
    """Four threads with a stream each, every one with its own data set and all with the same model."""
    m = model.AniModel(dtype=dtype, fit_charges=dtype == torch.float64, seed=3)
    sets = [_data(30 + 7 * k, 100 * k) for k in range(4)]
    want = [np.array(m.predict(d)) for d in sets]
    got, failed = [[] for _ in sets], []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(10):
                    got[k].append(np.array(m.predict(sets[k], batch_size=16)))
        except Exception as e:                        # (an assertion in a thread would be lost)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    for w, runs in zip(want, got):
        assert len(runs) == 10 and all(np.abs(g - w).max() <= tol * np.abs(w).max() for g in runs)
