"""The launch shapes that depend on the size of the batch, at the sizes where they change: the same molecules in a batch
that gives each of them more wavefronts or workgroups and in one that does not."""
import numpy as np
import pytest

from khan_amd import datagen

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from khan_amd import _lib, ops as _ops
    _lib.load()
    return _ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def passes(ops, b, n_mols, dtype, upstream, vectors):
    """Rows, gradients and Jacobian-vector rows, in atom order, of the first n_mols molecules of batch b run alone."""
    n = int(b.MOs[n_mols - 1] + b.MACs[n_mols - 1])
    X, Y, Z = (dev(v[:n]).to(dtype) for v in (b.X, b.Y, b.Z))
    macs, mos = ops.mol_offsets(dev(b.mol_idxs[:n]), n_mols)
    sc, ga, ac = ops.ani_sort(dev(b.A[:n]))
    acs, order, ga = ac.cpu().tolist(), ops.size_order(macs), ga.long()
    classes = order[-4:].cpu()
    args = (X, Y, Z, dev(b.A[:n]), mos, macs, sc, acs)
    rows = torch.cat(ops.featurize(*args, order=order, size_classes=classes)).view(-1, 384)[ga]
    buckets = torch.empty((n, 384), dtype=dtype, device=DEV)
    buckets[ga] = upstream[:n]
    grads = torch.stack(ops.featurize_grad(*args, *torch.split(buckets.view(-1), [c * 384 for c in acs]), order=order, size_classes=classes), dim=1)
    jvp = torch.cat(ops.featurize_grad_inverse(*args, *(v[:n].contiguous() for v in vectors), order=order, size_classes=classes)).view(-1, 384)[ga]
    return rows, grads, jvp


# sizes on both sides of the lines at which a molecule gets 2, 4, 8 (16) wavefronts or workgroups
@pytest.mark.parametrize("kind,dtype,most,sizes", [
    ("organic", torch.float32, 16500, (1, 1023, 1025, 2049, 4097, 8192)),
    ("organic", torch.float64, 8300, (1, 511, 1025, 2048, 4096)),
    ("boxes", torch.float32, 2200, (1, 127, 257, 1024)),
    ("boxes", torch.float64, 600, (1, 63, 65, 256)),
])
def test_molecules_shared_by_several_wavefronts(ops, kind, dtype, most, sizes):
    b = datagen.make_batch(kind, most)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(3)
    upstream = torch.randn((b.n_atoms, 384), dtype=dtype, device=DEV, generator=gen)
    vectors = torch.randn((3, b.n_atoms), dtype=dtype, device=DEV, generator=gen)
    rows, grads, jvp = passes(ops, b, most, dtype, upstream, vectors)
    tol = 2e-6 if dtype == torch.float32 else 4e-15       # forces are sums in another order
    for n_mols in sizes:
        r, g, j = passes(ops, b, n_mols, dtype, upstream, vectors)
        n = r.shape[0]
        print("   %s %s, %d molecules" % (kind, dtype, n_mols), flush=True)
        assert torch.equal(r, rows[:n]) and torch.equal(j, jvp[:n])
        assert float((g - grads[:n]).abs().max()) <= tol * float(grads[:n].abs().max())

@pytest.mark.parametrize("n_atoms,n_mols", [(0, 0), (0, 3), (1, 1), (63, 5), (2047, 100), (2048, 2048), (4096, 2047), (4097, 300), (5000, 1), (16384, 2048), (16385, 1300),
                                            (100003, 9000), (3000, 2049)])
def test_batch_preparation_in_one_call(ops, n_atoms, n_mols):
    """prepare_batch against mol_offsets, ani_sort and size_order, around the tile sizes and the line between its two forms."""
    rng = np.random.default_rng(n_atoms + n_mols)
    ids = np.sort(rng.integers(0, max(n_mols, 1), n_atoms)).astype(np.int32)
    types = rng.choice(4, size=n_atoms, p=[0.55, 0.3, 0.1, 0.05]).astype(np.int32)
    if n_atoms > 4:
        types[3] = 7                                             # out of range: counted as O
    pinned = torch.full((8,), -1, dtype=torch.int32, pin_memory=True)
    macs, mos, sc, ga, ac, order = ops.prepare_batch(dev(ids), dev(types), n_mols, pinned)
    torch.cuda.synchronize()
    want_sc, want_ga, want_ac = ops.ani_sort(dev(types))
    assert torch.equal(sc, want_sc) and torch.equal(ga, want_ga) and torch.equal(ac, want_ac)
    t = np.where((types < 0) | (types > 3), 3, types)
    assert np.array_equal(ga.cpu().numpy()[np.argsort(t, kind="stable")], np.arange(n_atoms))
    if n_mols == 0:
        return
    sizes = np.bincount(ids, minlength=n_mols)
    assert np.array_equal(macs.cpu().numpy(), sizes) and np.array_equal(mos.cpu().numpy(), np.cumsum(sizes) - sizes)
    want = ops.size_order(macs)
    assert torch.equal(order[n_mols:n_mols + 258], want[n_mols:n_mols + 258]) and torch.equal(order[-4:], want[-4:])
    o = order[:n_mols].cpu().numpy()
    assert np.array_equal(np.sort(o), np.arange(n_mols)) and np.all(np.diff(np.minimum(sizes[o], 257)) <= 0)
    assert pinned.tolist() == ac.cpu().tolist() + order[-4:].cpu().tolist()


@pytest.mark.parametrize("dtype,rtol", [(torch.float32, 1e-5), (torch.float64, 1e-12)])
@pytest.mark.parametrize("sizes", [(1,), (64, 65), (2, 63, 64, 65, 66, 127, 128, 129, 255, 256, 257, 513, 700), (12,) * 37 + (200,), (200,) * 9 + (5, 300)])
def test_charges_of_every_size_in_one_launch(ops, dtype, rtol, sizes):
    """Energies, dE/dq and dE/dxyz against float64 sums over all pairs: both sides of the limits between the forms, odd and
    even sizes, and batches of small molecules with a large one and the reverse (a workgroup per four molecules or per one)."""
    rng = np.random.default_rng(len(sizes))
    n = sum(sizes)
    xyz = rng.uniform(0, 1, (n, 3)) * (np.repeat(sizes, sizes)[:, None] / 0.1) ** (1 / 3)
    q, g = rng.normal(0, 0.3, n), rng.standard_normal(len(sizes))
    xyz, q, g = (v.astype(np.float32 if dtype == torch.float32 else np.float64).astype(np.float64) for v in (xyz, q, g))
    macs = np.array(sizes, dtype=np.int32)
    mos = (np.cumsum(sizes) - sizes).astype(np.int32)
    out = ops.ani_charge_all(*(dev(v).to(dtype) for v in (xyz[:, 0], xyz[:, 1], xyz[:, 2], q)), dev(mos), dev(macs), dev(g).to(dtype))
    e_alone = ops.ani_charge(*(dev(v).to(dtype) for v in (xyz[:, 0], xyz[:, 1], xyz[:, 2], q)), dev(mos), dev(macs))
    e, dq, dx, dy, dz = (v.cpu().numpy().astype(np.float64) for v in out)
    K, Rc = float(np.float32(0.529176917)), float(np.float32(4.6))
    for m, (o, k) in enumerate(zip(mos, macs)):
        s = slice(o, o + k)
        d = xyz[s][:, None] - xyz[s][None]
        r = np.sqrt((d ** 2).sum(-1)) + np.eye(k) * 1e9
        near = r <= Rc
        damp = np.where(near, 0.5 - 0.5 * np.cos(np.pi * r / Rc), 1.0) * (1 - np.eye(k))
        ddamp = np.where(near, 0.5 * np.pi / Rc * np.sin(np.pi * r / Rc), 0.0)
        pot = K * damp / r
        want_q = pot @ q[s]
        want_e = 0.5 * q[s] @ want_q
        fac = K * (ddamp / r - damp / r ** 2) / r * (1 - np.eye(k)) * q[s][:, None] * q[s][None]
        want_x = (fac[:, :, None] * d).sum(1)
        mag = 0.5 * np.abs(q[s]) @ (pot @ np.abs(q[s])) + 1e-30
        assert abs(e[m] - want_e) <= rtol * mag and abs(float(e_alone[m]) - want_e) <= rtol * mag, (m, k)
        assert np.abs(dq[s] - g[m] * want_q).max() <= rtol * (np.abs(g[m]) * (pot @ np.abs(q[s])).max() + 1e-30), (m, k)
        got = np.stack([dx[s], dy[s], dz[s]], axis=1)
        assert np.abs(got - g[m] * want_x).max() <= 2 * rtol * (np.abs(g[m]) * (np.abs(fac)[:, :, None] * np.abs(d)).sum(1).max() + 1e-30), (m, k)
