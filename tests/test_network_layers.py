"""The per-type networks of csrc/net_layers.hip (any widths, CELU) against library layers in float64 on the CPU: values,
gradients by rows and parameters, and the parameters' gradient of a loss on the row gradients."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ALPHA = 0.1
WIDTHS = [(384, 128, 128, 64, 1), (384, 256, 128, 64, 8, 1), (384, 5, 1), (7, 33, 17, 1), (64, 64, 66, 1)]
# rows per type around the 16- and 32-row tiles and the 64-row shares of the weight gradients; an empty type; one form for
# few rows and one for enough to fill the GPU
ROWS = [(0, 1, 15, 16), (17, 31, 33, 0), (64, 65, 1, 200), (9001, 8190, 0, 17)]


def _reference(widths, flat, xs, u, v):
    """[values], [row gradients], parameter gradients of sum(v . values) and of sum(u . row gradients)"""
    at, parts = 0, [[], []]
    for kind in (0, 1):
        for k, n in zip(widths, widths[1:]):
            size = k * n if kind == 0 else n
            parts[kind].append([flat[at + t * size:at + (t + 1) * size].reshape((k, n) if kind == 0 else (n,)) for t in range(4)])
            at += 4 * size
    values = []
    for t in range(4):
        a = xs[t]
        for l in range(len(widths) - 1):
            a = torch.addmm(parts[1][l][t], a, parts[0][l][t])
            if l < len(widths) - 2:
                a = torch.where(a >= 0, a, ALPHA * torch.expm1(torch.clamp(a, max=0.0) / ALPHA))
        values.append(a.reshape(-1))
    first = sum((v[t] * values[t]).sum() for t in range(4))
    rows = torch.autograd.grad(first, xs, create_graph=True)
    by_flat, = torch.autograd.grad(first, flat, retain_graph=True)
    second = sum((u[t] * rows[t]).sum() for t in range(4))
    by_flat2, by_v = torch.autograd.grad(second, (flat, v[1]))
    return values, rows, by_flat, by_flat2, by_v


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("widths", WIDTHS)
def test_networks_of_any_widths(widths, rows, dtype):
    from khan_amd import _native
    print("case:", widths, rows, dtype, flush=True)
    rng = np.random.default_rng(3)
    size = 4 * sum((k + 1) * n for k, n in zip(widths, widths[1:]))
    cast = lambda a: torch.from_numpy(a).to(dtype)
    flat = cast(rng.standard_normal(size) * 0.1)
    xs, u = ([cast(rng.standard_normal((n, widths[0]))) for n in rows] for _ in range(2))
    v = [cast(rng.standard_normal(n)) for n in rows]

    def leaves(to):
        return to(flat).requires_grad_(True), [to(x).requires_grad_(True) for x in xs], [to(x) for x in u], [to(x).requires_grad_(True) for x in v]

    want = _reference(widths, *leaves(lambda a: a.double().clone()))
    f, x, uu, vv = leaves(lambda a: a.cuda())
    native = _native.load()
    values = native.network_autograd(f, [a.reshape(-1) for a in x], list(widths), ALPHA)
    first = sum((vv[t] * values[t]).sum() for t in range(4))
    by_flat, *plain = torch.autograd.grad(first, [f] + x, retain_graph=True)
    grads = torch.autograd.grad(first, x, create_graph=True)
    by_flat2, by_v = torch.autograd.grad(sum((uu[t] * grads[t]).sum() for t in range(4)), (f, vv[1]))
    out = native.network_forward(f.detach(), [a.detach().reshape(-1) for a in x], list(widths), ALPHA, True)
    again = native.network_rows(f.detach(), [a.detach().reshape(-1) for a in x], list(widths), ALPHA, out[4:],
                                [a.detach() for a in vv], [a.reshape(-1).clone() for a in uu])

    tol = 2e-5 if dtype == torch.float32 else 1e-12

    def close(got, ref, what, but=0.0):
        ref = ref.detach()
        err = (got.detach().cpu().double() - ref).abs()
        size = ref.abs().max().item() if ref.numel() else 0.0
        assert (err > tol * (size + 1e-3)).sum().item() <= but * err.numel(), (what, err.max().item(), size)
    for t in range(4):
        close(values[t], want[0][t], "values")
        assert torch.equal(out[t], values[t])
        close(plain[t], want[1][t], "row gradients")
        assert torch.equal(plain[t], grads[t])
        close(again[t].reshape(-1) - uu[t].reshape(-1), want[1][t].reshape(-1), "row gradients added to others")
    close(by_flat, want[2], "parameter gradients")
    # CELU's second derivative jumps at 0: among a million activations in single precision one may lie on the other side,
    # which changes a few columns of the gradient
    close(by_flat2, want[3], "parameter gradients of a loss on the row gradients", but=0.02 if dtype == torch.float32 else 0.0)
    close(by_v, want[4], "factor gradients of a loss on the row gradients")
