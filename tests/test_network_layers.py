"""The per-type networks of csrc/net_layers.hip (any widths, CELU) against library layers in float64 on the CPU: values,
gradients by rows and parameters, and the parameters' gradient of a loss on the row gradients; single layers; what is left of
library operations."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ALPHA = 0.1
WIDTHS = [(384, 128, 128, 64, 1), (384, 256, 128, 64, 8, 1), (384, 5, 1), (7, 33, 17, 1), (64, 64, 66, 1)]
# rows per type around the 16- and 32-row tiles and the 64-row shares of the weight gradients; an empty type; one form for
# few rows and one for enough to fill the GPU
ROWS = [(0, 1, 15, 16), (17, 31, 33, 0), (64, 65, 1, 200), (9001, 8190, 0, 17)]


def _reference(widths, flat, xs, u, v, positive):
    """[values], [row gradients], parameter gradients of sum(v . values) and of sum(u . row gradients).  positive[l][t]: which
    side of 0 the activations of layer l lie on.  CELU and its first derivative are continuous there, its second jumps: an
    activation of the size of its rounding error counts as on the side that the tested pass found it on."""
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
                side = positive[l][t]
                assert (a.abs()[side != (a >= 0)] < 1e-5).all()
                a = torch.where(side, a, ALPHA * torch.expm1(torch.where(side, 0.0, a) / ALPHA))
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
    positive = [torch.split((a >= 0).cpu(), list(rows)) for a in out[4:-1]]
    want = _reference(widths, *leaves(lambda a: a.double().clone()), positive)

    tol = 2e-5 if dtype == torch.float32 else 1e-12

    def close(got, ref, what):
        ref = ref.detach()
        err = (got.detach().cpu().double() - ref).abs()
        size = ref.abs().max().item() if ref.numel() else 0.0
        assert (err <= tol * (size + 1e-3)).all(), (what, err.max().item(), size)
    for t in range(4):
        close(values[t], want[0][t], "values")
        assert torch.equal(out[t], values[t])
        close(plain[t], want[1][t], "row gradients")
        assert torch.equal(plain[t], grads[t])
        close(again[t].reshape(-1) - uu[t].reshape(-1), want[1][t].reshape(-1), "row gradients added to others")
    close(by_flat, want[2], "parameter gradients")
    close(by_flat2, want[3], "parameter gradients of a loss on the row gradients")
    close(by_v, want[4], "factor gradients of a loss on the row gradients")



class _Layer(ctypes.Structure):
    _fields_ = ([(name, ctypes.c_void_p * 4) for name in ("x", "w", "bias", "act", "d", "t", "scale", "out", "out2")] +
                [("n", ctypes.c_int32 * 4)] + [(name, ctypes.c_int32) for name in ("k", "n_out", "transposed", "kind", "accumulate")] +
                [("alpha", ctypes.c_double)])


# Float32 layers with split products: 64- and 128-column workgroups (from 128 and 512 tiles of 128 rows on), rows around the
# 128 of a workgroup, output widths that are no multiple of a tile, one or more chunks of 32 k, every kind of epilogue.
# What the split leaves out is below 2^-23 |x| |w|, the float32 sums of up to 96 products in 16s stay below 2e-6 of
# sum |x| |w| (as for the dense layers), and the epilogue adds a few roundings of its own terms (1e-6 of them).
@pytest.mark.parametrize("rows", [(16300, 127, 0, 1), (33000, 128, 129, 0)])
@pytest.mark.parametrize("k,n_out", [(32, 64), (64, 132), (96, 384)])
@pytest.mark.parametrize("transposed", [0, 1])
def test_split_products(rows, k, n_out, transposed):
    from khan_amd import _lib
    lib = _lib.load()
    print("case:", rows, k, n_out, transposed, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    make = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)
    x, w, bias = [make(n, k) for n in rows], [make(k, n_out) for _ in rows], [make(n_out) for _ in rows]
    stored = [(a.t() if transposed else a).contiguous() for a in w]
    act = [torch.nn.functional.celu(make(n, n_out), ALPHA) for n in rows]
    d, t = ([make(n, n_out) for n in rows] for _ in range(2))
    scale = [make(n) for n in rows]
    for kind, name in enumerate(("celu", "slope", "rows", "tangent", "second")):
        out, out2 = ([torch.ones(n, n_out, device="cuda") for n in rows] for _ in range(2))
        a = _Layer(k=k, n_out=n_out, transposed=transposed, kind=kind, accumulate=1, alpha=ALPHA)
        for i, n in enumerate(rows):
            a.n[i] = n
            for field, value in (("x", x), ("w", stored), ("act", act), ("d", d), ("t", t), ("scale", scale), ("out", out), ("out2", out2)):
                getattr(a, field)[i] = value[i].data_ptr()
            if name == "celu":
                a.bias[i] = bias[i].data_ptr()
        lib.khan_net_layer_f32.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        assert lib.khan_net_layer_f32(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        for i in range(4):
            y, size = x[i].double() @ w[i].double(), x[i].abs().double() @ w[i].abs().double()
            h, s = act[i].double(), scale[i].double()[:, None]
            slope = torch.where(h >= 0, 1.0, h / ALPHA + 1)
            want2 = None
            if name == "celu":
                want = torch.nn.functional.celu(y + bias[i].double(), ALPHA)
                bound = 2e-6 * size + 1e-6 * (bias[i].abs().double() + ALPHA)
            elif name == "slope":
                want, bound = y * slope, 2e-6 * size
            elif name == "rows":
                want, bound = y * s + 1, 2e-6 * size * s.abs() + 1e-6
            elif name == "tangent":
                want, bound = y * s * slope, 2e-6 * size * s.abs()
                want2 = torch.where(h >= 0, 0.0, y * s * d[i].double() / ALPHA)
                bound2 = 2e-6 * size * s.abs() * d[i].abs().double() / ALPHA
            else:
                want, bound = y * slope + s * t[i].double(), 2e-6 * size + 1e-6 * (s * t[i].double()).abs()
            assert ((out[i].double() - want).abs() <= bound).all(), (name, i)
            if want2 is not None:
                assert ((out2[i].double() - want2).abs() <= bound2).all(), (name, i)
            else:
                assert (out2[i] == 1).all(), (name, i)


class _Grads(ctypes.Structure):
    _fields_ = ([(name, ctypes.c_void_p * 4) for name in ("x", "x2", "scale")] +
                [(name, ctypes.c_void_p * 12) for name in ("left", "right", "left2", "right2")] +
                [("row0", ctypes.c_int64 * 4), ("n", ctypes.c_int32 * 4), ("layers", ctypes.c_int32), ("widths", ctypes.c_int32 * 13)] +
                [(name, ctypes.c_uint32) for name in ("first", "second")] + [(name, ctypes.c_int32) for name in ("scale_first", "scale_second")] +
                [(name, ctypes.c_void_p) for name in ("out", "workspace")])


# Weight gradients on split products (from 20,000 rows times tiles on): tiles of 128 x 128 and 128 x 64, widths that are no
# multiple of them, narrow layers beside them; rows around the 32 of a chunk and the 128 of a share; both pairs of operands or
# the first alone.  The float32 sums and the split stay below 2e-6 of sum |left| |right|.  Infinite and undefined operands
# give what they give in float64, element by element; odd row numbers and a pointer off its alignment take the other form.
@pytest.mark.parametrize("widths", [(384, 64, 128, 1), (64, 68, 132, 8, 1), (196, 192, 64, 1)])
@pytest.mark.parametrize("rows", [(9001, 33, 0, 1023), (127, 12800, 1, 31)])
@pytest.mark.parametrize("both", [False, True])
def test_weight_gradients_on_split_products(widths, rows, both):
    from khan_amd import _lib
    lib = _lib.load()
    print("case:", widths, rows, both, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(9)
    layers, total, row0 = len(widths) - 1, sum(rows), [sum(rows[:t]) for t in range(4)]
    # (the first column of the padding keeps arrays apart, so that `shift` may move them off their alignment)
    make = lambda w: torch.randn(total * w + 4, device="cuda", generator=gen)
    left, left2 = ([make(k) for k in widths[:-1]] for _ in range(2))
    right, right2 = ([make(k) for k in widths[1:]] for _ in range(2))
    scale = [torch.randn(n + 1, device="cuda", generator=gen) for n in rows]

    def gradients(shift=0):
        a = _Grads(layers=layers, first=(1 << layers) - 1, second=(1 << layers) - 1 if both else 0, scale_first=1, scale_second=0)
        for i, w in enumerate(widths):
            a.widths[i] = w
        for t in range(4):
            a.n[t], a.row0[t], a.scale[t] = rows[t], row0[t], scale[t].data_ptr()
            a.x[t], a.x2[t] = (v[0].data_ptr() + 4 * row0[t] * widths[0] for v in (left, left2))
        for l in range(layers):
            a.left[l], a.left2[l], a.right2[l] = left[l].data_ptr(), left2[l].data_ptr(), right2[l].data_ptr()
            a.right[l] = right[l].data_ptr() + 4 * (shift if l == 0 else 0) if l < layers - 1 else None
        out = torch.full((4 * sum((k + 1) * n for k, n in zip(widths, widths[1:])),), 7.0, device="cuda")
        work = torch.empty(lib.khan_net_grads_workspace_bytes_f32(ctypes.byref(a)), dtype=torch.uint8, device="cuda")
        a.out, a.workspace = out.data_ptr(), work.data_ptr()
        assert lib.khan_net_grads_f32(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        return out.cpu().double()

    def reference(shift=0):
        weights, sizes, sums, sum_sizes = [], [], [], []
        rows_of = lambda v, w, t, s=0: v[s:s + total * w].view(total, w)[row0[t]:row0[t] + rows[t]].cpu().double()
        for l, (k, n) in enumerate(zip(widths, widths[1:])):
            for t in range(4):
                s = scale[t][:rows[t]].cpu().double()[:, None]
                r = (rows_of(right[l], n, t, shift if l == 0 else 0) if l < layers - 1 else torch.ones(rows[t], 1, dtype=torch.float64)) * s
                pairs = [(rows_of(left[l], k, t), r)] + ([(rows_of(left2[l], k, t), rows_of(right2[l], n, t))] if both else [])
                weights.append(sum(p.t() @ q for p, q in pairs).reshape(-1))
                sizes.append(sum(p.abs().t() @ q.abs() for p, q in pairs).reshape(-1))
                sums.append(r.sum(0))
                sum_sizes.append(r.abs().sum(0))
        return torch.cat(weights + sums), torch.cat(sizes + sum_sizes)

    for shift in (0, 1):
        got, (want, size) = gradients(shift), reference(shift)
        assert ((got - want).abs() <= 2e-6 * size).all(), (shift, ((got - want).abs() / size).max().item())
    for what in (float("inf"), float("nan")):
        big = rows.index(max(rows))
        left[0][(row0[big] + 40) * widths[0] + 3] = what
        right[1][(row0[big] + 7) * widths[2] + 1] = -what
        got, (want, size) = gradients(), reference()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        known = torch.isfinite(want)
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
        assert ((got - want).abs() <= 2e-6 * size)[known].all()


def _one_layer_gradients(lib, left, right):
    """The weight and bias gradients of one layer with rows of one type: left [n, k], right [n, n_out] -> float64 on the CPU."""
    (n, k), n_out = left.shape, right.shape[1]
    a = _Grads(layers=1, first=1, second=0, scale_first=0, scale_second=0)
    a.widths[0], a.widths[1], a.n[0], a.x[0], a.right[0] = k, n_out, n, left.data_ptr(), right.data_ptr()
    out = torch.full((4 * (k + 1) * n_out,), 7.0, device="cuda")
    work = torch.empty(lib.khan_net_grads_workspace_bytes_f32(ctypes.byref(a)), dtype=torch.uint8, device="cuda")
    a.out, a.workspace = out.data_ptr(), work.data_ptr()
    assert lib.khan_net_grads_f32(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    return out[:k * n_out].view(k, n_out).cpu().double(), out[4 * k * n_out:][:n_out].cpu().double()


# Every plan of the weight gradients: few rows of many tiles (a wavefront to each run of the sums) and many rows of few (a
# workgroup), both sides of the lines between float32 and split products, several rounds of workgroups (36 tiles, 60,000 rows),
# narrow layers beside wide ones, with the same shares and (35,000 rows) larger ones, widths that are no multiple of anything.  A
# share's sum has at most 2,048 / 4 + 4 products one after the other on a lane and 64 on the split form's, shares and quarters
# carry their roundings: float64 stays below 520 units of 2^-53, float32 below the 2e-6 of the tests above (its sums over
# wavefronts and matrix steps are far from their worst case).
@pytest.mark.parametrize("dtype,bound", [(torch.float32, 2e-6), (torch.float64, 520 * 2.0 ** -53)])
@pytest.mark.parametrize("widths,rows", [((384, 512, 512, 256, 1), (5, 0, 1, 2)), ((384, 512, 512, 1), (31200, 20400, 3601, 4799)), ((384, 256, 1), (12000, 7000, 33, 1)),
                                         ((384, 128, 128, 64, 1), (1000, 700, 200, 98)), ((384, 128, 128, 64, 1), (1300, 850, 150, 200)),
                                         ((384, 128, 128, 64, 1), (2500, 1700, 300, 299)), ((384, 128, 128, 64, 1), (2500, 1700, 300, 301)),
                                         ((384, 128, 128, 64, 1), (18200, 11900, 2100, 2800)),
                                         ((384, 64, 1), (4000, 3000, 500, 499)), ((37, 66, 5, 1), (300, 0, 17, 1))])
def test_weight_gradients_of_every_plan(widths, rows, dtype, bound):
    from khan_amd import _lib
    lib = _lib.load()
    name = "f32" if dtype == torch.float32 else "f64"
    print("case:", widths, rows, name, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(11)
    layers, total, row0 = len(widths) - 1, sum(rows), [sum(rows[:t]) for t in range(4)]
    left = [torch.randn(total, w, device="cuda", dtype=dtype, generator=gen) for w in widths[:-1]]
    right = [torch.randn(total, w, device="cuda", dtype=dtype, generator=gen) for w in widths[1:]]
    a = _Grads(layers=layers, first=(1 << layers) - 1, second=0, scale_first=0, scale_second=0)
    for i, w in enumerate(widths):
        a.widths[i] = w
    for t in range(4):
        a.n[t], a.row0[t], a.x[t] = rows[t], row0[t], left[0][row0[t]:].data_ptr() if rows[t] else None
    for l in range(layers):
        a.left[l], a.right[l] = left[l].data_ptr(), right[l].data_ptr()
    out = torch.full((4 * sum((k + 1) * n for k, n in zip(widths, widths[1:])),), 7.0, device="cuda", dtype=dtype)
    work = torch.empty(getattr(lib, "khan_net_grads_workspace_bytes_" + name)(ctypes.byref(a)), dtype=torch.uint8, device="cuda")
    a.out, a.workspace = out.data_ptr(), work.data_ptr()
    for _ in range(2):                  # (twice: the same bits, whatever the workspace holds)
        previous = out.clone()
        assert getattr(lib, "khan_net_grads_" + name)(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, previous)
    at, bias_at = 0, 4 * sum(k * n for k, n in zip(widths, widths[1:]))
    for l, (k, n) in enumerate(zip(widths, widths[1:])):
        for t in range(4):
            x, y = (v[l][row0[t]:row0[t] + rows[t]].double() for v in (left, right))
            for got, want, size in ((out[at:at + k * n].view(k, n), x.t() @ y, x.abs().t() @ y.abs()), (out[bias_at:bias_at + n], y.sum(0), y.abs().sum(0))):
                assert ((got.double() - want).abs() <= bound * size).all(), (l, t, ((got.double() - want).abs() / size).max().item())
            at, bias_at = at + k * n, bias_at + n


# Operands at both ends of float32's exponents: near the bottom the third part of a bfloat16 split would run out of them, near
# the top the sums leave the split form.  Sums of 12,800 products in float32: the 2e-6 of sum |left| |right| of the test above.
# (sum |left| |right| stays below 2^127: beyond, which sums overflow depends on the order they are formed in.)
@pytest.mark.parametrize("left_exponent,right_exponent", [(0, -112), (0, -118), (0, -125), (-118, 0), (-125, 0), (-118, 40), (-60, -60), (0, 100),
                                                          (104, -104), (40, 30), (56, 56)])
def test_weight_gradients_of_tiny_and_huge_operands(left_exponent, right_exponent):
    from khan_amd import _lib
    lib = _lib.load()
    print("case:", left_exponent, right_exponent, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    make = lambda width, exponent: torch.ldexp(torch.randn(12800, width, device="cuda", generator=gen, dtype=torch.float64),
                                               torch.tensor(exponent, device="cuda")).float()
    left, right = make(384, left_exponent), make(128, right_exponent)
    weights, bias = _one_layer_gradients(lib, left, right)
    l, r = left.cpu().double(), right.cpu().double()
    want, size = l.t() @ r, l.abs().t() @ r.abs()
    assert size.max() < 2.0 ** 127
    assert ((weights - want).abs() <= 2e-6 * size).all(), ((weights - want).abs() / size).max().item()
    assert ((bias - r.sum(0)).abs() <= 2e-6 * r.abs().sum(0)).all()


@pytest.mark.parametrize("absolute", [False, True])
def test_celu_of_small_and_large_arguments(absolute):
    """The layers' float32 CELU over the binades of negative arguments from -1e-30 on (below, the split operands' smallest parts
    are subnormal): within 2^-21 of alpha expm1(z / alpha) (five roundings of 2^-24: alpha, its inverse, the argument, the
    function, the last product; the function has 1.5), never zero below zero, NaN kept; in its absolute form within
    2^-23 alpha more.  One input column and a weight of one make the layer's sum its argument."""
    from khan_amd import _lib
    lib = _lib.load()
    lib.khan_net_layer_f32.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    z = torch.cat([-torch.logspace(-30, 2, 40000), torch.tensor([0.0, -0.0, 1.5, -1e30, float("nan"), float("-inf"), float("inf")])]).cuda()
    x, w = torch.zeros(z.numel(), 32, device="cuda"), torch.zeros(32, 64, device="cuda")
    x[:, 0] = z
    w[0] = 1.0
    for first in (0, z.numel() - 64):                     # split products, which make NaN of infinities; the float32 instructions
        rows, arg = x[first:].contiguous(), z[first:].double()
        out = torch.empty(rows.shape[0], 64, device="cuda")
        a = _Layer(k=32, n_out=64, kind=5 if absolute else 0, alpha=ALPHA)
        a.n[1] = rows.shape[0]
        for field, value in (("x", rows), ("w", w), ("out", out)):
            getattr(a, field)[1] = value.data_ptr()
        assert lib.khan_net_layer_f32(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        got = out[:, 0].double()
        want = torch.where(arg < 0, ALPHA * torch.expm1(arg / ALPHA), arg)
        known = torch.isfinite(arg) if first == 0 else ~torch.isnan(arg)
        bound = torch.where(arg < 0, 2.0 ** -23 * ALPHA, 0.0) if absolute else 0.0
        assert ((got - want).abs() <= 2.0 ** -21 * want.abs() + bound)[known & ~torch.isinf(want)].all()
        assert ((got < 0) | absolute)[known & (arg < 0)].all() and torch.isnan(got[torch.isnan(arg)]).all()
        assert first == 0 or got[-1] == float("inf")


class _Top(ctypes.Structure):
    _fields_ = ([(name, ctypes.c_void_p * 4) for name in ("act", "w", "bias", "t", "scale", "value", "out")]
                + [("n", ctypes.c_int32 * 4), ("k", ctypes.c_int32), ("second", ctypes.c_int32), ("alpha", ctypes.c_double)])


@pytest.mark.parametrize("dtype,unit", [(torch.float32, 2.0 ** -24), (torch.float64, 2.0 ** -53)])
@pytest.mark.parametrize("k", [1, 5, 8, 63, 64, 68, 130, 256, 300])
def test_output_layer_of_any_width(k, dtype, unit):
    """The output layer alone, values and a w celu'(a) of it, and its second form scale t: widths on and off its steps of 64
    (32) values, rows that are 16-byte aligned and rows that are not, a type without rows.  A value is a sum over lanes of
    k / 16 + 1 products each, four steps and a bias: (k / 16 + 6) roundings of the products' sizes; celu' is three."""
    from khan_amd import _lib
    lib = _lib.load()
    run = getattr(lib, "khan_net_top_f32" if dtype == torch.float32 else "khan_net_top_f64")
    run.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    gen = torch.Generator(device="cuda").manual_seed(k)
    for shift in (0, 1):
        some = lambda *shape: torch.randn(int(np.prod(shape)) + shift, dtype=dtype, device="cuda", generator=gen)[shift:].view(*shape)
        rows = (17, 0, 1, 40)
        act, t = [[0.1 * some(n, k) if n else None for n in rows] for _ in range(2)]
        act = [torch.cat([torch.zeros(shift, dtype=dtype, device="cuda"), a.reshape(-1)])[shift:].view(-1, k) if a is not None else None for a in act]
        w, bias, scale = [some(k) for _ in rows], [some(1) for _ in rows], [some(max(n, 1)) for n in rows]
        out, value = [some(max(n, 1), k) for n in rows], [some(max(n, 1)) for n in rows]

        def launch(second, scaled):
            a = _Top(k=k, second=second, alpha=ALPHA)
            for i, n in enumerate(rows):
                a.n[i] = n
                if n == 0:
                    continue
                a.out[i] = out[i].data_ptr()
                if second:
                    a.t[i] = t[i].data_ptr()
                    if scaled:
                        a.scale[i] = scale[i].data_ptr()
                else:
                    a.act[i], a.w[i], a.bias[i], a.value[i] = (v[i].data_ptr() for v in (act, w, bias, value))
            assert run(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0

        launch(0, False)
        for i, n in enumerate(rows):
            if n:
                h, weight = act[i].double(), w[i].double()
                size = h.abs() @ weight.abs() + bias[i].double().abs()
                assert ((value[i].double() - (h @ weight + bias[i].double())).abs() <= (k / 16 + 6) * unit * 1.01 * size + 4e-16 * size).all()
                want = weight * torch.where(h >= 0, 1.0, h / ALPHA + 1)
                assert ((out[i].double() - want).abs() <= 3 * unit * 1.01 * weight.abs() * (1 + h.abs() / ALPHA) + 4e-16).all()
        for scaled in (False, True):
            launch(1, scaled)
            for i, n in enumerate(rows):
                if n:
                    assert torch.equal(out[i], t[i] * scale[i][:, None] if scaled else t[i])


@pytest.mark.parametrize("dtype,unit", [(torch.float32, 2.0 ** -24), (torch.float64, 2.0 ** -53)])
def test_bias_gradients_of_many_rows(dtype, unit):
    """Bias gradients are sums over all rows of factors of either sign: the output layer's of four types' 20,000 to 50,000 rows,
    ten sets of factors, lie within two roundings of the sums (2-norm; 0.9 measured in both precisions, 3.0 in single precision
    where the lanes' sums drop their rounding errors).  An infinite factor gives an infinity of its sign, not NaN."""
    from khan_amd import _native
    widths, rows = [8, 64, 1], (50000, 40000, 30000, 20000)
    rng = np.random.default_rng(8)
    flat = torch.from_numpy(rng.standard_normal(4 * sum((k + 1) * m for k, m in zip(widths, widths[1:])))).to(dtype).cuda().requires_grad_(True)
    xs = [torch.from_numpy(rng.standard_normal(n * 8)).to(dtype).cuda() for n in rows]
    values = _native.load().network_autograd(flat, xs, widths, ALPHA)
    got, want = [], []

    def of_outputs(factors):
        g, = torch.autograd.grad(values, flat, [torch.from_numpy(f).cuda() for f in factors], retain_graph=True)
        return g[-4:].cpu().numpy().astype(np.longdouble)

    for _ in range(10):
        factors = [torch.from_numpy(rng.standard_normal(n)).to(dtype).numpy() for n in rows]
        got.append(of_outputs(factors))
        want.append([f.astype(np.longdouble).sum() for f in factors])
    got, want = np.array(got), np.array(want)
    off = float(np.sqrt(((got - want) ** 2).sum() / (want ** 2).sum())) / unit
    print("bias gradients:", dtype, "%.3g units" % off, flush=True)
    assert off <= 2.0
    factors[1][17] = float("inf")
    assert np.isposinf(of_outputs(factors)[1])


class _Few(ctypes.Structure):
    _fields_ = ([("x", ctypes.c_void_p * 4), ("w", ctypes.c_void_p * 4 * 4), ("b", ctypes.c_void_p * 4 * 4), ("value", ctypes.c_void_p * 4),
                 ("grad", ctypes.c_void_p * 4), ("n", ctypes.c_int32 * 4), ("layers", ctypes.c_int32), ("widths", ctypes.c_int32 * 5),
                 ("alpha", ctypes.c_double)])


# Float64 networks in one launch: rows around its tiles of sixteen, an empty type, gradients by one workgroup a tile (from 86
# tiles on) and by three.  Float64 library layers on the CPU: 1e-12 for sums of a few hundred products, as for the layers.
@pytest.mark.parametrize("rows", [(0, 1, 15, 16), (17, 31, 33, 0), (1, 0, 0, 0), (1300, 50, 3, 0), (1400, 0, 0, 17)])
def test_float64_networks_in_one_launch(rows):
    from khan_amd import _lib
    lib = _lib.load()
    print("case:", rows, flush=True)
    gen = torch.Generator().manual_seed(6)
    widths = (384, 128, 128, 64, 1)
    rand = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)
    x = [rand(n, 384) for n in rows]
    w, b = [[rand(k, m) * 0.1 for _ in rows] for k, m in zip(widths, widths[1:])], [[rand(m) * 0.1 for _ in rows] for m in widths[1:]]

    def run(x, with_grad, shift=0):
        put = lambda t: t.cuda()
        xs, ws, bs = [torch.cat([torch.zeros(shift, dtype=t.dtype), t.reshape(-1)]).cuda()[shift:] for t in x], [list(map(put, v)) for v in w], [list(map(put, v)) for v in b]
        a = _Few(layers=4, alpha=ALPHA)
        values, grads = [torch.full((n + 1,), 7.0, device="cuda", dtype=torch.float64) for n in rows], [torch.full((n + 1, 384), 7.0, device="cuda", dtype=torch.float64) for n in rows]
        for i, k in enumerate(widths):
            a.widths[i] = k
        for t, n in enumerate(rows):
            a.n[t], a.x[t], a.value[t], a.grad[t] = n, xs[t].data_ptr(), values[t].data_ptr(), grads[t].data_ptr() if with_grad else None
            for l in range(4):
                a.w[l][t], a.b[l][t] = ws[l][t].data_ptr(), bs[l][t].data_ptr()
        status = lib.khan_net_few_f64(ctypes.byref(a), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert all((v[-1] == 7).item() and (g[-1] == 7).all().item() for v, g in zip(values, grads))
        return status, [v[:-1].cpu() for v in values], [g[:-1].cpu() for g in grads]

    want, want_grad = [], []
    for t in range(4):
        leaf = x[t].clone().requires_grad_(True)
        a = leaf
        for l in range(4):
            a = torch.addmm(b[l][t], a, w[l][t])
            if l < 3:
                a = torch.where(a >= 0, a, ALPHA * torch.expm1(torch.clamp(a, max=0.0) / ALPHA))
        want.append(a.detach().reshape(-1))
        want_grad.append(torch.autograd.grad(a.sum(), leaf)[0])
    close = lambda got, ref: ref.numel() == 0 or ((got - ref).abs() <= 1e-12 * (ref.abs().max() + 1e-3)).all().item()
    for with_grad in (True, False):
        status, values, grads = run(x, with_grad)
        assert status == 0 and all(map(close, values, want))
        assert all(map(close, grads, want_grad)) if with_grad else all((g == 7).all() for g in grads)
    # a row that is not a number stays alone
    big = rows.index(max(rows))
    spoilt = [t.clone() for t in x]
    spoilt[big][rows[big] // 2, 11] = float("nan")
    _, values, grads = run(x, True)
    _, other_values, other_grads = run(spoilt, True)
    others = torch.arange(rows[big]) != rows[big] // 2
    assert torch.isnan(other_values[big][~others]).all() and torch.isnan(other_grads[big][~others]).all()
    assert torch.equal(values[big][others], other_values[big][others]) and torch.equal(grads[big][others], other_grads[big][others])
    # operands off their alignment are refused; `infer` then goes layer by layer
    assert run(x, True, shift=1)[0] != 0
    widths_c = (ctypes.c_int32 * 5)(384, 128, 128, 65, 1)
    assert lib.khan_net_few_fits(widths_c, 4) == 0


class _Chain(ctypes.Structure):
    _fields_ = ([("x", ctypes.c_void_p * 4), ("w", ctypes.c_void_p * 4 * 12), ("b", ctypes.c_void_p * 4 * 12)] +
                [(name, ctypes.c_void_p * 4) for name in ("scale", "value", "grad")] + [("workspace", ctypes.c_void_p), ("n", ctypes.c_int32 * 4), ("layers", ctypes.c_int32),
                 ("widths", ctypes.c_int32 * 13), ("want_rows", ctypes.c_int32), ("accumulate", ctypes.c_int32), ("absolute", ctypes.c_uint32), ("alpha", ctypes.c_double)])


# Float32 networks in a launch each way: rows around the 32 and the 64 of a workgroup, either form (64 rows: with four wavefronts
# 262, 409 and 549 tiles of them, with eight 144, 262 and 409), an empty type; four wavefronts and eight, widths on and off the padding to 64, layers so narrow
# that two wavefronts share their columns, one hidden layer and eleven, row gradients of one and of more passes over a workgroup's
# columns.  A layer's sums are within 2e-6 of their products' sizes (as for single layers), and the weights are drawn to keep the
# sizes, so that a value is within 2e-6 of the largest a layer; a slope takes its activation's error over alpha, and
# the way back adds that of as many layers again.
@pytest.mark.parametrize("rows", [(0, 1, 31, 33), (32, 63, 64, 65), (16500, 33, 0, 129), (9001, 65, 0, 31), (26000, 63, 0, 33), (32800, 65, 0, 31), (20000, 15000, 33, 1)])
@pytest.mark.parametrize("widths", [(384, 128, 128, 64, 1), (128, 5, 1), (384, 256, 256, 200, 8, 1), (256, 129, 64, 1), (384,) + (64,) * 10 + (70, 1)])
def test_float32_networks_in_one_launch_each_way(widths, rows):
    from khan_amd import _lib
    lib = _lib.load()
    print("case:", widths, rows, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(6)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    layers, alpha, st = len(widths) - 1, 0.5, torch.cuda.current_stream().cuda_stream
    x, scale, start = [rand(n, widths[0]) for n in rows], [rand(n) for n in rows], [rand(n + 1, widths[0]) for n in rows]
    w, b = [[rand(k, m) * k ** -0.5 for _ in rows] for k, m in zip(widths, widths[1:])], [[rand(m) * 0.1 for _ in rows] for m in widths[1:]]

    def run(x, want_rows, plain=False):
        a = _Chain(layers=layers, want_rows=want_rows, accumulate=not plain, alpha=alpha, absolute=1)
        values, grads = [torch.full((n + 1,), 7.0, device="cuda") for n in rows], [g.clone() for g in start]
        for i, k in enumerate(widths):
            a.widths[i] = k
        for t, n in enumerate(rows):
            a.n[t], a.x[t], a.value[t], a.grad[t] = n, x[t].data_ptr(), values[t].data_ptr(), grads[t].data_ptr()
            a.scale[t] = None if plain else scale[t].data_ptr()
            for l in range(layers):
                a.w[l][t] = w[l][t].data_ptr()
                a.b[l][t] = None if l == 0 and t == 1 else b[l][t].data_ptr()
        size = lib.khan_net_chain_workspace_bytes(ctypes.byref(a))
        workspace = torch.full((size + 64,), 255, dtype=torch.uint8, device="cuda")      # NaN wherever it is read before it is written
        a.workspace = workspace.data_ptr()
        assert lib.khan_net_chain_values_f32(ctypes.byref(a), st) == 0
        if want_rows:
            assert lib.khan_net_chain_rows_f32(ctypes.byref(a), st) == 0
        else:
            assert lib.khan_net_chain_rows_f32(ctypes.byref(a), st) != 0
        assert all((v[-1] == 7).item() and torch.equal(g[-1], s[-1]) for v, g, s in zip(values, grads, start)) and (workspace[size:] == 255).all()
        return [v[:-1] for v in values], [g[:-1] for g in grads]

    want, want_grad = [], []
    for t in range(4):
        leaf = x[t].double().requires_grad_(True)
        h = leaf
        for l in range(layers):
            h = h @ w[l][t].double() + (0.0 if l == 0 and t == 1 else b[l][t].double())
            if l + 1 < layers:
                h = torch.nn.functional.celu(h, alpha)
        want.append(h.detach().reshape(-1))
        want_grad.append(torch.autograd.grad(h.sum(), leaf)[0])
    tol = 2e-6 * layers

    def close(got, ref, tol):
        off = max(((g.double() - r).abs().max().item() if r.numel() else 0.0) for g, r in zip(got, ref))
        size = max(r.abs().max().item() for r in ref if r.numel())
        assert off <= tol * size, (off, size)
    values, grads = run(x, True)
    close(values, want, tol)
    close([g - s[:-1] for g, s in zip(grads, start)], [g * c.double()[:, None] for g, c in zip(want_grad, scale)], tol * (1 + 1 / alpha) + 1e-6)
    close(run(x, True, plain=True)[1], want_grad, tol * (1 + 1 / alpha))
    assert all(map(torch.equal, run(x, False)[0], values))
    # a row that is not a number stays alone
    big = rows.index(max(rows))
    spoilt = [t.clone() for t in x]
    spoilt[big][rows[big] // 2, 11] = float("nan")
    other_values, other_grads = run(spoilt, True)
    others = torch.arange(rows[big], device="cuda") != rows[big] // 2
    assert torch.isnan(other_values[big][~others]).all() and torch.isnan(other_grads[big][~others]).all()
    assert torch.equal(values[big][others], other_values[big][others]) and torch.equal(grads[big][others], other_grads[big][others])


def _run_chain(widths, x, w, alpha):
    """The four types' values and row gradients, without biases."""
    from khan_amd import _lib
    lib, st, layers = _lib.load(), torch.cuda.current_stream().cuda_stream, len(widths) - 1
    a = _Chain(layers=layers, want_rows=1, alpha=alpha)
    values, grads = [torch.empty(r.shape[0], device="cuda") for r in x], [torch.empty_like(r) for r in x]
    for i, k in enumerate(widths):
        a.widths[i] = k
    for t, r in enumerate(x):
        a.n[t], a.x[t], a.value[t], a.grad[t] = r.shape[0], r.data_ptr(), values[t].data_ptr(), grads[t].data_ptr()
        for l in range(layers):
            a.w[l][t] = w[l][t].data_ptr()
    workspace = torch.full((lib.khan_net_chain_workspace_bytes(ctypes.byref(a)),), 255, dtype=torch.uint8, device="cuda")
    a.workspace = workspace.data_ptr()
    assert lib.khan_net_chain_values_f32(ctypes.byref(a), st) == 0
    assert lib.khan_net_chain_rows_f32(ctypes.byref(a), st) == 0
    return values, grads


# No operand loses a bit, whatever stands beside it: a column of zeros but for one weight, and positive sums, pass a value through
# every layer as it is, and the weight comes back as the row's gradient; beside them are values 2^40 and weights 2^10 times as large
# that do not reach the result.  Exact: a value times one is the sum of its three parts.
@pytest.mark.parametrize("rows", [(3, 70, 0, 33), (26000, 33, 0, 129)])
@pytest.mark.parametrize("widths", [(128, 5, 1), (128, 128, 64, 1), (384, 256, 64, 256, 1)])
def test_float32_networks_in_one_launch_keep_every_bit(widths, rows):
    print("case:", widths, rows, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(9)
    values_of = lambda n: (torch.rand(n, generator=gen, device="cuda") + 1.0) * torch.exp2(torch.randint(-60, 40, (n,), generator=gen, device="cuda").float())
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    x, w = [], [[torch.zeros(k, m, device="cuda") for _ in rows] for k, m in zip(widths, widths[1:])]
    for t, n in enumerate(rows):
        x.append(rand(n, widths[0]) * 2.0 ** 80)
        x[t][:, 7] = values_of(n)
        if n > 2:
            x[t][:3, 7] = torch.tensor([1.0 + 2049.0 * 2.0 ** -23, 1.0 - 2.0 ** -24, 2.0 ** 24 - 1.0], device="cuda")
        at = 7
        for l in range(len(widths) - 1):
            to = (5 * l + 3) % widths[l + 1]
            if l + 1 < len(widths) - 1:
                w[l][t][:8, 0 if to else 1] = rand(8) * 2.0 ** 10           # (a column that nothing takes)
            w[l][t][:, to] = 0.0
            w[l][t][at, to] = 1.0
            at = to
    values, grads = _run_chain(widths, x, w, 0.5)
    for t, n in enumerate(rows):
        assert torch.equal(values[t], x[t][:, 7])
        assert (grads[t][:, 7] == 1).all() and grads[t].count_nonzero() == n
    # the weights' bits, in every layer; and the slopes', which take theirs from the layer above
    for l in range(len(widths) - 1):
        for v in values_of(3).tolist() + [1.0 + 2049.0 * 2.0 ** -23]:
            ones = [torch.where(torch.arange(widths[0], device="cuda") == 7, 1.0, r * 2.0 ** -70) for r in x]
            with_v = [[m * v if k == l else m for m in layer] for k, layer in enumerate(w)]
            values, grads = _run_chain(widths, ones, with_v, 0.5)
            want = torch.tensor(v, device="cuda")
            assert all((g == want).all() for g in values) and all((g[:, 7] == want).all() and g.count_nonzero() == g.shape[0] for g in grads)


# A sum of 256 terms whose result float32 holds is finite, whatever the sizes of its factors.
def test_float32_networks_in_one_launch_reach_as_far_as_float32():
    widths = (256, 64, 1)
    for up, down in ((121, -20), (-20, 110), (100, 10), (-60, -40)):
        x = [torch.full((n, 256), 2.0 ** up, device="cuda") for n in (33, 0, 2, 65)]
        w = [[torch.full((256, 64), 2.0 ** down, device="cuda") for _ in x], [torch.full((64, 1), 0.5, device="cuda") for _ in x]]
        values, grads = _run_chain(widths, x, w, 0.5)
        assert all((v == 2.0 ** (up + down + 8 + 5)).all() for v in values) and all((g == 2.0 ** (down + 5)).all() for g in grads)


# Rows of very different sizes, and columns of a layer whose sizes the next layer's weights undo: every row has the accuracy of its own
# size, in its value and in its gradient.  Bound: a layer's sums are within 2e-6 of their products' sizes (root mean squares, four times
# for the largest of many); an activation's error is handed on by the next weights, a slope lies between those at both ends of
# its activation's error, and the way back hands on the slopes' errors and adds as much of its own.
@pytest.mark.parametrize("rows", [(3, 70, 0, 33), (26000, 33, 0, 129)])
@pytest.mark.parametrize("widths", [(128, 128, 64, 1), (384, 256, 64, 256, 1)])
def test_float32_networks_in_one_launch_over_float32s_range(widths, rows):
    print("case:", widths, rows, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    layers, alpha = len(widths) - 1, 0.5
    powers = lambda n, most: torch.exp2(torch.randint(-most, most + 1, (n,), generator=gen, device="cuda").float())
    size = [powers(n, 80) for n in rows]
    x = [rand(n, widths[0]) * s[:, None] for n, s in zip(rows, size)]
    w = [[rand(k, m) * k ** -0.5 for _ in rows] for k, m in zip(widths, widths[1:])]
    for l in range(layers - 1):
        for t in range(4):
            by = powers(widths[l + 1], 12)
            w[l][t] *= by
            w[l + 1][t] /= by[:, None]
    values, grads = _run_chain(widths, x, w, alpha)
    each = 2e-6 * 4
    slope = lambda z: torch.exp(z.clamp(max=0.0) / alpha)
    for t, n in enumerate(rows):
        if n == 0:
            continue
        h, err, zs, errs = x[t].double(), torch.zeros_like(x[t], dtype=torch.float64), [], []
        for l in range(layers):
            m = w[l][t].double()
            err = (err.square() @ m.square()).sqrt() + each * (h.square() @ m.square()).sqrt()
            h = h @ m
            if l + 1 < layers:
                zs.append(h)
                errs.append(err)
                h = torch.where(h > 0, h, alpha * torch.expm1(h.clamp(max=0.0) / alpha))
        assert ((values[t] - h[:, 0]).abs() <= err[:, 0]).all()
        d, off = torch.ones(n, 1, dtype=torch.float64, device="cuda"), torch.zeros(n, 1, dtype=torch.float64, device="cuda")
        for l in reversed(range(layers)):
            m = w[l][t].double().t()
            off = (off.square() @ m.square()).sqrt() + each * (d.square() @ m.square()).sqrt()
            d = d @ m
            if l > 0:
                z, e = zs[l - 1], errs[l - 1]
                off = off * slope(z + e) + d.abs() * (slope(z + e) - slope(z - e) + 1e-6)         # (1 + a / alpha, of a rounded a)
                d = d * slope(z)
        assert ((grads[t] - d).abs() <= off + each * d.abs()).all()


def test_networks_that_one_launch_does_not_take():
    """Feature widths off 128, hidden layers wider than 256, more than eleven of them or none, an output that is no single value."""
    from khan_amd import _lib
    lib = _lib.load()
    fits = lambda *widths: lib.khan_net_chain_fits((ctypes.c_int32 * 16)(*widths), len(widths) - 1)
    assert fits(384, 256, 1) and fits(128, *[8] * 11, 1)
    assert not any((fits(96, 64, 1), fits(0, 64, 1), fits(384, 257, 1), fits(384, 0, 1), fits(128, *[8] * 12, 1), fits(384, 1), fits(384, 64, 2)))


@pytest.mark.parametrize("layers,live", [((256, 64, 8, 1), 2), ((128, 128, 1), 2), ((128, 64, 1), 3), ((100, 1), 0)])
def test_parameters_behind_the_constant_layers_have_gradients(layers, live):
    """Without `weights_need_grad` the leading layers of a float32 network are constants and those behind them are not: their
    gradients, and those of a loss on the row gradients, are what `weights_need_grad` gives, and no other parameter has one."""
    from khan_amd import model
    net = model.MoleculeNN(layers, model.celu, torch.float32, "cuda:0", seed=2)
    gen = torch.Generator(device="cuda").manual_seed(1)
    feats = [torch.rand(n * 384, device="cuda", generator=gen).requires_grad_(True) for n in (300, 0, 17, 64)]
    params = net.parameters()
    results = []
    for need in (False, True):
        net.weights_need_grad = need
        energy = sum(v.sum() for v in net.type_outputs(feats))
        first = torch.autograd.grad(energy, params, allow_unused=True, retain_graph=True) if energy.requires_grad else [None] * len(params)
        rows = torch.autograd.grad(energy, feats, create_graph=True)
        loss = sum((r ** 2).sum() for r in rows)
        second = torch.autograd.grad(loss, params, allow_unused=True) if loss.requires_grad else [None] * len(params)
        results.append((first, second))
    layer_of = [k for t in model.TYPE_MAP for k, _ in enumerate(net.names[t]) for _ in (0, 1)]
    for (some, every) in zip(*results):
        for k, (a, b) in enumerate(zip(some, every)):
            if layer_of[k] < live:
                assert a is None
            else:
                assert a is not None and torch.equal(a, b)


def test_networks_under_tracing_and_transforms():
    """Forward mode, vmap, torch.func's gradients and tracers go through type_outputs as library operations did: a launch's values
    with the tangents, batches and graphs of those operations.  Float64: 1e-12 for sums of a few hundred products."""
    from khan_amd import model
    net = model.MoleculeNN((32, 16, 1), model.celu, torch.float64, "cuda:0", seed=2)
    gen = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *shape: torch.rand(*shape, device="cuda", generator=gen, dtype=torch.float64)
    rows = (5, 0, 3, 2)
    feats, tangents = [rand(n * 384) for n in rows], [rand(n * 384) for n in rows]
    energy = lambda *f: sum(v.sum() for v in net.type_outputs(f))
    plain = lambda *f: sum(net.atom_type_outputs(t, x.reshape(-1, 384)).sum() for t, x in enumerate(f))
    close = lambda a, b: bool(((a - b).detach().abs().max() <= 1e-12 * (1 + b.detach().abs().max())).item())
    grads = torch.func.grad(plain, argnums=(0, 2))(*feats)
    leaves = [f.clone().requires_grad_(True) for f in feats]
    directional = sum((g * v).sum() for g, v in zip(torch.autograd.grad(plain(*leaves), leaves), tangents))
    # forward mode, both forms
    value, tangent = torch.func.jvp(energy, tuple(feats), tuple(tangents))
    assert close(value, plain(*feats)) and close(tangent, directional)
    with torch.autograd.forward_ad.dual_level():
        duals = [torch.autograd.forward_ad.make_dual(f, v) for f, v in zip(feats, tangents)]
        assert close(torch.autograd.forward_ad.unpack_dual(energy(*duals)).tangent, directional)
    assert all(close(a, b) for a, b in zip(torch.func.grad(energy, argnums=(0, 2))(*feats), grads))
    batch = [torch.stack([f, v]) for f, v in zip(feats, tangents)]
    assert all(close(a, b) for a, b in zip(torch.vmap(energy)(*batch), (plain(*feats), plain(*tangents))))
    # tracers record operations, not the values of one call (torch.jit takes no constants that require gradients)
    for p in net.parameters():
        p.requires_grad_(False)
    assert close(torch.jit.trace(energy, tuple(feats), check_trace=False)(*tangents), plain(*tangents))
    from torch.fx.experimental.proxy_tensor import make_fx
    assert close(make_fx(energy)(*feats)(*tangents), plain(*tangents))
    assert close(energy(*feats), plain(*feats))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("layers,rows", [((128, 128, 64, 1), (40, 0, 3, 1)), ((100, 8, 1), (40, 0, 3, 1)), ((128, 100, 1), (40000, 0, 65, 17))])
def test_infinite_and_undefined_rows_stay_alone(layers, rows, dtype):
    """A feature that is NaN or infinite reaches its own row and no other: every other value and row gradient has the bits it has
    without it.  NaN stays NaN; in float64 an infinity gives what the library operations give."""
    from khan_amd import model
    net = model.MoleculeNN(layers, model.celu, dtype, "cuda:0", seed=2)
    gen = torch.Generator(device="cuda").manual_seed(1)
    clean = [torch.rand(n, 384, device="cuda", generator=gen, dtype=dtype) for n in rows]

    def passes(feats):
        leaves = [f.clone().requires_grad_(True) for f in feats]
        values = net.type_outputs([f.reshape(-1) for f in leaves])
        return values, torch.autograd.grad(sum(v.sum() for v in values), leaves)

    want, want_g = passes(clean)
    for what in (float("nan"), float("inf"), float("-inf")):
        feats = [f.clone() for f in clean]
        at = rows[0] // 2
        feats[0][at, 5] = what
        values, grads = passes(feats)
        others = torch.arange(rows[0], device="cuda") != at
        assert torch.equal(values[0][others], want[0][others]) and torch.equal(grads[0][others], want_g[0][others])
        assert all(torch.equal(a, b) for a, b in zip(values[1:], want[1:])) and all(torch.equal(a, b) for a, b in zip(grads[1:], want_g[1:]))
        if what != what:
            assert torch.isnan(values[0][at]) and torch.isnan(grads[0][at]).all()
        elif dtype == torch.float64:
            library = net.atom_type_outputs(0, feats[0][at:at + 1])[0].detach()
            assert torch.equal(torch.isnan(values[0][at]), torch.isnan(library)) and (torch.isnan(library) or values[0][at] == library)


def test_differentiable_layers_one_by_one():
    """autograd.dense, dense_first and dense_head (one layer of the four networks, the last one with the output layer): values and
    the gradients by rows, weights and biases, and of a loss on the row gradients, against float64; 2e-5 of the largest
    element, as for whole networks."""
    from khan_amd import autograd
    rng = np.random.default_rng(4)
    rows = (130, 0, 1, 40)
    f32 = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    for head, first in ((False, False), (False, True), (True, False)):
        k, n_out = 384 if first else 128, 64 if head else 128
        xs, ws, bs = [f32(n, k) for n in rows], [f32(k, n_out) * 0.1 for _ in rows], [f32(n_out) * 0.1 for _ in rows]
        hs, cs, us = [f32(64, 1) for _ in rows], [f32(1) for _ in rows], [f32(n, k) for n in rows]
        results = []
        for kernels in (True, False):
            put = lambda arrays: [torch.from_numpy(a).to("cuda" if kernels else "cpu", torch.float32 if kernels else torch.float64).requires_grad_(True)
                                  for a in arrays]
            x, w, b, h, c, u = (put(a) for a in (xs, ws, bs, hs, cs, us))
            if kernels and head:
                out = autograd.dense_head(x, w, b, h, c)
            elif kernels:
                out = autograd.dense_first([a.reshape(-1) for a in x], rows, w, b) if first else autograd.dense(x, w, b)
            else:
                out = [torch.nn.functional.celu(a @ m + v, 0.1) for a, m, v in zip(x, w, b)]
                out = [(o @ m + v).reshape(-1) for o, m, v in zip(out, h, c)] if head else out
            energy = sum((o ** 2).sum() for o in out)
            leaves = x + w + b + (h + c if head else [])
            grads = torch.autograd.grad(energy, leaves, retain_graph=True)
            by_rows = torch.autograd.grad(energy, x, create_graph=True)
            second = torch.autograd.grad(sum((g * v.detach()).sum() for g, v in zip(by_rows, u)), w)
            results.append([t.detach().cpu().double() for t in (*out, *grads, *second)])
        for got, want in zip(*results):
            assert got.shape == want.shape
            assert want.numel() == 0 or float((got - want).abs().max()) <= 2e-5 * (1 + float(want.abs().max())), (head, first)


# The kernels between a charge network's passes: rows to atoms and back, ones and sums, around the 256 elements of a workgroup; an
# index outside the rows gives NaN and writes nothing.  Copies and single additions: exact.
@pytest.mark.parametrize("n, other", [(1, 700), (255, 0), (256, 257), (1025, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_rows_to_atoms_and_back(dtype, n, other):
    from khan_amd import _lib
    lib, suffix, st = _lib.load(), "f32" if dtype == torch.float32 else "f64", torch.cuda.current_stream().cuda_stream
    print("case:", dtype, n, other, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(8)
    rand = lambda k: torch.randn(k, generator=gen, device="cuda", dtype=dtype)
    row_of, rows = torch.randperm(n, generator=gen, device="cuda").int(), rand(n)
    bad = row_of.clone()
    bad[n // 2] = n
    bad[-1] = -1
    inside = (bad >= 0) & (bad < n)
    for index in (row_of, bad):
        out, ones = torch.zeros(n + 1, device="cuda", dtype=dtype), torch.zeros(other + 1, device="cuda", dtype=dtype)
        assert getattr(lib, "khan_take_rows_" + suffix)(rows.data_ptr(), index.data_ptr(), n, n, out.data_ptr(), ones.data_ptr(), other, st) == 0
        back = torch.zeros(n + 1, device="cuda", dtype=dtype)
        assert getattr(lib, "khan_put_rows_" + suffix)(out.data_ptr(), index.data_ptr(), n, n, back.data_ptr(), st) == 0
        use = inside if index is bad else torch.ones_like(inside)
        assert torch.equal(out[:-1][use], rows[index[use].long()]) and torch.isnan(out[:-1][~use]).all()
        assert (ones[:-1] == 1).all() and ones[-1] == 0 and out[-1] == 0 and back[-1] == 0
        want = torch.zeros(n, device="cuda", dtype=dtype)
        want[index[use].long()] = rows[index[use].long()]
        assert torch.equal(back[:-1], want)
    a, b, c, d = rand(n + 1), rand(other + 1), rand(n + 1), rand(other + 1)
    want = torch.cat([a[:-1] + c[:-1], a[-1:]]), torch.cat([b[:-1] + d[:-1], b[-1:]])
    assert getattr(lib, "khan_add_two_" + suffix)(a.data_ptr(), c.data_ptr(), n, b.data_ptr(), d.data_ptr(), other, st) == 0
    assert torch.equal(a, want[0]) and torch.equal(b, want[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_charges_refuse_what_is_no_index_of_a_row(dtype):
    """A model with charges: indices from atoms to rows are integers, one to an atom; 64 bits and strides change nothing.  A row that no
    index names has an undefined gradient, in its molecule and no other (an index outside the rows is the library gather's device
    assertion, and no test's)."""
    from khan_amd import datagen, model
    from khan_amd.batching import DeviceBatch
    m = model.AniModel((128, 64, 1), model.celu, dtype, "cuda:0", fit_charges=True, seed=2)
    c = datagen.make_batch("organic", 40)
    xyz = [torch.from_numpy(v).to("cuda", dtype) for v in (c.X, c.Y, c.Z)]
    types, mols = torch.from_numpy(c.A).cuda(), torch.from_numpy(np.repeat(np.arange(40, dtype=np.int32), c.MACs)).cuda()

    def passes(index=None, need_grad=True):
        b = DeviceBatch.from_device_arrays(*xyz, types, mols, 40)
        if index is not None:
            b.gather_idxs = index(b.gather_idxs)
        return m.batch_energies(b, need_grad=need_grad)

    want, want_g = passes()
    assert torch.isfinite(want).all() and torch.isfinite(want_g).all()
    for index in (lambda g: g.long(), lambda g: torch.stack([g, g], dim=1)[:, 0]):
        e, g = passes(index)
        assert torch.equal(e, want) and torch.allclose(g, want_g, rtol=1e-4, atol=1e-6)
    for index in (lambda g: g.float(), lambda g: g.double(), lambda g: g.short(), lambda g: g[:-1], lambda g: g[:, None], lambda g: torch.cat([g, g[:1]])):
        for need_grad in (True, False):
            with pytest.raises((RuntimeError, IndexError, ValueError, TypeError)):
                passes(index, need_grad)

    def twice(g):
        g = g.clone()
        g[-1] = g[0]
        return g
    g = passes(twice)[1]
    last = mols == 39
    assert torch.isnan(g[last]).any() and not torch.isnan(g[~last]).any()
