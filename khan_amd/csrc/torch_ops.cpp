// The tensor side of khan_amd.ops in native code: argument checks, output allocation and the call into libkhan_aev.so.
//
// A call on a small batch is bound by the host: the checks, the allocations and the marshalling of a dozen pointers took
// 20-35 us per call in Python (ctypes) and take 3-5 us here, which is what the launch itself costs.  The library is opened
// by path (init), so that a build named by KHAN_AEV_LIBRARY is used here too; nothing is linked against it.
#include <dlfcn.h>

#include <torch/csrc/Exceptions.h>

#include "torch_common.h"

namespace khan_torch {

Api api;
PyObject* khan_error = nullptr;

void raise(PyObject* type, const std::string& message)
{
    if (PyGILState_Check()) {
        PyErr_SetString(type, message.c_str());
        throw py::error_already_set();
    }
    python_error e;
    {
        const py::gil_scoped_acquire lock;
        PyErr_SetString(type, message.c_str());
        e.persist();
    }
    throw python_error(std::move(e));
}

static void init(const std::string& path, py::object error_type)
{
    void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (!lib) throw std::runtime_error(dlerror());
#define X(name)                                                                                  \
    api.name = reinterpret_cast<decltype(api.name)>(dlsym(lib, #name));                          \
    if (!api.name) throw std::runtime_error(path + " does not export " #name);
    KHAN_API(X)
#undef X
    khan_error = error_type.release().ptr();
}

// four ints from a tensor (a device tensor is copied) or a sequence, whatever int() takes; fractions are cut off
Counts counts4(const py::object& o, const char* what)
{
    Counts c{};
    if (THPVariable_Check(o.ptr())) {
        Tensor t = THPVariable_Unpack(o.ptr());
        if (t.is_cuda() || t.scalar_type() != at::kInt || !t.is_contiguous()) t = t.detach().cpu().to(at::kInt).contiguous();
        same_size(t.numel() == 4, what);
        std::copy_n(t.data_ptr<int32_t>(), 4, c.v);
    } else {
        int k = 0;
        for (const auto& item : o) {
            same_size(k < 4, what);
            c.v[k++] = PyLong_CheckExact(item.ptr()) ? item.cast<int32_t>() : py::int_(py::reinterpret_borrow<py::object>(item)).cast<int32_t>();
        }
        same_size(k == 4, what);
    }
    return c;
}

// ---------------------------------------------------------------------------------------------- preparation
// -> (macs, mos, scatter_idxs, gather_idxs, atom_counts, order), slices of one allocation
static int64_t up4(int64_t v) { return (v + 3) & ~int64_t(3); }

static std::array<int64_t, 6> prepared_sizes(int64_t n, int64_t n_mols) { return {n_mols, n_mols, n, n, 4, n_mols + kOrderExtra}; }

int64_t prepare_batch_ints(int64_t n, int64_t n_mols)
{
    int64_t total = up4(api.khan_prepare_batch_workspace_bytes(n) / 4);
    for (const int64_t s : prepared_sizes(n, n_mols)) total += up4(s);
    return total;
}

std::vector<Tensor> prepare_batch_into(const Tensor& mol_idxs, const Tensor& types, int64_t n_mols, const c10::optional<Tensor>& counts_pinned,
                                       const Tensor& all)
{
    const int64_t n = types.numel();
    std::vector<Tensor> out;
    int64_t at = up4(api.khan_prepare_batch_workspace_bytes(n) / 4);
    for (const int64_t s : prepared_sizes(n, n_mols)) {
        out.push_back(all.narrow(0, at, s));
        at += up4(s);
    }
    const khan_stream_t st = stream();
    int32_t* host = nullptr;
    if (counts_pinned) {
        const Tensor& h = *counts_pinned;
        if (h.scalar_type() != at::kInt || h.numel() != 8 || !h.is_contiguous() || !h.is_pinned())
            raise(PyExc_ValueError, "counts_pinned must hold 8 int32 in pinned memory");
        host = h.data_ptr<int32_t>();
        std::fill_n(host, 8, n_mols == 0 ? 0 : -1);               // -1: not written yet (wait_for_counts)
        // the GPU writes to it: not to be handed out again before this work is done, whoever drops the tensor
        at::getHostAllocator(at::kCUDA)->record_event(h.data_ptr(), h.storage().data_ptr().get_context(),
                                                      c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().unwrap());
    }
    call(api.khan_prepare_batch, ptr<const int32_t>(mol_idxs), ptr<const int32_t>(types), n, static_cast<int32_t>(n_mols),
         ptr<int32_t>(out[0]), ptr<int32_t>(out[1]), ptr<int32_t>(out[2]), ptr<int32_t>(out[3]), ptr<int32_t>(out[4]),
         ptr<int32_t>(out[5]), static_cast<void*>(all.data_ptr()), host, st);
    return out;
}

// The counts that prepare_batch writes to pinned memory (a list of the atom counts, a tensor of the class totals), or None if
// they have not arrived within about a millisecond.  They are on the host while the kernel that wrote them still ranks atoms,
// some microseconds before an event behind it.
static py::object wait_for_counts(const Tensor& counts_pinned)
{
    same_size(counts_pinned.scalar_type() == at::kInt && counts_pinned.numel() == 8 && counts_pinned.is_contiguous() && !counts_pinned.is_cuda(),
              "counts_pinned must hold 8 int32 in host memory");
    const volatile int32_t* c = counts_pinned.data_ptr<int32_t>();
    const auto arrived = [&] {
        for (int k = 0; k < 8; ++k)
            if (c[k] < 0) return false;
        return true;
    };
    {
        py::gil_scoped_release release;
        for (int spin = 0; spin < 20000 && !arrived(); ++spin) __builtin_ia32_pause();
    }
    if (!arrived()) return py::none();
    py::list acs(4);
    const Tensor classes = at::empty({4}, at::kInt);
    for (int k = 0; k < 4; ++k) {
        PyList_SET_ITEM(acs.ptr(), k, PyLong_FromLong(c[k]));
        classes.data_ptr<int32_t>()[k] = c[4 + k];
    }
    return py::make_tuple(acs, classes);
}

static std::vector<Tensor> prepare_batch(const Tensor& mol_idxs, const Tensor& types, int64_t n_mols, const c10::optional<Tensor>& counts_pinned)
{
    dev(mol_idxs, at::kInt, "mol_idxs");
    dev(types, at::kInt, "atomic_numbers");
    same_size(mol_idxs.numel() == types.numel(), "mol_idxs and atomic_numbers must have the same length");
    same_size(n_mols >= 0, "n_mols must not be negative");
    return prepare_batch_into(mol_idxs, types, n_mols, counts_pinned, at::empty({prepare_batch_ints(types.numel(), n_mols)}, types.options()));
}

// ---------------------------------------------------------------------------------------------- AEV passes
struct Atoms {
    at::ScalarType dt;
    int64_t n;
    Counts acs;
    const int32_t* order = nullptr;
    bool ordered = false, classes_known = false;
    Counts classes{};
    const int32_t* classes_ptr() const { return classes_known ? classes.v : nullptr; }
};

AevArgs aev_args(const py::object& acs, const c10::optional<Tensor>& order, const py::object& size_classes)
{
    AevArgs a{counts4(acs, "acs must hold 4 atom counts"), order, c10::nullopt};
    if (!size_classes.is_none()) a.classes = counts4(size_classes, "size_classes must hold 4 counts");
    return a;
}

Atoms check_atoms(const Atoms7& in, const AevArgs& args)
{
    const Tensor &xs = in[0], &ys = in[1], &zs = in[2], &as = in[3], &mos = in[4], &macs = in[5], &sis = in[6];
    Atoms a;
    a.dt = float_dtype(xs, "coordinates");
    dev(xs, a.dt, "xs"); dev(ys, a.dt, "ys"); dev(zs, a.dt, "zs");
    dev(as, at::kInt, "as"); dev(mos, at::kInt, "mos"); dev(macs, at::kInt, "macs"); dev(sis, at::kInt, "sis");
    a.n = xs.numel();
    same_size(ys.numel() == a.n && zs.numel() == a.n && as.numel() == a.n && sis.numel() == a.n, "xs, ys, zs, as, sis must have the same length");
    same_size(mos.numel() == macs.numel(), "mos and macs must have the same length");
    a.acs = args.acs;
    if (a.acs.sum() != a.n)
        raise(PyExc_ValueError, "sum(acs)=" + std::to_string(a.acs.sum()) + " does not match the number of atoms " + std::to_string(a.n));
    if (args.order) {
        dev(*args.order, at::kInt, "order");
        same_size(args.order->numel() == macs.numel() + kOrderExtra, "order must come from size_order(macs) of this batch");
        a.order = ptr<const int32_t>(*args.order);
        a.ordered = true;
        if (args.classes) {
            a.classes = *args.classes;
            a.classes_known = true;
        }
    }
    return a;
}

// four consecutive slices of one array, acs[t] * 384 elements each
std::vector<Tensor> buckets(const Tensor& packed, const Counts& acs, int64_t width)
{
    std::vector<Tensor> out;
    int64_t at = 0;
    for (const int32_t c : acs.v) {
        out.push_back(packed.narrow(0, at, c * width));
        at += c * width;
    }
    return out;
}

template <typename T, typename Plain, typename Ordered>
void run_forward(Plain plain, Ordered ordered, const Atoms& a, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as,
                 const Tensor& mos, const Tensor& macs, const Tensor& sis, const std::vector<Tensor>& o)
{
    const khan_stream_t st = stream();
    const int32_t m = static_cast<int32_t>(mos.numel());
    if (a.ordered)
        call(ordered, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<T>(o[0]), ptr<T>(o[1]), ptr<T>(o[2]), ptr<T>(o[3]), a.acs.v, a.order, a.classes_ptr(), st);
    else
        call(plain, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<T>(o[0]), ptr<T>(o[1]), ptr<T>(o[2]), ptr<T>(o[3]), a.acs.v, st);
}

std::vector<Tensor> run_featurize(const Atoms7& in, const AevArgs& args)
{
    const Atoms a = check_atoms(in, args);
    auto out = buckets(at::empty({a.n * kFeats}, in[0].options()), a.acs, kFeats);
    const auto& [xs, ys, zs, as, mos, macs, sis] = in;
    if (a.dt == at::kFloat) run_forward<float>(api.khan_featurize_f32, api.khan_featurize_ordered_f32, a, xs, ys, zs, as, mos, macs, sis, out);
    else run_forward<double>(api.khan_featurize_f64, api.khan_featurize_ordered_f64, a, xs, ys, zs, as, mos, macs, sis, out);
    return out;
}

static std::vector<Tensor> featurize(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos, const Tensor& macs,
                                     const Tensor& sis, const py::object& acs, const c10::optional<Tensor>& order, const py::object& size_classes)
{
    return run_featurize({xs, ys, zs, as, mos, macs, sis}, aev_args(acs, order, size_classes));
}

template <typename T, typename Plain, typename Ordered>
void run_backward(Plain plain, Ordered ordered, const Atoms& a, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as,
                  const Tensor& mos, const Tensor& macs, const Tensor& sis, const std::array<Tensor, 4>& g, const std::vector<Tensor>& o)
{
    const khan_stream_t st = stream();
    const int32_t m = static_cast<int32_t>(mos.numel());
    if (a.ordered)
        call(ordered, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<const T>(g[0]), ptr<const T>(g[1]), ptr<const T>(g[2]), ptr<const T>(g[3]), ptr<T>(o[0]), ptr<T>(o[1]),
             ptr<T>(o[2]), a.acs.v, a.order, a.classes_ptr(), st);
    else
        call(plain, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<const T>(g[0]), ptr<const T>(g[1]), ptr<const T>(g[2]), ptr<const T>(g[3]), ptr<T>(o[0]), ptr<T>(o[1]),
             ptr<T>(o[2]), a.acs.v, st);
}

std::vector<Tensor> run_featurize_grad(const Atoms7& in, const AevArgs& args, const Four& upstream, std::vector<Tensor> out)
{
    const Atoms a = check_atoms(in, args);
    static const char* const names[4] = {"h_grads", "c_grads", "n_grads", "o_grads"};
    Four g;
    for (int t = 0; t < 4; ++t) {
        g[t] = upstream[t].reshape({-1});
        dev(g[t], a.dt, names[t]);
        if (g[t].numel() != a.acs.v[t] * kFeats)
            raise(PyExc_ValueError, std::string(names[t]) + " has " + std::to_string(g[t].numel()) + " elements, expected " +
                                  std::to_string(a.acs.v[t] * kFeats));
    }
    const auto& [xs, ys, zs, as, mos, macs, sis] = in;
    if (out.empty()) out = {at::empty({a.n}, xs.options()), at::empty({a.n}, xs.options()), at::empty({a.n}, xs.options())};
    if (a.dt == at::kFloat)
        run_backward<float>(api.khan_featurize_grad_f32, api.khan_featurize_grad_ordered_f32, a, xs, ys, zs, as, mos, macs, sis, g, out);
    else
        run_backward<double>(api.khan_featurize_grad_f64, api.khan_featurize_grad_ordered_f64, a, xs, ys, zs, as, mos, macs, sis, g, out);
    return out;
}

static std::vector<Tensor> featurize_grad(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos,
                                          const Tensor& macs, const Tensor& sis, const py::object& acs, const Tensor& h, const Tensor& c,
                                          const Tensor& n, const Tensor& o, const c10::optional<Tensor>& order, const py::object& size_classes)
{
    return run_featurize_grad({xs, ys, zs, as, mos, macs, sis}, aev_args(acs, order, size_classes), {h, c, n, o});
}

template <typename T, typename Plain, typename Ordered>
void run_inverse(Plain plain, Ordered ordered, const Atoms& a, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as,
                 const Tensor& mos, const Tensor& macs, const Tensor& sis, const Tensor& vx, const Tensor& vy, const Tensor& vz,
                 const std::vector<Tensor>& o)
{
    const khan_stream_t st = stream();
    const int32_t m = static_cast<int32_t>(mos.numel());
    if (a.ordered)
        call(ordered, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<const T>(vx), ptr<const T>(vy), ptr<const T>(vz), ptr<T>(o[0]), ptr<T>(o[1]), ptr<T>(o[2]), ptr<T>(o[3]),
             a.acs.v, a.order, a.classes_ptr(), st);
    else
        call(plain, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const int32_t>(as), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             m, ptr<const int32_t>(sis), ptr<const T>(vx), ptr<const T>(vy), ptr<const T>(vz), ptr<T>(o[0]), ptr<T>(o[1]), ptr<T>(o[2]), ptr<T>(o[3]),
             a.acs.v, st);
}

std::vector<Tensor> run_featurize_grad_inverse(const Atoms7& in, const AevArgs& args, const std::array<Tensor, 3>& v)
{
    const Atoms a = check_atoms(in, args);
    dev(v[0], a.dt, "x_grads"); dev(v[1], a.dt, "y_grads"); dev(v[2], a.dt, "z_grads");
    same_size(v[0].numel() == a.n && v[1].numel() == a.n && v[2].numel() == a.n, "x_grads, y_grads, z_grads must have one element per atom");
    auto out = buckets(at::empty({a.n * kFeats}, in[0].options()), a.acs, kFeats);
    const auto& [xs, ys, zs, as, mos, macs, sis] = in;
    if (a.dt == at::kFloat)
        run_inverse<float>(api.khan_featurize_grad_inverse_f32, api.khan_featurize_grad_inverse_ordered_f32, a, xs, ys, zs, as, mos, macs, sis, v[0],
                           v[1], v[2], out);
    else
        run_inverse<double>(api.khan_featurize_grad_inverse_f64, api.khan_featurize_grad_inverse_ordered_f64, a, xs, ys, zs, as, mos, macs, sis, v[0],
                            v[1], v[2], out);
    return out;
}

static std::vector<Tensor> featurize_grad_inverse(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos,
                                                  const Tensor& macs, const Tensor& sis, const py::object& acs, const Tensor& vx, const Tensor& vy,
                                                  const Tensor& vz, const c10::optional<Tensor>& order, const py::object& size_classes)
{
    return run_featurize_grad_inverse({xs, ys, zs, as, mos, macs, sis}, aev_args(acs, order, size_classes), {vx, vy, vz});
}

// ---------------------------------------------------------------------------------------------- charges
at::ScalarType check_charge(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs)
{
    const auto dt = float_dtype(xs, "coordinates");
    dev(xs, dt, "xs"); dev(ys, dt, "ys"); dev(zs, dt, "zs"); dev(qs, dt, "qs");
    dev(mos, at::kInt, "mos"); dev(macs, at::kInt, "macs");
    const int64_t n = xs.numel();
    same_size(ys.numel() == n && zs.numel() == n && qs.numel() == n, "xs, ys, zs, qs must have the same length");
    same_size(mos.numel() == macs.numel(), "mos and macs must have the same length");
    return dt;
}

Tensor ani_charge(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs)
{
    const auto dt = check_charge(xs, ys, zs, qs, mos, macs);
    const Tensor e = at::empty({mos.numel()}, xs.options());
    const khan_stream_t st = stream();
    auto run = [&](auto zero, auto fn) {
        using T = decltype(zero);
        call(fn, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const T>(qs), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             static_cast<int32_t>(mos.numel()), xs.numel(), static_cast<const T*>(nullptr), ptr<T>(e), static_cast<T*>(nullptr),
             static_cast<T*>(nullptr), static_cast<T*>(nullptr), static_cast<T*>(nullptr), 0, st);
    };
    if (dt == at::kFloat) run(0.0f, api.khan_ani_charges_f32);
    else run(0.0, api.khan_ani_charges_f64);
    return e;
}

// Gradients (and with `energies` the energies) of the damped charge energy.  One allocation cut into the outputs, zeroed by the
// launch that orders the molecules: atoms outside every molecule keep zeros.
std::vector<Tensor> ani_charge_grads(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs,
                                     const Tensor& grads, bool want_xyz, bool energies)
{
    const auto dt = check_charge(xs, ys, zs, qs, mos, macs);
    dev(grads, dt, "grads");
    same_size(grads.numel() == mos.numel(), "grads must have one element per molecule");
    const int64_t n = xs.numel(), m = mos.numel();
    const Tensor all = at::empty({n * (want_xyz ? 4 : 1) + (energies ? m : 0)}, xs.options());
    const Tensor order = m > 256 && n > 32 * m ? at::empty({m}, mos.options()) : Tensor();      // (elsewhere it would not be used)
    std::vector<Tensor> out;
    int64_t at = 0;
    auto take = [&](int64_t size) {
        out.push_back(all.narrow(0, at, size));
        at += size;
    };
    if (energies) take(m);
    for (int k = 0; k < (want_xyz ? 4 : 1); ++k) take(n);
    const khan_stream_t st = stream();
    auto run = [&](auto zero, auto fn) {
        using T = decltype(zero);
        const int q = energies ? 1 : 0;
        T* none = nullptr;
        call(fn, ptr<const T>(xs), ptr<const T>(ys), ptr<const T>(zs), ptr<const T>(qs), ptr<const int32_t>(mos), ptr<const int32_t>(macs),
             static_cast<int32_t>(m), n, ptr<const T>(grads), energies ? ptr<T>(out[0]) : none, ptr<T>(out[q]), want_xyz ? ptr<T>(out[q + 1]) : none,
             want_xyz ? ptr<T>(out[q + 2]) : none, want_xyz ? ptr<T>(out[q + 3]) : none, ptr<T>(all), all.numel(), order.defined() ? ptr<int32_t>(order) : nullptr, st);
    };
    if (dt == at::kFloat) run(0.0f, api.khan_ani_charges_begun_f32);
    else run(0.0, api.khan_ani_charges_begun_f64);
    return out;
}

// ---------------------------------------------------------------------------------------------- networks
Tensor run_mol_energy(const Four& type_outputs, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs, Tensor e)
{
    const auto dt = float_dtype(type_outputs[0], "type_outputs");
    Four o;
    int64_t n = 0;
    for (int t = 0; t < 4; ++t) {
        o[t] = type_outputs[t].reshape({-1});
        dev(o[t], dt, "type_outputs");
        n += o[t].numel();
    }
    dev(types, at::kInt, "atom_types"); dev(sis, at::kInt, "sis"); dev(mos, at::kInt, "mos"); dev(macs, at::kInt, "macs");
    same_size(n == types.numel() && sis.numel() == n && mos.numel() == macs.numel(),
              "the four vectors must hold one value per atom, and mos / macs one entry per molecule");
    if (!e.defined()) e = at::empty({macs.numel()}, o[0].options());
    const int32_t m = static_cast<int32_t>(macs.numel());
    const khan_stream_t st = stream();
    auto run = [&](auto zero, auto fn) {
        using T = decltype(zero);
        const T* p[4] = {ptr<const T>(o[0]), ptr<const T>(o[1]), ptr<const T>(o[2]), ptr<const T>(o[3])};
        call(fn, p, ptr<const int32_t>(types), ptr<const int32_t>(sis), ptr<const int32_t>(mos), ptr<const int32_t>(macs), m, ptr<T>(e), st);
    };
    if (dt == at::kFloat) run(0.0f, api.khan_mol_energy_f32);
    else run(0.0, api.khan_mol_energy_f64);
    return e;
}

static Tensor mol_energy(const std::vector<Tensor>& type_outputs, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs)
{
    same_size(type_outputs.size() == 4, "type_outputs must hold the four per-type vectors");
    return run_mol_energy({type_outputs[0], type_outputs[1], type_outputs[2], type_outputs[3]}, types, sis, mos, macs);
}

std::vector<Tensor> run_mol_energy_grad(const Tensor& e_grads, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs,
                                        const Counts& c)
{
    const auto dt = float_dtype(e_grads, "e_grads");
    dev(e_grads, dt, "e_grads");
    dev(types, at::kInt, "atom_types"); dev(sis, at::kInt, "sis"); dev(mos, at::kInt, "mos"); dev(macs, at::kInt, "macs");
    same_size(c.sum() == types.numel() && sis.numel() == types.numel() && mos.numel() == macs.numel() && e_grads.numel() == macs.numel(),
              "acs must add up to the number of atoms, and e_grads / mos / macs hold one entry per molecule");
    // one cleared array cut into the four vectors (atoms outside every molecule keep 0)
    auto out = buckets(at::zeros({c.sum()}, e_grads.options()), c, 1);
    const int32_t m = static_cast<int32_t>(macs.numel());
    const khan_stream_t st = stream();
    auto run = [&](auto zero, auto fn) {
        using T = decltype(zero);
        T* p[4] = {ptr<T>(out[0]), ptr<T>(out[1]), ptr<T>(out[2]), ptr<T>(out[3])};
        call(fn, ptr<const T>(e_grads), ptr<const int32_t>(types), ptr<const int32_t>(sis), ptr<const int32_t>(mos), ptr<const int32_t>(macs), m, p, st);
    };
    if (dt == at::kFloat) run(0.0f, api.khan_mol_energy_grad_f32);
    else run(0.0, api.khan_mol_energy_grad_f64);
    return out;
}

static std::vector<Tensor> mol_energy_grad(const Tensor& e_grads, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs,
                                           const py::object& acs)
{
    return run_mol_energy_grad(e_grads, types, sis, mos, macs, counts4(acs, "acs must hold 4 atom counts"));
}

}  // namespace khan_torch

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    using namespace khan_torch;
    m.def("init", &init);
    m.def("prepare_batch", &prepare_batch);
    m.def("wait_for_counts", &wait_for_counts);
    m.def("featurize", &featurize);
    m.def("featurize_grad", &featurize_grad);
    m.def("featurize_grad_inverse", &featurize_grad_inverse);
    m.def("ani_charge", &ani_charge);
    m.def("ani_charge_grads", &ani_charge_grads);
    m.def("mol_energy", &mol_energy);
    m.def("mol_energy_grad", &mol_energy_grad);
    bind_autograd(m);
    bind_feed(m);
}
