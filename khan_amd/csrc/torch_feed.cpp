// The host side of feeding a data set: molecules held as numpy arrays -> one pinned buffer -> one buffer on the GPU that holds
// a batch's arrays and everything its preparation makes (khan/data/dataset.py:118-183, trainer_multi_tower.py:767-792).
// What bounds it is the interpreter and cache misses: concatenating, splitting and casting a batch of 1,024 molecules in
// numpy, five copies, twelve tensors to tell the allocator about and the wait for the counts of the sort took more than
// the GPU's work on the batch.  Here a molecule costs one visit, and the counts are made on the way.
#include <pybind11/numpy.h>

#include <c10/core/StreamGuard.h>

#include "torch_common.h"

namespace khan_torch {

namespace {

constexpr int64_t kPad = 64;          // elements; keeps every array of the buffer on a 256-byte boundary

int64_t padded(int64_t n) { return (n + kPad - 1) / kPad * kPad; }

// The buffer: xs, ys, zs (padded), atom types, molecule indices
struct Staged {
    int64_t n, at;
    size_t w;
    Staged(int64_t n_, bool f64) : n(n_), at(padded(n_)), w(f64 ? 8 : 4) {}
    int64_t bytes() const { return at * static_cast<int64_t>(3 * w + 8); }
    int64_t coord(int k) const { return k * at * static_cast<int64_t>(w); }
    int64_t ints(int k) const { return at * static_cast<int64_t>(3 * w + 4 * k); }
};

// four atom counts and the molecules of up to 32, 64, 256 and more atoms, as the preparation on the GPU counts them
struct Totals {
    int32_t v[8] = {};
    void atom(int32_t type) { ++v[static_cast<uint32_t>(type) > 3u ? 3 : type]; }
    void molecule(int64_t atoms) { ++v[4 + (atoms > 32) + (atoms > 64) + (atoms > 256)]; }
    py::tuple pair() const { return py::make_tuple(py::make_tuple(v[0], v[1], v[2], v[3]), py::make_tuple(v[4], v[5], v[6], v[7])); }
};

struct Rows4 {
    const double* row;
    int64_t n;
};

template <typename T>
void fill(const std::vector<Rows4>& mols, const Staged& s, char* base, Totals& totals)
{
    T *x = reinterpret_cast<T*>(base + s.coord(0)), *y = reinterpret_cast<T*>(base + s.coord(1)), *z = reinterpret_cast<T*>(base + s.coord(2));
    int32_t *types = reinterpret_cast<int32_t*>(base + s.ints(0)), *ids = reinterpret_cast<int32_t*>(base + s.ints(1));
    int64_t at = 0;
    for (size_t m = 0; m < mols.size(); ++m) {
        // every molecule is an allocation of its own: fetch the ones to come
        if (m + 4 < mols.size())
            for (int64_t b = 0; b < 4 * mols[m + 4].n && b < 128; b += 8) __builtin_prefetch(mols[m + 4].row + b);
        const double* r = mols[m].row;
        for (int64_t i = 0; i < mols[m].n; ++i, ++at, r += 4) {
            const int32_t t = static_cast<int32_t>(r[0]);
            types[at] = t;
            totals.atom(t);
            x[at] = static_cast<T>(r[1]);
            y[at] = static_cast<T>(r[2]);
            z[at] = static_cast<T>(r[3]);
            ids[at] = static_cast<int32_t>(m);
        }
        totals.molecule(mols[m].n);
    }
}

void check_staging(const Tensor& staging)
{
    same_size(staging.scalar_type() == at::kByte && staging.is_contiguous() && !staging.is_cuda(), "staging must be a byte array on the host");
}

// The molecules `sel` of a list of arrays -> staging: (atoms, molecule sizes, totals); the bytes needed where staging is too
// small; None where a molecule is not a contiguous float64 array of (type, x, y, z) rows (the caller converts those itself).
py::object stage_molecules(const py::object& list, const py::array_t<int64_t>& sel, const Tensor& staging, bool f64)
{
    check_staging(staging);
    if (!PyList_Check(list.ptr())) return py::none();
    const py::list arrays = py::reinterpret_borrow<py::list>(list);
    const auto& api = py::detail::npy_api::get();
    static PyObject* const f64_type = py::dtype::of<double>().release().ptr();
    const int64_t *ids = sel.data(), count = sel.size(), have = static_cast<int64_t>(arrays.size());
    std::vector<Rows4> mols(static_cast<size_t>(count));
    int64_t n = 0;
    for (int64_t k = 0; k < count; ++k) {
        if (ids[k] < 0 || ids[k] >= have) throw py::index_error("molecule index out of range");
        PyObject* o = PyList_GET_ITEM(arrays.ptr(), ids[k]);
        if (!api.PyArray_Check_(o)) return py::none();
        const auto* a = py::detail::array_proxy(o);
        if (a->descr != f64_type || a->nd != 2 || a->dimensions[1] != 4 ||
            !(a->flags & py::detail::npy_api::NPY_ARRAY_C_CONTIGUOUS_) || !(a->flags & py::detail::npy_api::NPY_ARRAY_ALIGNED_))
            return py::none();
        mols[k] = {reinterpret_cast<const double*>(a->data), a->dimensions[0]};
        n += mols[k].n;
    }
    const Staged s(n, f64);
    if (staging.numel() < s.bytes()) return py::int_(s.bytes());
    py::list sizes(static_cast<size_t>(count));
    for (int64_t k = 0; k < count; ++k) PyList_SET_ITEM(sizes.ptr(), k, PyLong_FromLongLong(mols[k].n));
    Totals totals;
    char* base = static_cast<char*>(staging.data_ptr());
    if (f64) fill<double>(mols, s, base, totals);
    else fill<float>(mols, s, base, totals);
    return py::make_tuple(n, sizes, totals.pair());
}

// The totals of a batch that is in staging already; offsets: the molecules' positions in it
py::tuple staged_totals(const Tensor& staging, int64_t n, const py::array_t<int64_t>& offsets, bool f64)
{
    check_staging(staging);
    const Staged s(n, f64);
    same_size(staging.numel() >= s.bytes(), "staging is too small");
    const int32_t* types = reinterpret_cast<const int32_t*>(static_cast<const char*>(staging.data_ptr()) + s.ints(0));
    Totals totals;
    for (int64_t i = 0; i < n; ++i) totals.atom(types[i]);
    for (int64_t m = 0; m + 1 < offsets.size(); ++m) totals.molecule(offsets.data()[m + 1] - offsets.data()[m]);
    return totals.pair();
}

// [values[k] for k in sel] of a list (the interpreter's loop over 4,096 molecules is 60 us of a pass over the data set, 1,840 us for two)
py::list picked(const py::list& values, const py::array_t<int64_t>& sel)
{
    const int64_t count = sel.size();
    py::list out(static_cast<size_t>(count));
    for (int64_t k = 0; k < count; ++k) {
        const int64_t id = sel.data()[k];
        if (id < 0 || id >= PyList_GET_SIZE(values.ptr())) throw py::index_error("molecule index out of range");
        PyObject* o = PyList_GET_ITEM(values.ptr(), id);
        Py_INCREF(o);
        PyList_SET_ITEM(out.ptr(), k, o);
    }
    return out;
}

int64_t staging_bytes(int64_t n, bool f64) { return Staged(n, f64).bytes(); }

// The staging area's parts as host tensors: xs, ys, zs, types, molecule indices
std::vector<Tensor> staging_parts(const Tensor& staging, int64_t n, bool f64)
{
    const Staged s(n, f64);
    const auto dt = f64 ? at::kDouble : at::kFloat;
    const auto part = [&](int64_t from, size_t w, at::ScalarType t) { return staging.narrow(0, from, n * static_cast<int64_t>(w)).view(t); };
    return {part(s.coord(0), s.w, dt), part(s.coord(1), s.w, dt), part(s.coord(2), s.w, dt), part(s.ints(0), 4, at::kInt), part(s.ints(1), 4, at::kInt)};
}

// Staging -> GPU in one copy on a stream (its id, device and device type), and the batch's preparation behind it
// -> (the buffer, xs, ys, zs, types, molecule indices, and what prepare_batch returns), all of them parts of the buffer
std::vector<Tensor> feed_batch(const Tensor& staging, int64_t n, int64_t n_mols, bool f64, const at::Device& device, const c10::optional<Tensor>& counts_pinned,
                               const std::tuple<int64_t, int64_t, int64_t>& on)
{
    const c10::StreamGuard guard(c10::Stream::unpack3(std::get<0>(on), static_cast<c10::DeviceIndex>(std::get<1>(on)),
                                                      static_cast<c10::DeviceType>(std::get<2>(on))));
    check_staging(staging);
    const Staged s(n, f64);
    same_size(staging.numel() >= s.bytes(), "staging is too small");
    const int64_t ints = s.bytes() / 4;
    const Tensor all = at::empty({ints + prepare_batch_ints(n, n_mols)}, at::TensorOptions().device(device).dtype(at::kInt));
    if (n > 0) all.narrow(0, 0, ints).copy_(staging.narrow(0, 0, s.bytes()).view(at::kInt), true);
    std::vector<Tensor> out = {all};
    // tensors of their own on the buffer's memory: what is written to one in place is no change of the others
    const auto part = [&](int64_t from, at::ScalarType t) {
        return at::empty({0}, all.options().dtype(t)).set_(all.storage(), from / static_cast<int64_t>(c10::elementSize(t)), {n}, {1});
    };
    for (int k = 0; k < 3; ++k) out.push_back(part(s.coord(k), f64 ? at::kDouble : at::kFloat));
    for (int k = 0; k < 2; ++k) out.push_back(part(s.ints(k), at::kInt));
    for (const Tensor& part : prepare_batch_into(out[5], out[4], n_mols, counts_pinned, all.narrow(0, ints, all.numel() - ints))) out.push_back(part);
    return out;
}

// (x, y, z) [3, atoms] -> the molecules' [atoms, 3] arrays, views of one
py::list molecule_rows(const py::array& planes, const py::list& sizes)
{
    const auto& api = py::detail::npy_api::get();
    const auto* p = py::detail::array_proxy(planes.ptr());
    same_size(p->nd == 2 && p->dimensions[0] == 3 && (p->flags & py::detail::npy_api::NPY_ARRAY_C_CONTIGUOUS_), "an array of three rows");
    const py::ssize_t n = p->dimensions[1], w = planes.itemsize();
    const py::array rows(planes.dtype(), std::vector<py::ssize_t>{n, 3});
    const auto transpose = [&](auto zero) {
        using T = decltype(zero);
        const T* from = reinterpret_cast<const T*>(p->data);
        T* to = static_cast<T*>(const_cast<void*>(rows.data()));
        for (py::ssize_t i = 0; i < n; ++i)
            for (int k = 0; k < 3; ++k) to[3 * i + k] = from[k * n + i];
    };
    same_size(w == 4 || w == 8, "single or double precision");
    if (w == 4) transpose(float());
    else transpose(double());
    py::list out(sizes.size());
    auto* d = py::detail::array_proxy(rows.ptr());
    Py_intptr_t shape[2] = {0, 3}, strides[2] = {3 * w, w};
    char* at = d->data;
    py::ssize_t left = n;
    for (size_t k = 0; k < sizes.size(); ++k) {
        shape[0] = PyLong_AsLongLong(PyList_GET_ITEM(sizes.ptr(), k));
        same_size(shape[0] >= 0 && shape[0] <= left, "the sizes do not fit the array");
        Py_INCREF(d->descr);
        PyObject* v = api.PyArray_NewFromDescr_(api.PyArray_Type_, d->descr, 2, shape, strides, at, py::detail::npy_api::NPY_ARRAY_WRITEABLE_, nullptr);
        if (!v) throw py::error_already_set();
        PyList_SET_ITEM(out.ptr(), k, v);
        Py_INCREF(rows.ptr());
        if (api.PyArray_SetBaseObject_(v, rows.ptr()) != 0) throw py::error_already_set();
        at += shape[0] * strides[0];
        left -= shape[0];
    }
    return out;
}

}  // namespace

void bind_feed(py::module_& m)
{
    m.def("stage_molecules", &stage_molecules);
    m.def("picked", &picked);
    m.def("staged_totals", &staged_totals);
    m.def("staging_bytes", &staging_bytes);
    m.def("staging_parts", &staging_parts);
    m.def("feed_batch", &feed_batch);
    m.def("molecule_rows", &molecule_rows);
}

}  // namespace khan_torch
