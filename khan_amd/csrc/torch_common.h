// What the native tensor layer's translation units share: the opened library's entry points, argument checks, the call.
#pragma once
#include <array>
#include <string>
#include <vector>

#include <ATen/hip/CachingHostAllocator.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../include/khan_aev.h"

namespace khan_torch {

namespace py = pybind11;
using at::Tensor;
using Four = std::array<Tensor, 4>;

#define KHAN_API(X)                                                                                                    \
    X(khan_status_string) X(khan_last_hip_error) X(khan_mol_offsets) X(khan_ani_sort) X(khan_size_order)               \
    X(khan_prepare_batch_workspace_bytes) X(khan_prepare_batch)                                                        \
    X(khan_featurize_f32) X(khan_featurize_f64) X(khan_featurize_ordered_f32) X(khan_featurize_ordered_f64)            \
    X(khan_featurize_grad_f32) X(khan_featurize_grad_f64) X(khan_featurize_grad_ordered_f32)                           \
    X(khan_featurize_grad_ordered_f64) X(khan_featurize_grad_inverse_f32) X(khan_featurize_grad_inverse_f64)           \
    X(khan_featurize_grad_inverse_ordered_f32) X(khan_featurize_grad_inverse_ordered_f64)                              \
    X(khan_ani_charges_f32) X(khan_ani_charges_f64) X(khan_ani_charges_begun_f32) X(khan_ani_charges_begun_f64)         \
    X(khan_mol_energy_f32) X(khan_mol_energy_f64) X(khan_mol_energy_grad_f32)               \
    X(khan_mol_energy_grad_f64) X(khan_net_layer_f32) X(khan_net_layer_f64) X(khan_net_top_f32) X(khan_net_top_f64)      \
    X(khan_net_grads_workspace_bytes_f32) X(khan_net_grads_workspace_bytes_f64) X(khan_net_grads_f32) X(khan_net_grads_f64) \
    X(khan_net_few_fits) X(khan_net_few_f64) X(khan_net_chain_fits) X(khan_net_chain_workspace_bytes)                  \
    X(khan_take_rows_f32) X(khan_take_rows_f64) X(khan_put_rows_f32) X(khan_put_rows_f64) X(khan_add_two_f32) X(khan_add_two_f64)   \
    X(khan_net_chain_values_f32) X(khan_net_chain_rows_f32)                                                            \
    X(khan_atomic_networks_f32) X(khan_atomic_networks_packed_bytes) X(khan_atomic_networks_pack_stored_f32)

struct Api {
#define X(name) decltype(&::name) name = nullptr;
    KHAN_API(X)
#undef X
};
extern Api api;
extern PyObject* khan_error;

// A Python exception of that type; in a thread of the autograd engine (which does not hold the interpreter's lock) in the form
// that the engine carries over to the thread that asked for the gradients.
[[noreturn]] void raise(PyObject* type, const std::string& message);

inline void check(int status)
{
    if (status == KHAN_OK) return;
    const std::string detail = api.khan_last_hip_error();
    raise(khan_error, std::string("libkhan_aev: ") + api.khan_status_string(status) + (detail.empty() ? "" : " (" + detail + ")"));
}

// the launch, with the interpreter's lock (where this thread holds it) given back as a foreign-function call gives it back
template <typename Fn, typename... Args>
void call(Fn fn, Args... args)
{
    int status;
    if (PyGILState_Check()) {
        py::gil_scoped_release release;
        status = fn(args...);
    } else {
        status = fn(args...);
    }
    check(status);
}

inline khan_stream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

inline void dev(const Tensor& t, at::ScalarType dtype, const char* name)
{
    if (!t.is_cuda()) raise(PyExc_TypeError, std::string(name) + " must be a CUDA tensor");
    if (t.scalar_type() != dtype)
        raise(PyExc_TypeError, std::string(name) + " must have dtype " + c10::toString(dtype) + ", got " + c10::toString(t.scalar_type()));
    if (t.dim() != 1) raise(PyExc_ValueError, std::string(name) + " must be rank 1 (flat), got rank " + std::to_string(t.dim()));
    if (!t.is_contiguous()) raise(PyExc_ValueError, std::string(name) + " must be contiguous");
}

inline void same_size(bool ok, const char* what)
{
    if (!ok) raise(PyExc_ValueError, what);
}

template <typename T>
T* ptr(const Tensor& t)
{
    return t.defined() && t.numel() > 0 ? static_cast<T*>(t.data_ptr()) : nullptr;
}

inline at::ScalarType float_dtype(const Tensor& x, const char* what)
{
    const auto dt = x.scalar_type();
    if (dt != at::kFloat && dt != at::kDouble) raise(PyExc_TypeError, std::string(what) + " must be float32 or float64, got " + c10::toString(dt));
    return dt;
}

struct Counts {
    int32_t v[4];
    int64_t sum() const { return static_cast<int64_t>(v[0]) + v[1] + v[2] + v[3]; }
};

constexpr int64_t kFeats = 384;
constexpr int64_t kOrderExtra = 520;

// What the AEV passes take besides their tensors: the four atom counts, and of the size order the four class totals
struct AevArgs {
    Counts acs;
    c10::optional<Tensor> order;
    c10::optional<Counts> classes;
};
using Atoms7 = std::array<Tensor, 7>;      // xs, ys, zs, as, mos, macs, sis

std::vector<Tensor> run_featurize(const Atoms7& in, const AevArgs& args);
// (`out`: three vectors to write to, otherwise new ones)
std::vector<Tensor> run_featurize_grad(const Atoms7& in, const AevArgs& args, const Four& upstream, std::vector<Tensor> out = {});
std::vector<Tensor> run_featurize_grad_inverse(const Atoms7& in, const AevArgs& args, const std::array<Tensor, 3>& v);
Tensor ani_charge(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs);
std::vector<Tensor> ani_charge_grads(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs,
                                     const Tensor& grads, bool want_xyz, bool energies);
Tensor run_mol_energy(const Four& type_outputs, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs,
                      Tensor out = Tensor());
std::vector<Tensor> run_mol_energy_grad(const Tensor& e_grads, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs,
                                        const Counts& acs);
Counts counts4(const py::object& o, const char* what);
AevArgs aev_args(const py::object& acs, const c10::optional<Tensor>& order, const py::object& size_classes);
std::vector<Tensor> buckets(const Tensor& packed, const Counts& acs, int64_t width);
int64_t prepare_batch_ints(int64_t n, int64_t n_mols);          // int32 elements prepare_batch_into takes for its results and workspace
std::vector<Tensor> prepare_batch_into(const Tensor& mol_idxs, const Tensor& types, int64_t n_mols, const c10::optional<Tensor>& counts_pinned,
                                       const Tensor& all);
void bind_autograd(py::module_& m);
void bind_feed(py::module_& m);

}  // namespace khan_torch
