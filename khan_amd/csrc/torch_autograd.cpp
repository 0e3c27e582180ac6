// torch.autograd functions of the path in native code: the AEV passes, the sums by molecule, the charge energy, and the
// per-type networks with CELU (khan/training/trainer_multi_tower.py:23-120 for the gradient wiring, khan/model/nn.py:38-68
// for the networks).  A training step on a thousand molecules spent most of its time between launches: Python functions on
// either side of every node, a library product per layer and type, a transposed copy of every weight.
#include <torch/csrc/autograd/custom_function.h>

#include "torch_common.h"

namespace khan_torch {

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::Variable;
using torch::autograd::variable_list;
using Saved = std::vector<int64_t>;
// Inside a node nothing is recorded: its few dozen views and allocations go past autograd's own dispatch, which costs as much
// again as the work itself (a training step on 1,024 molecules is bound by the host).
using Unrecorded = at::AutoDispatchBelowADInplaceOrView;

Tensor flat1(const Tensor& t) { return t.dim() == 1 ? t : t.reshape({-1}); }

// ---------------------------------------------------------------------------------------------- AEV passes
void keep(AutogradContext* ctx, const AevArgs& a)
{
    ctx->saved_data["acs"] = Saved(a.acs.v, a.acs.v + 4);
    if (a.classes) ctx->saved_data["classes"] = Saved(a.classes->v, a.classes->v + 4);
}

AevArgs kept(AutogradContext* ctx, const Variable& order)
{
    AevArgs a{};
    const auto acs = ctx->saved_data["acs"].toIntVector();
    for (int t = 0; t < 4; ++t) a.acs.v[t] = static_cast<int32_t>(acs[t]);
    if (order.defined()) a.order = order;
    if (ctx->saved_data.count("classes")) {
        const auto c = ctx->saved_data["classes"].toIntVector();
        a.classes = Counts{};
        for (int t = 0; t < 4; ++t) a.classes->v[t] = static_cast<int32_t>(c[t]);
    }
    return a;
}

Atoms7 atoms_of(const variable_list& v) { return {v[0].detach(), v[1].detach(), v[2].detach(), v[3], v[4], v[5], v[6]}; }

variable_list with_order(const Atoms7& in, const AevArgs& args)
{
    variable_list v(in.begin(), in.end());
    v.push_back(args.order ? *args.order : Tensor());
    return v;
}

struct FeaturizeGradFn : Function<FeaturizeGradFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos,
                                 const Tensor& macs, const Tensor& sis, const Tensor& h, const Tensor& c, const Tensor& n, const Tensor& o,
                                 const AevArgs& args)
    {
        const Atoms7 in = {xs, ys, zs, as, mos, macs, sis};
        ctx->save_for_backward(with_order(in, args));
        keep(ctx, args);
        const Unrecorded quiet;
        return run_featurize_grad(in, args, {h.contiguous(), c.contiguous(), n.contiguous(), o.contiguous()});
    }
    // d / d(upstream rows): the Jacobian applied to the incoming vectors; no second derivative by the coordinates, as in
    // the reference (trainer_multi_tower.py:64-91)
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto saved = ctx->get_saved_variables();
        std::array<Tensor, 3> v;
        for (int k = 0; k < 3; ++k) v[k] = g[k].defined() ? g[k].contiguous() : at::zeros_like(saved[0]);
        const auto d = run_featurize_grad_inverse(atoms_of(saved), kept(ctx, saved[7]), v);
        variable_list out(12);
        for (int t = 0; t < 4; ++t) out[7 + t] = d[t];
        return out;
    }
};

struct FeaturizeFn : Function<FeaturizeFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos,
                                 const Tensor& macs, const Tensor& sis, const AevArgs& args)
    {
        const Unrecorded quiet;
        const Atoms7 in = {xs, ys, zs, as, mos, macs, sis};
        ctx->save_for_backward(with_order(in, args));
        keep(ctx, args);
        return run_featurize(in, args);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto saved = ctx->get_saved_variables();
        const AevArgs args = kept(ctx, saved[7]);
        for (int t = 0; t < 4; ++t)
            if (!g[t].defined()) g[t] = at::zeros({args.acs.v[t] * kFeats}, saved[0].options());
        const Atoms7 in = atoms_of(saved);
        const auto d = FeaturizeGradFn::apply(in[0], in[1], in[2], in[3], in[4], in[5], in[6], g[0], g[1], g[2], g[3], args);
        variable_list out(8);
        for (int k = 0; k < 3; ++k) out[k] = d[k];
        return out;
    }
};

std::vector<Tensor> featurize_autograd(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos, const Tensor& macs,
                                       const Tensor& sis, const py::object& acs, const c10::optional<Tensor>& order, const py::object& size_classes)
{
    const AevArgs args = aev_args(acs, order, size_classes);
    return FeaturizeFn::apply(xs, ys, zs, as, mos, macs, sis, args);
}

struct AniChargeFn : Function<AniChargeFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos,
                          const Tensor& macs)
    {
        ctx->save_for_backward({xs, ys, zs, qs, mos, macs});
        return ani_charge(xs, ys, zs, qs, mos, macs);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        const bool xyz = ctx->needs_input_grad(0) || ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
        const auto d = ani_charge_grads(s[0].detach(), s[1].detach(), s[2].detach(), s[3].detach(), s[4], s[5], g[0].contiguous(), xyz, false);
        if (!xyz) return {Tensor(), Tensor(), Tensor(), d[0], Tensor(), Tensor()};
        return {d[1], d[2], d[3], d[0], Tensor(), Tensor()};
    }
};

Tensor ani_charge_autograd(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& qs, const Tensor& mos, const Tensor& macs)
{
    return AniChargeFn::apply(xs, ys, zs, qs, mos, macs);
}

// ---------------------------------------------------------------------------------------------- sums by molecule
// Both maps are linear and each is the other's transpose: the pair is differentiable to any order.
struct MolEnergyGradFn;
struct MolEnergyFn : Function<MolEnergyFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs, const Tensor& o0,
                          const Tensor& o1, const Tensor& o2, const Tensor& o3)
    {
        ctx->save_for_backward({types, sis, mos, macs});
        ctx->saved_data["counts"] = Saved{o0.numel(), o1.numel(), o2.numel(), o3.numel()};
        std::vector<Saved> shapes;
        for (const Tensor* o : {&o0, &o1, &o2, &o3}) shapes.push_back(o->sizes().vec());
        ctx->saved_data["shapes"] = shapes;
        const Unrecorded quiet;
        return run_mol_energy({o0, o1, o2, o3}, types, sis, mos, macs);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g);
};
struct MolEnergyGradFn : Function<MolEnergyGradFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs, Saved counts,
                                 const Tensor& ge)
    {
        ctx->save_for_backward({types, sis, mos, macs});
        ctx->saved_data["counts"] = counts;
        ctx->saved_data["double"] = ge.scalar_type() == at::kDouble;
        Counts c{};
        for (int t = 0; t < 4; ++t) c.v[t] = static_cast<int32_t>(counts[t]);
        const Unrecorded quiet;
        return run_mol_energy_grad(ge.contiguous(), types, sis, mos, macs, c);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        const auto counts = ctx->saved_data["counts"].toIntVector();
        const auto dt = ctx->saved_data["double"].toBool() ? at::kDouble : at::kFloat;
        for (int t = 0; t < 4; ++t)
            g[t] = g[t].defined() ? g[t].contiguous() : at::zeros({counts[t]}, s[0].options().dtype(dt));
        return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), MolEnergyFn::apply(s[0], s[1], s[2], s[3], g[0], g[1], g[2], g[3])};
    }
};
variable_list MolEnergyFn::backward(AutogradContext* ctx, variable_list g)
{
    const auto s = ctx->get_saved_variables();
    auto d = MolEnergyGradFn::apply(s[0], s[1], s[2], s[3], ctx->saved_data["counts"].toIntVector(), g[0]);
    variable_list out(8);
    const auto shapes = ctx->saved_data["shapes"].toList();
    for (int t = 0; t < 4; ++t) {
        const auto shape = static_cast<c10::IValue>(shapes.get(t)).toIntVector();
        out[4 + t] = shape.size() == 1 ? d[t] : d[t].reshape(shape);
    }
    return out;
}

Tensor mol_energy_autograd(const std::vector<Tensor>& o, const Tensor& types, const Tensor& sis, const Tensor& mos, const Tensor& macs)
{
    same_size(o.size() == 4, "type_outputs must hold the four per-type vectors");
    return MolEnergyFn::apply(types, sis, mos, macs, o[0], o[1], o[2], o[3]);
}

// ---------------------------------------------------------------------------------------------- networks
// A network of `widths` (feature width first, 1 last) for the four types with its parameters in one flat array: for every
// layer the four types' weights [in, out], then for every layer the four types' biases.
struct Net {
    Saved widths;
    double alpha;
    int64_t live_from = 0;      // the parameters of earlier layers are constants: no gradients are formed for them
    uint32_t live() const { return ((1u << layers()) - 1u) & ~((1u << live_from) - 1u); }
    int layers() const { return static_cast<int>(widths.size()) - 1; }        // products, the output layer included
    int64_t weight_at(int l, int t) const
    {
        int64_t at = 0;
        for (int k = 0; k < l; ++k) at += 4 * widths[k] * widths[k + 1];
        return at + t * widths[l] * widths[l + 1];
    }
    int64_t bias_at(int l, int t) const
    {
        int64_t at = weight_at(layers(), 0);
        for (int k = 0; k < l; ++k) at += 4 * widths[k + 1];
        return at + t * widths[l + 1];
    }
    int64_t size() const { return bias_at(layers(), 0); }
};

struct Rows {
    Four x;                // [n_t, widths[0]]
    int64_t n[4], row0[4], total;
};

// Where a network's parameters lie: parts of one flat array, or the tensors themselves, read where they are, so that a pass
// takes the values they have when it runs, whoever wrote them.
struct Params {
    std::vector<Tensor> held;             // what the addresses point into
    std::vector<char*> at;                // for every layer the four types' weights, then for every layer their biases
    at::TensorOptions options;
    at::ScalarType dtype;

    Params(const Net& net, const Tensor& flat) : held{flat}, options(flat.options()), dtype(float_dtype(flat, "parameters"))
    {
        check_net(net);
        dev(flat, dtype, "parameters");
        same_size(flat.numel() == net.size(), "the parameters do not match the network's widths");
        char* base = static_cast<char*>(flat.data_ptr());
        const int64_t w = static_cast<int64_t>(c10::elementSize(dtype));
        for (int l = 0; l < net.layers(); ++l)
            for (int t = 0; t < 4; ++t) at.push_back(base + net.weight_at(l, t) * w);
        for (int l = 0; l < net.layers(); ++l)
            for (int t = 0; t < 4; ++t) at.push_back(base + net.bias_at(l, t) * w);
    }
    Params(const Net& net, const std::vector<Tensor>& tensors)
    {
        check_net(net);
        same_size(tensors.size() == 8 * static_cast<size_t>(net.layers()), "a weight and a bias for each layer and type");
        options = at::TensorOptions().dtype(tensors[0].scalar_type()).device(tensors[0].device());
        dtype = float_dtype(tensors[0], "parameters");
        for (size_t k = 0; k < tensors.size(); ++k) {
            const int l = static_cast<int>(k / 4) % net.layers();
            const bool weight = k / 4 < static_cast<size_t>(net.layers());
            const Tensor p = tensors[k].contiguous();
            if (!p.is_cuda() || p.scalar_type() != dtype) raise(PyExc_TypeError, "the parameters must be CUDA tensors of one type");
            same_size(p.numel() == (weight ? net.widths[l] * net.widths[l + 1] : net.widths[l + 1]),
                      "the parameters do not match the network's widths");
            held.push_back(p);
            at.push_back(static_cast<char*>(p.data_ptr()));
        }
    }
    char* weight(int l, int t) const { return at[4 * l + t]; }
    char* bias(int l, int t) const { return at[at.size() / 2 + 4 * l + t]; }

private:
    static void check_net(const Net& net)
    {
        if (net.widths.size() < 3 || net.layers() > KHAN_NET_MAX_LAYERS || net.widths.back() != 1)
            raise(PyExc_ValueError, "a network of 2 to " + std::to_string(KHAN_NET_MAX_LAYERS) + " layers, the last of width 1");
    }
};

Rows rows_of(const Net& net, const Params& params, const Tensor& h, const Tensor& c, const Tensor& n, const Tensor& o)
{
    const auto dt = params.dtype;
    Rows r;
    r.x = {h, c, n, o};
    r.total = 0;
    for (int t = 0; t < 4; ++t) {
        r.x[t] = flat1(r.x[t]);
        dev(r.x[t], dt, "feature rows");
        same_size(r.x[t].numel() % net.widths[0] == 0, "feature rows must be whole rows");
        r.n[t] = r.x[t].numel() / net.widths[0];
        r.row0[t] = r.total;
        r.total += r.n[t];
    }
    same_size(r.total <= INT32_MAX, "too many rows");
    return r;
}

// The passes over a network's layers (khan_net_*; the names are those of csrc/net_layers.hip).
struct Pass {
    const Net& net;
    const Rows& rows;
    const Params& params;
    khan_stream_t st = stream();
    bool f64 = params.dtype == at::kDouble;
    size_t w = f64 ? 8 : 4;
    int L = net.layers() - 1;                 // hidden layers

    Tensor make(int64_t width) const { return at::empty({rows.total, width}, params.options); }
    char* part(const Tensor& a, int64_t width, int t) const
    {
        return a.defined() && rows.n[t] > 0 ? static_cast<char*>(a.data_ptr()) + rows.row0[t] * width * w : nullptr;
    }
    khan_net_layer layer(int l, bool back, int kind) const
    {
        khan_net_layer a = {};
        a.k = static_cast<int32_t>(net.widths[back ? l + 1 : l]);
        a.n_out = static_cast<int32_t>(net.widths[back ? l : l + 1]);
        a.transposed = back;
        a.kind = kind;
        a.alpha = net.alpha;
        for (int t = 0; t < 4; ++t) {
            a.n[t] = static_cast<int32_t>(rows.n[t]);
            a.w[t] = params.weight(l, t);
        }
        return a;
    }
    void set(const void* (&p)[4], const Tensor& a, int64_t width) const
    {
        for (int t = 0; t < 4; ++t) p[t] = part(a, width, t);
    }
    void set(void* (&p)[4], const Tensor& a, int64_t width) const
    {
        for (int t = 0; t < 4; ++t) p[t] = part(a, width, t);
    }
    static void set(const void* (&p)[4], const Four& a)
    {
        for (int t = 0; t < 4; ++t) p[t] = ptr<char>(a[t]);
    }
    void run(const khan_net_layer& a) const { call(f64 ? api.khan_net_layer_f64 : api.khan_net_layer_f32, &a, st); }
    void run(const khan_net_top& a) const { call(f64 ? api.khan_net_top_f64 : api.khan_net_top_f32, &a, st); }

    // activations a_1 .. a_L.  `inference`: the leading layers of the widths that ops.dense takes have their CELU from exp(z) - 1,
    // as they have there (deep networks on 4,001 molecules 1,785 -> 1,740 us); what differentiates twice needs the sides of
    // 0 that small activations lie on.
    variable_list forward(bool inference) const
    {
        variable_list acts;
        bool leading = inference;
        for (int l = 0; l < L; ++l) {
            leading = leading && net.widths[l] % 32 == 0 && net.widths[l + 1] % 64 == 0;
            khan_net_layer a = layer(l, false, leading ? KHAN_NET_CELU_ABSOLUTE : KHAN_NET_CELU);
            for (int t = 0; t < 4; ++t) a.bias[t] = params.bias(l, t);
            if (l == 0) set(a.in, rows.x);
            else set(a.in, acts[l - 1], net.widths[l]);
            acts.push_back(make(net.widths[l + 1]));
            set(a.out, acts[l], net.widths[l + 1]);
            run(a);
        }
        return acts;
    }
    // the values (into `values`, where defined) and d_L (returned, where asked for)
    Tensor top(const Tensor& last, const Four* values, bool want_d) const
    {
        khan_net_top a = {};
        a.k = static_cast<int32_t>(net.widths[L]);
        a.alpha = net.alpha;
        const Tensor d = want_d ? make(net.widths[L]) : Tensor();
        set(a.act, last, net.widths[L]);
        set(a.out, d, net.widths[L]);
        for (int t = 0; t < 4; ++t) {
            a.n[t] = static_cast<int32_t>(rows.n[t]);
            a.w[t] = params.weight(L, t);
            a.bias[t] = params.bias(L, t);
            a.value[t] = values ? ptr<char>((*values)[t]) : nullptr;
        }
        run(a);
        return d;
    }
    // d_1 .. d_{L-1} from d_L (returned as d[0 .. L-1], d[l] of layer l + 1)
    variable_list slopes(const variable_list& acts, const Tensor& d_last) const
    {
        variable_list d(L);
        d[L - 1] = d_last;
        for (int l = L - 1; l >= 1; --l) {
            khan_net_layer a = layer(l, true, KHAN_NET_SLOPE);
            d[l - 1] = make(net.widths[l]);
            set(a.in, d[l], net.widths[l + 1]);
            set(a.act, acts[l - 1], net.widths[l]);
            set(a.out, d[l - 1], net.widths[l]);
            run(a);
        }
        return d;
    }
    // first . W_1^T, times the rows' factors (scale may hold undefined tensors: ones), into `out` or added to it
    void to_rows(const Tensor& first, const Four& scale, const Four& out, bool accumulate) const
    {
        khan_net_layer a = layer(0, true, KHAN_NET_ROWS);
        a.accumulate = accumulate;
        set(a.in, first, net.widths[1]);
        set(a.scale, scale);
        for (int t = 0; t < 4; ++t) a.out[t] = ptr<char>(out[t]);
        run(a);
    }
    khan_net_grads grads(const Four& scale) const
    {
        khan_net_grads g = {};
        g.layers = net.layers();
        for (size_t k = 0; k < net.widths.size(); ++k) g.widths[k] = static_cast<int32_t>(net.widths[k]);
        for (int t = 0; t < 4; ++t) {
            g.n[t] = static_cast<int32_t>(rows.n[t]);
            g.row0[t] = rows.row0[t];
        }
        set(g.x, rows.x);
        set(g.scale, scale);
        return g;
    }
    Tensor run(khan_net_grads& g) const
    {
        const int64_t bytes = (f64 ? api.khan_net_grads_workspace_bytes_f64 : api.khan_net_grads_workspace_bytes_f32)(&g);
        const Tensor ws = at::empty({bytes}, params.options.dtype(at::kByte)), out = at::empty({net.size()}, params.options);
        g.workspace = ws.data_ptr();
        g.out = out.data_ptr();
        call(f64 ? api.khan_net_grads_f64 : api.khan_net_grads_f32, &g, st);
        return out;
    }
    // gradient of sum_r scale_r value_r by the parameters
    Tensor first_order(const variable_list& acts, const variable_list& d, const Four& scale) const
    {
        khan_net_grads g = grads(scale);
        g.first = net.live();
        g.scale_first = 1;
        for (int l = 0; l <= L; ++l) {
            if (l > 0) g.left[l] = ptr<char>(acts[l - 1]);
            if (l < L) g.right[l] = ptr<char>(d[l]);         // the output layer: ones, times the factors
        }
        return run(g);
    }
};

// `all` cut into one part per type, `width` elements to a row
Four by_type(const Rows& rows, const Tensor& all, int64_t width)
{
    Four out;
    for (int t = 0; t < 4; ++t) out[t] = all.narrow(0, rows.row0[t] * width, rows.n[t] * width);
    return out;
}

Four like_values(const Rows& rows, const Params& params)
{
    return {at::empty({rows.n[0]}, params.options), at::empty({rows.n[1]}, params.options), at::empty({rows.n[2]}, params.options),
            at::empty({rows.n[3]}, params.options)};
}

Four like_rows(const Net& net, const Rows& rows, const Params& params)
{
    return by_type(rows, at::empty({rows.total * net.widths[0]}, params.options), net.widths[0]);
}

// The values from library operations, for derivatives of an order the kernels have no form for.
variable_list library_values(const Net& net, const Tensor& flat, const variable_list& x)
{
    variable_list out;
    for (int t = 0; t < 4; ++t) {
        Tensor a = x[t].reshape({-1, net.widths[0]});
        for (int l = 0; l < net.layers(); ++l) {
            const Tensor w = flat.narrow(0, net.weight_at(l, t), net.widths[l] * net.widths[l + 1]).view({net.widths[l], net.widths[l + 1]});
            a = at::addmm(flat.narrow(0, net.bias_at(l, t), net.widths[l + 1]), a, w);
            if (l + 1 < net.layers())
                a = at::where(a >= 0, a, net.alpha * at::expm1(at::clamp_max(a, 0.0) / net.alpha));
        }
        out.push_back(a.reshape({-1}));
    }
    return out;
}

variable_list library_grad(const variable_list& outputs, const variable_list& inputs, const variable_list& grads)
{
    variable_list o, g;
    for (size_t k = 0; k < outputs.size(); ++k)
        if (grads[k].defined() && outputs[k].requires_grad()) {
            o.push_back(outputs[k]);
            g.push_back(grads[k].reshape(outputs[k].sizes()));
        }
    variable_list in;
    for (const auto& v : inputs)
        if (v.requires_grad()) in.push_back(v);
    variable_list got = o.empty() || in.empty() ? variable_list(in.size()) : torch::autograd::grad(o, in, g, true, true, true), out;
    size_t k = 0;
    for (const auto& v : inputs) out.push_back(v.requires_grad() ? got[k++] : Tensor());
    return out;
}

Net net_of(AutogradContext* ctx)
{
    return Net{ctx->saved_data["widths"].toIntVector(), ctx->saved_data["alpha"].toDouble(), ctx->saved_data["live_from"].toInt()};
}
void keep(AutogradContext* ctx, const Net& net)
{
    ctx->saved_data["widths"] = net.widths;
    ctx->saved_data["alpha"] = net.alpha;
    ctx->saved_data["live_from"] = net.live_from;
}

Four or_zeros(const Rows& rows, const Tensor& flat, const variable_list& g, int from, int64_t width)
{
    Four out;
    for (int t = 0; t < 4; ++t) {
        const Tensor& v = g[from + t];
        out[t] = v.defined() ? flat1(v).contiguous() : at::zeros({rows.n[t] * width}, flat.options());
    }
    return out;
}

// The rows' gradients s_r d value_r / d x_r as a function of the parameters, the rows and s: what a loss on forces
// differentiates once more.
struct NetRowsFn : Function<NetRowsFn> {
    // inputs: flat, x[4], s[4]; saved behind them: the activations and d_1 .. d_L
    static variable_list forward(AutogradContext* ctx, const Tensor& flat, const Tensor& x0, const Tensor& x1, const Tensor& x2, const Tensor& x3,
                                 const Tensor& s0, const Tensor& s1, const Tensor& s2, const Tensor& s3, const variable_list& kept_acts, const Net& net)
    {
        const Unrecorded quiet;
        const Params params(net, flat);
        const Rows rows = rows_of(net, params, x0, x1, x2, x3);
        const Pass p{net, rows, params};
        const variable_list acts(kept_acts.begin(), kept_acts.begin() + p.L);
        const variable_list d = p.slopes(acts, kept_acts[p.L]);
        const Four s = {s0, s1, s2, s3};
        const Four out = like_rows(net, rows, params);
        p.to_rows(d[0], s, out, false);
        variable_list save = {flat, x0, x1, x2, x3, s0, s1, s2, s3};
        save.insert(save.end(), acts.begin(), acts.end());
        save.insert(save.end(), d.begin(), d.end());
        ctx->save_for_backward(save);
        keep(ctx, net);
        const Four xs = {x0, x1, x2, x3};
        variable_list res;
        for (int t = 0; t < 4; ++t) res.push_back(out[t].reshape(xs[t].sizes()));
        return res;
    }
    static variable_list backward(AutogradContext* ctx, variable_list u)
    {
        const auto saved = ctx->get_saved_variables();
        const Net net = net_of(ctx);
        const Tensor flat = saved[0];
        const variable_list x(saved.begin() + 1, saved.begin() + 5), s(saved.begin() + 5, saved.begin() + 9);
        variable_list out(11);
        if (at::GradMode::is_enabled()) {
            variable_list in = {flat};
            in.insert(in.end(), x.begin(), x.end());
            in.insert(in.end(), s.begin(), s.end());
            // (rows that carry no graph of their own still have to be differentiated by)
            variable_list xs = x;
            for (auto& v : xs)
                if (!v.requires_grad()) v = v.detach().requires_grad_(true);
            const auto rows = library_grad(library_values(net, flat, xs), xs, s);
            for (int t = 0; t < 4; ++t) in[1 + t] = xs[t];
            const auto g = library_grad(rows, in, u);
            for (int k = 0; k < 9; ++k)
                if (k == 0 || k > 4 || x[k - 1].requires_grad()) out[k] = g[k];
            return out;
        }
        const Unrecorded quiet;
        const Params params(net, flat);
        const Rows rows = rows_of(net, params, x[0], x[1], x[2], x[3]);
        const Pass p{net, rows, params};
        const int L = p.L;
        const variable_list acts(saved.begin() + 9, saved.begin() + 9 + L), d(saved.begin() + 9 + L, saved.begin() + 9 + 2 * L);
        const Four v = or_zeros(rows, flat, u, 0, net.widths[0]);
        const Four scale = {s[0].contiguous(), s[1].contiguous(), s[2].contiguous(), s[3].contiguous()};
        // the tangents along u
        variable_list dot, second;
        for (int l = 0; l < L; ++l) {
            khan_net_layer a = p.layer(l, false, KHAN_NET_TANGENT);
            if (l == 0) Pass::set(a.in, v);
            else p.set(a.in, dot[l - 1], net.widths[l]);
            dot.push_back(p.make(net.widths[l + 1]));
            second.push_back(p.make(net.widths[l + 1]));
            p.set(a.act, acts[l], net.widths[l + 1]);
            p.set(a.d, d[l], net.widths[l + 1]);
            p.set(a.out, dot[l], net.widths[l + 1]);
            p.set(a.out2, second[l], net.widths[l + 1]);
            p.run(a);
        }
        const bool need_x = ctx->needs_input_grad(1) || ctx->needs_input_grad(2) || ctx->needs_input_grad(3) || ctx->needs_input_grad(4);
        const bool need_s = ctx->needs_input_grad(5) || ctx->needs_input_grad(6) || ctx->needs_input_grad(7) || ctx->needs_input_grad(8);
        if (need_s) {          // the values' tangents
            khan_net_top a = {};
            a.k = static_cast<int32_t>(net.widths[L]);
            a.alpha = net.alpha;
            const Four e = like_values(rows, params);
            p.set(a.act, dot[L - 1], net.widths[L]);
            for (int t = 0; t < 4; ++t) {
                a.n[t] = static_cast<int32_t>(rows.n[t]);
                a.w[t] = params.weight(L, t);
                a.value[t] = ptr<char>(e[t]);
                out[5 + t] = e[t].reshape(s[t].sizes());
            }
            p.run(a);
        }
        if (!need_x && !ctx->needs_input_grad(0)) return out;
        // q_L .. q_1
        variable_list q(L);
        {
            khan_net_top a = {};
            a.k = static_cast<int32_t>(net.widths[L]);
            a.alpha = net.alpha;
            a.second = 1;
            q[L - 1] = p.make(net.widths[L]);
            p.set(a.t, second[L - 1], net.widths[L]);
            p.set(a.out, q[L - 1], net.widths[L]);
            Pass::set(a.scale, scale);
            for (int t = 0; t < 4; ++t) a.n[t] = static_cast<int32_t>(rows.n[t]);
            p.run(a);
        }
        for (int l = L - 1; l >= 1; --l) {
            khan_net_layer a = p.layer(l, true, KHAN_NET_SECOND);
            q[l - 1] = p.make(net.widths[l]);
            p.set(a.in, q[l], net.widths[l + 1]);
            p.set(a.act, acts[l - 1], net.widths[l]);
            p.set(a.t, second[l - 1], net.widths[l]);
            Pass::set(a.scale, scale);
            p.set(a.out, q[l - 1], net.widths[l]);
            p.run(a);
        }
        if (need_x) {
            const Four g = like_rows(net, rows, params);
            p.to_rows(q[0], Four{}, g, false);
            for (int t = 0; t < 4; ++t) out[1 + t] = g[t].reshape(x[t].sizes());
        }
        if (ctx->needs_input_grad(0)) {
            khan_net_grads g = p.grads(scale);
            g.first = net.live() & ((1u << L) - 1u);       // the hidden layers: a^T q ...
            g.second = net.live();                         // ... and all: a'^T (s d), d = 1 in the output layer
            g.scale_second = 1;
            Pass::set(g.x2, v);
            for (int l = 0; l <= L; ++l) {
                if (l > 0) {
                    g.left[l] = l < L ? ptr<char>(acts[l - 1]) : nullptr;
                    g.left2[l] = ptr<char>(dot[l - 1]);
                }
                if (l < L) {
                    g.right[l] = ptr<char>(q[l]);
                    g.right2[l] = ptr<char>(d[l]);
                }
            }
            out[0] = p.run(g);
        }
        return out;
    }
};

// The values of the four types' rows as a function of the parameters and the rows.
struct NetFn : Function<NetFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& flat, const Tensor& x0, const Tensor& x1, const Tensor& x2, const Tensor& x3,
                                 const Net& net, bool graph)
    {
        const Unrecorded quiet;
        const Params params(net, flat);
        const Rows rows = rows_of(net, params, x0, x1, x2, x3);
        const Pass p{net, rows, params};
        const Four values = like_values(rows, params);
        variable_list acts = p.forward(false);
        const Tensor d = p.top(acts.back(), &values, graph);
        if (graph) {
            variable_list save = {flat, x0, x1, x2, x3};
            save.insert(save.end(), acts.begin(), acts.end());
            save.push_back(d);
            ctx->save_for_backward(save);
            keep(ctx, net);
        }
        return {values[0], values[1], values[2], values[3]};
    }
    static variable_list backward(AutogradContext* ctx, variable_list gs)
    {
        const auto saved = ctx->get_saved_variables();
        const Net net = net_of(ctx);
        const Tensor flat = saved[0];
        const variable_list x(saved.begin() + 1, saved.begin() + 5);
        const bool need_x = ctx->needs_input_grad(1) || ctx->needs_input_grad(2) || ctx->needs_input_grad(3) || ctx->needs_input_grad(4);
        const bool need_p = ctx->needs_input_grad(0);
        variable_list out(7);
        if (at::GradMode::is_enabled() && need_p) {
            const auto g = library_grad(library_values(net, flat, x), {flat, x[0], x[1], x[2], x[3]}, gs);
            for (int k = 0; k < 5; ++k) out[k] = g[k];
            return out;
        }
        const Params params(net, flat);
        const Rows rows = rows_of(net, params, x[0], x[1], x[2], x[3]);
        if (at::GradMode::is_enabled()) {
            variable_list s(4);
            for (int t = 0; t < 4; ++t) s[t] = gs[t].defined() ? gs[t].contiguous() : at::zeros({rows.n[t]}, flat.options());
            const variable_list kept_acts(saved.begin() + 5, saved.end());
            const auto g = NetRowsFn::apply(flat, x[0], x[1], x[2], x[3], s[0], s[1], s[2], s[3], kept_acts, net);
            for (int t = 0; t < 4; ++t) out[1 + t] = g[t];
            return out;
        }
        const Unrecorded quiet;
        const Pass p{net, rows, params};
        const variable_list acts(saved.begin() + 5, saved.begin() + 5 + p.L);
        const variable_list d = p.slopes(acts, saved[5 + p.L]);
        const Four scale = or_zeros(rows, flat, gs, 0, 1);
        if (need_x) {
            const Four g = like_rows(net, rows, params);
            p.to_rows(d[0], scale, g, false);
            for (int t = 0; t < 4; ++t) out[1 + t] = g[t].reshape(x[t].sizes());
        }
        if (need_p) out[0] = p.first_order(acts, d, scale);
        return out;
    }
};

// live_from: the parameters of earlier layers are constants
std::vector<Tensor> network_autograd(const Tensor& flat, const std::vector<Tensor>& x, Saved widths, double alpha, int64_t live_from)
{
    same_size(x.size() == 4, "four feature buckets");
    const Net net{widths, alpha, live_from};
    same_size(live_from >= 0 && live_from <= net.layers(), "live_from must be a layer's number, or the number of layers");
    bool graph = flat.requires_grad();
    for (const Tensor& v : x) graph |= v.requires_grad();
    return NetFn::apply(flat, x[0], x[1], x[2], x[3], net, graph && at::GradMode::is_enabled());
}

// The parameters of a network (tensors of any shape) end to end in one array.
struct FlattenFn : Function<FlattenFn> {
    static Tensor forward(AutogradContext* ctx, at::TensorList params)
    {
        const Unrecorded quiet;
        std::vector<Saved> shapes;
        std::vector<Tensor> flat;
        for (const auto& p : params) {
            shapes.push_back(p.sizes().vec());
            flat.push_back(flat1(p));
        }
        ctx->saved_data["shapes"] = shapes;
        return at::cat(flat);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        variable_list out;
        const auto shapes = ctx->saved_data["shapes"].toList();
        int64_t at = 0;
        const auto parts = [&](bool strided) {
            for (size_t k = 0; k < shapes.size(); ++k) {
                const auto shape = static_cast<c10::IValue>(shapes.get(k)).toIntVector();
                const int64_t n = c10::multiply_integers(shape);
                if (strided) out.push_back(g[0].as_strided(shape, c10::contiguous_strides(shape), at));
                else out.push_back(g[0].narrow(0, at, n).view(shape));
                at += n;
            }
        };
        if (at::GradMode::is_enabled() || !g[0].is_contiguous() || g[0].storage_offset() != 0) {
            parts(false);
        } else {
            const Unrecorded quiet;
            parts(true);
        }
        return out;
    }
};

Tensor flatten(const std::vector<Tensor>& params)
{
    return FlattenFn::apply(at::TensorList(params));
}

// ---------------------------------------------------------------------------------------------- inference
// One network of a model: its parameters and, for the one-launch kernel, the weights split and packed
struct Weights {
    Net net;
    Params params;
    Tensor packed;
};

// A network's pass over a batch: the values, then the rows' gradients.
struct Inference {
    const Weights& w;
    const Rows rows;
    const Pass pass;
    Tensor values;                          // of all rows, type by type
    variable_list state;                    // activations and d_L; in the one-launch forms the rows' gradients
    bool few = false;                       // float64 in one launch (net_few.hip): see take_few
    bool chain = false;                     // float32, a launch each way (net_chain.hip): see take_chain; state: its workspace

    Inference(const Weights& w_, const Four& x)
        : w(w_), rows(rows_of(w.net, w.params, x[0], x[1], x[2], x[3])), pass{w.net, rows, w.params},
          values(at::empty({rows.total}, w.params.options))
    {
    }
    bool one_launch() const { return w.packed.defined(); }

    // Float64 networks of the widths net_few.hip takes, whose rows' gradients are not to be scaled: one launch up to
    // KHAN_NET_FEW_TILES tiles of KHAN_NET_FEW_ROWS rows of a type, one for every compute unit (us, values and gradients, layer by
    // layer -> one launch: 1 molecule 80 -> 67, 16 molecules 112 -> 86, 256 (2,970 rows) 152 -> 115, 330 (3,863) 175 -> 132; values
    // alone 41 -> 29, 54 -> 39, 67 -> 47).
    void take_few()
    {
        if (w.params.dtype != at::kDouble || w.net.layers() > KHAN_NET_FEW_LAYERS) return;
        int32_t widths[KHAN_NET_FEW_LAYERS + 1];
        for (size_t k = 0; k < w.net.widths.size(); ++k) widths[k] = static_cast<int32_t>(w.net.widths[k]);
        if (!api.khan_net_few_fits(widths, w.net.layers())) return;
        int64_t tiles = 0;
        uintptr_t bits = 0;
        for (int t = 0; t < 4; ++t) {
            tiles += (rows.n[t] + KHAN_NET_FEW_ROWS - 1) / KHAN_NET_FEW_ROWS;
            if (rows.n[t] > 0) bits |= reinterpret_cast<uintptr_t>(rows.x[t].data_ptr());
            for (int l = 0; l < w.net.layers(); ++l) bits |= reinterpret_cast<uintptr_t>(w.params.weight(l, t));
        }
        few = tiles <= KHAN_NET_FEW_TILES && (bits & 15u) == 0;
    }
    Tensor launch_few(bool want_rows)
    {
        const Tensor grads = want_rows ? at::empty({rows.total * w.net.widths[0]}, w.params.options) : Tensor();
        khan_net_few a = {};
        a.layers = w.net.layers();
        for (size_t k = 0; k < w.net.widths.size(); ++k) a.widths[k] = static_cast<int32_t>(w.net.widths[k]);
        a.alpha = w.net.alpha;
        for (int t = 0; t < 4; ++t) {
            a.n[t] = static_cast<int32_t>(rows.n[t]);
            a.x[t] = rows.n[t] > 0 ? rows.x[t].data_ptr() : nullptr;
            a.value[t] = pass.part(values, 1, t);
            a.grad[t] = pass.part(grads, w.net.widths[0], t);
            for (int l = 0; l < a.layers; ++l) {
                a.w[l][t] = w.params.weight(l, t);
                a.b[l][t] = w.params.bias(l, t);
            }
        }
        call(api.khan_net_few_f64, static_cast<const khan_net_few*>(&a), pass.st);
        return grads;
    }

    // Float32 networks that would go layer by layer otherwise, of hidden widths up to 256 and rows of a multiple of 128 (us, layer by layer
    // -> this; deep networks with gradients: 1 organic molecule 191 -> 168, 400 321 -> 202, 4,096 904 -> 814; values alone 1 104 -> 99,
    // 256 136 -> 107; default ones beside charges, values alone: 16 97 -> 91, 256 108 -> 98, 4,096 239 -> 201; with gradients 65,536
    // 5,013 -> 4,665).
    void take_chain()
    {
        if (w.params.dtype != at::kFloat || one_launch()) return;
        const khan_net_chain a = chain_net(false);
        uintptr_t bits = 0;
        for (int t = 0; t < 4; ++t) bits |= reinterpret_cast<uintptr_t>(a.x[t]);
        chain = rows.total > 0 && (bits & 15u) == 0 && api.khan_net_chain_fits(a.widths, a.layers);
    }
    khan_net_chain chain_net(bool want_rows) const
    {
        khan_net_chain a = {};
        a.layers = w.net.layers();
        a.alpha = w.net.alpha;
        a.want_rows = want_rows;
        for (size_t k = 0; k < w.net.widths.size(); ++k) a.widths[k] = static_cast<int32_t>(w.net.widths[k]);
        bool leading = true;                // (the CELU of Pass::forward)
        for (int l = 0; l < a.layers; ++l) {
            leading = leading && l + 1 < a.layers && a.widths[l] % 32 == 0 && a.widths[l + 1] % 64 == 0;
            if (leading) a.absolute |= 1u << l;
            for (int t = 0; t < 4; ++t) {
                a.w[l][t] = w.params.weight(l, t);
                a.b[l][t] = w.params.bias(l, t);
            }
        }
        for (int t = 0; t < 4; ++t) {
            a.n[t] = static_cast<int32_t>(rows.n[t]);
            a.x[t] = rows.n[t] > 0 ? rows.x[t].data_ptr() : nullptr;
            a.value[t] = pass.part(values, 1, t);
        }
        return a;
    }
    Tensor launch_chain(bool want_rows)
    {
        khan_net_chain a = chain_net(want_rows);
        const Tensor workspace = at::empty({api.khan_net_chain_workspace_bytes(&a)}, w.params.options.dtype(at::kByte));
        a.workspace = workspace.data_ptr();
        call(api.khan_net_chain_values_f32, static_cast<const khan_net_chain*>(&a), pass.st);
        return workspace;
    }

    Tensor launch(bool want_rows)
    {
        const Tensor grads = want_rows ? at::empty({rows.total * kFeats}, w.params.options) : Tensor();
        const float *x[4], *bias[12], *head_w[4], *head_b[4];
        float *value[4], *grad[4];
        int32_t n[4];
        for (int t = 0; t < 4; ++t) {
            x[t] = ptr<float>(rows.x[t]);
            n[t] = static_cast<int32_t>(rows.n[t]);
            for (int l = 0; l < 3; ++l) bias[4 * l + t] = reinterpret_cast<const float*>(w.params.bias(l, t));
            head_w[t] = reinterpret_cast<const float*>(w.params.weight(3, t));
            head_b[t] = reinterpret_cast<const float*>(w.params.bias(3, t));
            value[t] = ptr<float>(values) ? ptr<float>(values) + rows.row0[t] : nullptr;
            grad[t] = want_rows && ptr<float>(grads) ? ptr<float>(grads) + rows.row0[t] * kFeats : nullptr;
        }
        call(api.khan_atomic_networks_f32, x, n, static_cast<const float* const*>(nullptr), static_cast<const float* const*>(nullptr),
             static_cast<const void*>(w.packed.data_ptr()), bias, head_w, head_b, static_cast<const float* const*>(nullptr),
             static_cast<float>(w.net.alpha), value, want_rows ? grad : static_cast<float* const*>(nullptr), pass.st);
        return grads;
    }
    // want_rows: row gradients will be asked for; exact: as network_autograd forms the activations
    Four forward(bool want_rows, bool exact = false)
    {
        const Four v = by_type(rows, values, 1);
        if (one_launch()) {
            state = {launch(want_rows)};
        } else if (few) {
            state = {launch_few(want_rows)};
        } else if (chain) {
            state = {launch_chain(want_rows)};
        } else {
            state = pass.forward(!exact);
            state.push_back(pass.top(state.back(), &v, want_rows));
        }
        return v;
    }
    // the rows' gradients times scale (undefined: ones), added to `into` where defined -> [all rows, features]; the one-launch
    // forms have them already, and take neither scale nor anything to add to
    Tensor gradients(const Four& scale, Tensor into)
    {
        if (one_launch() || few) {
            for (const Tensor& s : scale) same_size(!s.defined(), "networks in one launch have no scaled gradients");
            same_size(!into.defined(), "networks in one launch add their gradients to nothing");
            return state[0];
        }
        const bool add = into.defined();
        if (!add) into = at::empty({rows.total * w.net.widths[0]}, w.params.options);
        if (chain) {
            khan_net_chain a = chain_net(true);
            a.workspace = state[0].data_ptr();
            a.accumulate = add;
            const Four out = by_type(rows, into, w.net.widths[0]);
            for (int t = 0; t < 4; ++t) {
                a.scale[t] = scale[t].defined() && rows.n[t] > 0 ? scale[t].data_ptr() : nullptr;
                a.grad[t] = rows.n[t] > 0 ? out[t].data_ptr() : nullptr;
            }
            call(api.khan_net_chain_rows_f32, static_cast<const khan_net_chain*>(&a), pass.st);
            return into;
        }
        const variable_list d = pass.slopes(variable_list(state.begin(), state.end() - 1), state.back());
        pass.to_rows(d[0], scale, by_type(rows, into, w.net.widths[0]), add);
        return into;
    }
};

Weights weights_of(const py::tuple& t, double alpha)
{
    const Net net{t[2].cast<Saved>(), alpha};
    Weights w{net, Params(net, t[0].cast<std::vector<Tensor>>()), Tensor()};
    if (t[1].cast<bool>()) {
        same_size(w.params.dtype == at::kFloat && net.widths == Saved{kFeats, 128, 128, 64, 1},
                  "the one-launch kernel takes 384-128-128-64-1 networks in float32");
        // One launch of 6 us on the stream that reads it: what the parameters are now, without a word about who may write to
        // them and when.
        w.packed = at::empty({api.khan_atomic_networks_packed_bytes()}, w.params.options.dtype(at::kByte));
        const float* stored[12];
        for (int k = 0; k < 12; ++k) stored[k] = reinterpret_cast<const float*>(w.params.weight(k / 4, k % 4));
        call(api.khan_atomic_networks_pack_stored_f32, static_cast<const float* const*>(stored), w.packed.data_ptr(), stream());
    }
    return w;
}

// The networks' part of `infer` alone, for a caller that has the rows: the values of the four types' rows and, with want_grad,
// what `network_rows` needs to form gradients -> (values[4], activations..., d_L)
std::vector<Tensor> network_forward(const Tensor& flat, const std::vector<Tensor>& x, Saved widths, double alpha, bool want_grad)
{
    same_size(x.size() == 4, "four feature buckets");
    const Net net{widths, alpha};
    const Weights w{net, Params(net, flat), Tensor()};
    Inference net_pass(w, {x[0], x[1], x[2], x[3]});
    const Four values = net_pass.forward(want_grad, true);
    std::vector<Tensor> out(values.begin(), values.end());
    if (want_grad) out.insert(out.end(), net_pass.state.begin(), net_pass.state.end());
    return out;
}

// scale_r d value_r / d x_r from what network_forward left behind the values (scale: four vectors, or none for ones), into
// new arrays or added to `into` (four arrays of rows, end to end in one) -> the four arrays
std::vector<Tensor> network_rows(const Tensor& flat, const std::vector<Tensor>& x, Saved widths, double alpha, const std::vector<Tensor>& state,
                                 const c10::optional<std::vector<Tensor>>& scale, const c10::optional<std::vector<Tensor>>& into)
{
    same_size(x.size() == 4, "four feature buckets");
    const Net net{widths, alpha};
    const Weights w{net, Params(net, flat), Tensor()};
    Inference net_pass(w, {x[0], x[1], x[2], x[3]});
    net_pass.state = state;
    same_size(static_cast<int>(state.size()) == net.layers() && (!scale || scale->size() == 4) && (!into || into->size() == 4),
              "state as network_forward returned it behind the values, and four scales and four arrays of rows");
    Four s;
    for (int t = 0; t < 4 && scale; ++t) {
        s[t] = (*scale)[t].reshape({-1});
        dev(s[t], w.params.dtype, "scale");
        same_size(s[t].numel() == net_pass.rows.n[t], "scale must have one element per row");
    }
    const Four out = by_type(net_pass.rows, net_pass.gradients(s, into ? at::cat(*into) : Tensor()), net.widths[0]);
    return {out[0], out[1], out[2], out[3]};
}

// A batch's energies and, with need_grad, their gradient by x, y and z: featurize, the networks' values and row gradients, the
// sums by molecule, the charge energy, featurize_grad.  No graph: the order of the passes is known, and the gradient of
// the near network's sum needs nothing from behind it.  near, charge: (the parameters as Params takes them, whether in
// one launch, widths).
// -> (energies,) or (energies, x, y, z); joined: all four are parts of one array, the last element of what is returned, which
// holds the energies, padded to 64 elements, then the three gradients
std::vector<Tensor> infer(const Tensor& xs, const Tensor& ys, const Tensor& zs, const Tensor& as, const Tensor& mos, const Tensor& macs,
                          const Tensor& sis, const Tensor& gather, const py::object& acs, const c10::optional<Tensor>& order,
                          const py::object& size_classes, const py::tuple& near, const py::object& charge, double alpha, bool need_grad, bool joined)
{
    const at::NoGradGuard no_graph;
    same_size(need_grad || !joined, "energies alone need no array to be joined in");
    const Atoms7 in = {xs.detach(), ys.detach(), zs.detach(), as, mos, macs, sis};
    const AevArgs args = aev_args(acs, order, size_classes);
    const int64_t n = xs.numel(), m = mos.numel(), from = joined ? (m + 63) / 64 * 64 : 0;
    const Tensor result = need_grad ? at::empty({from + 3 * n}, xs.options()) : Tensor();
    std::vector<Tensor> out = {joined ? result.narrow(0, 0, m) : at::empty({m}, xs.options())};
    if (need_grad)
        for (int k = 0; k < 3; ++k) out.push_back(result.narrow(0, from + k * n, n));
    if (joined) out.push_back(result);
    const auto f = run_featurize(in, args);
    const Four feats = {f[0], f[1], f[2], f[3]};
    const Weights near_w = weights_of(near, alpha);
    same_size(charge.is_none() || !near_w.packed.defined(), "networks beside a charge network take no packed weights");
    Inference near_net(near_w, feats);
    near_net.take_few();
    near_net.take_chain();
    run_mol_energy(near_net.forward(need_grad), as, sis, mos, macs, out[0]);
    if (charge.is_none()) {
        if (need_grad) run_featurize_grad(in, args, by_type(near_net.rows, near_net.gradients({}, Tensor()), kFeats), {out[1], out[2], out[3]});
        return out;
    }
    const Weights charge_w = weights_of(charge.cast<py::tuple>(), alpha);
    same_size(!charge_w.packed.defined(), "a charge network takes no packed weights");
    Inference charge_net(charge_w, feats);
    if (!need_grad) charge_net.take_few();
    charge_net.take_chain();
    charge_net.forward(need_grad);
    // (the library's gather, which refuses an index that is no integer or lies outside the rows)
    const Tensor qs = charge_net.values.index_select(0, gather);
    same_size(qs.numel() == n, "gather_idxs must have one element per atom");
    if (!need_grad) {
        out[0].add_(ani_charge(in[0], in[1], in[2], qs, mos, macs));
        return out;
    }
    const Tensor row_of = gather.to(at::kInt).contiguous(), ones = at::empty({m}, xs.options());
    const int64_t n_rows = charge_net.rows.total;
    same_size(n_rows <= n, "no more feature rows than atoms");
    const auto in_type = [&](auto f32, auto f64) { return xs.scalar_type() == at::kFloat ? f32(0.0f) : f64(0.0); };
    // the ones that the energies' gradients are and, of no rows at all, NaN for every row's derivative: what a row that no atom's index
    // names then has
    const Tensor by_value = at::empty({n_rows}, xs.options());
    const auto begin = [&](auto fn) {
        return [&, fn](auto zero) {
            using T = decltype(zero);
            call(fn, static_cast<const T*>(nullptr), ptr<const int32_t>(row_of), n_rows, int64_t{0}, ptr<T>(by_value), ptr<T>(ones), m, charge_net.pass.st);
        };
    };
    in_type(begin(api.khan_take_rows_f32), begin(api.khan_take_rows_f64));
    const auto c = ani_charge_grads(in[0], in[1], in[2], qs, mos, macs, ones, true, true);
    const auto put = [&](auto fn) {
        return [&, fn](auto zero) {
            using T = decltype(zero);
            call(fn, ptr<const T>(c[1]), ptr<const int32_t>(row_of), n, n_rows, ptr<T>(by_value), charge_net.pass.st);
        };
    };
    in_type(put(api.khan_put_rows_f32), put(api.khan_put_rows_f64));
    const Tensor g = charge_net.gradients(by_type(charge_net.rows, by_value, 1), near_net.gradients({}, Tensor()));
    run_featurize_grad(in, args, by_type(near_net.rows, g, kFeats), {out[1], out[2], out[3]});
    const auto add = [&](auto fn) {                                              // (x, y and z lie end to end)
        return [&, fn](auto zero) {
            using T = decltype(zero);
            call(fn, ptr<T>(out[0]), ptr<const T>(c[0]), m, ptr<T>(out[1]), ptr<const T>(c[2]), 3 * n, charge_net.pass.st);
        };
    };
    in_type(add(api.khan_add_two_f32), add(api.khan_add_two_f64));
    return out;
}

}  // namespace

void bind_autograd(py::module_& m)
{
    m.def("featurize_autograd", &featurize_autograd);
    m.def("ani_charge_autograd", &ani_charge_autograd);
    m.def("mol_energy_autograd", &mol_energy_autograd);
    m.def("network_autograd", &network_autograd, py::arg("flat"), py::arg("x"), py::arg("widths"), py::arg("alpha"), py::arg("live_from") = 0);
    m.def("flatten", &flatten);
    m.def("network_forward", &network_forward);
    m.def("network_rows", &network_rows);
    m.def("infer", &infer);
}

}  // namespace khan_torch
