// DDFPack (ddf/ddf.py:195-222 of the reference) as one native call: inference, and a
// training step's forward as one autograd node whose backward runs the operator's gradient
// kernels, the normalisation's and both branches'.  A layer made of torch modules issues
// some thirty launches per training step, each through the interpreter, the dispatcher and
// the convolution library: at ResNet-50's sizes a step was 0.7-0.8 ms of host time around
// 0.2 ms of kernels.
#pragma once

#include "module_guard.h"

#include <torch/csrc/autograd/functions/basic_ops.h>

namespace ddf_torch {

constexpr size_t kAlign = 256;
inline size_t aligned_bytes(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

// What a DDFPack is made of, collected by DDFPack._pack_plan in modules.py (which has
// checked that both branches are the stock ones): with a guard once, for calls through
// pack_forward, or without for a single call of pack_infer.
struct PackPlan {
    Refs refs;
    ModuleGuard *guard = nullptr;    // (owned by refs; null: a plan for one call)
    // 1x1 convolutions (weight, bias): spatial branch, first and second of the channel branch
    TensorRef ws, bs, w1, b1, w2, b2;
    // FilterNorm: learned gains and offsets, or the constant gain
    TensorRef sgain_vec, soffset_vec, cgain_vec, coffset_vec;
    double sgain, cgain;
    int64_t channels;     // that the channel filters are normalised by
    int k, d, s, head, combine;
    bool fuse_pool, fuse_norm;

    // tensors: those ten
    PackPlan(const py::object &guard_, const py::list &tensors, double sgain_, double cgain_, int64_t channels_, int k_,
             int d_, int s_, int head_, const std::string &combine_, bool fuse_pool_, bool fuse_norm_)
        : sgain(sgain_), cgain(cgain_), channels(channels_), k(k_), d(d_), s(s_), head(head_),
          combine(combine_code(combine_)), fuse_pool(fuse_pool_), fuse_norm(fuse_norm_) {
        TORCH_CHECK(tensors.size() == 10, "ten tensors expected");
        const std::vector<TensorRef> t = tensor_refs(refs, tensors);
        TORCH_CHECK(t[0].defined() && t[2].defined() && t[4].defined(), "weights expected");
        ws = t[0]; bs = t[1]; w1 = t[2]; b1 = t[3]; w2 = t[4]; b2 = t[5];
        sgain_vec = t[6]; soffset_vec = t[7]; cgain_vec = t[8]; coffset_vec = t[9];
        if (!guard_.is_none()) {
            guard = guard_.cast<ModuleGuard *>();
            refs.add(guard_.ptr());
        }
    }
    int traverse(visitproc visit, void *arg) const { return refs.traverse(visit, arg); }
    void clear() {
        guard = nullptr;
        for (TensorRef *t : {&ws, &bs, &w1, &b1, &w2, &b2, &sgain_vec, &soffset_vec, &cgain_vec, &coffset_vec}) *t = {};
        refs.clear();
    }
    bool holds() const { return guard && guard->holds(); }
    // Why the branch kernels cannot run these features with the plan's tensors as they are now
    // (parameters may have been resized, moved or re-laid in place), or null.
    const char *misfit(const at::Tensor &x) const {
        const auto type = x.scalar_type();
        const auto dev = x.device();
        const int64_t c = x.size(1), kk = (int64_t)k * k;
        if (has_tangent(x)) return "the branch kernels have no forward-mode derivative";
        if (head < 1 || c % head != 0) return "channels must divide into heads";
        if (channels != c) return "the channel filters' normalisation does not fit the features";
        for (const TensorRef *t : {&ws, &w1, &w2})
            if ((*t)->dim() != 4 || (*t)->size(2) != 1 || (*t)->size(3) != 1) return "branch weights do not fit the features";
        const int64_t mid = w1->size(0);
        if (ws->size(0) != head * kk || ws->size(1) != c || w1->size(1) != c || w2->size(0) != c * kk || w2->size(1) != mid)
            return "branch weights do not fit the features";
        const char *why = nullptr;
        auto ask = [&](const TensorRef &t, int64_t count) {
            if (why || !t.defined()) return;
            if (t->scalar_type() != type || t->device() != dev) why = "parameters must be of the features' type and device";
            else if (t->unsafeGetTensorImpl()->is_python_dispatch()) why = "parameters must be plain tensors";
            else if (has_tangent(*t)) why = "the branch kernels have no forward-mode derivative";
            else if (!t->is_contiguous()) why = "weights must be contiguous";
            else if (t->numel() != count) why = "branch parameters do not fit the features";
        };
        ask(ws, head * kk * c); ask(bs, head * kk);
        ask(w1, mid * c); ask(b1, mid);
        ask(w2, c * kk * mid); ask(b2, c * kk);
        ask(sgain_vec, head * kk); ask(soffset_vec, head * kk);
        ask(cgain_vec, c * kk); ask(coffset_vec, c * kk);
        return why;
    }
    bool wants_gradients(const at::Tensor &x) const {
        if (x.requires_grad()) return true;
        for (const TensorRef *t : {&ws, &bs, &w1, &b1, &w2, &b2, &sgain_vec, &soffset_vec, &cgain_vec, &coffset_vec})
            if (t->defined() && (*t)->requires_grad()) return true;
        return false;
    }
};

// Without gradients: spatial branch (leaving the planes' partial sums where its kernel
// can), channel branch, operator.  (The caller has asked misfit.)
inline at::Tensor pack_run(const PackPlan &p, const at::Tensor &features) {
    const int dt = dtype_code(features.scalar_type());
    const at::Tensor x = features.contiguous();
    const int64_t b = x.size(0), c = x.size(1), h = x.size(2), w = x.size(3), mid = p.w1->size(0);
    const int64_t ho = h / p.s, wo = w / p.s, kk = (int64_t)p.k * p.k;
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(x.device());
    hipStream_t st = current_stream(x);
    at::Tensor out = new_tensor({b, c, ho, wo}, x.scalar_type(), x.device());
    // both filters and the partial sums in one piece of scratch
    const size_t esz = x.element_size();
    const size_t cf_bytes = aligned_bytes(b * c * kk * esz), sf_bytes = aligned_bytes(b * p.head * kk * ho * wo * esz);
    const int64_t cap = p.fuse_pool ? b * c * ((ho * wo + 63) / 64 + 1) : 0;
    at::Tensor scratch = new_tensor({(int64_t)(cf_bytes + sf_bytes + cap * sizeof(float))}, at::kByte, x.device());
    char *base = static_cast<char *>(scratch.data_ptr());
    void *cf = base, *sf = base + cf_bytes;
    // The spatial branch reads every feature plane anyway: where its kernel can, it leaves
    // the planes' partial sums and the channel branch pools from those (one launch and
    // one read of the feature map fewer); else pool first.
    bool pooled_on_the_way = false;
    if (p.fuse_pool && b * c * ho * wo > 0) {
        float *parts = reinterpret_cast<float *>(base + cf_bytes + sf_bytes);
        int n_parts = 0;
        const int rc = ddf_hip_spatial_branch_pool(
            x.data_ptr(), p.ws->data_ptr(), ptr_or_null(p.bs), sf, parts, cap, &n_parts, b, c, h, w, p.head, p.k, p.s,
            p.sgain, ptr_or_null(p.sgain_vec), ptr_or_null(p.soffset_vec), dt, st);
        if (rc != DDF_ERR_UNSUPPORTED) {
            check_status(rc);
            check_status(ddf_hip_channel_branch_parts(
                parts, n_parts, 1.0 / (double)(h * w), p.w1->data_ptr(), ptr_or_null(p.b1), p.w2->data_ptr(),
                ptr_or_null(p.b2), cf, b, c, mid, p.k, p.cgain, ptr_or_null(p.cgain_vec),
                ptr_or_null(p.coffset_vec), dt, st));
            pooled_on_the_way = true;
        }
    }
    if (!pooled_on_the_way) {
        const at::Tensor pooled = at::mean(x, {2, 3});
        check_status(ddf_hip_channel_branch(
            pooled.data_ptr(), p.w1->data_ptr(), ptr_or_null(p.b1), p.w2->data_ptr(), ptr_or_null(p.b2), cf, b, c, mid,
            p.k, p.cgain, ptr_or_null(p.cgain_vec), ptr_or_null(p.coffset_vec), dt, st));
        check_status(ddf_hip_spatial_branch(
            x.data_ptr(), p.ws->data_ptr(), ptr_or_null(p.bs), sf, b, c, h, w, p.head, p.k, p.s, p.sgain,
            ptr_or_null(p.sgain_vec), ptr_or_null(p.soffset_vec), dt, st));
    }
    // heads are folded into the batch: (b * head, c / head, h, w)
    check_status(ddf_hip_forward(x.data_ptr(), cf, sf, out.data_ptr(), b * p.head, c / p.head, h, w, p.k, p.d, p.s,
                                 p.combine, dt, DDF_VARIANT_AUTO, st));
    return out;
}

// A training step's layer.  What the backward pass wants of the forward (the filters, the
// un-normalised taps, the pooled and hidden vectors) sits in one buffer:
//   cf | sf | raw sf (features' dtype) | pooled | hidden | channel taps (fp32)
struct PackSizes {
    int64_t b, c, h, w, ho, wo, mid, kk;
    size_t cf, sf, pooled, hidden, taps, saved;
    PackSizes(const at::Tensor &x, int64_t mid_, int k, int s, int head) {
        b = x.size(0); c = x.size(1); h = x.size(2); w = x.size(3);
        ho = h / s; wo = w / s; mid = mid_; kk = (int64_t)k * k;
        const size_t esz = x.element_size();
        cf = aligned_bytes(b * c * kk * esz);
        sf = aligned_bytes(b * head * kk * ho * wo * esz);
        pooled = aligned_bytes(b * c * sizeof(float));
        hidden = aligned_bytes(b * mid * sizeof(float));
        taps = aligned_bytes(b * c * kk * sizeof(float));
        saved = cf + 2 * sf + pooled + hidden + taps;
    }
};

class PackAutograd : public torch::autograd::Function<PackAutograd> {
public:
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &ws, const at::Tensor &bs,
                              const at::Tensor &w1, const at::Tensor &b1, const at::Tensor &w2, const at::Tensor &b2,
                              const at::Tensor &gain_vec, double sgain, int64_t k, int64_t d, int64_t s,
                              int64_t head, int64_t combine) {
        const PackSizes z(x, w1.size(0), k, s, head);
        const int dt = dtype_code(x.scalar_type());
        c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(x.device());
        hipStream_t st = current_stream(x);
        at::Tensor out = new_tensor({z.b, z.c, z.ho, z.wo}, x.scalar_type(), x.device());
        at::Tensor saved = new_tensor({(int64_t)z.saved}, at::kByte, x.device());
        const int64_t cap = z.b * z.c * ((z.ho * z.wo + 63) / 64 + 1);
        at::Tensor parts = new_tensor({cap}, at::kFloat, x.device());
        char *q = static_cast<char *>(saved.data_ptr());
        void *cf = q, *sf = q + z.cf, *raw = q + z.cf + z.sf;
        float *pooled = reinterpret_cast<float *>(q + z.cf + 2 * z.sf);
        float *hidden = pooled + z.pooled / sizeof(float), *taps = hidden + z.hidden / sizeof(float);
        check_status(ddf_hip_pack_filters(x.data_ptr(), ws.data_ptr(), bs.data_ptr(), w1.data_ptr(), b1.data_ptr(),
                                          w2.data_ptr(), b2.data_ptr(), raw, sf, cf, pooled, hidden, taps,
                                          parts.data_ptr<float>(), cap, z.b, z.c, z.h, z.w, z.mid, (int)head, (int)k,
                                          (int)s, sgain, 1.0, gain_vec.data_ptr(), dt, st));
        check_status(ddf_hip_forward(x.data_ptr(), cf, sf, out.data_ptr(), z.b * head, z.c / head, z.h, z.w, (int)k,
                                     (int)d, (int)s, (int)combine, dt, DDF_VARIANT_AUTO, st));
        ctx->save_for_backward({x, ws, w1, w2, gain_vec, bs, b1, b2, saved});
        ctx->saved_data["conf"] = std::vector<int64_t>{k, d, s, head, combine};
        ctx->saved_data["sgain"] = sgain;
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto sv = ctx->get_saved_variables();
        const at::Tensor &x = sv[0], &ws = sv[1], &w1 = sv[2], &w2 = sv[3], &gain_vec = sv[4], &saved = sv[8];
        const auto conf = ctx->saved_data["conf"].toIntVector();
        const int k = (int)conf[0], d = (int)conf[1], s = (int)conf[2], head = (int)conf[3], combine = (int)conf[4];
        const double sgain = ctx->saved_data["sgain"].toDouble();
        const PackSizes z(x, w1.size(0), k, s, head);
        const int dt = dtype_code(x.scalar_type());
        const at::Tensor go = grads[0].to(x.scalar_type()).contiguous();
        c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(x.device());
        hipStream_t st = current_stream(x);
        const bool want_dx = ctx->needs_input_grad(0);
        const unsigned need = (want_dx ? DDF_NEED_DX : 0u) | DDF_NEED_DCF | DDF_NEED_DSF;
        const int64_t n = z.b * head, cg = z.c / head;
        const size_t op_bytes = aligned_bytes(ddf_hip_backward_spatial_norm_workspace_bytes(
            n, cg, z.h, z.w, k, d, s, combine, dt, need, DDF_VARIANT_AUTO));
        const size_t br_bytes = ddf_hip_pack_backward_workspace_bytes(z.b, z.c, z.h, z.w, z.mid, head, k, s, dt);
        at::Tensor work = new_tensor({(int64_t)(z.cf + z.sf + op_bytes + br_bytes)}, at::kByte, x.device());
        char *wq = static_cast<char *>(work.data_ptr());
        void *dcf = wq, *draw = wq + z.cf, *op_ws = wq + z.cf + z.sf, *br_ws = wq + z.cf + z.sf + op_bytes;
        char *q = static_cast<char *>(saved.data_ptr());
        void *cf = q, *sf = q + z.cf, *raw = q + z.cf + z.sf;
        float *pooled = reinterpret_cast<float *>(q + z.cf + 2 * z.sf);
        float *hidden = pooled + z.pooled / sizeof(float), *taps = hidden + z.hidden / sizeof(float);
        auto like = [&](const at::Tensor &t) { return new_tensor(t.sizes(), t.scalar_type(), x.device()); };
        at::Tensor dx;
        if (want_dx) dx = like(x);
        at::Tensor dws = like(ws), dw1 = like(w1), dw2 = like(w2),
                   dgain = like(gain_vec), dbs = like(sv[5]), db1 = like(sv[6]),
                   db2 = like(sv[7]);
        void *dxp = want_dx ? dx.data_ptr() : nullptr;
        check_status(ddf_hip_backward_spatial_norm(
            go.data_ptr(), x.data_ptr(), cf, sf, raw, dxp, dcf, draw, nullptr, op_ws, op_bytes, n, cg, z.h, z.w, k, d,
            s, combine, dt, need, head, sgain, nullptr, DDF_VARIANT_AUTO, st));
        check_status(ddf_hip_pack_backward(
            x.data_ptr(), dcf, draw, pooled, hidden, taps, ws.data_ptr(), w1.data_ptr(), w2.data_ptr(),
            gain_vec.data_ptr(), 1.0, dxp, dws.data_ptr(), dbs.data_ptr(), dw1.data_ptr(), db1.data_ptr(),
            dw2.data_ptr(), db2.data_ptr(), dgain.data_ptr(), br_ws, br_bytes, z.b, z.c, z.h, z.w, z.mid, head, k, s,
            dt, st));
        variable_list out = {dx, dws, dbs, dw1, db1, dw2, db2, dgain};
        if (at::GradMode::is_enabled()) {
            // (create_graph: there is no second derivative; asking for one raises)
            for (auto &t : out)
                if (t.defined()) t.set_requires_grad(true);
            auto node = std::make_shared<torch::autograd::DelayedError>(
                "trying to differentiate twice a function that was marked with @once_differentiable",
                (int64_t)out.size());
            out = (*node)(std::move(out));
        }
        out.resize(14);
        return out;
    }
};

// The same for a caller without a standing plan; refuses with an error what the kernels do not
// take.
inline at::Tensor pack_infer(const PackPlan &p, const at::Tensor &x) {
    TORCH_CHECK(x.is_cuda() && x.dim() == 4, "features must be a 4-d device tensor");
    const int dt = dtype_code(x.scalar_type());
    TORCH_CHECK(dt == DDF_F16 || dt == DDF_F32, "the branch kernels cover fp16 and fp32");
    const char *why = p.misfit(x);
    TORCH_CHECK(why == nullptr, why);
    return pack_run(p, x);
}

// DDFPack.forward through a plan: the result, or None where the plan does not (any longer)
// describe the layer or the native path does not cover the call.
inline py::object pack_forward(const PackPlan &p, const at::Tensor &x) {
    if (!p.holds() || !x.is_cuda() || x.dim() != 4 || dispatch_watched(x)) return py::none();
    const int dt = dtype_code(x.scalar_type());
    // (a size the stride does not divide fails in the layer's own code, as in the reference
    // at ddf/ddf.py:215-218)
    if ((dt != DDF_F16 && dt != DDF_F32) || x.size(2) % p.s || x.size(3) % p.s || p.misfit(x))
        return py::none();
    if (!(at::GradMode::is_enabled() && p.wants_gradients(x))) return py::cast(pack_run(p, x));
    // Training: the stock configuration only (constant spatial gain, learned channel gain, no
    // offsets, biases present), everything trained.
    if (!p.fuse_norm || p.sgain_vec.defined() || p.soffset_vec.defined() || p.coffset_vec.defined() ||
        !p.cgain_vec.defined())
        return py::none();
    for (const TensorRef *t : {&p.ws, &p.bs, &p.w1, &p.b1, &p.w2, &p.b2, &p.cgain_vec})
        if (!t->defined() || !(*t)->requires_grad()) return py::none();
    if (at::autocast::is_autocast_enabled(at::kCUDA)) return py::none();
    if (x.numel() == 0) return py::none();
    // (the streaming kernel's addresses: weights in whole words, features in whole vectors)
    const bool covered =
        reinterpret_cast<uintptr_t>(p.ws->data_ptr()) % 4 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
        ddf_hip_pack_backward_workspace_bytes(x.size(0), x.size(1), x.size(2), x.size(3), p.w1->size(0), p.head, p.k,
                                              p.s, dt) > 0;
    if (!covered) return py::none();
    return py::cast(PackAutograd::apply(x.contiguous(), *p.ws, *p.bs, *p.w1, *p.b1, *p.w2, *p.b2, *p.cgain_vec, p.sgain,
                                        (int64_t)p.k, (int64_t)p.d, (int64_t)p.s, (int64_t)p.head,
                                        (int64_t)p.combine));
}

}  // namespace ddf_torch
