// Inference of a whole DDF-ResNet (ddf_resnet.py:34-111 of the reference) as one native
// call: the launches of csrc/ddf_net.hip on channels-last activations in one workspace.
#pragma once

#include "module_guard.h"

namespace ddf_torch {

// A convolution with what follows it: (weight, conv bias, BatchNorm weight, bias, running
// mean, running variance); missing ones undefined.
struct NetLayer {
    TensorRef t[6];
    ddf_net_norm_t norm() const {
        return ddf_net_norm_t{ptr_or_null(t[2]), ptr_or_null(t[3]), ptr_or_null(t[4]), ptr_or_null(t[5]),
                              ptr_or_null(t[1]), eps};
    }
    float eps = 0.f;
};

struct NetBlock {
    NetLayer conv1, conv3, down;
    NetLayer bn2;                 // (no convolution of its own)
    TensorRef ws, bs, w1, b1, w2, b2, cgain, coffset;
    double sgain, cgain_const;
    int stride, combine;
    int64_t width, mid;
};

using NetLayerArgs = std::pair<py::list, double>;

struct NetPlan {
    Refs refs;
    ModuleGuard *guard;              // (owned by refs)
    NetLayer stem, fc;
    std::vector<NetBlock> blocks;
    // every tensor and the sizes it must have
    std::vector<std::pair<TensorRef, std::vector<int64_t>>> all;

    explicit NetPlan(const py::object &guard_) : guard(guard_.cast<ModuleGuard *>()) { refs.add(guard_.ptr()); }
    int traverse(visitproc visit, void *arg) const { return refs.traverse(visit, arg); }
    void clear() {
        guard = nullptr;
        stem = fc = NetLayer();
        blocks.clear();
        all.clear();
        refs.clear();
    }
    bool holds() const { return guard && guard->holds(); }
    void expect(const TensorRef &t, std::vector<int64_t> sizes) {
        if (t.defined()) all.emplace_back(t, std::move(sizes));
    }
    // A convolution of these sizes (none: only what follows it) with what follows it.
    NetLayer layer(const NetLayerArgs &a, std::vector<int64_t> sizes, int64_t channels) {
        NetLayer l;
        const std::vector<TensorRef> t = tensor_refs(refs, a.first);
        TORCH_CHECK(t.size() == 6, "six tensors per layer expected");
        for (int i = 0; i < 6; ++i) {
            l.t[i] = t[i];
            expect(l.t[i], i == 0 ? sizes : std::vector<int64_t>{channels});
        }
        l.eps = (float)a.second;
        return l;
    }
    void set_ends(const NetLayerArgs &s, const NetLayerArgs &f, int64_t features, int64_t classes) {
        stem = layer(s, {64, 3, 7, 7}, 64);
        fc = layer(f, {classes, features}, classes);
    }
    // A bottleneck of `in` -> `width` -> `out` channels with `mid` hidden ones.
    void add_block(const NetLayerArgs &conv1, const NetLayerArgs &bn2, const NetLayerArgs &conv3,
                   const NetLayerArgs &down, const py::list &branches, double sgain,
                   double cgain, int stride, const std::string &combine, int64_t in, int64_t width, int64_t out,
                   int64_t mid) {
        NetBlock b;
        b.conv1 = layer(conv1, {width, in, 1, 1}, width);
        b.bn2 = layer(bn2, {}, width);
        b.conv3 = layer(conv3, {out, width, 1, 1}, out);
        b.down = layer(down, {out, in, 1, 1}, out);
        TensorRef *const to[8] = {&b.ws, &b.bs, &b.w1, &b.b1, &b.w2, &b.b2, &b.cgain, &b.coffset};
        const std::vector<int64_t> sizes[8] = {{9, width, 1, 1}, {9}, {mid, width, 1, 1}, {mid}, {9 * width, mid, 1, 1},
                                               {9 * width}, {9 * width}, {9 * width}};
        const std::vector<TensorRef> t = tensor_refs(refs, branches);
        TORCH_CHECK(t.size() == 8, "eight branch tensors expected");
        for (int i = 0; i < 8; ++i) {
            *to[i] = t[i];
            expect(*to[i], sizes[i]);
        }
        b.sgain = sgain; b.cgain_const = cgain;
        b.stride = stride;
        b.combine = combine_code(combine);
        b.width = width;
        b.mid = mid;
        blocks.push_back(b);
    }
    // Why the native inference cannot run this input with the network's tensors as they are now
    // (parameters may have been resized, moved or re-laid in place), or null.
    const char *misfit(const at::Tensor &x) const {
        if (x.scalar_type() != at::kHalf || x.dim() != 4 || x.size(1) != 3) return "images in fp16 expected";
        // (2^27 pixels: 32-bit offsets inside a sample of the stem and of the widest activation
        // under a 3 x 3, twice the channels at a quarter of the image's rows and columns)
        if (x.size(0) < 1 || x.size(0) > 65535 || x.size(2) % 32 || x.size(3) % 32 || x.numel() == 0 ||
            x.size(2) * x.size(3) >= (int64_t(1) << 27))
            return "image sizes not covered";
        const bool grad = at::GradMode::is_enabled();
        if ((grad && x.requires_grad()) || has_tangent(x)) return "gradients wanted";
        const auto dev = x.device();
        for (const auto &[ref, sizes] : all) {
            const at::Tensor &t = *ref;
            if (t.scalar_type() != at::kHalf || t.device() != dev) return "parameters must be fp16 and with the images";
            if (t.sizes() != sizes) return "parameters do not fit each other";
            if (!t.is_contiguous() || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return "parameters must be laid out densely";
            if ((grad && t.requires_grad()) || has_tangent(t)) return "gradients wanted";
            if (t.unsafeGetTensorImpl()->is_python_dispatch()) return "parameters must be plain tensors";
        }
        return nullptr;
    }
};

// A call whose sizes the library refuses, before or between launches.
struct NotCovered {};
inline void covered(int status) {
    if (status == DDF_ERR_UNSUPPORTED) throw NotCovered();
    check_status(status);
}

// Logits, or None where the plan does not (any longer) describe the network or the native
// path does not cover the call.
inline py::object net_forward(const NetPlan &p, const at::Tensor &input) {
    if (!input.is_cuda() || at::autocast::is_autocast_enabled(at::kCUDA) || dispatch_watched(input) || !p.holds() ||
        p.misfit(input))
        return py::none();
    const auto dev = input.device();
    const at::Tensor x = input.contiguous();
    const int64_t n = x.size(0), h0 = x.size(2), w0 = x.size(3);
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(dev);
    hipStream_t st = current_stream(x);

    // One workspace: a block's input and output trade places (a block without a projection
    // adds its result in place), between them the narrow activations and the filters.
    int64_t wide = 0, narrow = 0, taps = 0, filters = 0, parts = 0, totals = 0;
    // (more partial sums of the pooled vectors than the channel branch is left become totals)
    struct Parts { int count; bool summed; };
    // (0: b's last convolution and the first one of the block behind it are launches of their own)
    auto chain_parts = [n, &p](size_t i, int64_t ho, int64_t wo, int64_t c) -> int64_t {
        const NetBlock &b = p.blocks[i];
        const bool down = b.down.t[0].defined();
        if (i + 1 == p.blocks.size() || (down && b.stride != 1)) return 0;
        return ddf_hip_net_conv_chain_parts(n, ho, wo, b.width, down ? c : 0, b.conv3.t[0]->size(0), p.blocks[i + 1].width);
    };
    // (whether that launch makes block i's spatial branch and dynamic filter, too)
    auto filtered = [n, &p](size_t i, int64_t ho, int64_t wo, int64_t c) {
        const NetBlock &b = p.blocks[i];
        return b.stride == 1 && ddf_hip_net_filter_chain_parts(n, ho, wo, b.width, b.down.t[0].defined() ? c : 0,
                                                               b.conv3.t[0]->size(0), p.blocks[i + 1].width) > 0;
    };
    // chained: what the launch that made b's first results has left, 0 where that is one of its own
    auto parts_of = [n](const NetBlock &b, int64_t h, int64_t w, int64_t c, int64_t chained) {
        const int64_t count = chained ? chained : ddf_hip_net_conv_pool_parts(n, h, w, c, b.width);
        return Parts{(int)count, count > ddf_hip_net_parts_left(n, b.width, b.mid)};
    };
    {
        int64_t h = h0 / 4, w = w0 / 4, c = 64, chained = 0;
        wide = n * h * w * 64;
        for (size_t i = 0; i < p.blocks.size(); ++i) {
            const NetBlock &b = p.blocks[i];
            const int64_t ho = h / b.stride, wo = w / b.stride;
            narrow = std::max(narrow, n * h * w * b.width);
            wide = std::max(wide, n * ho * wo * b.conv3.t[0]->size(0));
            taps = std::max(taps, n * ho * wo * 12);
            filters = std::max(filters, n * b.width * 9);
            const Parts of = parts_of(b, h, w, c, chained);
            chained = chain_parts(i, ho, wo, c);
            parts = std::max(parts, n * b.width * of.count);
            if (of.summed) totals = std::max(totals, n * b.width);
            c = b.conv3.t[0]->size(0);
            h = ho; w = wo;
        }
    }
    const size_t wide_b = aligned_bytes(wide * 2), narrow_b = aligned_bytes(narrow * 2), taps_b = aligned_bytes(taps * 2),
                 filters_b = aligned_bytes(filters * 2), parts_b = aligned_bytes(parts * 4),
                 totals_b = aligned_bytes(totals * 4);
    at::Tensor work = new_tensor({(int64_t)(2 * wide_b + 2 * narrow_b + taps_b + filters_b + parts_b + totals_b)},
                                 at::kByte, x.device());
    char *q = static_cast<char *>(work.data_ptr());
    void *cur = q, *other = q + wide_b, *t1 = q + 2 * wide_b, *t2 = q + 2 * wide_b + narrow_b;
    void *sf = q + 2 * wide_b + 2 * narrow_b, *cf = static_cast<char *>(sf) + taps_b;
    float *pp = reinterpret_cast<float *>(static_cast<char *>(cf) + filters_b), *pt = pp + parts_b / sizeof(float);
    at::Tensor logits = new_tensor({n, p.fc.t[0]->size(0)}, at::kHalf, dev);
    try {
        py::gil_scoped_release release;    // (a network's launches take a while)
        ddf_net_norm_t nm = p.stem.norm();
        covered(ddf_hip_net_stem(x.data_ptr(), p.stem.t[0]->data_ptr(), &nm, cur, n, h0, w0, st));
        int64_t h = h0 / 4, w = w0 / 4, c = 64, chained = 0;
        for (size_t i = 0; i < p.blocks.size(); ++i) {
            const NetBlock &b = p.blocks[i];
            const int64_t ho = h / b.stride, wo = w / b.stride, width = b.width, wide_c = b.conv3.t[0]->size(0);
            if (!chained) {
                nm = b.conv1.norm();
                covered(ddf_hip_net_conv_pool(cur, b.conv1.t[0]->data_ptr(), &nm, t1, pp, n, h, w, c, width, 1, st));
            }
            const Parts of = parts_of(b, h, w, c, chained);
            chained = chain_parts(i, ho, wo, c);
            if (of.summed) covered(ddf_hip_net_sum_parts(pp, of.count, pt, n, width, st));
            const float *const pooled = of.summed ? pt : pp;
            const int count = of.summed ? 1 : of.count;
            const bool fused = chained && filtered(i, ho, wo, c);
            nm = b.bn2.norm();
            if (fused)
                covered(ddf_hip_channel_branch_parts(pooled, count, 1.0 / (double)(h * w), b.w1->data_ptr(), ptr_or_null(b.b1),
                                                     b.w2->data_ptr(), ptr_or_null(b.b2), cf, n, width, b.mid, 3, b.cgain_const,
                                                     ptr_or_null(b.cgain), ptr_or_null(b.coffset), DDF_F16, st));
            else
                covered(ddf_hip_net_ddf(t1, b.ws->data_ptr(), ptr_or_null(b.bs), sf, b.sgain, pooled, count,
                                        b.w1->data_ptr(), ptr_or_null(b.b1), b.w2->data_ptr(), ptr_or_null(b.b2), cf, b.mid,
                                        b.cgain_const, ptr_or_null(b.cgain), ptr_or_null(b.coffset), &nm, t2, n, h, w, width,
                                        b.stride, b.combine, st));
            const ddf_net_norm_t nm2 = nm;
            nm = b.conv3.norm();
            const ddf_net_norm_t down = b.down.norm();
            if (chained) {
                const NetBlock &next = p.blocks[i + 1];
                const ddf_net_norm_t nm1 = next.conv1.norm();
                const bool side = b.down.t[0].defined();
                void *to = side ? other : cur;
                const void *const res = side ? nullptr : cur, *const side_x = side ? cur : nullptr;
                if (fused) {
                    covered(ddf_hip_net_filter_chain(t1, cf, b.ws->data_ptr(), ptr_or_null(b.bs), b.sgain, &nm2, b.combine,
                                                     b.conv3.t[0]->data_ptr(), &nm, res, side_x, ptr_or_null(b.down.t[0]), &down, side ? c : 0, to, next.conv1.t[0]->data_ptr(),
                                                     &nm1, t2, pp, n, ho, wo, width, wide_c, next.width, st));
                    std::swap(t1, t2);
                } else {
                    covered(ddf_hip_net_conv_chain(t2, b.conv3.t[0]->data_ptr(), &nm, res, side_x, ptr_or_null(b.down.t[0]),
                                                   &down, side ? c : 0, to, next.conv1.t[0]->data_ptr(), &nm1, t1, pp, n, ho, wo,
                                                   width, wide_c, next.width, st));
                }
                if (side) std::swap(cur, other);
            } else if (b.down.t[0].defined()) {
                covered(ddf_hip_net_conv_pair(t2, b.conv3.t[0]->data_ptr(), &nm, width, cur,
                                                   b.down.t[0]->data_ptr(), &down, h, w, c, b.stride, other, n, wide_c, 1,
                                                   st));
                std::swap(cur, other);
            } else {
                covered(ddf_hip_net_conv(t2, b.conv3.t[0]->data_ptr(), &nm, cur, cur, n, ho, wo, width, wide_c, 1, 1,
                                              st));
            }
            h = ho; w = wo; c = wide_c;
        }
        covered(ddf_hip_net_pool(cur, other, n, h * w, c, st));
        nm = p.fc.norm();
        covered(ddf_hip_net_conv(other, p.fc.t[0]->data_ptr(), &nm, nullptr, logits.data_ptr(), n, 1, 1, c,
                                      logits.size(1), 1, 0, st));
    } catch (const NotCovered &) {
        return py::none();    // (the modules run; what was written so far is dropped)
    }
    return py::cast(logits);
}

}  // namespace ddf_torch
