// Inference of a whole DDF-ResNet (ddf_resnet.py:34-111 of the reference) as one native
// call: the launches of csrc/ddf_net.hip on channels-last activations in one workspace.
#pragma once

#include "module_guard.h"

namespace ddf_torch {

// A convolution with what follows it: (weight, conv bias, BatchNorm weight, bias, running
// mean, running variance); missing ones undefined.
struct NetLayer {
    at::Tensor t[6];
    ddf_net_norm_t norm() const {
        auto p = [](const at::Tensor &x) -> const void * { return x.defined() ? x.data_ptr() : nullptr; };
        return ddf_net_norm_t{p(t[2]), p(t[3]), p(t[4]), p(t[5]), p(t[1]), eps};
    }
    float eps = 0.f;
};

struct NetBlock {
    NetLayer conv1, conv3, down;
    NetLayer bn2;                 // (no convolution of its own)
    at::Tensor ws, bs, w1, b1, w2, b2, cgain, coffset;
    double sgain, cgain_const;
    int stride, combine;
    int64_t width, mid;
};

using NetLayerArgs = std::pair<std::vector<c10::optional<at::Tensor>>, double>;

struct NetPlan {
    std::shared_ptr<ModuleGuard> guard;
    NetLayer stem, fc;
    std::vector<NetBlock> blocks;
    std::vector<at::Tensor> all;

    explicit NetPlan(std::shared_ptr<ModuleGuard> guard_) : guard(std::move(guard_)) {}

    NetLayer layer(const NetLayerArgs &a) {
        NetLayer l;
        TORCH_CHECK(a.first.size() == 6, "six tensors per layer expected");
        for (int i = 0; i < 6; ++i)
            if (a.first[i].has_value() && a.first[i]->defined()) {
                l.t[i] = *a.first[i];
                all.push_back(l.t[i]);
            }
        l.eps = (float)a.second;
        return l;
    }
    void set_ends(const NetLayerArgs &s, const NetLayerArgs &f) { stem = layer(s); fc = layer(f); }
    void add_block(const NetLayerArgs &conv1, const NetLayerArgs &bn2, const NetLayerArgs &conv3,
                   const NetLayerArgs &down, std::vector<c10::optional<at::Tensor>> branches, double sgain,
                   double cgain, int stride, const std::string &combine) {
        NetBlock b;
        b.conv1 = layer(conv1); b.bn2 = layer(bn2); b.conv3 = layer(conv3); b.down = layer(down);
        at::Tensor *const to[8] = {&b.ws, &b.bs, &b.w1, &b.b1, &b.w2, &b.b2, &b.cgain, &b.coffset};
        TORCH_CHECK(branches.size() == 8, "eight branch tensors expected");
        for (int i = 0; i < 8; ++i)
            if (branches[i].has_value() && branches[i]->defined()) {
                *to[i] = *branches[i];
                all.push_back(*to[i]);
            }
        b.sgain = sgain; b.cgain_const = cgain;
        b.stride = stride;
        b.combine = combine == "add" ? DDF_ADD : DDF_MUL;
        b.width = b.conv1.t[0].size(0);
        b.mid = b.w1.size(0);
        blocks.push_back(b);
    }
};

// Logits, or None where the plan does not (any longer) describe the network or the native
// path does not cover the call.
inline py::object net_forward(const NetPlan &p, const at::Tensor &input) {
    if (!input.is_cuda() || input.scalar_type() != at::kHalf || input.dim() != 4 || input.size(1) != 3 ||
        input.size(0) < 1 || input.size(0) > 65535 || input.size(2) % 32 || input.size(3) % 32 || input.numel() == 0 ||
        at::autocast::is_autocast_enabled(at::kCUDA) || !p.guard->holds())
        return py::none();
    const auto dev = input.device();
    const bool grad = at::GradMode::is_enabled();
    if (grad && input.requires_grad()) return py::none();
    for (const at::Tensor &t : p.all)
        if (t.scalar_type() != at::kHalf || t.device() != dev || !t.is_contiguous() || (grad && t.requires_grad()) ||
            reinterpret_cast<uintptr_t>(t.data_ptr()) % 16)
            return py::none();
    const at::Tensor x = input.contiguous();
    const int64_t n = x.size(0), h0 = x.size(2), w0 = x.size(3);
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(dev);
    hipStream_t st = current_stream(x);

    // One workspace: a block's input and output trade places (a block without a projection
    // adds its result in place), between them the narrow activations and the filters.
    int64_t wide = 0, narrow = 0, taps = 0, filters = 0, parts = 0;
    {
        int64_t h = h0 / 4, w = w0 / 4;
        wide = n * h * w * 64;
        for (const NetBlock &b : p.blocks) {
            const int64_t ho = h / b.stride, wo = w / b.stride;
            narrow = std::max(narrow, n * h * w * b.width);
            wide = std::max(wide, n * ho * wo * b.conv3.t[0].size(0));
            taps = std::max(taps, n * ho * wo * 12);
            filters = std::max(filters, n * b.width * 9);
            parts = std::max(parts, n * b.width * 8);
            h = ho; w = wo;
        }
    }
    const size_t wide_b = aligned_bytes(wide * 2), narrow_b = aligned_bytes(narrow * 2), taps_b = aligned_bytes(taps * 2),
                 filters_b = aligned_bytes(filters * 2), parts_b = aligned_bytes(parts * 4);
    at::Tensor work = new_tensor({(int64_t)(2 * wide_b + 2 * narrow_b + taps_b + filters_b + parts_b)}, at::kByte, x.device());
    char *q = static_cast<char *>(work.data_ptr());
    void *cur = q, *other = q + wide_b, *t1 = q + 2 * wide_b, *t2 = q + 2 * wide_b + narrow_b;
    void *sf = q + 2 * wide_b + 2 * narrow_b, *cf = static_cast<char *>(sf) + taps_b;
    float *pp = reinterpret_cast<float *>(static_cast<char *>(cf) + filters_b);
    at::Tensor logits = new_tensor({n, p.fc.t[0].size(0)}, at::kHalf, dev);
    {
        py::gil_scoped_release release;    // (a network's launches take a while)
        ddf_net_norm_t nm = p.stem.norm();
        check_status(ddf_hip_net_stem(x.data_ptr(), p.stem.t[0].data_ptr(), &nm, cur, n, h0, w0, st));
        int64_t h = h0 / 4, w = w0 / 4, c = 64;
        for (const NetBlock &b : p.blocks) {
            const int64_t ho = h / b.stride, wo = w / b.stride, width = b.width, wide_c = b.conv3.t[0].size(0);
            nm = b.conv1.norm();
            check_status(ddf_hip_net_conv(cur, b.conv1.t[0].data_ptr(), &nm, nullptr, t1, n, h, w, c, width, 1, 1, st));
            int n_parts = 0;
            check_status(ddf_hip_net_spatial(t1, b.ws.data_ptr(), ptr_or_null(b.bs), sf, pp, &n_parts, n, h, w, width,
                                             b.stride, b.sgain, st));
            check_status(ddf_hip_channel_branch_parts(
                pp, n_parts, 1.0 / (double)(h * w), b.w1.data_ptr(), ptr_or_null(b.b1), b.w2.data_ptr(),
                ptr_or_null(b.b2), cf, n, width, b.mid, 3, b.cgain_const, ptr_or_null(b.cgain), ptr_or_null(b.coffset),
                DDF_F16, st));
            nm = b.bn2.norm();
            check_status(ddf_hip_net_filter(t1, cf, sf, &nm, t2, n, h, w, width, b.stride, b.combine, st));
            nm = b.conv3.norm();
            if (b.down.t[0].defined()) {
                const ddf_net_norm_t down = b.down.norm();
                check_status(ddf_hip_net_conv_pair(t2, b.conv3.t[0].data_ptr(), &nm, width, cur,
                                                   b.down.t[0].data_ptr(), &down, h, w, c, b.stride, other, n, wide_c, 1,
                                                   st));
                std::swap(cur, other);
            } else {
                check_status(ddf_hip_net_conv(t2, b.conv3.t[0].data_ptr(), &nm, cur, cur, n, ho, wo, width, wide_c, 1, 1,
                                              st));
            }
            h = ho; w = wo; c = wide_c;
        }
        check_status(ddf_hip_net_pool(cur, other, n, h * w, c, st));
        nm = p.fc.norm();
        check_status(ddf_hip_net_conv(other, p.fc.t[0].data_ptr(), &nm, nullptr, logits.data_ptr(), n, 1, 1, c,
                                      logits.size(1), 1, 0, st));
    }
    return py::cast(logits);
}

}  // namespace ddf_torch
