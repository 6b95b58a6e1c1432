// Host path of the shared MLPs (include/tk3d_mlp.h): which products, sums and small kernels a
// chain of "1x1 convolution, batch norm, ReLU" layers is made of, forward and backward.
#include "native.h"
#include "tk3d_mlp.h"

#include <ATen/TracerMode.h>
#include <ATen/native/Normalization.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/autograd.h>

namespace tk3d {

bool plain(const Tensor &t)
{
    using c10::DispatchKey;
    constexpr c10::DispatchKeySet odd({DispatchKey::Python, DispatchKey::PythonTLSSnapshot,
                                       DispatchKey::FuncTorchBatched,
                                       DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize,
                                       DispatchKey::Conjugate, DispatchKey::Negative,
                                       DispatchKey::ZeroTensor});
    return !t.key_set().has_any(odd) && !t._fw_grad(0).defined();
}

bool watched()
{
    return c10::impl::tls_is_dispatch_key_included(
               c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           c10::impl::TorchDispatchModeTLS::any_modes_set() || at::tracer::impl::is_dispatch_enabled();
}

variable_list dense(variable_list saved)
{
    for (Tensor &t : saved)
        if (t.defined())
            t = t.contiguous();
    return saved;
}

namespace {

using torch::autograd::AutogradContext;

float *f32(const Tensor &t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

// Whether the gradients of a training step are those of the stock modules, for rows of P values. On
// rows whose length is no multiple of four the library's batch norm backward loses values where
// they are longer than 1024, in large batches longer than 512: dgamma and dbeta of [2, 64, 1025] and
// of [40, 64, 515] are 1e-1 off from float64, 1e-7 at [2, 64, 1023] and [40, 64, 511]. The kernels
// here are not, but a step on such clouds goes on giving what it gave.
bool same_gradients(int64_t P) { return P <= 512 || P % 4 == 0; }

// Whether training goes through the library's batch norm, whose order of operations the backward
// repeats where it asks for a sign (normalised() in mlp_common.h). torch has a kernel of its own, which
// rounds differently, for what MIOpen does not take and where the user has switched it off
// (torch.backends.cudnn.enabled).
bool library_norm(const Tensor &like, at::IntArrayRef shape, const Tensor *params, const Tensor *buffers,
                  double eps)
{
    const Tensor y = at::empty({}, like.options()).expand(shape);
    return at::native::_select_batch_norm_backend(y, params[1], params[2], buffers[0], buffers[1], true,
                                                  eps) == at::native::BatchNormBackend::Miopen;
}

// What a chain is applied to and how.
struct Call {
    // dense input: x [B, C, P] and, if defined, x2 [B, C2, P] behind its channels
    Tensor x, x2;
    // grouped input: features [B, C, N] (x above, may be undefined), xyz [B, 3, N],
    // centre [B, 3, M], index [B, M, S]
    Tensor xyz, centre, index;
    int64_t pool = 0;  // maximum over groups of this many consecutive positions, 0: none
    bool whole = false;  // maximum over all positions (pool is their number), and its place
    int64_t rows = 0;  // of a dense input given as [B, C, rows, P / rows]
    bool training = false;
    std::vector<double> eps, momentum;
    std::vector<Tensor> params;   // weight, gamma, beta of every layer
    std::vector<Tensor> buffers;  // running mean, running variance, batch count of every layer

    bool grouped() const { return xyz.defined(); }
    int64_t layers() const { return (int64_t)params.size() / 3; }
    const Tensor &weight(int64_t l) const { return params[3 * l]; }
    int64_t out_channels(int64_t l) const { return params[3 * l].size(0); }
    int64_t in_channels(int64_t l) const { return params[3 * l].size(1); }
    int64_t batch() const { return grouped() ? xyz.size(0) : x.size(0); }
    int64_t positions() const { return grouped() ? index.size(1) * index.size(2) : x.size(2); }
    Tensor like() const { return grouped() ? xyz : x; }
};

// What the backward needs besides the call: the product of every layer (of a pooled last layer
// the extremes, and their places), and the statistics it was normalised with (training: `var` is
// 1 / sqrt(variance + eps), as batch norm saves it).
struct Kept {
    std::vector<Tensor> y, mean, var;
    Tensor arg;  // uint8; of a maximum over all positions int32
};

tk3d_mlp_norm norm_of(const Call &c, const Kept &k, int64_t l)
{
    return {f32(k.mean[l]), f32(k.var[l]), f32(c.params[3 * l + 1]), f32(c.params[3 * l + 2]),
            c.training ? -1.0f : (float)c.eps[l]};
}

tk3d_mlp_source source(const Tensor &x, const float *w, int64_t wk, int64_t wc)
{
    tk3d_mlp_source s{};
    s.x = f32(x);
    s.w = w;
    s.batch_stride = x.size(1) * x.size(2);
    s.K = (int32_t)x.size(1);
    s.wk = (int32_t)wk;
    s.wc = (int32_t)wc;
    return s;
}

tk3d_mlp_product product(int64_t B, int64_t C, int64_t P)
{
    tk3d_mlp_product p{};
    p.B = (int32_t)B;
    p.C = p.C0 = (int32_t)C;
    p.P = (int32_t)P;
    p.group = 1;
    p.M = (int32_t)P;
    return p;
}

// Partial sums [C][slots] of (double, double).
Tensor partial_sums(const Tensor &like, int64_t C, int slots)
{
    return at::empty({C, slots, 2}, like.options().dtype(at::kDouble));
}

// Runs a product with partial sums; returns them and their number per channel.
std::pair<Tensor, int> summed_product(int in, int out, tk3d_mlp_product &p, const Tensor &like,
                                      void *stream)
{
    const int slots = tk3d_mlp_product_slots(in, out, &p);
    const Tensor partial = partial_sums(like, p.C, slots);
    p.partial = partial.data_ptr();
    done(tk3d_mlp_product_f32(in, out, &p, stream), "tk3d_mlp_product_f32");
    return {partial, slots};
}

void run_product(int in, int out, tk3d_mlp_product &p, void *stream)
{
    done(tk3d_mlp_product_f32(in, out, &p, stream), "tk3d_mlp_product_f32");
}

// The product of the features with their weights in the first layer behind a grouping: [B, N, C], or
// undefined without features.
Tensor feature_product(const Call &c)
{
    if (!c.x.defined())
        return {};
    const int64_t B = c.batch(), C = c.out_channels(0), N = c.xyz.size(2);
    const Tensor u = at::empty({B, N, C}, c.xyz.options());
    tk3d_mlp_product q = product(B, C, N);
    q.src[0] = source(c.x, f32(c.weight(0)), 1, c.in_channels(0));
    q.out = f32(u);
    run_product(TK3D_MLP_IN_RAW, TK3D_MLP_OUT_POINTS, q, stream_of(c.xyz));
    return u;
}

// The product of the first layer behind a grouping, without the grouped tensor.
void first_grouped(const Call &c, const Tensor &y)
{
    const int64_t B = c.batch(), C = c.out_channels(0), K = c.in_channels(0);
    const int64_t M = c.index.size(1), S = c.index.size(2), N = c.xyz.size(2);
    const float *w = f32(c.weight(0));
    void *stream = stream_of(c.xyz);
    const Tensor u = feature_product(c);
    done(tk3d_mlp_group_f32(f32(u), f32(c.xyz), f32(c.centre), c.index.data_ptr<int64_t>(), w + (K - 3),
                            (int)K, (int)B, (int)C, (int)N, (int)M, (int)S, f32(y), stream),
         "tk3d_mlp_group_f32");
}

// Evaluation without gradients: every layer leaves its activations.
Tensor evaluate(const Call &c)
{
    const int64_t B = c.batch(), P = c.positions(), L = c.layers();
    const Tensor like = c.like();
    void *stream = stream_of(like);
    Kept k;
    for (int64_t l = 0; l < L; ++l) {
        k.mean.push_back(c.buffers[3 * l]);
        k.var.push_back(c.buffers[3 * l + 1]);
    }
    if (c.grouped() && c.pool && L == 3) {
        tk3d_mlp_grouped_pool p{};
        p.xyz = f32(c.xyz);
        p.centre = f32(c.centre);
        p.index = c.index.data_ptr<int64_t>();
        p.ldw = (int32_t)c.in_channels(0);
        p.wx = f32(c.weight(0)) + (p.ldw - 3);
        p.w2 = f32(c.weight(1));
        p.w3 = f32(c.weight(2));
        p.B = (int32_t)B;
        p.N = (int32_t)c.xyz.size(2);
        p.M = (int32_t)c.index.size(1);
        p.S = (int32_t)c.index.size(2);
        for (int l = 0; l < 3; ++l) {
            p.norm[l] = norm_of(c, k, l);
            p.C[l] = (int32_t)c.out_channels(l);
        }
        if (tk3d_mlp_grouped_pool_supported(&p)) {
            const Tensor u = feature_product(c), out = at::empty({B, p.C[2], p.M}, like.options());
            p.u = f32(u);
            p.out = f32(out);
            done(tk3d_mlp_grouped_pool_f32(&p, stream), "tk3d_mlp_grouped_pool_f32");
            return out;
        }
    }
    Tensor h;
    for (int64_t l = 0; l < L; ++l) {
        const int64_t C = c.out_channels(l), K = c.in_channels(l);
        const float *w = f32(c.weight(l));
        tk3d_mlp_product p = product(B, C, P);
        p.out_norm = norm_of(c, k, l);
        if (l == 0 && c.grouped()) {
            h = at::empty({B, C, P}, like.options());
            first_grouped(c, h);
            continue;
        }
        int in = TK3D_MLP_IN_RAW, out = TK3D_MLP_OUT_EVAL;
        if (l == 0) {
            p.src[0] = source(c.x, w, 1, K);
            if (c.x2.defined()) {
                in = TK3D_MLP_IN_RAW2;
                p.src[1] = source(c.x2, w + c.x.size(1), 1, K);
            }
        } else {
            p.src[0] = source(h, w, 1, K);
            if (l == 1 && c.grouped()) {
                in = TK3D_MLP_IN_ACT;
                p.in_norm = norm_of(c, k, 0);
            }
        }
        Tensor next;
        if (c.pool && l == L - 1) {
            out = TK3D_MLP_OUT_POOL_EVAL;
            p.group = (int32_t)c.pool;
            p.M = (int32_t)(P / c.pool);
            next = at::empty({B, C, p.M}, like.options());
        } else {
            next = at::empty({B, C, P}, like.options());
        }
        p.out = f32(next);
        run_product(in, out, p, stream);
        h = next;
    }
    return h;
}

// A layer of a training step: the library's product, and its batch norm with the statistics of this
// batch (the running ones updated) behind it.
struct Normalised {
    Tensor y, mean, inv_std;
    Tensor z;                 // the library's, where it took the batch norm
    tk3d_mlp_batch_norm norm{};  // else what the pass over y needs
    Tensor partial;
    int64_t *count = nullptr;    // the norm's count of batches, if that pass counts

    // Whether the pass over y takes the count along: a single int64 beside y. (Its version goes up
    // as with an addition in place.)
    bool counts(const Tensor &batches)
    {
        if (z.defined() || batches.device() != y.device() || batches.scalar_type() != at::kLong ||
            batches.numel() != 1)
            return false;
        batches.unsafeGetTensorImpl()->bump_version();
        count = batches.data_ptr<int64_t>();
        return true;
    }
};

Normalised stock_layer(const Tensor &h, const Tensor &weight, const Tensor &gamma, const Tensor &beta,
                       const Tensor &running_mean, const Tensor &running_var, double momentum,
                       double eps)
{
    Normalised n;
    n.y = h.dim() == 4 ? at::conv2d(h, weight) : at::conv1d(h, weight);
    const int64_t B = n.y.size(0), C = n.y.size(1), P = n.y.numel() / (B * C);
    if (n.y.is_contiguous() && tk3d_mlp_batch_norm_supported(B, C, P)) {
        n.mean = at::empty({C}, n.y.options());
        n.inv_std = at::empty({C}, n.y.options());
        n.partial = at::empty({tk3d_mlp_batch_norm_partial_bytes(C)}, n.y.options().dtype(at::kByte));
        n.norm = {n.partial.data_ptr(), f32(gamma), f32(beta), f32(running_mean), f32(running_var),
                  f32(n.mean), f32(n.inv_std), eps, (float)momentum, (int32_t)B, (int32_t)C, (int32_t)P};
        done(tk3d_mlp_batch_sums_f32(f32(n.y), (int)B, (int)C, (int)P, n.partial.data_ptr(),
                                     stream_of(n.y)),
             "tk3d_mlp_batch_sums_f32");
    } else {
        std::tie(n.z, n.mean, n.inv_std, std::ignore, std::ignore) =
            at::_batch_norm_impl_index(n.y, gamma, beta, running_mean, running_var, true, momentum, eps,
                                       at::globalContext().userEnabledCuDNN());
    }
    return n;
}

// ReLU of the normalised layer.
Tensor activate(const Normalised &n)
{
    if (n.z.defined())
        return Tensor(n.z).relu_();
    const Tensor z = at::empty_like(n.y);
    done(tk3d_mlp_batch_relu_counted_f32(f32(n.y), &n.norm, n.count, f32(z), stream_of(z)),
         "tk3d_mlp_batch_relu_f32");
    return z;
}

// ReLU and the maximum over the last dimension, with the y at the place of the maximum.
Tensor pool_max(const Normalised &n, Tensor &extreme, Tensor &arg)
{
    const Tensor y = n.y.contiguous();
    const int64_t B = y.size(0), C = y.size(1), M = y.size(2);
    const Tensor out = at::empty({B, C, M}, y.options());
    extreme = at::empty({B, C, M}, y.options());
    arg = at::empty({B, C, M}, y.options().dtype(at::kByte));
    if (n.z.defined()) {
        const Tensor z = n.z.contiguous();
        done(tk3d_mlp_pool_max_f32(f32(z), f32(y), B * C * M, (int)y.size(3), f32(out), f32(extreme),
                                   arg.data_ptr<uint8_t>(), stream_of(y)),
             "tk3d_mlp_pool_max_f32");
    } else {
        done(tk3d_mlp_batch_pool_counted_f32(f32(y), &n.norm, n.count, (int)y.size(3), f32(out), f32(extreme),
                                             arg.data_ptr<uint8_t>(), stream_of(y)),
             "tk3d_mlp_batch_pool_f32");
    }
    return out;
}

// The same over all positions, with the places as torch.max gives them behind a ReLU.
Tensor row_max(const Normalised &n, Tensor &extreme, Tensor &arg, Tensor &index)
{
    const Tensor y = n.y.contiguous(), z = n.z.defined() ? n.z.contiguous() : n.z;
    const int64_t B = y.size(0), C = y.size(1), P = y.numel() / (B * C);
    const Tensor out = at::empty({B, C}, y.options());
    extreme = at::empty({B, C}, y.options());
    arg = at::empty({B, C}, y.options().dtype(at::kInt));
    index = at::empty({B, C}, y.options().dtype(at::kLong));
    done(tk3d_mlp_batch_rows_counted_f32(f32(y), f32(z), &n.norm, n.count, (int)B, (int)C, (int)P, f32(out),
                                         f32(extreme), arg.data_ptr<int32_t>(), index.data_ptr<int64_t>(),
                                         stream_of(y)),
         "tk3d_mlp_batch_rows_f32");
    return out;
}

// Training: the activations of the stock modules, bit by bit. The gradient of a training step
// follows the signs and places that last-bit differences decide: with products and statistics of
// its own, however exact, one step in six of a PointNet++ or DGCNN had single gradients off by more
// than half their root mean square from the stock modules' (which are as far from float64). So the
// products are the library's, and the batch norms' sums come in its order (csrc/batch_norm.hip). Fused
// are the grouping, the batch norm with the ReLU or the maximum behind it, what is kept (the products
// alone, no activations, no edge of a pooled layer), and the whole backward.
Tensor forward_training(const Call &c, Kept &k, Tensor &index)
{
    const int64_t B = c.batch(), L = c.layers();
    Tensor h = c.x2.defined() ? at::cat({c.x, c.x2}, 1) : c.x;
    if (c.grouped()) {
        const int64_t M = c.index.size(1), S = c.index.size(2), N = c.xyz.size(2);
        const int64_t F = c.in_channels(0) - 3;
        h = at::empty({B, F + 3, M, S}, c.xyz.options());
        done(tk3d_group_points_concat_forward_f32(f32(c.x), f32(c.xyz), f32(c.centre),
                                                  c.index.data_ptr<int64_t>(), B, F, N, M, S, f32(h),
                                                  stream_of(h)),
             "tk3d_group_points_concat_forward_f32");
    } else if (c.params[0].dim() == 4) {
        h = h.view({B, h.size(1), c.rows, -1});
    }
    std::vector<Tensor> counts;  // of the layers whose own passes don't count (one launch for all of them)
    for (int64_t l = 0; l < L; ++l) {
        const Tensor *w = &c.params[3 * l], *s = &c.buffers[3 * l];
        Normalised n = stock_layer(h, w[0], w[1], w[2], s[0], s[1], c.momentum[l], c.eps[l]);
        if (s[2].defined() && !n.counts(s[2]))
            counts.push_back(s[2]);
        k.mean.push_back(n.mean);
        k.var.push_back(n.inv_std);
        if (c.pool && l == L - 1) {
            Tensor extreme;
            h = c.whole ? row_max(n, extreme, k.arg, index) : pool_max(n, extreme, k.arg);
            k.y.push_back(extreme);
        } else {
            h = activate(n);
            k.y.push_back(n.y.flatten(2).contiguous());
        }
    }
    if (!counts.empty())
        at::_foreach_add_(counts, 1);
    return h;
}

struct Grads {
    Tensor x, x2;
    std::vector<Tensor> params;
};

// A weight gradient in partial sums, and where their sum goes.
struct Pending {
    std::vector<tk3d_mlp_sum> sums;
    std::vector<Tensor> alive;
};

void pending_sum(const Tensor &partial, const tk3d_mlp_outer &o, float *out, int64_t ld, Pending &pending)
{
    pending.sums.push_back({f32(partial), out, (int64_t)o.row.K * o.col.K, (int32_t)partial.size(0),
                            o.row.K, o.col.K, (int32_t)ld});
    pending.alive.push_back(partial);
}

void outer(int row, int col, tk3d_mlp_outer &o, const Tensor &like, float *out, int64_t ld,
           Pending &pending, void *stream)
{
    const Tensor partial = at::empty({tk3d_mlp_outer_splits(&o), o.row.K, o.col.K}, like.options());
    o.partial = f32(partial);
    done(tk3d_mlp_outer_f32(row, col, &o, stream), "tk3d_mlp_outer_f32");
    pending_sum(partial, o, out, ld, pending);
}

// A layer's product and its weight gradient in one launch, where there is one for its size. Returns the
// partial sums of a masked product and their slots, and leaves those of the weight gradient (and of the rows)
// in o; 0 slots: nothing was launched.
struct Paired {
    int slots = 0;
    Tensor sums, outer, rows;
};
Paired pair(int in, int out, tk3d_mlp_product &p, tk3d_mlp_outer &o, const Tensor &like, void *stream)
{
    Paired r;
    r.slots = tk3d_mlp_pair_slots(&p, &o);
    if (r.slots == 0)
        return r;
    r.outer = at::empty({r.slots, o.row.K, o.col.K}, like.options());
    o.partial = f32(r.outer);
    if (out == TK3D_MLP_OUT_MASK) {
        r.sums = partial_sums(like, p.C, r.slots);
        p.partial = r.sums.data_ptr();
    }
    if (in == TK3D_MLP_IN_CENTRED) {
        r.rows = at::empty({r.slots, o.row.K}, like.options());
        o.rowsum = f32(r.rows);
    }
    done(tk3d_mlp_pair_f32(in, out, &p, &o, stream), "tk3d_mlp_pair_f32");
    return r;
}

Grads backward(const Call &c, const Kept &k, const Tensor &g, bool want_x, bool want_x2)
{
    const int64_t B = c.batch(), P = c.positions(), L = c.layers();
    const Tensor like = c.like();
    void *stream = stream_of(like);
    Grads out;
    out.params.resize(3 * L);
    for (int64_t l = 0; l < L; ++l) {
        out.params[3 * l] = at::empty(c.weight(l).sizes(), like.options());
        const Tensor affine = at::empty({2, c.out_channels(l)}, like.options());
        out.params[3 * l + 1] = affine.select(0, 0);
        out.params[3 * l + 2] = affine.select(0, 1);
    }
    Pending pending;
    std::vector<Tensor> coef(L);
    for (int64_t l = 0; l < L; ++l)
        coef[l] = at::empty({c.out_channels(l), 4}, like.options());
    const auto coefficients = [&](int64_t l, const void *partial, int slots) {
        const tk3d_mlp_norm norm = norm_of(c, k, l);
        done(tk3d_mlp_grad_coefficients_f32(partial, slots, B * P, (int)c.out_channels(l), &norm,
                                            f32(coef[l]), f32(out.params[3 * l + 1]),
                                            f32(out.params[3 * l + 2]), stream),
             "tk3d_mlp_grad_coefficients_f32");
    };

    int64_t l = L - 1;
    Tensor e = g;
    bool masked = false;  // whether e already is the gradient behind the norm
    if (c.whole) {
        // As below with a group that is a row. The layer's input is the activation of the layer in front, or
        // x itself, counted from its mean (as beta of `inner`: of either sign, unlike the centre of activations).
        const int64_t O = c.out_channels(l), I = c.in_channels(l);
        const bool first = l == 0;
        Tensor x = first ? c.x : k.y[l - 1];
        if (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15)  // (a hook's doing)
            x = x.clone();
        Tensor mean;
        if (first) {
            mean = at::empty({I}, like.options());
            done(tk3d_mlp_channel_means_f32(f32(x), (int)B, (int)I, (int)P, f32(mean), stream),
                 "tk3d_mlp_channel_means_f32");
        }
        const tk3d_mlp_norm norm = norm_of(c, k, l),
                            inner = first ? tk3d_mlp_norm{f32(mean), f32(mean), f32(mean), f32(mean), -1.0f}
                                          : norm_of(c, k, l - 1);
        const Tensor sel = at::empty({B, O, 2}, like.options());
        const Tensor sums = partial_sums(like, O, tk3d_mlp_pool_grad_slots((int)B, (int)O, 1));
        const float *w = f32(c.weight(l));
        done(tk3d_mlp_pool_grad_f32(f32(g), f32(k.y[l]), nullptr, k.arg.data_ptr<int32_t>(), (int)B, (int)O, 1,
                                    B * P, &norm, w, (int)I, &inner, first, sums.data_ptr(), sel.data_ptr(),
                                    f32(coef[l]), f32(out.params[3 * l + 1]), f32(out.params[3 * l + 2]),
                                    stream),
             "tk3d_mlp_pool_grad_f32");
        tk3d_mlp_outer o{};
        o.B = (int32_t)B;
        o.P = (int32_t)P;
        o.row = o.col = source(x, nullptr, 0, 0);
        o.row_norm = o.col_norm = inner;
        Paired both;
        if (!first || want_x) {
            const Tensor gram = at::empty({I + 1, I}, like.options());
            done(tk3d_mlp_pool_gram_f32(w, f32(coef[l]), (int)O, (int)I, f32(gram), f32(gram) + I * I, stream),
                 "tk3d_mlp_pool_gram_f32");
            e = at::empty({B, I, P}, like.options());
            done(tk3d_mlp_rows_scatter_f32(sel.data_ptr(), w, (int)B, (int)O, (int)I, (int)P, f32(e), stream),
                 "tk3d_mlp_rows_scatter_f32");
            tk3d_mlp_product p = product(B, I, P);
            p.src[0] = source(x, f32(gram), I, 1);
            p.in_norm = p.out_norm = inner;
            p.yprev = first ? nullptr : f32(x);
            p.bias = f32(gram) + I * I;
            p.add = p.out = f32(e);
            if (first) {
                run_product(TK3D_MLP_IN_SHIFTED, TK3D_MLP_OUT_PLAIN, p, stream);
                out.x = e;
            } else {
                both = pair(TK3D_MLP_IN_CENTRED, TK3D_MLP_OUT_MASK, p, o, like, stream);
                if (both.slots == 0)
                    std::tie(both.sums, both.slots) =
                        summed_product(TK3D_MLP_IN_CENTRED, TK3D_MLP_OUT_MASK, p, like, stream);
            }
        }
        if (!both.outer.defined()) {
            const int splits = tk3d_mlp_outer_splits(&o);
            both.outer = at::empty({splits, I, I}, like.options());
            both.rows = at::empty({splits, I}, like.options());
            o.partial = f32(both.outer);
            o.rowsum = f32(both.rows);
            done(tk3d_mlp_outer_f32(first ? TK3D_MLP_ROW_SHIFTED : TK3D_MLP_ROW_CENTRED,
                                    first ? TK3D_MLP_COL_SHIFTED : TK3D_MLP_COL_CENTRED, &o, stream),
                 "tk3d_mlp_outer_f32");
        }
        const Tensor sparse = at::empty({1, O, I}, like.options()), scratch = at::empty({I + 1, I}, like.options());
        done(tk3d_mlp_rows_outer_f32(sel.data_ptr(), f32(x), first, &inner, (int)B, (int)O, (int)I, (int)P,
                                     f32(sparse), stream),
             "tk3d_mlp_rows_outer_f32");
        done(tk3d_mlp_pool_weight_grad_f32(f32(sparse), 1, f32(both.outer), f32(both.rows),
                                           (int)both.outer.size(0), w, f32(coef[l]), (int)O, (int)I,
                                           f32(scratch), f32(out.params[3 * l]), stream),
             "tk3d_mlp_pool_weight_grad_f32");
        if (!first)
            coefficients(l - 1, both.sums.data_ptr(), both.slots);
        masked = true;
        --l;
    } else if (c.pool) {
        const int64_t O = c.out_channels(l), I = c.in_channels(l), M = P / c.pool;
        const tk3d_mlp_norm norm = norm_of(c, k, l), inner = norm_of(c, k, l - 1);
        const Tensor sel = at::empty({B, O, M, 2}, like.options());
        const Tensor scratch_sums = partial_sums(like, O, tk3d_mlp_pool_grad_slots((int)B, (int)O, (int)M));
        const float *w = f32(c.weight(l));
        done(tk3d_mlp_pool_grad_f32(f32(g), f32(k.y[l]), k.arg.data_ptr<uint8_t>(), nullptr, (int)B, (int)O,
                                    (int)M, B * P, &norm, w, (int)I, &inner, 0, scratch_sums.data_ptr(),
                                    sel.data_ptr(), f32(coef[l]), f32(out.params[3 * l + 1]),
                                    f32(out.params[3 * l + 2]), stream),
             "tk3d_mlp_pool_grad_f32");
        const Tensor gram = at::empty({I + 1, I}, like.options());
        done(tk3d_mlp_pool_gram_f32(w, f32(coef[l]), (int)O, (int)I, f32(gram), f32(gram) + I * I,
                                    stream),
             "tk3d_mlp_pool_gram_f32");
        e = at::empty({B, I, P}, like.options());
        done(tk3d_mlp_pool_scatter_f32(sel.data_ptr(), w, (int)B, (int)O, (int)I, (int)M, (int)c.pool,
                                       f32(e), stream),
             "tk3d_mlp_pool_scatter_f32");
        tk3d_mlp_product p = product(B, I, P);
        p.src[0] = source(k.y[l - 1], f32(gram), I, 1);
        p.in_norm = p.out_norm = inner;
        p.yprev = f32(k.y[l - 1]);
        p.bias = f32(gram) + I * I;
        p.add = p.out = f32(e);
        const int sparse_splits = tk3d_mlp_pool_outer_splits((int)B, (int)O, (int)I, (int)M);
        const Tensor sparse = at::empty({sparse_splits, O, I}, like.options());
        done(tk3d_mlp_pool_outer_f32(sel.data_ptr(), f32(k.y[l - 1]), &inner, (int)B, (int)O, (int)I,
                                     (int)M, (int)c.pool, f32(sparse), stream),
             "tk3d_mlp_pool_outer_f32");
        tk3d_mlp_outer o{};
        o.B = (int32_t)B;
        o.P = (int32_t)P;
        o.col = source(k.y[l - 1], nullptr, 0, 0);
        o.col_norm = o.row_norm = inner;
        o.row = o.col;
        Paired both = pair(TK3D_MLP_IN_CENTRED, TK3D_MLP_OUT_MASK, p, o, like, stream);
        if (both.slots == 0) {
            std::tie(both.sums, both.slots) =
                summed_product(TK3D_MLP_IN_CENTRED, TK3D_MLP_OUT_MASK, p, like, stream);
            const int splits = tk3d_mlp_outer_splits(&o);
            both.outer = at::empty({splits, I, I}, like.options());
            both.rows = at::empty({splits, I}, like.options());
            o.partial = f32(both.outer);
            o.rowsum = f32(both.rows);
            done(tk3d_mlp_outer_f32(TK3D_MLP_ROW_CENTRED, TK3D_MLP_COL_CENTRED, &o, stream),
                 "tk3d_mlp_outer_f32");
        }
        const Tensor scratch = at::empty({I + 1, I}, like.options());
        done(tk3d_mlp_pool_weight_grad_f32(f32(sparse), sparse_splits, f32(both.outer), f32(both.rows),
                                           (int)both.outer.size(0), w, f32(coef[l]), (int)O, (int)I,
                                           f32(scratch), f32(out.params[3 * l]), stream),
             "tk3d_mlp_pool_weight_grad_f32");
        coefficients(l - 1, both.sums.data_ptr(), both.slots);
        masked = true;
        --l;
    } else {
        const tk3d_mlp_norm norm = norm_of(c, k, l);
        const int C = (int)c.out_channels(l);
        const int slots = tk3d_mlp_mask_slots((int)B, C, (int)P);
        const Tensor partial = partial_sums(like, C, slots);
        done(tk3d_mlp_mask_sums_f32(f32(g), f32(k.y[l]), (int)B, C, (int)P, &norm,
                                    partial.data_ptr(), stream),
             "tk3d_mlp_mask_sums_f32");
        coefficients(l, partial.data_ptr(), slots);
    }

    for (; l >= 0; --l) {
        const int64_t O = c.out_channels(l), I = c.in_channels(l);
        const float *w = f32(c.weight(l));
        float *dw = f32(out.params[3 * l]);
        tk3d_mlp_outer o{};
        o.B = (int32_t)B;
        o.P = (int32_t)P;
        o.row = source(e, nullptr, 0, 0);
        o.row.y = f32(k.y[l]);
        o.row.coef = f32(coef[l]);
        o.row_norm = norm_of(c, k, l);
        const int row = masked ? TK3D_MLP_ROW_GRAD : TK3D_MLP_ROW_GRAD_OUT;
        const int in = masked ? TK3D_MLP_IN_GRAD : TK3D_MLP_IN_GRAD_OUT;
        const auto gradient_product = [&](int64_t channels) {
            tk3d_mlp_product p = product(B, channels, P);
            p.src[0] = source(e, w, I, 1);
            p.src[0].y = f32(k.y[l]);
            p.src[0].coef = f32(coef[l]);
            p.in_norm = norm_of(c, k, l);
            return p;
        };
        if (l > 0) {
            o.col = source(k.y[l - 1], nullptr, 0, 0);
            o.col_norm = norm_of(c, k, l - 1);
            tk3d_mlp_product p = gradient_product(I);
            p.out_norm = o.col_norm;
            p.yprev = f32(k.y[l - 1]);
            const Tensor before = at::empty({B, I, P}, like.options());
            p.out = f32(before);
            Paired both = pair(in, TK3D_MLP_OUT_MASK, p, o, like, stream);
            if (both.slots) {
                pending_sum(both.outer, o, dw, I, pending);
            } else {
                outer(row, TK3D_MLP_COL_ACT, o, like, dw, I, pending, stream);
                std::tie(both.sums, both.slots) = summed_product(in, TK3D_MLP_OUT_MASK, p, like, stream);
            }
            coefficients(l - 1, both.sums.data_ptr(), both.slots);
            e = before;
            masked = true;
            continue;
        }
        if (!c.grouped()) {
            const int64_t C1 = c.x.size(1);
            o.col = source(c.x, nullptr, 0, 0);
            if (want_x)
                out.x = at::empty(c.x.sizes(), like.options());
            Paired both;
            if (want_x && !want_x2) {
                tk3d_mlp_product p = gradient_product(C1);
                p.out = f32(out.x);
                both = pair(in, TK3D_MLP_OUT_PLAIN, p, o, like, stream);
            }
            if (both.slots)
                pending_sum(both.outer, o, dw, I, pending);
            else
                outer(row, TK3D_MLP_COL_RAW, o, like, dw, I, pending, stream);
            if (c.x2.defined()) {
                o.col = source(c.x2, nullptr, 0, 0);
                outer(row, TK3D_MLP_COL_RAW, o, like, dw + C1, I, pending, stream);
            }
            if ((want_x || want_x2) && !both.slots) {
                tk3d_mlp_product p = gradient_product(I);
                p.C0 = (int32_t)C1;
                if (want_x2)
                    out.x2 = at::empty(c.x2.sizes(), like.options());
                p.out = f32(out.x);
                p.out2 = f32(out.x2);
                run_product(in, TK3D_MLP_OUT_PLAIN, p, stream);
            }
            continue;
        }
        const int64_t M = c.index.size(1), S = c.index.size(2), N = c.xyz.size(2), F = I - 3;
        const int64_t *index = c.index.data_ptr<int64_t>();
        if (!want_x && F <= 29) {
            // The grouped input itself, in one tile of columns: it is small, and nothing else of
            // this layer's gradient is needed.
            const Tensor grouped = at::empty({B, I, P}, like.options());
            done(tk3d_group_points_concat_forward_f32(f32(c.x), f32(c.xyz), f32(c.centre), index, B,
                                                      F, N, M, S, f32(grouped), stream),
                 "tk3d_group_points_concat_forward_f32");
            o.col = source(grouped, nullptr, 0, 0);
            outer(row, TK3D_MLP_COL_RAW, o, like, dw, I, pending, stream);
            continue;
        }
        // dy, summed per point; the rest is per point.
        const Tensor rel = at::empty({B, 3, P}, like.options());
        done(tk3d_group_points_concat_forward_f32(nullptr, f32(c.xyz), f32(c.centre), index, B, 0, N,
                                                  M, S, f32(rel), stream),
             "tk3d_group_points_concat_forward_f32");
        const Tensor partial = at::empty({tk3d_mlp_grad_apply_splits((int)B, (int)P), O, 3}, like.options());
        done(tk3d_mlp_grad_apply_f32(f32(e), f32(k.y[0]), f32(coef[0]), f32(rel), (int)B, (int)O, (int)P,
                                     f32(partial), stream),
             "tk3d_mlp_grad_apply_f32");
        o.col = source(rel, nullptr, 0, 0);
        pending_sum(partial, o, dw + F, I, pending);
        const Tensor du = at::empty({B, O, N}, like.options());
        done(tk3d_group_points_backward_f32(f32(e), index, B, O, N, M, S, f32(du), stream),
             "tk3d_group_points_backward_f32");
        tk3d_mlp_outer q{};
        q.B = (int32_t)B;
        q.P = (int32_t)N;
        q.row = source(du, nullptr, 0, 0);
        q.col = source(c.x, nullptr, 0, 0);
        outer(TK3D_MLP_ROW_RAW, TK3D_MLP_COL_RAW, q, like, dw, I, pending, stream);
        if (want_x) {
            out.x = at::empty(c.x.sizes(), like.options());
            tk3d_mlp_product p = product(B, F, N);
            p.src[0] = source(du, w, I, 1);
            p.out = f32(out.x);
            run_product(TK3D_MLP_IN_RAW, TK3D_MLP_OUT_PLAIN, p, stream);
        }
    }
    done(tk3d_mlp_sum_f32(pending.sums.data(), (int)pending.sums.size(), stream), "tk3d_mlp_sum_f32");
    return out;
}

// The same chain in stock operators (training): for gradients of gradients.
Tensor in_stock_operators(const Call &c)
{
    Tensor h;
    if (c.grouped()) {
        const int64_t B = c.batch(), M = c.index.size(1), S = c.index.size(2);
        const Tensor valid = (c.index.ge(0) & c.index.lt(c.xyz.size(2))).view({B, 1, M * S});
        const Tensor flat = c.index.view({B, 1, M * S}).clamp(0, c.xyz.size(2) - 1);
        const auto gather = [&](const Tensor &t) {
            return at::where(valid, at::gather(t, 2, flat.expand({B, t.size(1), M * S})),
                             at::zeros({}, t.options()));
        };
        h = gather(c.xyz) - c.centre.unsqueeze(3).expand({B, 3, M, S}).reshape({B, 3, M * S});
        if (c.x.defined())
            h = at::cat({gather(c.x), h}, 1);
    } else {
        h = c.x2.defined() ? at::cat({c.x, c.x2}, 1) : c.x;
    }
    for (int64_t l = 0; l < c.layers(); ++l) {
        h = at::conv1d(h, c.weight(l).view({c.out_channels(l), c.in_channels(l), 1}));
        h = at::batch_norm(h, c.params[3 * l + 1], c.params[3 * l + 2], Tensor(), Tensor(), true, 0.0,
                           c.eps[l], false);
        h = at::relu(h);
    }
    if (c.whole)
        return std::get<0>(at::max(h, 2));
    if (c.pool)
        h = std::get<0>(at::max(h.view({h.size(0), h.size(1), h.size(2) / c.pool, c.pool}), 3));
    return h;
}

struct Node : torch::autograd::Function<Node> {  // (made in training mode alone)
    // Saved: x, x2, xyz, centre, index, arg, then of every layer weight, gamma, beta, y, mean, var.
    // (The tensors in front of the call are what autograd sees; the call holds them too.)
    // The maximum over all positions has their places behind it.
    static variable_list forward(AutogradContext *ctx, const std::optional<Tensor> &,
                                 const std::optional<Tensor> &, at::TensorList, const Call &call)
    {
        Kept k;
        Tensor index;
        const Tensor z = forward_training(call, k, index);
        variable_list saved = {call.x, call.x2, call.xyz, call.centre, call.index, k.arg};
        for (int64_t l = 0; l < call.layers(); ++l) {
            for (int64_t i = 0; i < 3; ++i)
                saved.push_back(call.params[3 * l + i]);
            saved.push_back(k.y[l]);
            saved.push_back(k.mean[l]);
            saved.push_back(k.var[l]);
        }
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["pool"] = call.pool;
        ctx->saved_data["whole"] = call.whole;
        ctx->saved_data["eps"] = call.eps;
        ctx->saved_data["want_x"] = call.x.defined() && call.x.requires_grad();
        ctx->saved_data["want_x2"] = call.x2.defined() && call.x2.requires_grad();
        if (!call.whole)
            return {z};
        ctx->mark_non_differentiable({index});
        return {z, index};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list s = dense(ctx->get_saved_variables());
        Call c;
        Kept k;
        c.x = s[0];
        c.x2 = s[1];
        c.xyz = s[2];
        c.centre = s[3];
        c.index = s[4];
        k.arg = s[5];
        c.pool = ctx->saved_data["pool"].toInt();
        c.whole = ctx->saved_data["whole"].toBool();
        c.training = true;
        c.eps = ctx->saved_data["eps"].toDoubleVector();
        const int64_t L = ((int64_t)s.size() - 6) / 6;
        for (int64_t l = 0; l < L; ++l) {
            const Tensor *t = &s[6 + 6 * l];
            for (int i = 0; i < 3; ++i)
                c.params.push_back(t[i]);
            k.y.push_back(t[3]);
            k.mean.push_back(t[4]);
            k.var.push_back(t[5]);
        }
        const bool want_x = ctx->saved_data["want_x"].toBool();
        const bool want_x2 = ctx->saved_data["want_x2"].toBool();
        // One gradient per tensor that apply() was given.
        variable_list result;
        if (c10::GradMode::is_enabled()) {  // a gradient of this gradient will be asked for
            const Tensor z = in_stock_operators(c);
            variable_list inputs;
            if (want_x)
                inputs.push_back(c.x);
            if (want_x2)
                inputs.push_back(c.x2);
            for (const Tensor &t : c.params)
                if (t.requires_grad())
                    inputs.push_back(t);
            const variable_list d =
                torch::autograd::grad({z}, inputs, {grads[0].reshape(z.sizes())}, std::nullopt, true,
                                      true);
            size_t i = 0;
            result.push_back(want_x ? d[i++] : Tensor());
            result.push_back(want_x2 ? d[i++] : Tensor());
            for (const Tensor &t : c.params)
                result.push_back(t.requires_grad() ? d[i++] : Tensor());
        } else {
            OnDeviceOf guard(c.like().device());
            const Grads d = tk3d::backward(c, k, grads[0].contiguous(), want_x, want_x2);
            result.push_back(d.x);
            result.push_back(d.x2);
            for (int64_t l = 0; l < L; ++l)
                for (int i = 0; i < 3; ++i)
                    result.push_back(d.params[3 * l + i]);
        }
        result.push_back(Tensor());  // (the call itself)
        return result;
    }
};

// ---- EdgeConv with one layer ---------------------------------------------------------------------

struct EdgeCall {
    Tensor x, index;   // [B, C, N], [B, N, K]
    Tensor lists;      // the inverse of the graph, where the caller has it
    Tensor weight, gamma, beta, running_mean, running_var, batches;
    double eps = 0.0, momentum = 0.0;
    bool training = false;

    int64_t batch() const { return x.size(0); }
    int64_t points() const { return x.size(2); }
    int64_t neighbours() const { return index.size(2); }
    int64_t out_channels() const { return weight.size(0); }
};

struct EdgeKept {
    Tensor extreme, arg, mean, var;
};

tk3d_mlp_norm norm_of(const EdgeCall &c, const EdgeKept &k)
{
    return {f32(k.mean), f32(k.var), f32(c.gamma), f32(c.beta), c.training ? -1.0f : (float)c.eps};
}

Tensor edge_forward(const EdgeCall &c, EdgeKept &k)
{
    const int64_t B = c.batch(), N = c.points(), K = c.neighbours(), O = c.out_channels();
    const int64_t C = c.x.size(1);
    const auto options = c.x.options();
    void *stream = stream_of(c.x);
    if (c.training) {  // (bit by bit what the stock modules give, see forward_training)
        const Tensor edges = at::empty({B, 2 * C, N, K}, options);
        done(tk3d_mlp_edge_features_f32(f32(c.x), c.index.data_ptr<int64_t>(), (int)B, (int)C, (int)N,
                                        (int)K, f32(edges), stream),
             "tk3d_mlp_edge_features_f32");
        Normalised n = stock_layer(edges, c.weight, c.gamma, c.beta, c.running_mean, c.running_var, c.momentum,
                                   c.eps);
        if (c.batches.defined() && !n.counts(c.batches))
            Tensor(c.batches).add_(1);
        k.mean = n.mean;
        k.var = n.inv_std;
        return pool_max(n, k.extreme, k.arg);
    }
    k.extreme = at::empty({B, O, N}, options);
    k.mean = c.running_mean;
    k.var = c.running_var;
    const Tensor workspace =
        at::empty({tk3d_mlp_edge_forward_bytes((int)B, (int)N, (int)C, (int)O)}, options.dtype(at::kByte));
    done(tk3d_mlp_edge_forward_f32(f32(c.x), c.index.data_ptr<int64_t>(), f32(c.weight), f32(c.gamma),
                                   (int)B, (int)N, (int)K, (int)C, (int)O, workspace.data_ptr(),
                                   f32(k.extreme), stream),
         "tk3d_mlp_edge_forward_f32");
    const Tensor z = at::empty({B, O, N}, options);
    const tk3d_mlp_norm norm = norm_of(c, k);
    done(tk3d_mlp_activate_f32(f32(k.extreme), B * O, (int)O, (int)N, &norm, f32(z), stream),
         "tk3d_mlp_activate_f32");
    return z;
}

variable_list edge_backward(const EdgeCall &c, const EdgeKept &k, const Tensor &g, bool want_x)
{
    const int64_t B = c.batch(), N = c.points(), K = c.neighbours(), O = c.out_channels();
    const int64_t C = c.x.size(1);
    const auto options = c.x.options();
    void *stream = stream_of(c.x);
    const tk3d_mlp_norm norm = norm_of(c, k);
    const Tensor affine = at::empty({2, O}, options), coef = at::empty({O, 4}, options);
    const int slots = tk3d_mlp_mask_slots((int)B, (int)O, (int)N);
    const Tensor partial = partial_sums(c.x, O, slots);
    done(tk3d_mlp_mask_sums_f32(f32(g), f32(k.extreme), (int)B, (int)O, (int)N, &norm,
                                partial.data_ptr(), stream),
         "tk3d_mlp_mask_sums_f32");
    done(tk3d_mlp_grad_coefficients_f32(partial.data_ptr(), slots, B * N * K, (int)O, &norm,
                                        f32(coef), f32(affine), f32(affine) + O, stream),
         "tk3d_mlp_grad_coefficients_f32");
    const Tensor dw = at::empty(c.weight.sizes(), options);
    Tensor dx;
    if (want_x)
        dx = at::empty(c.x.sizes(), options);
    const Tensor workspace =
        at::empty({tk3d_mlp_edge_backward_bytes((int)B, (int)N, (int)O, (int)C)}, options.dtype(at::kByte));
    done(tk3d_mlp_edge_backward_f32(f32(g), f32(k.extreme), k.arg.data_ptr<uint8_t>(), f32(c.x),
                                    c.index.data_ptr<int64_t>(), c.lists.data_ptr<int32_t>(),
                                    f32(c.weight), (int)B, (int)N, (int)K, (int)C, (int)O, &norm,
                                    f32(coef), workspace.data_ptr(), f32(dx), f32(dw), stream),
         "tk3d_mlp_edge_backward_f32");
    return {dx, dw, affine.select(0, 0), affine.select(0, 1)};
}

Tensor edge_in_stock_operators(const EdgeCall &c)
{
    const int64_t B = c.batch(), N = c.points(), K = c.neighbours(), C = c.x.size(1);
    const Tensor valid = (c.index.ge(0) & c.index.lt(N)).view({B, 1, N * K});
    const Tensor flat = c.index.view({B, 1, N * K}).clamp(0, N - 1).expand({B, C, N * K});
    const Tensor query = c.x.unsqueeze(3).expand({B, C, N, K}).reshape({B, C, N * K});
    const Tensor near = at::where(valid, at::gather(c.x, 2, flat), at::zeros({}, c.x.options()));
    Tensor h = at::conv1d(at::cat({near - query, query}, 1),
                          c.weight.view({c.out_channels(), 2 * C, 1}));
    h = at::batch_norm(h, c.gamma, c.beta, Tensor(), Tensor(), true, 0.0, c.eps, false);
    return std::get<0>(at::max(at::relu(h).view({B, c.out_channels(), N, K}), 3));
}

struct EdgeNode : torch::autograd::Function<EdgeNode> {  // (made in training mode alone)
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &, const Tensor &,
                          const Tensor &, const EdgeCall &call)
    {
        EdgeKept k;
        const Tensor z = edge_forward(call, k);
        ctx->save_for_backward({call.x, call.index, call.lists, call.weight, call.gamma, call.beta,
                                k.extreme, k.arg, k.mean, k.var});
        ctx->saved_data["eps"] = call.eps;
        ctx->saved_data["want_x"] = x.requires_grad();
        return z;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list s = dense(ctx->get_saved_variables());
        EdgeCall c;
        EdgeKept k;
        c.x = s[0];
        c.index = s[1];
        c.lists = s[2];
        c.weight = s[3];
        c.gamma = s[4];
        c.beta = s[5];
        k.extreme = s[6];
        k.arg = s[7];
        k.mean = s[8];
        k.var = s[9];
        c.training = true;
        c.eps = ctx->saved_data["eps"].toDouble();
        const bool want_x = ctx->saved_data["want_x"].toBool();
        variable_list d;
        if (c10::GradMode::is_enabled()) {
            const Tensor z = edge_in_stock_operators(c);
            variable_list inputs;
            for (const Tensor &t : {c.x, c.weight, c.gamma, c.beta})
                if (t.requires_grad())
                    inputs.push_back(t);
            const variable_list found =
                torch::autograd::grad({z}, inputs, {grads[0]}, std::nullopt, true, true);
            size_t i = 0;
            for (const Tensor &t : {c.x, c.weight, c.gamma, c.beta})
                d.push_back(t.requires_grad() ? found[i++] : Tensor());
        } else {
            OnDeviceOf guard(c.x.device());
            d = edge_backward(c, k, grads[0].contiguous(), want_x);
        }
        d.push_back(Tensor());
        return d;
    }
};

bool usable(const Tensor &t, const Tensor &like)
{
    return t.is_cuda() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided &&
           t.device() == like.device() && plain(t);
}

bool usable_index(const Tensor &t, const Tensor &like)
{
    return t.scalar_type() == at::kLong && t.layout() == at::kStrided && t.device() == like.device() &&
           plain(t);
}

// Weight, gamma and beta, running mean, running variance and batch count of one layer.
bool usable_layer(const Tensor *params, const Tensor *buffers, const Tensor &like)
{
    const int64_t C = params[0].dim() > 1 ? params[0].size(0) : -1;
    for (int i = 0; i < 3; ++i)
        if (!usable(params[i], like) || !params[i].is_contiguous() || (i && params[i].numel() != C))
            return false;
    for (int i = 0; i < 2; ++i)
        if (!usable(buffers[i], like) || !buffers[i].is_contiguous() || buffers[i].numel() != C)
            return false;
    return !buffers[2].defined() || (usable_index(buffers[2], like) && buffers[2].numel() == 1);
}

}  // namespace

// Whether the backward of a maximum over all positions takes this layer: its products are as wide as the layer's input.
// That pays from twice as many outputs and 4096 positions on (64 -> 128 -> 256 channels, 4 x 1024 forward and backward
// 296 -> 277 us; more launches, each of its 5 us), and where the positions are worth the products of the weights alone,
// O I (I + 1) in fp64, a cloud's O maxima on top: a position for every 32 weights (last layer 256 -> 1024, 32 x 128
// dense 284, so 289 us, 64 x 64 286, 341, 128 x 128 522, 461; 512 -> 1024, 32 x 128 302, 417, 64 x 128 494, 568,
// 128 x 128 883, 888, 256 x 128 1703, 1568). Rows under 16 gain at any number (256 -> 1024, 512 x 8 994 -> 828, 512 ->
// 1024 1719, 1710). A first layer gains from 128 positions a row on (330 -> 700 channels, 128 x 128 557 -> 488), not on
// shorter ones (128 -> 512, 256 x 16 252, 310; 320 -> 1024, 128 x 32 333, 415; 330 -> 700, 64 x 64 247, 304).
bool whole_rows(const Call &c)
{
    const int64_t l = c.layers() - 1, O = c.out_channels(l), I = c.in_channels(l), B = c.batch(), P = c.positions();
    if (P % 4 != 0 || O < 2 * I || B * P < 4096 || (P >= 16 && 32 * B * P < O * I) || B > (1 << 20))
        return false;
    if (l > 0)
        return true;
    if (P < 128)
        return false;
    tk3d_mlp_product p = product(B, I, P);
    p.src[0] = source(c.x, nullptr, I, 1);
    return tk3d_mlp_product_slots(TK3D_MLP_IN_SHIFTED, TK3D_MLP_OUT_PLAIN, &p) > 0;
}

// x [B,C,P] (or [B,C,M,S]); a chain applied to it. Declines (undefined result) what the kernels
// do not take: the caller then runs the stock modules.
// With pool -1 the maximum over all positions: [B, C] and the places, for training alone.
variable_list mlp(Tensor x, Tensor x2, const Tensor &xyz, const Tensor &centre, const Tensor &index,
                  std::vector<Tensor> params, std::vector<Tensor> buffers, std::vector<double> eps,
                  std::vector<double> momentum, bool training, int64_t pool)
{
    Call c;
    const int64_t L = (int64_t)params.size() / 3;
    c.whole = pool < 0;
    if (c.whole) {
        if (!training || !x.defined() || x.dim() != 3 || x.size(2) == 0)
            return {};
        pool = 0;
    }
    // (Pooled forms: groups of 32 or 64, which fill whole tiles of every shape; other groups take
    // the dense chain and a maximum behind it.)
    if (L == 0 || (pool && (L < 2 || (pool != 32 && pool != 64))) || watched())
        return {};
    const bool grouped = xyz.defined();
    std::vector<int64_t> shape;
    if (grouped) {
        if (L < 2 || !pool || !usable(xyz, xyz) || !usable(centre, xyz) || !usable_index(index, xyz) ||
            xyz.dim() != 3 || centre.dim() != 3 || index.dim() != 3 || index.size(2) != pool || centre.size(2) != index.size(1) || xyz.size(1) != 3 ||
            centre.size(1) != 3 || index.size(0) != xyz.size(0) || centre.size(0) != xyz.size(0))
            return {};
        c.xyz = xyz.contiguous();
        c.centre = centre.contiguous();
        c.index = index.contiguous();
        if (x.defined() && (x.dim() != 3 || x.size(2) != xyz.size(2) || x.size(0) != xyz.size(0)))
            return {};
    } else {
        if (!x.defined() || x.dim() < 3 || x.dim() > 4 || (pool && x.size(-1) != pool))
            return {};
        if (x2.defined() && (x.dim() != 3 || x2.dim() != 3 || x2.size(0) != x.size(0) ||
                             x2.size(2) != x.size(2)))
            return {};
        shape = x.sizes().vec();
    }
    const bool has_x = x.defined(), has_x2 = x2.defined();
    const Tensor &first = grouped ? xyz : x;
    if ((has_x && !usable(x, first)) || (has_x2 && !usable(x2, first)))
        return {};
    int64_t channels = (has_x ? x.size(1) : 0) + (has_x2 ? x2.size(1) : 0) + (grouped ? 3 : 0);
    bool tracked = (has_x && x.requires_grad()) || (has_x2 && x2.requires_grad());
    for (int64_t l = 0; l < L; ++l) {
        if (!usable_layer(&params[3 * l], &buffers[3 * l], first))
            return {};
        for (int i = 0; i < 3; ++i)
            tracked = tracked || params[3 * l + i].requires_grad();
        if (params[3 * l].size(1) != channels)
            return {};
        channels = params[3 * l].size(0);
    }
    if (params[0].dim() != (grouped ? 4 : x.dim()))
        return {};  // (a Conv1d on [B, C, M, S] and the like: stock torch has the error)
    c.rows = !grouped && x.dim() == 4 ? x.size(2) : 0;
    if (has_x)
        c.x = x.dim() == 4 ? x.flatten(2).contiguous() : x.contiguous();
    if (has_x2)
        c.x2 = x2.contiguous();
    c.pool = pool;
    c.training = training;
    c.params = std::move(params);
    c.buffers = std::move(buffers);
    c.eps = std::move(eps);
    c.momentum = std::move(momentum);
    const int64_t B = c.batch(), P = c.positions();
    // The stock modules run training mode without gradients, and evaluation mode with them: there,
    // too, signs and places decide the gradients, and nothing of the forward would be left to fuse.
    const bool grads = c10::GradMode::is_enabled() && tracked;
    if (training != grads || (training && !same_gradients(P)))
        return {};
    if (c.whole) {
        c.pool = P;
        if (!whole_rows(c))
            return {};
    }
    int64_t widest = has_x ? c.x.size(1) : 0;
    if (has_x2)
        widest = std::max(widest, c.x2.size(1));
    for (int64_t l = 0; l < L; ++l)
        widest = std::max(widest, c.out_channels(l));
    const int64_t longest = grouped ? std::max(P, c.xyz.size(2)) : P;
    // (one value per channel has no variance: stock batch norm raises the error)
    if (B == 0 || P == 0 || longest == 0 || B * P < 2 || widest > 2048 ||
        (widest + 8) * longest > (1 << 29) || B * longest > (1 << 30))
        return {};
    OnDeviceOf guard(c.like().device());
    for (int64_t l = 0; training && l < L; ++l) {
        const int64_t C = c.out_channels(l), rows = grouped ? index.size(1) : c.rows;
        const std::vector<int64_t> y =
            rows ? std::vector<int64_t>{B, C, rows, P / rows} : std::vector<int64_t>{B, C, P};
        if (!library_norm(c.like(), y, &c.params[3 * l], &c.buffers[3 * l], c.eps[l]))
            return {};
    }
    Tensor z;
    if (training) {
        const auto given = [](const Tensor &t) {
            return t.defined() ? std::optional<Tensor>(t) : std::nullopt;
        };
        const variable_list made = Node::apply(given(c.x), given(c.x2), at::TensorList(c.params), c);
        if (c.whole)
            return made;
        z = made[0];
    } else {
        z = evaluate(c);
    }
    if (!grouped && x.dim() == 4 && !pool)
        z = z.reshape({shape[0], z.size(1), shape[2], shape[3]});
    return {z};
}

// The inverse of a graph [B, N, K] over N points, for edge_conv(); undefined where the kernels do
// not take its size.
Tensor edge_lists(const Tensor &index_, int64_t n)
{
    if (!index_.is_cuda() || !usable_index(index_, index_) || index_.dim() != 3 || watched() ||
        index_.size(1) != n || !tk3d_mlp_edge_supported(index_.size(0), n, index_.size(2), 1))
        return Tensor();
    const Tensor index = index_.contiguous();
    const int64_t B = index.size(0), K = index.size(2);
    OnDeviceOf guard(index.device());
    const Tensor lists = at::empty({B, n + 1 + n * K}, index.options().dtype(at::kInt));
    done(tk3d_mlp_edge_lists(index.data_ptr<int64_t>(), (int)B, (int)n, (int)K,
                             lists.data_ptr<int32_t>(), stream_of(index)),
         "tk3d_mlp_edge_lists");
    return lists;
}

// EdgeConv with one layer on the graph of x with itself; undefined where the caller has to run it
// layer by layer.
Tensor edge_conv(const Tensor &x, const Tensor &index, const Tensor &lists,
                 const std::vector<Tensor> &params, const std::vector<Tensor> &buffers, double eps,
                 double momentum, bool training)
{
    if (!usable(x, x) || x.dim() != 3 || !usable_index(index, x) || index.dim() != 3 ||
        index.size(0) != x.size(0) || index.size(1) != x.size(2) || params.size() != 3 || watched() ||
        params[0].dim() != 4 || !usable_layer(params.data(), buffers.data(), x))
        return Tensor();
    const int64_t B = x.size(0), C = x.size(1), N = x.size(2), K = index.size(2);
    const int64_t O = params[0].size(0);
    if (lists.defined() &&
        (lists.scalar_type() != at::kInt || lists.device() != x.device() || !plain(lists) ||
         lists.dim() != 2 || lists.size(0) != B || lists.size(1) != N + 1 + N * K ||
         !lists.is_contiguous()))
        fail("lists must be edge_lists(key_ind, N): contiguous int32 [B, N + 1 + N K] on the GPU of "
             "the features.");
    if (params[0].size(1) != 2 * C || !tk3d_mlp_edge_supported(B, N, K, O) || B * N * K < 2 ||
        C > 4096 || (std::max(C, 2 * O) + 8) * N > (1 << 29) || (training && !same_gradients(N * K)))
        return Tensor();
    EdgeCall c;
    c.x = x.contiguous();
    c.index = index.contiguous();
    c.weight = params[0];
    c.gamma = params[1];
    c.beta = params[2];
    c.running_mean = buffers[0];
    c.running_var = buffers[1];
    c.batches = buffers[2];
    c.eps = eps;
    c.momentum = momentum;
    c.training = training;
    OnDeviceOf guard(x.device());
    const bool grads = c10::GradMode::is_enabled() && (x.requires_grad() || c.weight.requires_grad() ||
                                                       c.gamma.requires_grad() || c.beta.requires_grad());
    if (training != grads ||  // (as for mlp())
        (training && !library_norm(x, {B, O, N, K}, params.data(), buffers.data(), eps)))
        return Tensor();
    if (grads) {
        c.lists = lists.defined() ? lists : edge_lists(c.index, N);
        return EdgeNode::apply(c.x, c.weight, c.gamma, c.beta, c);
    }
    EdgeKept k;
    return edge_forward(c, k);
}

}  // namespace tk3d
