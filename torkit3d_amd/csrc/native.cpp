// Host path of the operators: argument checks, output allocation, autograd nodes and the calls
// into the C ABI (include/tk3d.h), as a Python extension module (torkit3d_amd/_host.so).
// A small call is host work only: through ctypes and Python's autograd.Function a chamfer
// forward + backward on 2 x 1024 points took 100 to 160 us around 27 us of kernels.
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "native.h"

namespace py = pybind11;
using namespace tk3d;
using torch::autograd::AutogradContext;

namespace {

// ---- checks (messages as the reference's TORCH_CHECKs give them; RuntimeError in Python) ----

void check(bool ok, const std::string &message)
{
    if (!ok)
        fail(message);
}

void check_eq(int64_t a, int64_t b, const char *what)
{
    if (a != b)
        fail("Check failed: " + std::string(what) + " (" + std::to_string(a) + " vs. " +
             std::to_string(b) + ")");
}

Tensor tensor_arg(const char *name, py::handle h)
{
    if (!THPVariable_Check(h.ptr()))
        fail(std::string(name) + " must be a tensor.");
    return THPVariable_Unpack(h.ptr());
}

void check_cuda(const char *name, const Tensor &t)
{
    if (!t.is_cuda())
        fail(std::string(name) + " must be a CUDA tensor.");
}

void check_contiguous_cuda(const char *name, const Tensor &t)
{
    check_cuda(name, t);
    if (!t.is_contiguous())
        fail(std::string(name) + " must be contiguous.");
}

void check_index(const char *name, const Tensor &t)
{
    if (t.scalar_type() != at::kLong)
        fail(std::string(name) + " must be an int64 tensor.");
}

void check_same(const char *a_name, const Tensor &a, const char *b_name, const Tensor &b)
{
    if (a.scalar_type() != b.scalar_type())
        fail(std::string(a_name) + " and " + b_name + " must have the same dtype.");
    if (a.device() != b.device())
        fail(std::string(a_name) + " and " + b_name + " must be on the same device.");
}

// float32 (true) or float64 (false); anything else is an error.
bool is_f32(const Tensor &t)
{
    if (t.scalar_type() == at::kFloat)
        return true;
    if (t.scalar_type() != at::kDouble)
        fail(std::string("torkit3d_amd supports float32 and float64 tensors, got ") +
             c10::toString(t.scalar_type()));
    return false;
}

// ---- device pointers, outputs, stream ---------------------------------------------------------

struct Ptr {  // becomes whatever pointer the entry point takes
    void *p;
    template <typename T> operator T *() const { return static_cast<T *>(p); }
};

Ptr ptr(const Tensor &t)
{
    return {t.defined() && t.numel() > 0 ? const_cast<void *>(t.const_data_ptr()) : nullptr};
}

Tensor like(const Tensor &t, at::IntArrayRef shape) { return at::empty(shape, t.options()); }

Tensor index_like(const Tensor &t, at::IntArrayRef shape)
{
    return at::empty(shape, t.options().dtype(at::kLong));
}

Tensor scratch(const Tensor &t, size_t bytes)
{
    return bytes ? at::empty({(int64_t)bytes}, t.options().dtype(at::kByte)) : Tensor();
}

#define TK3D_CALL(is32, name, ...)                                                             \
    done((is32) ? name##_f32(__VA_ARGS__) : name##_f64(__VA_ARGS__), #name)

// ---- operators ---------------------------------------------------------------------------------

struct Cloud {
    int64_t b, n;
};

Cloud cloud_dims(const char *name, const Tensor &t, bool channels_first)
{
    check_contiguous_cuda(name, t);
    check_eq(t.dim(), 3, (std::string(name) + ".dim() == 3").c_str());
    check_eq(t.size(channels_first ? 1 : 2), 3,
             (std::string(name) + (channels_first ? ".size(1) == 3" : ".size(2) == 3")).c_str());
    return {t.size(0), t.size(channels_first ? 2 : 1)};
}

std::tuple<Tensor, Tensor> fps(const Tensor &points, int64_t num_samples, bool channels_first,
                               bool want_xyz)
{
    const Cloud c = cloud_dims("points", points, channels_first);
    check(num_samples > 0,
          "Check failed: num_samples > 0 (" + std::to_string(num_samples) + " vs. 0)");
    check(c.n >= num_samples, "Check failed: points.size(1) >= num_samples (" +
                                  std::to_string(c.n) + " vs. " + std::to_string(num_samples) + ")");
    OnDeviceOf guard(points.device());
    const Tensor index = index_like(points, {c.b, num_samples});
    Tensor sampled;
    if (want_xyz)
        sampled = channels_first ? like(points, {c.b, 3, num_samples})
                                 : like(points, {c.b, num_samples, 3});
    const size_t bytes =
        tk3d_sample_farthest_points_workspace_bytes(c.b, c.n, points.element_size());
    const Tensor ws = scratch(points, bytes);
    TK3D_CALL(is_f32(points), tk3d_sample_farthest_points_gather, ptr(points), channels_first, c.b,
              c.n, num_samples, ptr(index), ptr(sampled), ptr(ws), bytes, stream_of(points));
    return {index, sampled};
}

Tensor ball_query(const Tensor &query, const Tensor &key, double radius, int64_t max_neighbors,
                  bool channels_first)
{
    const Cloud q = cloud_dims("query", query, channels_first);
    const Cloud k = cloud_dims("key", key, channels_first);
    check_eq(q.b, k.b, "query.size(0) == key.size(0)");
    check_same("query", query, "key", key);
    check(max_neighbors >= 0, "max_neighbors must be non-negative.");
    OnDeviceOf guard(query.device());
    const Tensor index = index_like(query, {q.b, q.n, max_neighbors});
    if (channels_first)
        TK3D_CALL(is_f32(query), tk3d_ball_query_bcn, ptr(query), ptr(key), q.b, q.n, k.n,
                  (float)radius, max_neighbors, ptr(index), stream_of(query));
    else
        TK3D_CALL(is_f32(query), tk3d_ball_query, ptr(query), ptr(key), q.b, q.n, k.n,
                  (float)radius, max_neighbors, ptr(index), stream_of(query));
    return index;
}

// Empty when the library has no kernel for this k on [B,3,N] clouds, or none that puts the rows in
// order or takes roots (k > 64).
std::vector<Tensor> knn(const Tensor &query, const Tensor &key, int64_t k, int64_t version,
                        bool channels_first, bool sorted = false, bool root = false)
{
    const Cloud q = cloud_dims("query", query, channels_first);
    const Cloud c = cloud_dims("key", key, channels_first);
    check_eq(c.b, q.b, "key.size(0) == query.size(0)");
    check(c.n >= k, "Check failed: key.size(1) >= k (" + std::to_string(c.n) + " vs. " +
                        std::to_string(k) + ")");
    check_same("query", query, "key", key);
    check(version == 0 || version == 1, "Invalid version");
    check(k >= 0, "k must be non-negative.");
    if ((channels_first || sorted || root) && k > 64)
        return {};
    OnDeviceOf guard(query.device());
    const Tensor distance = like(query, {q.b, q.n, k});
    const Tensor index = index_like(query, {q.b, q.n, k});
    if (k > 0 && (sorted || root)) {
        TK3D_CALL(is_f32(query), tk3d_knn_distance_ordered, ptr(query), ptr(key), channels_first, q.b,
                  q.n, c.n, k, sorted, root, ptr(distance), ptr(index), stream_of(query));
    } else if (k > 0 && channels_first) {
        const int code =
            is_f32(query)
                ? tk3d_knn_distance_bcn_f32(ptr(query), ptr(key), q.b, q.n, c.n, k, (int)version,
                                            ptr(distance), ptr(index), stream_of(query))
                : tk3d_knn_distance_bcn_f64(ptr(query), ptr(key), q.b, q.n, c.n, k, (int)version,
                                            ptr(distance), ptr(index), stream_of(query));
        if (code == TK3D_ERR_UNSUPPORTED)
            return {};
        done(code, "tk3d_knn_distance_bcn");
    } else if (k > 0) {
        TK3D_CALL(is_f32(query), tk3d_knn_distance, ptr(query), ptr(key), q.b, q.n, c.n, k,
                  (int)version, ptr(distance), ptr(index), stream_of(query));
    }
    return {distance, index};
}

std::tuple<Tensor, Tensor, Tensor> three_nn(const Tensor &query, const Tensor &key,
                                            bool channels_first, double eps)
{
    const Cloud q = cloud_dims("query", query, channels_first);
    const Cloud c = cloud_dims("key", key, channels_first);
    check_eq(q.b, c.b, "query.size(0) == key.size(0)");
    check_same("query", query, "key", key);
    check(c.n >= 3, "Check failed: key.size(1) >= k (" + std::to_string(c.n) + " vs. 3)");
    OnDeviceOf guard(query.device());
    const Tensor distance = like(query, {q.b, q.n, 3});
    const Tensor index = index_like(query, {q.b, q.n, 3});
    const Tensor weight = like(query, {q.b, q.n, 3});
    TK3D_CALL(is_f32(query), tk3d_three_nn, ptr(query), ptr(key), channels_first, q.b, q.n, c.n,
              eps, ptr(distance), ptr(index), ptr(weight), stream_of(query));
    return {distance, index, weight};
}

// sqrt(max(d, eps)) of both directions.
std::vector<Tensor> roots(const Tensor &d1, const Tensor &d2, double eps)
{
    OnDeviceOf guard(d1.device());
    const Tensor r1 = like(d1, d1.sizes()), r2 = like(d2, d2.sizes());
    TK3D_CALL(is_f32(d1), tk3d_chamfer_roots, ptr(d1), ptr(d2), d1.numel(), d2.numel(), eps, ptr(r1),
              ptr(r2), stream_of(d1));
    return {r1, r2};
}

// dist1, idx1, dist2, idx2 and, where `root`, sqrt(max(dist, eps)) of both.
std::vector<Tensor> chamfer_forward(const Tensor &xyz1, const Tensor &xyz2, bool channels_first,
                                    bool root = false, double eps = 0.0)
{
    const Cloud a = cloud_dims("xyz1", xyz1, channels_first);
    const Cloud c = cloud_dims("xyz2", xyz2, channels_first);
    check_eq(a.b, c.b, "xyz1.size(0) == xyz2.size(0)");
    check_same("xyz1", xyz1, "xyz2", xyz2);
    OnDeviceOf guard(xyz1.device());
    const Tensor dist1 = like(xyz1, {a.b, a.n}), idx1 = index_like(xyz1, {a.b, a.n});
    const Tensor dist2 = like(xyz1, {a.b, c.n}), idx2 = index_like(xyz1, {a.b, c.n});
    void *stream = stream_of(xyz1);
    const bool in_place =
        is_f32(xyz1) && tk3d_chamfer_distance_forward_in_place(a.b, a.n, c.n, channels_first);
    if (in_place && root) {
        const Tensor r1 = like(xyz1, {a.b, a.n}), r2 = like(xyz1, {a.b, c.n});
        done(tk3d_chamfer_distance_forward_roots_f32(ptr(xyz1), ptr(xyz2), channels_first, a.b, a.n, c.n,
                                                     eps, ptr(dist1), ptr(idx1), ptr(dist2), ptr(idx2),
                                                     ptr(r1), ptr(r2), stream),
             "tk3d_chamfer_distance_forward_roots_f32");
        return {dist1, idx1, dist2, idx2, r1, r2};
    }
    if (is_f32(xyz1)) {
        // Clouds of a few thousand points and more are sorted along a space-filling curve in a
        // scratch buffer, and only key tiles near a wave's queries are swept. (On [B,3,N]
        // clouds the sorted path goes up to 16384 points.)
        const bool sortable = !channels_first || std::max(a.n, c.n) <= 16384;
        const size_t bytes =
            sortable ? tk3d_chamfer_distance_forward_workspace_bytes(a.b, a.n, c.n, 0) : 0;
        const size_t copy_bytes =
            bytes || in_place ? 0 : tk3d_chamfer_distance_forward_rows_bytes(a.b, a.n, c.n, channels_first);
        const Tensor ws = scratch(xyz1, bytes ? bytes : copy_bytes);
        const auto call = channels_first ? tk3d_chamfer_distance_forward_bcn_f32
                                         : tk3d_chamfer_distance_forward_ws_f32;
        if (copy_bytes)
            done(tk3d_chamfer_distance_forward_rows_f32(
                     ptr(xyz1), ptr(xyz2), channels_first, a.b, a.n, c.n, ptr(dist1), ptr(idx1),
                     ptr(dist2), ptr(idx2), ptr(ws), copy_bytes, stream),
                 "tk3d_chamfer_distance_forward_rows_f32");
        else
            done(call(ptr(xyz1), ptr(xyz2), a.b, a.n, c.n, ptr(dist1), ptr(idx1), ptr(dist2),
                      ptr(idx2), ptr(ws), bytes, stream),
                 "tk3d_chamfer_distance_forward_f32");
    } else {
        const auto call = channels_first ? tk3d_chamfer_distance_forward_bcn_f64
                                         : tk3d_chamfer_distance_forward_f64;
        done(call(ptr(xyz1), ptr(xyz2), a.b, a.n, c.n, ptr(dist1), ptr(idx1), ptr(dist2),
                  ptr(idx2), stream),
             "tk3d_chamfer_distance_forward_f64");
    }
    if (root) {
        const std::vector<Tensor> r = roots(dist1, dist2, eps);
        return {dist1, idx1, dist2, idx2, r[0], r[1]};
    }
    return {dist1, idx1, dist2, idx2};
}

void check_chamfer_backward(const Tensor &grad1, const Tensor &grad2, const Tensor &xyz1, const Tensor &xyz2,
                            const Tensor &idx1, const Tensor &idx2, bool channels_first = false)
{
    check_contiguous_cuda("grad_dist1", grad1);
    check_contiguous_cuda("grad_dist2", grad2);
    check_contiguous_cuda("xyz1", xyz1);
    check_contiguous_cuda("xyz2", xyz2);
    check_contiguous_cuda("idx1", idx1);
    check_contiguous_cuda("idx2", idx2);
    check(grad1.dim() == 2 && grad2.dim() == 2, "grad_dist must be 2-D tensors.");
    const int64_t b = grad1.size(0), n1 = grad1.size(1), n2 = grad2.size(1);
    check_eq(grad2.size(0), b, "grad_dist2.size(0) == bs");
    check(xyz1.dim() == 3 && xyz2.dim() == 3, "xyz1 and xyz2 must be 3-D tensors.");
    check_eq(xyz1.size(0), b, "xyz1.size(0) == bs");
    check_eq(xyz2.size(0), b, "xyz2.size(0) == bs");
    if (channels_first) {
        check_eq(xyz1.size(2), n1, "xyz1.size(2) == n1");
        check_eq(xyz2.size(2), n2, "xyz2.size(2) == n2");
        check_eq(xyz1.size(1), 3, "xyz1.size(1) == 3");
        check_eq(xyz2.size(1), 3, "xyz2.size(1) == 3");
    } else {
        check_eq(xyz1.size(1), n1, "xyz1.size(1) == n1");
        check_eq(xyz2.size(1), n2, "xyz2.size(1) == n2");
        check_eq(xyz1.size(2), 3, "xyz1.size(2) == 3");
        check_eq(xyz2.size(2), 3, "xyz2.size(2) == 3");
    }
    check(idx1.dim() == 2 && idx2.dim() == 2, "idx1 and idx2 must be 2-D tensors.");
    check_eq(idx1.size(0), b, "idx1.size(0) == bs");
    check_eq(idx2.size(0), b, "idx2.size(0) == bs");
    check_eq(idx1.size(1), n1, "idx1.size(1) == n1");
    check_eq(idx2.size(1), n2, "idx2.size(1) == n2");
    check_index("idx1", idx1);
    check_index("idx2", idx2);
    check_same("grad_dist1", grad1, "xyz1", xyz1);
    check_same("grad_dist2", grad2, "xyz2", xyz2);
    check_same("xyz1", xyz1, "xyz2", xyz2);
}

// The gradients from clouds [B,N,3] and gradients of distances at `x` and `grad`; `xyz` says type and device.
std::vector<Tensor> chamfer_gradients(const Tensor &xyz, int64_t b, const int64_t (&n)[2], const Ptr (&grad)[2],
                                      const Ptr (&x)[2], const Tensor &idx1, const Tensor &idx2, bool want1, bool want2)
{
    if (!is_f32(xyz) || std::max(n[0], n[1]) > (1 << 27))
        want1 = want2 = true;  // (one gradient alone: the fp32 kernel)
    Tensor grad_xyz1, grad_xyz2;
    if (want1)
        grad_xyz1 = like(xyz, {b, n[0], 3});
    if (want2)
        grad_xyz2 = like(xyz, {b, n[1], 3});
    TK3D_CALL(is_f32(xyz), tk3d_chamfer_distance_backward, grad[0], grad[1], x[0], x[1], ptr(idx1), ptr(idx2), b,
              n[0], n[1], ptr(grad_xyz1), ptr(grad_xyz2), stream_of(xyz));
    return {grad_xyz1, grad_xyz2};
}

std::vector<Tensor> chamfer_backward(const Tensor &grad1, const Tensor &grad2, const Tensor &xyz1,
                                     const Tensor &xyz2, const Tensor &idx1, const Tensor &idx2)
{
    check_chamfer_backward(grad1, grad2, xyz1, xyz2, idx1, idx2);
    OnDeviceOf guard(xyz1.device());
    return chamfer_gradients(xyz1, grad1.size(0), {grad1.size(1), grad2.size(1)}, {ptr(grad1), ptr(grad2)},
                             {ptr(xyz1), ptr(xyz2)}, idx1, idx2, true, true);
}

// The same of what the forward call leaves: clouds of either layout, and gradients of the distances or of their roots
// (`of` then holds both distances and both roots).
std::vector<Tensor> chamfer_backward_forms(const Tensor &grad1, const Tensor &grad2, const Tensor &xyz1,
                                           const Tensor &xyz2, const Tensor &idx1, const Tensor &idx2,
                                           const Tensor *of, double eps, bool channels_first, bool want1, bool want2)
{
    check_chamfer_backward(grad1, grad2, xyz1, xyz2, idx1, idx2, channels_first);
    for (int i = 0; of && i < 4; ++i) {
        check_contiguous_cuda("dist", of[i]);
        check_same("dist", of[i], "xyz1", xyz1);
        check(of[i].sizes() == (i % 2 ? grad2 : grad1).sizes(), "distances and grad_dist differ in shape.");
    }
    OnDeviceOf guard(xyz1.device());
    const int64_t b = grad1.size(0), n[2] = {grad1.size(1), grad2.size(1)};
    void *const stream = stream_of(xyz1);
    // (asked before anything is allocated: a call on few long clouds takes as long as its host work)
    if (is_f32(xyz1) && (channels_first || of) &&
        tk3d_chamfer_distance_backward_takes_forms(channels_first, of != nullptr, n[0], n[1])) {
        Tensor grad_xyz1, grad_xyz2;
        if (want1)
            grad_xyz1 = like(xyz1, {b, n[0], 3});
        if (want2)
            grad_xyz2 = like(xyz2, {b, n[1], 3});
        done(tk3d_chamfer_distance_backward_forms_f32(
                 ptr(grad1), ptr(grad2), ptr(xyz1), ptr(xyz2), ptr(idx1), ptr(idx2), of ? ptr(of[0]) : Ptr{},
                 of ? ptr(of[1]) : Ptr{}, of ? ptr(of[2]) : Ptr{}, of ? ptr(of[3]) : Ptr{}, eps, channels_first, b, n[0],
                 n[1], ptr(grad_xyz1), ptr(grad_xyz2), stream),
             "tk3d_chamfer_distance_backward_forms_f32");
        return {grad_xyz1, grad_xyz2};
    }
    // The other kernels work on [B,N,3] and gradients of distances: copies and gradients, all in one tensor.
    Ptr x[2] = {ptr(xyz1), ptr(xyz2)}, g[2] = {ptr(grad1), ptr(grad2)};
    Tensor work;
    const int64_t points = b * (n[0] + n[1]);
    if (points > 0 && (channels_first || of)) {
        work = like(xyz1, {points * ((channels_first ? 3 : 0) + (of ? 1 : 0))});
        char *at = static_cast<char *>(work.data_ptr());
        const auto take = [&](int64_t elements) {
            const Ptr p{at};
            at += elements * (int64_t)work.element_size();
            return p;
        };
        const Ptr rows[2] = {channels_first ? take(b * n[0] * 3) : Ptr{}, channels_first ? take(b * n[1] * 3) : Ptr{}};
        const Ptr of_dist[2] = {of ? take(b * n[0]) : Ptr{}, of ? take(b * n[1]) : Ptr{}};
        if (of && channels_first && is_f32(xyz1))
            done(tk3d_chamfer_root_grads_rows_f32(g[0], g[1], ptr(of[0]), ptr(of[1]), ptr(of[2]), ptr(of[3]), x[0], x[1],
                                                  b, n[0], n[1], eps, of_dist[0], of_dist[1], rows[0], rows[1], stream),
                 "tk3d_chamfer_root_grads_rows_f32");
        else {
            if (of)
                TK3D_CALL(is_f32(xyz1), tk3d_chamfer_root_grads, g[0], g[1], ptr(of[0]), ptr(of[1]), ptr(of[2]),
                          ptr(of[3]), grad1.numel(), grad2.numel(), eps, of_dist[0], of_dist[1], stream);
            if (channels_first)
                TK3D_CALL(is_f32(xyz1), tk3d_chamfer_rows, x[0], x[1], 1, b, n[0], n[1], n[0], n[1], rows[0], rows[1],
                          stream);
        }
        for (int i = 0; i < 2; ++i) {
            x[i] = channels_first ? rows[i] : x[i];
            g[i] = of ? of_dist[i] : g[i];
        }
    }
    return chamfer_gradients(xyz1, b, n, g, x, idx1, idx2, want1, want2);
}

// Like the reference (which goes through at::gather) non-contiguous tensors are accepted.
Tensor group_forward(const Tensor &input_, const Tensor &index_)
{
    check_cuda("input", input_);
    check_cuda("index", index_);
    check_eq(input_.dim(), 3, "input.dim() == 3");
    check_eq(index_.dim(), 3, "index.dim() == 3");
    check_eq(input_.size(0), index_.size(0), "input.size(0) == index.size(0)");
    check_index("index", index_);
    OnDeviceOf guard(input_.device());
    const Tensor input = input_.contiguous(), index = index_.contiguous();
    const int64_t b = input.size(0), c = input.size(1), n2 = index.size(1), k = index.size(2);
    const Tensor output = like(input, {b, c, n2, k});
    TK3D_CALL(is_f32(input), tk3d_group_points_forward, ptr(input), ptr(index), b, c,
              input.size(2), n2, k, ptr(output), stream_of(input));
    return output;
}

void check_grouped_grad(const Tensor &grad, const Tensor &index)
{
    check_contiguous_cuda("grad_output", grad);
    check_contiguous_cuda("index", index);
    check_eq(grad.dim(), 4, "grad_output.dim() == 4");
    check_eq(index.dim(), 3, "index.dim() == 3");
    check_eq(index.size(0), grad.size(0), "index.size(0) == grad_output.size(0)");
    check_eq(index.size(1), grad.size(2), "index.size(1) == grad_output.size(2)");
    check_eq(index.size(2), grad.size(3), "index.size(2) == grad_output.size(3)");
    check_index("index", index);
}

Tensor group_backward(const Tensor &grad, const Tensor &index, int64_t n1)
{
    check_grouped_grad(grad, index);
    OnDeviceOf guard(grad.device());
    const Tensor out = like(grad, {grad.size(0), grad.size(1), n1});
    TK3D_CALL(is_f32(grad), tk3d_group_points_backward, ptr(grad), ptr(index), grad.size(0),
              grad.size(1), n1, grad.size(2), grad.size(3), ptr(out), stream_of(grad));
    return out;
}

Tensor group_concat_forward(const Tensor &feature, const Tensor &xyz, const Tensor &centre,
                            const Tensor &index)
{
    const Cloud p = cloud_dims("xyz", xyz, true);
    const Cloud m = cloud_dims("centre", centre, true);
    check_eq(p.b, m.b, "xyz.size(0) == centre.size(0)");
    check_same("xyz", xyz, "centre", centre);
    check_contiguous_cuda("index", index);
    check_index("index", index);
    check_eq(index.dim(), 3, "index.dim() == 3");
    check_eq(index.size(0), p.b, "index.size(0) == xyz.size(0)");
    check_eq(index.size(1), m.n, "index.size(1) == centre.size(2)");
    int64_t c = 0;
    if (feature.defined()) {
        check_contiguous_cuda("feature", feature);
        check_eq(feature.dim(), 3, "feature.dim() == 3");
        check_eq(feature.size(0), p.b, "feature.size(0) == xyz.size(0)");
        check_eq(feature.size(2), p.n, "feature.size(2) == xyz.size(2)");
        check_same("feature", feature, "xyz", xyz);
        c = feature.size(1);
    }
    OnDeviceOf guard(xyz.device());
    const Tensor out = like(xyz, {p.b, c + 3, m.n, index.size(2)});
    TK3D_CALL(is_f32(xyz), tk3d_group_points_concat_forward, ptr(feature), ptr(xyz), ptr(centre),
              ptr(index), p.b, c, p.n, m.n, index.size(2), ptr(out), stream_of(xyz));
    return out;
}

std::tuple<Tensor, Tensor> group_concat_backward(const Tensor &grad, const Tensor &index,
                                                 int64_t n1, bool want_feature, bool want_xyz)
{
    check_grouped_grad(grad, index);
    const int64_t b = grad.size(0), c = grad.size(1) - 3;
    check(c >= 0, "grad_output must have at least 3 channels.");
    OnDeviceOf guard(grad.device());
    Tensor feature, xyz;
    if (want_feature && c > 0)
        feature = like(grad, {b, c, n1});
    if (want_xyz)
        xyz = like(grad, {b, 3, n1});
    if (feature.defined() || xyz.defined())
        TK3D_CALL(is_f32(grad), tk3d_group_points_concat_backward, ptr(grad), ptr(index), b, c, n1,
                  grad.size(2), grad.size(3), ptr(feature), ptr(xyz), stream_of(grad));
    return {feature, xyz};
}

void check_interpolate(const char *name, const Tensor &first, const Tensor &index,
                       const Tensor &weight)
{
    const std::string n(name);
    check_contiguous_cuda(name, first);
    check_contiguous_cuda("index", index);
    check_contiguous_cuda("weight", weight);
    check_eq(first.dim(), 3, (n + ".dim() == 3").c_str());
    check_eq(index.dim(), 3, "index.dim() == 3");
    check_eq(weight.dim(), 3, "weight.dim() == 3");
    check_eq(first.size(0), index.size(0), (n + ".size(0) == index.size(0)").c_str());
    check_eq(first.size(0), weight.size(0), (n + ".size(0) == weight.size(0)").c_str());
    check_eq(index.size(1), weight.size(1), "index.size(1) == weight.size(1)");
    check_eq(index.size(2), weight.size(2), "index.size(2) == weight.size(2)");
    check_index("index", index);
    check_same(name, first, "weight", weight);
}

Tensor interpolate_forward(const Tensor &input, const Tensor &index, const Tensor &weight)
{
    check_interpolate("input", input, index, weight);
    check_eq(index.size(2), 3, "index.size(2) == 3");
    OnDeviceOf guard(input.device());
    const Tensor out = like(input, {input.size(0), input.size(1), index.size(1)});
    TK3D_CALL(is_f32(input), tk3d_interpolate_forward, ptr(input), ptr(index), ptr(weight),
              input.size(0), input.size(1), input.size(2), index.size(1), index.size(2), ptr(out),
              stream_of(input));
    return out;
}

Tensor interpolate_backward(const Tensor &grad, const Tensor &index, const Tensor &weight,
                            int64_t n1)
{
    check_interpolate("grad_output", grad, index, weight);
    check_eq(grad.size(2), index.size(1), "grad_output.size(2) == index.size(1)");
    check(index.size(2) == 3, "Only support k=3.");
    OnDeviceOf guard(grad.device());
    const Tensor out = like(grad, {grad.size(0), grad.size(1), n1});
    TK3D_CALL(is_f32(grad), tk3d_interpolate_backward, ptr(grad), ptr(index), ptr(weight),
              grad.size(0), grad.size(1), n1, grad.size(2), index.size(2), ptr(out),
              stream_of(grad));
    return out;
}

// ---- autograd nodes ------------------------------------------------------------------------------

template <typename... T> bool tracked(const T &...t)
{
    return c10::GradMode::is_enabled() && ((t.defined() && t.requires_grad()) || ...);
}

struct ChamferNode : torch::autograd::Function<ChamferNode> {
    static variable_list forward(AutogradContext *ctx, const Tensor &xyz1, const Tensor &xyz2,
                                 bool channels_first, bool root, double eps)
    {
        const Tensor a = xyz1.contiguous(), c = xyz2.contiguous();
        const std::vector<Tensor> out = chamfer_forward(a, c, channels_first, root, eps);
        ctx->saved_data["channels_first"] = channels_first;
        ctx->saved_data["want"] = (xyz1.requires_grad() ? 1 : 0) + (xyz2.requires_grad() ? 2 : 0);
        if (!root) {
            ctx->save_for_backward({a, c, out[1], out[3]});
            return {out[0], out[2]};
        }
        ctx->saved_data["eps"] = eps;
        ctx->save_for_backward({a, c, out[1], out[3], out[0], out[2], out[4], out[5]});
        return {out[4], out[5]};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = dense(ctx->get_saved_variables());
        const int64_t want = ctx->saved_data["want"].toInt();
        const bool channels_first = ctx->saved_data["channels_first"].toBool();
        const Tensor g1 = grads[0].contiguous(), g2 = grads[1].contiguous();
        const bool roots = saved.size() > 4;
        std::vector<Tensor> g = chamfer_backward_forms(g1, g2, saved[0], saved[1], saved[2], saved[3],
                                                       roots ? &saved[4] : nullptr,
                                                       roots ? ctx->saved_data["eps"].toDouble() : 0.0, channels_first,
                                                       (want & 1) != 0, (want & 2) != 0);
        for (int i = 0; i < 2; ++i) {
            if (!(want & (1 << i)))
                g[i] = Tensor();
            else if (channels_first)
                g[i] = g[i].transpose(1, 2);
        }
        return {g[0], g[1], Tensor(), Tensor(), Tensor()};
    }
};

std::tuple<Tensor, Tensor> chamfer(const Tensor &xyz1, const Tensor &xyz2, bool channels_first,
                                   bool root, double eps)
{
    if (tracked(xyz1, xyz2)) {
        const variable_list out = ChamferNode::apply(xyz1, xyz2, channels_first, root, eps);
        return {out[0], out[1]};
    }
    const std::vector<Tensor> out =
        chamfer_forward(xyz1.contiguous(), xyz2.contiguous(), channels_first, root, eps);
    return root ? std::tuple<Tensor, Tensor>{out[4], out[5]} : std::tuple<Tensor, Tensor>{out[0], out[2]};
}

struct GroupNode : torch::autograd::Function<GroupNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &points, const Tensor &index)
    {
        ctx->save_for_backward({index});
        ctx->saved_data["n"] = points.size(2);
        return group_forward(points, index);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        return {group_backward(grads[0].contiguous(), saved[0].contiguous(),
                               ctx->saved_data["n"].toInt()),
                Tensor()};
    }
};

Tensor group_points(const Tensor &points, const Tensor &index)
{
    if (tracked(points))
        return GroupNode::apply(points, index);
    return group_forward(points, index);
}

struct GroupConcatNode : torch::autograd::Function<GroupConcatNode> {
    static Tensor forward(AutogradContext *ctx, const std::optional<Tensor> &maybe_feature,
                          const Tensor &xyz, const Tensor &centre, const Tensor &index)
    {
        const Tensor feature = maybe_feature.value_or(Tensor());
        ctx->save_for_backward({index});
        ctx->saved_data["n"] = xyz.size(2);
        ctx->saved_data["feature"] = feature.defined() && feature.requires_grad();
        ctx->saved_data["xyz"] = xyz.requires_grad();
        ctx->saved_data["centre"] = centre.requires_grad();
        return group_concat_forward(feature.defined() ? feature.contiguous() : feature,
                                    xyz.contiguous(), centre.contiguous(), index.contiguous());
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor grad = grads[0].contiguous();
        auto [feature, xyz] = group_concat_backward(
            grad, saved[0].contiguous(), ctx->saved_data["n"].toInt(),
            ctx->saved_data["feature"].toBool(), ctx->saved_data["xyz"].toBool());
        Tensor centre;
        if (ctx->saved_data["centre"].toBool())
            centre = grad.narrow(1, grad.size(1) - 3, 3).sum(3).neg();
        return {feature, xyz, centre, Tensor()};
    }
};

Tensor group_points_with_xyz(const Tensor &feature, const Tensor &xyz, const Tensor &centre,
                             const Tensor &index)
{
    if (tracked(feature, xyz, centre))
        return GroupConcatNode::apply(
            feature.defined() ? std::optional<Tensor>(feature) : std::nullopt, xyz, centre, index);
    return group_concat_forward(feature.defined() ? feature.contiguous() : feature,
                                xyz.contiguous(), centre.contiguous(), index.contiguous());
}

struct InterpolateNode : torch::autograd::Function<InterpolateNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &feature, const Tensor &index,
                          const Tensor &weight)
    {
        ctx->save_for_backward({index, weight});
        ctx->saved_data["n"] = feature.size(2);
        return interpolate_forward(feature.contiguous(), index.contiguous(), weight.contiguous());
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        return {interpolate_backward(grads[0].contiguous(), saved[0].contiguous(),
                                     saved[1].contiguous(), ctx->saved_data["n"].toInt()),
                Tensor(), Tensor()};
    }
};

Tensor interpolate(const Tensor &feature, const Tensor &index, const Tensor &weight)
{
    if (tracked(feature, weight))
        return InterpolateNode::apply(feature, index, weight);
    return interpolate_forward(feature.contiguous(), index.contiguous(), weight.contiguous());
}

// ---- Python ----------------------------------------------------------------------------------------

Tensor optional_arg(const char *name, py::handle h)
{
    return h.is_none() ? Tensor() : tensor_arg(name, h);
}

// Runs an operator without the interpreter lock.
template <typename F> auto unlocked(F &&f)
{
    py::gil_scoped_release release;
    return f();
}

}  // namespace

PYBIND11_MODULE(_host, m)
{
    m.def("sample_farthest_points",
          [](py::handle points, int64_t k, bool channels_first, bool want_xyz) {
              const Tensor p = tensor_arg("points", points);
              return unlocked([&] { return fps(p, k, channels_first, want_xyz); });
          });
    m.def("ball_query", [](py::handle query, py::handle key, double radius, int64_t k,
                           bool channels_first) {
        const Tensor q = tensor_arg("query", query), c = tensor_arg("key", key);
        return unlocked([&] { return ball_query(q, c, radius, k, channels_first); });
    });
    m.def(
        "knn",
        [](py::handle query, py::handle key, int64_t k, int64_t version, bool channels_first,
           bool sorted, bool root) {
            const Tensor q = tensor_arg("query", query), c = tensor_arg("key", key);
            return unlocked([&] { return knn(q, c, k, version, channels_first, sorted, root); });
        },
        py::arg("query"), py::arg("key"), py::arg("k"), py::arg("version"),
        py::arg("channels_first"), py::arg("sorted") = false, py::arg("root") = false);
    m.def("three_nn", [](py::handle query, py::handle key, bool channels_first, double eps) {
        const Tensor q = tensor_arg("query", query), c = tensor_arg("key", key);
        return unlocked([&] { return three_nn(q, c, channels_first, eps); });
    });
    m.def("chamfer_forward", [](py::handle xyz1, py::handle xyz2, bool channels_first) {
        const Tensor a = tensor_arg("xyz1", xyz1), c = tensor_arg("xyz2", xyz2);
        return unlocked([&] { return chamfer_forward(a, c, channels_first); });
    });
    m.def("chamfer_backward", [](py::handle grad1, py::handle grad2, py::handle xyz1,
                                 py::handle xyz2, py::handle idx1, py::handle idx2) {
        const Tensor t[] = {tensor_arg("grad_dist1", grad1), tensor_arg("grad_dist2", grad2),
                            tensor_arg("xyz1", xyz1),        tensor_arg("xyz2", xyz2),
                            tensor_arg("idx1", idx1),        tensor_arg("idx2", idx2)};
        return unlocked([&] { return chamfer_backward(t[0], t[1], t[2], t[3], t[4], t[5]); });
    });
    m.def("group_forward", [](py::handle input, py::handle index) {
        const Tensor x = tensor_arg("input", input), i = tensor_arg("index", index);
        return unlocked([&] { return group_forward(x, i); });
    });
    m.def("group_backward", [](py::handle grad, py::handle index, int64_t n1) {
        const Tensor g = tensor_arg("grad_output", grad), i = tensor_arg("index", index);
        return unlocked([&] { return group_backward(g, i, n1); });
    });
    m.def("group_concat_forward", [](py::handle feature, py::handle xyz, py::handle centre,
                                     py::handle index) {
        const Tensor f = optional_arg("feature", feature), x = tensor_arg("xyz", xyz),
                     c = tensor_arg("centre", centre), i = tensor_arg("index", index);
        return unlocked([&] { return group_concat_forward(f, x, c, i); });
    });
    m.def("group_concat_backward", [](py::handle grad, py::handle index, int64_t n1,
                                      bool want_feature, bool want_xyz) {
        const Tensor g = tensor_arg("grad_output", grad), i = tensor_arg("index", index);
        return unlocked([&] { return group_concat_backward(g, i, n1, want_feature, want_xyz); });
    });
    m.def("interpolate_forward", [](py::handle input, py::handle index, py::handle weight) {
        const Tensor x = tensor_arg("input", input), i = tensor_arg("index", index),
                     w = tensor_arg("weight", weight);
        return unlocked([&] { return interpolate_forward(x, i, w); });
    });
    m.def("interpolate_backward", [](py::handle grad, py::handle index, py::handle weight,
                                     int64_t n1) {
        const Tensor g = tensor_arg("grad_output", grad), i = tensor_arg("index", index),
                     w = tensor_arg("weight", weight);
        return unlocked([&] { return interpolate_backward(g, i, w, n1); });
    });

    // Whether a call on these arguments may go straight to the functions here. Where a tracer, a
    // function transform or a dispatch mode is active, or a tensor carries a forward-mode tangent,
    // these would leave nothing to see: a trace would hold memory that nobody fills, a tangent would
    // be lost. The caller then takes its torch.autograd.Function, which such things know.
    m.def("direct", [](py::args args) {
        if (watched())
            return false;
        for (const py::handle h : args)
            if (THPVariable_Check(h.ptr()) && !plain(THPVariable_Unpack(h.ptr())))
                return false;
        return true;
    });

    // differentiable forms
    m.def("chamfer", [](py::handle xyz1, py::handle xyz2, bool channels_first, bool root,
                        double eps) {
        const Tensor a = tensor_arg("xyz1", xyz1), c = tensor_arg("xyz2", xyz2);
        return unlocked([&] { return chamfer(a, c, channels_first, root, eps); });
    });
    m.def("group_points", [](py::handle points, py::handle index) {
        const Tensor x = tensor_arg("input", points), i = tensor_arg("index", index);
        return unlocked([&] { return group_points(x, i); });
    });
    m.def("group_points_with_xyz", [](py::handle feature, py::handle xyz, py::handle centre,
                                      py::handle index) {
        const Tensor f = optional_arg("feature", feature), x = tensor_arg("xyz", xyz),
                     c = tensor_arg("centre", centre), i = tensor_arg("index", index);
        return unlocked([&] { return group_points_with_xyz(f, x, c, i); });
    });
    m.def("interpolate", [](py::handle feature, py::handle index, py::handle weight) {
        const Tensor x = tensor_arg("input", feature), i = tensor_arg("index", index),
                     w = tensor_arg("weight", weight);
        return unlocked([&] { return interpolate(x, i, w); });
    });
    m.def("mlp", [](py::handle x, py::handle x2, py::handle xyz, py::handle centre,
                    py::handle index, std::vector<Tensor> params, std::vector<Tensor> buffers,
                    std::vector<double> eps, std::vector<double> momentum, bool training,
                    int64_t pool) {
        const Tensor t[] = {optional_arg("x", x), optional_arg("x2", x2), optional_arg("xyz", xyz),
                            optional_arg("centre", centre), optional_arg("index", index)};
        return unlocked([&] {
            const variable_list made = mlp(t[0], t[1], t[2], t[3], t[4], std::move(params),
                                           std::move(buffers), std::move(eps), std::move(momentum),
                                           training, pool);
            return made.empty() ? Tensor() : made[0];
        });
    });
    // (values, places), or an empty list
    m.def("mlp_max", [](py::handle x, std::vector<Tensor> params, std::vector<Tensor> buffers,
                        std::vector<double> eps, std::vector<double> momentum, bool training) {
        const Tensor in = tensor_arg("x", x), none;
        return unlocked([&] {
            return mlp(in, none, none, none, none, std::move(params), std::move(buffers),
                       std::move(eps), std::move(momentum), training, -1);
        });
    });
    m.def("edge_lists", [](py::handle index, int64_t n) {
        const Tensor i = tensor_arg("index", index);
        return unlocked([&] { return edge_lists(i, n); });
    });
    m.def("edge_conv", [](py::handle x, py::handle index, py::handle lists,
                          std::vector<Tensor> params, std::vector<Tensor> buffers, double eps,
                          double momentum, bool training) {
        const Tensor t[] = {tensor_arg("x", x), tensor_arg("index", index),
                            optional_arg("lists", lists)};
        return unlocked([&] {
            return edge_conv(t[0], t[1], t[2], params, buffers, eps, momentum, training);
        });
    });
}
