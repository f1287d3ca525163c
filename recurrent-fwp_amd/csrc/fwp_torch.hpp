// What the host bindings of libfwp_hip.so share: errors, tensor checks, views, the current stream.
#pragma once
#include <torch/extension.h>

// FWP_HOST_STUB: a build for tests of the host logic on a machine without a GPU (tests/host_stub/):
// tensors may live in host memory, the stream handed to the C ABI is NULL, and the library it is linked
// against is a stand-in whose entry points launch nothing.  The product is built without it.
#ifndef FWP_HOST_STUB
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#endif

#include <stdexcept>
#include <string>

#include "fwp_hip.h"

namespace fwp_host {

// Raised to Python as the package's FwpError (set_error_class), a RuntimeError otherwise.
struct fwp_failure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
[[noreturn]] inline void fail(const std::string &what) { throw fwp_failure(what); }

// The reference checks shapes with assert; so do the Python Functions, and so does this.
struct fwp_assertion : std::runtime_error {
    using std::runtime_error::runtime_error;
};
inline void require(bool ok, const char *what) {
    if (!ok) throw fwp_assertion(what);
}

inline bool same_shape(const at::Tensor &t, std::initializer_list<int64_t> shape) { return t.sizes() == at::IntArrayRef(shape); }

inline void require_state(const at::Tensor &t, const char *name) {
    if (!t.is_contiguous() || t.scalar_type() != at::kFloat) fail(std::string(name) + " must be a contiguous fp32 tensor");
}

inline void check(int rc, const char *what) {
    if (rc != 0)
        fail(std::string(what) + " failed: " + fwp_strerror(rc) + " (code " + std::to_string(rc) + ")");
}

inline std::string shape_of(const at::Tensor &t) {
    std::string s = "(";
    for (int64_t i = 0; i < t.dim(); i++) s += (i ? ", " : "") + std::to_string(t.size(i));
    return s + ")";
}

// A view argument for a 4-D fp32 tensor.  Permuted views are passed as they are; a copy is made
// when the last axis is strided, and when rows of a multiple of 4 floats are not 16-byte aligned
// (one elementwise pass costs far less than giving up the kernels that read 16 bytes at a time).
inline at::Tensor rows(const at::Tensor &t_in, fwp_view &v) {
    at::Tensor t = t_in;
    if (t.scalar_type() != at::kFloat) fail("fast-weight operators are fp32 only");
    if (t.dim() != 4) fail("expected a 4-D [N,H,L,D] tensor, got " + std::to_string(t.dim()) + "-D");
    const int64_t d = t.size(3);
    if (t.is_contiguous()) {
        if (d % 4 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) t = t.clone();
    } else {
        const auto s = t.strides();
        if (d != 1 && s[3] != 1) t = t.contiguous();
        else if (d % 4 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 || s[0] % 4 || s[1] % 4 || s[2] % 4))
            t = t.contiguous();
    }
    v.ptr = t.data_ptr<float>();
    v.sN = t.stride(0);
    v.sH = t.stride(1);
    v.sL = t.stride(2);
    return t;
}

#ifndef FWP_HOST_STUB
// The device check of a GPU runs once per thread that uses it: the last device a thread saw pass is
// remembered without a lock.
inline void require_device(const at::Tensor &t) {
    if (!t.is_cuda()) fail("fast-weight operators need tensors on an MI355X GPU, got device '" + t.device().str() + "'");
    thread_local int passed = -1;
    const int idx = t.get_device();
    if (idx == passed) return;
    {
        c10::DeviceGuard guard(t.device());
        check(fwp_check_device(), "device check");
    }
    passed = idx;
}

inline void *stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

struct LaunchGuard {      // makes the tensors' GPU current for a launch when it is not
    c10::OptionalDeviceGuard guard;
    explicit LaunchGuard(const at::Tensor &t) {
        if (t.get_device() != c10::hip::current_device()) guard.reset_device(t.device());
    }
};
#else
inline void require_device(const at::Tensor &) {}
inline void *stream_of(const at::Tensor &) { return nullptr; }
struct LaunchGuard {
    explicit LaunchGuard(const at::Tensor &) {}
};
#endif

// The view of a tensor that rows() has already passed (a saved tensor in a backward pass).
inline fwp_view view_of(const at::Tensor &t) {
    return {static_cast<const float *>(t.const_data_ptr()), t.stride(0), t.stride(1), t.stride(2)};
}

// Scratch for a delta-rule call whose sequences run as several segments at once; undefined: they do not.
inline at::Tensor segment_work(int64_t N, int64_t H, int64_t L, int64_t E, int64_t M, int chunk, const at::TensorOptions &opts,
                               bool backward) {
    const int64_t n = (backward ? fwp_delta_bwd_segment_floats : fwp_delta_segment_floats)((int)N, (int)H, (int)L, (int)E, (int)M, chunk);
    return n > 0 ? at::empty({n}, opts) : at::Tensor();
}

// Several contiguous fp32 results of one call in one allocation: `sizes[i]` floats each, every part
// starting at a multiple of 4 floats (16 bytes, which the kernels that store 16 bytes at a time need).
struct Parts {
    at::Tensor buf;
    int64_t at = 0;
    Parts(std::initializer_list<int64_t> sizes, const at::TensorOptions &opts) {
        int64_t total = 0;
        for (int64_t n : sizes) total += (n + 3) & ~int64_t(3);
        buf = at::empty({total}, opts);
    }
    // the next part, shaped [a, b, c, d] (contiguous)
    at::Tensor take(int64_t a, int64_t b, int64_t c, int64_t d) {
        const at::Tensor t = buf.as_strided({a, b, c, d}, {b * c * d, c * d, d, 1}, at);
        at += (a * b * c * d + 3) & ~int64_t(3);
        return t;
    }
};

// Every tensor of a call lives on the first one's GPU: the kernels get raw addresses, and an address
// of host memory or of another GPU would be a memory fault there, not an exception.
inline void same_device(const at::Tensor &ref, std::initializer_list<at::Tensor> others) {
    for (const at::Tensor &t : others)
        if (t.defined() && t.device() != ref.device())
            fail("all tensors of a call must be on the same device: got '" + t.device().str() + "' beside '" +
                 ref.device().str() + "'");
}

}  // namespace fwp_host

using namespace fwp_host;
