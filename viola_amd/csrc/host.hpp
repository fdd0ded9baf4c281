// Shared by the two native host files (host.cpp: modules, host_optim.cpp: optimizer and wire codec): calling the library's
// entry points, tensor helpers, arenas.
#pragma once
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "../../include/viola_hip.h"

namespace viola_host {

namespace py = pybind11;
using at::Tensor;

// ---------------------------------------------------------------------------------------------------- calls
// Instrumented mode (the `timeline` of viola_amd._lib): every call is bracketed by two timing events on the current stream.
inline std::atomic<bool> recording{false};
// the list and torch.cuda.Event; process-wide and never released (the interpreter may be gone before static destructors run)
inline py::object* timeline_sink = nullptr;
inline py::object* event_class = nullptr;

inline void check(const char* name, int status) {
    TORCH_CHECK(status == 0, name, " failed: ", viola_error_string(status), " (status ", status, ")");
}

template <typename F>
int timed(const char* name, F&& f) {
    if (__builtin_expect(!recording.load(std::memory_order_relaxed), 1)) return f();
    py::gil_scoped_acquire gil;
    if (!timeline_sink || timeline_sink->is_none()) return f();
    py::object start = (*event_class)(py::arg("enable_timing") = true), end = (*event_class)(py::arg("enable_timing") = true);
    start.attr("record")();
    const int status = f();
    end.attr("record")();
    timeline_sink->attr("append")(py::make_tuple(name, start, end));
    return status;
}
// VIOLA_CALL raises on a non-zero status, VIOLA_TRY hands VIOLA_EUNSUPPORTED back to a caller that has another route
#define VIOLA_CALL(fn, ...) check(#fn, timed(#fn, [&] { return fn(__VA_ARGS__); }))
#define VIOLA_TRY(fn, ...) timed(#fn, [&] { return fn(__VA_ARGS__); })

inline int code_of(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return VIOLA_F32;
        case at::kBFloat16: return VIOLA_BF16;
        case at::kHalf: return VIOLA_F16;
        case at::kFloat8_e4m3fn: return VIOLA_E4M3;
        case at::kFloat8_e5m2: return VIOLA_E5M2;
        default: TORCH_CHECK(false, "viola_amd kernels do not take tensors of type ", t);
    }
}

inline viola_stream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline const void* ptr(const Tensor& t) { return t.defined() && t.numel() ? t.const_data_ptr() : nullptr; }
inline int64_t ceil_to(int64_t n, int64_t unit) { return (n + unit - 1) / unit * unit; }
inline int64_t ceil_div(int64_t n, int64_t unit) { return (n + unit - 1) / unit; }

// Several buffers of one lifetime as one allocation: take() reserves, make() allocates, at() hands out addresses.
class Arena {
public:
    int64_t take(int64_t bytes) {
        const int64_t begin = size_;
        size_ += ceil_to(bytes, 256);
        return begin;
    }
    void make(const at::Device& device) {
        if (size_) buffer_ = at::empty({size_}, at::TensorOptions().dtype(at::kByte).device(device));
    }
    void* at(int64_t offset) const { return static_cast<char*>(buffer_.mutable_data_ptr()) + offset; }
    template <typename T> T* as(int64_t offset) const { return static_cast<T*>(at(offset)); }
    void release() { buffer_ = Tensor(); }
    const Tensor& tensor() const { return buffer_; }
    int64_t size() const { return size_; }

private:
    int64_t size_ = 0;
    Tensor buffer_;
};

void register_optimizer(py::module_& m);                         // host_optim.cpp

}  // namespace viola_host
