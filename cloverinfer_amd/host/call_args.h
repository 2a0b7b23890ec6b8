// call_args.h - argument blocks of the C ABI from tensors (call_args.cpp).
#pragma once

#include <torch/extension.h>

namespace clv_host {

// Each fills the ctypes structure at address dst (clv_decode_args,
// clv_prefill_args, clv_cache_args) and returns true, or returns false having
// written nothing.
bool fill_decode_args(uintptr_t dst, py::object out, py::object q, py::object k, py::object v,
                      py::object bt, py::object cl, int64_t block_size, int64_t max_context_len,
                      py::object scale);
bool fill_prefill_args(uintptr_t dst, py::object out, py::object q, py::object k, py::object v,
                       py::object bt, py::object cl, py::object qsl, int64_t max_query_len,
                       py::object scale);
bool fill_cache_args(uintptr_t dst, py::object key, py::object value, py::object k, py::object v,
                     py::object slots);

// What the blocks' layout was when this was compiled (cloverinfer_amd/_native.py,
// call_args_layout): the functions above are called only where it still is.
py::tuple call_args_layout();

}  // namespace clv_host
