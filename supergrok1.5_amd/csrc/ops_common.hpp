// Argument checks and workspace shared by the translation units of the torch
// extension (plain C++: no device code).
#pragma once
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>

#include "../../include/sg_abi.h"

inline void* current_stream(const torch::Tensor& t) {
    return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

inline int dtype_code(const torch::Tensor& t, const char* what) {
    switch (t.scalar_type()) {
        case torch::kFloat32: return SG_F32;
        case torch::kFloat16: return SG_F16;
        case torch::kBFloat16: return SG_BF16;
        default: TORCH_CHECK(false, what, ": unsupported dtype ", t.scalar_type());
    }
    return -1;
}

inline void check_gpu(const torch::Tensor& t, const char* fn, const char* what) {
    if (!t.is_cuda()) throw std::runtime_error(std::string(fn) + " requires CUDA tensors (" + what + " is on the CPU).");
    TORCH_CHECK(t.is_contiguous(), fn, ": ", what, " must be contiguous");
}
inline void check_f32(const torch::Tensor& t, const char* fn, const char* what) {
    check_gpu(t, fn, what);
    TORCH_CHECK(t.scalar_type() == torch::kFloat32, fn, ": ", what, " must be float32");
}

inline torch::Tensor make_workspace(size_t bytes, const torch::Tensor& like) {
    return torch::empty({(int64_t)std::max<size_t>(bytes, 256)},
                        torch::TensorOptions().device(like.device()).dtype(torch::kUInt8));
}

inline void check_status(int rc, const char* fn) { TORCH_CHECK(rc == 0, fn, ": ", sg_last_error()); }

extern int g_sg15_gelu_mode;   // 0 exact erf GELU, 1 sigmoid approximation

// the 33 meta-net weight tensors of the v2 step: fp32, on the GPU, of the sizes that the dimensions ask for
void check_sg2_weights(const char* fn, const torch::Tensor* const (&w)[SG2_NUM_WEIGHTS], const SgDims& d, Sg2Weights* W);

void bind_group_steps(pybind11::module_& m);      // ops_group.cpp
