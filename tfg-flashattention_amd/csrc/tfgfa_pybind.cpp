// tfgfa_pybind.cpp - pybind11 module `custom_flash_attn._C`, a thin layer over the C ABI.
//
// Plays the role of the reference's PYBIND11_MODULE (src/cpp/torch_bind.cpp:47-49), but it
// does not depend on libtorch: it takes raw device pointers, sizes and a stream handle.  The
// Python package (custom_flash_attn/__init__.py) does the tensor checks and allocation that
// torch_bind.cpp:13-31 does in C++.  The GIL is released around the launch, and a non-zero
// C-ABI status becomes a Python RuntimeError (the reference drops launcher errors,
// torch_bind.cpp:34-39).
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <array>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "tfgfa.h"
#include "tfgfa_gpt2.h"
#include "tfgfa_plan.h"

namespace py = pybind11;

namespace {

void fwd(std::uintptr_t q, std::uintptr_t k, std::uintptr_t v, std::uintptr_t o, std::uintptr_t lse,
         int B, int H, int N, int D, float softmax_scale, bool causal, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgfa_fwd_bf16(reinterpret_cast<const void*>(q), reinterpret_cast<const void*>(k),
                        reinterpret_cast<const void*>(v), reinterpret_cast<void*>(o),
                        reinterpret_cast<float*>(lse), B, H, N, D, softmax_scale, causal ? 1 : 0,
                        reinterpret_cast<void*>(stream));
  }
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_fwd_bf16 failed (status ") + std::to_string(st) +
                             "): " + tfgfa_strerror(st));
  }
}

using Strides4 = std::array<std::int64_t, 4>;

void fwd_strided(std::uintptr_t q, const Strides4& qs, std::uintptr_t k, const Strides4& ks,
                 std::uintptr_t v, const Strides4& vs, std::uintptr_t o, const Strides4& os,
                 std::uintptr_t lse, int B, int H, int N, int D, float softmax_scale, bool causal,
                 std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgfa_fwd_bf16_strided(
        reinterpret_cast<const void*>(q), qs.data(), reinterpret_cast<const void*>(k), ks.data(),
        reinterpret_cast<const void*>(v), vs.data(), reinterpret_cast<void*>(o), os.data(),
        reinterpret_cast<float*>(lse), B, H, N, D, softmax_scale, causal ? 1 : 0,
        reinterpret_cast<void*>(stream));
  }
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_fwd_bf16_strided failed (status ") +
                             std::to_string(st) + "): " + tfgfa_strerror(st));
  }
}

void fwd_general(std::uintptr_t q, const Strides4& qs, std::uintptr_t k, const Strides4& ks,
                 std::uintptr_t v, const Strides4& vs, std::uintptr_t o, const Strides4& os,
                 std::uintptr_t lse, int B, int H, int N_q, int N_k, int D, int dtype,
                 float softmax_scale, bool causal, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgfa_fwd(reinterpret_cast<const void*>(q), qs.data(), reinterpret_cast<const void*>(k),
                   ks.data(), reinterpret_cast<const void*>(v), vs.data(),
                   reinterpret_cast<void*>(o), os.data(), reinterpret_cast<float*>(lse), B, H, N_q,
                   N_k, D, dtype, softmax_scale, causal ? 1 : 0, reinterpret_cast<void*>(stream));
  }
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_fwd failed (status ") + std::to_string(st) +
                             "): " + tfgfa_strerror(st));
  }
}

using Strides3 = std::array<std::int64_t, 3>;

void decode(std::uintptr_t q, const Strides3& qs, std::uintptr_t kc, const Strides4& ks,
            std::uintptr_t vc, const Strides4& vs, std::uintptr_t kn, const Strides3& kns,
            std::uintptr_t vn, const Strides3& vns, std::uintptr_t seqlens, std::uintptr_t o,
            const Strides3& os, std::uintptr_t lse, int B, int H, int N_max, int D,
            float softmax_scale, std::uintptr_t workspace, std::size_t workspace_bytes,
            std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgfa_decode_bf16(
        reinterpret_cast<const void*>(q), qs.data(), reinterpret_cast<void*>(kc), ks.data(),
        reinterpret_cast<void*>(vc), vs.data(), reinterpret_cast<const void*>(kn), kns.data(),
        reinterpret_cast<const void*>(vn), vns.data(), reinterpret_cast<const int*>(seqlens),
        reinterpret_cast<void*>(o), os.data(), reinterpret_cast<float*>(lse), B, H, N_max, D,
        softmax_scale, reinterpret_cast<void*>(workspace), workspace_bytes,
        reinterpret_cast<void*>(stream));
  }
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_decode_bf16 failed (status ") +
                             std::to_string(st) + "): " + tfgfa_strerror(st));
  }
}

void decode_general(std::uintptr_t q, const Strides3& qs, std::uintptr_t kc, const Strides4& ks,
                    std::uintptr_t vc, const Strides4& vs, std::uintptr_t kn, const Strides3& kns,
                    std::uintptr_t vn, const Strides3& vns, std::uintptr_t seqlens,
                    std::uintptr_t o, const Strides3& os, std::uintptr_t lse, int B, int H,
                    int N_max, int D, int dtype, float softmax_scale, std::uintptr_t workspace,
                    std::size_t workspace_bytes, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgfa_decode(
        reinterpret_cast<const void*>(q), qs.data(), reinterpret_cast<void*>(kc), ks.data(),
        reinterpret_cast<void*>(vc), vs.data(), reinterpret_cast<const void*>(kn), kns.data(),
        reinterpret_cast<const void*>(vn), vns.data(), reinterpret_cast<const int*>(seqlens),
        reinterpret_cast<void*>(o), os.data(), reinterpret_cast<float*>(lse), B, H, N_max, D,
        dtype, softmax_scale, reinterpret_cast<void*>(workspace), workspace_bytes,
        reinterpret_cast<void*>(stream));
  }
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_decode failed (status ") + std::to_string(st) +
                             "): " + tfgfa_strerror(st));
  }
}

void check(int st, const char* what) {
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(st) +
                             "): " + tfgfa_strerror(st));
  }
}

void gpt2_layernorm(std::uintptr_t x, std::uintptr_t delta, std::uintptr_t sum,
                    std::uintptr_t scale, std::uintptr_t shift, std::uintptr_t y, int y_kind,
                    std::int64_t rows, int d, float eps, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgpt2_layernorm(reinterpret_cast<const float*>(x), reinterpret_cast<const void*>(delta),
                          reinterpret_cast<float*>(sum), reinterpret_cast<const float*>(scale),
                          reinterpret_cast<const float*>(shift), reinterpret_cast<void*>(y),
                          y_kind, rows, d, eps, reinterpret_cast<void*>(stream));
  }
  check(st, "tfgpt2_layernorm");
}

void gpt2_gelu(std::uintptr_t x, std::uintptr_t y, std::int64_t n, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgpt2_gelu(reinterpret_cast<const float*>(x), reinterpret_cast<float*>(y), n,
                     reinterpret_cast<void*>(stream));
  }
  check(st, "tfgpt2_gelu");
}

// casts: (source, destination, count) of each array.
void gpt2_cast_bf16(
    const std::vector<std::tuple<std::uintptr_t, std::uintptr_t, std::int64_t>>& casts,
    std::uintptr_t stream) {
  if (casts.size() > TFGPT2_MAX_CASTS) check(TFGFA_ERR_BAD_SHAPE, "tfgpt2_cast_bf16");
  const float* src[TFGPT2_MAX_CASTS];
  void* dst[TFGPT2_MAX_CASTS];
  std::int64_t n[TFGPT2_MAX_CASTS];
  for (std::size_t i = 0; i < casts.size(); ++i) {
    src[i] = reinterpret_cast<const float*>(std::get<0>(casts[i]));
    dst[i] = reinterpret_cast<void*>(std::get<1>(casts[i]));
    n[i] = std::get<2>(casts[i]);
  }
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgpt2_cast_bf16((int)casts.size(), src, dst, n, reinterpret_cast<void*>(stream));
  }
  check(st, "tfgpt2_cast_bf16");
}

// parts: (weight, bias or 0, output) of each weight matrix.
void gpt2_linear_rows(
    std::uintptr_t x, bool x_bf16, std::uintptr_t ln_scale, std::uintptr_t ln_shift, float eps,
    const std::vector<std::tuple<std::uintptr_t, std::uintptr_t, std::uintptr_t>>& parts,
    bool gelu, std::uintptr_t residual, bool y_bf16, int M, int N, int K, std::uintptr_t stream) {
  constexpr std::size_t kMax = 3;
  if (parts.size() > kMax) check(TFGFA_ERR_BAD_SHAPE, "tfgpt2_linear_rows");
  const float* w[kMax] = {};
  const float* bias[kMax] = {};
  void* y[kMax] = {};
  for (std::size_t i = 0; i < parts.size(); ++i) {
    w[i] = reinterpret_cast<const float*>(std::get<0>(parts[i]));
    bias[i] = reinterpret_cast<const float*>(std::get<1>(parts[i]));
    y[i] = reinterpret_cast<void*>(std::get<2>(parts[i]));
  }
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgpt2_linear_rows(reinterpret_cast<const void*>(x), x_bf16 ? 1 : 0,
                            reinterpret_cast<const float*>(ln_scale),
                            reinterpret_cast<const float*>(ln_shift), eps, (int)parts.size(), w,
                            bias, gelu ? 1 : 0, reinterpret_cast<const float*>(residual), y,
                            y_bf16 ? 1 : 0, M, N, K, reinterpret_cast<void*>(stream));
  }
  check(st, "tfgpt2_linear_rows");
}

void gpt2_linear_planes(std::uintptr_t x, std::uintptr_t w, std::uintptr_t bias, bool gelu_planes,
                        std::uintptr_t residual, std::uintptr_t y, std::uintptr_t part, int splits,
                        int M, int N, int K, std::uintptr_t stream) {
  int st;
  {
    py::gil_scoped_release nogil;
    st = tfgpt2_linear_planes(reinterpret_cast<const void*>(x), reinterpret_cast<const float*>(w),
                              reinterpret_cast<const float*>(bias), gelu_planes ? 1 : 0,
                              reinterpret_cast<const float*>(residual), reinterpret_cast<void*>(y),
                              reinterpret_cast<float*>(part), splits, M, N, K,
                              reinterpret_cast<void*>(stream));
  }
  check(st, "tfgpt2_linear_planes");
}

py::dict device_info() {
  int cu = 0, mhz = 0;
  char arch[128] = {0};
  const int st = tfgfa_device_info(&cu, &mhz, arch, sizeof(arch));
  if (st != TFGFA_OK) {
    throw std::runtime_error(std::string("tfgfa_device_info failed: ") + tfgfa_strerror(st));
  }
  py::dict d;
  d["cu_count"] = cu;
  d["sclk_mhz"] = mhz;
  d["arch"] = std::string(arch);
  return d;
}

}  // namespace

PYBIND11_MODULE(_C, m) {
  m.doc() = "MI355X causal FlashAttention forward (C-ABI binding)";
  m.def("fwd", &fwd, "Launch the bf16 attention forward on raw device pointers", py::arg("q"),
        py::arg("k"), py::arg("v"), py::arg("o"), py::arg("lse"), py::arg("B"), py::arg("H"),
        py::arg("N"), py::arg("D"), py::arg("softmax_scale"), py::arg("causal"),
        py::arg("stream"));
  m.def("fwd_strided", &fwd_strided,
        "Launch the bf16 attention forward on strided operands (element strides b, h, n, d)",
        py::arg("q"), py::arg("q_strides"), py::arg("k"), py::arg("k_strides"), py::arg("v"),
        py::arg("v_strides"), py::arg("o"), py::arg("o_strides"), py::arg("lse"), py::arg("B"),
        py::arg("H"), py::arg("N"), py::arg("D"), py::arg("softmax_scale"), py::arg("causal"),
        py::arg("stream"));
  m.def("fwd_general", &fwd_general,
        "Attention forward, any strides, bf16/fp16, head dim a multiple of 8 up to 128, N_q != N_k",
        py::arg("q"), py::arg("q_strides"), py::arg("k"), py::arg("k_strides"), py::arg("v"),
        py::arg("v_strides"), py::arg("o"), py::arg("o_strides"), py::arg("lse"), py::arg("B"),
        py::arg("H"), py::arg("N_q"), py::arg("N_k"), py::arg("D"), py::arg("dtype"),
        py::arg("softmax_scale"), py::arg("causal"), py::arg("stream"));
  m.attr("DTYPE_BF16") = TFGFA_DTYPE_BF16;
  m.attr("DTYPE_F16") = TFGFA_DTYPE_F16;
  m.def("decode", &decode,
        "One decode step over a KV cache on raw device pointers (element strides)",
        py::arg("q"), py::arg("q_strides"), py::arg("k_cache"), py::arg("k_strides"),
        py::arg("v_cache"), py::arg("v_strides"), py::arg("k_new"), py::arg("k_new_strides"),
        py::arg("v_new"), py::arg("v_new_strides"), py::arg("cache_seqlens"), py::arg("o"),
        py::arg("o_strides"), py::arg("lse"), py::arg("B"), py::arg("H"), py::arg("N_max"),
        py::arg("D"), py::arg("softmax_scale"), py::arg("workspace"),
        py::arg("workspace_bytes"), py::arg("stream"));
  m.def("decode_general", &decode_general,
        "One decode step, bf16/fp16, head dim a multiple of 8 up to 128 (element strides)",
        py::arg("q"), py::arg("q_strides"), py::arg("k_cache"), py::arg("k_strides"),
        py::arg("v_cache"), py::arg("v_strides"), py::arg("k_new"), py::arg("k_new_strides"),
        py::arg("v_new"), py::arg("v_new_strides"), py::arg("cache_seqlens"), py::arg("o"),
        py::arg("o_strides"), py::arg("lse"), py::arg("B"), py::arg("H"), py::arg("N_max"),
        py::arg("D"), py::arg("dtype"), py::arg("softmax_scale"), py::arg("workspace"),
        py::arg("workspace_bytes"), py::arg("stream"));
  m.def("stream_read", [](std::uintptr_t p, std::size_t bytes, std::uintptr_t sink, std::uintptr_t stream) {
    const int st = tfgfa_stream_read(reinterpret_cast<const void*>(p), bytes,
                                     reinterpret_cast<void*>(sink), reinterpret_cast<void*>(stream));
    if (st != TFGFA_OK)
      throw std::runtime_error(std::string("tfgfa_stream_read failed: ") + tfgfa_strerror(st));
  }, "A plain streaming read of `bytes` device bytes (a measurement floor)", py::arg("p"),
        py::arg("bytes"), py::arg("sink"), py::arg("stream"));
  m.def("decode_workspace_bytes", [](int B, int H, int N_max) {
    return tfgfa_decode_workspace_bytes(B, H, N_max);
  });
  m.def("decode_workspace_size", [](int B, int H, int N_max, int D) {
    return tfgfa_decode_workspace_size(B, H, N_max, D);
  });
  m.def("gpt2_layernorm", &gpt2_layernorm, "LayerNorm, with an optional residual add before it",
        py::arg("x"), py::arg("delta"), py::arg("sum"), py::arg("scale"), py::arg("shift"),
        py::arg("y"), py::arg("y_kind"), py::arg("rows"), py::arg("d"), py::arg("eps"),
        py::arg("stream"));
  m.def("gpt2_gelu", &gpt2_gelu, "GELU (tanh form), elementwise", py::arg("x"), py::arg("y"),
        py::arg("n"), py::arg("stream"));
  m.def("gpt2_cast_bf16", &gpt2_cast_bf16, "float32 -> bf16 copies in one launch",
        py::arg("casts"), py::arg("stream"));
  m.def("gpt2_linear_rows", &gpt2_linear_rows,
        "A linear layer on few rows, with LayerNorm, bias, GELU and residual", py::arg("x"),
        py::arg("x_bf16"), py::arg("ln_scale"), py::arg("ln_shift"), py::arg("eps"),
        py::arg("parts"), py::arg("gelu"), py::arg("residual"), py::arg("y_bf16"), py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("stream"));
  m.def("gpt2_linear_planes", &gpt2_linear_planes,
        "A float32 linear layer on the bf16 matrix units, from three-way splits", py::arg("x"),
        py::arg("w"), py::arg("bias"), py::arg("gelu_planes"), py::arg("residual"), py::arg("y"),
        py::arg("part"), py::arg("splits"), py::arg("M"), py::arg("N"), py::arg("K"),
        py::arg("stream"));
  m.def("gpt2_linear_planes_splits", [](int M, int N, int K) {
    int cu = 0;
    check(tfgfa_device_info(&cu, nullptr, nullptr, 0), "tfgfa_device_info");
    return tfgpt2_linear_planes_splits(M, N, K, cu);
  });
  m.def("fwd_plan",
        [](long long heads, int cu_count, int Nq, int Nk, int D, bool causal) {
          static const char* const names[] = {"kWhole", "kHalves", "kGroups2", "kPairs", "kGroups4"};
          return names[(int)tfgfa::choose_plan(heads, cu_count, Nq, Nk, D, causal)];
        },
        "The kernel that runs a forward of these sizes", py::arg("heads"), py::arg("cu_count"),
        py::arg("Nq"), py::arg("Nk"), py::arg("D"), py::arg("causal"));
  m.attr("GPT2_F32") = TFGPT2_F32;
  m.attr("GPT2_BF16") = TFGPT2_BF16;
  m.attr("GPT2_PLANES") = TFGPT2_PLANES;
  m.attr("GPT2_MAX_NORM_DIM") = TFGPT2_MAX_NORM_DIM;
  m.attr("GPT2_MAX_ROWS") = TFGPT2_MAX_ROWS;
  m.attr("GPT2_MAX_NORM_ROWS") = TFGPT2_MAX_NORM_ROWS;
  m.attr("GPT2_MAX_VALUES") = TFGPT2_MAX_VALUES;
  m.attr("GPT2_MAX_OUTPUTS") = TFGPT2_MAX_OUTPUTS;
  m.def("device_info", &device_info, "CU count, shader clock (MHz) and arch of the current device");
  m.def("strerror", [](int st) { return std::string(tfgfa_strerror(st)); });
  m.def("abi_version", []() { return tfgfa_abi_version(); });
}
