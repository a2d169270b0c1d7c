// Host path of a matmul call (CPython extension): the checks, the output
// allocation and the pmi_matmul_w4a16 call that pare_amd.kernels and
// pare_amd.linear otherwise make from Python. Calls at decode sizes take 3-15 us
// on the GPU, and the Python path issued one every 20 us (QuantizedLinear at one
// row); this one every 7.
//
// Only plain calls are taken: dense tensors of the expected types on the current
// device. For everything else, and where the library refuses, matmul() returns
// None and the caller's general path runs, with its own conversions and errors.
// Nothing is kept between calls, and no HIP header is needed: the library's entry
// points arrive as addresses, the stream as its handle.
#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>

namespace py = pybind11;

namespace {

using MatmulFn = int (*)(const void*, int, const uint8_t*, const float*, const void*, int, const int32_t*,
                         const uint16_t*, const float*, const uint8_t*, const uint8_t*, void*, int, int64_t,
                         int64_t, int64_t, int64_t, void*, size_t, void*);
using ChoiceFn = int (*)(int64_t, int64_t, int64_t, int64_t, int);
using WorkspaceFn = size_t (*)(int64_t, int64_t, int64_t, int64_t, int);
using RouteFn = int (*)(int64_t, int64_t, int64_t, int64_t, int, int, size_t);

MatmulFn g_matmul = nullptr;
ChoiceFn g_choice = nullptr;
WorkspaceFn g_workspace = nullptr;
RouteFn g_route = nullptr;

constexpr int kF16 = 0, kBf16 = 1, kU8 = 3;  // PMI_F16, PMI_BF16, PMI_U8
constexpr int kChoiceTiled = 1, kChoicePerm = 2, kChoiceGm = 4;

void bind(uintptr_t matmul, uintptr_t choice, uintptr_t workspace, uintptr_t route) {
  g_matmul = reinterpret_cast<MatmulFn>(matmul);
  g_choice = reinterpret_cast<ChoiceFn>(choice);
  g_workspace = reinterpret_cast<WorkspaceFn>(workspace);
  g_route = reinterpret_cast<RouteFn>(route);
}

bool plain(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj() &&
         !at::isTensorSubclassLike(t);
}

// A buffer the kernels read in place.
bool buffer(const at::Tensor& t, const at::Device& dev, at::ScalarType dtype, int64_t numel, size_t align) {
  return plain(t) && t.device() == dev && t.scalar_type() == dtype && t.numel() == numel && t.is_contiguous() &&
         reinterpret_cast<uintptr_t>(t.const_data_ptr()) % align == 0;
}

// [N] (one group), [N, G] or [N, G, 1].
bool per_group(const at::Tensor& t, int64_t N, int64_t G) {
  const int64_t d = t.dim();
  return d >= 1 && d <= 3 && t.size(0) == N && (d > 1 ? t.size(1) == G : G == 1) && (d < 3 || t.size(2) == 1);
}

template <typename T>
const T* ptr(const std::optional<at::Tensor>& t) {
  return t ? static_cast<const T*>(t->const_data_ptr()) : nullptr;
}

// x [.., K] @ dequant(w [N, K/2])^T (+ bias) -> [.., N]. cast: other dtypes of x
// are computed in fp16 and converted back (without it they are not taken). bf16:
// x in bf16 is computed in bf16. build_tiled: the caller could make the tiled
// copy that it has not; calls that would run on it are then left to it.
// workspace_fn(nbytes) gives the stream's workspace.
py::object matmul(const at::Tensor& x, const at::Tensor& w, const at::Tensor& scales, const at::Tensor& zeros,
                  int64_t gs, const std::optional<at::Tensor>& perm, const std::optional<at::Tensor>& perm16,
                  const std::optional<at::Tensor>& s_gm, const std::optional<at::Tensor>& z_gm,
                  const std::optional<at::Tensor>& w_tiled, bool build_tiled, bool cast, bool bf16,
                  const std::optional<at::Tensor>& bias, int64_t device, uintptr_t stream,
                  const py::function& workspace_fn) {
  if (!g_matmul || !plain(x) || !plain(w) || x.dim() < 1 || w.dim() != 2 || gs <= 0) return py::none();
  const at::Device dev = x.device();
  const int64_t N = w.size(0), K = 2 * w.size(1);
  if (dev.index() != device || x.size(-1) != K || K == 0 || N == 0 || K % gs != 0 || x.numel() == 0)
    return py::none();
  const at::ScalarType in = x.scalar_type();
  const bool native = in == at::kBFloat16 && bf16;
  if (!native && in != at::kHalf && !(cast && (in == at::kBFloat16 || in == at::kFloat))) return py::none();
  const int64_t M = x.numel() / K, G = K / gs;
  if (!buffer(w, dev, at::kByte, N * (K / 2), 16) || !buffer(scales, dev, at::kFloat, N * G, 4) ||
      !buffer(zeros, dev, at::kByte, N * G, 1) || !per_group(scales, N, G) || !per_group(zeros, N, G))
    return py::none();
  if (perm && !buffer(*perm, dev, at::kInt, K, 4)) return py::none();
  if (perm16 && (!perm || !buffer(*perm16, dev, at::kShort, K, 16))) return py::none();
  if (s_gm.has_value() != z_gm.has_value()) return py::none();
  if (s_gm && (!buffer(*s_gm, dev, at::kFloat, N * G, 4) || !buffer(*z_gm, dev, at::kByte, N * G, 4) ||
               s_gm->dim() != 2 || s_gm->size(0) != G || z_gm->dim() != 2 || z_gm->size(0) != G))
    return py::none();
  if (w_tiled && !buffer(*w_tiled, dev, at::kByte, (N + 63) / 64 * 64 * (K / 2), 16)) return py::none();
  const int act = perm ? kChoicePerm : 0;
  if (!w_tiled && build_tiled && !(native && perm)) {
    const int c = g_choice(M, N, K, gs, kChoiceTiled | act);
    if (c == 5 || c == 6) return py::none();
  }
  const size_t need = g_workspace(M, N, K, gs, perm ? 1 : 0);
  if (!w_tiled && build_tiled && native &&
      g_route(M, N, K, gs, kBf16, kChoiceTiled | act, need) != g_route(M, N, K, gs, kBf16, kChoiceGm | act, need))
    return py::none();
  at::Tensor ws;
  if (need) {
    ws = workspace_fn(need).cast<at::Tensor>();
    if (!plain(ws) || ws.device() != dev) return py::none();
  }
  // other threads run meanwhile: a launch waits where the stream's queue is full
  std::optional<py::gil_scoped_release> unlocked(std::in_place);
  at::Tensor xc = native || in == at::kHalf ? x : x.to(at::kHalf);
  xc = xc.contiguous();
  if (reinterpret_cast<uintptr_t>(xc.const_data_ptr()) % 16) xc = xc.clone();
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = N;
  at::Tensor y = at::empty(shape, at::TensorOptions().dtype(xc.scalar_type()).device(dev));

  const int code = native ? kBf16 : kF16;
  const int rc = g_matmul(xc.const_data_ptr(), code, static_cast<const uint8_t*>(w.const_data_ptr()),
                          static_cast<const float*>(scales.const_data_ptr()), zeros.const_data_ptr(), kU8,
                          ptr<int32_t>(perm), ptr<uint16_t>(perm16), ptr<float>(s_gm), ptr<uint8_t>(z_gm),
                          ptr<uint8_t>(w_tiled), y.mutable_data_ptr(), code, M, N, K, gs,
                          need ? ws.mutable_data_ptr() : nullptr, need ? (size_t)ws.numel() : 0,
                          reinterpret_cast<void*>(stream));
  if (rc == 0 && y.scalar_type() != in) y = y.to(in);
  if (rc == 0 && bias) y = y + *bias;
  unlocked.reset();
  return rc == 0 ? py::cast(y) : py::none();
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("bind", &bind);
  m.def("matmul", &matmul);
}
