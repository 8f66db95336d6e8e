// Shared host glue of the torch-facing modules: tensor checks, current stream,
// device guard, workspace from the caching allocator, status -> exception.
#pragma once
#include <torch/extension.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <map>
#include <memory>
#include <mutex>
#include <optional>
#include <utility>

#include "teletron_op.h"

namespace tt_glue {

inline void check_act(const torch::Tensor& t, const char* name, int64_t rows, int64_t cols) {
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16, got ", t.scalar_type());
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.numel() == rows * cols, name, " has ", t.numel(), " elements, expected rows*cols = ", rows * cols);
}
inline void check_param(const torch::Tensor& t, const char* name, int64_t cols, const torch::Tensor& ref) {
  TORCH_CHECK(t.is_cuda() && t.device() == ref.device(), name, " must be on the input's device");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16, got ", t.scalar_type());
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.numel() == cols, name, " has ", t.numel(), " elements, expected cols = ", cols);
}
inline void check_rowstat(const torch::Tensor& t, const char* name, int64_t rows, const torch::Tensor& ref) {
  TORCH_CHECK(t.is_cuda() && t.device() == ref.device(), name, " must be on the input's device");
  TORCH_CHECK(t.scalar_type() == at::kFloat, name, " must be float32, got ", t.scalar_type());
  TORCH_CHECK(t.is_contiguous() && t.numel() == rows, name, " must be contiguous with rows = ", rows, " elements");
}
inline void check_shape(int64_t rows, int64_t cols) {
  TORCH_CHECK(rows >= 0 && cols > 0, "rows must be >= 0 and cols > 0");
}
inline void* current_stream(const torch::Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}
// Backward workspace (per-workgroup partial sums): one tensor per (device, stream), grown on demand
// and reused from call to call, so a backward call does not go to the allocator (the reference
// allocates its fp32 [32, C] scratch on every call, teletron_op/fused_rmsnorm/weight_backward.cu:229).
struct Workspace {
  std::mutex mu;          // held from the look at `memory` until everything that uses it is queued
  torch::Tensor memory;
};
struct Workspaces {
  std::mutex mu;
  std::map<std::pair<int, hipStream_t>, std::shared_ptr<Workspace>> kept;
};
// Never destroyed: the HIP runtime may be gone by the time static destructors run.
inline Workspaces& workspaces() {
  static auto* w = new Workspaces();
  return *w;
}
constexpr int64_t kKeepBytes = 64 << 20;   // more than this is not kept between calls

// Calls launch(memory, bytes), which queues a backward call's two kernels on the current stream of ref's
// device, and returns its result; `bytes` is what was asked for, however large the kept memory is.  Launches on one stream run in order, so consecutive calls never overlap in
// the workspace; the lock keeps two host threads from queueing kernel, kernel, reduction, reduction.  The GIL
// is released first (the launch may wait for room in the queue, and the lock for another Python thread).
// A stream under graph capture gets memory of its own from the capture's pool: the graph keeps the pointer.
template <typename F>
auto with_workspace(size_t bytes, const torch::Tensor& ref, F launch) {
  std::optional<pybind11::gil_scoped_release> unlocked;
  if (PyGILState_Check()) unlocked.emplace();   // a call through torch.ops comes without it
  const auto opts = at::TensorOptions().dtype(at::kByte).device(ref.device());
  const int64_t need = static_cast<int64_t>(bytes < 16 ? 16 : bytes);
  const int device = static_cast<int>(ref.device().index());
  hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) (void)hipGetLastError();
  if (capturing != hipStreamCaptureStatusNone || need > kKeepBytes) {
    const torch::Tensor own = at::empty({need}, opts);
    return launch(own.data_ptr(), static_cast<size_t>(need));
  }
  std::shared_ptr<Workspace> ws;
  {
    std::lock_guard<std::mutex> lock(workspaces().mu);
    auto& entry = workspaces().kept[{device, stream}];
    if (!entry) entry = std::make_shared<Workspace>();
    ws = entry;
  }
  std::lock_guard<std::mutex> lock(ws->mu);
  if (!ws->memory.defined() || ws->memory.numel() < need) ws->memory = at::empty({need}, opts);
  return launch(ws->memory.data_ptr(), static_cast<size_t>(need));
}
inline void check_status(int rc, const char* what) {
  TORCH_CHECK(rc == TT_OK, what, " failed: ", tt_error_string(rc),
              rc == TT_ERR_HIP ? " (hipError_t " + std::to_string(tt_last_hip_error()) + ")" : std::string());
}

}  // namespace tt_glue
