// What the operator layer's translation units share: the conversion of tensors to the C ABI's
// pointers, error translation, the launch context and the library's side streams.
#pragma once
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>

#include <hip/hip_runtime_api.h>

#include <mutex>
#include <optional>

#include "../../include/mi355_moe.h"

namespace mi355_torch {

// A second stream per device (default priority, not synchronising with the null stream) and the
// events of a fork / join around it.  The backward's weight gradients do not depend on its
// input gradient: launched there, their workgroups fill the CUs that the last, partly filled
// round of the other product's tiles leaves idle, and the bandwidth-bound row sum runs beside
// matrix work instead of between two launches.  Created on first use; never under stream
// capture (a caller who captures first runs a step uncaptured, as for every lazily built state);
// nullptr means "stay on one stream".
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t entry = nullptr;                // a fork in front of a call's first launch
  hipEvent_t fork = nullptr, join = nullptr;  // one behind a launch of the call, and a join
  std::mutex order;  // an event is recorded and waited for as one step: host threads share the three

  // `to` waits for everything enqueued on `from` so far
  bool chain(hipEvent_t event, hipStream_t from, hipStream_t to) {
    std::lock_guard<std::mutex> lock(order);
    return hipEventRecord(event, from) == hipSuccess && hipStreamWaitEvent(to, event, 0) == hipSuccess;
  }
};

// which: 0 the weight gradients of the fused backward, 1 the shared expert (handed to the Python
// layer as a raw pointer, see aux_stream below)
inline SideStream* side_stream(int device, hipStream_t current, int which = 0) {
  static std::mutex mu;
  static SideStream streams[2][64];
  static bool attempted[2][64];
  if (device < 0 || device >= 64 || which < 0 || which > 1) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  SideStream& s = streams[which][device];
  bool* tried = attempted[which];
  if (!tried[device]) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(current, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone)
      return nullptr;  // not now: try again on a later, uncaptured call
    tried[device] = true;
    // Without the system-scope fences of an ordinary event where what stands before it on its stream is a kernel of the same call and what waits for it one of the
    // same device: the kernels' own device-scope fences order the two, that kernel began behind whatever a copy or another device had written for its stream (its own start
    // drops stale lines from every L2), and whatever later hands results to the host or another device has fences of its own.  In front of a call's first launch no kernel
    // has done that, a copy of the tokens may be the last thing on the stream: an ordinary event.  A step or forward, us, all with / all without: 3000 tokens of 64
    // experts of 1024 x 512 364 / 359, 300 of 128 of 2048 x 768 701 / 695; one rank's share of 7168 x 2048 with its shared expert, forward of 16 and 128 tokens 182 / 178, 348 / 345,
    // a step of 500 1492 / 1482.
    constexpr unsigned kEvent = hipEventDisableTiming | hipEventDisableSystemFence;
    if (hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&s.entry, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s.fork, kEvent) != hipSuccess ||
        hipEventCreateWithFlags(&s.join, kEvent) != hipSuccess) {
      (void)hipGetLastError();
      s.stream = nullptr;
    }
  }
  return s.stream ? &s : nullptr;
}

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// A registered operator, to be called through the dispatcher.
template <class Sig>
auto typed_op(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}

// An operator has written an argument through its pointer: a backward that saved its earlier value is to raise.  (An inference tensor has no
// version, and no backward saves one.)
inline void wrote(const OptTensor& t) {
  if (t.has_value() && t->defined() && !t->is_inference()) t->unsafeGetTensorImpl()->bump_version();
}

inline int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return MI355_F32;
  if (t.scalar_type() == at::kBFloat16) return MI355_BF16;
  if (t.scalar_type() == at::kDouble) return MI355_F64;
  TORCH_CHECK_TYPE(false, "MI355 MoE kernels support float32, bfloat16 and float64, got ", t.scalar_type());
}

inline void* ptr(const Tensor& t) { return (t.defined() && t.numel() > 0) ? t.data_ptr() : nullptr; }
inline void* ptr(const OptTensor& t) { return t.has_value() ? ptr(*t) : nullptr; }
inline const int32_t* iptr(const Tensor& t) { return static_cast<const int32_t*>(ptr(t)); }
inline const int32_t* iptr(const OptTensor& t) { return static_cast<const int32_t*>(ptr(t)); }
inline const float* fptr(const Tensor& t) { return static_cast<const float*>(ptr(t)); }
inline const float* fptr(const OptTensor& t) { return static_cast<const float*>(ptr(t)); }

// Device guard + the current stream of that device, for the duration of one operator.
struct Launch {
  c10::DeviceGuard guard;
  void* stream;
  explicit Launch(const Tensor& t)
      : guard(t.device()),
        stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()) {
    TORCH_CHECK(t.is_cuda(), "MI355 MoE kernels need tensors on a HIP device (got ", t.device(),
                "); there is no CPU implementation");
  }
};

inline void check(int rc, const char* what) {
  if (rc == MI355_OK) return;
  const char* msg = mi355_moe_last_error();
  TORCH_CHECK_VALUE(rc != MI355_EINVAL, what, " failed (", rc, "): ", msg);
  TORCH_CHECK(false, what, " failed (", rc, "): ", msg);
}

// The tensor as the kernels read it: contiguous, and starting on a 16-byte boundary as an allocation of its own
// does.  A view into a flat buffer need not, and the kernels fetch 16 bytes at a time: such a one is copied.
inline Tensor dense(const Tensor& t) {
  Tensor c = t.contiguous();
  if (!c.is_cuda()) return c;  // (shapes only: no memory to look at)
  return reinterpret_cast<uintptr_t>(ptr(c)) % 16 == 0 ? c : c.clone();
}
inline Tensor dense(const OptTensor& t) { return t.has_value() && t->defined() ? dense(*t) : Tensor(); }
inline Tensor cf(const Tensor& t) { return dense(t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)); }
inline Tensor bytes(int64_t n, const Tensor& like) {
  return at::empty({n > 0 ? n : 1}, like.options().dtype(at::kByte));
}
inline Tensor none_like(const Tensor& like) { return at::empty({0}, like.options()); }

}  // namespace mi355_torch
