// Whether the kernels in front of an event are done; wait: the host waits for them.  The thread asks by its own relaxed capture mode:
// an event of work outside a graph may be looked at while a graph is recorded, but by default asking for it ends the recording.
#pragma once
#include <torch/extension.h>
#include <hip/hip_runtime.h>

inline bool event_done(uintptr_t event, bool wait) {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  TORCH_CHECK(hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess, "event_done: capture mode");
  const hipError_t rc = wait ? hipEventSynchronize((hipEvent_t)event) : hipEventQuery((hipEvent_t)event);
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (rc == hipErrorNotReady) {
    (void)hipGetLastError();
    return false;
  }
  TORCH_CHECK(rc == hipSuccess, "event_done: ", hipGetErrorString(rc));
  return true;
}
