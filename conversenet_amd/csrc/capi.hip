// Library-wide C-ABI entry points: version, error string, cache no-op, calibration copy kernel.
#include <algorithm>

#include "cvn_common.h"

namespace cvn {
std::string& last_error_slot() {
  static thread_local std::string s;
  return s;
}

// 16-byte grid-stride copy with a scalar tail; used to calibrate HBM byte counters and to measure
// the attainable HBM bandwidth.  Stores are non-temporal (streaming), as in the library's kernels
// whose outputs are not read back by the same launch.
typedef float copy_f32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) k_copy(const copy_f32x4* __restrict__ src, copy_f32x4* __restrict__ dst,
                                              int64_t n4, const float* __restrict__ src1,
                                              float* __restrict__ dst1, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride)
    __builtin_nontemporal_store(src[i], &dst[i]);
  for (int64_t i = 4 * n4 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst1[i] = src1[i];
}
}  // namespace cvn

using namespace cvn;

extern "C" const char* cvn_version(void) { return "conversenet_amd 0.1 (gfx950)"; }

extern "C" const char* cvn_last_error(void) { return last_error_slot().c_str(); }

extern "C" int cvn_clear_cache(void) { return CVN_OK; }

namespace {
int event_rc(hipError_t e, const char* what) {
  return e == hipSuccess ? CVN_OK : fail(CVN_ERR_HIP, "event %s: %s", what, hipGetErrorString(e));
}
// Whether a stream records a graph (the null stream cannot).  HIP refuses waits for events of such a stream, and
// the attempt spoils the recording.
hipError_t recording(hipStream_t stream, bool* yes) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  const hipError_t e = stream ? hipStreamIsCapturing(stream, &status) : hipSuccess;
  *yes = status != hipStreamCaptureStatusNone;
  return e;
}
}  // namespace

extern "C" int cvn_event_create(void** event) {
  if (!event) return fail(CVN_ERR_ARG, "null event");
  return event_rc(hipEventCreateWithFlags((hipEvent_t*)event, hipEventDisableTiming | hipEventDisableSystemFence),
                  "create");
}

extern "C" int cvn_event_record(void* event, cvn_stream_t stream) {
  if (!event) return fail(CVN_ERR_ARG, "null event");
  return event_rc(hipEventRecord((hipEvent_t)event, (hipStream_t)stream), "record");
}

extern "C" int cvn_event_join(void* event, cvn_stream_t recorded_on, cvn_stream_t stream) {
  if (!event) return fail(CVN_ERR_ARG, "null event");
  bool busy = false;
  const hipError_t e = recording((hipStream_t)recorded_on, &busy);
  if (e != hipSuccess) return event_rc(e, "join");
  if (busy) return fail(CVN_ERR_UNSUPPORTED, "event join: the event's stream records a graph");
  return event_rc(hipStreamWaitEvent((hipStream_t)stream, (hipEvent_t)event, 0), "join");
}

extern "C" int cvn_event_wait(void* event, cvn_stream_t stream) {
  if (!event) return fail(CVN_ERR_ARG, "null event");
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
  if (e == hipSuccess) {
    bool busy = false;
    e = recording((hipStream_t)stream, &busy);
    if (e == hipSuccess && !busy) e = hipEventSynchronize((hipEvent_t)event);
    const hipError_t back = hipThreadExchangeStreamCaptureMode(&mode);
    if (e == hipSuccess) e = back;
  }
  return event_rc(e, "wait");
}

extern "C" int cvn_copy_f32(const float* src, float* dst, int64_t n, cvn_stream_t stream) {
  if (n < 0 || (n > 0 && (!src || !dst))) return fail(CVN_ERR_ARG, "bad copy arguments");
  if (n == 0) return CVN_OK;
  if (((uintptr_t)src | (uintptr_t)dst) & 15) return fail(CVN_ERR_ARG, "copy needs 16-byte aligned buffers");
  const int64_t n4 = n / 4;
  const int64_t blocks = std::min<int64_t>((n4 + 255) / 256 + 1, 256 * 64);
  hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const copy_f32x4*)src, (copy_f32x4*)dst, n4, src, dst, n);
  return check_launch("copy");
}
