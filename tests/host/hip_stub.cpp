// A stand-in for the HIP runtime, so that the library's host code (its sources
// compiled for the host only) runs on a CPU.  It keeps what the host code can get
// wrong: which stream each launch, event and wait goes to, stream validity, capture
// states, memory that runs out, and the error that hipGetLastError returns until
// it is asked.  Kernels do nothing.
//
// The log has one line per call, streams and events by number:
//   launch <kernel> <stream> [<workspace pointer>]   record <event> <stream>
//   wait <stream> <event>   sync <stream>   sync_event <event>   sync_device
//   malloc <bytes> <pointer>   free <pointer>
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include "../../gemma4.kt_amd/csrc/g4_internal.hpp"

namespace {

hipError_t last = hipSuccess;
size_t free_bytes = ~size_t(0);
std::string text;
std::map<const void *, std::string> kernels;
std::map<void *, size_t> blocks;
hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;

struct Stream {
  int id;
  bool live, capturing;
};
Stream streams[64];
int n_streams = 0;
int n_events = 0;

hipError_t fail(hipError_t e) { return last = e; }

Stream *at(hipStream_t s) {
  Stream *p = (Stream *)s;
  return p && p->live ? p : nullptr;
}

// a call that a capture in the process forbids
bool forbidden() {
  if (mode == hipStreamCaptureModeRelaxed) return false;
  for (int i = 0; i < n_streams; ++i)
    if (streams[i].live && streams[i].capturing) return true;
  return false;
}

void log(const char *fmt, ...) {
  char b[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(b, sizeof(b), fmt, ap);
  va_end(ap);
  text += b;
  text += '\n';
}

struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} config;

}  // namespace

extern "C" {

// ------------------------------------------------------ the test's controls ---
const char *stub_log() { return text.c_str(); }
void stub_clear() { text.clear(); }
void stub_free_bytes(size_t n) { free_bytes = n; }
void stub_capture(void *s, int on) { ((Stream *)s)->capturing = on; }
int stub_stream_id(void *s) { return ((Stream *)s)->id; }
int stub_last_error() { return last; }

// ------------------------------------------------------------------ runtime ---
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "error of the stand-in runtime"; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeWarpSize ? 64 : 1024;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 2, hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { return *p = const_cast<void *>(s), hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) {
  if (forbidden()) return fail(hipErrorStreamCaptureUnsupported);
  if (n > free_bytes) return fail(hipErrorOutOfMemory);
  *p = malloc(n ? n : 1);
  if (free_bytes != ~size_t(0)) free_bytes -= n;
  blocks[*p] = n;
  log("malloc %zu %p", n, *p);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  if (forbidden()) return fail(hipErrorStreamCaptureUnsupported);
  log("free %p", p);
  if (free_bytes != ~size_t(0)) free_bytes += blocks[p];
  blocks.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = malloc(n ? n : 1), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }

// a destroyed stream's handle is given out again, as allocators do
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  static int ids = 0;
  int i = 0;
  while (i < n_streams && streams[i].live) ++i;
  if (i == n_streams) ++n_streams;
  streams[i] = Stream{ids++, true, false};
  return *s = (hipStream_t)&streams[i], hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorInvalidHandle);
  p->live = false;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorContextIsDestroyed);
  *st = p->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
  const hipStreamCaptureMode old = mode;
  mode = *m;
  *m = old;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorContextIsDestroyed);
  if (p->capturing) return fail(hipErrorStreamCaptureUnsupported);
  log("sync %d", p->id);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  if (forbidden()) return fail(hipErrorStreamCaptureUnsupported);
  log("sync_device");
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)(intptr_t)++n_events, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) {
  log("sync_event %d", (int)(intptr_t)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorContextIsDestroyed);
  log("record %d %d", (int)(intptr_t)e, p->id);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorContextIsDestroyed);
  log("wait %d %d", p->id, (int)(intptr_t)e);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s) {
  Stream *p = at(s);
  if (!p) return fail(hipErrorContextIsDestroyed);
  const std::string &k = kernels[f];
  // the workspace a kernel writes (k_split: its seventh argument; the 16-token tiles:
  // the partial sums) or reads (k_tok_reduce: its first)
  void *ws = nullptr;
  if (k.find("k_mat") != std::string::npos || k.find("k_tok_q4k") != std::string::npos)
    ws = ((const g4::TokArgs *)args[0])->part;
  if (k.find("k_split") != std::string::npos) memcpy(&ws, args[6], sizeof(ws));
  if (k.find("k_tok_reduce") != std::string::npos) memcpy(&ws, args[0], sizeof(ws));
  if (ws)
    log("launch %s %d %p", k.c_str(), p->id, ws);
  else
    log("launch %s %d", k.c_str(), p->id);
  return hipSuccess;
}

// ------------------------------------- what the compiler's launch stubs call ---
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) {
  config = Config{g, b, n, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
  *g = config.grid, *b = config.block, *n = config.shared, *s = config.stream;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}

}  // extern "C"
