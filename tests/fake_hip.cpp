// The HIP calls of csrc/host_copy.hip for a test on the CPU: transfers happen at once, and what each stream knows to have ended
// on the caller's stream is kept (an event carries it from the stream it is recorded on to those that wait for it).
#include <algorithm>
#include <cstdarg>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "runtime.h"

namespace {
std::map<hipStream_t, int> known;   // pieces of work of the caller's stream
std::map<hipEvent_t, int> carried;
hipStream_t caller = nullptr;
int early = 0, transfers = 0;
int know(hipStream_t s) { return known[s]; }
}  // namespace

namespace mobula_hip {
CallState& call_state() { static CallState state; return state; }
void set_error(const char* fmt, ...) { call_state().error = fmt; }
}  // namespace mobula_hip

extern "C" {
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new int); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(new int); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { carried[e] = know(s); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { known[s] = std::max(know(s), carried[e]); return hipSuccess; }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t s) {
  ++transfers;
  if (know(s) < know(caller)) ++early;
  std::memcpy(to, from, n);
  return hipSuccess;
}

// Three calls with arrays of `bytes` bytes, there and back, each behind work on the caller's stream.  -1: a byte did not
// arrive; else the transfers that did not wait for that work, times 1000, and the transfers.
int run_copies(size_t bytes) {
  std::vector<char> in(bytes), out(bytes);
  for (size_t i = 0; i < bytes; ++i) in[i] = static_cast<char>(i * 31 + i / 4096);
  for (int call = 0; call < 3; ++call) {
    ++known[caller];
    std::memset(out.data(), 0, bytes);
    mobula_hip::HostStaging stage;
    stage.reserve({bytes, bytes});
    void* const a = stage.in(in.data(), bytes);
    void* const b = stage.inout(out.data(), bytes, false);
    std::memcpy(b, a, bytes);   // (the call's kernel)
    ++known[caller];
    if (!stage.flush(caller) || in != out) return -1;
  }
  return early * 1000 + transfers;
}
}
