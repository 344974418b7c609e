// faults.cpp -- failures on demand for the host code over its CPU stand-ins (hip_host_stub.cpp,
// resident_stub.cpp).  TEST INFRASTRUCTURE ONLY: linked with --wrap, so that the calls named below
// pass through here; a test sets the counters through ctypes.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <mutex>
#include <system_error>
#include <thread>
#include <unordered_map>

#include "../../pannde_amd/csrc/rsg_internal.h"

extern "C" {

// threads that may still be started; -1: any number
int fault_threads = -1;

#define START_THREAD _ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE
#define PASTE(a, b) a##b
#define NAME(a, b) PASTE(a, b)

void NAME(__real_, START_THREAD)(std::thread* self, void* state, void (*depend)());
void NAME(__wrap_, START_THREAD)(std::thread* self, void* state, void (*depend)()) {
  if (fault_threads == 0) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
  if (fault_threads > 0) fault_threads--;
  NAME(__real_, START_THREAD)(self, state, depend);
}

// Resident launches that decide against their steps, how many ms after its launch a decision becomes
// known (or when the host waits for the stream), whether one is not known yet, launches so far, and what the per-step kernels were launched with: the first
// channel's amplitude and the trace row's address.
int fault_refuse = 0, fault_late = 0, fault_undecided = 0;
int fault_resident = 0, fault_velocity = 0, fault_stress = 0;
// resident launches that fail, and which of the event records from now on does (1: the next)
int fault_launch = 0, fault_record = 0;
// resident launches whose tiles lose each other
int fault_lost = 0;
double fault_amp[4096], fault_stress_amp[4096];
const double* fault_trace[4096];
// device allocations so far, and the bytes from which on there is no memory for one (0: there is)
int fault_allocs = 0, fault_no_memory = 0;
}  // extern "C"

namespace {
thread_local int current = 0;
std::mutex devices_mu;
std::unordered_map<const void*, int> devices;
void put_device(const void* p) {
  std::lock_guard<std::mutex> lock(devices_mu);
  devices[p] = current;
}
int device_of(const void* p) {
  std::lock_guard<std::mutex> lock(devices_mu);
  return devices.count(p) ? devices[p] : 0;
}

// the status word, what it will hold, and when
int32_t* late_word = nullptr;
int32_t late_value = 0;
std::chrono::steady_clock::time_point late_at;
void decide(int32_t* status, uint32_t decision) {
  late_word = status + rsg::kResidentDecision;
  late_value = (int32_t)decision;
  late_at = std::chrono::steady_clock::now() + std::chrono::milliseconds(fault_late);
  fault_undecided = fault_late > 0;
  if (!fault_undecided) *late_word = late_value;
}
void decided() {
  *late_word = late_value;
  fault_undecided = 0;
}

template <typename A, typename F>
hipError_t resident(const A& a, F&& real) {
  if (fault_launch > 0 && fault_launch--) return hipErrorLaunchFailure;
  fault_resident++;
  if (fault_lost > 0 && fault_lost--) a.status[rsg::kResidentLost] = 1;
  if (a.ntiles == 1) return real();
  uint32_t* const decision = a.ctrl + 1;  // as the kernel keeps it
  if (a.chained && *decision == 2 * (a.seq - 1)) {
    *decision = 2 * a.seq;
    return hipSuccess;
  }
  *decision = 2 * a.seq + !fault_refuse;
  decide(a.status, *decision);
  if (fault_refuse == 0) return real();
  fault_refuse--;
  return hipSuccess;
}
template <typename A>
void velocity(const A& a) {
  fault_amp[fault_velocity % 4096] = a.amp[0];
  fault_trace[fault_velocity++ % 4096] = a.trace;
}
template <typename A>
void stress(const A& a) {
  fault_stress_amp[fault_stress++ % 4096] = a.amp[0];
}
}  // namespace

extern "C" {

hipError_t __real_hipEventQuery(hipEvent_t e);
hipError_t __wrap_hipEventQuery(hipEvent_t e) {
  if (fault_undecided) {
    if (std::chrono::steady_clock::now() < late_at) return hipErrorNotReady;
    decided();
  }
  return __real_hipEventQuery(e);
}

// pinned allocations made and freed so far, and whether there is no pinned memory for more
int fault_pinned = 0, fault_unpinned = 0, fault_no_pinned = 0;
hipError_t __real_hipHostMalloc(void** p, size_t bytes, unsigned int flags);
hipError_t __wrap_hipHostMalloc(void** p, size_t bytes, unsigned int flags) {
  if (fault_no_pinned) return hipErrorOutOfMemory;
  __atomic_fetch_add(&fault_pinned, 1, __ATOMIC_RELAXED);
  return __real_hipHostMalloc(p, bytes, flags);
}
hipError_t __real_hipHostFree(void* p);
hipError_t __wrap_hipHostFree(void* p) {
  __atomic_fetch_add(&fault_unpinned, 1, __ATOMIC_RELAXED);
  return __real_hipHostFree(p);
}

// waits for a stream so far
int fault_waits = 0;
hipError_t __real_hipStreamSynchronize(hipStream_t s);
hipError_t __wrap_hipStreamSynchronize(hipStream_t s) {
  __atomic_fetch_add(&fault_waits, 1, __ATOMIC_RELAXED);
  if (fault_undecided) decided();
  return __real_hipStreamSynchronize(s);
}

hipError_t __real_hipMallocFromPoolAsync(void** p, size_t bytes, hipMemPool_t pool, hipStream_t s);
hipError_t __wrap_hipMallocFromPoolAsync(void** p, size_t bytes, hipMemPool_t pool, hipStream_t s) {
  if (device_of(s) != current) return hipErrorInvalidValue;
  if (fault_no_memory && bytes >= (size_t)fault_no_memory) return hipErrorOutOfMemory;
  __atomic_fetch_add(&fault_allocs, 1, __ATOMIC_RELAXED);
  return __real_hipMallocFromPoolAsync(p, bytes, pool, s);
}

// Two devices: a stream or event is on the device current where it was made, memory is taken from
// the current device's pool, and mixing them is an error.
void fault_set_device(int d) { current = d; }
void fault_get_device(int* d) { *d = current; }
hipError_t __real_hipGetDevice(int* d);
hipError_t __wrap_hipGetDevice(int* d) {
  *d = current;
  return hipSuccess;
}
hipError_t __real_hipSetDevice(int d);
hipError_t __wrap_hipSetDevice(int d) {
  current = d;
  return hipSuccess;
}
hipError_t __real_hipStreamCreateWithFlags(hipStream_t* s, unsigned int flags);
hipError_t __wrap_hipStreamCreateWithFlags(hipStream_t* s, unsigned int flags) {
  const hipError_t e = __real_hipStreamCreateWithFlags(s, flags);
  put_device(*s);
  return e;
}
hipError_t __real_hipEventCreateWithFlags(hipEvent_t* v, unsigned flags);
hipError_t __wrap_hipEventCreateWithFlags(hipEvent_t* v, unsigned flags) {
  const hipError_t e = __real_hipEventCreateWithFlags(v, flags);
  put_device(*v);
  return e;
}

hipError_t __real_hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t __wrap_hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (device_of(e) != device_of(s)) return hipErrorInvalidHandle;
  if (fault_record > 0 && --fault_record == 0) return hipErrorUnknown;
  return __real_hipEventRecord(e, s);
}

#define RESIDENT_F64 _ZN3rsg19launch_resident_f64ERKNS_12ResidentArgsIdEEiP12ihipStream_t
#define RESIDENT_F32 _ZN3rsg19launch_resident_f32ERKNS_12ResidentArgsIfEEiP12ihipStream_t
hipError_t NAME(__real_, RESIDENT_F64)(const rsg::ResidentArgs<double>& a, int threads, hipStream_t s);
hipError_t NAME(__wrap_, RESIDENT_F64)(const rsg::ResidentArgs<double>& a, int threads, hipStream_t s) {
  return resident(a, [&]() { return NAME(__real_, RESIDENT_F64)(a, threads, s); });
}
hipError_t NAME(__real_, RESIDENT_F32)(const rsg::ResidentArgs<float>& a, int threads, hipStream_t s);
hipError_t NAME(__wrap_, RESIDENT_F32)(const rsg::ResidentArgs<float>& a, int threads, hipStream_t s) {
  return resident(a, [&]() { return NAME(__real_, RESIDENT_F32)(a, threads, s); });
}

#define VELOCITY_F64 _ZN3rsg19launch_velocity_f64ERKNS_12VelocityArgsIdEEiP12ihipStream_t
#define STRESS_F64 _ZN3rsg17launch_stress_f64ERKNS_10StressArgsIdEEiP12ihipStream_t
hipError_t NAME(__real_, VELOCITY_F64)(const rsg::VelocityArgs<double>& a, int block, hipStream_t s);
hipError_t NAME(__wrap_, VELOCITY_F64)(const rsg::VelocityArgs<double>& a, int block, hipStream_t s) {
  velocity(a);
  return NAME(__real_, VELOCITY_F64)(a, block, s);
}
hipError_t NAME(__real_, STRESS_F64)(const rsg::StressArgs<double>& a, int block, hipStream_t s);
hipError_t NAME(__wrap_, STRESS_F64)(const rsg::StressArgs<double>& a, int block, hipStream_t s) {
  stress(a);
  return NAME(__real_, STRESS_F64)(a, block, s);
}

}  // extern "C"
