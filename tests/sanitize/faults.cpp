// faults.cpp -- failures on demand for the host code over its CPU stand-ins (hip_host_stub.cpp,
// resident_stub.cpp).  TEST INFRASTRUCTURE ONLY: linked with --wrap, so that the calls named below
// pass through here; a test sets the counters through ctypes.
#include <system_error>
#include <thread>

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

}  // extern "C"
