// A stand-in for the HIP runtime, for tests of the library's host code without a
// GPU: built as libamdhip64.so.7 and found before the real one through
// LD_LIBRARY_PATH, it defines every runtime function that libhkmoe.so imports.
// Nothing runs; each call that matters for ordering is appended to a log that
// the test reads (fake_hip_log): kernel launches with their demangled name, grid
// and stream, events, streams.
#include <cxxabi.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
struct Call {
  Dim3 grid, block;
  size_t lds;
  void* stream;
};
std::mutex mu;
std::string text, log_copy;
std::map<const void*, std::string> kernels;
std::map<std::string, int> fail_in;  // function -> calls until it fails (0: the next)
int delay_ms = 0, capturing = 0, last_error = 0;
intptr_t next_handle = 1;
std::string watch_name;
int watch_arg = -1;
thread_local std::vector<Call> calls;

void say(const std::string& s) { text += s + "\n"; }
bool fails(const char* fn) {
  auto it = fail_in.find(fn);
  if (it == fail_in.end() || it->second-- > 0) return false;
  fail_in.erase(it);
  last_error = 2;
  say(std::string("failed ") + fn);
  return true;
}
std::string id(const void* p) { return std::to_string(reinterpret_cast<intptr_t>(p)); }
int launch(const void* f, Dim3 grid, void** args, void* stream) {
  std::lock_guard<std::mutex> g(mu);
  const std::string& name = kernels[f];
  say("launch " + name + " grid=" + std::to_string(grid.x) + " stream=" + id(stream));
  if (watch_arg >= 0 && name.find(watch_name) != std::string::npos)
    say("arg " + std::to_string(*static_cast<int32_t*>(args[watch_arg])));
  return 0;
}
int make(const char* fn, const char* what, void** out) {
  if (delay_ms) std::this_thread::sleep_for(std::chrono::milliseconds(delay_ms));
  std::lock_guard<std::mutex> g(mu);
  if (fails(fn)) return 2;
  *out = reinterpret_cast<void*>(next_handle++);
  say(std::string(what) + "_create " + id(*out));
  return 0;
}
int destroy(const char* what, void* h) {
  std::lock_guard<std::mutex> g(mu);
  say(std::string(what) + "_destroy " + id(h));
  return 0;
}
}  // namespace

extern "C" {
// ---- the test's side ------------------------------------------------------
const char* fake_hip_log() {
  std::lock_guard<std::mutex> g(mu);
  log_copy = text;
  return log_copy.c_str();
}
void fake_hip_clear() {
  std::lock_guard<std::mutex> g(mu);
  text.clear();
}
void fake_hip_delay(int ms) { delay_ms = ms; }          // of every stream and event creation
void fake_hip_capturing(int on) { capturing = on; }     // every stream reports an active capture
void fake_hip_fail(const char* fn, int after) {         // fn fails once, after `after` good calls
  std::lock_guard<std::mutex> g(mu);
  fail_in[fn] = after;
}
void fake_hip_watch(const char* name, int arg) {        // log int argument `arg` of these kernels
  std::lock_guard<std::mutex> g(mu);
  watch_name = name;
  watch_arg = arg;
}

// ---- the runtime ------------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  int status = 0;
  char* d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  std::string s = status == 0 ? d : name;
  std::free(d);
  if (s.rfind("void ", 0) == 0) s = s.substr(5);
  int depth = 0;  // cut the parameter list, not a "(" inside the template arguments
  for (size_t i = 0; i < s.size(); ++i) {
    if (s[i] == '<') ++depth;
    else if (s[i] == '>') --depth;
    else if (s[i] == '(' && depth == 0) {
      s.resize(i);
      break;
    }
  }
  for (char& c : s)
    if (c == ' ') c = '_';
  kernels[host] = s;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  calls.push_back(Call{grid, block, lds, stream});
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  const Call c = calls.back();
  calls.pop_back();
  *grid = c.grid;
  *block = c.block;
  *lds = c.lds;
  *stream = c.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void** args, size_t, void* stream) {
  return launch(f, grid, args, stream);
}
int hipExtLaunchKernel(const void* f, Dim3 grid, Dim3, void** args, size_t, void* stream, void*, void*, int) {
  return launch(f, grid, args, stream);
}
int hipGetDevice(int* d) { return *d = 0; }
int hipDeviceGetAttribute(int* v, int, int) {  // only asked for the CU count
  *v = 256;
  return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetLastError() {
  std::lock_guard<std::mutex> g(mu);
  const int e = last_error;
  last_error = 0;
  return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetSymbolAddress(void** p, const void*) {
  *p = reinterpret_cast<void*>(intptr_t{1} << 40);
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { return make("hipStreamCreateWithFlags", "stream", s); }
int hipStreamDestroy(void* s) { return destroy("stream", s); }
int hipStreamIsCapturing(void*, int* status) {
  *status = capturing;
  return 0;
}
int hipEventCreate(void** e) { return make("hipEventCreate", "event", e); }
int hipEventCreateWithFlags(void** e, unsigned) { return make("hipEventCreateWithFlags", "event", e); }
int hipEventDestroy(void* e) { return destroy("event", e); }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.0f;
  return 0;
}
int hipEventRecord(void* e, void* s) {
  std::lock_guard<std::mutex> g(mu);
  say("record " + id(e) + " stream=" + id(s));
  return 0;
}
int hipStreamWaitEvent(void* s, void* e, unsigned) {
  std::lock_guard<std::mutex> g(mu);
  say("wait " + id(e) + " stream=" + id(s));
  return 0;
}
}
