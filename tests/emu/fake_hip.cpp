// The HIP calls of libspeckle_hip.so as host functions, for tests of its host
// code without a GPU: which kernels a call launches, in which grids, and what
// it does when an allocation or a launch fails.  Device memory is host memory,
// no kernel runs, copies and small fills are made.  Loaded RTLD_GLOBAL in
// front of the library (fake_run.py), so that its calls come here.
#include <cxxabi.h>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <sstream>
#include <string>

namespace {
struct Dim { uint32_t x, y, z; };
std::map<const void*, std::string> names;
std::map<void*, size_t> blocks;
std::map<std::string, long long> knob{{"cus", 256}, {"occupancy", 1}};
std::string log_text;
size_t live = 0;
int last = 0;
Dim cfg_grid, cfg_block;

int ret(int e) { if (e) last = e; return e; }
// knob `name` counts down the calls that still fail
bool fails(const char* name) {
  auto it = knob.find(name);
  if (it == knob.end() || it->second <= 0) return false;
  --it->second;
  return true;
}
int launch(const char* how, const void* f, Dim g, Dim b, void** args) {
  const std::string& name = names[f];
  std::ostringstream o;
  o << how << ' ' << name << ' ' << g.x << ' ' << g.y << ' ' << g.z << ' ' << b.x;
  if (name == "k_resident_begin")   // words of flags, values to empty, whether
    o << " begin " << *(int*)args[1] << ' ' << *(int*)args[4] << ' ' << *(int*)args[5];
  const bool bad = *how == 'c' ? fails("fail_cooperative") : false;
  if (bad) o << " failed";
  log_text += o.str() + "\n";
  return ret(bad ? 720 : 0);   // hipErrorCooperativeLaunchTooLarge
}
}  // namespace

extern "C" {
void fake_set(const char* name, long long v) { knob[name] = v; }
long long fake_get(const char* name) { return knob[name]; }
const char* fake_log() { return log_text.c_str(); }
void fake_clear() { log_text.clear(); }
unsigned long long fake_live() { return live; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* dev, unsigned, void*, void*,
                           void*, void*, int*) {
  int st = 0;
  char* d = abi::__cxa_demangle(dev, nullptr, nullptr, &st);
  std::string s = d ? d : dev;
  std::free(d);
  // "void spk::(anonymous namespace)::k_x<1, 2>(args)" -> "k_x<1,2>"
  const size_t k = s.find("k_"), a = s.find_first_of("<(", k);
  size_t end = a;
  if (a != std::string::npos && s[a] == '<') {
    int depth = 0;
    for (end = a; end < s.size(); ++end) {
      if (s[end] == '<') ++depth;
      if (s[end] == '>' && --depth == 0) { ++end; break; }
    }
  }
  std::string t;
  for (char c : s.substr(k, end - k))
    if (c != ' ') t += c;
  names[host] = t;
}
int __hipPushCallConfiguration(Dim g, Dim b, size_t, void*) { cfg_grid = g; cfg_block = b; return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* sh, void** st) {
  *g = cfg_grid; *b = cfg_block; *sh = 0; *st = nullptr;
  return 0;
}
int hipLaunchKernel(const void* f, Dim g, Dim b, void** args, size_t, void*) {
  return launch("plain", f, g, b, args);
}
int hipExtLaunchKernel(const void* f, Dim g, Dim b, void** args, size_t, void*, void*, void*, int) {
  return launch("plain", f, g, b, args);
}
int hipLaunchCooperativeKernel(const void* f, Dim g, Dim b, void** args, unsigned, void*) {
  return launch("coop", f, g, b, args);
}

int hipMalloc(void** p, size_t n) {
  const auto limit = knob.find("malloc_limit");   // bytes in all
  if (limit != knob.end() && limit->second > 0 && live + n > (size_t)limit->second) {
    *p = nullptr;
    return ret(2);
  }
  *p = std::malloc(n);
  blocks[*p] = n;
  live += n;
  return 0;
}
int hipFree(void* p) {
  if (!p) return 0;
  live -= blocks.at(p);   // throws on a pointer that hipMalloc did not give
  blocks.erase(p);
  std::free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return 0; }
int hipHostFree(void* p) { std::free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) {
  std::memcpy(d, s, n);
  if (n == 3 * sizeof(int)) ((int*)d)[2] = (int)knob["sticky"];   // a plan's wait flags
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { std::memset(d, v, n); return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char sym[1 << 20]; *p = sym; return 0; }

int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int, size_t) {
  ++knob["queries"];
  *n = (int)(names[f].find(",2,true>") != std::string::npos ? 2 * knob["occupancy"]
                                                             : knob["occupancy"]);
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) { *v = (int)knob["cus"]; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void*, int* s) { *s = (int)knob["capturing"]; return 0; }
int hipGetLastError() { const int e = last; last = 0; return e; }
const char* hipGetErrorString(int) { return "an error that the test asked for"; }
int hipEventCreate(void** e) { *e = std::malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = std::malloc(1); return 0; }
int hipEventDestroy(void* e) { std::free(e); return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0; return 0; }
}
