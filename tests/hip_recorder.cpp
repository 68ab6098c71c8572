/* A HIP runtime without a device, preloaded over the real one by
 * test_host_calls.py: memory is host memory, kernels do not run, and every
 * call is recorded as a line of text. What the library does around its
 * kernels -- which buffers it holds, on which stream it launches, what it
 * waits for -- can so be tested where there is no GPU, also after a failed
 * allocation and under stream capture, and without a kernel that would write
 * through a wrong pointer.
 *
 * What a stream was given is done once it, a stream that waited for it, an event
 * recorded behind it or the device is synchronised. While a stream is captured
 * in another mode than relaxed, allocating and freeing fail as on a device. */
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <utility>
#include <vector>

namespace {
enum { OK = 0, BAD_VALUE = 1, NO_MEMORY = 2, CAPTURING = 900 };
struct Dim3 { uint32_t x, y, z; };
struct Event { void* stream; int order; };

std::vector<std::string> log_;
std::map<const void*, std::string> kernels;
std::map<void*, size_t> live;
std::map<void*, std::set<Event*>> waits; /* per stream */
/* calls' numbers that a stream is to write to host memory */
struct Done { void* stream; uint32_t* to; uint32_t value; int order; };
std::vector<Done> done;
int order = 0;
size_t fail_above = SIZE_MAX;
int fail_in = 0; /* the allocation to fail: 1 the next */
void* captured = nullptr;
int capture_mode = 0;
Dim3 grid_, block_;
size_t shared_;
void* stream_;

template<class... A> void note(const char* fmt, A... a)
{
  char line[256];
  snprintf(line, sizeof(line), fmt, a...);
  log_.push_back(line);
}

/* what a stream (or all) was given up to `last' is done */
void finish(void* s, bool all, int last)
{
  for(auto& d : done)
    if(d.to && (all || d.stream == s) && d.order <= last) { *d.to = d.value; d.to = nullptr; }
}

bool refused() { return captured && capture_mode != 2; }
} /* namespace */

extern "C" {
/* the tests' side */
size_t recorder_log(char* out, size_t n)
{
  std::string s;
  for(auto& l : log_) s += l + "\n";
  if(n > s.size()) memcpy(out, s.c_str(), s.size() + 1);
  return s.size() + 1;
}
void recorder_clear(void) { log_.clear(); }
void recorder_fail_above(size_t n) { fail_above = n; }
void recorder_fail_in(int n) { fail_in = n; }
size_t recorder_live_bytes(void)
{
  size_t n = 0;
  for(auto& l : live) n += l.second;
  return n;
}

/* the runtime's */
void** __hipRegisterFatBinary(const void*) { static void* mod; return &mod; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*,
                           void*, int*)
{
  kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* s)
{
  grid_ = g; block_ = b; shared_ = sh; stream_ = s;
  return OK;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** s)
{
  *g = grid_; *b = block_; *sh = shared_; *s = stream_;
  return OK;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3, void** args, size_t, void* s)
{
  if(kernels[f].find("done_kernel") != std::string::npos)
    done.push_back({s, *(uint32_t**)args[0], *(uint32_t*)args[1], ++order});
  note("launch %.160s grid %u stream %p", kernels[f].c_str(), g.x, s);
  return OK;
}
int hipMalloc(void** p, size_t n)
{
  if(refused() || n > fail_above || (fail_in && !--fail_in)) {
    note("malloc %zu refused", n);
    return refused() ? (int)CAPTURING : (int)NO_MEMORY;
  }
  *p = calloc(n, 1);
  live[*p] = n;
  note("malloc %zu %p", n, *p);
  return OK;
}
int hipFree(void* p)
{
  if(!p) return OK;
  if(refused()) { note("free %p refused", p); return CAPTURING; }
  if(!live.count(p)) { note("free %p unknown", p); return BAD_VALUE; }
  note("free %zu %p", live[p], p);
  live.erase(p);
  free(p);
  return OK;
}
int hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(n, 1); return OK; }
int hipHostFree(void* p) { free(p); return OK; }
int hipMemcpy(void* d, const void* s, size_t n, int)
{
  if(refused()) return CAPTURING;
  memcpy(d, s, n);
  return OK;
}
int hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int)
{
  for(size_t y = 0; y < h; ++y) memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
  return OK;
}
int hipMemset(void* p, int v, size_t n) { memset(p, v, n); return OK; }
int hipMemsetAsync(void* p, int v, size_t n, void*) { memset(p, v, n); return OK; }
int hipGetDevice(int* d) { *d = 0; return OK; }
int hipGetLastError(void) { return OK; }
/* 256 compute units; the clock rate of the other attribute asked for */
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int block, size_t)
{
  *n = 3 * 256 / block;
  return OK;
}
int hipGetSymbolAddress(void** p, const void*)
{
  static void* scratch = calloc(64 << 20, 1);
  *p = scratch;
  return OK;
}
int hipDeviceSynchronize(void)
{
  note("sync device%s", "");
  finish(nullptr, true, order);
  return OK;
}
int hipStreamCreateWithFlags(void** s, unsigned) { *s = malloc(16); note("stream %p", *s); return OK; }
int hipStreamDestroy(void* s) { free(s); return OK; }
int hipStreamSynchronize(void* s)
{
  note("sync stream %p", s);
  finish(s, false, order);
  for(Event* e : waits[s]) finish(e->stream, false, e->order);
  waits[s].clear();
  return OK;
}
int hipStreamWaitEvent(void* s, void* e, unsigned)
{
  note("wait stream %p event %p", s, e);
  waits[s].insert((Event*)e);
  return OK;
}
int hipStreamGetPriority(void*, int* p) { *p = 0; return OK; }
int hipExtStreamGetCUMask(void*, uint32_t n, uint32_t* m) { memset(m, 255, 4 * n); return OK; }
int hipStreamIsCapturing(void* s, int* status) { *status = s && s == captured; return OK; }
int hipThreadExchangeStreamCaptureMode(int* mode)
{
  std::swap(*mode, capture_mode);
  return OK;
}
int hipStreamBeginCapture(void* s, int mode) { captured = s; capture_mode = mode; return OK; }
int hipStreamEndCapture(void*, void** g) { captured = nullptr; *g = malloc(16); return OK; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = malloc(16); return OK; }
int hipGraphLaunch(void*, void* s) { note("graph stream %p", s); return OK; }
int hipGraphDestroy(void* g) { free(g); return OK; }
int hipGraphExecDestroy(void* x) { free(x); return OK; }
int hipEventCreateWithFlags(void** e, unsigned)
{
  *e = new Event{nullptr, 0};
  return OK;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e)
{
  for(auto& w : waits) w.second.erase((Event*)e);
  delete (Event*)e;
  return OK;
}
int hipEventRecord(void* e, void* s)
{
  note("record stream %p event %p", s, e);
  *(Event*)e = Event{s, ++order};
  return OK;
}
int hipEventSynchronize(void* e)
{
  note("sync event %p", e);
  finish(((Event*)e)->stream, false, ((Event*)e)->order);
  return OK;
}
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 1.f; return OK; }
}
