// Test harness: a stand-in for the HIP runtime calls liberod.so makes, loaded
// before it, so that what the library does on the host (plans, allocations,
// copies, which device they are on) can be checked with no GPU.  "Device"
// memory is host memory, copies are copies, kernels only leave a line in the
// log.  Two devices, each of a size the test sets.
#include <sys/mman.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>

namespace {
  using Error = int;
  constexpr Error kOk = 0, kInvalid = 1, kNoMemory = 2, kBadHandle = 400;
  struct Dim3 {
    uint32_t x, y, z;
  };
  struct Handle {
    int device;
    double clock = 0.0;  // events: the time of their last record
  };
  struct Block {
    size_t bytes;
    int device;  // -1: pinned host memory
  };

  std::recursive_mutex g_mutex;
  std::map<const void*, Block> g_blocks;
  std::map<const void*, std::string> g_kernels;
  size_t g_capacity = size_t(64) << 30, g_live[2] = {};
  double g_clock = 0.0;
  long g_left = -1;
  Error g_last = kOk;
  std::string g_log, g_fast[2];
  thread_local int t_device = 0;
  struct Call {
    Dim3 grid, block;
    size_t shmem;
    Handle* stream;
  };
  thread_local Call t_call;

  template <typename... A>
  void note(const char* fmt, A... a) {
    char buf[512];
    (void)std::snprintf(buf, sizeof(buf), fmt, a...);
    std::lock_guard<std::recursive_mutex> lock(g_mutex);
    g_log += buf;
    g_log += '\n';
  }

  // the block an address lies in, or null
  const Block* owner(const void* p) {
    auto it = g_blocks.upper_bound(p);
    if (it == g_blocks.begin()) return nullptr;
    --it;
    const char* b = static_cast<const char*>(it->first);
    return static_cast<const char*>(p) < b + it->second.bytes ? &it->second : nullptr;
  }

  Error take(void** p, size_t bytes, int device) {
    std::lock_guard<std::recursive_mutex> lock(g_mutex);
    *p = nullptr;
    if (device >= 0 && g_live[device] + bytes > g_capacity) return kNoMemory;
    void* m = mmap(nullptr, bytes + 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return kNoMemory;
    g_blocks[m] = {bytes + 1, device};
    if (device >= 0) g_live[device] += bytes;
    *p = m;
    return kOk;
  }

  Error give(void* p) {
    std::lock_guard<std::recursive_mutex> lock(g_mutex);
    if (!p) return kOk;
    auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return kInvalid;
    if (it->second.device >= 0) g_live[it->second.device] -= it->second.bytes - 1;
    munmap(p, it->second.bytes);
    g_blocks.erase(it);
    return kOk;
  }

  // state pointers (four each in arguments 0 and 1) that are not memory of the device
  int foreign(void** args, int device) {
    int n = 0;
    for (int a = 0; a < 2; ++a)
      for (int i = 0; i < 4; ++i) {
        const Block* b = owner(static_cast<void**>(args[a])[i]);
        n += !b || b->device != device;
      }
    return n;
  }
}  // namespace

extern "C" {
// ---- what a test sets and reads
void double_capacity(size_t bytes) { g_capacity = bytes; }
size_t double_live(int device) { return g_live[device]; }
// kernels whose name holds `name` take a hundredth of the time, those whose name holds `faster` far less
void double_fast(const char* name, const char* faster) {
  g_fast[0] = name;
  g_fast[1] = faster;
}
const char* double_log() { return g_log.c_str(); }
void double_clear() { g_log.clear(); }
void double_fail_after(long n) { g_left = n; }  // launches until one is refused
int double_set_device(int d) { return t_device = d, 0; }

// ---- the runtime's calls
Error hipGetDeviceCount(int* n) { return *n = 2, kOk; }
Error hipGetDevice(int* d) { return *d = t_device, kOk; }
Error hipSetDevice(int d) { return t_device = d, kOk; }
Error hipDeviceGetAttribute(int* v, int, int) { return *v = 256, kOk; }  // (only the compute units are asked for)
Error hipGetLastError() { return std::exchange(g_last, kOk); }
const char* hipGetErrorString(Error e) { return e == kNoMemory ? "out of memory" : "error"; }

Error hipMalloc(void** p, size_t bytes) {
  const Error e = take(p, bytes, t_device);
  note("malloc %d %zu%s", t_device, bytes, e ? " refused" : "");
  return e;
}
Error hipFree(void* p) { return give(p); }
Error hipHostMalloc(void** p, size_t bytes, unsigned) {
  note("pinned %d %zu", t_device, bytes);
  return take(p, bytes, -1);
}
Error hipHostFree(void* p) { return give(p); }
Error hipMemGetInfo(size_t* free, size_t* total) {
  *total = g_capacity;
  *free = g_capacity - g_live[t_device];
  return kOk;
}
Error hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), kOk; }

Error hipMemcpyAsync(void* dst, const void* src, size_t bytes, int, Handle*) {
  const Block* b = owner(dst);
  note("copy %s %zu", !b ? "pageable" : (b->device < 0 ? "pinned" : "device"), bytes);
  std::memmove(dst, src, bytes);
  return kOk;
}
Error hipMemcpy2DAsync(void* dst, size_t dp, const void* src, size_t sp, size_t w, size_t h, int, Handle*) {
  note("copy2d %zu x %zu", w, h);
  for (size_t i = 0; i < h; ++i) std::memmove(static_cast<char*>(dst) + i * dp, static_cast<const char*>(src) + i * sp, w);
  return kOk;
}
Error hipMemsetAsync(void* dst, int v, size_t bytes, Handle*) {
  // (fresh memory is zero and stays untouched)
  if (v || bytes < (size_t(1) << 20)) std::memset(dst, v, bytes);
  return kOk;
}

Error hipStreamCreateWithFlags(Handle** s, unsigned) { return *s = new Handle{t_device}, kOk; }
Error hipStreamDestroy(Handle* s) { return delete s, kOk; }
Error hipStreamSynchronize(Handle*) { return kOk; }
Error hipEventCreateWithFlags(Handle** e, unsigned) { return *e = new Handle{t_device}, kOk; }
Error hipEventCreate(Handle** e) { return hipEventCreateWithFlags(e, 0); }
Error hipEventDestroy(Handle* e) { return delete e, kOk; }
Error hipEventRecord(Handle* e, Handle* s) {
  if (e->device != s->device) return kBadHandle;
  e->clock = g_clock;
  return kOk;
}
Error hipEventSynchronize(Handle*) { return kOk; }
Error hipStreamWaitEvent(Handle* s, Handle* e, unsigned) { return s->device == e->device ? kOk : kBadHandle; }
Error hipEventElapsedTime(float* ms, Handle* a, Handle* b) { return *ms = static_cast<float>(b->clock - a->clock), kOk; }

Error hipStreamBeginCapture(Handle*, int) {
  note("%s", "capture");
  return kOk;
}
Error hipStreamEndCapture(Handle*, void** g) { return *g = &g_log, kOk; }
Error hipGraphGetNodes(void*, void**, size_t* n) { return *n = 2, kOk; }
Error hipGraphInstantiate(void** x, void*, void**, char*, size_t) { return *x = &g_log, kOk; }
Error hipGraphDestroy(void*) { return kOk; }
Error hipGraphExecDestroy(void*) { return kOk; }
Error hipGraphLaunch(void*, Handle*) {
  note("%s", "replay");
  return kOk;
}

Error hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t, Handle* stream) {
  if (g_left >= 0 && g_left-- == 0) return g_last = kInvalid;
  const std::string& name = g_kernels[f];
  double unit = 1.0;
  for (int i = 0; i < 2; ++i)
    if (!g_fast[i].empty() && name.find(g_fast[i]) != std::string::npos) unit = i ? 1e-5 : 1e-2;
  if (name.find("k_fused") != std::string::npos) {
    const int total = *static_cast<int*>(args[13]), split = *static_cast<int*>(args[14]);
    note("launch %s grid %u steps %d split %d foreign %d", name.c_str(), grid.x, total, split, foreign(args, stream->device));
    g_clock += unit * (total + 8) * (1.0 + 1e-3 * grid.x);
  } else if (name.find("k_steps") != std::string::npos) {
    note("launch %s grid %u steps %d left %d own %d foreign %d", name.c_str(), grid.x, *static_cast<int*>(args[10]),
         *static_cast<int*>(args[11]), *static_cast<int*>(args[12]), foreign(args, stream->device));
  } else {
    note("launch %s grid %u block %u", name.c_str(), grid.x, block.x);
    g_clock += unit;
  }
  return kOk;
}
Error __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, Handle* s) { return t_call = {grid, block, shmem, s}, kOk; }
Error __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shmem, Handle** s) {
  *grid = t_call.grid;
  *block = t_call.block;
  *shmem = t_call.shmem;
  *s = t_call.stream;
  return kOk;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
