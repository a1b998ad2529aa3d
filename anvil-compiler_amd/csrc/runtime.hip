// Context, memory, timing and error reporting of the anvil_mi355x C ABI.
#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

#include "common.h"

namespace anvil {

static thread_local std::string g_last_error;
__thread KernelTimer g_timer;

// A recorded launch: the kernel and a copy of its arguments (ptrs into bytes).
struct LaunchRecord {
  const void* sym;
  hipFunction_t fn;
  dim3 grid, block;
  unsigned lds;
  std::vector<char> bytes;
  std::vector<void*> ptrs;
  std::vector<unsigned short> sizes;
};

// What anvil_graph_end and anvil_record_end return: the recorded launches, or (exec set) a captured HIP graph whose
// nodes are not all launches that the capturing thread made through launch_kernel.
struct LaunchList {
  std::vector<LaunchRecord> launches;
  hipGraphExec_t exec = nullptr;
  bool incomplete = false;             // a launch could not be noted
};

// The recordings under way in the order they began. Each notes the launches that the thread which began it makes on its
// stream. A capture may end on another thread and a context may be destroyed with recordings open, so they are held for
// all threads; g_recording, their number, keeps launches outside of any recording from taking the lock.
struct Recording {
  hipStream_t stream;
  unsigned long long thread;
  bool capture;
  LaunchList* list;
};
static std::mutex g_recordings_lock;
static std::vector<Recording> g_recordings;
static std::atomic<int> g_recording{0};

static unsigned long long this_thread() {            // never given twice, unlike a thread id
  static std::atomic<unsigned long long> next{1};
  static thread_local unsigned long long id = next++;
  return id;
}

static bool record_start(hipStream_t s, bool capture) {
  std::lock_guard<std::mutex> hold(g_recordings_lock);
  LaunchList* l = new (std::nothrow) LaunchList();
  if (!l) return false;
  try {
    g_recordings.push_back({s, this_thread(), capture, l});
  } catch (const std::bad_alloc&) {
    delete l;
    return false;
  }
  ++g_recording;
  return true;
}

// The innermost recording of this kind on the stream, ended: a capture's whichever thread began it, a list's on its own
// thread. Null when there is none.
static LaunchList* record_stop(hipStream_t s, bool capture) {
  std::lock_guard<std::mutex> hold(g_recordings_lock);
  for (size_t i = g_recordings.size(); i-- > 0;) {
    const Recording r = g_recordings[i];
    if (r.stream != s || r.capture != capture || (!capture && r.thread != this_thread())) continue;
    g_recordings.erase(g_recordings.begin() + (long)i);
    --g_recording;
    return r.list;
  }
  return nullptr;
}

static void record_drop(hipStream_t s) {             // a destroyed stream's
  std::lock_guard<std::mutex> hold(g_recordings_lock);
  for (size_t i = g_recordings.size(); i-- > 0;)
    if (g_recordings[i].stream == s) {
      delete g_recordings[i].list;
      g_recordings.erase(g_recordings.begin() + (long)i);
      --g_recording;
    }
}

static void note(LaunchList& list, const void* sym, dim3 grid, dim3 block, unsigned lds, void** args,
                 const unsigned short* sizes, int n) {
  LaunchRecord r{sym, nullptr, grid, block, lds, {}, {}, {sizes, sizes + n}};
  if (hipGetFuncBySymbol(&r.fn, sym) != hipSuccess) {
    (void)hipGetLastError();
    list.incomplete = true;
    return;
  }
  size_t total = 0;
  for (int i = 0; i < n; ++i) total = (total + 15) / 16 * 16 + sizes[i];
  r.bytes.resize(total + 1);
  size_t at = 0;
  for (int i = 0; i < n; ++i) {
    at = (at + 15) / 16 * 16;
    std::memcpy(r.bytes.data() + at, args[i], sizes[i]);
    r.ptrs.push_back(r.bytes.data() + at);
    at += sizes[i];
  }
  list.launches.push_back(std::move(r));             // moving the vectors keeps their storage, and so the pointers
}

// A launch that cannot be noted has still run: it only spoils the recordings, which then end in an error.
static void note_launch(const void* sym, dim3 grid, dim3 block, unsigned lds, hipStream_t s, void** args,
                        const unsigned short* sizes, int n) {
  std::lock_guard<std::mutex> hold(g_recordings_lock);
  for (const Recording& rec : g_recordings) {
    if (rec.stream != s || rec.thread != this_thread()) continue;
    try {
      note(*rec.list, sym, grid, block, lds, args, sizes, n);
    } catch (const std::bad_alloc&) {
      rec.list->incomplete = true;
    }
  }
}

int launch_kernel(const void* sym, dim3 grid, dim3 block, unsigned lds, hipStream_t s, void** args,
                  const unsigned short* sizes, int n) {
  hipError_t e;
  if (g_timer.stop && g_timer.stream == s) {
    hipEvent_t start = g_timer.start;
    g_timer.start = nullptr;
    e = hipExtLaunchKernel(sym, grid, block, args, lds, s, start, g_timer.stop, 0);
  } else {
    e = hipLaunchKernel(sym, grid, block, args, lds, s);
  }
  if (e == hipSuccess && g_recording.load(std::memory_order_relaxed)) note_launch(sym, grid, block, lds, s, args, sizes, n);
  return e == hipSuccess ? ANVIL_OK : hip_fail(e, "kernel launch");
}

int set_error(int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return set_error(ANVIL_E_RUNTIME, "%s: %s (%d)", what, hipGetErrorString(e), (int)e);
}

int check_ctx(anvil_ctx* ctx) {
  if (!ctx) return set_error(ANVIL_E_VALUE, "null context");
  ANVIL_HIP(hipSetDevice(ctx->device));
  return ANVIL_OK;
}

__global__ void zero_kernel(uint8_t* __restrict__ p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  // 16-byte body on an aligned pointer, byte head/tail otherwise
  if (((uintptr_t)p & 15) == 0) {
    size_t n16 = n / 16;
    uint4 z = {0, 0, 0, 0};
    for (size_t j = i; j < n16; j += stride) reinterpret_cast<uint4*>(p)[j] = z;
    for (size_t j = n16 * 16 + i; j < n; j += stride) p[j] = 0;
  } else {
    for (size_t j = i; j < n; j += stride) p[j] = 0;
  }
}

int zero_fill(hipStream_t s, void* dst, size_t bytes) {
  size_t blocks = (bytes / 16 + 255) / 256;
  blocks = blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks);
  ANVIL_LAUNCH(zero_kernel, dim3((unsigned)blocks), dim3(256), 0, s, (uint8_t*)dst, bytes);
  ANVIL_LAUNCHED();
  return ANVIL_OK;
}

}  // namespace anvil

using namespace anvil;

// Device buffers and the context's flags into page-locked host memory by one kernel, instead of one copy command each.
// Measured with the wait (the buffer, 4 KiB more and the flags; copy commands -> kernel): 4 KiB 18 -> 14 us, 32 KiB 29 ->
// 14, 512 KiB 38 -> 22, 4 MiB 103 -> 88, 16 MiB 323 -> 318: there the link bounds both, and the copy engine leaves the CUs
// free. A small forward's read-back was two copies, a wait and a copy of the flags, about 45 us of a 64-wide block's 175.
constexpr int FETCH_MAX = 8;                            // buffers of one launch
constexpr size_t FETCH_KERNEL_MAX = 4 << 20;
struct FetchArgs {
  const int8_t* src[FETCH_MAX];
  int8_t* dst[FETCH_MAX];
  long long bytes[FETCH_MAX];
  int n;
  const unsigned* flags;                                // null: not fetched
  unsigned* host_flags;
};

__global__ __launch_bounds__(256) void fetch_kernel(FetchArgs a) {
  const long long first = (long long)blockIdx.x * 256 + threadIdx.x, step = (long long)gridDim.x * 256;
  for (int i = 0; i < a.n; ++i) {
    const long long chunks = a.bytes[i] / 16;
    for (long long c = first; c < chunks; c += step)
      reinterpret_cast<int4*>(a.dst[i])[c] = reinterpret_cast<const int4*>(a.src[i])[c];
    for (long long b = 16 * chunks + first; b < a.bytes[i]; b += step) a.dst[i][b] = a.src[i][b];
  }
  if (a.flags && first == 0) *a.host_flags = *a.flags;
}

static int report_flags(anvil_ctx* ctx, bool nonfinite_first) {
  const unsigned flags = *(volatile unsigned*)ctx->host_flags;
  if (!flags) return ANVIL_OK;
  ANVIL_HIP(hipMemset(ctx->flags, 0, sizeof(unsigned)));
  const char* nonfinite = "a float input holds NaN or infinite values";
  if (nonfinite_first && (flags & FLAG_NONFINITE)) return set_error(ANVIL_E_VALUE, "%s", nonfinite);
  if (flags & FLAG_OVERFLOW) return set_error(ANVIL_E_OVERFLOW, "an int32 intermediate overflowed on the device");
  if (flags & FLAG_ZERODIV) return set_error(ANVIL_E_ZERODIV, "a softmax row summed to zero");
  if (flags & FLAG_SHIFT) return set_error(ANVIL_E_VALUE, "an rmsnorm shift s + k left [0, 31]");
  if (flags & FLAG_NONFINITE) return set_error(ANVIL_E_VALUE, "%s", nonfinite);
  return set_error(ANVIL_E_VALUE, "an operand left its dtype range on the device (flags %u)", flags);
}

extern "C" {

const char* anvil_last_error(void) { return g_last_error.c_str(); }

int anvil_version(void) { return 1; }

int anvil_init(int device, anvil_ctx** out) {
  if (!out) return set_error(ANVIL_E_VALUE, "anvil_init: null output pointer");
  *out = nullptr;
  int n = 0;
  ANVIL_HIP(hipGetDeviceCount(&n));
  if (device < 0 || device >= n) return set_error(ANVIL_E_VALUE, "anvil_init: device %d of %d", device, n);
  ANVIL_HIP(hipSetDevice(device));
  hipDeviceProp_t prop;
  ANVIL_HIP(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return set_error(ANVIL_E_RUNTIME, "anvil_init: device %d is %s, this library is built for gfx950", device,
                     prop.gcnArchName);
  anvil_ctx* c = new anvil_ctx();
  c->device = device;
  c->num_cu = prop.multiProcessorCount;
  if (const char* cfg = std::getenv("ANVIL_GEMM_CFG")) c->gemm_cfg = std::atoi(cfg);
  hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc(&c->flags, 256);
  if (e == hipSuccess) e = hipMemset(c->flags, 0, 256);
  if (e == hipSuccess) e = hipHostMalloc((void**)&c->host_flags, 64, hipHostMallocDefault);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    anvil_destroy(c);
    return hip_fail(e, "anvil_init");
  }
  if (int r = gemm_scratch_setup(device)) {
    anvil_destroy(c);
    return r;
  }
  *out = c;
  return ANVIL_OK;
}

int anvil_destroy(anvil_ctx* ctx) {
  if (!ctx) return ANVIL_OK;
  if (g_timer.stream == ctx->stream) g_timer = KernelTimer{};
  hipSetDevice(ctx->device);
  if (ctx->stream) hipStreamSynchronize(ctx->stream);
  gemm_scratch_release(ctx);
  for (auto& ev : ctx->events)
    if (ev) hipEventDestroy(ev);
  if (ctx->flags) hipFree(ctx->flags);
  if (ctx->host_flags) hipHostFree(ctx->host_flags);
  if (ctx->ws) hipFree(ctx->ws);
  for (int* w : ctx->ws_retired) hipFree(w);
  if (ctx->stream) {
    record_drop(ctx->stream);
    hipStreamDestroy(ctx->stream);
  }
  delete ctx;
  return ANVIL_OK;
}

int anvil_sync(anvil_ctx* ctx) {
  if (int r = check_ctx(ctx)) return r;
  FetchArgs a{};
  a.flags = ctx->flags, a.host_flags = ctx->host_flags;
  fetch_kernel<<<1, 256, 0, ctx->stream>>>(a);
  ANVIL_HIP(hipGetLastError());
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  return report_flags(ctx, false);
}

int anvil_fetch(anvil_ctx* ctx, int n, const void* const* src, void* const* dst, const size_t* bytes, int check) {
  if (n < 0 || (n > 0 && (!src || !dst || !bytes))) return set_error(ANVIL_E_VALUE, "anvil_fetch: null pointer");
  if (int r = check_ctx(ctx)) return r;
  for (int i = 0; i < n; ++i)
    if (!src[i] || !dst[i] || (uintptr_t)src[i] % 16 || (uintptr_t)dst[i] % 16)
      return set_error(ANVIL_E_VALUE, "anvil_fetch: buffer %d is null or not 16-byte aligned", i);
  FetchArgs a{};
  size_t total = 0;
  auto launch = [&]() {
    const unsigned grid = (unsigned)std::min<size_t>(256, std::max<size_t>(1, (total + 4095) / 4096));
    fetch_kernel<<<grid, 256, 0, ctx->stream>>>(a);
    a = FetchArgs{};
    total = 0;
    return hipGetLastError();
  };
  for (int i = 0; i < n; ++i) {
    if (bytes[i] > FETCH_KERNEL_MAX) {
      ANVIL_HIP(hipMemcpyAsync(dst[i], src[i], bytes[i], hipMemcpyDeviceToHost, ctx->stream));
      continue;
    }
    a.src[a.n] = (const int8_t*)src[i], a.dst[a.n] = (int8_t*)dst[i], a.bytes[a.n] = (long long)bytes[i];
    total += bytes[i];
    if (++a.n == FETCH_MAX) ANVIL_HIP(launch());
  }
  if (check) a.flags = ctx->flags, a.host_flags = ctx->host_flags;
  if (a.n || check) ANVIL_HIP(launch());
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  return check ? report_flags(ctx, true) : ANVIL_OK;
}

int anvil_alloc(anvil_ctx* ctx, size_t bytes, void** dptr) {
  if (int r = check_ctx(ctx)) return r;
  if (!dptr) return set_error(ANVIL_E_VALUE, "anvil_alloc: null output pointer");
  *dptr = nullptr;
  ANVIL_HIP(hipMalloc(dptr, bytes ? bytes : 1));
  return ANVIL_OK;
}

int anvil_free(anvil_ctx* ctx, void* dptr) {
  if (int r = check_ctx(ctx)) return r;
  if (!dptr) return ANVIL_OK;
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  ANVIL_HIP(hipFree(dptr));
  return ANVIL_OK;
}

int anvil_host_alloc(anvil_ctx* ctx, size_t bytes, void** hptr) {
  if (int r = check_ctx(ctx)) return r;
  if (!hptr) return set_error(ANVIL_E_VALUE, "anvil_host_alloc: null output pointer");
  *hptr = nullptr;
  ANVIL_HIP(hipHostMalloc(hptr, bytes ? bytes : 1, hipHostMallocDefault));
  return ANVIL_OK;
}

int anvil_host_free(anvil_ctx* ctx, void* hptr) {
  if (int r = check_ctx(ctx)) return r;
  if (!hptr) return ANVIL_OK;
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  ANVIL_HIP(hipHostFree(hptr));
  return ANVIL_OK;
}

int anvil_upload(anvil_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (int r = check_ctx(ctx)) return r;
  if (!bytes) return ANVIL_OK;
  if (!dst || !src) return set_error(ANVIL_E_VALUE, "anvil_upload: null pointer");
  ANVIL_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  return ANVIL_OK;
}

int anvil_download(anvil_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (int r = check_ctx(ctx)) return r;
  if (!bytes) return ANVIL_OK;
  if (!dst || !src) return set_error(ANVIL_E_VALUE, "anvil_download: null pointer");
  ANVIL_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  return ANVIL_OK;
}

int anvil_zero(anvil_ctx* ctx, void* dst, size_t bytes) {
  if (int r = check_ctx(ctx)) return r;
  if (!bytes) return ANVIL_OK;
  if (!dst) return set_error(ANVIL_E_VALUE, "anvil_zero: null pointer");
  return zero_fill(ctx->stream, dst, bytes);
}

int anvil_graph_begin(anvil_ctx* ctx) {
  if (int r = check_ctx(ctx)) return r;
  ANVIL_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeRelaxed));
  (void)record_start(ctx->stream, true);                 // without a list the capture keeps its executable form
  return ANVIL_OK;
}

int anvil_graph_end(anvil_ctx* ctx, void** graph) {
  if (int r = check_ctx(ctx)) return r;
  LaunchList* l = record_stop(ctx->stream, true);
  if (!graph) {
    delete l;
    return set_error(ANVIL_E_VALUE, "anvil_graph_end: null output pointer");
  }
  *graph = nullptr;
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(ctx->stream, &g);   // ends the capture whatever happened inside it
  if (e != hipSuccess) {
    delete l;
    return hip_fail(e, "hipStreamEndCapture(ctx->stream, &g)");
  }
  // Where the captured nodes are the noted launches of the thread that began, one after another on one stream, they are
  // replayed as launches from the list. hipGraphLaunch of the same kernels costs more on both sides: 28 us of host time for one
  // node to 43 us for twelve, and about 0.7 us more a node on the device (measured: a 768-wide block on one sequence,
  // 7 nodes, 61.4 us a forward through hipGraphLaunch, 55 us as launches; the 128-wide two-layer model, 12 nodes,
  // 96.5 against 89.7 us). A graph that holds anything else keeps its executable form.
  size_t nodes = 0;
  e = hipGraphGetNodes(g, nullptr, &nodes);
  if (!l) l = new (std::nothrow) LaunchList();
  if (!l) {
    hipGraphDestroy(g);
    return set_error(ANVIL_E_RUNTIME, "anvil_graph_end: out of memory");
  }
  if (e != hipSuccess || nodes != l->launches.size() || l->incomplete) {
    l->launches.clear();
    e = hipGraphInstantiate(&l->exec, g, nullptr, nullptr, 0);
  }
  hipGraphDestroy(g);
  if (e != hipSuccess) {
    delete l;
    return hip_fail(e, "hipGraphInstantiate");
  }
  *graph = l;
  return ANVIL_OK;
}

int anvil_record_begin(anvil_ctx* ctx) {
  if (int r = check_ctx(ctx)) return r;
  if (!record_start(ctx->stream, false)) return set_error(ANVIL_E_RUNTIME, "anvil_record_begin: out of memory");
  return ANVIL_OK;
}

int anvil_record_end(anvil_ctx* ctx, void** list) {
  if (int r = check_ctx(ctx)) return r;
  LaunchList* l = record_stop(ctx->stream, false);
  if (!list) {
    delete l;
    return set_error(ANVIL_E_VALUE, "anvil_record_end: null output pointer");
  }
  *list = nullptr;
  if (!l) return set_error(ANVIL_E_VALUE, "anvil_record_end: nothing is being recorded on this thread");
  if (l->incomplete) {
    delete l;
    return set_error(ANVIL_E_RUNTIME, "anvil_record_end: a launch could not be recorded");
  }
  *list = l;
  return ANVIL_OK;
}

int anvil_graph_launch(anvil_ctx* ctx, void* graph) {
  if (int r = check_ctx(ctx)) return r;
  if (!graph) return set_error(ANVIL_E_VALUE, "anvil_graph_launch: null graph");
  LaunchList* l = (LaunchList*)graph;
  if (l->exec) {
    ANVIL_HIP(hipGraphLaunch(l->exec, ctx->stream));
    return ANVIL_OK;
  }
  const bool plain = !g_recording.load(std::memory_order_relaxed) && !(g_timer.stop && g_timer.stream == ctx->stream);
  for (LaunchRecord& r : l->launches) {
    if (plain) {
      ANVIL_HIP(hipModuleLaunchKernel(r.fn, r.grid.x, r.grid.y, r.grid.z, r.block.x, r.block.y, r.block.z, r.lds,
                                      ctx->stream, r.ptrs.data(), nullptr));
    } else if (int e = launch_kernel(r.sym, r.grid, r.block, r.lds, ctx->stream, r.ptrs.data(), r.sizes.data(),
                                     (int)r.sizes.size())) {
      return e;
    }
  }
  return ANVIL_OK;
}

int anvil_graph_destroy(anvil_ctx* ctx, void* graph) {
  if (int r = check_ctx(ctx)) return r;
  if (!graph) return ANVIL_OK;
  LaunchList* l = (LaunchList*)graph;
  hipError_t e = hipSuccess;
  if (l->exec) {
    e = hipStreamSynchronize(ctx->stream);
    if (e == hipSuccess) e = hipGraphExecDestroy(l->exec);
  }
  delete l;
  return e == hipSuccess ? ANVIL_OK : hip_fail(e, "hipGraphExecDestroy");
}

// The context's events only time work (anvil_event_elapsed, anvil_time_kernels); nothing reads device memory through
// them, so they are created without the system-scope release / acquire fence: recording one then costs no L2
// writeback and invalidation, which would also slow the next kernel.
static int ensure_event(anvil_ctx* ctx, int slot) {
  if (!ctx->events[slot]) ANVIL_HIP(hipEventCreateWithFlags(&ctx->events[slot], hipEventDisableSystemFence));
  return ANVIL_OK;
}

int anvil_event_record(anvil_ctx* ctx, int slot) {
  if (slot < 0 || slot >= EVENT_SLOTS)
    return set_error(ANVIL_E_VALUE, "event slot %d outside [0, %d)", slot, EVENT_SLOTS);
  if (int r = check_ctx(ctx)) return r;
  if (int r = ensure_event(ctx, slot)) return r;
  ANVIL_HIP(hipEventRecord(ctx->events[slot], ctx->stream));
  return ANVIL_OK;
}

int anvil_time_kernels(anvil_ctx* ctx, int slot0, int slot1) {
  if (int r = check_ctx(ctx)) return r;
  if (slot0 < 0 && slot1 < 0) {
    if (g_timer.stream == ctx->stream) g_timer = KernelTimer{};
    return ANVIL_OK;
  }
  if (slot0 < 0 || slot0 >= EVENT_SLOTS || slot1 < 0 || slot1 >= EVENT_SLOTS || slot0 == slot1)
    return set_error(ANVIL_E_VALUE, "anvil_time_kernels: slots %d, %d must be two distinct slots in [0, %d)", slot0,
                     slot1, EVENT_SLOTS);
  for (int s : {slot0, slot1})
    if (int r = ensure_event(ctx, s)) return r;
  g_timer = KernelTimer{ctx->stream, ctx->events[slot0], ctx->events[slot1]};
  return ANVIL_OK;
}

int anvil_event_elapsed(anvil_ctx* ctx, int slot0, int slot1, float* ms) {
  if (slot0 < 0 || slot0 >= EVENT_SLOTS || slot1 < 0 || slot1 >= EVENT_SLOTS || !ms)
    return set_error(ANVIL_E_VALUE, "anvil_event_elapsed: bad slot or null output");
  if (int r = check_ctx(ctx)) return r;
  if (!ctx->events[slot0] || !ctx->events[slot1])
    return set_error(ANVIL_E_VALUE, "anvil_event_elapsed: slot never recorded");
  ANVIL_HIP(hipEventSynchronize(ctx->events[slot1]));
  ANVIL_HIP(hipEventElapsedTime(ms, ctx->events[slot0], ctx->events[slot1]));
  return ANVIL_OK;
}

}  // extern "C"
