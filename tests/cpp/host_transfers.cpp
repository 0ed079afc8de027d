// The host side of the library without a GPU: this program defines the runtime functions that the
// library calls (an executable's definitions come before a shared library's), so that what
// the stream does can be put off as long as a real one may put it off, and can be made to fail.
//
// The stream executes what is queued on it when somebody waits for it, or piece by piece while
// an event is polled.  Kernels are known by name; those that a check does not look at do nothing.
#include <hip/hip_runtime_api.h>
#include <malloc.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "coalsack_moe.h"

namespace fake {
std::recursive_mutex m;
// (used by the library's own initialisation, before this program's)
std::map<const void*, std::string>& kernels() {  // host stub -> device name
  static std::map<const void*, std::string> k;
  return k;
}
std::map<const void*, std::vector<char>>& vars() {
  static std::map<const void*, std::vector<char>> v;
  return v;
}
std::map<void*, size_t> device;              // live allocations
size_t device_bytes = 0;
std::deque<std::function<void()>> queue;     // the library's stream
std::deque<std::function<void()>> null_queue;  // the null stream, which nothing orders against it
long executed = 0, queued = 0;               // of the library's stream
int fail_launch_in = -1;                     // launches until one fails
hipError_t last = hipSuccess;
long launches = 0;
std::vector<std::string> launched;           // names since the last clear()
bool refuse_pinned = false;
bool fail_wait = false;                      // waiting for the stream reports an error
double stream_busy_until = 0.0;              // by the process's wall clock: the stream does nothing before
unsigned char* packed_scales = nullptr;      // scale plane that the last pack kernel wrote
std::map<const void*, std::vector<char>> packed;  // by plane: the blocks that were staged when its pack kernel ran
dim3 grid, block;
size_t shmem;
hipStream_t st;

std::function<void()> before_kernel;         // called once, when the next add_kernel is queued
double now() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }
void run(std::deque<std::function<void()>>& q, size_t n) {
  for (; n && !q.empty(); --n) {
    auto f = q.front();
    q.pop_front();
    f();
    if (&q == &queue) ++executed;
  }
}
void wait_for_stream() {
  while (now() < stream_busy_until) std::this_thread::sleep_for(std::chrono::milliseconds(1));
}
void run_all() {
  wait_for_stream();
  run(queue, (size_t)-1);
}
void put(std::function<void()> f) {
  queue.push_back(std::move(f));
  ++queued;
}
struct Event {
  long at = 0;
};

hipError_t launch(const void* f, void** args) {
  std::lock_guard<std::recursive_mutex> g(m);
  ++launches;
  if (fail_launch_in >= 0 && fail_launch_in-- == 0) return last = hipErrorLaunchFailure;
  const std::string& name = kernels()[f];
  launched.push_back(name);
  auto is = [&](const char* s) { return name.find(s) != std::string::npos; };
  if (is("link_copy_kernel")) {
    auto src = *(const char**)args[0];
    auto dst = *(char**)args[1];
    auto n = *(size_t*)args[2];
    put([=] { std::memmove(dst, src, n); });
  } else if (is("fill_cells_kernel")) {
    auto p = *(unsigned long long**)args[0];
    auto n = *(int*)args[1];
    auto v = *(unsigned long long*)args[2];
    put([=] {
      for (int i = 0; i < n; ++i) p[i] = v;
    });
  } else if (is("fill_words_kernel")) {
    auto p = *(uint32_t**)args[0];
    auto n = *(long*)args[1];
    auto v = *(uint32_t*)args[2];
    put([=] {
      for (long i = 0; i < 4 * n; ++i) p[i] = v;
    });
  } else if (is("pack_mxfp4_kernel")) {
    auto src = *(const char**)args[0];
    auto q = *(const void**)args[1];
    auto s = *(unsigned char**)args[2];
    const size_t n = (size_t)*(int*)args[3] * *(int*)args[4] * 17;
    packed_scales = s;
    put([=] {
      packed[q].assign(src, src + n);
      std::memset(s, 0x55, 256);
    });
  } else if (is("export_mxfp4_kernel")) {
    auto q = *(const void**)args[0];
    auto dst = *(char**)args[2];
    put([=] { std::memcpy(dst, packed[q].data(), packed[q].size()); });
  } else if (is("10add_kernel")) {
    auto a = *(const float**)args[0];
    auto b = *(const float**)args[1];
    auto o = *(float**)args[2];
    auto n = *(long*)args[3];
    if (before_kernel) run_all(), before_kernel(), before_kernel = nullptr;
    put([=] {
      for (long i = 0; i < n; ++i) o[i] = a[i] + b[i];
    });
  } else {
    put([] {});
  }
  return hipSuccess;
}
}  // namespace fake

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  fake::kernels()[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { fake::vars()[var].resize(size); }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t t) {
  fake::grid = g, fake::block = b, fake::shmem = s, fake::st = t;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* t) {
  *g = fake::grid, *b = fake::block, *s = fake::shmem, *t = fake::st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) { return fake::launch(f, args); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
  return fake::launch(f, args);
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  const hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "(stated by the test)"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *t = (size_t)288 << 30;
  *f = *t - fake::device_bytes;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = fake::vars()[s].data();
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)8;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  fake::run_all();
  return fake::fail_wait ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  *p = std::calloc(n, 1);
  fake::device[*p] = n;
  fake::device_bytes += n;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {  // waits for the device, as the real one does
  std::lock_guard<std::recursive_mutex> g(fake::m);
  fake::run_all();
  fake::run(fake::null_queue, (size_t)-1);
  fake::device_bytes -= fake::device[p];
  fake::device.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (fake::refuse_pinned) return fake::last = hipErrorOutOfMemory;
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipMemset(void* p, int v, size_t n) {  // on the null stream; device memory: not awaited
  std::lock_guard<std::recursive_mutex> g(fake::m);
  fake::null_queue.push_back([=] { std::memset(p, v, n); });
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  fake::run(fake::null_queue, (size_t)-1);
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  fake::put([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t) new fake::Event;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  ((fake::Event*)e)->at = fake::queued;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  const long at = ((fake::Event*)e)->at;
  if (fake::executed < at && fake::now() >= fake::stream_busy_until && std::rand() % 4 == 0) fake::run(fake::queue, 1);
  return fake::executed >= at ? hipSuccess : (fake::last = hipErrorNotReady);
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::recursive_mutex> g(fake::m);
  const long at = ((fake::Event*)e)->at;
  if (fake::executed < at) fake::wait_for_stream();
  while (fake::executed < at) fake::run(fake::queue, 1);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}
}  // extern "C"

#define CHECK(cond)                                                                        \
  do {                                                                                     \
    if (!(cond)) {                                                                         \
      std::printf("line %d: %s (last error: %s)\n", __LINE__, #cond, csk_last_error());    \
      return 1;                                                                            \
    }                                                                                      \
  } while (0)
#define OK(call) CHECK((call) == CSK_OK)

// A call fails between two results on their way down; the layer they were meant for goes away
// and the next call ends.  (Vectors above 64 KiB are mappings of their own here: one that is
// gone cannot be written without notice.)
static int results_of_a_failed_call() {
  mallopt(M_MMAP_THRESHOLD, 64 << 10);
  const int64_t E = 2, k = 2, H = 2880, F = 32, T = 8;
  std::vector<float> gate(E * H), hidden(T * H, 1.f), out(T * H), pairs(T * k * 2), norm(H);
  std::vector<uint8_t> bytes(F * H / 32 * 17, 1);
  csk_mxfp4 *u, *g, *d;
  OK(csk_mxfp4_upload(bytes.data(), F, H, &u));
  OK(csk_mxfp4_upload(bytes.data(), F, H, &g));
  OK(csk_mxfp4_upload(bytes.data(), H, F, &d));
  csk_layer *L, *other;
  OK(csk_layer_create_view(E, k, H, F, &L));
  OK(csk_layer_create_view(E, k, H, F, &other));
  OK(csk_layer_set_router(L, gate.data(), nullptr));
  for (int e = 0; e < E; ++e) OK(csk_layer_attach_expert(L, e, u, g, d, nullptr, nullptr, nullptr));
  int running = 0;
  OK(csk_moe_frame_begin(L, hidden.data(), T, pairs.data(), 0, &running));
  CHECK(running);
  fake::fail_launch_in = 1;  // the rows' copy is queued, that of their positions is refused
  CHECK(csk_moe_frame_expert_rows(L, 0, out.data()) == CSK_ERR_HIP);
  fake::fail_launch_in = -1;
  csk_layer_destroy(L);
  OK(csk_layer_set_norm(other, norm.data(), 1e-5f));
  return 0;
}

// A call fails with a copy into the pinned area still queued; the next call's values pass
// through the same place.
static int pinned_area_after_a_failed_call() {
  const int64_t T = 8, H = 256, E = 16, k = 4, n = 60000;
  std::vector<double> hidden(T * H, 1.0), gate(E * H, 1.0), logits(T * E);
  std::vector<float> pairs(T * k * 2), a(n), b(n), out(n);
  fake::fail_launch_in = 5;  // gate, hidden, logits, selection, pairs down, logits down
  CHECK(csk_moe_router_f64(hidden.data(), T, H, gate.data(), E, nullptr, k, 0, pairs.data(), logits.data()) == CSK_ERR_HIP);
  CHECK(fake::fail_launch_in == -1);
  for (int64_t i = 0; i < n; ++i) a[i] = (float)i, b[i] = 0.5f;
  OK(csk_add(a.data(), b.data(), out.data(), n));
  for (int64_t i = 0; i < n; ++i) CHECK(out[i] == a[i] + b[i]);
  return 0;
}

// Pageable memory is enough for every call where the machine gives no pinned memory.
static int no_pinned_memory() {
  fake::refuse_pinned = true;
  for (int64_t n : {100, 300000}) {
    std::vector<float> a(n), b(n), out(n);
    for (int64_t i = 0; i < n; ++i) a[i] = (float)i, b[i] = 0.5f;
    OK(csk_add(a.data(), b.data(), out.data(), n));
    for (int64_t i = 0; i < n; ++i) CHECK(out[i] == a[i] + b[i]);
  }
  return 0;
}

// Processor time of the whole process while the stream is at work for half a second in front of a
// result, and in front of the room that an upload waits for: the threads sleep, the caller too.
static int threads_sleep_while_the_stream_works() {
  const int64_t n = 6000000;  // 24 MB: larger than the ring
  std::vector<float> a(n, 1.f), b(n, 2.f), out(n);
  OK(csk_add(a.data(), b.data(), out.data(), n));
  for (int part = 0; part < 2; ++part) {
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    const double t0 = fake::now();
    const std::clock_t c0 = std::clock();
    if (part == 0) {
      fake::stream_busy_until = t0 + 0.5;  // the uploads find the ring full
      OK(csk_add(a.data(), b.data(), out.data(), n));
    } else {
      fake::before_kernel = [] { fake::stream_busy_until = fake::now() + 0.5; };  // the result comes late
      OK(csk_add(a.data(), b.data(), out.data(), n));
    }
    const double wall = fake::now() - t0, cpu = double(std::clock() - c0) / CLOCKS_PER_SEC;
    std::printf("part %d: %.3f s wall, %.3f s of processor time\n", part, wall, cpu);
    CHECK(wall >= 0.5);
    CHECK(cpu < 0.25);
    CHECK(out[0] == 3.f && out[n - 1] == 3.f);
  }
  return 0;
}

// What an upload stages on the device is given back if it is large: an output head of 300 MB
// must not cost that much memory for good.
static int staging_memory_after_a_large_upload() {
  const int64_t rows = 65536, K = 2304;
  const size_t before = fake::device_bytes;
  std::vector<uint16_t> w((size_t)rows * K);
  csk_f16* m;
  OK(csk_f16_upload(w.data(), rows, K, &m));
  CHECK(fake::device_bytes >= before + w.size() * 2);
  csk_f16_free(m);
  CHECK(fake::device_bytes <= before + ((size_t)256 << 20));
  // an expert's matrices, on the other hand, find it there the second time
  std::vector<uint8_t> bytes(2880 * 90 * 17, 1);
  csk_mxfp4* q;
  OK(csk_mxfp4_upload(bytes.data(), 2880, 2880, &q));
  csk_mxfp4_free(q);
  uint64_t count0 = 0, count1 = 0;
  OK(csk_alloc_count(&count0));
  OK(csk_mxfp4_upload(bytes.data(), 2880, 2880, &q));
  OK(csk_alloc_count(&count1));
  CHECK(count1 - count0 == 2);  // the two planes
  return 0;
}

// The kernels that a batch takes.  Where an expert cannot hold more tokens than one pass of the streaming
// kernel contracts, no weight is streamed twice, however large the matrices.
static int kernels_of_a_batch() {
  struct Call {
    int64_t E, k, H, F, T;
    bool stream;
  };
  const Call calls[] = {
      {8, 8, 4096, 8192, 1, true},    {16, 8, 6144, 8192, 1, true},  {8, 8, 4096, 6144, 4, true},
      {1, 1, 8192, 8192, 4, true},    {8, 8, 4096, 6144, 5, false},  {8, 4, 4096, 6144, 8, false},
      {4, 4, 2880, 1536, 33, true},   {4, 4, 2880, 1536, 37, false}, {32, 4, 2880, 2880, 16, true},
      {128, 4, 2880, 2880, 64, true}, {32, 4, 2880, 2880, 64, false}, {8, 2, 8224, 64, 1, false},
      // (what the GPU tests of these shapes say they run)
      {4, 2, 8224, 64, 3, false},     {4, 2, 64, 8224, 64, false},    {4, 2, 3200, 64, 6, true},
      {32, 4, 2880, 2880, 32, true},  {32, 4, 2880, 2880, 48, true},  {128, 4, 2880, 2880, 128, true},
      {128, 4, 2880, 2880, 160, false},
  };
  for (const Call& c : calls) {
    csk_layer* L;
    OK(csk_layer_create(c.E, c.k, c.H, c.F, &L));
    std::vector<float> gate(c.E * c.H), hidden(c.T * c.H), out(c.T * c.H);
    OK(csk_layer_set_router(L, gate.data(), nullptr));
    OK(csk_layer_fill_synthetic(L, 1, 0, 117, 5));
    fake::launched.clear();
    OK(csk_moe_forward(L, hidden.data(), c.T, out.data(), 0));
    auto count = [](const char* s) {
      int n = 0;
      for (const std::string& name : fake::launched) n += name.find(s) != std::string::npos;
      return n;
    };
    if (count("expert_stream_kernel") != (c.stream ? 2 : 0) || count("expert_gemm_mx_kernel") != (c.stream ? 0 : 2)) {
      std::printf("E %ld k %ld H %ld F %ld T %ld: not the kernels expected\n", c.E, c.k, c.H, c.F, c.T);
      return 1;
    }
    // a single token on the streaming kernels is routed by the first of them
    if (c.T == 1) CHECK((count("route_") + count("dispatch_") == 0) == (c.stream && c.E > 1));
    csk_layer_destroy(L);
  }
  return 0;
}

// Token groups of four in passes, or tiles of up to 64 tokens.
static int groups_of_a_batch() {
  struct Call {
    int64_t E, k, H, F, T;
    int wbf;
    bool tiles;
  };
  const Call calls[] = {
      {8, 4, 2880, 2880, 4, 0, false},    {8, 4, 2880, 2880, 8, 0, true},    {32, 4, 2880, 2880, 16, 0, false},
      {32, 4, 2880, 2880, 24, 0, true},   {128, 4, 2880, 2880, 16, 0, false}, {128, 4, 2880, 2880, 20, 0, false},
      {128, 4, 2880, 2880, 64, 0, true},  {64, 8, 2048, 768, 50, 0, true},   {1, 1, 2880, 2880, 8, 0, false},
      {1, 1, 2880, 2880, 17, 0, true},    {16, 2, 3328, 544, 19, 1, false},  {16, 2, 3328, 544, 19, 0, true},
      {4, 4, 2880, 1536, 33, 1, true},
  };
  for (const Call& c : calls) {
    csk_layer* L;
    OK(csk_layer_create(c.E, c.k, c.H, c.F, &L));
    std::vector<float> gate(c.E * c.H), hidden(c.T * c.H), out(c.T * c.H);
    OK(csk_layer_set_router(L, gate.data(), nullptr));
    OK(csk_layer_set_options(L, 0, CSK_ACT_MODIFIED_SWIGLU, c.wbf));
    OK(csk_layer_fill_synthetic(L, 1, 0, 117, 5));
    fake::launched.clear();
    OK(csk_moe_forward(L, hidden.data(), c.T, out.data(), 0));
    int tiles = 0, all = 0;
    for (const std::string& name : fake::launched) {
      tiles += name.find("expert_stream_kernel_tiles") != std::string::npos;
      all += name.find("expert_stream_kernel") != std::string::npos;
    }
    if (all != 2 || tiles != (c.tiles ? 2 : 0)) {
      std::printf("E %ld k %ld H %ld F %ld T %ld: not the kernels expected\n", c.E, c.k, c.H, c.F, c.T);
      return 1;
    }
    csk_layer_destroy(L);
  }
  return 0;
}

// The pinned ring (16 MiB, quarters of 4, pieces of 64 KiB) entered at many offsets and gone round
// several times within a call, on a stream that reads and writes it as late as it may.
static int ring_entered_anywhere() {
  uint32_t x = 1;
  auto random = [&x] { return (x = x * 1664525u + 1013904223u) >> 8; };
  for (int round = 0; round < 6; ++round) {
    const int64_t H = 32 * (8 + random() % 120), F = 32 * (8 + random() % 200);
    csk_layer* L;
    OK(csk_layer_create(1, 1, H, F, &L));
    std::vector<uint8_t> w[3];
    for (auto& m : w) {
      m.resize(H * F / 32 * 17);
      for (auto& b : m) b = (uint8_t)random();
    }
    fake::packed.clear();
    OK(csk_layer_set_expert(L, 0, w[0].data(), w[1].data(), w[2].data(), nullptr, nullptr, nullptr));
    const int which[3] = {CSK_W_UP, CSK_W_GATE, CSK_W_DOWN};
    for (int i = 0; i < 3; ++i) {
      std::vector<uint8_t> back(w[i].size());
      OK(csk_layer_export(L, 0, which[i], back.data()));
      CHECK(back == w[i]);
    }
    csk_layer_destroy(L);
  }
  return 0;
}

// An expert whose matrices did not arrive is not there, whichever format they have.
static int expert_that_did_not_arrive() {
  const int64_t H = 64, F = 64;
  std::vector<uint16_t> halves(H * F);
  std::vector<uint8_t> blocks(H * F / 32 * 17, 1);
  std::vector<float> gate(H), x(H), y(H);
  for (int f16 = 0; f16 < 3; ++f16) {
    csk_layer* L;
    OK(f16 ? csk_layer_create_f16(1, 1, H, F, &L) : csk_layer_create(1, 1, H, F, &L));
    OK(csk_layer_set_router(L, gate.data(), nullptr));
    auto set = [&] {
      if (f16 == 2) {  // matrix by matrix
        for (int which = 0; which < 3; ++which)
          if (const int rc = csk_layer_set_expert_matrix(L, 0, which, 1, halves.data()); rc != CSK_OK) return rc;
        return CSK_OK;
      }
      return f16 ? csk_layer_set_expert_f16(L, 0, halves.data(), halves.data(), halves.data(), nullptr, nullptr, nullptr)
                 : csk_layer_set_expert(L, 0, blocks.data(), blocks.data(), blocks.data(), nullptr, nullptr, nullptr);
    };
    for (int first = 1; first >= 0; --first) {  // an expert that had none, and one that loses its old ones
      fake::fail_wait = true;
      CHECK(set() == CSK_ERR_HIP);
      fake::fail_wait = false;
      CHECK(csk_moe_forward(L, x.data(), 1, y.data(), 0) == CSK_ERR_STATE);
      OK(set());
      OK(csk_moe_forward(L, x.data(), 1, y.data(), 0));
    }
    csk_layer_destroy(L);
  }
  return 0;
}

// Nothing orders the null stream against the library's: what is written there may land late.
static int scales_of_an_uploaded_matrix() {
  std::vector<uint8_t> bytes(16 * 17, 1);
  csk_mxfp4* m;
  OK(csk_mxfp4_upload(bytes.data(), 16, 32, &m));
  fake::run(fake::null_queue, (size_t)-1);
  for (int i = 0; i < 256; ++i) CHECK(fake::packed_scales[i] == 0x55);
  // padding (this plane has 2 KiB) holds the scale of 1
  for (int i = 256; i < 2048; ++i) CHECK(fake::packed_scales[i] == 127);
  return 0;
}

// The expert kernels of one batch, by name: a layer's (layer E k H F T weight_before_ffn), or a single expert's (expert k H F T
// weight_before_ffn, expert_f16 the same, expert_eighth where every eighth token takes the expert).
static int names_of_a_batch(const std::string& what, const std::vector<int64_t>& v) {
  const bool layer = what == "layer", f16 = what == "expert_f16";
  const int64_t E = layer ? v[0] : 1, k = v[layer], H = v[layer + 1], F = v[layer + 2], T = v[layer + 3];
  const int wbf = (int)v[layer + 4];
  std::vector<float> hidden(T * H), out(T * H);
  if (layer) {
    csk_layer* L;
    std::vector<float> gate(E * H);
    OK(csk_layer_create(E, k, H, F, &L));
    OK(csk_layer_set_router(L, gate.data(), nullptr));
    OK(csk_layer_set_options(L, 0, CSK_ACT_MODIFIED_SWIGLU, wbf));
    OK(csk_layer_fill_synthetic(L, 1, 0, 117, 5));
    fake::launched.clear();
    OK(csk_moe_forward(L, hidden.data(), T, out.data(), 0));
    csk_layer_destroy(L);
  } else {
    std::vector<float> pairs(T * k * 2);
    for (int64_t i = 0; i < T * k; ++i) pairs[2 * i] = what == "expert_eighth" && i / k % 8 ? 1.0f : 0.0f;
    int empty = 0;
    if (f16) {
      std::vector<uint16_t> w(H * F);
      csk_f16 *u, *g, *d;
      OK(csk_f16_upload(w.data(), F, H, &u));
      OK(csk_f16_upload(w.data(), F, H, &g));
      OK(csk_f16_upload(w.data(), H, F, &d));
      fake::launched.clear();
      OK(csk_expert_mlp_f16(0, hidden.data(), T, H, F, u, g, d, nullptr, nullptr, nullptr, pairs.data(), k, 0, wbf, out.data(), &empty));
    } else {
      std::vector<uint8_t> w(H * F / 32 * 17, 1);
      csk_mxfp4 *u, *g, *d;
      OK(csk_mxfp4_upload(w.data(), F, H, &u));
      OK(csk_mxfp4_upload(w.data(), F, H, &g));
      OK(csk_mxfp4_upload(w.data(), H, F, &d));
      fake::launched.clear();
      OK(csk_expert_mlp_mxfp4(0, hidden.data(), T, H, F, u, g, d, nullptr, nullptr, nullptr, pairs.data(), k, 0, wbf, out.data(), &empty));
    }
  }
  for (const std::string& name : fake::launched)
    for (const char* kernel : {"expert_stream_kernel_tiles", "expert_stream_kernel", "expert_gemm_mx_kernel", "expert_f16_gemm_kernel", "expert_f16_kernel"})
      if (name.find(kernel) != std::string::npos) {
        std::printf("%s\n", kernel);
        break;
      }
  return 0;
}

int main(int argc, char** argv) {
  if (argc > 2) {
    std::vector<int64_t> v;
    for (int i = 2; i < argc; ++i) v.push_back(std::atoll(argv[i]));
    const std::string what = argv[1];
    if (v.size() != (what == "layer" ? 6u : 5u) || csk_init(0) != CSK_OK) return 2;
    const int rc = names_of_a_batch(what, v);
    std::fflush(stdout);
    std::_Exit(rc);
  }
  const std::map<std::string, int (*)()> checks = {
      {"results_of_a_failed_call", results_of_a_failed_call},
      {"pinned_area_after_a_failed_call", pinned_area_after_a_failed_call},
      {"no_pinned_memory", no_pinned_memory},
      {"threads_sleep_while_the_stream_works", threads_sleep_while_the_stream_works},
      {"staging_memory_after_a_large_upload", staging_memory_after_a_large_upload},
      {"kernels_of_a_batch", kernels_of_a_batch},
      {"groups_of_a_batch", groups_of_a_batch},
      {"ring_entered_anywhere", ring_entered_anywhere},
      {"expert_that_did_not_arrive", expert_that_did_not_arrive},
      {"scales_of_an_uploaded_matrix", scales_of_an_uploaded_matrix},
  };
  if (argc != 2 || !checks.count(argv[1])) return 2;
  if (csk_init(0) != CSK_OK) {
    std::printf("csk_init: %s\n", csk_last_error());
    return 3;
  }
  const int rc = checks.at(argv[1])();
  std::printf("%s: %s\n", argv[1], rc ? "failed" : "ok");
  std::fflush(stdout);
  std::_Exit(rc);
}
