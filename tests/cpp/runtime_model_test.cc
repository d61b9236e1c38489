// The library's host side run against a model of the HIP runtime: this program
// defines the runtime's functions itself (they take precedence over those of
// libamdhip64), with "device" memory in host memory and one stream whose work
// is performed only when something waits for it. Kernels are not executed, but
// for the two that copy between host and device; every launch is logged by
// name. That shows in which order a call enqueues its work, what it does when a
// launch fails, what it asks for while its stream records a graph and which
// kernel it runs on, none of which a GPU is needed (or, for the failures,
// wanted) for.
//
//   runtime_model_test failed_upload | page_locked_sources | page_locked_destinations | skinny_shapes |
//       timing | capture | raw_rows | scratch_blocks | staged_rule | routes | kernels
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "kernels/host_copy.h"
#include "ruy_amd/c_api.h"

static int g_failures = 0;
#define EXPECT(cond, ...)                                                              \
  do {                                                                                 \
    if (!(cond)) {                                                                     \
      std::fprintf(stderr, "%s:%d: EXPECT failed: %s: ", __FILE__, __LINE__, #cond);   \
      std::fprintf(stderr, __VA_ARGS__);                                               \
      std::fprintf(stderr, "\n");                                                      \
      ++g_failures;                                                                    \
    }                                                                                  \
  } while (0)

namespace {

// Everything the model knows. (A function-local object: the library registers
// its kernels before this program's own static objects are constructed.)
struct Runtime {
  std::map<const void*, std::string> kernels;
  std::map<const char*, std::size_t> device, pinned;  // base -> size
  std::vector<std::function<void()>> queue;           // enqueued, not performed yet
  std::vector<std::string> log;                       // kernel names and "event"
  std::vector<std::vector<char>> uploads;             // what each upload that was performed brought
  std::string fail_kernel;                            // fail the fail_at-th launch of a kernel so named
  int fail_at = 0;
  hipError_t last_error = hipSuccess;
  bool capturing = false;
  bool captured_elsewhere = false;                    // by another thread, in the mode that binds all of them
  hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;  // of this thread
  int capture_violations = 0;
  int allocations = 0;                                // of device memory, refused ones too
  int frees = 0;
  std::size_t device_limit = ~std::size_t(0);         // bytes of device memory there are
  bool fill_allocations = true;
  dim3 grid, block;
  std::size_t shared = 0;
  hipStream_t stream = nullptr;
};
Runtime& R() {
  static Runtime* r = new Runtime;
  return *r;
}

void Drain() {
  std::vector<std::function<void()>> work;
  work.swap(R().queue);
  for (auto& f : work) f();
}

// What a stream that records a graph cannot take.
void NotWhileCapturing() {
  if (R().capturing) ++R().capture_violations;
}

const char* In(const std::map<const char*, std::size_t>& ranges, const void* p) {
  auto it = ranges.upper_bound(static_cast<const char*>(p));
  if (it == ranges.begin()) return nullptr;
  --it;
  return static_cast<const char*>(p) < it->first + it->second ? it->first : nullptr;
}

void Upload(void* to, const void* from, std::size_t bytes, std::size_t moved) {
  std::memcpy(to, from, moved);
  const char* c = static_cast<const char*>(from);
  R().uploads.emplace_back(c, c + bytes);
}

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* module = nullptr;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  R().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, std::size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, std::size_t shared, hipStream_t stream) {
  R().grid = grid;
  R().block = block;
  R().shared = shared;
  R().stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, std::size_t* shared, hipStream_t* stream) {
  *grid = R().grid;
  *block = R().block;
  *shared = R().shared;
  *stream = R().stream;
  return hipSuccess;
}

hipError_t hipLaunchKernel(const void* function, dim3, dim3, void** args, std::size_t, hipStream_t) {
  const std::string& name = R().kernels[function];
  if (!R().fail_kernel.empty() && name.find(R().fail_kernel) != std::string::npos && --R().fail_at == 0) {
    R().last_error = hipErrorLaunchOutOfResources;
    return R().last_error;
  }
  R().log.push_back(name);
  if (name.find("UploadKernel") != std::string::npos) {
    const ruyamd::UploadPieces pieces = *static_cast<const ruyamd::UploadPieces*>(args[0]);
    R().queue.push_back([pieces] {
      for (int i = 0; i < pieces.count; ++i) {
        EXPECT(reinterpret_cast<std::uintptr_t>(pieces.from[i]) % 16 == 0, "piece %d", i);
        Upload(pieces.to[i], pieces.from[i], pieces.bytes[i], (pieces.bytes[i] + 15) / 16 * 16);
      }
    });
  }
  if (name.find("DownloadKernel") != std::string::npos) {
    const void* from = *static_cast<const void**>(args[0]);
    void* to = *static_cast<void**>(args[1]);
    const uint32_t bytes = *static_cast<uint32_t*>(args[2]);
    uint32_t* done = *static_cast<uint32_t**>(args[3]);
    const uint32_t value = *static_cast<uint32_t*>(args[4]);
    R().queue.push_back([=] {
      std::memcpy(to, from, (bytes + 15) / 16 * 16);
      for (int b = 0; b < ruyamd::DownloadBlocks(bytes); ++b) done[b] = value;
    });
    Drain();  // (a GPU gets there by itself)
  }
  return hipSuccess;
}

// ... nor another thread meanwhile do.
static void NotWhileAnyoneCaptures() {
  NotWhileCapturing();
  if (R().captured_elsewhere && R().mode != hipStreamCaptureModeRelaxed) ++R().capture_violations;
}
static hipError_t Take(std::map<const char*, std::size_t>* ranges, void** p, std::size_t bytes) {
  *p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096 + 4096);
  if (R().fill_allocations) std::memset(*p, 0xCD, bytes);
  (*ranges)[static_cast<char*>(*p)] = bytes;
  NotWhileAnyoneCaptures();
  return hipSuccess;
}
static hipError_t Give(std::map<const char*, std::size_t>* ranges, void* p) {
  Drain();
  if (p) ranges->erase(static_cast<char*>(p));
  std::free(p);
  NotWhileAnyoneCaptures();
  return hipSuccess;
}
hipError_t hipMalloc(void** p, std::size_t bytes) {
  ++R().allocations;
  std::size_t held = bytes;
  for (const auto& range : R().device) held += range.second;
  if (held > R().device_limit) return R().last_error = hipErrorOutOfMemory;
  return Take(&R().device, p, bytes);
}
hipError_t hipFree(void* p) {
  ++R().frees;
  return Give(&R().device, p);
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* mode) {
  std::swap(*mode, R().mode);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, std::size_t bytes, unsigned) { return Take(&R().pinned, p, bytes); }
hipError_t hipHostFree(void* p) { return Give(&R().pinned, p); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof(*a));
  const bool device = In(R().device, p), host = In(R().pinned, p);
  if (!device && !host) return R().last_error = hipErrorInvalidValue;
  a->type = device ? hipMemoryTypeDevice : hipMemoryTypeHost;
  a->devicePointer = const_cast<void*>(p);
  if (host) a->hostPointer = const_cast<void*>(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, std::size_t bytes, hipMemcpyKind kind, hipStream_t) {
  NotWhileCapturing();
  R().queue.push_back([=] {
    if (kind == hipMemcpyHostToDevice)
      Upload(to, from, bytes, bytes);
    else
      std::memcpy(to, from, bytes);
  });
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, std::size_t bytes, hipMemcpyKind) {
  Drain();
  std::memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* to, std::size_t to_pitch, const void* from, std::size_t from_pitch, std::size_t width,
                            std::size_t height, hipMemcpyKind, hipStream_t) {
  NotWhileCapturing();
  R().queue.push_back([=] {
    for (std::size_t i = 0; i < height; ++i)
      std::memcpy(static_cast<char*>(to) + i * to_pitch, static_cast<const char*>(from) + i * from_pitch, width);
  });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int value, std::size_t bytes, hipStream_t) {
  NotWhileCapturing();
  R().queue.push_back([=] { std::memset(p, value, bytes); });
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  R().log.push_back("event");
  NotWhileCapturing();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) {
  Drain();
  NotWhileCapturing();
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "an error of the runtime model"; }
hipError_t hipGetLastError() {
  const hipError_t e = R().last_error;
  R().last_error = hipSuccess;
  return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* area = nullptr;
  if (!area) (void)Take(&R().device, &area, std::size_t(64) << 20);
  *p = area;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = R().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  Drain();
  NotWhileCapturing();
  return hipSuccess;
}

}  // extern "C"

namespace {

int SizeOf(int dtype) {
  switch (dtype) {
    case RUYAMD_DTYPE_U8:
    case RUYAMD_DTYPE_I8:
      return 1;
    case RUYAMD_DTYPE_I16:
      return 2;
    case RUYAMD_DTYPE_F64:
      return 8;
    default:
      return 4;
  }
}

ruyamd_mat Mat(int dtype, void* data, int rows, int cols, int order, int zero_point = 0,
               int cache = RUYAMD_CACHE_NEVER) {
  ruyamd_mat m = {};
  m.data = data;
  m.rows = rows;
  m.cols = cols;
  m.stride = order == RUYAMD_ORDER_COL_MAJOR ? rows : cols;
  m.zero_point = zero_point;
  m.order = static_cast<uint8_t>(order);
  m.dtype = static_cast<uint8_t>(dtype);
  m.cache_policy = static_cast<uint8_t>(cache);
  return m;
}

ruyamd_mul_params Params(int dst) {
  ruyamd_mul_params p = {};
  const bool fp = dst == RUYAMD_DTYPE_F32 || dst == RUYAMD_DTYPE_F64;
  p.accum_dtype = static_cast<uint8_t>(fp ? dst : RUYAMD_DTYPE_I32);
  p.clamp_min = fp ? -1e30 : -128;
  p.clamp_max = fp ? 1e30 : 127;
  p.multiplier_fixedpoint = fp ? 0 : 1 << 30;
  p.multiplier_exponent = fp ? 0 : -9;
  return p;
}

struct Context {
  ruyamd_ctx* ctx = nullptr;
  Context() {
    if (ruyamd_ctx_create(&ctx) != RUYAMD_OK) std::abort();
    R().log.clear();
    R().uploads.clear();
    R().capture_violations = 0;
  }
  ~Context() { ruyamd_ctx_destroy(ctx); }
};

int Count(const char* name) {
  return static_cast<int>(std::count_if(R().log.begin(), R().log.end(),
                                        [&](const std::string& s) { return s.find(name) != std::string::npos; }));
}

struct Types {
  const char* name;
  int lhs, rhs, dst;
};
const Types kTypes[] = {{"int8", RUYAMD_DTYPE_I8, RUYAMD_DTYPE_I8, RUYAMD_DTYPE_I8},
                        {"fp32", RUYAMD_DTYPE_F32, RUYAMD_DTYPE_F32, RUYAMD_DTYPE_F32},
                        {"int8 x int16", RUYAMD_DTYPE_I8, RUYAMD_DTYPE_I16, RUYAMD_DTYPE_I16},
                        {"generic", RUYAMD_DTYPE_F64, RUYAMD_DTYPE_F64, RUYAMD_DTYPE_F64}};

// A cached operand whose upload could not be launched leaves no entry: the next
// call uploads and packs it.
void FailedUpload() {
  const int M = 96, K = 160, N = 64;
  for (const Types& t : kTypes) {
    for (int fail_at = 1; fail_at <= 2; ++fail_at) {
      Context c;
      std::vector<char> lhs(M * K * 8, 1), rhs(K * N * 8, 2), dst(M * N * 8);
      const ruyamd_mat l = Mat(t.lhs, lhs.data(), M, K, RUYAMD_ORDER_ROW_MAJOR, 0, RUYAMD_CACHE_ALWAYS);
      const ruyamd_mat r = Mat(t.rhs, rhs.data(), K, N, RUYAMD_ORDER_COL_MAJOR, 0, RUYAMD_CACHE_ALWAYS);
      const ruyamd_mat d = Mat(t.dst, dst.data(), M, N, RUYAMD_ORDER_COL_MAJOR);
      const ruyamd_mul_params p = Params(t.dst);
      R().fail_kernel = "UploadKernel";
      R().fail_at = fail_at;
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) != RUYAMD_OK, "%s, upload %d", t.name, fail_at);
      R().fail_kernel.clear();
      // The operands go up one after the other: those before the failure are cached.
      EXPECT(ruyamd_ctx_cache_matrix_count(c.ctx) == fail_at - 1, "%s, upload %d: %d entries", t.name, fail_at,
             ruyamd_ctx_cache_matrix_count(c.ctx));
      R().uploads.clear();
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", t.name);
      EXPECT(static_cast<int>(R().uploads.size()) == 3 - fail_at, "%s, upload %d: %d operands uploaded by the next call",
             t.name, fail_at, static_cast<int>(R().uploads.size()));
      EXPECT(ruyamd_ctx_cache_matrix_count(c.ctx) == 2, "%s", t.name);
    }
  }
}

// Page-locked memory whose last bytes are those in front of a page that cannot
// be touched: `bytes` bytes that start `from_end` bytes before it.
struct PageLocked {
  char* base;
  char* data;
  std::size_t room;
  PageLocked(std::size_t bytes, std::size_t from_end) {
    room = (std::max(bytes, from_end) + 4095) / 4096 * 4096;
    base = static_cast<char*>(mmap(nullptr, room + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (base == MAP_FAILED || mprotect(base + room, 4096, PROT_NONE) != 0) std::abort();
    data = base + room - from_end;
    R().pinned[base] = room;
  }
  ~PageLocked() {
    R().pinned.erase(base);
    munmap(base, room + 4096);
  }
};

// A page-locked operand is read in stream order: what work enqueued in front of
// the call writes to it is what the call multiplies by. At any address and
// size, and nothing outside the 16 aligned bytes that hold a byte of it.
void PageLockedSources() {
  const int M = 70, N = 40;
  for (int K : {33, 48, 128, 20000}) {       // (the last: 1.4 MB and 0.8 MB, either side of the kernel copies' limit)
    for (int misalign : {0, 1, 4}) {
      Context c;
      const std::size_t sizes[4] = {std::size_t(M) * K, std::size_t(K) * N, std::size_t(M) * 4, std::size_t(M) * 4};
      std::vector<PageLocked*> operands;
      for (std::size_t size : sizes) {
        // As close to the end as the alignment allows.
        operands.push_back(new PageLocked(size, size + (16 - (size + misalign) % 16) % 16));
      }
      for (int i = 0; i < 4; ++i) std::memset(operands[i]->data, 0x11, sizes[i]);
      std::vector<char> mf(M * 4, 0x22), dst(M * N);  // (a pageable one among them)
      const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, operands[0]->data, M, K, RUYAMD_ORDER_ROW_MAJOR);
      const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, operands[1]->data, K, N, RUYAMD_ORDER_COL_MAJOR, 3);
      const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, dst.data(), M, N, RUYAMD_ORDER_COL_MAJOR);
      ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
      p.bias = operands[2]->data;
      p.multiplier_fixedpoint_perchannel = reinterpret_cast<const int32_t*>(mf.data());
      p.multiplier_exponent_perchannel = reinterpret_cast<const int32_t*>(operands[3]->data);
      R().queue.push_back([&] {  // work on the call's stream, in front of it
        for (int i = 0; i < 4; ++i) std::memset(operands[i]->data, 0x40 + i, sizes[i]);
      });
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
      for (int i = 0; i < 4; ++i) {
        const std::vector<char> want(sizes[i], static_cast<char>(0x40 + i));
        EXPECT(std::count(R().uploads.begin(), R().uploads.end(), want) == 1, "depth %d, %d bytes off: operand %d", K,
               misalign, i);
      }
      EXPECT(std::count(R().uploads.begin(), R().uploads.end(), mf) == 1, "pageable operand");
      for (PageLocked* o : operands) delete o;
    }
  }
}

// A page-locked destination comes back by a kernel and the CPU only while that
// is the shorter way, in one run or in many; either way all of it is there when
// the call returns, and nothing between its runs.
void PageLockedDestinations() {
  struct {
    int rows, cols, pad;
    bool locked, by_kernel;
  } const cases[] = {
      {1024, 384, 0, true, true},  {1024, 385, 0, true, false},  {1024, 128, 32, true, true},
      {1024, 129, 32, true, false}, {1024, 1024, 0, false, true}, {1024, 1024, 32, false, true},
      {1024, 1025, 0, false, false}, {3000, 1, 64, true, true},
  };
  for (const auto& k : cases) {
    Context c;
    const int K = 33, rows = k.rows - k.pad;
    std::vector<char> lhs(k.rows * K, 1), rhs(K * k.cols, 2), pageable(std::size_t(k.rows) * k.cols);
    PageLocked locked(pageable.size(), pageable.size());
    char* dst = k.locked ? locked.data : pageable.data();
    std::memset(dst, 0x5A, pageable.size());
    const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, lhs.data(), rows, K, RUYAMD_ORDER_ROW_MAJOR);
    const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, rhs.data(), K, k.cols, RUYAMD_ORDER_COL_MAJOR);
    ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, dst, rows, k.cols, RUYAMD_ORDER_COL_MAJOR);
    d.stride = k.rows;
    const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
    EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
    EXPECT(Count("DownloadKernel") == k.by_kernel, "%d x %d, %d between the runs", rows, k.cols, k.pad);
    // (No kernel has written the device's image of it: it is as memory is allocated here.)
    int wrong = 0;
    for (int j = 0; j < k.cols; ++j)
      for (int i = 0; i < k.rows; ++i)
        wrong += dst[std::size_t(j) * k.rows + i] != (i < rows ? static_cast<char>(0xCD) : 0x5A);
    EXPECT(wrong == 0, "%d x %d, %d between the runs: %d bytes", rows, k.cols, k.pad, wrong);
  }
}

// Kernel timing of a call on host memory brackets the product, not the upload.
void Timing() {
  const int M = 96, K = 160;
  for (const Types& t : kTypes) {
    if (t.dst == RUYAMD_DTYPE_F64) continue;  // (the generic kernel is not timed)
    for (int N : {64, 4}) {
      Context c;
      (void)ruyamd_ctx_set_kernel_timing(c.ctx, 1);
      std::vector<char> lhs(M * K * 8, 1), rhs(K * N * 8, 2), dst(M * N * 8), bias(M * 4, 3);
      const ruyamd_mat l = Mat(t.lhs, lhs.data(), M, K, RUYAMD_ORDER_ROW_MAJOR);
      const ruyamd_mat r = Mat(t.rhs, rhs.data(), K, N, RUYAMD_ORDER_COL_MAJOR);
      const ruyamd_mat d = Mat(t.dst, dst.data(), M, N, RUYAMD_ORDER_COL_MAJOR);
      ruyamd_mul_params p = Params(t.dst);
      p.bias = bias.data();
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
      const auto begin = std::find(R().log.begin(), R().log.end(), "event");
      const auto end = std::find(begin == R().log.end() ? begin : begin + 1, R().log.end(), "event");
      EXPECT(end - begin == 2, "%s x %d: %d launches inside the bracket", t.name, N, static_cast<int>(end - begin) - 1);
      EXPECT(Count("UploadKernel") == 1, "%s", t.name);
    }
  }
}

// A product of device operands that no kernel here ever reads.
struct DeviceCall {
  void* lhs;
  void* rhs;
  void* dst;
  DeviceCall(std::size_t lhs_bytes, std::size_t rhs_bytes, std::size_t dst_bytes) {
    (void)hipMalloc(&lhs, lhs_bytes);
    (void)hipMalloc(&rhs, rhs_bytes);
    (void)hipMalloc(&dst, dst_bytes);
  }
  ~DeviceCall() {
    (void)hipFree(lhs);
    (void)hipFree(rhs);
    (void)hipFree(dst);
  }
};

// The streaming kernel's waves to a group of 16 rows: four only where all
// groups run at once (three workgroups to a CU), or one would have too little
// in flight.
void SkinnyShapes() {
  struct {
    int rows, depth_bytes, narrow;
    const char* shape;  // stages, bytes of one, waves, narrow vectors staged
  } const cases[] = {
      {768 * 16, 1024, 8, "Li2ELi256ELi4ELi8E"},     {768 * 16 + 1, 1024, 8, "Li2ELi256ELi1ELi8E"},
      {900 * 16, 512, 2, "Li2ELi256ELi1ELi8E"},      {1023 * 16, 4096, 4, "Li2ELi256ELi1ELi8E"},
      {1023 * 16, 8192, 8, "Li2ELi256ELi1ELi8E"},    {1023 * 16, 8208, 8, "Li2ELi256ELi4ELi8E"},
      {1023 * 16 + 1, 8208, 8, "Li2ELi256ELi1ELi8E"}, {900 * 16, 1024, 9, "Li2ELi256ELi2ELi16E"},
  };
  for (const auto& c : cases) {
    for (const Types& t : {kTypes[0], kTypes[1]}) {
      Context ctx;
      const int depth = c.depth_bytes / SizeOf(t.lhs);
      DeviceCall call(std::size_t(c.rows) * c.depth_bytes, std::size_t(c.narrow) * c.depth_bytes,
                      std::size_t(c.rows) * c.narrow * SizeOf(t.dst));
      const ruyamd_mat l = Mat(t.lhs, call.lhs, c.rows, depth, RUYAMD_ORDER_ROW_MAJOR);
      const ruyamd_mat r = Mat(t.rhs, call.rhs, depth, c.narrow, RUYAMD_ORDER_COL_MAJOR);
      const ruyamd_mat d = Mat(t.dst, call.dst, c.rows, c.narrow, RUYAMD_ORDER_COL_MAJOR);
      const ruyamd_mul_params p = Params(t.dst);
      EXPECT(ruyamd_mul(ctx.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(ctx.ctx));
      EXPECT(R().log.size() == 1 && Count("GemvMmaKernel") == 1 && Count(c.shape) == 1, "%s %d x %d bytes x %d: %s", t.name,
             c.rows, c.depth_bytes, c.narrow, R().log.empty() ? "nothing" : R().log.back().c_str());
    }
  }
}

// A call can be recorded once it has run: what it then needs of scratch memory
// is there, although a recorded call forms some sums in a launch of their own.
// One that is refused, on a context that has run nothing or a smaller call,
// records nothing.
void Capture() {
  struct {
    int M, K, N, lhs_order, rhs_order, lhs_zero, rhs_zero;
  } const cases[] = {
      {2048, 2048, 2048, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_COL_MAJOR, 0, 3},   // packed, its sums with the product
      {2048, 2048, 2048, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_ROW_MAJOR, 3, 3},
      {2048, 2048, 2048, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_ROW_MAJOR, -5, 3},
      {2048, 2048, 2048, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 3, 3},   // in place
      {3000, 4096, 2500, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 0, 3},
      {4096, 1024, 4096, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 0, 3},
      {1000, 1500, 700, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_COL_MAJOR, 4, -3},
      {1000, 4099, 700, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 4, -3},
      {1100, 1100, 1100, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_ROW_MAJOR, 4, -3},
      {1104, 1104, 1104, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 4, -3},
      {300, 16384, 260, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_ROW_MAJOR, 4, -3},   // a depth in parts
      {64, 8192, 100, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 4, -3},
      {4096, 5000, 7, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_ROW_MAJOR, 4, -3},     // skinny
      {77, 131, 45, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_ROW_MAJOR, 4, -3},
      {100000, 512, 256, RUYAMD_ORDER_COL_MAJOR, RUYAMD_ORDER_COL_MAJOR, 0, 3},   // more rows than a context has room for
      {100000, 512, 256, RUYAMD_ORDER_ROW_MAJOR, RUYAMD_ORDER_COL_MAJOR, 0, 3},
  };
  for (const auto& k : cases) {
    for (const Types& t : kTypes) {
      if (t.dst == RUYAMD_DTYPE_F64) continue;
      const bool zero_points = t.rhs == RUYAMD_DTYPE_I8;
      DeviceCall call(std::size_t(k.M) * k.K * SizeOf(t.lhs), std::size_t(k.K) * k.N * SizeOf(t.rhs),
                      std::size_t(k.M) * k.N * SizeOf(t.dst));
      const ruyamd_mat l = Mat(t.lhs, call.lhs, k.M, k.K, k.lhs_order, zero_points ? k.lhs_zero : 0);
      const ruyamd_mat r = Mat(t.rhs, call.rhs, k.K, k.N, k.rhs_order, zero_points ? k.rhs_zero : 0);
      const ruyamd_mat d = Mat(t.dst, call.dst, k.M, k.N, RUYAMD_ORDER_COL_MAJOR);
      const ruyamd_mul_params p = Params(t.dst);
      for (const std::string before : {"nothing", "a smaller call", "the same call"}) {
        Context c;
        ruyamd_mat sl = l, sr = r, sd = d;
        if (before == "a smaller call") {
          sl.rows = sd.rows = std::min(k.M, 40);
          sr.cols = sd.cols = std::min(k.N, 40);
          sl.cols = sr.rows = std::min(k.K, 77);
        }
        if (before != "nothing")
          EXPECT(ruyamd_mul(c.ctx, &sl, &sr, &p, &sd) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
        R().log.clear();
        R().capturing = true;
        const int rc = ruyamd_mul(c.ctx, &l, &r, &p, &d);
        R().capturing = false;
        EXPECT(R().capture_violations == 0, "%s %d x %d x %d", t.name, k.M, k.K, k.N);
        EXPECT(rc == RUYAMD_OK || before != "the same call", "%s %d x %d x %d (orders %d %d): %s", t.name, k.M, k.K, k.N, k.lhs_order,
               k.rhs_order, ruyamd_ctx_last_error(c.ctx));
        EXPECT(rc == RUYAMD_OK || R().log.empty(), "%s %d x %d x %d (orders %d %d) after %s: refused with %d launches recorded",
               t.name, k.M, k.K, k.N, k.lhs_order, k.rhs_order, before.c_str(), static_cast<int>(R().log.size()));
      }
    }
  }
}

// Rows of any length and alignment that a kernel reads where they lie, without a
// packed copy: recorded on a context that has run nothing, taken without room in
// the static area, and an ordinary call takes no scratch memory for them either.
void RawRowsNeedNoScratch() {
  struct {
    int dtype, M, K, N;
  } const cases[] = {
      {RUYAMD_DTYPE_I8, 64, 100, 64},    {RUYAMD_DTYPE_I8, 300, 777, 300},    {RUYAMD_DTYPE_U8, 200, 333, 200},
      {RUYAMD_DTYPE_U8, 64, 147, 12544}, {RUYAMD_DTYPE_I8, 1000, 1001, 900},  {RUYAMD_DTYPE_I8, 64, 1023, 16384},
      {RUYAMD_DTYPE_I8, 1000, 511, 900}, {RUYAMD_DTYPE_U8, 1024, 1024, 1024},
  };
  for (const auto& k : cases) {
    DeviceCall call(std::size_t(k.M) * k.K, std::size_t(k.K) * k.N, std::size_t(k.M) * k.N);
    const ruyamd_mat l = Mat(k.dtype, call.lhs, k.M, k.K, RUYAMD_ORDER_ROW_MAJOR, 4);
    const ruyamd_mat r = Mat(k.dtype, call.rhs, k.K, k.N, RUYAMD_ORDER_COL_MAJOR, 3);
    const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, k.M, k.N, RUYAMD_ORDER_COL_MAJOR);
    const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
    Context c;
    R().capturing = true;
    EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%d x %d x %d recorded first: %s", k.M, k.K, k.N,
           ruyamd_ctx_last_error(c.ctx));
    R().capturing = false;
    EXPECT(ruyamd_mul_no_alloc(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%d x %d x %d without allocation: %s", k.M, k.K, k.N,
           ruyamd_ctx_last_error(c.ctx));
    R().allocations = 0;
    EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
    EXPECT(R().allocations == 0, "%d x %d x %d: %d allocations", k.M, k.K, k.N, R().allocations);
    EXPECT(R().log.size() == 3, "%d x %d x %d: %d launches", k.M, k.K, k.N, static_cast<int>(R().log.size()));
  }
}

// Sums left to the product cost a call no scratch memory, although a recorded
// call forms some of them in a launch of their own: a first call takes a block
// for an operand that is packed and the sums the pack forms, nothing more.
void ScratchBlocks() {
  struct {
    int M, K, N, lhs_order, lhs_zero, rhs_zero, blocks;
  } const cases[] = {
      {2048, 2048, 2048, RUYAMD_ORDER_COL_MAJOR, 0, 3, 1},  // its sums formed by the product
      {2048, 2048, 2048, RUYAMD_ORDER_COL_MAJOR, 4, 3, 1},  // ... and those of the other operand, used in place
      {1024, 128, 8192, RUYAMD_ORDER_COL_MAJOR, 0, 3, 1},   // by the pack
      {2048, 2048, 2048, RUYAMD_ORDER_COL_MAJOR, 0, 0, 1},  // none
      {2048, 2048, 2048, RUYAMD_ORDER_ROW_MAJOR, 0, 3, 0},  // in place, its sums shared out (not so when recorded)
      {256, 256, 256, RUYAMD_ORDER_ROW_MAJOR, 0, 3, 0},     // in place, formed by each workgroup by itself
  };
  for (const auto& k : cases) {
    DeviceCall call(std::size_t(k.M) * k.K, std::size_t(k.K) * k.N, std::size_t(k.M) * k.N);
    const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, call.lhs, k.M, k.K, k.lhs_order, k.lhs_zero);
    const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, call.rhs, k.K, k.N, RUYAMD_ORDER_COL_MAJOR, k.rhs_zero);
    const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, k.M, k.N, RUYAMD_ORDER_COL_MAJOR);
    const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
    Context c;
    for (int want : {k.blocks, 0}) {
      R().allocations = 0;
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
      EXPECT(R().allocations == want, "%d x %d x %d, zero points %d %d: %d allocations, expected %d", k.M, k.K,
             k.N, k.lhs_zero, k.rhs_zero, R().allocations, want);
    }
  }
}

// A workspace whose calls take turns with its pieces: made large enough once, from
// the eighth call that needs scratch on, by no more than four times what a call
// takes; a call that is recorded finds its room whoever's turn it is, also one that
// takes more than a piece, and a growing one only adds what it needs. Not where a call
// takes so much that the pieces would crowd the operands out of the caches.
void ScratchInTurns() {
  auto on_device = [] {
    std::size_t sum = 0;
    for (const auto& range : R().device) sum += range.second;
    return sum;
  };
  struct {
    int M, K, N;
    bool turns;
  } const cases[] = {{1000, 1501, 700, true}, {2000, 4099, 2100, true}, {160, 4027, 6300, false},
                     {160, 6260, 8768, false}, {6000, 15000, 1100, false}};
  for (const auto& k : cases) {
    DeviceCall call(std::size_t(k.M) * k.K, std::size_t(k.K) * k.N, std::size_t(k.M) * k.N);
    const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, call.lhs, k.M, k.K, RUYAMD_ORDER_COL_MAJOR, 4);
    const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, call.rhs, k.K, k.N, RUYAMD_ORDER_ROW_MAJOR, 3);
    const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, k.M, k.N, RUYAMD_ORDER_COL_MAJOR);
    ruyamd_mat small_l = l, small_d = d;
    small_l.rows = small_d.rows = k.M / 3;
    const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
    Context c;
    const std::size_t before = on_device();
    std::size_t once = 0;
    for (int i = 1; i <= 20; ++i) {
      R().allocations = 0;
      EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
      if (i == 1) once = on_device() - before;
      EXPECT(R().allocations == 0 || i <= 2 || (k.turns && i <= 10), "call %d: %d allocations", i, R().allocations);
      EXPECT(on_device() - before <= (k.turns ? 4 : 1) * once + (1 << 20), "call %d: %zu bytes, one call %zu", i,
             on_device() - before, once);
      if (i >= 15) {
        R().capturing = true;
        EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "recorded behind call %d: %s", i, ruyamd_ctx_last_error(c.ctx));
        R().capturing = false;
        EXPECT(R().capture_violations == 0, "behind call %d", i);
      }
    }
    Context fresh;
    for (int i = 1; i <= 24; ++i) {
      const bool small = i <= 12 || i % 3 == 0;
      EXPECT(ruyamd_mul(fresh.ctx, small ? &small_l : &l, &r, &p, small ? &small_d : &d) == RUYAMD_OK, "%s",
             ruyamd_ctx_last_error(fresh.ctx));
    }
    R().allocations = 0;
    for (int i = 0; i < 9; ++i)
      EXPECT(ruyamd_mul(fresh.ctx, i % 3 ? &l : &small_l, &r, &p, i % 3 ? &d : &small_d) == RUYAMD_OK, "%s",
             ruyamd_ctx_last_error(fresh.ctx));
    EXPECT(R().allocations == 0, "%d allocations", R().allocations);
    for (const bool small : {false, true, false}) {
      R().capturing = true;
      EXPECT(ruyamd_mul(fresh.ctx, small ? &small_l : &l, &r, &p, small ? &small_d : &d) == RUYAMD_OK, "%s",
             ruyamd_ctx_last_error(fresh.ctx));
      R().capturing = false;
      EXPECT(ruyamd_mul(fresh.ctx, small ? &l : &small_l, &r, &p, small ? &d : &small_d) == RUYAMD_OK, "%s",
             ruyamd_ctx_last_error(fresh.ctx));
    }
    EXPECT(R().capture_violations == 0, "%d x %d x %d", k.M, k.K, k.N);
  }
}

// A device with no room for a workspace whose calls take turns: it is asked once (or
// once more for a smaller size that calls come in), the block that there was stays, and calls go on in it
// without a further allocation or free, which waits for the device.
void ScratchInTurnsRefused() {
  const int M = 2000, K = 2051, N = 1800;
  DeviceCall call(std::size_t(M) * K, std::size_t(K) * N, std::size_t(M) * N);
  const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, call.lhs, M, K, RUYAMD_ORDER_COL_MAJOR, 4);
  const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, call.rhs, K, N, RUYAMD_ORDER_ROW_MAJOR, 3);
  const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, M, N, RUYAMD_ORDER_COL_MAJOR);
  ruyamd_mat small_l = l, small_d = d;
  small_l.rows = small_d.rows = M / 3;
  const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
  for (const bool two_sizes : {false, true}) {
    Context c;
    auto run = [&](int i) {
      const bool small = two_sizes && i % 2;
      EXPECT(ruyamd_mul(c.ctx, small ? &small_l : &l, &r, &p, small ? &small_d : &d) == RUYAMD_OK, "%s",
             ruyamd_ctx_last_error(c.ctx));
    };
    for (int i = 0; i < 4; ++i) run(i);
    const auto held = R().device;
    std::size_t bytes = 0;
    for (const auto& range : held) bytes += range.second;
    R().device_limit = bytes + (std::size_t(1) << 20);
    R().allocations = R().frees = 0;
    for (int i = 0; i < 20; ++i) run(i);
    // (What is larger than a size refused before is not asked for either.)
    EXPECT(R().allocations >= 1 && R().allocations <= 1 + two_sizes && R().frees == 0, "%d allocations, %d frees",
           R().allocations, R().frees);
    EXPECT(R().device == held, "the block that there was is gone");
    EXPECT(R().last_error == hipSuccess, "an error is left behind");
    R().capturing = true;
    run(0);
    R().capturing = false;
    EXPECT(R().capture_violations == 0, "while recording");
    R().device_limit = ~std::size_t(0);
  }
}

// The calls after a program's first ones while another thread records a graph: whatever
// the workspace does for them does not end the recording.
void ScratchInTurnsBesideACapture() {
  const int M = 1000, K = 1501, N = 700;
  DeviceCall call(std::size_t(M) * K, std::size_t(K) * N, std::size_t(M) * N);
  const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, call.lhs, M, K, RUYAMD_ORDER_COL_MAJOR, 4);
  const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, call.rhs, K, N, RUYAMD_ORDER_ROW_MAJOR, 3);
  const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, M, N, RUYAMD_ORDER_COL_MAJOR);
  const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
  Context c;
  for (int i = 0; i < 20; ++i) {
    R().captured_elsewhere = i >= 2;
    EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
  }
  R().captured_elsewhere = false;
  EXPECT(R().capture_violations == 0, "%d violations", R().capture_violations);
  EXPECT(R().mode == hipStreamCaptureModeGlobal, "the thread's mode was not given back");
  R().capture_violations = 0;
}

bool Staged(const std::string& kernel) {
  return kernel.find("MfmaGemmKernel") != std::string::npos &&
         (kernel.find("Lb0ELi1EEEv") != std::string::npos || kernel.find("Lb0ELi2EEEv") != std::string::npos);
}

// Which products of operands usable in place the staged form of the smallest
// tile takes: with one workgroup a CU whole stages of depth only, since the end of
// a row costs it more than a direct load does; with two also those whose sums it
// forms, or whose columns end in many rows that are stored one by one.
void StagedRule() {
  struct {
    int M, K, N, rhs_zero;
    bool staged;
  } const cases[] = {
      {2048, 128, 1024, 0, true},  {2048, 384, 1024, 0, true},  {2048, 320, 1024, 0, false}, {2048, 320, 1024, 3, true},
      {2048, 144, 1024, 0, false}, {2048, 144, 1024, 3, true},  {2048, 240, 1024, 3, true},  {2048, 256, 1024, 3, true},
      {2048, 272, 1024, 3, true},  {2048, 496, 1024, 3, true},  {2048, 512, 1024, 3, true},  {2048, 528, 1024, 3, false},
      {2039, 320, 1024, 0, false}, {2040, 320, 1024, 0, true},  {2047, 144, 1024, 0, true},  {2040, 528, 1024, 0, false},
      {1024, 384, 1024, 0, false}, {1024, 400, 1024, 0, false}, {1024, 512, 1024, 0, true},  {1024, 624, 1024, 3, false},
      {1024, 640, 1024, 0, true},  {1024, 784, 1024, 0, false}, {1024, 896, 1024, 3, true},  {1024, 1024, 1024, 0, false},
      {1024, 144, 1024, 3, false}, {1016, 496, 1024, 0, false}, {2112, 128, 1024, 0, false},
  };
  for (const auto& k : cases) {
    Context c;
    DeviceCall call(std::size_t(k.M) * k.K, std::size_t(k.K) * k.N, std::size_t(k.M) * k.N);
    const ruyamd_mat l = Mat(RUYAMD_DTYPE_I8, call.lhs, k.M, k.K, RUYAMD_ORDER_ROW_MAJOR);
    const ruyamd_mat r = Mat(RUYAMD_DTYPE_I8, call.rhs, k.K, k.N, RUYAMD_ORDER_COL_MAJOR, k.rhs_zero);
    const ruyamd_mat d = Mat(RUYAMD_DTYPE_I8, call.dst, k.M, k.N, RUYAMD_ORDER_COL_MAJOR);
    const ruyamd_mul_params p = Params(RUYAMD_DTYPE_I8);
    EXPECT(ruyamd_mul(c.ctx, &l, &r, &p, &d) == RUYAMD_OK, "%s", ruyamd_ctx_last_error(c.ctx));
    EXPECT(Staged(R().log.back()) == k.staged, "%d x %d x %d, zero point %d: %s", k.M, k.K, k.N, k.rhs_zero,
           R().log.back().c_str());
  }
}

// What calls read from the standard input run on: a line each of "ordinary",
// "recorded" or "without_allocation", the types of LHS, RHS and destination, rows,
// depth, columns, the three storage orders, what the three strides are longer
// than the rows or columns, the operands' zero points, whether each is cached, the
// address of their first element modulo 16 and the tile that is forced (0 0: none).
// Answered by a line of the call's result, its allocations and what it launched.
// Ordinary calls use one context, the others a new one each. (No operand is
// touched.)
int Routes() {
  const std::size_t room = std::size_t(1) << 38;
  char* const at = static_cast<char*>(mmap(nullptr, 3 * room, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0));
  if (at == MAP_FAILED) std::abort();
  R().device[at] = 3 * room;
  R().fill_allocations = false;
  Context shared;
  char how[32];
  int types[3], m, k, n, order[3], pad[3], zero[2], cached[2], misaligned, tile[2];
  while (std::scanf("%31s %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d", how, &types[0], &types[1], &types[2], &m,
                    &k, &n, &order[0], &order[1], &order[2], &pad[0], &pad[1], &pad[2], &zero[0], &zero[1], &cached[0],
                    &cached[1], &misaligned, &tile[0], &tile[1]) == 20) {
    ruyamd_mat mats[3];
    for (int i = 0; i < 3; ++i) {
      mats[i] = Mat(types[i], at + i * room + misaligned, i == 1 ? k : m, i == 0 ? k : n, order[i], i < 2 ? zero[i] : 0,
                    i < 2 && cached[i] ? RUYAMD_CACHE_ALWAYS : RUYAMD_CACHE_NEVER);
      mats[i].stride += pad[i];
    }
    ruyamd_mul_params p = Params(types[2]);
    if (types[2] == RUYAMD_DTYPE_I32) p.multiplier_fixedpoint = p.multiplier_exponent = 0;
    const bool ordinary = std::strcmp(how, "ordinary") == 0;
    Context* own = ordinary ? nullptr : new Context;
    ruyamd_ctx* const ctx = ordinary ? shared.ctx : own->ctx;
    (void)ruyamd_ctx_force_tile(ctx, tile[0], tile[1], 0);
    R().log.clear();
    R().allocations = 0;
    R().capturing = std::strcmp(how, "recorded") == 0;
    const int rc = (std::strcmp(how, "without_allocation") == 0 ? ruyamd_mul_no_alloc : ruyamd_mul)(ctx, &mats[0], &mats[1],
                                                                                                  &p, &mats[2]);
    R().capturing = false;
    std::printf("%d %d", rc, R().allocations);
    for (const std::string& kernel : R().log) std::printf(" %s", kernel.c_str());
    std::printf("\n");
    ruyamd_ctx_clear_prepacked_cache(ctx);
    delete own;
  }
  return 0;
}

// The names of the library's kernels.
int Kernels() {
  for (const auto& k : R().kernels) std::printf("%s\n", k.second.c_str());
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "routes") return Routes();
  if (which == "kernels") return Kernels();
  if (which == "failed_upload") FailedUpload();
  else if (which == "page_locked_sources") PageLockedSources();
  else if (which == "page_locked_destinations") PageLockedDestinations();
  else if (which == "skinny_shapes") SkinnyShapes();
  else if (which == "timing") Timing();
  else if (which == "capture") Capture();
  else if (which == "raw_rows") RawRowsNeedNoScratch();
  else if (which == "scratch_blocks") ScratchBlocks();
  else if (which == "scratch_in_turns") ScratchInTurns();
  else if (which == "scratch_in_turns_refused") ScratchInTurnsRefused();
  else if (which == "scratch_in_turns_beside_a_capture") ScratchInTurnsBesideACapture();
  else if (which == "staged_rule") StagedRule();
  else return 2;
  if (g_failures) {
    std::printf("%d failures\n", g_failures);
    return 1;
  }
  std::printf("%s: all passed\n", which.c_str());
  return 0;
}
