// Per-caller state behind ruyamd_ctx: the counterpart of ruy::CtxImpl
// (ruy/ctx_impl.h:57-82) for a device: a stream, a grow-only device workspace
// that replaces the bump allocator (ruy/allocator.h:56-97), the
// prepacked-matrix cache, and the knobs ruy::Context exposes.
#ifndef RUY_AMD_CSRC_CONTEXT_H_
#define RUY_AMD_CSRC_CONTEXT_H_

#include <hip/hip_runtime.h>

#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "internal.h"
#include "kernels/host_copy.h"
#include "prepacked_cache.h"

namespace ruyamd {

// Device scratch memory handed out by bumping a pointer; everything is
// released together at the start of the next call (ruy's
// Allocator::FreeAll, ruy/frontend.cc:34). If a call outgrows the current
// block an extra block is taken, and the next Reset replaces all blocks with
// one that is large enough. Once Pin() has been called (work that refers to
// the scratch was recorded for later replay) blocks are never released or
// replaced before the workspace is destroyed, and while growth is disabled
// Alloc fails instead of taking a new block.
class Workspace {
 public:
  ~Workspace();
  // 256-byte aligned device memory valid until the next Reset; nullptr on
  // allocation failure.
  void* Alloc(std::size_t bytes);
  // The same for memory the caller can do without (it runs another way when
  // there is none): a failure is not recorded by exhausted().
  void* AllocOptional(std::size_t bytes);
  // Call only when no kernel still uses the previous call's scratch.
  void Reset();
  std::size_t capacity() const;
  void Pin() { pinned_ = true; }
  void set_growth_allowed(bool allowed) { growth_allowed_ = allowed; }
  // Makes this a workspace over memory it does not own: one block that is
  // never released, replaced or added to. For a workspace that owns nothing.
  void UseFixed(void* base, std::size_t size);
  // Whether an Alloc has failed since the last Reset.
  bool exhausted() const { return exhausted_; }

 private:
  std::size_t Piece() const;
  struct Block {
    char* base;
    std::size_t size;
    std::size_t used;
  };
  // Calls take turns with the pieces of a workspace of one block, where each needs
  // no more than one: the lines of a packed operand are still held by the caches of
  // the XCDs that have read it, and are slower to write to than others. (8.9 MB packed
  // and then read by all XCDs, call after call: 18.9 us in one place, 17.4 in two. int8,
  // both sides packed, one place -> these: 2048 x 2051 x 2048 23.5 -> 17.7 us, 1024 x 4099 x
  // 1024 20.8 -> 15.6, 1000 x 1500 x 700 13.9 -> 12.8, in two places 14.0; 4000 x 4003 x 1008
  // 31.1 -> 27.6.) Four pieces while a call takes no more than kFourTurnsUpTo, two (as good
  // there) up to kTurnsUpTo. None beyond: what the XCDs' caches (4 MiB each) hold of
  // such a call is hardly in the way (160 x 4027 x 8000, 32 MiB packed, 24.1 -> 23.6 us; x 6260
  // 34.2 -> 33.8), but two contexts' pieces and operands no longer fit the 256 MiB of the
  // cache in front of memory: 160 x 6260 x 8768 36.2 -> 44.6, 160 x 8003 x 7500 40.5 -> 47.8.
  // (24 MiB, 160 x 3011 x 8000: 21.3 -> 19.3, two contexts 19.3 and 19.3.) From its kTurnsFrom-th call that needs scratch
  // on, a workspace is made large enough for that, once: a program's first calls do not
  // wait for it. What the device has refused is not asked for again: an allocation and
  // a free each call would cost more than the turns give.
  static constexpr std::size_t kFourTurnsUpTo = std::size_t(8) << 20;
  static constexpr std::size_t kTurnsUpTo = std::size_t(24) << 20;
  static constexpr int kTurnsFrom = 8;
  static std::size_t TurnsFor(std::size_t taken) { return taken <= kFourTurnsUpTo ? 4 : 2; }
  std::vector<Block> blocks_;
  std::size_t taken_ = 0;       // by the call so far
  int calls_ = 0;               // that needed scratch, up to kTurnsFrom
  std::size_t refused_ = ~std::size_t(0);  // the smallest block for turns that could not be had
  std::size_t turns_ = 2;                  // pieces,
  std::size_t turn_ = 0;                   // the one this call starts in,
  std::size_t wrapped_used_ = 0;           // and what did not fit behind has taken in front of it
  bool pinned_ = false;
  bool growth_allowed_ = true;
  bool fixed_ = false;
  bool exhausted_ = false;
};

// What the runtime knows about a buffer of a call.
enum class Memory {
  kDevice,            // (managed memory too)
  kPageable,          // ordinary host memory
  kPageLocked,        // hipHostMalloc, torch's pinned tensors
  kPageLockedMapped,  // the same, at the same address for kernels
};
Memory MemoryOf(const void* p);

// Moves pageable host memory to and from the device through a small ring of
// pinned chunks: the CPU copies into (out of) a chunk while the copy engine
// works on the previous ones, and every transfer the engine sees is a true
// asynchronous pinned copy. Small operands share a chunk. A source that is
// already page-locked skips the chunks: it is read where it lies, in stream
// order, so that a call may follow the work that fills it on the same stream;
// a large page-locked destination is written by the copy engine directly.
// Small transfers (kByKernel bytes) do not use the copy engine at all: what a
// call uploads is collected - in a chunk, or where it lies if that is 16-byte
// aligned page-locked memory - and moved by one kernel when the first kernel
// that may read it is about to be launched (Flush), and a small destination
// comes back through a chunk by a kernel whose completion the host sees in host
// memory (kernels/host_copy.hip). Used only by calls
// that were handed host pointers; such a call ends with a stream
// synchronisation or a download seen to be complete, after which Reset()
// makes all chunks available again.
class HostStaging {
 public:
  ~HostStaging();
  // dst_dev[0, bytes) = src_host[0, bytes), ordered on `stream` once Flush has
  // been called. dst_dev is 16-byte aligned and has room for a whole number of
  // 16-byte granules. A pageable source is read before this returns, a
  // page-locked one (`source`) when the stream gets there.
  bool ToDevice(void* dst_dev, const void* src_host, std::size_t bytes, Memory source, hipStream_t stream);
  // Copies `outer` runs of `inner_bytes`, `pitch` bytes apart in both images,
  // from device to host after everything already enqueued on `stream`; the
  // bytes between the runs of the host image are not written. The host image
  // is complete when this returns (pageable or small destination) or once the
  // stream has been synchronised (page-locked `destination` above kThroughChunk,
  // written directly). *drained is set if everything enqueued on `stream` so far is
  // known to have finished. src_dev as dst_dev in ToDevice.
  bool ToHost2D(void* dst_host, const void* src_dev, std::size_t pitch, std::size_t inner_bytes,
                std::size_t outer, Memory destination, hipStream_t stream, bool* drained);
  // Forgets uploads that a failed call has left behind.
  void DropPending() { pending_.count = 0; }
  // Enqueues the uploads collected so far: before any kernel that may read them.
  bool Flush(hipStream_t stream) { return pending_.count == 0 || FlushPending(stream); }
  // Call after the stream has been synchronised (or seen drained).
  void Reset();

 private:
  static constexpr std::size_t kChunkBytes = std::size_t(4) << 20;
  static constexpr int kChunks = 4;
  // Up to here a kernel moves a transfer faster than the copy engine does,
  // counting what it costs the streams to hand over to that engine and back
  // (int8, cached weights, whole calls by the copy engine -> by kernels: 200 KB
  // each way 73 -> 40 us, 1 MiB each way 141 -> 118 us; 2 MiB and more gain from
  // the engine's higher rate and from the CPU filling the next chunk meanwhile).
  static constexpr std::size_t kByKernel = std::size_t(1) << 20;
  // A page-locked destination the engine writes directly, where the kernel's way
  // ends with the CPU's copy out of a chunk, which costs more when it is one of
  // many runs (whole calls, destination by the engine -> by the kernel: 64 KiB 33
  // to 37 -> 24 us, 196 KiB 40 to 44 -> 35, 384 KiB 41 to 45 -> 41, 640 KiB 46 to
  // 50 -> 53, 1000 KiB 82 to 86 -> 105; in runs 64 KiB 32 to 34 -> 25, 196 KiB 37
  // to 41 -> 42, 512 KiB 44 to 47 -> 65).
  static constexpr std::size_t kThroughChunk = std::size_t(384) << 10;
  static constexpr std::size_t kRunsThroughChunk = std::size_t(128) << 10;
  // Behind the chunks: one word per workgroup of a download.
  static constexpr std::size_t kDoneBytes = kByKernel / kHostCopyBlockBytes * sizeof(uint32_t);
  bool Init();
  bool Collect(void* to, const void* from, std::size_t bytes, hipStream_t stream);
  bool FlushPending(hipStream_t stream);
  bool SmallToHost2D(char* dst, const void* src_dev, std::size_t pitch, std::size_t inner_bytes, std::size_t outer,
                     hipStream_t stream, bool* drained);
  // Makes chunk c reusable: waits for the transfer that last used it.
  bool WaitFree(int c);
  bool RetireCurrent(hipStream_t stream);
  char* pinned_ = nullptr;
  hipEvent_t done_[kChunks] = {};
  bool busy_[kChunks] = {};
  int current_ = 0;            // chunk being filled by ToDevice
  std::size_t fill_ = 0;       // bytes of it already handed to the copy engine or collected in pending_
  UploadPieces pending_;       // pieces (of the current chunk or page-locked sources) that no launch has moved yet
  uint32_t downloads_ = 0;     // the value the last download's workgroups left in their words
};

}  // namespace ruyamd

struct ruyamd_ctx {
  int device = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  bool synchronous = true;
  bool capturing = false;  // this call's stream is recording a graph
  // This call may not allocate device memory (ruyamd_mul_no_alloc): scratch
  // comes from the GPU's static area, the prepacked cache is only looked up.
  bool no_alloc = false;
  int last_used_path = RUYAMD_PATH_NONE;
  int runtime_enabled_paths = RUYAMD_PATH_NONE;  // kNone = not decided yet
  int max_num_threads = 1;
  int explicit_tuning = 0;        // ruy::Tuning::kAuto
  int num_threads_strategy = 0;   // ruy::NumThreadsStrategy::kDefault
  int performance_advisories = 0;
  int last_kernel = RUYAMD_KERNEL_NONE;
  bool force_generic = false;
  int forced_depth_parts = 0;
  bool forced_split_without_waiting = false;
  int forced_tile_rows = 0, forced_tile_cols = 0;  // diagnostics: 0 = the timing model picks
  std::string last_error;
  ruyamd::Workspace workspace;         // grows on demand (hipMalloc)
  ruyamd::Workspace static_workspace;  // over this GPU's static scratch area
  ruyamd::Workspace* ws = &workspace;  // the one the current call draws from
  ruyamd::HostStaging staging;
  std::unique_ptr<ruyamd::PrepackedCache> cache;
  int multiprocessor_count = 0;
  // Arrival counters of the depth-split matrix-core kernels: zero between
  // launches (the kernels leave them so), allocated with the context.
  uint32_t* split_counters = nullptr;
  // The same in this GPU's static scratch area, for calls that may not allocate.
  uint32_t* static_split_counters = nullptr;
  // Room for sums formed by a launch of their own, of one operand and of the
  // other (fused_sums::kMaxRows each; more come from the workspace): there from
  // the start, since a call that is being recorded needs it where an ordinary
  // one does not.
  int32_t* sums_words = nullptr;
  // Row sums formed inside the launch of the largest int8 tile
  // (kernels/fused_sums.h): two sets of 64-bit words, one per row, all zero
  // when a launch starts. A launch uses set `row_sums_next` and clears what
  // the launch before it left in the other one (`row_sums_dirty_rows`).
  long long* row_sums_sets[2] = {nullptr, nullptr};
  int row_sums_dirty_rows[2] = {0, 0};
  int row_sums_next = 0;
  bool row_sums_in_launch = true;
  bool row_sums_fetch_late = false;
  int64_t row_sums_calls = 0;
  int row_sums_spin_limit = 1 << 14;
  // Optional timing of the dominant kernel of each call.
  bool kernel_timing = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> timing_pending;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> timing_pool;
  // The stream for a kernel that may read the call's operands: whatever has
  // been collected for upload is enqueued first (upload_failed if that fails;
  // the call then reports it).
  hipStream_t LaunchStream() {
    if (!staging.Flush(stream)) upload_failed = true;
    return stream;
  }
  bool upload_failed = false;
  // Brackets for the dispatcher: Begin returns false if timing is off.
  bool TimingBegin();
  void TimingEnd();
};

#endif  // RUY_AMD_CSRC_CONTEXT_H_
