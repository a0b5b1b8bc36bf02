// Library plumbing: last-error slot, per-stream scratch arena, buffer knobs.
#include <atomic>
#include <chrono>
#include <thread>
#include <map>
#include <mutex>

#include "common.h"

namespace mnt {

static thread_local std::string g_last_error;

void set_last_error(const std::string &message) { g_last_error = message; }

static std::mutex g_arena_mutex;
static std::map<std::pair<int, hipStream_t>, Arena *> g_arenas;

// ---- one caller thread per stream ------------------------------------------

static std::atomic<unsigned long long> g_next_thread_token{1};
static thread_local unsigned long long t_token = 0;
static thread_local int t_depth = 0;
static thread_local std::vector<Arena *> t_taken;      // arenas this thread took during the call under way

static unsigned long long thread_token() {
  if (t_token == 0) t_token = g_next_thread_token.fetch_add(1, std::memory_order_relaxed);
  return t_token;
}

void enter_call() { ++t_depth; }

// Current device, or -1 on a machine without one (the registry and its
// ownership rules work there too; anything that allocates fails later).
static int registry_device() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    device = -1;
  }
  return device;
}

Arena &Arena::of(hipStream_t stream) {
  const int device = registry_device();
  const unsigned long long me = thread_token();
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  auto key = std::make_pair(device, stream);
  auto it = g_arenas.find(key);
  if (it == g_arenas.end()) it = g_arenas.emplace(key, new Arena(stream)).first;
  Arena &arena = *it->second;
  if ((arena.held_ || arena.pinned_by_thread_) && arena.holder_ != me) {
    MNT_FAIL("stream %p is in use by another thread: the library keeps per-stream state (scratch arena, "
             "two-phase build state) and takes one caller thread per stream at a time",
             static_cast<void *>(stream));
  }
  if (t_depth > 0 && !arena.held_) {
    arena.held_ = true;
    arena.holder_ = me;
    t_taken.push_back(&arena);
  }
  return arena;
}

void leave_call() {
  if (--t_depth > 0 || t_taken.empty()) return;
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  for (Arena *arena : t_taken) arena->held_ = false;
  t_taken.clear();
}

void Arena::pin(hipStream_t stream) {
  Arena &arena = Arena::of(stream);              // fails when another thread is inside or has pinned it
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  arena.pinned_by_thread_ = true;
  arena.holder_ = thread_token();
}

void Arena::unpin(hipStream_t stream) {
  Arena &arena = Arena::of(stream);
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  arena.pinned_by_thread_ = false;
}

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

void Arena::add_page(size_t bytes) {
  Page page;
  page.size = align_up(bytes, 256);
  page.used = 0;
  MNT_HIP(hipMalloc(reinterpret_cast<void **>(&page.base), page.size));
  pages_.push_back(page);
}

void *Arena::alloc(size_t bytes) {
  bytes = align_up(bytes ? bytes : 1, 256);
  for (size_t p = cursor_; p < pages_.size(); ++p) {
    if (p != cursor_) pages_[p].used = 0;
    if (pages_[p].used + bytes <= pages_[p].size) {
      void *ptr = pages_[p].base + pages_[p].used;
      pages_[p].used += bytes;
      cursor_ = p;
      return ptr;
    }
  }
  size_t want = static_cast<size_t>(static_cast<double>(bytes) * (1.0 + (growth_ > 0 ? growth_ : 0)));
  size_t pages = (want + page_size_ - 1) / page_size_;
  add_page(pages * page_size_);
  cursor_ = pages_.size() - 1;
  pages_[cursor_].used = bytes;
  return pages_[cursor_].base;
}

Arena::Mark Arena::mark() const {
  if (pages_.empty()) return Mark{0, 0};
  return Mark{cursor_, pages_[cursor_].used};
}

void Arena::release(const Mark &m) {
  if (pages_.empty()) return;
  for (size_t p = m.page + 1; p < pages_.size(); ++p) pages_[p].used = 0;
  cursor_ = m.page;
  if (cursor_ < pages_.size()) pages_[cursor_].used = m.used;
}

void Arena::preallocate(size_t bytes) {
  size_t have = 0;
  for (const auto &p : pages_) have = p.size > have ? p.size : have;
  if (have >= bytes) return;
  add_page(align_up(bytes, page_size_));
}

void Arena::free_all(bool synchronise) {
  if (synchronise) MNT_HIP(hipStreamSynchronize(stream_));
  for (auto &p : pages_) MNT_HIP(hipFree(p.base));
  pages_.clear();
  cursor_ = 0;
  for (int slot = 0; slot < kPersistentSlots; ++slot) {
    if (persistent_[slot]) {
      MNT_HIP(hipFree(persistent_[slot]));
      persistent_[slot] = nullptr;
      persistent_size_[slot] = 0;
    }
  }
  pending.valid = false;
  map_state_valid = false;
  pass_pending = false;
  zero_bitmap_words = 0;
  words_cleared_ = false;
}

void Arena::reset_device() {
  int device = 0;
  MNT_HIP(hipGetDevice(&device));
  const unsigned long long me = thread_token();
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  for (const auto &entry : g_arenas) {
    const Arena *arena = entry.second;
    MNT_CHECK(entry.first.first != device || !(arena->held_ || arena->pinned_by_thread_) || arena->holder_ == me,
              "another thread is inside the library on stream %p of this device: no reset while it is",
              static_cast<void *>(entry.first.second));
  }
  for (Arena *arena : t_taken) arena->held_ = false;     // this thread's own: they are about to go
  t_taken.clear();
  for (auto it = g_arenas.begin(); it != g_arenas.end();) {
    if (it->first.first != device) {
      ++it;
      continue;
    }
    Arena *arena = it->second;
    arena->free_all(false);               // the caller has waited for the whole device; the stream may be gone
    if (arena->pinned_ != nullptr) {
      MNT_HIP(hipHostFree(arena->pinned_));
      arena->pinned_ = nullptr;
      arena->pinned_device_ = nullptr;
    }
    delete arena;
    it = g_arenas.erase(it);
  }
}

size_t Arena::total() const {
  size_t t = 0;
  for (const auto &p : pages_) t += p.size;
  return t;
}

size_t Arena::used() const {
  size_t t = 0;
  for (size_t p = 0; p < pages_.size() && p <= cursor_; ++p) t += pages_[p].used;
  return t;
}

void *Arena::pinned() {
  if (!pinned_) {
    constexpr size_t bytes = kPinnedBytes + sizeof(unsigned long long) * kPinnedWords;
    MNT_HIP(hipHostMalloc(&pinned_, bytes, hipHostMallocMapped | hipHostMallocCoherent));
    memset(pinned_, 0, bytes);
    MNT_HIP(hipHostGetDevicePointer(&pinned_device_, pinned_, 0));
  }
  return pinned_;
}

void *Arena::pinned_device() {
  pinned();
  return pinned_device_;
}

unsigned long long *Arena::flag_device(int slot) {
  return reinterpret_cast<unsigned long long *>(static_cast<char *>(pinned_device()) + kFlagOffset +
                                                static_cast<size_t>(slot) * 64);
}

static std::atomic<long long> g_host_waits{0}, g_host_wait_ns{0};

void Arena::wait_flag(int slot, unsigned long long sequence) {
  wait_word(reinterpret_cast<volatile unsigned long long *>(static_cast<char *>(pinned()) + kFlagOffset +
                                                            static_cast<size_t>(slot) * 64),
            sequence);
}

template <typename Done>
void Arena::spin(Done done) {
  const auto start = std::chrono::steady_clock::now();
  struct Tally {
    std::chrono::steady_clock::time_point since;
    ~Tally() {
      g_host_waits.fetch_add(1, std::memory_order_relaxed);
      g_host_wait_ns.fetch_add(std::chrono::duration_cast<std::chrono::nanoseconds>(
                                   std::chrono::steady_clock::now() - since).count(),
                               std::memory_order_relaxed);
    }
  } tally{start};
  unsigned spins = 0;
  while (!done()) {
    if ((++spins & 0x3FFFu) == 0) {
      const auto waited = std::chrono::steady_clock::now() - start;
      if (waited > std::chrono::seconds(2)) {
        MNT_HIP(hipStreamSynchronize(stream_));
        MNT_CHECK(done(), "a kernel finished without signalling its completion flag");
        break;
      }
    }
    __builtin_ia32_pause();
  }
  std::atomic_thread_fence(std::memory_order_acquire);
}

const volatile unsigned long long *Arena::wait_words(int count, unsigned long long sequence) {
  const volatile unsigned long long *words =
      reinterpret_cast<const volatile unsigned long long *>(static_cast<char *>(pinned()) + kPinnedBytes);
  int at = 0;
  spin([&] {
    while (at < count && static_cast<unsigned>(words[at] >> 32) == static_cast<unsigned>(sequence)) ++at;
    return at == count;
  });
  return words;
}

void Arena::wait_word(volatile unsigned long long *flag, unsigned long long sequence) {
  spin([&] { return *flag == sequence; });
}

void *Arena::persistent(int slot, size_t bytes) {
  if (bytes > persistent_size_[slot]) {
    if (persistent_[slot]) {
      MNT_HIP(hipStreamSynchronize(stream_));
      MNT_HIP(hipFree(persistent_[slot]));
    }
    persistent_size_[slot] = align_up(bytes + bytes / 4, 1 << 20);
    MNT_HIP(hipMalloc(&persistent_[slot], persistent_size_[slot]));
    if (slot == 0) zero_bitmap_words = 0;
  }
  return persistent_[slot];
}

__global__ __launch_bounds__(Arena::kWords) void clear_words_kernel(unsigned long long *__restrict__ words) {
  words[threadIdx.x] = 0ull;
}

unsigned long long *Arena::words() {
  auto *block = static_cast<unsigned long long *>(persistent(3, sizeof(unsigned long long) * kWords));
  if (!words_cleared_) {
    clear_words_kernel<<<1, kWords, 0, stream_>>>(block);
    check_launch("clear_words_kernel");
    words_cleared_ = true;
  }
  return block;
}

// ---- stage profiler -------------------------------------------------------

static bool g_profile_on = false;
static std::vector<std::pair<const char *, hipEvent_t>> g_marks;
static std::vector<hipEvent_t> g_event_pool;
static constexpr size_t kMaxMarks = 4096;

static std::thread::id g_profile_thread;

int compute_units() {
  static std::atomic<int> known[64];
  int device = 0;
  MNT_HIP(hipGetDevice(&device));
  const int slot = device & 63;
  int units = known[slot].load(std::memory_order_relaxed);
  if (units == 0) {
    MNT_HIP(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
    units = units > 0 ? units : 256;
    known[slot].store(units, std::memory_order_relaxed);
  }
  return units;
}

void profile_mark(const char *label, hipStream_t stream) {
  // marks are kept for the thread that turned profiling on: the look-ahead
  // worker runs the same entry points on another stream at the same time
  if (!g_profile_on || std::this_thread::get_id() != g_profile_thread || g_marks.size() >= kMaxMarks) return;
  hipEvent_t event;
  if (!g_event_pool.empty()) {
    event = g_event_pool.back();
    g_event_pool.pop_back();
  } else {
    MNT_HIP(hipEventCreate(&event));
  }
  MNT_HIP(hipEventRecord(event, stream));
  g_marks.emplace_back(label, event);
}

// ---- plain streaming kernels: the memory ceilings a benchmark quotes -------

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kStreamBlock = 256;
constexpr int kStreamUnroll = 4;            // 16-byte vectors in flight per lane

__global__ __launch_bounds__(kStreamBlock) void stream_copy_kernel(const u32x4 *__restrict__ src,
                                                                  u32x4 *__restrict__ dst, long long vectors) {
  const long long stride = static_cast<long long>(gridDim.x) * kStreamBlock;
  long long i = static_cast<long long>(blockIdx.x) * kStreamBlock + threadIdx.x;
  for (; i + (kStreamUnroll - 1) * stride < vectors; i += kStreamUnroll * stride) {
    u32x4 v[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) v[u] = __builtin_nontemporal_load(src + i + u * stride);
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) __builtin_nontemporal_store(v[u], dst + i + u * stride);
  }
  for (; i < vectors; i += stride) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

__global__ __launch_bounds__(kStreamBlock) void stream_read_kernel(const u32x4 *__restrict__ src,
                                                                  long long vectors, unsigned *__restrict__ sink) {
  const long long stride = static_cast<long long>(gridDim.x) * kStreamBlock;
  long long i = static_cast<long long>(blockIdx.x) * kStreamBlock + threadIdx.x;
  unsigned acc = 0;
  for (; i + (kStreamUnroll - 1) * stride < vectors; i += kStreamUnroll * stride) {
    u32x4 v[kStreamUnroll];
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) v[u] = __builtin_nontemporal_load(src + i + u * stride);
#pragma unroll
    for (int u = 0; u < kStreamUnroll; ++u) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
  }
  for (; i < vectors; i += stride) {
    const u32x4 v = __builtin_nontemporal_load(src + i);
    acc ^= v.x ^ v.y ^ v.z ^ v.w;
  }
  // the data is all zero, so nothing is ever stored; the test keeps the loads alive
  if (acc == 0x9e3779b9u) sink[0] = acc;
}

__global__ __launch_bounds__(kStreamBlock) void stream_write_kernel(u32x4 *__restrict__ dst, long long vectors,
                                                                   unsigned value) {
  const long long stride = static_cast<long long>(gridDim.x) * kStreamBlock;
  const u32x4 v = {value, value, value, value};
  for (long long i = static_cast<long long>(blockIdx.x) * kStreamBlock + threadIdx.x; i < vectors; i += stride) {
    __builtin_nontemporal_store(v, dst + i);
  }
}

static void profile_clear() {
  for (auto &m : g_marks) g_event_pool.push_back(m.second);
  g_marks.clear();
}

}  // namespace mnt

using namespace mnt;

extern "C" {

int mnt_abi_version(void) { return 1; }

const char *mnt_last_error(void) { return g_last_error.c_str(); }

int mnt_buffer_preallocate(void *stream, size_t bytes) {
  return guarded([&] { Arena::of(static_cast<hipStream_t>(stream)).preallocate(bytes); });
}

int mnt_buffer_free(void *stream) {
  return guarded([&] { Arena::of(static_cast<hipStream_t>(stream)).free_all(); });
}

int mnt_buffer_set_growth(void *stream, float growth) {
  return guarded([&] { Arena::of(static_cast<hipStream_t>(stream)).set_growth(growth); });
}

int mnt_buffer_set_page_size(void *stream, size_t bytes) {
  return guarded([&] { Arena::of(static_cast<hipStream_t>(stream)).set_page_size(bytes); });
}

size_t mnt_buffer_total_size(void *stream) {
  size_t value = 0;
  guarded([&] { value = Arena::of(static_cast<hipStream_t>(stream)).total(); });
  return value;
}

size_t mnt_buffer_used_size(void *stream) {
  size_t value = 0;
  guarded([&] { value = Arena::of(static_cast<hipStream_t>(stream)).used(); });
  return value;
}

int mnt_stream_acquire(void *stream) {
  return guarded([&] { Arena::pin(static_cast<hipStream_t>(stream)); });
}

int mnt_stream_release(void *stream) {
  return guarded([&] { Arena::unpin(static_cast<hipStream_t>(stream)); });
}

int mnt_time_memory(int kind, size_t bytes, int repeats, float *ms_out, void *stream_) {
  return guarded([&] {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MNT_CHECK(kind >= 0 && kind <= 2, "kind must be 0 (copy), 1 (read) or 2 (write), found %d", kind);
    MNT_CHECK(bytes >= 4096 && bytes % 16 == 0 && bytes <= (size_t(64) << 30), "bytes = %zu out of range", bytes);
    MNT_CHECK(repeats >= 1 && repeats <= 1000 && ms_out != nullptr, "bad argument");
    Scope scope(stream);
    const long long vectors = static_cast<long long>(bytes / 16);
    u32x4 *a = scope.alloc<u32x4>(vectors);
    u32x4 *b = kind == 0 ? scope.alloc<u32x4>(vectors) : nullptr;
    unsigned *sink = scope.alloc<unsigned>(4);
    // enough workgroups to keep every compute unit's load queues full, few
    // enough that each lane streams a long run
    const unsigned grid = static_cast<unsigned>(compute_units()) * 16u;
    stream_write_kernel<<<grid, kStreamBlock, 0, stream>>>(a, vectors, 0u);          // also faults the pages in
    if (b != nullptr) stream_write_kernel<<<grid, kStreamBlock, 0, stream>>>(b, vectors, 0u);
    auto once = [&] {
      if (kind == 0) stream_copy_kernel<<<grid, kStreamBlock, 0, stream>>>(a, b, vectors);
      else if (kind == 1) stream_read_kernel<<<grid, kStreamBlock, 0, stream>>>(a, vectors, sink);
      else stream_write_kernel<<<grid, kStreamBlock, 0, stream>>>(a, vectors, 1u);
    };
    once();
    check_launch("stream kernel");
    hipEvent_t start, stop;
    MNT_HIP(hipEventCreate(&start));
    MNT_HIP(hipEventCreate(&stop));
    MNT_HIP(hipEventRecord(start, stream));
    for (int r = 0; r < repeats; ++r) once();
    MNT_HIP(hipEventRecord(stop, stream));
    hipError_t status = hipEventSynchronize(stop);
    float ms = 0.0f;
    if (status == hipSuccess) status = hipEventElapsedTime(&ms, start, stop);
    (void)hipEventDestroy(start);
    (void)hipEventDestroy(stop);
    MNT_HIP(status);
    *ms_out = ms / static_cast<float>(repeats);
  });
}

int mnt_device_facts(int64_t *facts_out, int capacity) {
  return guarded([&] {
    MNT_CHECK(facts_out != nullptr && capacity >= 6, "facts_out needs room for 6 values");
    int device = 0;
    MNT_HIP(hipGetDevice(&device));
    const hipDeviceAttribute_t wanted[5] = {hipDeviceAttributeMultiprocessorCount, hipDeviceAttributeClockRate,
                                            hipDeviceAttributeMemoryClockRate, hipDeviceAttributeMemoryBusWidth,
                                            hipDeviceAttributeL2CacheSize};
    for (int i = 0; i < 5; ++i) {
      int value = 0;
      MNT_HIP(hipDeviceGetAttribute(&value, wanted[i], device));
      facts_out[i] = value;
    }
    size_t free_bytes = 0, total_bytes = 0;
    MNT_HIP(hipMemGetInfo(&free_bytes, &total_bytes));
    facts_out[5] = static_cast<int64_t>(total_bytes);
  });
}

int mnt_profile_enable(int on) {
  return guarded([&] {
    profile_clear();
    g_profile_thread = std::this_thread::get_id();
    g_profile_on = on != 0;
  });
}

int mnt_profile_read(int capacity, float *ms_out, char *labels_out, int label_stride,
                     int *count_out) {
  return guarded([&] {
    MNT_CHECK(ms_out != nullptr && labels_out != nullptr && count_out != nullptr && label_stride > 1,
              "bad argument");
    int count = 0;
    if (!g_marks.empty()) MNT_HIP(hipEventSynchronize(g_marks.back().second));
    for (size_t i = 1; i < g_marks.size() && count < capacity; ++i) {
      float ms = 0.0f;
      MNT_HIP(hipEventElapsedTime(&ms, g_marks[i - 1].second, g_marks[i].second));
      ms_out[count] = ms;
      snprintf(labels_out + static_cast<size_t>(count) * label_stride, label_stride, "%s",
               g_marks[i].first);
      ++count;
    }
    *count_out = count;
    profile_clear();
  });
}

int mnt_reset_error(void) {
  (void)hipGetLastError();
  g_last_error.clear();
  return 0;
}

int mnt_host_wait_stats(int64_t *waits_out, int64_t *nanoseconds_out, int reset) {
  return guarded([&] {
    if (waits_out != nullptr) *waits_out = g_host_waits.load(std::memory_order_relaxed);
    if (nanoseconds_out != nullptr) *nanoseconds_out = g_host_wait_ns.load(std::memory_order_relaxed);
    if (reset) {
      g_host_waits.store(0, std::memory_order_relaxed);
      g_host_wait_ns.store(0, std::memory_order_relaxed);
    }
  });
}

int mnt_device_reset(void) {
  return guarded([&] {
    if (mnt_lookahead_finish(nullptr) != 0) throw Error{mnt_last_error()};
    MNT_HIP(hipDeviceSynchronize());
    Arena::reset_device();
    (void)hipGetLastError();
    g_last_error.clear();
  });
}

}  // extern "C"
