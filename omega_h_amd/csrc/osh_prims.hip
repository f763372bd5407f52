// Stream-ordered primitives: offset scans, compaction, fills, reductions and
// the stable tuple sort used when building meshes.
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cstring>

#include "osh_runtime.hpp"

// Scratch of the scans that allocate nothing (offset_scans_noalloc): the
// tile status words of up to kNoAllocTiles tiles, then the tile ticket
// counter.  Each GPU holds its own copy (128 KiB) for the life of the
// process; host code reaches it only through the address that
// hipGetSymbolAddress returns for the current device.
static constexpr unsigned kNoAllocTiles = 16384;
static __device__ __align__(256) unsigned long long scratch[kNoAllocTiles + 1];

namespace osh {

std::size_t Pool::round_up(std::size_t bytes) {
  if (bytes <= 256) return 256;
  int lg = 63 - __builtin_clzll(bytes - 1);  // 2^lg < bytes <= 2^(lg+1)
  std::size_t step = std::size_t(1) << (lg - 1);
  return (bytes + step - 1) / step * step;
}

void* Pool::get(std::size_t bytes) {
  std::size_t size = round_up(bytes);
  {
    std::lock_guard<std::mutex> g(mu_);
    auto it = free_.find(size);
    if (it != free_.end() && !it->second.empty()) {
      void* p = it->second.back();
      it->second.pop_back();
      cached_ -= size;
      return p;
    }
  }
  void* p = nullptr;
  if (hipMalloc(&p, size) != hipSuccess) {
    (void)hipGetLastError();
    release_all();
    OSH_HIP(hipMalloc(&p, size));
  }
  return p;
}

// Over the cap the largest cached blocks go first: those of a mesh that has
// shrunk since would otherwise fill the cache for good, and every later array
// would be allocated and freed by the runtime (5.2 s instead of 0.75 s for an
// adapt of 24.6 M tets that ends with 0.5 M).
void Pool::put(void* p, std::size_t bytes) {
  std::size_t size = round_up(bytes);
  std::vector<void*> out;
  {
    std::lock_guard<std::mutex> g(mu_);
    while (!closed_ && cached_ + size > cap_) {
      std::size_t most = 0;
      for (auto const& kv : free_)
        if (!kv.second.empty() && kv.first > most) most = kv.first;
      if (most <= size) break;
      out.push_back(free_[most].back());
      free_[most].pop_back();
      cached_ -= most;
    }
    if (!closed_ && cached_ + size <= cap_) {
      free_[size].push_back(p);
      cached_ += size;
      p = nullptr;
    }
  }
  for (void* q : out) (void)hipFree(q);
  if (p) (void)hipFree(p);
}

void Pool::release_all() {
  std::unordered_map<std::size_t, std::vector<void*>> blocks;
  {
    std::lock_guard<std::mutex> g(mu_);
    blocks.swap(free_);
    cached_ = 0;
  }
  for (auto& kv : blocks)
    for (void* p : kv.second) (void)hipFree(p);
}

Ctx::Ctx() : pool(std::make_shared<Pool>()) {
  OSH_HIP(hipGetDevice(&device));
  OSH_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  OSH_HIP(hipHostMalloc(&pinned, 8 * kSlots + 192, hipHostMallocDefault));
  std::memset(pinned, 0, 8 * kSlots + 192);
  OSH_HIP(hipMalloc((void**)&words, sizeof(unsigned) * kWords));
  unsigned none[kWords] = {0};
  OSH_HIP(hipMemcpy(words, none, sizeof(none), hipMemcpyHostToDevice));
  OSH_HIP(hipHostMalloc((void**)&partials, sizeof(Partial) * kPartials, hipHostMallocDefault));
  std::memset(partials, 0, sizeof(Partial) * kPartials);
  OSH_HIP(hipMalloc((void**)&tile_counter, sizeof(unsigned)));
  OSH_HIP(hipMalloc((void**)&tile_sums, sizeof(LO) * kScanTiles * kMaxScanJobs));
  unsigned zero = 0;
  OSH_HIP(hipMemcpy(tile_counter, &zero, sizeof(zero), hipMemcpyHostToDevice));
  noalloc_setup(device);
  profile.from_environment();
}

Ctx::~Ctx() {
  if (profile.print_at_close) {
    std::string r = profile.report(profile.chop, profile.percent, profile_now() - profile.origin);
    std::fputs(r.c_str(), stdout);
    std::fflush(stdout);
  }
  if (stream) {
    (void)hipStreamSynchronize(stream);
    (void)hipStreamDestroy(stream);
  }
  if (scan_status) (void)hipFree(scan_status);
  if (tile_counter) (void)hipFree(tile_counter);
  if (tile_sums) (void)hipFree(tile_sums);
  if (words) (void)hipFree(words);
  if (pool) pool->close();
  if (partials) (void)hipHostFree(partials);
  if (pinned) (void)hipHostFree(pinned);
}

void range_begin(Ctx& c, char const* name) {
  if (c.profile.flags & kProfileMarkers) roctxRangePushA(name);
  if (c.profile.flags & kProfileTree) c.profile.start(name, profile_now());
}

void range_end(Ctx& c) {
  // a failed wait is left for the next sync() to report: a range may end
  // while an error unwinds the stack
  if (c.profile.flags & kProfileSync) (void)hipStreamSynchronize(c.stream);
  if (c.profile.flags & kProfileTree) c.profile.stop(profile_now());
  if (c.profile.flags & kProfileMarkers) roctxRangePop();
}

void Ctx::sync() {
  OSH_HIP(hipStreamSynchronize(stream));
  raise_device_error();
}

namespace {

// stores made by the stream's earlier kernels happen before this release
__global__ void signal_kernel(unsigned const* words, unsigned* host_words, unsigned* word,
    unsigned value) {
  for (int i = 0; i < Ctx::kWords; ++i) host_words[i] = words[i];
  __hip_atomic_store(word, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// how long wait() polls before it leaves the core to other threads
constexpr double kPollSeconds = 200e-6;

}  // namespace

// A pass waits for its counts four to six times, each wait with the device
// idle until the host has seen it and launched again.  hipStreamSynchronize
// adds 8 to 30 us to the kernels it waits for (a system-scope barrier packet
// and often an interrupt); a one-thread kernel that stores into pinned memory
// with the host polling that word adds 6 to 8 us.  Scans bring their totals
// with the tag themselves (put_total) and need no such kernel: 0.1 ms of the
// 1.85 ms of the smallest adapt and 1.8 of the 97.6 ms of the 64^3 workload.
void Ctx::wait() {
  hipLaunchKernelGGL(signal_kernel, dim3(1), dim3(1), 0, stream,
      static_cast<unsigned const*>(words), host_words(), signal_word(), wait_tag());
  OSH_HIP(hipGetLastError());
  wait_signalled();
}

template <class Arrived>
void Ctx::poll(Arrived const& arrived) {
  double limit = 0.0;
  for (unsigned polls = 1;; ++polls) {
    if (arrived()) {
      raise_device_error();
      return;
    }
    __builtin_ia32_pause();
    if (polls % 64 == 0) {
      double t = profile_now();
      if (limit == 0.0) limit = t + kPollSeconds;
      if (t > limit) break;
    }
  }
  sync();
}

void Ctx::wait_signalled() {
  unsigned value = signal_value = wait_tag();
  unsigned* word = signal_word();
  poll([=] { return __atomic_load_n(word, __ATOMIC_ACQUIRE) == value; });
}

void Ctx::wait_totals(unsigned slots) {
  unsigned tag = signal_value = wait_tag();
  unsigned long long const* words = static_cast<unsigned long long const*>(pinned);
  auto arrived = [=] {
    for (int i = 0; i < kSlots; ++i)
      if (((slots >> i) & 1u) && unsigned(__atomic_load_n(words + i, __ATOMIC_ACQUIRE) >> 32) != tag)
        return false;
    return true;
  };
  poll(arrived);
  OSH_CHECK(arrived(), "a scan's total is missing");
}

void Ctx::wait_partials(int n) {
  unsigned long long tag = signal_value = wait_tag();
  Partial const* a = partials;
  auto arrived = [=] {
    for (int i = 0; i < n; ++i)
      if (__atomic_load_n(&a[i].tag, __ATOMIC_ACQUIRE) != tag) return false;
    return true;
  };
  poll(arrived);
  OSH_CHECK(arrived(), "a reduction's result is missing");
}

void Ctx::raise_device_error() {
  int* err = error_word();
  if (*err != kNoError) {
    int code = *err;
    *err = kNoError;
    if (code == kReflectDownNoMatch) throw Error(kNoMatchMessage);
    if (code == kScanTimeout) throw Error("scan: a tile waited too long for its predecessor");
    if (code == kScanTicket) throw Error("scan: tile tickets out of step");
    if (code == kKeyWithoutUp) throw Error("modify: a key entity has no adjacent entity above it");
    if (code == kNonManifoldSide) throw Error("a side has more than two elements");
    if (code == kBrokenSwapLoop)
      throw Error("swap: the elements around an edge do not close a loop");
    if (code == kBadPart) throw Error("split: a vertex without a valid part number");
    if (code == kFlipNormals)
      throw Error("prevent_coarsen_flip: too many exposed sides at a vertex, or no most normal "
                  "normal");
    if (code == kZeroSizeCavity)
      throw Error("conservation: an integral error in a cavity of zero size");
    if (code == kPolytopeOverflow)
      throw Error("conservation: a simplex intersection left the polytope buffer");
    if (code == kDegenerateEigen)
      throw Error("eigen: no eigenvector for a simple eigenvalue (degenerate metric)");
    throw Error("device error " + std::to_string(code));
  }
}

namespace {

constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;  // 4096 values per block
constexpr int kWave = 64;

// both with every lane active: the lane before takes part in the addition itself
// (row_shr 1, 2, 4, 8, then the last lanes of rows 0 and 2 and of rows 0-1)
__device__ __forceinline__ LO wave_inclusive_scan(LO v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

__device__ __forceinline__ LO wave_sum(LO v) {
  return __builtin_amdgcn_readlane(wave_inclusive_scan(v), kWave - 1);
}

// Block-wide exclusive scan of one value per thread; returns the block total.
__device__ __forceinline__ LO block_exclusive_scan(LO v, LO* total) {
  __shared__ LO wave_sums[kBlock / kWave];
  int lane = threadIdx.x & (kWave - 1);
  int wave = threadIdx.x / kWave;
  LO inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) wave_sums[wave] = inc;
  __syncthreads();
  LO before = 0;
  LO sum = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    LO s = wave_sums[w];
    if (w < wave) before += s;
    sum += s;
  }
  __syncthreads();
  *total = sum;
  return before + inc - v;
}

template <class T>
__global__ void fill_kernel(LO n, T* out, T value) {
  LO i = thread_index();
  if (i < n) out[i] = value;
}

// Single-pass exclusive scan with decoupled look-back.  Each workgroup of a
// multi-tile scan takes the next tile ticket from a counter (so every tile it
// waits on belongs to a workgroup that is already running), scans its 4096
// values and publishes its aggregate; its first wave then reads the words of
// the 64 preceding tiles at once, one per lane, and adds the aggregates back
// to the nearest inclusive prefix, moving the window back 64 tiles at a time
// until it meets one.  A status word is [epoch:24 | flag:8 | value:32]; the
// epoch changes every scan, so words left by earlier scans read as "not yet
// published" and no clearing pass is needed.  The word carries the value
// itself, so relaxed agent-scope atomics suffice.  A wait that outlasts
// kSpinLimit polls (it cannot happen on a correct schedule) stops, sets the
// context's error word and lets every workgroup finish; the next stream sync
// raises it.  Values pass through LDS so that global loads and stores are
// coalesced while each thread scans 16 consecutive values; LDS index
// j + j/16 keeps both access patterns free of bank conflicts.
constexpr unsigned kFlagAggregate = 1u;
constexpr unsigned kFlagInclusive = 2u;
constexpr unsigned kSpinLimit = 1u << 20;

__device__ __forceinline__ unsigned long long status_word(unsigned epoch, unsigned flag, LO v) {
  return (static_cast<unsigned long long>(epoch) << 40) |
         (static_cast<unsigned long long>(flag) << 32) | static_cast<unsigned>(v);
}

// the exclusive prefix of `tile` from its predecessors' status words; run by
// the 64 lanes of one wave, returns the same value in every lane
__device__ __forceinline__ LO look_back(unsigned long long* status, unsigned tile,
    unsigned epoch, int* error) {
  int lane = threadIdx.x & (kWave - 1);
  LO prefix = 0;
  long long window = static_cast<long long>(tile) - 1;  // the tile lane 0 reads
  unsigned spins = 0;
  for (;;) {
    long long j = window - lane;
    unsigned long long w = status_word(epoch, kFlagInclusive, 0);  // before tile 0
    if (j >= 0) w = __hip_atomic_load(&status[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned flag = unsigned(w >> 32) & 0xffu;
    bool ready = unsigned(w >> 40) == epoch && flag != 0;
    if (__ballot(!ready) != 0ull) {
      if (++spins > kSpinLimit) {
        if (lane == 0) *error = kScanTimeout;
        return prefix;
      }
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    LO v = LO(unsigned(w));
    unsigned long long inclusive = __ballot(flag == kFlagInclusive);
    if (inclusive != 0ull) {
      int nearest = __ffsll(static_cast<long long>(inclusive)) - 1;
      if (lane > nearest) v = 0;
      return prefix + wave_sum(v);
    }
    prefix += wave_sum(v);
    window -= kWave;
  }
}

// up to kMaxScanJobs independent scans share one launch: job j owns the
// tiles [first[j], first[j + 1]) of the launch and the same range of status
// words, so its look-back never leaves its own tiles
struct ScanBatch {
  struct Job {
    void const* in;
    LO* out;
    LO* list;
    unsigned long long* total;
    LO n;
    int kind;
  };
  // a job's arguments are one load
  Job job[kMaxScanJobs];
  unsigned first[kMaxScanJobs + 1];
  int count;
  unsigned tag;
};

// a grand total goes to its pinned slot as one word with the tag that the host
// polls for, so that a scan ends its own wait: no order among the totals, and
// no kernel after the scan, is needed
__device__ __forceinline__ void put_total(unsigned long long* slot, unsigned tag, LO total) {
  if (slot)
    __hip_atomic_store(slot,
        (static_cast<unsigned long long>(tag) << 32) | static_cast<unsigned>(total),
        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ LO scan_input(void const* in, int kind, LO i) {
  if (kind == kScanLO) return static_cast<LO const*>(in)[i];
  return LO(static_cast<I8 const*>(in)[i] != 0);
}

// without tickets (every job one tile) a workgroup's tile is its index
__global__ void __launch_bounds__(kBlock) scan_lookback(ScanBatch b,
    unsigned long long* status, unsigned* tile_counter, unsigned ticket_base, int tickets,
    unsigned epoch, int* error) {
  __shared__ LO s_vals[kScanTile + kScanTile / 16];
  __shared__ unsigned s_tile;
  __shared__ LO s_prefix;
  if (tickets) {
    if (threadIdx.x == 0) s_tile = atomicAdd(tile_counter, 1u) - ticket_base;
    __syncthreads();
  }
  unsigned t = tickets ? s_tile : blockIdx.x;
  if (t >= gridDim.x) {  // the ticket base is out of step: refuse to write
    if (threadIdx.x == 0) *error = kScanTicket;
    return;
  }
  int job = 0;
  while (job + 1 < b.count && t >= b.first[job + 1]) ++job;
  unsigned tile = t - b.first[job];
  unsigned ntiles = b.first[job + 1] - b.first[job];
  LO n = b.job[job].n;
  int kind = b.job[job].kind;
  void const* in = b.job[job].in;
  LO* out = b.job[job].out;
  LO* list = b.job[job].list;
  unsigned long long* st = status + b.first[job];
  LO tile_base = LO(tile) * kScanTile;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int j = k * kBlock + int(threadIdx.x);
    LO i = tile_base + j;
    s_vals[j + (j >> 4)] = (i < n) ? scan_input(in, kind, i) : 0;
  }
  __syncthreads();
  int row = int(threadIdx.x) * (kScanItems + 1);  // padded index of value 16 * threadIdx.x
  LO vals[kScanItems];
  LO acc = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    acc += s_vals[row + k];
    vals[k] = acc;
  }
  LO total;
  LO excl = block_exclusive_scan(acc, &total);
  if (threadIdx.x < kWave) {
    LO prefix = 0;
    if (tile != 0) {
      if (threadIdx.x == 0)
        __hip_atomic_store(&st[tile], status_word(epoch, kFlagAggregate, total),
            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      prefix = look_back(st, tile, epoch, error);
    }
    if (threadIdx.x == 0) {
      if (ntiles > 1)
        __hip_atomic_store(&st[tile], status_word(epoch, kFlagInclusive, prefix + total),
            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_prefix = prefix;
      if (tile == 0 && out) out[0] = 0;
      if (tile == ntiles - 1) put_total(b.job[job].total, b.tag, prefix + total);
    }
  }
  __syncthreads();
  LO prefix = s_prefix + excl;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s_vals[row + k] = prefix + vals[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int j = k * kBlock + int(threadIdx.x);
    LO i = tile_base + j;
    if (i < n) {
      LO inc = s_vals[j + (j >> 4)];
      if (out) out[1 + i] = inc;
      if (list && scan_input(in, kind, i)) list[inc - 1] = i;
    }
  }
}

// Scans of moderate jobs take two launches instead: one sums each tile, the
// next scans each tile behind the sum of its job's earlier tile sums, which
// every workgroup adds up for itself.  A look-back has to carry the prefix
// from workgroup to workgroup across the XCDs, a device-scope round trip at
// a time: 10 us from two tiles on, 21 us at 542, against 7.4 us for the two
// launches.  Jobs of one tile of 1024, 4096 or 16384 values need only the second
// launch, with 256 threads or, for the largest, 1024; in moderate jobs
// (kOwnTiles) each workgroup adds up the values in front of its tile itself,
// from L2, which costs less than the first launch.
//
// Small scans are bound by the chain of latencies from the arguments to the
// stores.  A job's arguments are one load, a workgroup of a one-tile job knows
// its job from its index, the lanes add with DPP moves instead of LDS
// permutes, and every wave scans the partial sums itself behind one barrier:
// 2.65 us for up to 1024 values, 3.3 for 4096 and 4.0 for 16384, against 5.7,
// 5.7 and 6.5 before.
//
// A thread takes four consecutive values per round (one 16-byte load, or one
// 4-byte load of byte values, where the array is so aligned) and writes the
// four offsets in front of them, so loads and stores are wide and coalesced
// without a pass through LDS.
template <int BLOCK, int ROUNDS>
struct TileScan {
  static constexpr int kWaves = BLOCK / kWave;
  static constexpr int kParts = ROUNDS * kWaves;
  static constexpr int kTile = BLOCK * ROUNDS * 4;
  static_assert(kParts <= kWave, "one wave scans the partial sums");
};

__device__ __forceinline__ void load_four(void const* in, int kind, LO i, LO n, bool wide,
    LO* v) {
  if (wide && i + 4 <= n) {
    if (kind == kScanLO) {
      int4 q = *reinterpret_cast<int4 const*>(static_cast<LO const*>(in) + i);
      v[0] = q.x;
      v[1] = q.y;
      v[2] = q.z;
      v[3] = q.w;
    } else {
      char4 q = *reinterpret_cast<char4 const*>(static_cast<I8 const*>(in) + i);
      v[0] = LO(q.x != 0);
      v[1] = LO(q.y != 0);
      v[2] = LO(q.z != 0);
      v[3] = LO(q.w != 0);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = (i + k < n) ? scan_input(in, kind, i + k) : 0;
  }
}

__device__ __forceinline__ bool wide_input(void const* in, int kind) {
  return (reinterpret_cast<std::uintptr_t>(in) & (kind == kScanLO ? 15u : 3u)) == 0;
}

__device__ __forceinline__ int job_of(ScanBatch const& b, unsigned t) {
  int job = 0;
  while (job + 1 < b.count && t >= b.first[job + 1]) ++job;
  return job;
}

constexpr int kSumBlock = 256;
constexpr int kSumRounds = 2;
constexpr int kSumTile = TileScan<kSumBlock, kSumRounds>::kTile;
constexpr int kLeastTile = TileScan<kSumBlock, 1>::kTile;
constexpr int kOneBlock = 1024;
constexpr int kOneRounds = 4;
constexpr int kOneTile = TileScan<kOneBlock, kOneRounds>::kTile;
// every workgroup reads its job's earlier tile sums: up to this many tiles
// (16.7 M values) that costs less than the look-back's chain
constexpr unsigned kMaxSumTiles = Ctx::kScanTiles;
// a workgroup of the one-launch form reads at most this many tiles of 4096
// values, and all of a launch at most kOwnBytes: at up to 16 tiles it takes 6
// us against 7.4 us for the two launches and 10 us for the look-back, at 32
// tiles 10 us
constexpr int kOwnTile = TileScan<kOneBlock, 1>::kTile;
static_assert(kOwnTile == TileScan<kSumBlock, 4>::kTile && kOneTile == 4 * kOwnTile, "one tile");
constexpr unsigned kOwnTiles = 16;
constexpr double kOwnBytes = 8e6;

__global__ void __launch_bounds__(kSumBlock) sum_tiles(ScanBatch b, LO* sums) {
  unsigned t = blockIdx.x;
  int job = job_of(b, t);
  ScanBatch::Job a = b.job[job];
  LO base = LO(t - b.first[job]) * kSumTile;
  bool wide = wide_input(a.in, a.kind);
  LO acc = 0;
#pragma unroll
  for (int r = 0; r < kSumRounds; ++r) {
    LO v[4];
    load_four(a.in, a.kind, base + (r * kSumBlock + LO(threadIdx.x)) * 4, a.n, wide, v);
    acc += (v[0] + v[1]) + (v[2] + v[3]);
  }
  __shared__ LO part[kSumBlock / kWave];
  acc = wave_sum(acc);
  if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    LO s = 0;
    for (int w = 0; w < kSumBlock / kWave; ++w) s += part[w];
    sums[t] = s;
  }
}

// How a workgroup knows what lies in front of its tile: kOnly, nothing does,
// every job being one tile; kSums, from the tile sums; kOwn, by adding up its
// job's earlier values itself.
enum ScanBefore { kOnly, kSums, kOwn };

template <int BLOCK, int ROUNDS, ScanBefore BEFORE>
__global__ void __launch_bounds__(BLOCK) scan_tiles(ScanBatch b, LO const* sums) {
  using T = TileScan<BLOCK, ROUNDS>;
  __shared__ LO part[T::kParts];
  __shared__ LO before[T::kWaves];
  unsigned t = blockIdx.x;
  int job = BEFORE == kOnly ? int(t) : job_of(b, t);
  ScanBatch::Job a = b.job[job];
  unsigned tile = BEFORE == kOnly ? 0u : t - b.first[job];
  bool last = BEFORE == kOnly || t + 1 == b.first[job + 1];
  LO n = a.n;
  int lane = int(threadIdx.x) & (kWave - 1);
  int wave = int(threadIdx.x) / kWave;
  LO base = LO(tile) * T::kTile;
  bool wide = wide_input(a.in, a.kind);
  LO v[ROUNDS][4];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r)
    load_four(a.in, a.kind, base + (r * BLOCK + LO(threadIdx.x)) * 4, n, wide, v[r]);
  if constexpr (BEFORE != kOnly) {
    LO earlier = 0;
    if constexpr (BEFORE == kOwn) {
      // whole tiles, all in range
#pragma unroll 4
      for (LO i = LO(threadIdx.x) * 4; i < base; i += BLOCK * 4) {
        LO u[4];
        load_four(a.in, a.kind, i, n, wide, u);
        earlier += (u[0] + u[1]) + (u[2] + u[3]);
      }
    } else {
      for (unsigned j = threadIdx.x; j < tile; j += BLOCK) earlier += sums[b.first[job] + j];
    }
    if (tile) earlier = wave_sum(earlier);
    if (lane == 0) before[wave] = earlier;
  }
  LO inc[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    inc[r] = wave_inclusive_scan((v[r][0] + v[r][1]) + (v[r][2] + v[r][3]));
    if (lane == kWave - 1) part[r * T::kWaves + wave] = inc[r];
  }
  __syncthreads();
  // every wave scans the partial sums for itself
  LO p = lane < T::kParts ? part[lane] : 0;
  LO i = wave_inclusive_scan(p);
  LO prefix = 0;
  if constexpr (BEFORE != kOnly) prefix = wave_sum(lane < T::kWaves ? before[lane] : 0);
  LO total = prefix + __builtin_amdgcn_readlane(i, kWave - 1);
  if (last && threadIdx.x == 0) {
    if (a.out) a.out[n] = total;
    put_total(a.total, b.tag, total);
  }
  i += prefix - p;
  LO* out = a.out;
  LO* list = a.list;
  bool wide_out = (reinterpret_cast<std::uintptr_t>(out) & 15u) == 0;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    LO at = base + (r * BLOCK + LO(threadIdx.x)) * 4;
    LO o0 = __builtin_amdgcn_readlane(i, __builtin_amdgcn_readfirstlane(r * T::kWaves + wave)) +
            inc[r] - ((v[r][0] + v[r][1]) + (v[r][2] + v[r][3]));
    LO o1 = o0 + v[r][0], o2 = o1 + v[r][1], o3 = o2 + v[r][2];
    if (list) {
      // values past the end are 0
      if (v[r][0]) list[o0] = at;
      if (v[r][1]) list[o1] = at + 1;
      if (v[r][2]) list[o2] = at + 2;
      if (v[r][3]) list[o3] = at + 3;
    }
    if (!out) continue;
    if (wide_out && at + 4 <= n) {
      *reinterpret_cast<int4*>(out + at) = make_int4(o0, o1, o2, o3);
    } else {
      if (at < n) out[at] = o0;
      if (at + 1 < n) out[at + 1] = o1;
      if (at + 2 < n) out[at + 2] = o2;
      if (at + 3 < n) out[at + 3] = o3;
    }
  }
}

__global__ void zero_u64(LO n, unsigned long long* a) {
  LO i = thread_index();
  if (i < n) a[i] = 0ull;
}

// the context's tile status words, grown (and cleared) when a scan needs
// more tiles than they hold; a new epoch per scan, with a clearing pass
// before the 24-bit epoch field would overflow (epochs run 1 .. 2^24 - 1;
// cleared words carry epoch 0)
unsigned long long* scan_status_words(Ctx& c, LO ntiles, unsigned* epoch) {
  if (ntiles > c.scan_status_cap || c.scan_epoch >= Ctx::kMaxScanEpoch) {
    LO cap = ntiles > c.scan_status_cap ? (ntiles > 2 * c.scan_status_cap ? ntiles
                                                                          : 2 * c.scan_status_cap)
                                        : c.scan_status_cap;
    if (cap != c.scan_status_cap) {
      if (c.scan_status) OSH_HIP(hipStreamSynchronize(c.stream));
      if (c.scan_status) (void)hipFree(c.scan_status);
      c.scan_status = nullptr;
      OSH_HIP(hipMalloc(&c.scan_status, sizeof(unsigned long long) * std::size_t(cap)));
      c.scan_status_cap = cap;
    }
    OSH_LAUNCH(zero_u64, cap, c, static_cast<unsigned long long*>(c.scan_status));
    c.scan_epoch = 0;
  }
  *epoch = ++c.scan_epoch;
  return static_cast<unsigned long long*>(c.scan_status);
}

}  // namespace

namespace {

// the jobs as a batch in tiles of `tile` values; returns the tile count and
// the largest job's in *most
unsigned batch_jobs(ScanJob const* jobs, int njobs, int tile, ScanBatch& b, unsigned* most) {
  unsigned tiles = 0;
  *most = 0;
  for (int j = 0; j < njobs; ++j) {
    OSH_CHECK(jobs[j].n >= 0 && (jobs[j].out || jobs[j].list), "offset_scans: bad job");
    b.job[j] = {jobs[j].in, jobs[j].out, jobs[j].list, jobs[j].total, jobs[j].n, jobs[j].kind};
    // a value of another kind left in the slot could look like the coming tag
    if (jobs[j].total) __atomic_store_n(jobs[j].total, 0ull, __ATOMIC_RELAXED);
    b.first[j] = tiles;
    // an empty job still takes one tile, which writes its 0 and its total
    unsigned nt = jobs[j].n == 0 ? 1u : unsigned((std::int64_t(jobs[j].n) + tile - 1) / tile);
    *most = nt > *most ? nt : *most;
    tiles += nt;
  }
  b.first[njobs] = tiles;
  b.count = njobs;
  return tiles;
}

}  // namespace

void offset_scans(Ctx& c, ScanJob const* jobs, int njobs) {
  OSH_CHECK(njobs >= 1 && njobs <= kMaxScanJobs, "offset_scans: 1 to 12 jobs per launch");
  ScanBatch b{};
  b.tag = c.wait_tag();
  unsigned most = 0;
  unsigned tiles = batch_jobs(jobs, njobs, kOwnTile, b, &most);
  if (most <= 1) {
    LO n = 0;
    for (int j = 0; j < njobs; ++j) n = jobs[j].n > n ? jobs[j].n : n;
    if (n <= kLeastTile)
      hipLaunchKernelGGL((scan_tiles<kSumBlock, 1, kOnly>), dim3(tiles), dim3(kSumBlock), 0,
          c.stream, b, (LO const*)nullptr);
    else
      hipLaunchKernelGGL((scan_tiles<kSumBlock, 4, kOnly>), dim3(tiles), dim3(kSumBlock), 0,
          c.stream, b, (LO const*)nullptr);
    OSH_HIP(hipGetLastError());
    return;
  }
  if (most <= 4) {
    tiles = batch_jobs(jobs, njobs, kOneTile, b, &most);
    hipLaunchKernelGGL((scan_tiles<kOneBlock, kOneRounds, kOnly>), dim3(tiles), dim3(kOneBlock),
        0, c.stream, b, (LO const*)nullptr);
    OSH_HIP(hipGetLastError());
    return;
  }
  if (most <= kOwnTiles) {
    double read = 0.0;
    for (int j = 0; j < njobs; ++j) {
      double nt = double(b.first[j + 1] - b.first[j]);
      read += 0.5 * nt * nt * kOwnTile * (jobs[j].kind == kScanLO ? 4.0 : 1.0);
    }
    if (read <= kOwnBytes) {
      hipLaunchKernelGGL((scan_tiles<kOneBlock, 1, kOwn>), dim3(tiles), dim3(kOneBlock), 0,
          c.stream, b, (LO const*)nullptr);
      OSH_HIP(hipGetLastError());
      return;
    }
  }
  tiles = batch_jobs(jobs, njobs, kSumTile, b, &most);
  if (most <= kMaxSumTiles) {
    LO* sums = c.tile_sums;
    hipLaunchKernelGGL(sum_tiles, dim3(tiles), dim3(kSumBlock), 0, c.stream, b, sums);
    OSH_HIP(hipGetLastError());
    hipLaunchKernelGGL((scan_tiles<kSumBlock, kSumRounds, kSums>), dim3(tiles), dim3(kSumBlock), 0,
        c.stream, b, static_cast<LO const*>(sums));
    OSH_HIP(hipGetLastError());
    return;
  }
  tiles = batch_jobs(jobs, njobs, kScanTile, b, &most);
  unsigned epoch = 0;
  unsigned ticket_base = c.tile_tickets;
  unsigned long long* status = scan_status_words(c, LO(tiles), &epoch);
  c.tile_tickets += tiles;
  hipLaunchKernelGGL(scan_lookback, dim3(tiles), dim3(kBlock), 0, c.stream, b, status,
      c.tile_counter, ticket_base, 1, epoch, c.error_word());
  OSH_HIP(hipGetLastError());
}

namespace {

// per device: the address of its `scratch`, and the epoch and ticket count
// of the scans made in it so far
struct NoAllocDevice {
  unsigned long long* words = nullptr;
  unsigned epoch = 0;
  unsigned tickets = 0;
  bool cleared = false;
};
constexpr int kMaxNoAllocDevices = 64;
std::mutex noalloc_mu;
NoAllocDevice noalloc_devices[kMaxNoAllocDevices];

}  // namespace

void noalloc_setup(int device) {
  OSH_CHECK(device >= 0 && device < kMaxNoAllocDevices, "device number out of range");
  std::lock_guard<std::mutex> g(noalloc_mu);
  NoAllocDevice& d = noalloc_devices[device];
  if (d.words) return;
  void* p = nullptr;
  OSH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  OSH_CHECK(p != nullptr, "no device address for the scan scratch");
  d.words = static_cast<unsigned long long*>(p);
}

void offset_scans_noalloc(Ctx& c, ScanJob const* jobs, int njobs) {
  OSH_CHECK(njobs >= 1 && njobs <= kMaxScanJobs, "offset_scans: 1 to 12 jobs per launch");
  ScanBatch b{};
  std::int64_t tiles = 0;
  bool multi = false;
  for (int j = 0; j < njobs; ++j) {
    OSH_CHECK(jobs[j].n >= 0 && jobs[j].out, "offset_scans: bad job");
    b.job[j] = {jobs[j].in, jobs[j].out, nullptr, jobs[j].total, jobs[j].n, jobs[j].kind};
    b.first[j] = unsigned(tiles);
    std::int64_t nt = jobs[j].n == 0 ? 1 : (std::int64_t(jobs[j].n) + kScanTile - 1) / kScanTile;
    multi = multi || nt > 1;
    tiles += nt;
    OSH_CHECK(tiles <= std::int64_t(kNoAllocTiles),
        "offset_scans_noalloc: more than 16384 tiles of 4096 values in one call");
  }
  b.first[njobs] = unsigned(tiles);
  b.count = njobs;
  unsigned epoch = 0, ticket_base = 0;
  unsigned long long* words = nullptr;
  {
    std::lock_guard<std::mutex> g(noalloc_mu);
    OSH_CHECK(c.device >= 0 && c.device < kMaxNoAllocDevices, "device number out of range");
    NoAllocDevice& d = noalloc_devices[c.device];
    OSH_CHECK(d.words, "the scan scratch of this device is not set up");
    words = d.words;
    if (multi) {
      // status words left by earlier scans read as unpublished under a new
      // epoch; before the 24-bit epoch field wraps (and before the first
      // use) a fill kernel clears them
      if (!d.cleared || d.epoch >= Ctx::kMaxScanEpoch) {
        hipLaunchKernelGGL(zero_u64, dim3(nblocks(LO(kNoAllocTiles))), dim3(kBlock), 0,
            c.stream, LO(kNoAllocTiles), words);
        OSH_HIP(hipGetLastError());
        d.epoch = 0;
        d.cleared = true;
      }
      epoch = ++d.epoch;
      ticket_base = d.tickets;
      d.tickets += unsigned(tiles);
    }
  }
  hipLaunchKernelGGL(scan_lookback, dim3(unsigned(tiles)), dim3(kBlock), 0, c.stream, b,
      multi ? words : nullptr, reinterpret_cast<unsigned*>(words + kNoAllocTiles), ticket_base,
      multi ? 1 : 0, epoch, c.error_word());
  OSH_HIP(hipGetLastError());
}

namespace {

__global__ void iota_kernel(LO n, LO* out, LO start, LO stride) {
  LO i = thread_index();
  if (i < n) out[i] = start + i * stride;
}

enum ReduceOp { kMin, kMax };

template <class T>
__host__ __device__ __forceinline__ T combine(int op, T a, T b) {
  if (op == kMin) return (b < a) ? b : a;
  return (a < b) ? b : a;
}

// Reductions: each job's workgroups write their partial results to pinned
// memory, tagged for the host, which polls for the tags and combines the few
// there are.  A second launch for that, and a wait a job, cost a pass 7 us and
// the start of an adapt two more waits.
//
// The host's share grows with the workgroups, so a job has at most 64 until each
// of them has 32 values a thread, and from there up to one a CU (fewer where
// many jobs share the partials).  A call over 12.6 M values takes 28 us with 256
// workgroups and 68 with 64; over 664,000, 12.7 with 64 and 18.4 with 162.
template <class T>
struct ReduceBatch {
  struct Job {
    T const* in;
    LO n;
    LO stride;
    int op;
    unsigned first;
  };
  Job job[kMaxReduceJobs + 1];  // one past the last: where its workgroups end
  int count;
  unsigned tag;
  Ctx::Partial* out;
};
constexpr int kReduceBlock = 1024;
constexpr int kFewValues = kReduceBlock * 4;  // a workgroup's
constexpr unsigned kFewBlocks = 64;
constexpr int kManyValues = kReduceBlock * 32;
constexpr unsigned kManyBlocks = 256;
static_assert(Ctx::kPartials >= kMaxReduceJobs, "a partial for each job");

template <class T, class A>
__global__ void __launch_bounds__(kReduceBlock) reduce_partials(ReduceBatch<T> b, A init_min,
    A init_max) {
  __shared__ A part[kReduceBlock / kWave];
  int w = 0;
  while (w + 1 < b.count && blockIdx.x >= b.job[w + 1].first) ++w;
  typename ReduceBatch<T>::Job a = b.job[w];
  unsigned block = blockIdx.x - a.first, blocks = b.job[w + 1].first - a.first;
  A acc = a.op == kMin ? init_min : init_max;
  std::int64_t step = std::int64_t(blocks) * blockDim.x;
#pragma unroll 4
  for (std::int64_t i = std::int64_t(block) * blockDim.x + threadIdx.x; i < a.n; i += step)
    acc = combine<A>(a.op, acc, A(a.in[i * a.stride]));
  for (int d = kWave / 2; d > 0; d >>= 1) acc = combine<A>(a.op, acc, __shfl_xor(acc, d, kWave));
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (unsigned k = 1; k < blockDim.x / kWave; ++k) acc = combine<A>(a.op, acc, part[k]);
  unsigned long long bits = 0;
  __builtin_memcpy(&bits, &acc, sizeof(A));
  b.out[blockIdx.x].value = bits;
  __hip_atomic_store(&b.out[blockIdx.x].tag, static_cast<unsigned long long>(b.tag),
      __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the reductions of up to kMaxReduceJobs jobs, waited for; an empty one gives
// its init
template <class T, class A>
void reduce(Ctx& c, ReduceBatch<T>& b, A const (&init)[2], A* out) {
  unsigned blocks = 0, share = unsigned(Ctx::kPartials / b.count);
  LO most = 0;
  for (int j = 0; j < b.count; ++j) {
    b.job[j].first = blocks;
    unsigned nb = std::max(std::min(nblocks(b.job[j].n, kFewValues), kFewBlocks),
        std::min(nblocks(b.job[j].n, kManyValues), kManyBlocks));
    blocks += std::min(nb, share);
    most = b.job[j].n > most ? b.job[j].n : most;
  }
  b.job[b.count].first = blocks;
  b.out = c.partials;
  b.tag = c.wait_tag();
  if (blocks) {
    hipLaunchKernelGGL((reduce_partials<T, A>), dim3(blocks),
        dim3(most > kBlock * 4 ? kReduceBlock : kBlock), 0, c.stream, b, init[0], init[1]);
    OSH_HIP(hipGetLastError());
    c.wait_partials(int(blocks));
  }
  for (int j = 0; j < b.count; ++j) {
    out[j] = init[b.job[j].op];
    for (unsigned k = b.job[j].first; k < b.job[j + 1].first; ++k) {
      A v;
      std::memcpy(&v, &c.partials[k].value, sizeof(A));
      out[j] = combine<A>(b.job[j].op, out[j], v);
    }
  }
}

constexpr Real kRealInit[2] = {1.79769313486231570815e+308, -1.79769313486231570815e+308};
constexpr LO kWholeInit[2] = {0x7fffffff, -0x7fffffff - 1};

template <class T, class A>
A reduce_one(Ctx& c, DArray<T> const& a, int op, A const (&init)[2]) {
  ReduceBatch<T> b{};
  b.count = 1;
  b.job[0] = {a.data(), a.size(), 1, op, 0u};
  A out;
  reduce<T, A>(c, b, init, &out);
  return out;
}

}  // namespace

void reduce_reals(Ctx& c, ReduceJob const* jobs, int njobs, Real* out) {
  for (int at = 0; at < njobs; at += kMaxReduceJobs) {
    ReduceBatch<Real> b{};
    for (; b.count < kMaxReduceJobs && at + b.count < njobs; ++b.count) {
      ReduceJob const& j = jobs[at + b.count];
      b.job[b.count] = {j.in, j.n, j.stride, j.max ? kMax : kMin, 0u};
    }
    reduce<Real, Real>(c, b, kRealInit, out + at);
  }
}

LOs offset_scan(Ctx& c, LOs const& counts, LO* total) {
  LOs out(c, counts.size() + 1);
  ScanJob job{counts.data(), kScanLO, counts.size(), out.data(),
      total ? total_slot(c, 0) : nullptr};
  offset_scans(c, &job, 1);
  if (total) *total = scan_total(c, 0);
  return out;
}

LOs collect_marked(Ctx& c, Bytes const& marks) { return collect_marked(c, marks, nullptr); }

LOs collect_marked(Ctx& c, Bytes const& marks, LOs* offsets_out) {
  LO n = marks.size();
  // the scan counts nonzero marks directly and lists them in the same launch,
  // in an array sized for all of them
  LOs out(c, n);
  if (offsets_out) *offsets_out = LOs(c, n + 1);
  ScanJob job{marks.data(), kScanNonzero, n, offsets_out ? offsets_out->data() : nullptr,
      total_slot(c, 0), out.data()};
  if (n == 0) {
    if (offsets_out) *offsets_out = fill_lo(c, 1, 0);
    return out;
  }
  offset_scans(c, &job, 1);
  out.shrink(scan_total(c, 0));
  return out;
}

namespace {

struct FillJobs {
  int n;
  unsigned first[25];
  void* p[24];
  std::size_t bytes[24];
  unsigned pattern[24];
};

// 16 bytes a thread; blocks come from the pool, so every start is aligned and
// only the last bytes of a job need single stores
__global__ void __launch_bounds__(kBlock) fill_jobs(FillJobs j) {
  int w = 0;
  while (w + 1 < j.n && blockIdx.x >= j.first[w + 1]) ++w;
  std::size_t at = (std::size_t(blockIdx.x - j.first[w]) * kBlock + threadIdx.x) * 16;
  std::size_t bytes = j.bytes[w];
  char* p = static_cast<char*>(j.p[w]) + at;
  unsigned v = j.pattern[w];
  if (at + 16 <= bytes) {
    *reinterpret_cast<uint4*>(p) = make_uint4(v, v, v, v);
  } else {
    for (int k = 0; at + k < bytes && k < 16; ++k) p[k] = char(v >> (8 * (k & 3)));
  }
}

}  // namespace

void Fills::add(void* p, std::size_t bytes, unsigned pattern) {
  if (bytes == 0) return;
  OSH_CHECK(n_ < kMax, "too many fills");
  p_[n_] = p;
  bytes_[n_] = bytes;
  pattern_[n_] = pattern;
  ++n_;
}

void Fills::run() {
  FillJobs j{};
  unsigned blocks = 0;
  for (int i = 0; i < n_; ++i) {
    j.p[i] = p_[i];
    j.bytes[i] = bytes_[i];
    j.pattern[i] = pattern_[i];
    j.first[i] = blocks;
    blocks += unsigned((bytes_[i] + 16 * kBlock - 1) / (16 * kBlock));
    j.first[i + 1] = blocks;
  }
  j.n = n_;
  n_ = 0;
  if (blocks == 0) return;
  hipLaunchKernelGGL(fill_jobs, dim3(blocks), dim3(kBlock), 0, c_.stream, j);
  OSH_HIP(hipGetLastError());
}

LOs iota(Ctx& c, LO n, LO start, LO stride) {
  LOs out(c, n);
  OSH_LAUNCH(iota_kernel, n, c, out.data(), start, stride);
  return out;
}

LOs fill_lo(Ctx& c, LO n, LO value) {
  LOs out(c, n);
  OSH_LAUNCH(fill_kernel<LO>, n, c, out.data(), value);
  return out;
}

Bytes fill_i8(Ctx& c, LO n, I8 value) {
  Bytes out(c, n);
  OSH_LAUNCH(fill_kernel<I8>, n, c, out.data(), value);
  return out;
}

Reals fill_real(Ctx& c, LO n, Real value) {
  Reals out(c, n);
  OSH_LAUNCH(fill_kernel<Real>, n, c, out.data(), value);
  return out;
}

I8 max_i8(Ctx& c, Bytes const& a) {
  return a.size() ? I8(reduce_one<I8, LO>(c, a, kMax, kWholeInit)) : I8(-128);
}
Real min_real(Ctx& c, Reals const& a) { return reduce_one<Real, Real>(c, a, kMin, kRealInit); }
Real min_real_wait(Ctx& c, Reals const& a) {
  if (a.size() == 0) c.wait();
  return min_real(c, a);
}
Real max_real(Ctx& c, Reals const& a) { return reduce_one<Real, Real>(c, a, kMax, kRealInit); }

namespace {

// ---- stable LSD radix sort of (64-bit key, 32-bit value) pairs
//
// Keys are signed; flipping the sign bit (sort_word) orders them as unsigned
// words.  A pass sorts by one 8-bit digit: a count kernel histograms the digits of each
// 4096-item tile into counts[digit * ntiles + tile], one exclusive scan of
// those counts (digit-major) gives every (digit, tile) its first output
// position, and a scatter kernel places each item at that position plus its
// rank among the tile's items with the same digit that precede it, so equal
// digits keep their order.  A tile's items are read striped (item r * 256 +
// t is thread t's r-th), so that loads coalesce and the tile order is
// "round, then thread": the rank is the digit's count in earlier rounds (a
// running LDS counter) plus its count in earlier waves of this round (LDS)
// plus the lanes below in the same wave with the same digit (eight ballots).
// Keys are packed (see sort_by_keys), so passes run only over bits that differ.
constexpr int kSortItems = 16;
constexpr int kSortTile = kBlock * kSortItems;
constexpr int kSortBins = 256;
constexpr int kSortWaves = kBlock / kWave;

__device__ __forceinline__ unsigned long long sort_word(I64 k) {
  return static_cast<unsigned long long>(k) ^ (1ull << 63);
}

// the OR and the AND of each tuple component's key words (their XOR shows
// the bits that differ) in one sweep.  At most kBitsBlocks workgroups, each
// combining its share through LDS, so the two words of a component see few
// atomics: one atomic per wave instead serialised 72,000 of them on one
// cache line (358 us a column in the build of a 40^3 box; the sweep over all
// columns now takes 18 us).
constexpr int kBitsBlocks = 256;
constexpr int kMaxKeyWidth = 8;

__global__ void __launch_bounds__(kBlock) sort_bits_kernel(LO n, int width, I64 const* keys,
    unsigned long long* or_and) {
  __shared__ unsigned long long s_or[kBlock / kWave], s_and[kBlock / kWave];
  int lane = int(threadIdx.x) & (kWave - 1);
  int wave = int(threadIdx.x) / kWave;
  for (int k = 0; k < width; ++k) {
    unsigned long long o = 0ull, a = ~0ull;
    for (std::int64_t i = std::int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n;
         i += std::int64_t(gridDim.x) * kBlock) {
      unsigned long long w = sort_word(keys[i * width + k]);
      o |= w;
      a &= w;
    }
    for (int d = kWave / 2; d > 0; d >>= 1) {
      o |= __shfl_xor(o, d, kWave);
      a &= __shfl_xor(a, d, kWave);
    }
    if (lane == 0) {
      s_or[wave] = o;
      s_and[wave] = a;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kBlock / kWave; ++w) {
        o |= s_or[w];
        a &= s_and[w];
      }
      atomicOr(or_and + 2 * k, o);
      atomicAnd(or_and + 2 * k + 1, a);
    }
    __syncthreads();
  }
}

__global__ void init_or_and(LO n, unsigned long long* or_and) {
  LO i = thread_index();
  if (i < n) or_and[i] = (i & 1) ? ~0ull : 0ull;
}

// the bit fields of the tuple components that one packed key holds, the
// last packed component lowest
struct PackedFields {
  int first, count;  // components [first, first + count)
  int shift[kMaxKeyWidth];
  int bits[kMaxKeyWidth];
};

__global__ void pack_keys(LO n, int width, I64 const* keys, LO const* perm, PackedFields f,
    I64* out) {
  LO i = thread_index();
  if (i >= n) return;
  I64 const* row = keys + std::int64_t(perm ? perm[i] : i) * width;
  unsigned long long r = 0ull;
  for (int k = 0; k < f.count; ++k) {
    int b = f.bits[k];
    if (b == 0) continue;
    unsigned long long w = sort_word(row[f.first + k]) >> f.shift[k];
    if (b < 64) w &= (1ull << b) - 1ull;
    r = (b < 64) ? ((r << b) | w) : w;
  }
  out[i] = I64(r);
}

__global__ void find_ties(LO n, I64 const* sorted, int* ties) {
  LO i = thread_index();
  if (i + 1 < n && sorted[i] == sorted[i + 1]) *ties = 1;
}

__global__ void __launch_bounds__(kBlock) sort_count(LO n, I64 const* keys, int shift,
    LO ntiles, LO* counts) {
  __shared__ LO hist[kSortBins];
  hist[threadIdx.x] = 0;
  __syncthreads();
  LO base = LO(blockIdx.x) * kSortTile;
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    LO i = base + r * kBlock + LO(threadIdx.x);
    if (i < n)
      atomicAdd(&hist[int(static_cast<unsigned long long>(keys[i]) >> shift) & (kSortBins - 1)],
          1);
  }
  __syncthreads();
  counts[LO(threadIdx.x) * ntiles + LO(blockIdx.x)] = hist[threadIdx.x];
}

__global__ void __launch_bounds__(kBlock) sort_scatter(LO n, I64 const* keys, LO const* vals,
    int shift, LO ntiles, LO const* offsets, I64* out_keys, LO* out_vals) {
  __shared__ LO running[kSortBins];
  __shared__ LO wave_counts[kSortWaves][kSortBins];
  int t = int(threadIdx.x);
  int lane = t & (kWave - 1);
  int wave = t / kWave;
  running[t] = offsets[LO(t) * ntiles + LO(blockIdx.x)];
  for (int w = 0; w < kSortWaves; ++w) wave_counts[w][t] = 0;
  __syncthreads();
  LO base = LO(blockIdx.x) * kSortTile;
  unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
  for (int r = 0; r < kSortItems; ++r) {
    LO i = base + r * kBlock + t;
    bool valid = i < n;
    I64 k = valid ? keys[i] : 0;
    int d = valid ? int(static_cast<unsigned long long>(k) >> shift) & (kSortBins - 1) : 0;
    // the lanes of this wave holding the same digit
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      unsigned long long bit = __ballot(valid && ((d >> b) & 1));
      same &= ((d >> b) & 1) ? bit : ~bit;
    }
    int rank_in_wave = __popcll(same & below);
    bool leader = valid && rank_in_wave == 0;
    if (leader) wave_counts[wave][d] = __popcll(same);
    __syncthreads();
    if (valid) {
      LO pos = running[d] + rank_in_wave;
      for (int w = 0; w < wave; ++w) pos += wave_counts[w][d];
      out_keys[pos] = k;
      out_vals[pos] = vals[i];
    }
    __syncthreads();
    // advance the running offsets by this round's counts and clear them
    LO add = 0;
    for (int w = 0; w < kSortWaves; ++w) {
      add += wave_counts[w][t];
      wave_counts[w][t] = 0;
    }
    running[t] += add;
    __syncthreads();
  }
}

// sorts (keys, vals) by the digits that hold a bit of `differ` in place
// (stable), using the second pair of buffers; returns with the result in the
// first pair
void radix_sort_pairs(Ctx& c, DArray<I64>& keys, LOs& vals, DArray<I64>& keys_tmp,
    LOs& vals_tmp, unsigned long long differ) {
  LO n = keys.size();
  LO ntiles = LO((std::int64_t(n) + kSortTile - 1) / kSortTile);
  OSH_CHECK(std::int64_t(ntiles) * kSortBins < std::int64_t(0x7fffffff), "sort: too many items");
  LOs counts(c, ntiles * kSortBins), offsets(c, ntiles * kSortBins + 1);
  for (int shift = 0; shift < 64; shift += 8) {
    if (((differ >> shift) & 0xffull) == 0ull) continue;
    hipLaunchKernelGGL(sort_count, dim3(unsigned(ntiles)), dim3(kBlock), 0, c.stream, n,
        keys.data(), shift, ntiles, counts.data());
    OSH_HIP(hipGetLastError());
    ScanJob job{counts.data(), kScanLO, ntiles * kSortBins, offsets.data(), nullptr};
    offset_scans(c, &job, 1);
    hipLaunchKernelGGL(sort_scatter, dim3(unsigned(ntiles)), dim3(kBlock), 0, c.stream, n,
        keys.data(), vals.data(), shift, ntiles, offsets.data(), keys_tmp.data(),
        vals_tmp.data());
    OSH_HIP(hipGetLastError());
    std::swap(keys, keys_tmp);
    std::swap(vals, vals_tmp);
  }
}

}  // namespace

// Stable lexical sort.  Only the span of bits in which a component's keys
// differ decides its order, so neighbouring components are packed into one
// 64-bit key while their spans fit (the vertex triples of a 40^3 box need 51
// bits: seven digit passes instead of three per component).  Components that
// don't fit one key form several groups; the leading group is sorted first,
// and when no two of its keys tie (Hilbert keys of distinct points differ
// early) the rest decides nothing.  Otherwise the groups are sorted LSD, the
// last one first, each stable.
LOs sort_by_keys(Ctx& c, DArray<I64> const& keys, int width) {
  LO n = keys.size() / width;
  LOs perm = iota(c, n);
  if (n <= 1) return perm;
  OSH_CHECK(width <= kMaxKeyWidth, "sort_by_keys: at most 8 keys per tuple");
  DArray<unsigned long long> or_and(c, 2 * width);
  OSH_LAUNCH(init_or_and, 2 * width, c, or_and.data());
  unsigned nb = nblocks(n) < unsigned(kBitsBlocks) ? nblocks(n) : unsigned(kBitsBlocks);
  hipLaunchKernelGGL(sort_bits_kernel, dim3(nb), dim3(kBlock), 0, c.stream, n, width,
      keys.data(), or_and.data());
  OSH_HIP(hipGetLastError());
  std::vector<unsigned long long> oa = to_host(c, or_and);
  std::vector<PackedFields> groups;
  std::vector<int> group_bits;
  std::vector<unsigned long long> group_differ;
  for (int k = 0; k < width; ++k) {
    unsigned long long differ = oa[std::size_t(2 * k)] ^ oa[std::size_t(2 * k + 1)];
    int shift = differ ? __builtin_ctzll(differ) : 0;
    int bits = differ ? 64 - __builtin_clzll(differ) - shift : 0;
    if (groups.empty() || group_bits.back() + bits > 64) {
      PackedFields f{};
      f.first = k;
      groups.push_back(f);
      group_bits.push_back(0);
      group_differ.push_back(0ull);
    }
    PackedFields& f = groups.back();
    f.shift[f.count] = shift;
    f.bits[f.count] = bits;
    ++f.count;
    group_bits.back() += bits;
    unsigned long long& gd = group_differ.back();
    gd = bits == 0 ? gd : (bits < 64 ? (gd << bits) | (differ >> shift) : differ >> shift);
  }
  DArray<I64> packed(c, n), packed_tmp(c, n);
  LOs perm_tmp(c, n);
  int ngroups = int(groups.size());
  if (ngroups > 1) {
    OSH_LAUNCH(pack_keys, n, c, width, keys.data(), (LO const*)nullptr, groups[0],
        packed.data());
    radix_sort_pairs(c, packed, perm, packed_tmp, perm_tmp, group_differ[0]);
    int* ties = slot_ptr<int>(c, 0);
    *ties = 0;  // nothing queued so far writes slot 0
    OSH_LAUNCH(find_ties, n, c, packed.data(), ties);
    if (pinned_value<int>(c) == 0) return perm;
    perm = iota(c, n);
  }
  for (int g = ngroups - 1; g >= 0; --g) {
    OSH_LAUNCH(pack_keys, n, c, width, keys.data(),
        g == ngroups - 1 ? (LO const*)nullptr : perm.data(), groups[std::size_t(g)],
        packed.data());
    radix_sort_pairs(c, packed, perm, packed_tmp, perm_tmp, group_differ[std::size_t(g)]);
  }
  return perm;
}

}  // namespace osh
