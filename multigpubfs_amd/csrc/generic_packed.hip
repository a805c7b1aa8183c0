// Generic backend on graphs whose states are one packed word (wide.hpp):
// any action over full history.
//
// The row form (generic_kernels.hip) hashes a child from its SoA entries,
// compares full states entry by entry and keeps a row list per layer.  Here
// a state is its word: all states found lie in one array in discovery
// order, so a layer is a range of it, and the visited table holds the words
// themselves (equality of words is equality of states).  Rows beyond the
// capacity stop the run with the row form's error bit.
#include <algorithm>
#include <cstring>
#include <vector>
#include "common.hpp"
#include "engine.hpp"
#include "kernels.hpp"
#include "wide.hpp"

namespace mgbfs {

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kGrid = 2048;
constexpr int kItems = 4;         // child slots per thread and tile at most
constexpr uint32_t kAhead = 16;   // layers queued per host wait
constexpr uint64_t kNone = ~0ull;

// One queued layer: states [start, start + count) of the array are its
// parents; `count` of the next one is counted by this one's launch.
struct PackedLayer {
  unsigned long long start, count;
  uint32_t error, pad;
};

// Probes of one claim at most.  The table has twice the slots of the rows it
// may hold, so a longer run means that the layer has outgrown them (its
// claims are counted only at the end of each tile).
constexpr uint64_t kProbes = 1u << 16;

// True when this thread put `key` into the table.  A plain read first: a
// word never changes once written, so a stale one can only be empty.
__device__ __forceinline__ bool claim_word(uint64_t* table, uint64_t mask, uint64_t key, uint32_t* error) {
  uint64_t slot = mix64(key) & mask;
  const uint64_t most = mask < kProbes ? mask + 1 : kProbes;
  for (uint64_t probe = 0; probe < most; ++probe) {
    uint64_t seen = table[slot];
    if (seen == key) return false;
    if (seen == kNone) {
      uint64_t old = kNone;
      if (__hip_atomic_compare_exchange_strong(table + slot, &old, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        return true;
      if (old == key) return false;
    }
    slot = (slot + 1) & mask;
  }
  atomicOr(error, kErrVisitedCap);
  return false;
}

// One layer: child slots generator-major over the parents (rounded up to a
// multiple of 64, so a wave shares its generator), `items` per thread: one
// until the grid is full, so small layers keep every CU busy.  Bound by the
// chain parent -> child -> table word -> claim -> array row (about 9 us with
// the launch); large layers by random table lines.
__global__ __launch_bounds__(kThreads) void packed_expand_kernel(uint64_t* states, PackedLayer* layer, uint64_t* table,
                                                                 uint64_t mask, uint64_t capacity, WideAction act) {
  __shared__ uint32_t wave_sums[kThreads / kWave];
  __shared__ unsigned long long wg_base;
  __shared__ uint32_t full_up;
  if (threadIdx.x == 0) full_up = 0;
  __syncthreads();
  const uint64_t start = layer[0].start, count = layer[0].count;
  if (layer[0].error) {  // an earlier layer ran out of rows
    if (blockIdx.x == 0 && threadIdx.x == 0) layer[1].error = layer[0].error;
    return;
  }
  const uint64_t end = start + count;
  if (blockIdx.x == 0 && threadIdx.x == 0) layer[1].start = end;
  const uint64_t rows = (count + kWave - 1) / kWave * kWave, slots = rows * act.count();
  const uint64_t full = static_cast<uint64_t>(kGrid) * kThreads;
  const uint32_t items = slots <= full ? 1u : (slots <= 2 * full ? 2u : kItems);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x)) / kWave;
  const uint64_t tile = static_cast<uint64_t>(items) * kThreads;
  for (uint64_t t0 = blockIdx.x * tile; t0 < slots; t0 += kGrid * tile) {
    if (__hip_atomic_load(&layer[1].error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) full_up = 1;
    __syncthreads();
    if (full_up) return;  // the rows ran out in another tile: the layer is lost anyway
    uint64_t fresh[kItems];
    uint32_t mine = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      fresh[k] = kNone;
      uint64_t s = t0 + static_cast<uint64_t>(k) * kThreads + wave * kWave;  // the wave's first slot
      if (k >= static_cast<int>(items) || s >= slots) continue;
      uint32_t g = 0;
      for (; s >= rows; s -= rows) ++g;
      if (s + lane < count) {
        const uint64_t child = act.child(states[start + s + lane], g);
        if (claim_word(table, mask, child, &layer[1].error)) {
          fresh[k] = child;
          ++mine;
        }
      }
    }
    // Workgroup scan of the new states, one reservation per tile.
    uint32_t incl = mine;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t v = __shfl_up(incl, off, kWave);
      if (lane >= static_cast<uint32_t>(off)) incl += v;
    }
    if (lane == kWave - 1) wave_sums[wave] = incl;
    __syncthreads();
    uint32_t before = 0, sum = 0;
#pragma unroll
    for (uint32_t w = 0; w < kThreads / kWave; ++w) {
      before += w < wave ? wave_sums[w] : 0u;
      sum += wave_sums[w];
    }
    if (threadIdx.x == 0 && sum) wg_base = atomicAdd(&layer[1].count, static_cast<unsigned long long>(sum));
    __syncthreads();
    if (mine) {
      uint64_t pos = end + wg_base + before + incl - mine;
      if (pos + mine > capacity) {
        atomicOr(&layer[1].error, kErrVisitedCap);
      } else {
#pragma unroll
        for (int k = 0; k < kItems; ++k)
          if (fresh[k] != kNone) states[pos++] = fresh[k];
      }
    }
    __syncthreads();  // wave_sums and wg_base are reused
  }
}

__global__ void packed_seed_kernel(uint64_t key, uint64_t* states, uint64_t* table, uint64_t mask) {
  if (threadIdx.x != 0) return;
  states[0] = key;
  table[mix64(key) & mask] = key;
}

// The layers about to be queued: the current one, then empty ones.
__global__ void packed_begin_kernel(PackedLayer* layer, uint64_t start, uint64_t count) {
  if (threadIdx.x > kAhead) return;
  layer[threadIdx.x] = PackedLayer{threadIdx.x == 0 ? start : 0, threadIdx.x == 0 ? count : 0, 0, 0};
}

}  // namespace

class GenericPackedEngine final : public Engine {
 public:
  GenericPackedEngine(const Graph& g, const mgbfs_engine_options& o, uint64_t state_bound, const WideCode& code)
      : code_(code), generators_(g.generators), elements_(g.elements) {
    device_ = o.device;
    backend = MGBFS_BACKEND_GENERIC;
    history_layers = 0;
    state_bytes = generic_state_bytes(g);
    MGBFS_HIP(hipSetDevice(device_));
    MGBFS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    MGBFS_HIP(hipEventCreate(&ev0_));
    MGBFS_HIP(hipEventCreate(&ev1_));
    cap_ = o.capacity;
    if (!cap_) {
      cap_ = generic_capacity(g, vram_budget(o), state_bound);
      if (!cap_) throw std::runtime_error("GENERIC_VRAM_CAPACITY");
    }
    if (cap_ > kGenericMaxArena) throw std::runtime_error("GENERIC_ARENA_SHAPE");
    generic_plan_bytes(elements_, cap_, state_bytes, &slots_);
    slots_ = std::max<uint64_t>(slots_, 64);
    states_.allocate(cap_ * 8);
    table_.allocate(slots_ * 8);
    layer_.allocate(sizeof(PackedLayer) * (kAhead + 1));
    wide_.allocate(sizeof(WideTable));
    MGBFS_HIP(hipMemcpy(wide_.as<void>(), &code_.table, sizeof(WideTable), hipMemcpyHostToDevice));
    MGBFS_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_), sizeof(PackedLayer) * (kAhead + 1), hipHostMallocDefault));
    device_bytes = states_.bytes() + table_.bytes() + layer_.bytes() + wide_.bytes();
    reset();
  }
  ~GenericPackedEngine() override {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (host_) (void)hipHostFree(host_);
    if (ev0_) (void)hipEventDestroy(ev0_);
    if (ev1_) (void)hipEventDestroy(ev1_);
    if (stream_) (void)hipStreamDestroy(stream_);
  }

  void reset() override {
    MGBFS_HIP(hipSetDevice(device_));
    MGBFS_HIP(fill_u64(table_.as<uint64_t>(), ~0ull, slots_, stream_));
    hipLaunchKernelGGL(packed_seed_kernel, dim3(1), dim3(64), 0, stream_, code_.start_key, states_.as<uint64_t>(),
                       table_.as<uint64_t>(), slots_ - 1);
    MGBFS_HIP(hipGetLastError());
    start_ = 0;
    layers.assign(1, 1);
    candidates = unique_candidates = 0;
    kernel_seconds = 0;
    launches = 0;
    streamed_bytes = 0;
    terminal = false;
  }

  int advance(uint64_t* next_count, uint32_t* fatal) override {
    if (terminal) throw std::runtime_error("ENGINE_TERMINAL");
    const int s = run_layers(1, fatal);
    *next_count = s == MGBFS_LAYER ? layers.back() : 0;
    return s;
  }

  int run_to_end() override {
    int s = MGBFS_LAYER;
    uint32_t fatal = 0;
    while (!terminal) s = run_layers(kAhead, &fatal);
    return s;
  }

  void layer_keys(std::vector<uint64_t>&) override { throw std::runtime_error("GENERIC_NO_PACKED_KEYS"); }

  void sample(uint32_t which, uint64_t limit, std::vector<int64_t>& rows, uint64_t& count) override {
    rows.clear();
    count = 0;
    if (which != 0 && layers.size() < 2) return;
    const uint64_t size = which == 0 ? layers.back() : layers[layers.size() - 2];
    const uint64_t first = which == 0 ? start_ : start_ - size;
    count = std::min(limit, size);
    std::vector<uint64_t> keys(count);
    if (count) {
      MGBFS_HIP(hipMemcpyAsync(keys.data(), states_.as<uint64_t>() + first, count * 8, hipMemcpyDeviceToHost, stream_));
      MGBFS_HIP(hipStreamSynchronize(stream_));
    }
    rows.resize(count * elements_);
    for (uint64_t r = 0; r < count; ++r)
      for (uint32_t e = 0; e < elements_; ++e) rows[r * elements_ + e] = code_.value(keys[r], e);
  }

  const char* name() const override { return "GENERIC_EXACT_ALL_VISITED"; }

 private:
  // Queues up to `most` layers, waits once and takes their counts.
  int run_layers(uint32_t most, uint32_t* fatal) {
    MGBFS_HIP(hipSetDevice(device_));
    PackedLayer* layer = layer_.as<PackedLayer>();
    MGBFS_HIP(hipEventRecord(ev0_, stream_));
    hipLaunchKernelGGL(packed_begin_kernel, dim3(1), dim3(64), 0, stream_, layer, start_, layers.back());
    for (uint32_t i = 0; i < most; ++i)
      hipLaunchKernelGGL(packed_expand_kernel, dim3(kGrid), dim3(kThreads), 0, stream_, states_.as<uint64_t>(),
                         layer + i, table_.as<uint64_t>(), slots_ - 1, cap_,
                         WideAction{wide_.as<WideTable>(), generators_});
    MGBFS_HIP(hipGetLastError());
    MGBFS_HIP(hipEventRecord(ev1_, stream_));
    MGBFS_HIP(hipMemcpyAsync(host_, layer, sizeof(PackedLayer) * (most + 1), hipMemcpyDeviceToHost, stream_));
    MGBFS_HIP(hipStreamSynchronize(stream_));
    float ms = 0;
    MGBFS_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
    kernel_seconds += ms * 1e-3;
    for (uint32_t i = 0; i < most; ++i) {
      const uint64_t parents = host_[i].count, kids = host_[i + 1].count;
      ++launches;
      candidates += parents * generators_;
      if (host_[i + 1].error) {
        *fatal = host_[i + 1].error;
        terminal = true;
        return MGBFS_RESOURCE;
      }
      if (kids == 0) {
        terminal = true;
        return MGBFS_COMPLETE;
      }
      start_ += parents;
      layers.push_back(kids);
    }
    return MGBFS_LAYER;
  }

  WideCode code_;
  uint32_t generators_, elements_;
  uint64_t cap_ = 0, slots_ = 0, start_ = 0;  // start_: the current layer's first state
  DeviceBuffer states_, table_, layer_, wide_;
  PackedLayer* host_ = nullptr;
  hipEvent_t ev0_ = nullptr, ev1_ = nullptr;
};

Engine* make_generic_packed_engine(const Graph& g, const mgbfs_engine_options& o, uint64_t state_bound,
                                   const WideCode& code) {
  return new GenericPackedEngine(g, o, state_bound, code);
}

}  // namespace mgbfs
