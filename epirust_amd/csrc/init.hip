// Population synthesis on gfx950.
//
// The reference builds the population on the CPU (engine/src/geography/grid.rs:83-155,
// engine/src/citizen/citizen_factory.rs:31-134, epidemiology_simulation.rs:75-192); in
// deterministic mode every draw is a Philox block at hour 0xFFFFFFFF, so each step is a
// data-parallel kernel over agents or houses of every simulation of a batch at once (a block
// finds its simulation in a table of first blocks, in which it searches by halving):
//   k_init_agents  : per agent, working / public transport / work status / immunity
//                    (sites INIT_A, INIT_B, INIT_C); the public-transport draw is kept in
//                    F_PT and counted per block;
//   k_scan         : exclusive prefix sums of such counts, a block per array;
//   k_select_pass  : radix selection over the 96-bit composite (INIT_C key, id), 8 bits
//                    a pass, finds the agents of given ranks without sorting; the starting
//                    infections (the `total` smallest composites, taking exposed /
//                    asymptomatic / mild / severe in composite order) need at most four
//                    such ranks, narrowed side by side;
//   k_init_finish  : per agent, the transport cap in id order (citizen_factory.rs:72-83) as a
//                    rank test against the scanned counts, then its group of starting
//                    infections from the four rank bounds;
//   k_init_cells   : per house, random_points(k) of the 2x2 house for its agents, and their
//                    bytes of the occupancy grid.
// All of it is integer work over a few bytes per agent and runs once per handle, a chain of
// launches that nothing on the host waits for: 32 simulations of 100k agents are created in
// 13.1 -> 1.7 ms, 64 of mixed sizes in 26.8 -> 3.3, one of 10k in 0.57 -> 0.46 (before: a simulation at a
// time, a read-back after each of its up to 32 selection passes, temporaries for each).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>
#include <vector>

#include "disease.hpp"
#include "init.hpp"
#include "philox.hpp"

namespace epi {
namespace {

constexpr uint32_t kInitBlock = 256;
constexpr uint32_t kSelectBits = 8;
constexpr uint32_t kSelectBins = 1u << kSelectBits;
constexpr uint32_t kSelectTopShift = 96 - kSelectBits;  // 88
constexpr uint32_t kSelectBlocks = 512;                 // at most, for one simulation
static_assert(kSelectBins == kInitBlock, "a thread per bin");

// A point of the 96-bit order (key, id): key in bits 95..32, id in bits 31..0.
struct Composite {
  unsigned long long key;
  uint32_t id;
};

// One simulation of the batch. first_* are its first blocks in the launches over agents,
// selection strides and houses.
struct InitSim {
  uint32_t n;
  uint32_t seed_lo, seed_hi;
  uint64_t thr_work, thr_pt, thr_staff, thr_ess;
  const uint8_t* csv_working;  // Population::Csv columns, or null for Auto
  const uint8_t* csv_pt;
  uint32_t pt_cap;  // ~0u: none (Population::Csv records keep their flag)
  uint32_t* pos;
  uint32_t* st;
  uint32_t* tm;
  uint32_t* wsa;
  uint8_t* occ;
  uint32_t strip;
  DiseaseParams dz;
  int32_t house_sx, house_sy, house_nx;
  uint32_t n_houses;
  uint32_t* block_pt;  // per agent block: public-transport draws, then their exclusive prefix
  uint32_t infected;   // starting infections of all kinds
  uint32_t zero;       // bit j: the first j + 1 kinds together are none
  uint32_t first_block, first_select, first_house;
};
// The same for the office layout's maps, with offices and chunks of houses.
struct OfficeSim {
  uint32_t n, n_offices, n_houses;
  const uint32_t* st;
  uint32_t *office_agent, *office_slot;
  uint32_t *cnt, *base;    // per office: its workers, and their exclusive prefix
  uint32_t *rcnt, *rbase;  // per chunk of houses: the other agents, and their exclusive prefix
  uint32_t first_office, first_chunk;
};

// The last of n simulations whose first block (member F) is at most `block`: those with no
// blocks share the next one's first.
template <auto F, class Sim>
__device__ __forceinline__ uint32_t sim_of_block(const Sim* sims, uint32_t n, uint32_t block) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (sims[mid].*F <= block) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint64_t seed_of(const InitSim& a) { return join64(a.seed_hi, a.seed_lo); }

__device__ __forceinline__ uint64_t infection_key(uint32_t seed_lo, uint32_t seed_hi, uint32_t i) {
  const u32x4 c = philox4x32_10(i, kInitHour, SITE_INIT_C, 0, seed_lo, seed_hi);
  return join64(c.w[2], c.w[3]);
}

// Bits [shift, shift + kSelectBits) of the composite.
__device__ __forceinline__ uint32_t digit(uint64_t key, uint32_t id, uint32_t shift) {
  if (shift >= 32) return static_cast<uint32_t>(key >> (shift - 32)) & (kSelectBins - 1);
  const uint64_t low = (key << 32) | id;
  return static_cast<uint32_t>(low >> shift) & (kSelectBins - 1);
}

__device__ __forceinline__ void set_digit(Composite& c, uint32_t shift, uint32_t d) {
  if (shift >= 32) {
    c.key |= static_cast<unsigned long long>(d) << (shift - 32);
  } else {
    const uint64_t v = static_cast<uint64_t>(d) << shift;
    c.id |= static_cast<uint32_t>(v);
    c.key |= v >> 32;
  }
}

// Blocks of a simulation in a selection pass, each striding over its agents, at least 16 a
// thread: the last block adds up the others' counts.
__host__ __device__ inline uint32_t select_blocks(uint32_t n) {
  const uint32_t blocks = (n + 16u * kInitBlock - 1u) / (16u * kInitBlock);
  return blocks < kSelectBlocks ? blocks : kSelectBlocks;
}

__device__ __forceinline__ bool greater(uint64_t key, uint32_t id, const Composite& c) {
  return key > c.key || (key == c.key && id > c.id);
}

__global__ __launch_bounds__(kInitBlock) void k_init_agents(const InitSim* sims, uint32_t n_sims) {
  const InitSim& a = sims[sim_of_block<&InitSim::first_block>(sims, n_sims, blockIdx.x)];
  const uint32_t block = blockIdx.x - a.first_block, i = block * kInitBlock + threadIdx.x;
  bool pt = false;
  if (i < a.n) {
    const uint64_t seed = seed_of(a);
    const u32x4 A = draw(seed, i, kInitHour, SITE_INIT_A, 0);
    const u32x4 B = draw(seed, i, kInitHour, SITE_INIT_B, 0);
    const u32x4 C = draw(seed, i, kInitHour, SITE_INIT_C, 0);
    bool working;
    if (a.csv_working) {  // Citizen::from_record (citizen/mod.rs:155-180)
      working = a.csv_working[i] != 0;
      pt = a.csv_pt[i] != 0;
    } else {
      working = bernoulli(a.thr_work, join64(A.w[0], A.w[1]));
      pt = working && bernoulli(a.thr_pt, join64(A.w[2], A.w[3]));
    }
    uint32_t ws;
    if (!working) ws = WS_NA;
    else if (bernoulli(a.thr_staff, join64(B.w[0], B.w[1]))) ws = WS_STAFF;
    else ws = bernoulli(a.thr_ess, join64(C.w[0], C.w[1])) ? WS_ESSENTIAL : WS_NORMAL;
    const uint32_t imm = below(B.w[2], 5);  // immunity -2..2 stored as immunity + 2
    a.st[i] = (ST_S << B_STATE) | (ws << B_WS) | (AREA_HOME << B_AREA) | (imm << B_IMM) | (pt ? F_PT : 0u);
    a.wsa[i] = ws == WS_STAFF ? 8u : 0u;  // HospitalStaff { work_start_at: ROUTINE_WORK_TIME }
    a.tm[i] = 0;
  }
  const int count = __syncthreads_count(pt);
  if (threadIdx.x == 0) a.block_pt[block] = static_cast<uint32_t>(count);
}

// Exclusive prefix sum of from[0..n) into to (the same array or another), one block of 1024
// threads per array: each thread sums a contiguous chunk, the chunk sums are scanned in LDS,
// then each chunk is written.
struct ScanJob {
  const uint32_t* from;
  uint32_t* to;
  uint32_t n;
};
__global__ __launch_bounds__(1024) void k_scan(const ScanJob* jobs) {
  __shared__ uint32_t part[1024];
  const ScanJob a = jobs[blockIdx.x];
  const uint32_t per = (a.n + 1023u) / 1024u;
  const uint32_t b = min(a.n, threadIdx.x * per), e = min(a.n, b + per);
  uint32_t sum = 0;
  for (uint32_t k = b; k < e; ++k) sum += a.from[k];
  part[threadIdx.x] = sum;
  __syncthreads();
  for (uint32_t off = 1; off < 1024u; off <<= 1) {
    const uint32_t t = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
    __syncthreads();
    part[threadIdx.x] += t;
    __syncthreads();
  }
  uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0u;
  for (uint32_t k = b; k < e; ++k) {
    const uint32_t x = a.from[k];
    a.to[k] = run;
    run += x;
  }
}

// Selection of up to four ranks of one simulation: bound[j] is the composite of rank
// c_j - 1 for the cumulative group sizes c = (exposed, +asymptomatic, +mild, +severe), once
// bit j of `done` is set; until then its top bits, with the rank that is left among the agents
// that share them. An agent of rank r belongs to group #{j : r >= c_j}; group 4 means not
// selected.
struct Select {
  Composite bound[4];
  uint32_t rank[4];
  uint32_t done;
  uint32_t finished;  // blocks that have counted in this pass
};

// Bits below `shift` of the composite.
__device__ __forceinline__ Composite low_bits(uint32_t shift) {
  if (shift >= 32) return Composite{(1ull << (shift - 32)) - 1ull, ~0u};
  return Composite{0ull, shift ? ~0u >> (32 - shift) : 0u};
}

// One pass: a histogram of digit(shift) over the agents that share each open bound's top bits.
// In the first pass these are all agents: counted in LDS, each block's counts stored to `top`
// (as atomics, up to 512 to one address, they take longer than the draws).
// Later they are next to none, counted by atomics in the simulation's slice of `hist`. The
// block that finishes last takes each bound's bin, clears what it read for the next pass, and
// closes a bound whose bin holds one agent: all lower bits set then compare as that agent's own
// do. So most of the twelve launches find nothing to do. What other blocks wrote is read by
// device-scope atomics.
__global__ __launch_bounds__(kInitBlock) void k_select_pass(const InitSim* sims, uint32_t n_sims, Select* selects,
                                                            uint32_t* top, uint32_t* hist, uint32_t shift) {
  __shared__ uint32_t h[kSelectBins];
  __shared__ uint32_t last, single;
  const uint32_t sim = sim_of_block<&InitSim::first_select>(sims, n_sims, blockIdx.x);
  const InitSim& a = sims[sim];
  Select& s = selects[sim];
  const uint32_t done = s.done;
  if (done == 15u) return;  // uniform, over all the simulation's blocks
  const uint32_t n_blocks = select_blocks(a.n), t = threadIdx.x;
  hist += static_cast<size_t>(sim) * 4 * kSelectBins;
  const bool first = shift == kSelectTopShift;
  // read before the loop, whose atomics could change them for all the compiler knows
  const uint32_t n = a.n, seed_lo = a.seed_lo, seed_hi = a.seed_hi;
  Composite bound[4];
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) bound[j] = s.bound[j];
  const Composite low = low_bits(shift + kSelectBits);  // not compared
  h[t] = 0;
  __syncthreads();
  for (uint32_t i = (blockIdx.x - a.first_select) * kInitBlock + t; i < n; i += n_blocks * kInitBlock) {
    const uint64_t key = infection_key(seed_lo, seed_hi, i);
    const uint32_t d = digit(key, i, shift);
    if (first) {
      atomicAdd(&h[d], 1u);
      continue;
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      if (!((done >> j) & 1u) && ((key ^ bound[j].key) & ~low.key) == 0 && ((i ^ bound[j].id) & ~low.id) == 0)
        atomicAdd(&hist[j * kSelectBins + d], 1u);
  }
  __syncthreads();
  if (first)
    __hip_atomic_store(&top[static_cast<size_t>(blockIdx.x) * kSelectBins + t], h[t], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  __threadfence();
  __syncthreads();
  if (t == 0) last = atomicAdd(&s.finished, 1u) == n_blocks - 1u;
  __syncthreads();
  if (!last) return;
  __threadfence();
  uint32_t all = 0;  // agents of this thread's bin
  if (first) {
    const uint32_t* of = top + static_cast<size_t>(a.first_select) * kSelectBins + t;
#pragma unroll 16
    for (uint32_t b = 0; b < n_blocks; ++b)
      all += __hip_atomic_load(of + static_cast<size_t>(b) * kSelectBins, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  uint32_t closed = done;
  for (uint32_t j = 0; j < 4; ++j) {
    if ((done >> j) & 1u) continue;  // uniform
    uint32_t count = all;
    if (!first) {
      count = __hip_atomic_load(&hist[j * kSelectBins + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&hist[j * kSelectBins + t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t r = s.rank[j];  // before the barriers: one thread changes it after them
    if (t == 0) single = 0;
    h[t] = count;
    __syncthreads();
    for (uint32_t off = 1; off < kSelectBins; off <<= 1) {
      const uint32_t before = t >= off ? h[t - off] : 0u;
      __syncthreads();
      h[t] += before;
      __syncthreads();
    }
    const uint32_t before = h[t] - count;
    if (r >= before && r - before < count) {  // one thread
      Composite c = bound[j];
      set_digit(c, shift, t);
      if (count == 1u || shift == 0u) {
        const Composite rest = low_bits(shift);
        c.key |= rest.key;
        c.id |= rest.id;
        single = 1;
      }
      s.bound[j] = c;
      s.rank[j] = r - before;
    }
    __syncthreads();
    if (single) closed |= 1u << j;
    __syncthreads();
  }
  if (t == 0) {
    s.done = closed;
    s.finished = 0;
  }
}

__global__ __launch_bounds__(kInitBlock) void k_init_finish(const InitSim* sims, uint32_t n_sims,
                                                            const Select* selects) {
  __shared__ uint32_t wave_count[kInitBlock / 64];
  const uint32_t sim = sim_of_block<&InitSim::first_block>(sims, n_sims, blockIdx.x);
  const InitSim& a = sims[sim];
  const uint32_t block = blockIdx.x - a.first_block, i = block * kInitBlock + threadIdx.x;
  const uint32_t w_in = i < a.n ? a.st[i] : 0u;
  uint32_t w = w_in;
  // clears F_PT on every public-transport draw whose rank in id order is >= the cap
  const uint64_t mask = __ballot((w & F_PT) != 0);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0) wave_count[wave] = static_cast<uint32_t>(__popcll(mask));
  __syncthreads();
  if (w & F_PT) {
    uint32_t rank = a.block_pt[block] + static_cast<uint32_t>(__popcll(mask & ((1ull << lane) - 1ull)));
    for (uint32_t q = 0; q < wave; ++q) rank += wave_count[q];
    if (rank >= a.pt_cap) w &= ~F_PT;
  }
  if (i >= a.n) return;
  if (a.infected) {  // uniform
    const Select& s = selects[sim];
    const uint64_t key = infection_key(a.seed_lo, a.seed_hi, i);
    uint32_t group = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (((a.zero >> j) & 1u) || greater(key, i, s.bound[j])) ++group;
    if (group < 4) {
      // starting_infections.rs: exposed {at_hour 0}; infected asymptomatic / mild / severe on day 1
      const uint32_t state = group == 0 ? ST_E : ST_I;
      const uint32_t sev = group == 0 ? 0u : (group == 1 ? SEV_ASYM : (group == 2 ? SEV_MILD : SEV_SEVERE));
      const uint32_t day = group == 0 ? 0u : 1u;
      w = (w & ~((M_STATE << B_STATE) | (M_SEV << B_SEV) | (M_DAY << B_DAY))) | (state << B_STATE) | (sev << B_SEV) |
          (day << B_DAY);
    }
  }
  if (w != w_in) a.st[i] = w;  // tm is 0 already
}

// Partial Fisher-Yates over {lo, lo + 1} from fixed words: min(m, 2) values.
__device__ __forceinline__ uint32_t choose2(int32_t lo, uint32_t m, uint32_t w0, uint32_t w1, int32_t* out) {
  int32_t v0 = lo, v1 = lo + 1;
  if (m > 2) m = 2;
  if (m >= 1 && below(w0, 2) == 1) {
    const int32_t t = v0;
    v0 = v1;
    v1 = t;
  }
  // the second step draws from a one-element range and swaps nothing (below(w1, 1) == 0)
  (void)w1;
  out[0] = v0;
  out[1] = v1;
  return m;
}

// House h holds agents h, h + H, ...; they take random_points(k) of the house in id order, and
// each cell its agent's grid byte: 1 occupied, 2 / 3 infectious in the regular / high window.
__global__ __launch_bounds__(kInitBlock) void k_init_cells(const InitSim* sims, uint32_t n_sims) {
  const InitSim& a = sims[sim_of_block<&InitSim::first_house>(sims, n_sims, blockIdx.x)];
  const uint32_t h = (blockIdx.x - a.first_house) * kInitBlock + threadIdx.x;
  const uint32_t H = a.n_houses;
  if (h >= min(H, a.n)) return;
  const uint32_t k = (a.n - h + H - 1) / H;
  const int32_t x0 = a.house_sx + static_cast<int32_t>(h % static_cast<uint32_t>(a.house_nx)) * 2;
  const int32_t y0 = a.house_sy + static_cast<int32_t>(h / static_cast<uint32_t>(a.house_nx)) * 2;
  const u32x4 w = draw(seed_of(a), h, kInitHour, SITE_INIT_HOUSE, 0);
  uint32_t side = 1;  // ceil(sqrt(k)) in integers
  while (side * side < k) ++side;
  int32_t xs[2], ys[2];
  const uint32_t mx = choose2(x0, side, w.w[0], w.w[1], xs);
  const uint32_t my = choose2(y0, side, w.w[2], w.w[3], ys);
  uint32_t j = 0;
  for (uint32_t p = 0; p < mx && j < k; ++p)
    for (uint32_t q = 0; q < my && j < k; ++q, ++j) {
      const uint32_t id = h + j * H, x = static_cast<uint32_t>(xs[p]), y = static_cast<uint32_t>(ys[q]);
      a.pos[id] = x | (y << 16);
      const uint8_t byte = occupant_byte(a.dz, a.st[id]);
      const GridPlace g = grid_place(a.strip, x, y);
      a.occ[g.at] = byte;
      if (in_two_strips(g)) a.occ[second_place(a.strip, g)] = byte;
    }
}

// One allocation for all of a call's scratch arrays: add() them, then alloc().
struct DeviceTemp {
  template <class T>
  void add(T** p, size_t count) {
    arrays.push_back({reinterpret_cast<void**>(p), bytes});
    bytes += (count * sizeof(T) + 255) / 256 * 256;
  }
  hipError_t alloc() {
    const hipError_t e = hipMalloc(&memory, std::max<size_t>(bytes, 1));
    if (e != hipSuccess) {
      memory = nullptr;
      return e;
    }
    for (const auto& a : arrays) *a.first = static_cast<char*>(memory) + a.second;
    return e;
  }
  ~DeviceTemp() {
    if (memory) (void)hipFree(memory);
  }
  std::vector<std::pair<void**, size_t>> arrays;
  size_t bytes = 0;
  void* memory = nullptr;
};

template <class T>
hipError_t upload(T* to, const std::vector<T>& from, hipStream_t stream) {
  return hipMemcpyAsync(to, from.data(), from.size() * sizeof(T), hipMemcpyHostToDevice, stream);
}

uint32_t div_up(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

#define INIT_TRY(step, expr)      \
  do {                            \
    hipError_t e_ = (expr);       \
    if (e_ != hipSuccess) {       \
      err = step;                 \
      return e_;                  \
    }                             \
  } while (0)

// ---- office layout slot maps (model.hpp): Normal and Essential workers office by office
// (office j = id % n_offices), each office's in id order, then the other agents house by house.
__device__ __forceinline__ bool office_worker(uint32_t w) {
  const uint32_t ws = (w >> B_WS) & M_WS;
  return ws == WS_NORMAL || ws == WS_ESSENTIAL;
}

// One thread per office: its workers (ids j, j + O, ... in order, coalesced over offices), the
// state words of kAhead of them in flight.
constexpr uint32_t kAhead = 16;
template <class F>
__device__ __forceinline__ void for_each_id(const OfficeSim& a, uint32_t j, F&& f) {
  for (uint64_t id0 = j; id0 < a.n; id0 += static_cast<uint64_t>(kAhead) * a.n_offices) {
    uint32_t w[kAhead];
#pragma unroll
    for (uint32_t k = 0; k < kAhead; ++k) {
      const uint64_t id = id0 + static_cast<uint64_t>(k) * a.n_offices;
      w[k] = id < a.n ? a.st[id] : (WS_NA << B_WS);
    }
#pragma unroll
    for (uint32_t k = 0; k < kAhead; ++k)
      if (office_worker(w[k])) f(static_cast<uint32_t>(id0 + static_cast<uint64_t>(k) * a.n_offices));
  }
}

__global__ __launch_bounds__(kInitBlock) void k_office_count(const OfficeSim* sims, uint32_t n_sims) {
  const OfficeSim& a = sims[sim_of_block<&OfficeSim::first_office>(sims, n_sims, blockIdx.x)];
  const uint32_t j = (blockIdx.x - a.first_office) * kInitBlock + threadIdx.x;
  if (j >= a.n_offices) return;
  uint32_t c = 0;
  for_each_id(a, j, [&](uint32_t) { ++c; });
  a.cnt[j] = c;
}

__global__ __launch_bounds__(kInitBlock) void k_office_place(const OfficeSim* sims, uint32_t n_sims) {
  const OfficeSim& a = sims[sim_of_block<&OfficeSim::first_office>(sims, n_sims, blockIdx.x)];
  const uint32_t j = (blockIdx.x - a.first_office) * kInitBlock + threadIdx.x;
  if (j >= a.n_offices) return;
  uint32_t slot = a.base[j];
  for_each_id(a, j, [&](uint32_t id) {
    a.office_agent[slot] = id;
    a.office_slot[id] = slot;
    ++slot;
  });
}

// The other agents go house by house, so that those of a wave stand close together and share the
// lines of their neighbourhoods and claims (in id order instead: 1M agents 18.0 us an hour, 17.1 so;
// 333k 11.3, 10.6; 64 runs of mixed sizes 134.8, 129.8; 10M 124.0, 121.3).
// The other agents of house h (ids h, h + H, ... in order), one thread per house, kInitBlock houses
// a block: how many, and how many the block's earlier houses have.
__device__ __forceinline__ uint32_t rest_of_house(const OfficeSim& a, uint32_t h, uint32_t& before, uint32_t& total) {
  __shared__ uint32_t sum[kInitBlock];
  uint32_t c = 0;
  if (h < a.n_houses)
    for (uint64_t id = h; id < a.n; id += a.n_houses) c += office_worker(a.st[id]) ? 0u : 1u;
  sum[threadIdx.x] = c;
  __syncthreads();
  for (uint32_t off = 1; off < kInitBlock; off <<= 1) {
    const uint32_t t = threadIdx.x >= off ? sum[threadIdx.x - off] : 0u;
    __syncthreads();
    sum[threadIdx.x] += t;
    __syncthreads();
  }
  before = sum[threadIdx.x] - c;
  total = sum[kInitBlock - 1u];
  return c;
}

__global__ __launch_bounds__(kInitBlock) void k_rest_count(const OfficeSim* sims, uint32_t n_sims) {
  const OfficeSim& a = sims[sim_of_block<&OfficeSim::first_chunk>(sims, n_sims, blockIdx.x)];
  const uint32_t chunk = blockIdx.x - a.first_chunk;
  uint32_t before, total;
  rest_of_house(a, chunk * kInitBlock + threadIdx.x, before, total);
  if (threadIdx.x == 0) a.rcnt[chunk] = total;
}

// The workers come first: as many as the last office's base and count make.
__global__ __launch_bounds__(kInitBlock) void k_rest_place(const OfficeSim* sims, uint32_t n_sims) {
  const OfficeSim& a = sims[sim_of_block<&OfficeSim::first_chunk>(sims, n_sims, blockIdx.x)];
  const uint32_t chunk = blockIdx.x - a.first_chunk, h = chunk * kInitBlock + threadIdx.x;
  uint32_t before, total;
  if (rest_of_house(a, h, before, total) == 0) return;
  uint32_t slot = a.base[a.n_offices - 1u] + a.cnt[a.n_offices - 1u] + a.rbase[chunk] + before;
  for (uint64_t id = h; id < a.n; id += a.n_houses)
    if (!office_worker(a.st[id])) {
      a.office_agent[slot] = static_cast<uint32_t>(id);
      a.office_slot[id] = slot;
      ++slot;
    }
}

}  // namespace

hipError_t synthesize_on_device(const std::vector<InitJob>& jobs, hipStream_t stream, std::string& err) {
  const uint32_t n_sims = static_cast<uint32_t>(jobs.size());
  std::vector<InitSim> sims(n_sims);
  std::vector<Select> selects(n_sims);
  std::vector<ScanJob> scans;
  uint32_t blocks = 0, strides = 0, house_blocks = 0;
  size_t csv_bytes = 0;
  for (uint32_t i = 0; i < n_sims; ++i) {
    const Config& cfg = *jobs[i].cfg;
    const Geometry& geo = *jobs[i].geo;
    InitSim& a = sims[i];
    a = InitSim{};
    a.n = cfg.number_of_agents;
    a.seed_lo = static_cast<uint32_t>(jobs[i].seed);
    a.seed_hi = static_cast<uint32_t>(jobs[i].seed >> 32);
    a.thr_work = bernoulli_threshold(cfg.working_percentage);
    a.thr_pt = bernoulli_threshold(cfg.public_transport_percentage);
    a.thr_staff = bernoulli_threshold(0.002);  // HOSPITAL_STAFF_PERCENTAGE
    a.thr_ess = bernoulli_threshold(cfg.has_lockdown ? cfg.essential_workers_population : 0.0);
    a.pt_cap = cfg.csv_population ? ~0u : geo.n_transport_points;
    a.pos = jobs[i].pos;
    a.st = jobs[i].st;
    a.tm = jobs[i].tm;
    a.wsa = jobs[i].wsa;
    a.occ = jobs[i].occ;
    a.strip = jobs[i].strip;
    a.dz = Disease::params(cfg);
    a.house_sx = geo.house_sx;
    a.house_sy = geo.house_sy;
    a.house_nx = std::max(geo.house_nx, 1);
    a.n_houses = geo.n_houses;
    const uint64_t c[4] = {cfg.si_exposed, 0ull + cfg.si_exposed + cfg.si_asymptomatic,
                           0ull + cfg.si_exposed + cfg.si_asymptomatic + cfg.si_mild,
                           0ull + cfg.si_exposed + cfg.si_asymptomatic + cfg.si_mild + cfg.si_severe};
    a.infected = a.n && c[3] ? static_cast<uint32_t>(c[3]) : 0u;
    if (a.n && c[3] > a.n) {
      err = "select: rank beyond the population";
      return hipErrorInvalidValue;
    }
    selects[i] = Select{};
    for (uint32_t j = 0; j < 4; ++j) {
      if (c[j] == 0) a.zero |= 1u << j;
      else selects[i].rank[j] = static_cast<uint32_t>(c[j] - 1);
    }
    selects[i].done = a.zero;
    a.first_block = blocks;
    a.first_select = strides;
    a.first_house = house_blocks;
    blocks += div_up(a.n, kInitBlock);
    if (a.infected) strides += select_blocks(a.n);
    house_blocks += div_up(std::min(geo.n_houses, a.n), kInitBlock);
    if (cfg.csv_population) csv_bytes += 2 * static_cast<size_t>(a.n);
  }
  if (blocks == 0) return hipSuccess;
  DeviceTemp tmp;
  uint32_t *block_pt = nullptr, *top = nullptr, *hist = nullptr;
  uint8_t* csv = nullptr;
  InitSim* d_sims = nullptr;
  Select* d_selects = nullptr;
  ScanJob* d_scans = nullptr;
  const size_t bins = strides ? static_cast<size_t>(n_sims) * 4 * kSelectBins : 0;
  tmp.add(&d_sims, n_sims);
  tmp.add(&d_selects, n_sims);
  tmp.add(&d_scans, n_sims);
  tmp.add(&block_pt, blocks);
  tmp.add(&top, static_cast<size_t>(strides) * kSelectBins);
  tmp.add(&hist, bins);
  tmp.add(&csv, csv_bytes);
  INIT_TRY("alloc scratch", tmp.alloc());
  for (uint32_t i = 0; i < n_sims; ++i) {
    InitSim& a = sims[i];
    a.block_pt = block_pt + a.first_block;
    if (a.n) scans.push_back(ScanJob{a.block_pt, a.block_pt, div_up(a.n, kInitBlock)});
    const Config& cfg = *jobs[i].cfg;
    if (!cfg.csv_population || a.n == 0) continue;
    INIT_TRY("upload csv working", hipMemcpyAsync(csv, cfg.csv_working.data(), a.n, hipMemcpyHostToDevice, stream));
    INIT_TRY("upload csv pub_transport",
             hipMemcpyAsync(csv + a.n, cfg.csv_pub_transport.data(), a.n, hipMemcpyHostToDevice, stream));
    a.csv_working = csv;
    a.csv_pt = csv + a.n;
    csv += 2 * static_cast<size_t>(a.n);
  }
  INIT_TRY("upload simulations", upload(d_sims, sims, stream));
  INIT_TRY("upload selections", upload(d_selects, selects, stream));
  INIT_TRY("upload scans", upload(d_scans, scans, stream));
  hipLaunchKernelGGL(k_init_agents, dim3(blocks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
  INIT_TRY("k_init_agents", hipGetLastError());
  hipLaunchKernelGGL(k_scan, dim3(static_cast<uint32_t>(scans.size())), dim3(1024), 0, stream, d_scans);
  INIT_TRY("k_scan", hipGetLastError());
  if (strides) {
    INIT_TRY("clear histograms", hipMemsetAsync(hist, 0, bins * sizeof(uint32_t), stream));
    for (int shift = static_cast<int>(kSelectTopShift); shift >= 0; shift -= static_cast<int>(kSelectBits)) {
      hipLaunchKernelGGL(k_select_pass, dim3(strides), dim3(kInitBlock), 0, stream, d_sims, n_sims, d_selects, top, hist,
                         static_cast<uint32_t>(shift));
      INIT_TRY("k_select_pass", hipGetLastError());
    }
  }
  hipLaunchKernelGGL(k_init_finish, dim3(blocks), dim3(kInitBlock), 0, stream, d_sims, n_sims, d_selects);
  INIT_TRY("k_init_finish", hipGetLastError());
  if (house_blocks) {
    hipLaunchKernelGGL(k_init_cells, dim3(house_blocks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
    INIT_TRY("k_init_cells", hipGetLastError());
  }
  // the scratch is freed on return: finish with it first
  INIT_TRY("init sync", hipStreamSynchronize(stream));
  return hipSuccess;
}

hipError_t build_office_maps_on_device(const std::vector<OfficeJob>& jobs,
                                       std::vector<std::vector<uint32_t>>& workers_per_office, hipStream_t stream,
                                       std::string& err) {
  const uint32_t n_sims = static_cast<uint32_t>(jobs.size());
  std::vector<OfficeSim> sims(n_sims);
  std::vector<ScanJob> scans;
  uint32_t office_blocks = 0, chunks = 0;
  size_t offices = 0;
  workers_per_office.assign(n_sims, {});
  for (uint32_t i = 0; i < n_sims; ++i) {
    OfficeSim& a = sims[i];
    a = OfficeSim{};
    a.n = jobs[i].n;
    a.n_offices = std::max(jobs[i].n_offices, 1u);
    a.n_houses = std::max(jobs[i].n_houses, 1u);
    a.st = jobs[i].st;
    a.office_agent = jobs[i].office_agent;
    a.office_slot = jobs[i].office_slot;
    a.first_office = office_blocks;
    a.first_chunk = chunks;
    workers_per_office[i].assign(a.n_offices, 0);
    if (a.n == 0) continue;
    office_blocks += div_up(a.n_offices, kInitBlock);
    chunks += div_up(std::min(a.n_houses, a.n), kInitBlock);
    offices += a.n_offices;
  }
  if (chunks == 0) return hipSuccess;
  DeviceTemp tmp;
  uint32_t *cnt = nullptr, *base = nullptr, *rcnt = nullptr, *rbase = nullptr;
  OfficeSim* d_sims = nullptr;
  ScanJob* d_scans = nullptr;
  tmp.add(&d_sims, n_sims);
  tmp.add(&d_scans, 2 * static_cast<size_t>(n_sims));
  tmp.add(&cnt, offices);
  tmp.add(&base, offices);
  tmp.add(&rcnt, chunks);
  tmp.add(&rbase, chunks);
  INIT_TRY("office maps: alloc", tmp.alloc());
  size_t office = 0;
  for (OfficeSim& a : sims) {
    if (a.n == 0) continue;
    a.cnt = cnt + office;
    a.base = base + office;
    a.rcnt = rcnt + a.first_chunk;
    a.rbase = rbase + a.first_chunk;
    scans.push_back(ScanJob{a.cnt, a.base, a.n_offices});
    scans.push_back(ScanJob{a.rcnt, a.rbase, div_up(std::min(a.n_houses, a.n), kInitBlock)});
    office += a.n_offices;
  }
  INIT_TRY("office maps: upload", upload(d_sims, sims, stream));
  INIT_TRY("office maps: upload", upload(d_scans, scans, stream));
  hipLaunchKernelGGL(k_office_count, dim3(office_blocks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
  INIT_TRY("k_office_count", hipGetLastError());
  hipLaunchKernelGGL(k_rest_count, dim3(chunks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
  INIT_TRY("k_rest_count", hipGetLastError());
  hipLaunchKernelGGL(k_scan, dim3(static_cast<uint32_t>(scans.size())), dim3(1024), 0, stream, d_scans);
  INIT_TRY("k_scan", hipGetLastError());
  hipLaunchKernelGGL(k_office_place, dim3(office_blocks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
  INIT_TRY("k_office_place", hipGetLastError());
  hipLaunchKernelGGL(k_rest_place, dim3(chunks), dim3(kInitBlock), 0, stream, d_sims, n_sims);
  INIT_TRY("k_rest_place", hipGetLastError());
  std::vector<uint32_t> counts(offices);
  INIT_TRY("office maps: read counts",
           hipMemcpyAsync(counts.data(), cnt, offices * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
  // the scratch is freed on return: finish with it first
  INIT_TRY("office maps: sync", hipStreamSynchronize(stream));
  office = 0;
  for (uint32_t i = 0; i < n_sims; ++i) {
    if (sims[i].n == 0) continue;
    std::copy_n(counts.begin() + static_cast<ptrdiff_t>(office), sims[i].n_offices, workers_per_office[i].begin());
    office += sims[i].n_offices;
  }
  return hipSuccess;
}

}  // namespace epi
