// Citizen-state stream on gfx950: one hour's per-agent records formatted as JSON text on
// the device.
//
// The reference buffers (citizen id, state letter, location) for every agent each hour
// (engine/src/models/events/citizen_state.rs:26-68, filled from allocation_map.rs:122-124)
// and publishes the buffer with serde_json as one message per hour
// (listeners/events_kafka_producer.rs:62-67, 90-99). Here the message body, the records
// joined by commas, is written by two kernels:
//   k_record_len   : the total length of each block of 256 agents' records, and of each 16
//                    blocks together;
//   k_record_write : each block adds up the lengths before it, builds its text in LDS and
//                    stores it in aligned 16-byte pieces at its offset.
// The lengths are few and the prefix is summed where it is used, so there is no scan launch
// between the two (a one-block scan took 5 us of 39 at 1M agents and 79 of 341 at 10M).
// A record is {"citizen_id":"<id>","state":"<s|e|i|r|d>","location":{"x":<x>,"y":<y>}},
// preceded by a comma for every agent but the first. Agent ids are the dense deterministic
// ids, written as a JSON string where the reference writes a UUID string. A simulation
// that did not step the requested hour writes a total of 0.
#include <hip/hip_runtime.h>

#include <mutex>

#include "stream.hpp"

namespace epi {

// Scratch of the no-allocation formatter (epi_citizen_states_text_noalloc): the record
// lengths, one entry per 256-agent block, for at most kNoAllocMaxAgents agents (512 KiB on
// each GPU the library runs on, held until the process ends). Host code never passes this
// name to a kernel: it is a host-side stand-in, not a device address. noalloc_scratch()
// resolves the device's own copy once per device with hipGetSymbolAddress, and that
// address is what the kernels get.
static __device__ __align__(256) unsigned long long scratch[kNoAllocMaxBlocks];

namespace {

constexpr uint32_t kStreamBlock = 256, kWaves = kStreamBlock / 64;
constexpr uint32_t kGroup = 16;  // record blocks whose lengths are also added up together
static_assert(kNoAllocMaxBlocks * kStreamBlock == kNoAllocMaxAgents, "no-allocation scratch size");

// {"citizen_id":"  ","state":"?","location":{"x":  ,"y":  }}
constexpr uint32_t kFixed = 15 + 11 + 1 + 18 + 5 + 2;
static_assert(1 + kFixed + 10 + 5 + 5 == kMaxRecord, "record bound");

// The scratch array as 32-bit lengths: one per record block, then one per group (there are
// two words per block).
__device__ __forceinline__ uint32_t* block_lens(const StreamArgs& a) { return reinterpret_cast<uint32_t*>(a.block_off); }
__device__ __forceinline__ uint32_t* group_lens(const StreamArgs& a) {
  return block_lens(a) + (a.n + kStreamBlock - 1) / kStreamBlock;
}

__device__ __forceinline__ char state_letter(uint32_t w) {
  switch ((w >> B_STATE) & M_STATE) {  // CitizenState::state_str (citizen_state.rs:35-43)
    case ST_S: return 's';
    case ST_E: return 'e';
    case ST_I: return 'i';
    case ST_R: return 'r';
    default: return 'd';
  }
}

__device__ __forceinline__ bool stepped(const StreamArgs& a) { return a.state->hour == a.hour; }

// Digits of a coordinate (below 100,000) and of an id.
__device__ __forceinline__ uint32_t digits5(uint32_t v) {
  return 1u + (v >= 10u) + (v >= 100u) + (v >= 1000u) + (v >= 10000u);
}
__device__ __forceinline__ uint32_t digits10(uint32_t v) {
  return digits5(min(v, 99999u)) + (v >= 100000u) + (v >= 1000000u) + (v >= 10000000u) + (v >= 100000000u) +
         (v >= 1000000000u);
}

// Length of the records of ids 0 .. i-1 without their coordinates' digits: the fixed text, a
// comma before every record but the first, and i + sum over k of max(0, i - 10^k) id digits.
__device__ __forceinline__ uint64_t length_before(uint32_t i) {
  uint64_t s = static_cast<uint64_t>(i) * (kFixed + 2u) - (i ? 1u : 0u);
  uint32_t p = 10u;
#pragma unroll
  for (int k = 0; k < 9; ++k, p *= 10u) s += i > p ? i - p : 0u;
  return s;
}

// Coordinate digits of the lanes in `of`, over a wave: one for each coordinate, and one more
// for each power of ten it reaches.
template <class F>
__device__ __forceinline__ void for_powers(uint32_t p, F&& add) {
  const uint32_t x = p & 0xFFFFu, y = p >> 16;
  add(x >= 10u);
  add(y >= 10u);
  add(x >= 100u);
  add(y >= 100u);
  add(x >= 1000u);
  add(y >= 1000u);
  add(x >= 10000u);
  add(y >= 10000u);
}

// One block per group: wave w adds up record blocks w, w + 4, ... of it, all their words in
// flight together, with a ballot and a popcount per power of ten.
__global__ __launch_bounds__(kStreamBlock) void k_record_len(StreamArgs a) {
  __shared__ uint32_t part[kWaves];
  if (!stepped(a)) return;  // uniform
  constexpr uint32_t kPer = kGroup / kWaves;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t blocks = (a.n + kStreamBlock - 1) / kStreamBlock;
  uint32_t p[kPer * 4];
#pragma unroll
  for (uint32_t k = 0; k < kPer * 4; ++k) {
    const uint64_t i = (static_cast<uint64_t>(blockIdx.x) * kGroup + wave + kWaves * (k / 4)) * kStreamBlock +
                       64u * (k % 4) + lane;
    p[k] = i < a.n ? a.pos[i] : 0u;  // (0, 0) reaches no power of ten
  }
  uint32_t group = 0;
#pragma unroll
  for (uint32_t s = 0; s < kPer; ++s) {
    const uint32_t b = blockIdx.x * kGroup + wave + kWaves * s;
    if (b >= blocks) break;  // uniform
    const uint32_t first = b * kStreamBlock, past = min(a.n, first + kStreamBlock);
    uint32_t len = static_cast<uint32_t>(length_before(past) - length_before(first)) + 2u * (past - first);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
      for_powers(p[4 * s + k], [&](bool reaches) { len += static_cast<uint32_t>(__popcll(__ballot(reaches))); });
    group += len;
    if (lane == 0) block_lens(a)[b] = len;
  }
  if (lane == 0) part[wave] = group;
  __syncthreads();
  if (threadIdx.x == 0) group_lens(a)[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Four decimal digits of v < 10,000 as ASCII, first digit in the lowest byte.
__device__ __forceinline__ uint32_t ascii4(uint32_t v) {
  const uint32_t hi = v / 100u, lo = v % 100u;
  return (hi / 10u) | (hi % 10u) << 8 | (lo / 10u) << 16 | (lo % 10u) << 24 | 0x30303030u;
}
// The nd digits of a coordinate, first digit in the lowest byte, nothing above the last.
__device__ __forceinline__ uint64_t ascii5(uint32_t v, uint32_t nd) {
  const uint64_t all = (static_cast<uint64_t>(ascii4(v % 10000u)) << 8) | (0x30u + v / 10000u);
  return all >> (8u * (5u - nd));
}
// The last (at most eight) digits of an id that has nd of them.
__device__ __forceinline__ uint64_t ascii8(uint32_t v, uint32_t nd) {
  const uint64_t all = (static_cast<uint64_t>(ascii4(v % 10000u)) << 32) | ascii4(v / 10000u % 10000u);
  return all >> (8u * (8u - min(nd, 8u)));
}

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
constexpr uint64_t text8(const char (&s)[9]) {
  uint64_t v = 0;
  for (int k = 0; k < 8; ++k) v |= static_cast<uint64_t>(static_cast<unsigned char>(s[k])) << (8 * k);
  return v;
}
__device__ __forceinline__ void put8(char* o, uint64_t v) { __builtin_memcpy(o, &v, 8); }  // one ds_write_b64

// A lane writes its record from front to back in eleven 8-byte stores, each piece's surplus
// bytes overwritten by the next; the last one ends with the record. The text lies in LDS as
// far past a 16-byte boundary as in memory, so that whole 16-byte pieces are stored, past
// the caches (nothing here reads them again). 8 bytes read and 62 written per agent: 22 us at
// 1M agents (3.2 TB/s), 26.5 with a store per character, 62 of them, and one-byte stores to
// memory; the whole call 68 -> 37 us.
__global__ __launch_bounds__(kStreamBlock) void k_record_write(StreamArgs a) {
  __shared__ __align__(16) char text[16 + 16 + kStreamBlock * kMaxRecord + 16];
  __shared__ unsigned long long s_before[kWaves];
  __shared__ uint32_t s_wave[kWaves];
  if (!stepped(a)) {  // uniform: no text
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.total = 0;
    return;
  }
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t first = blockIdx.x * kStreamBlock, i = first + threadIdx.x;
  const bool valid = i < a.n;
  const uint32_t p = valid ? a.pos[i] : 0u, w = valid ? a.st[i] : 0u;
  // the text before this block: the groups before its own, then its group's blocks before it
  unsigned long long before = 0;
  const uint32_t group = blockIdx.x / kGroup;
  for (uint32_t k = threadIdx.x; k < group; k += kStreamBlock) before += group_lens(a)[k];
  if (threadIdx.x < blockIdx.x % kGroup) before += block_lens(a)[group * kGroup + threadIdx.x];
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  // coordinate digits before this lane in its wave, and the wave's
  uint32_t mine = 0, all = 0;
  for_powers(p, [&](bool reaches) {
    const uint64_t m = __ballot(reaches);
    mine += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
    all += static_cast<uint32_t>(__popcll(m));
  });
  if (lane == 0) {
    s_before[wave] = before;
    s_wave[wave] = all;
  }
  __syncthreads();
  before = s_before[0] + s_before[1] + s_before[2] + s_before[3];
  const uint64_t base = length_before(first);
  for (uint32_t v = 0; v < wave; ++v) mine += s_wave[v];
  const uint32_t past = min(a.n, first + kStreamBlock);
  const uint32_t len = static_cast<uint32_t>(length_before(past) - base) + 2u * (past - first) + s_wave[0] + s_wave[1] +
                       s_wave[2] + s_wave[3];
  char* const dst = a.text + before;
  const uint32_t phase = 16u + static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst) & 15u);
  if (valid) {
    const uint32_t at = static_cast<uint32_t>(length_before(i) - base) + 2u * threadIdx.x + mine;
    char* o = text + phase + at + (i ? 1u : 0u);  // at the brace; the first record has no comma
    put8(o - 1, text8(",{\"citiz"));
    put8(o + 7, text8("en_id\":\""));
    o += 15;
    const uint32_t nd = digits10(i);
    if (nd > 8u) {  // the digits above the last eight
      const uint32_t high = i / 100000000u;
      if (nd > 9u) *o++ = static_cast<char>('0' + high / 10u);
      *o++ = static_cast<char>('0' + high % 10u);
    }
    put8(o, ascii8(i, nd));
    o += min(nd, 8u);
    put8(o, text8("\",\"state"));
    put8(o + 8, text8("\":\"?\",\"l") ^ (static_cast<uint64_t>('?' ^ state_letter(w)) << 24));
    put8(o + 16, text8("ocation\""));
    put8(o + 22, text8("n\":{\"x\":"));
    o += 30;
    const uint32_t x = p & 0xFFFFu, y = p >> 16, nx = digits5(x), ny = digits5(y);
    put8(o, ascii5(x, nx));
    o += nx;
    // ,"y":<digits>}} is 7 + ny bytes: its first eight, then its last eight
    const uint64_t tail = ascii5(y, ny) | (static_cast<uint64_t>('}' | '}' << 8) << (8u * ny));
    const uint64_t t0 = (text8(",\"y\":   ") & 0xFFFFFFFFFFull) | (tail << 40), t1 = tail >> 24;
    const uint32_t sh = 8u * (ny - 1u);
    put8(o, t0);
    put8(o + ny - 1u, sh ? (t0 >> sh) | (t1 << (64u - sh)) : t0);
  }
  __syncthreads();
  // whole 16-byte pieces, and the bytes of the first and last one
  const uint32_t end = phase + len;
  for (uint32_t k = 16u + 16u * threadIdx.x; k < end; k += 16u * kStreamBlock) {
    if (k >= phase && k + 16u <= end) {
      __builtin_nontemporal_store(*reinterpret_cast<const v4u*>(text + k), reinterpret_cast<v4u*>(dst + (k - phase)));
    } else {
      for (uint32_t q = max(k, phase); q < min(k + 16u, end); ++q) dst[q - phase] = text[q];
    }
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *a.total = before + len;
}

}  // namespace

uint32_t max_record_bytes(uint32_t n, uint32_t stride, uint32_t height) {
  uint32_t nd_id = 1, nd_x = 1, nd_y = 1;
  for (uint32_t v = n ? n - 1 : 0; v >= 10u; v /= 10u) ++nd_id;
  for (uint32_t v = stride; v >= 10u; v /= 10u) ++nd_x;
  for (uint32_t v = height; v >= 10u; v /= 10u) ++nd_y;
  return 1u + kFixed + nd_id + nd_x + nd_y;
}

uint32_t stream_blocks(uint32_t n) { return (n + kStreamBlock - 1) / kStreamBlock; }

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned long long* g_scratch[kMaxDevices] = {};
}  // namespace

hipError_t noalloc_scratch(unsigned long long** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {  // the current device's copy of the array, resolved once
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch[dev] = static_cast<unsigned long long*>(p);
  }
  *out = g_scratch[dev];
  return hipSuccess;
}

hipError_t launch_citizen_states(const StreamArgs& a, hipStream_t stream) {
  const uint32_t blocks = stream_blocks(a.n);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_record_len, dim3((blocks + kGroup - 1) / kGroup), dim3(kStreamBlock), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_record_write, dim3(blocks), dim3(kStreamBlock), 0, stream, a);
  return hipGetLastError();
}

}  // namespace epi
