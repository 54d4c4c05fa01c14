// Device functions shared by the hour-step kernels: state-word fields, the 3 x 3 neighbourhood
// as masks, claim keys and decided sweeps.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "disease.hpp"
#include "kernels.hpp"
#include "philox.hpp"

namespace epi {
namespace {

constexpr int kWave = 64;
__device__ __forceinline__ uint32_t first_lane(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// A value at a uniform address that nothing in the launch changes before the read, by scalar
// loads: the constant address space says so where the compiler cannot prove it (it turns
// descriptor reads into vector loads when it sees a store that might come before).
template <class T>
__device__ __forceinline__ T scalar_copy(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  typedef const __attribute__((address_space(4))) uint32_t* Words;
  const Words q = (Words)reinterpret_cast<uintptr_t>(p);
  uint32_t w[sizeof(T) / 4];
#pragma unroll
  for (uint32_t k = 0; k < sizeof(T) / 4; ++k) w[k] = q[k];
  T t;
  __builtin_memcpy(&t, w, sizeof(T));
  return t;
}

// Makes the values pass through registers at this point: the loads producing them are
// issued before it and waited for once, together. Without it the compiler sinks each load
// to its first use, behind the wait for another, and a lane pays one memory round trip per
// word instead of one for all of them. The asm has outputs and no side effects, so it is
// no memory clobber: descriptor reads after it still come from the scalar cache.
__device__ __forceinline__ void loaded_together(uint32_t& a, uint32_t& b, uint32_t& c) {
  asm("" : "+v"(a), "+v"(b), "+v"(c));
}
// The same with a uniform word that the next branch tests: it passes through too, so the loads
// are not sunk behind the branch (and behind the wait for that word).
__device__ __forceinline__ void loaded_together(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& uniform) {
  asm("" : "+v"(a), "+v"(b), "+v"(c), "+s"(uniform));
}
// And for two loaded words and a draw block computed while they are in flight: the
// draw's words pass through the barrier too, so its rounds are scheduled before the wait.
__device__ __forceinline__ void loaded_together(uint32_t& a, uint32_t& b, Philox9& d, uint32_t& uniform) {
  asm("" : "+v"(a), "+v"(b), "+v"(d.c0), "+v"(d.c1), "+v"(d.c2), "+v"(d.c3), "+s"(uniform));
}

// Sum over the wave, in lane 63: adds across lanes by DPP (rows of 16, then their last lanes
// broadcast on), a few cycles a step where a shuffle through LDS takes over a hundred (the
// epilogue's six sums: 3,250 cycles of its 7,000).
__device__ __forceinline__ uint32_t wave_sum(uint32_t x) {
#define EPI_DPP_ADD(ctrl, rows) \
  x += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), ctrl, rows, 0xF, false))
  EPI_DPP_ADD(0x111, 0xF);  // row_shr:1
  EPI_DPP_ADD(0x112, 0xF);  // row_shr:2
  EPI_DPP_ADD(0x114, 0xF);  // row_shr:4
  EPI_DPP_ADD(0x118, 0xF);  // row_shr:8
  EPI_DPP_ADD(0x142, 0xA);  // row_bcast:15 into rows 1 and 3
  EPI_DPP_ADD(0x143, 0xC);  // row_bcast:31 into rows 2 and 3
#undef EPI_DPP_ADD
  return x;
}

// Lanes set in a wave's mask, and `x` with lane `lane` replaced, both on the scalar unit.
__device__ __forceinline__ uint32_t wave_count(uint64_t mask) { return static_cast<uint32_t>(__builtin_popcountll(mask)); }
template <int LANE>
__device__ __forceinline__ uint32_t lane_word(uint32_t x, uint32_t value) {
  asm("v_writelane_b32 %0, %1, %2" : "+v"(x) : "s"(value), "n"(LANE));
  return x;
}

__device__ __forceinline__ bool contains(const Rect& a, int32_t x, int32_t y) {
  return (a.x0 <= x) & (a.x1 >= x) & (a.y0 <= y) & (a.y1 >= y);  // no branches
}
__device__ __forceinline__ bool same_rect(const Rect& a, const Rect& b) {
  return a.x0 == b.x0 && a.y0 == b.y0 && a.x1 == b.x1 && a.y1 == b.y1;
}

// Moore neighbour order (point.rs:57-61): (-1,-1) (0,-1) (1,-1) (-1,0) (1,0) (-1,1) (0,1) (1,1),
// offsets as two-bit fields of a constant, and the neighbours of each edge as eight bits.
__device__ __forceinline__ int32_t moore_dx(uint32_t k) {
  return static_cast<int32_t>((0x9224u >> (2u * k)) & 3u) - 1;
}
__device__ __forceinline__ int32_t moore_dy(uint32_t k) {
  return static_cast<int32_t>((0xA940u >> (2u * k)) & 3u) - 1;
}
constexpr uint32_t kMooreLeft = 0x29u, kMooreRight = 0x94u, kMooreTop = 0x07u, kMooreBottom = 0xE0u;

__device__ __forceinline__ uint32_t fld(uint32_t w, uint32_t b, uint32_t m) { return (w >> b) & m; }
__device__ __forceinline__ uint32_t set_fld(uint32_t w, uint32_t b, uint32_t m, uint32_t v) {
  return (w & ~(m << b)) | ((v & m) << b);
}

// Index of cell (x, y) in the claim array of one simulation. A simulation
// has fewer than 2^32 padded cells (grid_size <= 32,000), so the index is 32-bit and a
// load adds it to the simulation's base as an unsigned offset.
__device__ __forceinline__ uint32_t cell_index(uint32_t pitch, int32_t x, int32_t y) {
  return __umul24(static_cast<uint32_t>(y) + kPadY, pitch) + static_cast<uint32_t>(x) + kPadX;
}
__device__ __forceinline__ uint32_t cell_index(const SimDesc& D, int32_t x, int32_t y) {
  return cell_index(D.pitch, x, y);
}

// 3 x 3 neighbourhood masks: bit 3 * (dy + 1) + (dx + 1) stands for the cell at offset
// (dx, dy), row-major, so bit 4 is the centre. moore8 drops the centre, which leaves the
// Moore order of point.rs:57-61: (-1,-1) (0,-1) (1,-1) (-1,0) (1,0) (-1,1) (0,1) (1,1).
// Index of the n-th (0-based) set bit of an 8-bit mask m, n < popcount(m): two halving
// steps on popcounts and a last compare, the same work for every n (a loop clearing n bits
// runs as long as the wavefront's largest n).
__device__ __forceinline__ uint32_t nth_bit8(uint32_t m, uint32_t n) {
  uint32_t base = 0;
  const uint32_t c4 = __builtin_popcount(m & 0xFu);
  if (n >= c4) {
    n -= c4;
    m >>= 4;
    base = 4;
  }
  const uint32_t c2 = __builtin_popcount(m & 0x3u);
  if (n >= c2) {
    n -= c2;
    m >>= 2;
    base += 2;
  }
  return base + (n >= (m & 1u) ? 1u : 0u);
}

__device__ __forceinline__ uint32_t moore8(uint32_t m9) { return (m9 & 0xFu) | ((m9 >> 1) & 0xF0u); }

// Bit j (j = 0..2) set iff lo <= base + j <= hi.
__device__ __forceinline__ uint32_t span3(int32_t base, int32_t lo, int32_t hi) {
  const int32_t from = min(max(lo - base, 0), 3), past = min(max(base + 2 - hi, 0), 3);
  return (0x7u << from) & (0x7u >> past) & 0x7u;
}

typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;
// Two words at base + off, off a multiple of 4.
__device__ __forceinline__ uint2 load_words2(GlobalBytes base, uint32_t off) {
  typedef uint64_t Words __attribute__((aligned(4)));
  const uint64_t q = *reinterpret_cast<const __attribute__((address_space(1))) Words*>(base + off);
  return make_uint2(static_cast<uint32_t>(q), static_cast<uint32_t>(q >> 32));
}
// The bytes of q from byte `first` (0..3) on.
__device__ __forceinline__ uint64_t from_byte(uint2 q, uint32_t first) {
  return join64(q.y >> (8u * first), __builtin_amdgcn_alignbyte(q.y, q.x, first));
}
// Bytes `first` .. first + 3 (first <= 3) of a window row: columns px-1, px, px+1 and one more.
__device__ __forceinline__ uint32_t three(uint64_t row, uint32_t first) {
  return __builtin_amdgcn_alignbyte(static_cast<uint32_t>(row >> 32), static_cast<uint32_t>(row), first);
}
// Bit 0 of the low three bytes of three words (rows y-1, y, y+1) as the eight neighbours, the
// centre dropped: products with byte weights, added up.
__device__ __forceinline__ uint32_t pack8(uint32_t top, uint32_t mid, uint32_t bottom) {
  constexpr uint32_t kBit0 = 0x01010101u;
  return __builtin_amdgcn_udot4(
      top & kBit0, 0x00040201u,
      __builtin_amdgcn_udot4(mid & kBit0, 0x00100008u,
                             __builtin_amdgcn_udot4(bottom & kBit0, 0x00804020u, 0u, false), false),
      false);
}
// Four grid bytes (0..3) as four bits, set where occupied.
__device__ __forceinline__ uint32_t occupied4(uint32_t bytes) {
  return __builtin_amdgcn_udot4((bytes | (bytes >> 1)) & 0x01010101u, 0x08040201u, 0u, false);
}
// The vacant ones among the eight neighbours of the cell in byte 2 of the middle row; a
// grid byte is 0..3, so a cell is occupied iff one of its two low bits is set.
__device__ __forceinline__ uint32_t vacant8(uint64_t above, uint64_t row, uint64_t below) {
  const uint32_t t = three(above, 1), m = three(row, 1), b = three(below, 1);
  return pack8(t | (t >> 1), m | (m >> 1), b | (b >> 1)) ^ 0xFFu;
}

// Claim key of agent `id` at `hour`: hours of day 7..23, 0 (the hours that move anyone)
// rank 0..17 since the reset at hour of day 2; a later hour takes a smaller top field, so
// its claims undercut any left from earlier hours of the day, and within an hour the
// lowest id wins.
__device__ __forceinline__ uint32_t claim_key(uint32_t hour, uint32_t id) {
  const uint32_t rank = (hour % 24u + 17u) % 24u;
  return ((31u - rank) << kClaimIdBits) | id;
}

// A decided sweep (allocation_map.rs:349-387): vaccination of susceptible agents (a
// Bernoulli keyed by the vaccination hour), lockdown isolation of everyone but essential
// workers, unlock. Applying it twice gives the same word.
struct Sweep {
  uint32_t mask, vacc_hour;
  unsigned long long vacc_thr;
};
// The sweep in the slot of parity p (filled by the epilogue of an hour of that parity).
__device__ __forceinline__ Sweep sweep_slot(const SimState& S, uint32_t p) {
  return Sweep{S.sweep[p], S.sweep_vacc_hour[p], S.sweep_vacc_thr[p]};
}
__device__ __forceinline__ uint32_t apply_sweep(uint32_t w, const Sweep& sw, uint32_t local, const SimDesc& D) {
  const uint32_t sweep = sw.mask;
  if ((sweep & SWEEP_VACC) && fld(w, B_STATE, M_STATE) == ST_S) {
    const u32x4 d = philox4x32_10(local, sw.vacc_hour, SITE_VACCINATE, 0, D.seed_lo, D.seed_hi);
    if (bernoulli(sw.vacc_thr, join64(d.w[0], d.w[1]))) w |= F_VACC;
  }
  if ((sweep & SWEEP_LOCK) && fld(w, B_WS, M_WS) != WS_ESSENTIAL) w |= F_ISO;
  if (sweep & SWEEP_UNLOCK) w &= ~F_ISO;
  return w;
}

}  // namespace
}  // namespace epi
