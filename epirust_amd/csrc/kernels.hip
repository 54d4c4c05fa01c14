// Hour-step kernels for gfx950.
//
// One hour of EpiRust's standalone engine (engine/src/allocation_map.rs:67-134 and
// :306-337, engine/src/citizen/mod.rs:227-454, default_disease_handler.rs:31-103) is
//   [hour-of-day 0 only] k_hospital_scan : first vacant hospital cell of the snapshot
//   k_step   : [hours of day 0, 7..23] per agent, the previous hour's vaccination /
//              lockdown sweep, then routine + disease update against the start-of-hour
//              grid; state written in place (it is read by no other agent) when it
//              changes, the chosen cell written to the target word and claimed with a
//              32-bit atomicMin keyed (claim hour, agent id) unless the office filter or
//              housemate arbitration settles it; S/E/I/H/R/D counted with wavefront
//              ballots into per-block partials.
//   k_commit : hours of day 0 and 7..23. Its first blocks, one per simulation, run the epilogue:
//              reduce the partials, write the row, run the intervention triggers and the
//              stop rule on device; the row and the state go to device memory and to the
//              host's pinned copies, which a step call reads after its one drain. The other
//              blocks run the hour's agent pass, which
//              reads nothing the same hour's epilogue writes (its hour and its sweep come
//              from parity slots the previous epilogue filled), so the two share a launch.
//              The agent pass commits the moves (the claim winner moves, grid bytes are
//              updated).
//   k_rest   : hours of day 1..6, which move nobody and change no state but flags and areas
//              (citizen/mod.rs:244-248): the epilogue repeats the last counts and the agent
//              pass applies the pending sweep, sets non-staff areas to home at hour of day 1
//              and resets the claim array at 2.
//   k_relayout: [hours of day 8 and 16] moves st and pos between the home layout
//              (slot = agent id) and the office layout that hours of day 8..15 run on:
//              each office's workers in consecutive slots, packed whole into blocks,
//              then everyone else house by house. There k_step resolves the claims of each
//              office's cells among the block's workers in LDS, and the winners on
//              offices that lie wholly in one block (all of them when an office fits a
//              block) claim nothing globally.
//              Small handles, and days on which most agents are isolated, stay in the home
//              layout throughout.
//   k_night / k_quiet_hours: hours of day 1..6 (or 3..6) of one call as one launch when no
//              sweep can be pending inside them (no vaccination there).
// A sweep decided at hour h (allocation_map.rs:306-337) is applied by the agent pass of
// hour h+1 (before the routine, in k_step), which is what the reference's next hour sees;
// sweeps are idempotent, so k_apply_sweep re-applies the last one before the host reads
// agents.
// Every kernel is batched: blocks map to (simulation, agent range) through a table, so
// many independent replicates share one launch. Nothing here uses MFMA: the step is
// integer work, priced against HBM bandwidth (its per-agent bytes are few; at 1M agents
// the grid stays in the caches and the step is bound by VALU issue and memory latency).
#include <hip/hip_runtime.h>

#include <cstddef>

#include "kernels.hpp"
#include "step_device.hpp"

namespace epi {
namespace {

// Office-hour block claim filter: 100 cells per 10 x 10 office, for the at most
// kMaxFilterOffices offices of a block.
constexpr uint32_t kOfficeCells = 100u, kFilterCells = kMaxFilterOffices * kOfficeCells, kNoCell = ~0u;
// Target word flags (x and y never exceed 32000, so bits 15 and 31 are free):
//   kTgtWon   the move has already won (office-hour block claim filter);
//   kTgtHouse a home-layout move into a cell of the agent's own house, arbitrated in the
//             commit among the house's agents instead of by a global claim.
// Every agent writes its target word at every step hour, movers or not, so the commit
// tells movers by it (no flag in the state word, which then changes, and is written, only
// when the agent's state does) and the words housemates read are this hour's.
constexpr uint32_t kTgtWon = 1u << 31;
constexpr uint32_t kTgtHouse = 1u << 15;
constexpr uint32_t kTgtCell = ~(kTgtWon | kTgtHouse);
// A non-mover: its cell part (x = y = 32767) is no cell, so it equals no move's word.
constexpr uint32_t kTgtNone = ~0u;
constexpr uint32_t kNoState = 5u;  // in the state bits of a lane without an agent
constexpr uint32_t kMaxWaves = 16;  // of a block of 1,024 threads

// k_step is compiled once per class of hours of day that take the same branches of the
// routine: every test of the hour folds, and with it the code of the other hours (static
// VALU / SALU instructions and scalar loads of an evening hour: 1,314 / 1,180 / 79 in one
// kernel for all hours, 832 / 556 / 37 in its own), which shortens what a small simulation's
// few waves wait for (10k agents 7.64 -> 7.25 us an hour, 100k 8.57 -> 8.31).
enum HourClass : uint32_t {
  HOURS_0,      // hospital admission
  HOURS_7_17,   // public transport, the others stay
  HOURS_8,      // to work
  HOURS_9_15,   // in the office; non-workers in the housing area until 12, at home after
  HOURS_16,     // home
  HOURS_18_22,  // where one is
  HOURS_23      // recovery or death
};
constexpr uint32_t first_hour(HourClass c) {
  return c == HOURS_0 ? 0u : c == HOURS_7_17 ? 7u : c == HOURS_8 ? 8u : c == HOURS_9_15 ? 9u : c == HOURS_16 ? 16u
         : c == HOURS_18_22 ? 18u : 23u;
}
constexpr uint32_t last_hour(HourClass c) {
  return c == HOURS_7_17 ? 17u : c == HOURS_9_15 ? 15u : c == HOURS_18_22 ? 22u : first_hour(c);
}
constexpr bool on_office_layout(HourClass c) { return c == HOURS_8 || c == HOURS_9_15; }
// Whether an hour of day of class C is `at`.
template <HourClass C>
__device__ __forceinline__ bool is_hour(uint32_t hd, uint32_t at) {
  if (at < first_hour(C) || at > last_hour(C)) return false;
  if (C == HOURS_7_17 && at != 7u && at != 17u) return false;
  return first_hour(C) == last_hour(C) || hd == at;
}

// Hour of day 2: block b of a simulation's n_blocks resets its share of the claim array
// (all padded cells, in 16-byte stores; the array of each simulation is a multiple of 4
// cells long and starts at a multiple of 4). The share is computed before the block's
// first store, while the descriptor still comes from the scalar cache.
struct ClaimShare {
  uint4* q;
  uint32_t begin, end;
};
__device__ __forceinline__ ClaimShare claim_share(const DevView& v, const SimDesc& D, uint32_t b) {
  const uint32_t quads = D.pitch / 4u * (D.height + 2u * kPadY);
  const uint32_t per = (quads + D.n_blocks - 1u) / D.n_blocks;
  return ClaimShare{reinterpret_cast<uint4*>(v.claim + D.cell_off), b * per, min(quads, (b + 1u) * per)};
}
__device__ __forceinline__ void reset_claims(const ClaimShare& c) {
  for (uint32_t k = c.begin + threadIdx.x; k < c.end; k += blockDim.x) c.q[k] = make_uint4(~0u, ~0u, ~0u, ~0u);
}

// Per-thread state of one agent's hour.
struct Agent {
  const SimDesc& D;
  const SimState& S;
  const uint8_t* __restrict__ occ;  // this simulation's grid
  const uint32_t seed_lo, seed_hi;  // read up front too
  // Transmission thresholds, read once up front: a per-lane choice between two descriptor
  // fields would otherwise become a per-lane load of the chosen field.
  const uint64_t thr_regular, thr_high;
  uint32_t id, h, w, tm, wsa;
  uint32_t tm0 = 0;  // tm as stored: loaded for the states that carry an at_hour, else 0
  uint32_t* tm_arr = nullptr;  // this agent's stored tm word
  int32_t x, y;                     // current cell
  int32_t tx, ty;                   // chosen cell
  int32_t hx = 0, hy = 0;           // home house origin (house id % H)
  int32_t ox = 0, oy = 0;           // office origin (office id % O)
  // The hour's movement and disease draw blocks, computed once up front (one inlined
  // Philox each) for the hours / states that can use them; the movement's last round is left
  // to the words that are read (all but a few agents read one).
  Philox9 mv{};
  u32x4 dz{{0, 0, 0, 0}};
  // 5x5 grid window around (wx, wy): the eight bytes of each row from column wx - 2 on.
  int32_t wx = 0, wy = 0;
  uint64_t r0 = 0, r1 = 0, r2 = 0, r3 = 0, r4 = 0;  // named, so no variable-index access exists

  __device__ Agent(const SimDesc& d, const SimState& s, const uint8_t* o)
      : D(d), S(s), occ(o), seed_lo(d.seed_lo), seed_hi(d.seed_hi), thr_regular(Disease::transmission_threshold(d.dz, 1u)),
        thr_high(Disease::transmission_threshold(d.dz, 2u)) {}

  __device__ __forceinline__ u32x4 dr(uint32_t site, uint32_t block) const {
    return philox4x32_10(id, h, site, block, seed_lo, seed_hi);
  }
  __device__ __forceinline__ void draw_move() { mv = philox4x32_9(id, h, SITE_MOVE, seed_lo, seed_hi); }
  __device__ __forceinline__ const u32x4& disease_words() const { return dz; }

  __device__ __forceinline__ uint32_t state() const { return fld(w, B_STATE, M_STATE); }
  __device__ __forceinline__ uint32_t sev() const { return fld(w, B_SEV, M_SEV); }
  __device__ __forceinline__ uint32_t ws() const { return fld(w, B_WS, M_WS); }
  __device__ __forceinline__ bool symptomatic() const {
    static_assert(SEV_MILD == 2 && SEV_SEVERE == 3, "both have the field's high bit set");
    return (w & ((M_STATE << B_STATE) | (2u << B_SEV))) == ((ST_I << B_STATE) | (2u << B_SEV));
  }
  __device__ __forceinline__ bool can_move() const {  // citizen/mod.rs:452-454
    return !(symptomatic() || (w & (F_HOSP | F_ISO)) || state() == ST_D);
  }
  // Home house id % H and office id % O, tiled row-major (area.rs:95-117), once per hour
  // with the division constants of the tiling. The office is needed only at hours of day
  // 8..16: a worker's area is its office from 8 to 16 (goto home resets it at 16, the
  // sleep hours reset it to home), the office is the target at 8, and the symptomatic-at-
  // work override of goto home is tested at 16; at other hours ox, oy are left unset and
  // every expression that reads them is masked by a condition that is false then.
  __device__ __forceinline__ void locate_buildings(bool office) {
    const uint32_t hk = fast_mod(id, D.fd_houses), hrow = fast_div(hk, D.fd_house_nx);
    hx = D.house_sx + static_cast<int32_t>(hk - hrow * D.fd_house_nx.d) * 2;
    hy = D.house_sy + static_cast<int32_t>(hrow) * 2;
    if (office) {
      const uint32_t ok = fast_mod(id, D.fd_offices), orow = fast_div(ok, D.fd_office_nx);
      ox = D.office_sx + static_cast<int32_t>(ok - orow * D.fd_office_nx.d) * 10;
      oy = D.office_sy + static_cast<int32_t>(orow) * 10;
    }
  }
  __device__ __forceinline__ Rect home() const { return Rect{hx, hy, hx + 1, hy + 1}; }
  __device__ __forceinline__ bool in_house(int32_t cx, int32_t cy) const {
    return static_cast<uint32_t>((cx - hx) | (cy - hy)) <= 1u;
  }
  __device__ __forceinline__ Rect work() const {  // non-workers' work location is home
    return ws() == WS_NA ? home() : Rect{ox, oy, ox + 9, oy + 9};
  }
  __device__ __forceinline__ Rect area_rect(uint32_t tag) const {
    Rect a = home();
    if (tag != AREA_HOME) {
      if (tag == AREA_WORK) a = work();
      else if (tag == AREA_TRANSPORT) a = D.transport;
      else if (tag == AREA_HOUSING) a = D.housing;
      else if (tag == AREA_HOSP0) a = D.hosp[0];
      else a = D.hosp[1];
    }
    return a;
  }
  __device__ __forceinline__ Rect current_area() const { return area_rect(fld(w, B_AREA, M_AREA)); }
  __device__ __forceinline__ void set_area(uint32_t tag) { w = set_fld(w, B_AREA, M_AREA, tag); }

  __device__ __forceinline__ bool vacant(int32_t cx, int32_t cy) const {
    return occ[grid_place(D.strip, static_cast<uint32_t>(cx), static_cast<uint32_t>(cy)).at] == 0;
  }
  // The cells around (cx, cy) that lie in rect a and in the grid (area.rs:83-88 and
  // allocation_map.rs:156-159 for each neighbour), in the order of the eight neighbours.
  // Areas start at coordinates >= 0 but may end past the grid.
  __device__ __forceinline__ uint32_t allowed8(const Rect& a, int32_t cx, int32_t cy) const {
    const int32_t last = static_cast<int32_t>(D.g) - 1;
    const int32_t x1 = min(a.x1, last), y1 = min(a.y1, last);
    if ((cx >= a.x0) & (cx <= x1) & (cy >= a.y0) & (cy <= y1))  // nearly always: only the edges' neighbours are out
      return 0xFFu & ~((cx == a.x0 ? kMooreLeft : 0u) | (cx == x1 ? kMooreRight : 0u) |
                       (cy == a.y0 ? kMooreTop : 0u) | (cy == y1 ? kMooreBottom : 0u));
    const uint32_t cols = span3(cx - 1, a.x0, x1), rows = span3(cy - 1, a.y0, y1);
    return moore8(cols * ((rows & 1u) | ((rows & 2u) << 2) | ((rows & 4u) << 4)));  // cols copied to each row
  }
  // Five independent loads of the two aligned words that hold columns cx-2..cx+2 of a row (an
  // unaligned eight-byte load takes twice the L1 accesses: 10M agents 161 us an hour, 153 with
  // these), a strip's row apart, then shifted to column cx-2.
  __device__ __forceinline__ void load_window(int32_t cx, int32_t cy) {
    const uint32_t first = static_cast<uint32_t>(cx) + (kPadX - 2u), k = strip_of(first);
    const uint32_t b = first - k * kStripStep;
    const uint32_t off = strip_start(D.strip, k) + (static_cast<uint32_t>(cy) + (kPadY - 2u)) * kStripRow + (b & ~3u);
    const GlobalBytes base = (GlobalBytes)occ;
    uint2 q[5];
#pragma unroll
    for (uint32_t r = 0; r < 5; ++r) q[r] = load_words2(base + r * kStripRow, off);
    r0 = from_byte(q[0], b & 3u);
    r1 = from_byte(q[1], b & 3u);
    r2 = from_byte(q[2], b & 3u);
    r3 = from_byte(q[3], b & 3u);
    r4 = from_byte(q[4], b & 3u);
    wx = cx;
    wy = cy;
  }
  // Make the window cover the 3x3 neighbourhood of (cx, cy).
  __device__ __forceinline__ void cover(int32_t cx, int32_t cy) {
    if (static_cast<uint32_t>(cx - wx + 1) > 2u || static_cast<uint32_t>(cy - wy + 1) > 2u) load_window(cx, cy);
  }
  __device__ __forceinline__ void random_point(const Rect& a, int32_t& px, int32_t& py) {  // area.rs:76-81
    px = a.x0 + static_cast<int32_t>(below(mv.word0(), static_cast<uint32_t>(a.x1 - a.x0 + 1)));
    py = a.y0 + static_cast<int32_t>(below(mv.word1(), static_cast<uint32_t>(a.y1 - a.y0 + 1)));
  }
  // move_agent (allocation_map.rs:136-142): the target if vacant in the snapshot, else stay
  __device__ __forceinline__ void move_to(int32_t px, int32_t py) {
    if (vacant(px, py)) { tx = px; ty = py; }
  }

  // The hour's movement primitive. Every path of perform_movements ends in at most one of
  //   ACT_LOCAL: move_agent_from (citizen/mod.rs:415-432): from the current cell, or from a
  //              random point of the current area when outside it, to a random vacant
  //              Moore neighbour inside the area;
  //   ACT_TELE : goto_area for a working citizen (citizen/mod.rs:367-395): a random point
  //              of the target area if vacant (a non-worker's goto_area is ACT_LOCAL).
  // Lanes choose their primitive first and one shared copy runs, so a wavefront mixing work
  // statuses pays for one window load and one neighbour scan.
  enum : uint32_t { ACT_NONE = 0, ACT_LOCAL = 1, ACT_TELE = 2 };

  // goto_area's gate for a working citizen: can_move, or the symptomatic-at-work override.
  __device__ __forceinline__ uint32_t tele_act(const Rect& target) const {
    const uint32_t s = ws();
    const bool override_movement = (s == WS_NORMAL || s == WS_ESSENTIAL) && symptomatic() &&
                                   same_rect(target, home()) && contains(work(), x, y);
    return (can_move() || override_movement) ? ACT_TELE : ACT_NONE;
  }

  // Every lane takes the window of the cell that it may move from, or of its own when it stays
  // (the infection scan reads it), so that the common case has no branches. A wave of an
  // evening hour issues 345 vector instructions, 415 with a path per case (10M agents 158 -> 151
  // us an hour, 1M 19.6 -> 18.9, 32 runs of 100k 48.9 -> 45.4; loads through L1 bound it next).
  // `tag` is the area of the move: the target's for ACT_TELE, else the current one.
  __device__ __forceinline__ void move(uint32_t act, uint32_t tag) {
    const bool tele = act == ACT_TELE, local = (act == ACT_LOCAL) & can_move();
    const Rect a = area_rect(tag);
    int32_t lx = x, ly = y;
    if (tele | (local & !contains(a, x, y))) random_point(a, lx, ly);  // vacancy not checked
    load_window(lx, ly);
    // vacant Moore neighbours of (lx, ly) in the area and the grid: bytes 1..3 of the rows
    // ly-1 .. ly+1
    const uint32_t cand = local ? vacant8(r1, r2, r3) & allowed8(a, lx, ly) : 0u;
    const uint32_t n = __builtin_popcount(cand);
    const uint32_t k = nth_bit8(cand, below(mv.word2(), n));
    if (n != 0) {
      tx = lx + moore_dx(k);
      ty = ly + moore_dy(k);
    }
    if (tele & ((static_cast<uint32_t>(r2) & 0xFF0000u) == 0)) {  // the point itself
      tx = lx;
      ty = ly;
    }
  }

  // default_disease_handler.rs:64-86 as an OR over fixed per-neighbour draws: first the
  // mask of eligible infectious neighbours of (tx, ty) from the window (rows chosen with
  // bit masks, so no variable indexing), then the draws (infected_by).
  uint32_t hot = 0, high = 0;  // infectious neighbours, in Moore order, and those in the high window
  __device__ __forceinline__ void find_infectious() {
    if (!Disease::can_catch(w)) return;
    cover(tx, ty);
    // No infectious cell (byte >= 2) anywhere in the 5 x 5 window, a superset of the
    // neighbourhood: nothing to test, and no draw is made. Most agents, and whole waves,
    // take this exit while infections are rare.
    if (((r0 | r1 | r2 | r3 | r4) & 0xFEFEFEFEFEull) == 0) return;
    const int32_t ox = tx - wx, oy = ty - wy;  // both in [-1, 1]
    const uint64_t mm = oy < 0 ? ~0ull : 0ull, m0 = oy == 0 ? ~0ull : 0ull, mp = oy > 0 ? ~0ull : 0ull;
    const uint64_t top = (r0 & mm) | (r1 & m0) | (r2 & mp);
    const uint64_t mid = (r1 & mm) | (r2 & m0) | (r3 & mp);
    const uint64_t bot = (r2 & mm) | (r3 & m0) | (r4 & mp);
    // infectious neighbours (grid byte >= 2, i.e. a byte with a bit above bit 0) and the
    // high-window ones (byte 3) among the cells of the area and the grid
    const uint32_t c = static_cast<uint32_t>(ox + 1);
    const uint32_t bt = three(top, c), bm = three(mid, c), bb = three(bot, c);
    const uint32_t infectious = pack8(bt >> 1, bm >> 1, bb >> 1);
    if (infectious == 0) return;  // before the area's masks, which few agents need
    hot = infectious & allowed8(current_area(), tx, ty);
    high = pack8(bt & (bt >> 1), bm & (bm >> 1), bb & (bb >> 1)) & hot;
  }
  // The draws of agent `who` against its infectious neighbours: one Philox block per pair of
  // neighbours, drawn in Moore order only for infectious ones.
  __device__ __forceinline__ bool infected_by(uint32_t who, uint32_t infectious, uint32_t in_high) const {
    int blk = -1;
    uint32_t q0 = 0, q1 = 0, q2 = 0, q3 = 0;
    while (infectious) {
      const int k = __builtin_ctz(infectious);
      infectious &= infectious - 1;
      if ((k >> 1) != blk) {
        blk = k >> 1;
        const u32x4 q = philox4x32_10(who, h, SITE_INFECT, static_cast<uint32_t>(blk), seed_lo, seed_hi);
        q0 = q.w[0]; q1 = q.w[1]; q2 = q.w[2]; q3 = q.w[3];
      }
      const uint64_t v = (k & 1) ? join64(q2, q3) : join64(q0, q1);
      const uint64_t thr = ((in_high >> k) & 1u) ? thr_high : thr_regular;
      if (bernoulli(thr, v)) return true;
    }
    return false;
  }

  // The stored at_hour of a state that carries one (Exposed, Pre), read where it is needed.
  __device__ __forceinline__ void load_tm() {
    if (Disease::timed(w)) tm = tm0 = *tm_arr;
  }

  // DiseaseStateMachine::next (disease_state_machine.rs:53-70): the handler's transition of
  // the current state; on_susceptible is the neighbour scan and the draws above.
  __device__ __forceinline__ void update_infection_dynamics() {
    const uint32_t s = state();
    if (s == ST_S) {
      find_infectious();
      if (hot && infected_by(id, hot, high)) Disease::on_caught(h, w, tm);
    } else if (s == ST_E) {
      load_tm();
      Disease::on_exposed(D.dz, h, disease_words(), w, tm);
    } else if (s == ST_I) {
      load_tm();
      Disease::on_infected(D.dz, h, disease_words(), w, tm);
    }
  }

  // citizen/mod.rs:257-349: choose the primitive and the area it leads to, run it, then the
  // disease update (skipped by the hospital-staff quarantine transitions, which return early).
  template <HourClass C>
  __device__ __forceinline__ void perform_movements(uint32_t hd) {
    const uint32_t s = ws(), here = fld(w, B_AREA, M_AREA);
    uint32_t act = ACT_LOCAL, tag = here;
    bool disease = true;
    if (s == WS_STAFF) {
      const uint32_t since = h > wsa ? h - wsa : 0u;  // saturating_sub
      act = ACT_NONE;
      if (since == 24u * 14u) {
        w |= F_WQ;
        disease = false;
      } else if (since == 24u * 14u * 2u) {
        act = tele_act(home());
        tag = AREA_HOME;
        wsa = h + 24u * 14u;
        disease = false;
      } else if (is_hour<C>(hd, 8)) {
        const uint32_t ver = S.hosp_version;
        if (!same_rect(current_area(), D.hosp[ver]) && wsa <= h) {
          act = tele_act(D.hosp[ver]);
          tag = AREA_HOSP0 + ver;
          wsa = h;
        }
        w &= ~F_WQ;
      } else if (is_hour<C>(hd, 16)) {
        w |= F_WQ;
      } else if (!(w & F_WQ)) {
        act = ACT_LOCAL;
      }
    } else if (s != WS_NA) {
      if (C == HOURS_7_17 && (w & F_PT)) {
        act = tele_act(D.transport);
        tag = AREA_TRANSPORT;
      } else if (is_hour<C>(hd, 8)) {
        act = can_move() ? ACT_TELE : ACT_NONE;  // an office is no home
        tag = AREA_WORK;
      } else if (is_hour<C>(hd, 16)) {
        act = tele_act(home());
        tag = AREA_HOME;
      }
    }
    move(act, tag);
    // goto_area of a non-worker is move_agent_from in the area it is still in
    if (s == WS_NA && is_hour<C>(hd, 8)) tag = AREA_HOUSING;
    if (s == WS_NA && is_hour<C>(hd, 12)) tag = AREA_HOME;
    if (tag != here) set_area(tag);
    if (disease) update_infection_dynamics();
  }

  // citizen/mod.rs:351-365 with allocation_map.rs:144-150
  __device__ __forceinline__ void hospitalize() {
    if ((w & F_HOSP) || !Disease::is_to_be_hospitalize(D.dz, w)) return;
    const uint32_t fv = S.first_vacant;
    if (fv != ~0u) {
      const Rect hr = D.hosp[S.hosp_version];
      const uint32_t wd = static_cast<uint32_t>(hr.x1 - hr.x0 + 1);
      tx = hr.x0 + static_cast<int32_t>(fv % wd);
      ty = hr.y0 + static_cast<int32_t>(fv / wd);
      w |= F_HOSP;
    } else {
      draw_move();  // hour of day 0 draws it only here
      int32_t px, py;
      random_point(home(), px, py);
      move_to(px, py);
    }
  }

  // citizen/mod.rs:397-413: the handler's on_routine_end, then the recovered go home and the
  // recovered or deceased leave hospital.
  __device__ __forceinline__ void deceased() {
    load_tm();
    Disease::on_routine_end(D.dz, disease_words(), w, tm);
    if (state() == ST_R) {
      draw_move();  // hour of day 23 draws it only here
      int32_t px, py;
      random_point(home(), px, py);
      move_to(px, py);
    }
    if ((state() == ST_R || state() == ST_D) && (w & F_HOSP)) w &= ~F_HOSP;
  }
};

// The descriptor fields the epilogue reads.
struct EpiDesc {
  uint64_t row_off, event_off;
  uint32_t event_cap, hours, n_vacc, vacc_off;
  uint32_t has_lockdown, lockdown_at, has_hospital, spread_rate_threshold;
  uint32_t block_begin, n_blocks;  // its blocks in the view's table
};

__device__ __forceinline__ void add_event(const DevView& v, const EpiDesc& D, SimState& st, uint32_t hour,
                                          uint32_t kind) {
  const uint32_t n = st.n_events;
  if (n < D.event_cap) v.events[D.event_off + n] = Event{hour, kind};
  st.n_events = n + 1;
}

// What the epilogue reads besides the counts, loaded before the counts are reduced so the loads
// overlap, by the whole block, so that it lies in scalar registers (thread 0's copy in vector
// registers would set the register count of the whole commit): the simulation's descriptor and
// state, and the next entry of the vaccination schedule.
struct EpilogueIn {
  EpiDesc D;
  SimState st;
  uint32_t vacc_h;           // hour of schedule entry st.vacc_next, ~0u past the end
  unsigned long long vacc_t;
};

__device__ __forceinline__ void load_epilogue_in(const DevView& v, const SimDesc* desc, const SimState* state,
                                                 uint32_t sim, EpilogueIn& in) {
  const SimDesc d = scalar_copy(desc + sim);
  in.D = EpiDesc{d.row_off, d.event_off, d.event_cap, d.hours, d.n_vacc, d.vacc_off,
                 d.has_lockdown, d.lockdown_at, d.has_hospital, d.spread_rate_threshold,
                 v.office ? d.office_block_begin : d.block_begin, v.office ? d.office_n_blocks : d.n_blocks};
  in.st = scalar_copy(state + sim);
  const bool more = in.st.vacc_next < in.D.n_vacc;
  in.vacc_h = more ? scalar_copy(v.vacc_hour + in.D.vacc_off + in.st.vacc_next) : ~0u;
  in.vacc_t = more ? scalar_copy(v.vacc_thr + in.D.vacc_off + in.st.vacc_next) : 0ull;
}

// A stopped simulation only clears the commit slot of the parity it last stepped (the slot of
// the next commit but one). Constant indices keep the state in registers.
__device__ __forceinline__ void clear_commit_slot(SimState& st) {
  if (st.hour & 1u) st.commit_hour[1] = 0u;
  else st.commit_hour[0] = 0u;
}

// The next entry of the vaccination schedule.
__device__ __forceinline__ void next_vaccination(const DevView& v, EpilogueIn& in) {
  const uint32_t k = ++in.st.vacc_next;
  const bool more = k < in.D.n_vacc;
  in.vacc_h = more ? v.vacc_hour[in.D.vacc_off + k] : ~0u;
  in.vacc_t = more ? v.vacc_thr[in.D.vacc_off + k] : 0ull;
}

// Hour epilogue for one simulation (after k_step):
// the CSV row (counts.rs:126-140), interventions (allocation_map.rs:306-337,
// lockdown.rs:55-73, hospital.rs:51-74, vaccination.rs:52-54) and the standalone stop
// rule (epidemiology_simulation.rs:564-575). Works on the registers of `in`, which
// store_state writes back after the last of a launch's hours.
__device__ void hour_epilogue(const DevView& v, EpilogueIn& in, uint32_t h, const uint32_t* c) {
  const EpiDesc& D = in.D;
  SimState& st = in.st;
  const Counts7 row{h, c[0], c[1], c[2], c[3], c[4], c[5]};
  v.rows[D.row_off + (h - 1)] = row;
  v.host_rows[D.row_off + (h - 1)] = row;  // what a step call returns, without a copy kernel
  const uint32_t infected = c[2];
  uint32_t sweep = 0;
  unsigned long long vacc_thr = 0;
  // schedule sorted by hour, one entry per hour (the last config entry wins); hours
  // advance by one per call, so a cursor replaces a search
  while (in.vacc_h < h) next_vaccination(v, in);
  if (in.vacc_h == h) {
    sweep |= SWEEP_VACC;
    vacc_thr = in.vacc_t;
    add_event(v, D, st, h, EV_VACCINATION);
    next_vaccination(v, in);
  }
  if (D.has_lockdown && !st.locked && h % 24u == 0 && infected > D.lockdown_at) {
    st.locked = 1;
    sweep |= SWEEP_LOCK;
    add_event(v, D, st, h, EV_LOCKED);
  }
  if (st.locked && h == st.zero_infection_hour + 21u * 24u) {
    sweep |= SWEEP_UNLOCK;
    st.locked = 0;
    st.zero_infection_hour = 0;
    add_event(v, D, st, h, EV_UNLOCKED);
  }
  if (h % 24u == 0) st.hosp_new_infections = infected > st.hosp_new_infections ? infected - st.hosp_new_infections : 0u;
  if (!st.hosp_applied && h % 24u == 0 && D.has_hospital && st.hosp_new_infections >= D.spread_rate_threshold) {
    st.hosp_version = 1;
    st.hosp_applied = 1;
    add_event(v, D, st, h, EV_HOSPITAL);
  }
  if ((c[1] == 0 && c[2] == 0 && c[3] == 0) || h + 1 >= D.hours) st.active = 0;
  st.hour = h;
  st.rows_written = h;
  st.first_vacant = ~0u;  // this hour's scan is consumed; the next one starts fresh
#pragma unroll
  for (int k = 0; k < 6; ++k) st.last_counts[k] = c[k];
  // Slots of this hour's parity: the sweep (read by the next hour's agent pass) and the
  // next hour's agent pass (0 once stopped). Constant indices keep st in registers.
  const uint32_t next = st.active ? h + 1u : 0u;
  if (h % 24u == 0) {
    st.night_sweep = sweep;
    st.night_vacc_hour = h;
    st.night_vacc_thr = vacc_thr;
  }
  if (h & 1u) {
    st.sweep[1] = sweep;
    st.sweep_vacc_hour[1] = h;
    st.sweep_vacc_thr[1] = vacc_thr;
    st.commit_hour[0] = next;
  } else {
    st.sweep[0] = sweep;
    st.sweep_vacc_hour[0] = h;
    st.sweep_vacc_thr[0] = vacc_thr;
    st.commit_hour[1] = next;
  }
}

__device__ __forceinline__ void store_state(const DevView& v, uint32_t sim, const EpilogueIn& in) {
  v.state[sim] = in.st;
  v.host_state[sim] = in.st;
}

// Adds up n blocks' partial counts (eight words each, two of them unused) over the block's
// threads, four blocks' loads of a thread in flight at once.
__device__ __forceinline__ void add_partials(uint32_t (&acc)[6], const uint32_t* counts, uint32_t n) {
  constexpr uint32_t kFlight = 4;
  for (uint32_t b0 = threadIdx.x; b0 < n; b0 += kFlight * blockDim.x) {
    uint4 lo[kFlight];
    uint2 hi[kFlight];
#pragma unroll
    for (uint32_t f = 0; f < kFlight; ++f) {
      const uint32_t b = b0 + f * blockDim.x;
      const uint32_t* c = counts + 8ull * min(b, n - 1u);
      lo[f] = *reinterpret_cast<const uint4*>(c);
      hi[f] = *reinterpret_cast<const uint2*>(c + 4);
    }
#pragma unroll
    for (uint32_t f = 0; f < kFlight; ++f)
      if (b0 + f * blockDim.x < n) {
        acc[0] += lo[f].x;
        acc[1] += lo[f].y;
        acc[2] += lo[f].z;
        acc[3] += lo[f].w;
        acc[4] += hi[f].x;
        acc[5] += hi[f].y;
      }
  }
}

// The epilogue of an hour of day 0 or 7..23 of simulation `sim` by one block: adds up the hour's
// per-block partial counts, then hour_epilogue on thread 0, whose other inputs are loaded first so they arrive with the
// partials. At up to 100k agents the commit is as long as this block, a chain of latencies:
// descriptor and state once by scalar loads, the counts in two wide loads per block, sums by
// DPP and one barrier; the state is worked on in registers and written once. With the step's
// and commit's agent words loaded right after the table entry, an hour of 10k agents took
// 8.60 -> 7.72 us, of 100k 9.69 -> 8.68 and of 1M 21.2 -> 20.4.
template <bool ONE>
__device__ __forceinline__ void epilogue_block(const DevView& v, const SimDesc* desc, SimState* state, uint32_t block) {
  const uint32_t sim = ONE ? 0u : block;
  __shared__ uint32_t s_sum[kMaxWaves][8];
  EpilogueIn in;
  load_epilogue_in(v, desc, state, sim, in);  // uniform: scalar registers
  if (!in.st.active) {           // uniform
    if (threadIdx.x == 0) {
      clear_commit_slot(in.st);
      state[sim] = in.st;
    }
    return;
  }
  const uint32_t h = in.st.hour + 1u;
  uint32_t acc[6] = {0, 0, 0, 0, 0, 0}, c[6] = {0, 0, 0, 0, 0, 0};
  add_partials(acc, v.block_counts + 8ull * (ONE ? 0u : in.D.block_begin), in.D.n_blocks);
  // Each wave's six sums to its own LDS words, then thread 0 adds up the waves'.
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const uint32_t x = wave_sum(acc[k]);
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_sum[threadIdx.x / kWave][k] = x;
  }
  __syncthreads();
  for (uint32_t q = 0; q < blockDim.x / kWave; ++q)
#pragma unroll
    for (int k = 0; k < 6; ++k) c[k] += s_sum[q][k];
  if (threadIdx.x == 0) {
    hour_epilogue(v, in, h, c);
    store_state(v, sim, in);
  }
}

// 80 scalar registers: a wave takes 16 more than its code, in steps of 16 out of 800 a SIMD, so
// the 90 that most classes would take leave six waves of a 512-thread block's two per SIMD where
// eight fit (10M agents 166 -> 158 us an hour, 1M 20.2 -> 19.6).
// The first arguments repeat fields of the view: they arrive in registers with the wave
// (kernel argument preload). ONE: the view has one simulation, whose descriptor and state need
// not wait for the block's entry to name it. With both, an hour of 10k agents takes 7.08 -> 6.99
// us, of 100k 7.99 -> 7.90, of 10M 150.9 -> 149.7 (with the preload alone 7.06, 8.00, 150.3).
// HOME: hours of day 8..15 on the home layout, for days on which most agents are isolated and
// stay at home or wherever the lockdown met them: nothing keeps a house's or an office's
// claims to their own agents there then, so every move claims its cell.
template <HourClass C, bool ONE, bool HOME>
__global__ __attribute__((amdgpu_num_sgpr(80))) void k_step(const AgentBlock* blocks, const SimDesc* desc,
                                                            SimState* state, const uint32_t* st, const uint32_t* pos,
                                                            const uint32_t* ids, DevView v) {
  constexpr bool office = on_office_layout(C) && !HOME;
  const AgentBlock bm = scalar_copy(blocks + blockIdx.x);
  const uint32_t count = first_lane(bm.count);
  // Every slot below the block's count holds an agent (the office slot map is a
  // permutation of the ids), so validity does not wait for the slot -> id read, and the
  // agent words are loaded alongside it, and alongside the descriptor; lanes past the count
  // read the block's last agent.
  const bool valid = threadIdx.x < count;
  const uint32_t lane_slot = min(threadIdx.x, count - 1u);
  const uint64_t g0 = (ONE ? 0ull : bm.agent_off) + first_lane(bm.first);
  uint32_t local = first_lane(bm.first) + lane_slot;  // the agent id, its words
  uint32_t w_stored = (st + g0)[lane_slot], p = (pos + g0)[lane_slot];
  if (office) local = (ids + g0)[lane_slot];
  const uint32_t sim = ONE ? 0u : first_lane(bm.sim);
  const SimDesc& D = desc[sim];
  SimState* S = state + sim;
  uint32_t active = S->active;
  const uint32_t h = S->hour + 1;  // an hour of day 0 or 7..23
  const uint32_t hd = first_hour(C) == last_hour(C) ? first_hour(C) : h % 24u;
  constexpr uint32_t kFirst = first_hour(C), kLast = last_hour(C);
  __builtin_assume(hd >= kFirst && hd <= kLast);
  const Sweep sweep = sweep_slot(*S, (h - 1u) & 1u);  // decided at hour h - 1
  const uint8_t* occ = v.occ + D.grid_off;

  // This lane's claim and state word, carried past the block's claim filter to the stores.
  bool moves = false;
  uint32_t key = 0, w_out = kNoState, w_in = kNoState, tgt_word = 0, office_cell = kNoCell;
  bool whole_office = false;  // the claimed cell's office has all its slots in this block
  bool house_move = false;    // a home-layout move into the agent's own house
  uint64_t ci = 0;
  uint32_t wsa0 = 0;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  // Office hours: the offices of this block's workers (j_lo .. j_hi, none in a block of
  // other agents and in the home layout), each with 100 cells in the block's claim filter.
  const uint32_t j_lo = first_lane(bm.j_lo), j_hi = first_lane(bm.j_hi);
  const bool filter = office && j_lo <= j_hi && (j_hi - j_lo + 1u) <= kMaxFilterOffices;
  // st and pos are in flight while the work that needs neither is done (the buildings and the
  // hour's movement draw, which hours of day 0 and 23 do not use: hospitalize draws it for its
  // rare fallback, deceased for the recovered, who go home), then one wait (wsa and tm are read
  // by few agents and loaded where they are needed).
  Agent a(D, *S, occ);
  a.id = local;
  a.h = h;
  a.locate_buildings(on_office_layout(C) || C == HOURS_16);
  if (C != HOURS_0 && C != HOURS_23) a.draw_move();
  loaded_together(w_stored, p, a.mv, active);
  if (!active) return;  // uniform over the block
  if (valid) {
    a.w = sweep.mask ? apply_sweep(w_stored, sweep, local, D) : w_stored;
    a.x = static_cast<int32_t>(p & 0xFFFFu);
    a.y = static_cast<int32_t>(p >> 16);
    a.tx = a.x;
    a.ty = a.y;
    a.tm = 0;
    const uint64_t gid = (ONE ? 0ull : bm.agent_off) + local;  // tm and wsa stay in the home layout (by id)
    a.tm_arr = v.tm + gid;
    a.wsa = wsa0 = a.ws() == WS_STAFF ? v.wsa[gid] : 0u;
    w_in = w_stored;

    if (Disease::draws_needed(a.w, hd)) a.dz = a.dr(SITE_DISEASE, 0);
    if constexpr (C == HOURS_0) {
      if (a.state() == ST_I) {  // increment_infection_day (state.rs:69-73)
        const uint32_t day = fld(a.w, B_DAY, M_DAY);
        a.w = set_fld(a.w, B_DAY, M_DAY, day < kMaxDay ? day + 1 : day);
      }
      a.hospitalize();
    } else if constexpr (C == HOURS_23) {
      a.deceased();
    } else {
      a.perform_movements<C>(hd);
    }
    // Everything the stores need is computed first: a descriptor field read after a store
    // can no longer come from the scalar cache and costs a vector round trip.
    key = claim_key(h, local);
    tgt_word = static_cast<uint32_t>(a.tx) | (static_cast<uint32_t>(a.ty) << 16);
    moves = tgt_word != p;
    ci = D.cell_off + cell_index(D, a.tx, a.ty);
    // a worker's claim of a cell of its own office (the only agents that claim office
    // cells at these hours) enters the filter
    const uint32_t j = fast_mod(local, D.fd_offices);  // the agent's office
    if (filter && moves && a.tx >= a.ox && a.tx <= a.ox + 9 && a.ty >= a.oy && a.ty <= a.oy + 9 && j >= j_lo &&
        j <= j_hi) {
      office_cell = (j - j_lo) * kOfficeCells + static_cast<uint32_t>(a.ty - a.oy) * 10u +
                    static_cast<uint32_t>(a.tx - a.ox);
      whole_office = bm.whole != 0u;
    }
    // Hours of day 16..23 and 0..7: only a house's own agents (ids congruent mod
    // n_houses) choose cells of that house. Local moves stay in the current area, which is
    // home for everyone but public-transport users (transport area) and hospital staff;
    // the teleports into a house (going home at 16, recovered going home at 23, the
    // hospital fallback at 0) are its own agents'; no one has the housing area then. So
    // the lowest-id claimant of such a cell is found among the agent's lower housemates,
    // whose target words the commit reads: no global claim is made.
    house_move = !on_office_layout(C) && moves && a.in_house(a.tx, a.ty);
  }
  // Block claim filter (office hours). The office layout puts each office's workers in one
  // or two blocks, and they are the only claimants of its cells, so most same-cell rivals
  // meet here: an LDS atomicMin per claimed cell leaves only the block's lowest key, and a
  // lane that is not it has lost to a lower id and makes no global claim. At most one
  // global atomic per cell and block remains, instead of one per rival. On an office whose
  // workers all lie in this block the filter has seen every claimant, so its survivor has
  // won: it makes no global claim and flags its target word for the commit.
  if (filter) {  // uniform
    __shared__ uint32_t s_cell[kFilterCells];
    const uint32_t n_cells = (j_hi - j_lo + 1u) * kOfficeCells;
    for (uint32_t i = threadIdx.x; i < n_cells; i += blockDim.x) s_cell[i] = ~0u;
    __syncthreads();
    if (office_cell != kNoCell) atomicMin(&s_cell[office_cell], key);
    __syncthreads();
    if (office_cell != kNoCell && s_cell[office_cell] != key) moves = false;
  }
  if (valid) {
    // the grid byte depends only on the state, the hospitalized flag, the infection day and
    // the immunity, so it is recomputed only when one of those changed this hour
    constexpr uint32_t kByteFields = (M_STATE << B_STATE) | F_HOSP | (M_DAY << B_DAY) | (M_IMM << B_IMM);
    if ((a.w ^ w_in) & kByteFields) {
      const DiseaseParams dz = scalar_copy(&D.dz);
      if (occupant_byte(dz, a.w) != occupant_byte(dz, w_in)) a.w |= F_DIRTY;
    }
    w_out = a.w;
    if (a.tm != a.tm0) *a.tm_arr = a.tm;
    if (a.wsa != wsa0) v.wsa[(ONE ? 0ull : bm.agent_off) + local] = a.wsa;
    if (moves) {
      if (whole_office) tgt_word |= kTgtWon;
      else if (house_move) tgt_word |= kTgtHouse;
      else atomicMin(&v.claim[ci], key);
    }
    (v.tgt + g0)[lane_slot] = moves ? tgt_word : kTgtNone;
    if (w_out != w_in) (v.st + g0)[lane_slot] = w_out;
  }

  // S/E/I/H/R/D from the wave's masks of the state's bits, each wave's into its own LDS words
  // (nothing to clear first), then one plain store per block and category; the epilogue adds up
  // the blocks'. Lanes without an agent hold no state.
  static_assert(ST_S == 0 && ST_E == 1 && ST_I == 2 && ST_R == 3 && ST_D == 4 && kNoState == 5 && B_STATE == 0, "bits");
  __shared__ uint32_t s_counts[kMaxWaves][8];
  const uint64_t b0 = __ballot(w_out & 1u), b1 = __ballot(w_out & 2u), b2 = __ballot(w_out & 4u);
  const uint64_t in_hospital = __ballot(w_out & F_HOSP), infected = b1 & ~b0;
  uint32_t mine = wave_count(~(b0 | b1 | b2));
  mine = lane_word<1>(mine, wave_count(b0 & ~(b1 | b2)));
  mine = lane_word<2>(mine, wave_count(infected & ~in_hospital));
  mine = lane_word<3>(mine, wave_count(infected & in_hospital));
  mine = lane_word<4>(mine, wave_count(b0 & b1));
  mine = lane_word<5>(mine, wave_count(b2 & ~b0));
  if (lane < 6) s_counts[threadIdx.x / kWave][lane] = mine;
  __syncthreads();
  if (threadIdx.x < 6) {
    uint32_t sum = 0;
    for (uint32_t q = 0; q < blockDim.x / kWave; ++q) sum += s_counts[q][threadIdx.x];
    v.block_counts[8ull * blockIdx.x + threadIdx.x] = sum;
  }
}

// Epilogues of hours of day 1..6 (thread 0 of a block walks the hours): nobody's state changes
// then, so each repeats the last counts.
__device__ void quiet_epilogues(const DevView& v, uint32_t sim, uint32_t n_hours) {
  EpilogueIn in;
  load_epilogue_in(v, v.desc, v.state, sim, in);
  for (uint32_t k = 0; k < n_hours; ++k) {
    if (!in.st.active) {
      clear_commit_slot(in.st);
      continue;
    }
    uint32_t c[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) c[q] = in.st.last_counts[q];
    hour_epilogue(v, in, in.st.hour + 1u, c);
  }
  store_state(v, sim, in);
}
// Hours of day 3..6 in one launch, one block per simulation, for days with no vaccination at
// hours of day 2..5. Then no sweep is pending at any of those hours (lockdown, unlock and hospital
// decisions fall on hours of day 0 only), so their agent passes would change nothing.
__global__ void k_quiet_hours(DevView v, uint32_t n_hours) {
  if (threadIdx.x == 0) quiet_epilogues(v, blockIdx.x, n_hours);
}

// Hours of day 1..6 in one launch, for days with no vaccination at hours of day 1..5 (so the only
// sweep pending in the night is hour of day 0's) and no simulation's last hour at 1..6. Blocks
// 0 .. n_epi-1 walk the six epilogues of simulation blockIdx.x; the agent blocks (home
// layout) do the night's agent work: hour of day 0's sweep, every non-staff current area
// to home (hour of day 1), and their share of the daily claim reset (hour of day 2). The
// epilogues rewrite the parity slots meanwhile, so the agent blocks read hour of day 0's
// sweep from its own slot, and whether the simulation runs from `active`, which these
// hours cannot change (counts repeat, and no simulation's hours end there).
__global__ __attribute__((amdgpu_num_sgpr(80))) void k_night(DevView v, uint32_t n_epi) {
  if (blockIdx.x < n_epi) {  // uniform
    if (threadIdx.x == 0) quiet_epilogues(v, blockIdx.x, 6);
    return;
  }
  const uint32_t b = blockIdx.x - n_epi;
  const AgentBlock bm = scalar_copy(v.agent_blocks + b);
  const uint32_t sim = first_lane(bm.sim);
  const SimDesc& D = v.desc[sim];
  const SimState* S = v.state + sim;
  if (!S->active) return;  // uniform
  const Sweep sweep{S->night_sweep, S->night_vacc_hour, S->night_vacc_thr};
  const ClaimShare share = claim_share(v, D, b - D.block_begin);
  const uint32_t local = first_lane(bm.first) + threadIdx.x;
  if (local < D.n) {
    const uint64_t gi = D.agent_off + local;
    const uint32_t w = v.st[gi];
    uint32_t nw = sweep.mask ? apply_sweep(w, sweep, local, D) : w;
    if (fld(nw, B_WS, M_WS) != WS_STAFF) nw = set_fld(nw, B_AREA, M_AREA, AREA_HOME);
    if (nw != w) v.st[gi] = nw;
  }
  reset_claims(share);
}

// One hour of day 1..6 (home layout). Blocks 0 .. n_epi-1 run the epilogue of simulation
// blockIdx.x; the rest its agent work: nobody moves and no disease update runs while asleep
// (citizen/mod.rs:244-248), so only the sweep decided at hour h - 1 is applied, hour of day 1 sets
// every non-staff current area to home, and hour of day 2 resets the claim array before the day's
// first claim hour. A kernel of its own, whose blocks read the agents only where one of these asks
// for them (hours of day 1, 2 and 3..6 of 10M agents as a branch of the commit behind its loads 47,
// 62 and 30 us; so 27, 30 and 15-16, which is the time to start 19,500 blocks).
__global__ __attribute__((amdgpu_num_sgpr(80))) void k_rest(DevView v, uint32_t parity, uint32_t n_epi) {
  if (blockIdx.x < n_epi) {  // uniform
    if (threadIdx.x == 0) quiet_epilogues(v, blockIdx.x, 1);
    return;
  }
  const uint32_t b = blockIdx.x - n_epi;
  const AgentBlock bm = scalar_copy(v.agent_blocks + b);
  const uint32_t sim = first_lane(bm.sim);
  const SimDesc& D = v.desc[sim];
  const SimState* S = v.state + sim;
  const uint32_t h = S->commit_hour[parity];
  if (h == 0) return;  // uniform: the simulation did not step this hour
  const uint32_t hd = h % 24u, local = first_lane(bm.first) + threadIdx.x;
  const Sweep sweep = sweep_slot(*S, (h - 1u) & 1u);
  ClaimShare share{nullptr, 0, 0};
  if (hd == 2) share = claim_share(v, D, b - D.block_begin);
  if (local < D.n && (sweep.mask || hd == 1)) {
    const uint64_t gi = D.agent_off + local;
    const uint32_t w = v.st[gi];
    uint32_t nw = sweep.mask ? apply_sweep(w, sweep, local, D) : w;
    if (hd == 1 && fld(nw, B_WS, M_WS) != WS_STAFF) nw = set_fld(nw, B_AREA, M_AREA, AREA_HOME);
    if (nw != w) v.st[gi] = nw;
  }
  reset_claims(share);
}

// The grid byte of cell `c` (x | y << 16), in both its places.
__device__ __forceinline__ void put_byte(uint8_t* occ, uint32_t strip, uint32_t c, uint8_t byte) {
  const GridPlace g = grid_place(strip, c & 0xFFFFu, c >> 16);
  occ[g.at] = byte;
  if (in_two_strips(g)) occ[second_place(strip, g)] = byte;
}

// The commit of an hour of day 0 or 7..23. `parity` is the hour's parity (an hour of day 24k + j
// has the parity of j). Blocks 0 .. n_epi-1 run the epilogue of simulation blockIdx.x; the rest
// run the agent pass. Eight waves per SIMD (64 VGPRs)
// for the agent pass, whose waves mostly wait for the grid: with the 98 VGPRs that the
// epilogue would take, an hour of 10M agents takes 177 us instead of 160.
// Arguments and ONE as in k_step.
template <bool ONE>
__global__ __attribute__((amdgpu_waves_per_eu(8))) void k_commit(const AgentBlock* blocks, const SimDesc* desc,
                                                                 SimState* state, uint32_t* st, uint32_t* pos,
                                                                 const uint32_t* tgt, uint32_t parity, uint32_t n_epi,
                                                                 DevView v) {
  if (blockIdx.x < (ONE ? 1u : n_epi)) {  // uniform
    epilogue_block<ONE>(v, desc, state, blockIdx.x);
    return;
  }
  const AgentBlock bm = scalar_copy(blocks + (blockIdx.x - (ONE ? 1u : n_epi)));
  const uint32_t count = first_lane(bm.count);
  const uint32_t slot = first_lane(bm.first) + min(threadIdx.x, count - 1u);  // as in k_step
  const uint64_t gi = (ONE ? 0ull : bm.agent_off) + slot;
  // st, pos and tgt are loaded together, and at home-layout hours with them the target
  // words of the agent's lower housemates (ids local - k * n_houses, k = 1..3: a house
  // holds at most 4 agents, grid.rs:133-142), consecutive for consecutive ids. A house
  // move then pays one round trip; a claimed move two (these words, then its claim).
  uint32_t w = st[gi];
  uint32_t p = pos[gi];
  uint32_t t = tgt[gi];
  uint32_t local = slot;  // the agent id
  uint32_t m1 = kTgtNone, m2 = kTgtNone, m3 = kTgtNone;
  if (v.office) {  // uniform
    local = v.office_agent[gi];
  } else {
    const uint32_t lower = fast_div(slot, bm.houses);  // lower housemates
    const uint32_t H = bm.houses.d;
    if (lower >= 1) m1 = tgt[gi - H];
    if (lower >= 2) m2 = tgt[gi - 2ull * H];
    if (lower >= 3) m3 = tgt[gi - 3ull * H];
  }
  const uint32_t sim = ONE ? 0u : first_lane(bm.sim);
  const SimDesc& D = desc[sim];
  const SimState* S = state + sim;
  uint32_t h = scalar_copy(&S->commit_hour[parity]);
  // The movers' part of the descriptor comes while the agent words are in flight, not after them
  // (an hour of 32 runs of 100k agents 39.01 -> 38.74 us, 10M 121.6 -> 121.2, 1M 17.17 -> 17.12).
  uint64_t cell_off = scalar_copy(&D.cell_off), grid_off = scalar_copy(&D.grid_off);
  uint32_t pitch = scalar_copy(&D.pitch), strip = scalar_copy(&D.strip);
  const DiseaseParams dz = scalar_copy(&D.dz);
  asm("" : "+s"(cell_off), "+s"(grid_off), "+s"(pitch), "+s"(strip), "+s"(h));
  loaded_together(m1, m2, m3);
  loaded_together(w, p, t, h);
  if (h == 0) return;  // uniform: the simulation did not step this hour
  if (threadIdx.x < count) {
    const bool mover = t != kTgtNone;
    if (mover || (w & F_DIRTY)) {
      uint8_t* occ = v.occ + grid_off;
      const uint8_t byte = occupant_byte(dz, w);
      bool moved = false;
      if (mover) {
        // won: decided by the office-hour claim filter; a house move wins unless a lower
        // housemate chose the same cell (the same word, kTgtHouse included); any other
        // move reads back its claim
        const bool house = (t & kTgtHouse) != 0u;
        const bool won = house ? (m1 != t && m2 != t && m3 != t) : (t & kTgtWon) != 0u;
        t &= kTgtCell;
        const uint32_t ci = cell_index(pitch, static_cast<int32_t>(t & 0xFFFFu), static_cast<int32_t>(t >> 16));
        if (won || (!house && (v.claim + cell_off)[ci] == claim_key(h, local))) {
          put_byte(occ, strip, p, 0);
          put_byte(occ, strip, t, byte);
          pos[gi] = t;
          moved = true;
        }
      }
      if (!moved && (w & F_DIRTY)) put_byte(occ, strip, p, byte);
      if (w & F_DIRTY) st[gi] = w & ~F_DIRTY;
    }
  }
}

// Re-applies each simulation's last decided sweep (idempotent) so that agent state read
// by the host includes it; the next hour's agent pass applies it again to the same words.
__global__ void k_apply_sweep(DevView v) {
  const AgentBlock bm = scalar_copy(v.agent_blocks + blockIdx.x);
  const uint32_t sim = first_lane(bm.sim);
  const SimDesc& D = v.desc[sim];
  const SimState* S = v.state + sim;
  const Sweep sweep = sweep_slot(*S, S->hour & 1u);
  const uint32_t local = first_lane(bm.first) + threadIdx.x;
  if (sweep.mask == 0 || local >= D.n) return;
  const uint64_t gi = D.agent_off + local;
  const uint32_t w = v.st[gi];
  const uint32_t nw = apply_sweep(w, sweep, local, D);
  if (nw != w) v.st[gi] = nw;
}

// First vacant cell of the current hospital area in row-major order (area.rs:119-146 +
// allocation_map.rs:145) of the snapshot grid. A thread takes a strip's 60 cells of a row, the
// items of a block in row-major order too, so the block's first vacant cell is the one of its
// first wave and lane that has any. One atomicMin per block that beats what is there: atomics to
// one address, from every wave of a mostly vacant hospital, were the scan's time (10M agents
// 109 -> 15 us a day; 7 with a strip's row per thread).
__global__ void k_hospital_scan(DevView v, uint32_t items_per_thread) {
  __shared__ uint32_t s_first[kMaxWaves];
  const BlockRef bm = v.hosp_blocks[blockIdx.x];
  const uint32_t sim = first_lane(bm.sim), first = first_lane(bm.first);
  const SimDesc& D = v.desc[sim];
  SimState* S = v.state + sim;
  if (!S->active || (S->hour + 1) % 24u != 0) return;
  const Rect hr = D.hosp[S->hosp_version];
  const uint32_t wd = static_cast<uint32_t>(hr.x1 - hr.x0 + 1), rows = static_cast<uint32_t>(hr.y1 - hr.y0 + 1);
  const uint32_t per_row = hospital_items(hr), n = per_row * rows;
  if (first >= n) return;
  const uint32_t strip0 = strip_of(static_cast<uint32_t>(hr.x0) + kPadX);
  const uint32_t lead = static_cast<uint32_t>(hr.x0) + kPadX - strip0 * kStripStep;  // of the first item, before the area
  const uint32_t row0 = first / per_row, item0 = first - row0 * per_row;
  const uint32_t cell0 = row0 * wd + (item0 ? item0 * kStripStep - lead : 0u);  // the block's first cell
  // Whether an earlier block already found one. Other blocks lower the word in the meantime, so each
  // wave may see its own answer: it decides only what that wave scans, and every wave writes its
  // result and reaches the barrier.
  const bool found_before =
      __hip_atomic_load(&S->first_vacant, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < cell0;
  const uint8_t* occ = v.occ + D.grid_off;
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, waves = blockDim.x / kWave;
  uint32_t best = ~0u;
  for (uint32_t k = 0; k < items_per_thread && best == ~0u && !found_before; ++k) {  // uniform over the wave
    const uint32_t q = first + (k * waves + wave) * kWave + lane;
    const uint32_t row = q / per_row, item = q - row * per_row;
    uint32_t mine = ~0u;
    if (q < n) {
      const uint32_t y = static_cast<uint32_t>(hr.y0) + row + kPadY;
      const uint4* words = reinterpret_cast<const uint4*>(occ + (static_cast<size_t>(strip0 + item) * D.strip + y * kStripRow));
      // a bit per vacant cell (grid bytes are 0..3), those outside the area left out
      uint64_t occupied = 0;
#pragma unroll
      for (uint32_t c = 0; c < kStripRow / 16u; ++c) {
        const uint4 b = words[c];
        occupied |= static_cast<uint64_t>(occupied4(b.x) | (occupied4(b.y) << 4) | (occupied4(b.z) << 8) | (occupied4(b.w) << 12)) << (16u * c);
      }
      uint64_t vacant = ~occupied & ((1ull << kStripStep) - 1u);
      const uint32_t past = wd + lead - item * kStripStep;  // cells of the area from this item's first on
      if (item == 0) vacant &= ~0ull << lead;
      if (past < kStripStep) vacant &= (1ull << past) - 1u;
      if (vacant) mine = row * wd + item * kStripStep - lead + static_cast<uint32_t>(__builtin_ctzll(vacant));
    }
    const uint64_t found = __ballot(mine != ~0u);
    if (found) best = __shfl(mine, __builtin_ctzll(found), kWave);
  }
  if (lane == 0) s_first[wave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t q = 1; q < waves; ++q) best = min(best, s_first[q]);
    if (best < __hip_atomic_load(&S->first_vacant, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin(&S->first_vacant, best);
  }
}

// Layout move of st and pos (tm and wsa, which few agents read, stay in the home layout and
// are indexed by id in both), one tile of 32 x 32 agents id = k * n_offices + j per block.
// Along j the ids are consecutive: the home side and the slot map are read (or written)
// 128 B at a time; the office slots of the tile's other agents, who lie house by house, are
// as close together as a house's agents are few. Along k lie the workers of one office, which hold consecutive office slots: the
// workers go through LDS rows of 33 words so that their office side is also accessed a
// column of the tile at a time. Each thread owns four rows of the tile and issues the loads
// of all four before any store, so that a wave keeps four times the bytes in flight.
__global__ void __launch_bounds__(256) k_relayout(DevView home, DevView office, const TileRef* tiles,
                                                  uint32_t to_office) {
  constexpr uint32_t kRows = 4;           // rows r = ly + 8 * i of the tile per thread
  __shared__ uint32_t tile[2][32][33];  // [array][k - k0][j - j0]: workers' words
  __shared__ uint32_t tslot[32][33];    // office slot of (k, j); ~0u: no agent or not a worker
  const TileRef tr = tiles[blockIdx.x];
  const SimDesc& D = home.desc[first_lane(tr.sim)];
  const uint32_t O = D.n_offices, W = D.n_workers, n = D.n;
  const uint64_t base = D.agent_off;
  const uint32_t k0 = first_lane(tr.k0), j0 = first_lane(tr.j0);
  const uint32_t lx = threadIdx.x & 31u, ly = threadIdx.x >> 5;
  const uint32_t j = j0 + lx;
  // along j: the slot map, the home words, and the non-workers' office words
  uint64_t id[kRows];
  uint32_t slot[kRows], w[kRows], p[kRows];
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i) {
    id[i] = static_cast<uint64_t>(k0 + ly + 8u * i) * O + j;
    const bool valid = j < O && id[i] < n;
    slot[i] = valid ? office.office_slot[base + id[i]] : ~0u;  // ~0u >= W: never a worker
    if (to_office && valid) {
      w[i] = home.st[base + id[i]];
      p[i] = home.pos[base + id[i]];
    }
  }
  if (!to_office) {  // uniform: the non-workers' office words, by slot
#pragma unroll
    for (uint32_t i = 0; i < kRows; ++i)
      if (slot[i] >= W && slot[i] != ~0u) {
        w[i] = office.st[base + slot[i]];
        p[i] = office.pos[base + slot[i]];
      }
  }
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i) {
    const uint32_t r = ly + 8u * i;
    if (slot[i] < W) {
      if (to_office) {
        tile[0][r][lx] = w[i];
        tile[1][r][lx] = p[i];
      }
    } else if (slot[i] != ~0u) {
      if (to_office) {
        office.st[base + slot[i]] = w[i];
        office.pos[base + slot[i]] = p[i];
      } else {
        home.st[base + id[i]] = w[i];
        home.pos[base + id[i]] = p[i];
      }
    }
    tslot[r][lx] = slot[i] < W ? slot[i] : ~0u;
  }
  __syncthreads();
  // along k: the workers of office j0 + r, in consecutive office slots
  uint32_t ks[kRows];
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i) ks[i] = tslot[lx][ly + 8u * i];
  if (to_office) {  // uniform
#pragma unroll
    for (uint32_t i = 0; i < kRows; ++i)
      if (ks[i] != ~0u) {
        office.st[base + ks[i]] = tile[0][lx][ly + 8u * i];
        office.pos[base + ks[i]] = tile[1][lx][ly + 8u * i];
      }
    return;
  }
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i)
    if (ks[i] != ~0u) {
      w[i] = office.st[base + ks[i]];
      p[i] = office.pos[base + ks[i]];
    }
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i)
    if (ks[i] != ~0u) {
      tile[0][lx][ly + 8u * i] = w[i];
      tile[1][lx][ly + 8u * i] = p[i];
    }
  __syncthreads();
  // along j: the workers' home words
#pragma unroll
  for (uint32_t i = 0; i < kRows; ++i) {
    const uint32_t r = ly + 8u * i;
    if (tslot[r][lx] == ~0u) continue;
    home.st[base + id[i]] = tile[0][r][lx];
    home.pos[base + id[i]] = tile[1][r][lx];
  }
}

__global__ void k_export_active(DevView v, uint32_t n_sims, uint32_t* active) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_sims) active[i] = v.state[i].active;
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t value) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t k = i; k < n; k += stride) p[k] = value;
}

}  // namespace

hipError_t launch_hospital_scan(const DevView& v, const LaunchShape& s, hipStream_t stream) {
  if (s.hosp_blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_hospital_scan, dim3(s.hosp_blocks), dim3(s.hosp_block), 0, stream, v, s.hosp_items_per_thread);
  return hipGetLastError();
}

template <HourClass C, bool HOME = false>
hipError_t launch_step_class(const DevView& v, const LaunchShape& s, uint32_t blocks, uint32_t threads,
                             hipStream_t stream) {
  const auto kernel = s.n_sims == 1 ? k_step<C, true, HOME> : k_step<C, false, HOME>;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(threads), 0, stream, v.agent_blocks, v.desc, v.state, v.st, v.pos,
                     v.office_agent, v);
  return hipGetLastError();
}

hipError_t launch_step(const DevView& v, const LaunchShape& s, uint32_t hour, hipStream_t stream) {
  const uint32_t hd = hour % 24u, blocks = v.office ? s.office_agent_blocks : s.agent_blocks;
  const uint32_t threads = v.office ? s.office_block : s.block;
  if (blocks == 0) return hipSuccess;
  switch (hd) {
    case 0: return launch_step_class<HOURS_0>(v, s, blocks, threads, stream);
    case 7: case 17: return launch_step_class<HOURS_7_17>(v, s, blocks, threads, stream);
    case 8:
      return v.office ? launch_step_class<HOURS_8>(v, s, blocks, threads, stream)
                      : launch_step_class<HOURS_8, true>(v, s, blocks, threads, stream);
    case 16: return launch_step_class<HOURS_16>(v, s, blocks, threads, stream);
    case 23: return launch_step_class<HOURS_23>(v, s, blocks, threads, stream);
    default:
      if (hd > 16u) return launch_step_class<HOURS_18_22>(v, s, blocks, threads, stream);
      return v.office ? launch_step_class<HOURS_9_15>(v, s, blocks, threads, stream)
                      : launch_step_class<HOURS_9_15, true>(v, s, blocks, threads, stream);
  }
}

hipError_t launch_commit(const DevView& v, const LaunchShape& s, uint32_t hour, hipStream_t stream) {
  const uint32_t blocks = v.office ? s.office_agent_blocks : s.agent_blocks;
  if (blocks + s.n_sims == 0) return hipSuccess;
  const auto kernel = s.n_sims == 1 ? k_commit<true> : k_commit<false>;
  hipLaunchKernelGGL(kernel, dim3(s.n_sims + blocks), dim3(v.office ? s.office_block : s.block), 0, stream,
                     v.agent_blocks, v.desc, v.state, v.st, v.pos, v.tgt, hour & 1u, s.n_sims, v);
  return hipGetLastError();
}

hipError_t launch_rest(const DevView& v, const LaunchShape& s, uint32_t hour, hipStream_t stream) {
  if (s.agent_blocks + s.n_sims == 0) return hipSuccess;
  hipLaunchKernelGGL(k_rest, dim3(s.n_sims + s.agent_blocks), dim3(s.block), 0, stream, v, hour & 1u, s.n_sims);
  return hipGetLastError();
}

hipError_t launch_night(const DevView& v, const LaunchShape& s, hipStream_t stream) {
  if (s.agent_blocks + s.n_sims == 0) return hipSuccess;
  hipLaunchKernelGGL(k_night, dim3(s.n_sims + s.agent_blocks), dim3(s.block), 0, stream, v, s.n_sims);
  return hipGetLastError();
}

hipError_t launch_quiet_hours(const DevView& v, const LaunchShape& s, uint32_t n_hours, hipStream_t stream) {
  if (s.n_sims == 0) return hipSuccess;
  hipLaunchKernelGGL(k_quiet_hours, dim3(s.n_sims), dim3(64), 0, stream, v, n_hours);
  return hipGetLastError();
}

hipError_t launch_apply_sweep(const DevView& v, const LaunchShape& s, hipStream_t stream) {
  if (s.agent_blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_apply_sweep, dim3(s.agent_blocks), dim3(s.block), 0, stream, v);
  return hipGetLastError();
}

hipError_t launch_relayout(const DevView& home, const DevView& office, const TileRef* tiles, uint32_t n_tiles,
                           bool to_office, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  hipLaunchKernelGGL(k_relayout, dim3(n_tiles), dim3(256), 0, stream, home, office, tiles, to_office ? 1u : 0u);
  return hipGetLastError();
}

hipError_t launch_export_active(const DevView& v, uint32_t n_sims, uint32_t* active, hipStream_t stream) {
  if (n_sims == 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_active, dim3((n_sims + 255) / 256), dim3(256), 0, stream, v, n_sims, active);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t value, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_fill_u32, dim3(static_cast<uint32_t>(blocks < 65536 ? blocks : 65536)), dim3(256), 0, stream, p,
                     n, value);
  return hipGetLastError();
}

}  // namespace epi
