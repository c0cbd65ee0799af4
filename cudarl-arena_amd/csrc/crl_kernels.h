// gfx950 kernels of the batched grid-world + tabular Q-learning engine.
//
// Data layout in HBM (all structure-of-arrays, one entry per env):
//   s, ep_step, episode : int32    reward : fp32    done, action : uint8
//   start               : int32 cell index
//   map                 : 2 bits per cell, 16 cells per uint32, map_words per map
//   moves               : 2 bits per (cell, action), derived from map, mv_words per map
//   cell_reward         : fp32 per cell (optional)
//   Q                   : fp32 [table][s][a], one table per env or one shared
//
// Nothing here is a contraction, so there is no MFMA: every kernel is bound by
// HBM traffic or by dependent-access latency.
#pragma once
#include <type_traits>

#include "crl_device.h"
#include "crl_reduce.h"

namespace crl {

struct Ptrs {
  int32_t* s;
  int32_t* ep_step;
  int32_t* episode;
  const int32_t* start;
  float* reward;
  uint8_t* done;
  uint8_t* action;
  const uint32_t* map;
  const uint32_t* moves;  // packed move codes of every cell, mv_words per map
  const float* cell_reward;
  float* Q;
  const float* eps_tab;
  // supplied exploration stream [sup_n][N], valid for steps sup_t0 .. sup_t0+sup_n-1
  const float* u_sup;
  const int32_t* a_sup;
  uint64_t sup_t0;
  int sup_n;
  // trace [cap][trace_n]
  int32_t* tr_s;
  uint8_t* tr_a;
  float* tr_r;
  uint8_t* tr_d;
  int trace_n, trace_cursor, trace_cap;
  // episode statistics (all null unless tracked): running return of the open
  // episode, return / length of the last finished one, sums over finished ones
  float* ret_acc;
  float* ret_last;
  float* ret_sum;
  int32_t* len_last;
  int32_t* len_sum;
  // geometry
  int N;
  int map_words;   // uint32 words per map
  int mv_words;    // uint32 words of move codes per map
  int map_shared;  // 1: one map for all envs
  int table_shared;  // 1: one table for all envs
  size_t S;        // cells per map
};

// an episode of `env` just ended with return `ret` after `len` steps
__device__ __forceinline__ void record_episode(const Ptrs& P, int env, float ret, int len) {
  P.ret_last[env] = ret;
  P.len_last[env] = len;
  P.ret_sum[env] = P.ret_sum[env] + ret;
  P.len_sum[env] = P.len_sum[env] + len;
}

// trace row of an env that has used up its episode budget: it stays where it is
__device__ __forceinline__ void trace_idle(const Ptrs& P, int env, int row, int s) {
  if (env < P.trace_n && row < P.trace_cap) {
    const size_t o = (size_t)row * P.trace_n + env;
    P.tr_s[o] = s;
    P.tr_a[o] = 0;
    P.tr_r[o] = 0.0f;
    P.tr_d[o] = 0;
  }
}

// the two draws of step t for one env
struct Draw {
  float u;
  int a;
};

__device__ __forceinline__ Draw pick_draw(const Philox4 blk, uint64_t t, int A) {
  const uint32_t w0 = (t & 1) ? blk.w2 : blk.w0;
  const uint32_t w1 = (t & 1) ? blk.w3 : blk.w1;
  Draw d;
  d.u = u01(w0);
  d.a = (int)below(w1, (uint32_t)A);
  return d;
}

// ---------------------------------------------------------------------------
// Fused select -> step -> update, per-env tables, one lane per env, n_steps per
// launch.  The env's position, episode counters and the Q row of the cell it
// stands on live in registers for the whole launch: per step the only table
// traffic is the row of the new cell (asked for twice when the episode goes on:
// as the TD target's row and as the next row to act from - one cache line) and
// one 4-byte write.
// ---------------------------------------------------------------------------

// where an env's table lives while it is being stepped
constexpr int kTouchFloats = 2048;  // tables up to 8 KB are pulled into the caches whole ...
constexpr int kTouchMinSteps = 64;  // ... by launches long enough to use most of their lines
template <int A>
struct GlobalTable {  // in HBM / the caches
  float* __restrict__ q;
  __device__ __forceinline__ Row<A> load(int s) const { return load_row<A>(q + (size_t)s * A); }
  __device__ __forceinline__ void store(int s, int a, float v) const { q[(size_t)s * A + a] = v; }
  // Reads one word of every 128-byte line of a small table before its env starts
  // to step.  Left to the steps, each line's first use is a miss all the way to
  // HBM that holds up the whole wave - 64 envs x 32 lines, one or two at a time;
  // asked for together they cost one round trip (measured on 4 KB tables: +18 %).
  __device__ __forceinline__ void touch(int floats) const {
    if (floats > kTouchFloats) return;
    float acc = 0.0f;
    for (int i = 0; i < floats; i += 32) acc += q[i];
    asm volatile("" ::"v"(acc));
  }
};
template <int A>
struct LdsTable {  // staged into LDS for the whole launch
  float* q;
  __device__ __forceinline__ Row<A> load(int s) const { return load_row<A>(q + s * A); }
  __device__ __forceinline__ void store(int s, int a, float v) const { q[s * A + a] = v; }
};

// Where the fused loops get the move codes of a cell from.
// Pre-built codes staged in LDS, word-interleaved over the wave's lanes:
template <int A>
struct MovesLds {
  const uint32_t* base;  // the lane's first word
  int stride;            // words between two consecutive words of one env
  __device__ __forceinline__ uint32_t at(int s, int, int) const {
    constexpr unsigned kCells = (unsigned)move_cells_per_word<A>();
    const unsigned c = (unsigned)s;  // cell indices are never negative: shifts, not signed division
    return base[(c / kCells) * (unsigned)stride] >> ((c % kCells) * 2u * A);
  }
};
// Derived from the class map in LDS when the codes of all lanes do not fit: one
// map word per action, asked for while the table row is in flight.
template <int A>
struct MovesFromMap {
  const uint32_t* base;  // the lane's first map word, words 64 apart
  int W, H;
  __device__ __forceinline__ uint32_t at(int s, int x, int y) const {
    return moves_of_cell<A>([&](int word) -> uint32_t { return base[word * 64]; }, W, H, x, y, s);
  }
};

// Read from global memory, for maps whose codes do not fit LDS: one load, in
// flight together with the table row of the same cell.
template <int A>
struct MovesGlobal {
  const uint32_t* base;  // the env's (or the shared) packed move codes
  __device__ __forceinline__ uint32_t at(int s, int, int) const {
    constexpr unsigned kCells = (unsigned)move_cells_per_word<A>();
    const unsigned c = (unsigned)s;
    return base[c / kCells] >> ((c % kCells) * 2u * A);
  }
};

// n_steps of one env, any configuration.  `moves.at(cell, x, y)` gives the move
// codes of a cell of the env's map, `own_map` is the env's packed class map in
// global memory (read twice per launch, and only for the goal test on the
// resulting cell), `cr` its per-cell rewards (or null), `tab` its table.
// The step rule is step_rule()'s, restated on move codes: the class of the
// target cell is two bits of the codes of the cell the env stands on.
// THREE: which form of Philox (xor3).
template <int A, bool THREE, class Table, class Moves>
__device__ __forceinline__ void run_env_steps(const Rules& R, const Ptrs& P, const int env,
                                              const uint64_t t0, const int n_steps, const Moves moves,
                                              const uint32_t* __restrict__ own_map,
                                              const float* __restrict__ cr, const Table tab) {
  // The class rewards as plain register values.  As loads from the kernel's
  // argument block, "cell reward or class reward" is turned into one load through
  // a selected pointer, which needs the class rewards copied to scratch memory.
  float r_step = R.step_reward, r_goal = R.goal_reward, r_trap = R.trap_reward;
  asm volatile("" : "+v"(r_step), "+v"(r_goal), "+v"(r_trap));
  const int W = R.W;
  const bool cells = (R.reward_flags & 1) != 0;
  const bool base_cells = cells && (R.reward_flags & 2) != 0;
  const bool goal_on_result = R.goal_mode != 0;
  int start = P.start[env];
  const int sx = start % W, sy = start / W;
  int s = P.s[env];
  int x = s % W, y = s / W;  // only followed when the move codes are derived from the map
  int ep_step = P.ep_step[env];
  int episode = P.episode[env];
  bool done = P.done[env] != 0;
  float reward = P.reward[env];  // rewritten unchanged if the env's episode budget is used up
  int action = P.action[env];
  Row<A> row = tab.load(s);
  uint32_t mv = moves.at(s, x, y);
  // goal test on the resulting cell: whether the env stands on a goal is carried
  // along (a move onto a cell tells its class); the start cell's answer is fixed
  int on_goal = 0, start_goal = 0;
  if (goal_on_result) {
    on_goal = cell_class_of(own_map[s >> 4], s) == kGoal;
    start_goal = cell_class_of(own_map[start >> 4], start) == kGoal;
  }
  Philox4 blk = explore_block<THREE>(R.seed, (uint32_t)env, t0 >> 1);
  // Epsilon of a per-episode schedule stays in a register and is looked up again
  // only when an episode of the wave ends: as a load at the top of every step it
  // was a second round trip to memory per step, in front of the action.
  float eps = eps_of(R, P.eps_tab, t0, episode);
  const bool track = P.ret_acc != nullptr;
  float ret = track ? P.ret_acc[env] : 0.0f;
  // nothing loaded above is still in flight when the loop starts (a value still in
  // flight at the loop's entry makes the loop wait for ALL outstanding memory
  // operations on every iteration, the previous step's stores included)
  row_opaque(row);
  asm volatile("" : "+v"(ep_step), "+v"(episode), "+v"(reward), "+v"(action), "+v"(ret), "+v"(mv),
               "+v"(start), "+v"(s), "+v"(on_goal), "+v"(start_goal), "+v"(eps));

  for (int k = 0; k < n_steps; ++k) {
    if (R.max_episodes > 0 && episode >= R.max_episodes) {
      // budget used up: for ever, so the rest of the launch only fills the trace
      for (int kk = k; kk < n_steps; ++kk) trace_idle(P, env, P.trace_cursor + kk, s);
      break;
    }
    const uint64_t t = t0 + (uint64_t)k;
    Draw d = pick_draw(blk, t, A);
    if (P.u_sup && t >= P.sup_t0 && t - P.sup_t0 < (uint64_t)P.sup_n) {
      const size_t o = (size_t)(t - P.sup_t0) * P.N + env;
      d.u = P.u_sup[o];
      d.a = P.a_sup[o];
    }
    // indexed by the step: one address for the whole wave, read every step
    if (R.eps_mode == 1) eps = eps_of(R, P.eps_tab, t, episode);
    const int a = (d.u < eps) ? d.a : row_argmax(row);

    // the move (src/kernels.cu:13-66; goal on the resulting cell: src/environment.cu:43)
    const int s0 = s;
    const uint32_t code = (mv >> (2 * a)) & 3u;  // class of the target cell, WALL outside the grid
    const bool moved = code < (uint32_t)kTrap;
    const bool trap = code == (uint32_t)kTrap;
    int dx, dy;
    action_delta(a, A, dx, dy);
    const int tgt = s0 + __mul24(dy, W) + dx;  // inside the map whenever it is used
    const int s2 = moved ? tgt : s0;
    dx = moved ? dx : 0;
    dy = moved ? dy : 0;
    const int on_goal2 = moved ? (int)(code == (uint32_t)kGoal) : on_goal;
    const bool hit = goal_on_result ? on_goal2 != 0 : code == (uint32_t)kGoal;
    // goal beats trap; the goal pays on the goal cell (= s2 under both rules), the
    // trap on the target cell, anything else on s2: one load at one index
    const float by_class = hit ? r_goal : trap ? r_trap : r_step;
    float by_cell = 0.0f;
    if (cells) by_cell = cr[(trap && !hit) ? tgt : s2];
    reward = (cells && (hit || trap || base_cells)) ? by_cell : by_class;
    done = hit || (!R.auto_reset && done);

    // Everything the rest of this step and the start of the next one read from
    // memory is asked for here, in one go: the reward above, the row of the cell
    // the move ends on (for the TD target), the row and the move codes of the cell
    // the env acts from next - the same cell unless the episode ends with this
    // step and the env restarts.  One round trip per step, no branch around a
    // load.  An env that stays where it is reads its own row again (the pre-update
    // values: the write below comes later).
    ep_step += 1;
    const bool ends = R.auto_reset && (done || (R.episode_len > 0 && ep_step >= R.episode_len));
    s = ends ? start : s2;
    x = ends ? sx : x + dx;
    y = ends ? sy : y + dy;
    on_goal = ends ? start_goal : on_goal2;
    // (the second row only when an episode of the wave ends: a request that
    // nobody needs still takes its turn in the memory pipeline)
    const bool any_ends = __builtin_amdgcn_ballot_w64(ends) != 0;
    const Row<A> row2 = tab.load(s2);
    Row<A> row_restart{};
    if (any_ends) row_restart = tab.load(s);
    mv = moves.at(s, x, y);
    // the next step's draws depend on nothing: the Philox rounds run while the
    // loads are in flight
    if ((t & 1) == 1) blk = explore_block<THREE>(R.seed, (uint32_t)env, (t + 1) >> 1);
    const float m = row_max(row2, done, R.max_mode);
    const float qn = td_value(row_get(row, a), reward, m, R.lr, R.gamma);
    tab.store(s0, a, qn);
    // the value just written, patched in from registers
    row = row_set(row_pick(ends, row_restart, row2), s == s0 ? a : -1, qn);

    action = a;
    ret = ret + reward;
    if (env < P.trace_n && P.trace_cursor + k < P.trace_cap) {
      const size_t o = (size_t)(P.trace_cursor + k) * P.trace_n + env;
      P.tr_s[o] = s2;
      P.tr_a[o] = (uint8_t)a;
      P.tr_r[o] = reward;
      P.tr_d[o] = done ? 1 : 0;
    }
    if (ends && track) record_episode(P, env, ret, ep_step);
    ret = ends ? 0.0f : ret;
    ep_step = ends ? 0 : ep_step;
    episode += ends ? 1 : 0;
    if (R.eps_mode >= 2 && any_ends) {
      eps = eps_of(R, P.eps_tab, t, episode);
      asm volatile("" : "+v"(eps));  // arrived before the loop goes round
    }
  }

  P.s[env] = s;
  P.ep_step[env] = ep_step;
  P.episode[env] = episode;
  if (track) P.ret_acc[env] = ret;
  P.reward[env] = reward;
  P.done[env] = done ? 1 : 0;
  P.action[env] = (uint8_t)action;
}

// u01(w) < eps  <=>  (w >> 8) < eps * 2^24, both sides exact: an integer compare
__device__ __forceinline__ uint32_t explore_threshold(float eps) {
  const float scaled = ceilf(eps * 16777216.0f);
  return !(scaled > 0.0f) ? 0u : scaled >= 16777216.0f ? (1u << 24) : (uint32_t)scaled;
}

// The same loop for the common configuration, with everything that is fixed
// there folded away: fixed epsilon, class rewards (no per-cell array), goal test
// on the target cell, auto-reset, true max, no trace and no supplied stream.
// Fewer live scalars and no optional branches: about half the instructions of
// the general loop, which matters because a wave that waits for one row per
// step is also issue-bound on the arithmetic between two rows.
// Between the arrival of one row and the request for the next lie only the
// argmax, the draw and one shift of the cell's move codes; the codes of the next
// cell, the Philox rounds and the bookkeeping run while the row is in flight.
//
// RICH adds the two things that configurations with large maps bring along and
// that cost one more request per step at most: per-cell rewards (`cr`, may be
// null) and an epsilon that follows the env's episode count.  The threshold
// stays in a register and is looked up again only when an episode of the wave
// ends, and so is the row of the start cell: with long episodes both are rare.
template <int A, bool RICH, class Table, class Moves>
__device__ __forceinline__ void run_env_fast(const Rules& R, const Ptrs& P, const int env,
                                             const uint64_t t0, const int n_steps, const Moves moves,
                                             const float* __restrict__ cr, const Table tab) {
  const int W = R.W, T = R.episode_len;
  const float lr = R.lr, gamma = R.gamma;
  uint32_t explore_below = explore_threshold(R.eps0);
  float r_step = R.step_reward, r_goal = R.goal_reward, r_trap = R.trap_reward;
  if (RICH) asm volatile("" : "+v"(r_step), "+v"(r_goal), "+v"(r_trap));  // plain values: no select of loads
  const bool cells = RICH && cr != nullptr;
  const bool base_cells = cells && (R.reward_flags & 2) != 0;
  const bool scheduled = RICH && R.eps_mode >= 2;
  int start = P.start[env];
  const int sx = start % W, sy = start / W;
  int s = P.s[env];
  int x = s % W, y = s / W;  // only followed when the move codes are derived from the map
  int ep_step = P.ep_step[env];
  int episode = P.episode[env];
  float reward = 0.0f;
  int action = 0;
  bool hit = false;
  Row<A> row = tab.load(s);
  uint32_t mv = moves.at(s, x, y);
  if (scheduled) explore_below = explore_threshold(eps_of(R, P.eps_tab, t0, episode));
  uint64_t next_block = (t0 >> 1) + 1;
  Philox4 blk = explore_block(R.seed, (uint32_t)env, t0 >> 1);
  bool odd = (t0 & 1) != 0;
  // everything loaded above has arrived before the loop starts: a value still in
  // flight at the loop's entry makes the loop's first instruction wait for ALL
  // outstanding memory operations on every iteration, the previous step's store
  // included
  row_opaque(row);
  asm volatile("" : "+v"(ep_step), "+v"(episode), "+v"(mv), "+v"(start), "+v"(s));
  if (RICH) asm volatile("" : "+v"(explore_below));

  for (int k = 0; k < n_steps; ++k) {
    const uint32_t w0 = odd ? blk.w2 : blk.w0;
    const uint32_t w1 = odd ? blk.w3 : blk.w1;
    // both candidates are computed and one is selected: cheaper than a divergent branch
    const int greedy = row_argmax(row);
    const int a = ((w0 >> 8) < explore_below) ? (int)below(w1, (uint32_t)A) : greedy;

    const uint32_t code = (mv >> (2 * a)) & 3u;
    const bool moved = code < (uint32_t)kTrap;
    int dx, dy;
    action_delta(a, A, dx, dy);
    hit = code == (uint32_t)kGoal;
    const bool trap = code == (uint32_t)kTrap;
    reward = hit ? r_goal : (trap ? r_trap : r_step);
    float by_cell = 0.0f;
    if (RICH && cells) {
      // the goal pays on the goal cell (where the move ends), the trap on the
      // cell it guards, anything else where the move ends: one load at one index
      const int tgt = s + __mul24(dy, W) + dx;
      by_cell = cr[trap ? tgt : (moved ? tgt : s)];
    }
    dx = moved ? dx : 0;
    dy = moved ? dy : 0;
    const int s2 = s + __mul24(dy, W) + dx;

    // Two rows are asked for together: the one of the cell the move ends on (for
    // the TD target) and the one of the cell the env acts from next - the same
    // cell, and the same cache line, unless the episode ends with this step and the
    // env restarts.  No branch, and a restart costs no second round trip.  An env
    // that stays where it is reads its own row again (the pre-update values: the
    // write below comes later).
    ep_step += 1;
    const bool ends = hit || (T > 0 && ep_step >= T);
    const int s_next = ends ? start : s2;
    const Row<A> row2 = tab.load(s2);
    Row<A> row_next{};
    const bool any_ends = !RICH || __builtin_amdgcn_ballot_w64(ends) != 0;
    if (any_ends) row_next = tab.load(s_next);
    x = ends ? sx : x + dx;
    y = ends ? sy : y + dy;
    mv = moves.at(s_next, x, y);
    if (odd) blk = explore_block(R.seed, (uint32_t)env, next_block++);  // in the loads' shadow
    if (RICH) reward = (cells && (hit || trap || base_cells)) ? by_cell : reward;
    const float m = row_max(row2, hit, 0);
    const float qn = td_value(row_get(row, a), reward, m, lr, gamma);
    tab.store(s, a, qn);

    // the cell to act from next, with the value just written patched in from registers
    row = row_set(RICH ? row_pick(ends, row_next, row2) : row_next, s_next == s ? a : -1, qn);
    ep_step = ends ? 0 : ep_step;
    episode += ends ? 1 : 0;
    s = s_next;
    action = a;
    odd = !odd;
    if (RICH && scheduled && any_ends) {
      explore_below = explore_threshold(eps_of(R, P.eps_tab, t0, episode));
      asm volatile("" : "+v"(explore_below));  // arrived before the loop goes round
    }
  }

  P.s[env] = s;
  P.ep_step[env] = ep_step;
  P.episode[env] = episode;
  P.reward[env] = reward;
  P.done[env] = hit ? 1 : 0;
  P.action[env] = (uint8_t)action;
}

// The folded loop for calls whose tables outgrow the caches, where what costs is the number of scattered
// requests: the rows an env comes to are kept in LDS and written back when others take their place or the
// call is over, so that a cell visited again costs none.
// An env has four places, each for a run of kRun cells beside each other (cut off at the map's edge), 32 bytes
// of the table, and a word: the run's name - first cell << 1, 1 more where it is cut off; kNone: none - and (CODES), from
// bit 16 on, the move codes of its cells.  Which place follows from the lowest bits of x / kRun and of y, so that the runs next to each
// other are in different ones.  Two lanes move a run together, 16 bytes each, first for one of them and then for the other.
// [place][piece][lane], the lane mixed with the piece against bank conflicts; then the words, [place][lane].
//
// What bounds it: memory, in requests of 128 bytes of which an env wants 32 and in partial writes, and that these and the steps overlap
// but in part: 1M envs of 16x16, 20 steps, 369 us, without loads and stores 169, with the stores only 187, the loads only 271.  A step
// waits for the lanes whose cell is new - with 64 envs there is always one.  257 vector instructions a step are not the bound (a
// variant with 14 % fewer took the same time).  What it came from: 627 us with a row and a value per step from and to
// HBM (21M reads of 16 bytes that meet the L2 in 5.9M lines, 21M stores of 4 bytes); rows kept one by one, each lane moving
// its own 474 (11.9M lines: with 16 waves to a compute unit none of it is met again in the L2); runs of two, each lane moving its own
// 430, of four 484; runs of two moved by two lanes and only what was written put back 383, with nothing in flight at the loop's
// entry and a word of 16 bits, so that 12 waves fit, 369; of four moved by four 474 (seven waves fit); more places would ask for
// 10.7 rows in 20 steps where four ask for 12, and cost waves.  32 and 64 steps 910 and 1571 us -> 500 and 890.
template <int A, bool CODES, int PLACES>
struct RowCache {
  using Word = std::conditional_t<CODES, uint32_t, uint16_t>;
  static constexpr int kRun = 8 / A, kPlaces = PLACES, kBytes = 64 * kPlaces * (32 + (int)sizeof(Word));
  static constexpr uint32_t kNone = 0xffffu, kRowBytes = 4 * A;
  crl_f4* pieces;
  Word* words;                  // the lane's
  unsigned char* tables;        // of the wave's first env
  const unsigned char* codes;
  uint32_t table_at, codes_at;  // from there to the lane's env's
  int lane, W;

  static __device__ __forceinline__ int place(int x, int y) { return ((unsigned)x / kRun & 1) | ((unsigned)y % (PLACES / 2)) << 1; }
  static __device__ __forceinline__ int offset(int x) { return x & (kRun - 1); }
  __device__ __forceinline__ uint32_t name(int s, int x) const {
    return A == 4 ? (uint32_t)(s - offset(x)) << 1 | ((x | 1) == W ? 1u : 0u) : (uint32_t)s << 1;
  }
  __device__ __forceinline__ Word& word(int p) const { return words[p * 64]; }
  __device__ __forceinline__ crl_f4* piece(int p, int c, int of_lane) const { return pieces + (p * 2 + c) * 64 + (of_lane ^ c); }
  __device__ __forceinline__ Row<A> row(int p, int off) const {
    if constexpr (A == 4) {
      return load_row4(reinterpret_cast<const float*>(piece(p, off, lane)));
    } else {
      const crl_f4 t = *piece(p, 0, lane), u = *piece(p, 1, lane);
      return Row<8>{t.x, t.y, t.z, t.w, u.x, u.y, u.z, u.w};
    }
  }
  // which of a run's two pieces holds the value of that cell and action
  static __device__ __forceinline__ int piece_of(int off, int a) { return A == 4 ? off : a >> 2; }
  __device__ __forceinline__ float* value(int p, int off, int a) const {
    return reinterpret_cast<float*>(piece(p, piece_of(off, a), lane)) + (a & 3);
  }
  // v of the even / odd one of the two lanes
  template <int J>
  static __device__ __forceinline__ uint32_t from(uint32_t v) {
    constexpr int j = J, k = 2 + J;
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, j | j << 2 | k << 4 | k << 6, 0xf, 0xf, true);
  }
  // a run in HBM: where it starts and, in the two lowest bits, which of its pieces
  __device__ __forceinline__ uint32_t run(uint32_t name, uint32_t pieces) const { return table_at + (name >> 1) * kRowBytes + pieces; }
  __device__ __forceinline__ crl_f4* global(uint32_t run) const {
    return reinterpret_cast<crl_f4*>(tables + ((run & ~15u) + (uint32_t)(lane & 1) * 16u));
  }
  __device__ __forceinline__ bool has(uint32_t run) const { return (run & (1u << (lane & 1))) != 0u; }

  // (what comes from another lane is fetched while that is at work too: not under a condition)
  struct Pieces {
    crl_f4 even, odd;
  };
  __device__ __forceinline__ void ask(uint32_t run, Pieces& v) const {
    const uint32_t even = from<0>(run), odd = from<1>(run);
    if (has(even)) v.even = *global(even);
    if (has(odd)) v.odd = *global(odd);
  }
  __device__ __forceinline__ Pieces take(int p) const {
    const int even = (int)from<0>(p), odd = (int)from<1>(p);
    return Pieces{*piece(even, lane & 1, lane & ~1), *piece(odd, lane & 1, lane | 1)};
  }
  __device__ __forceinline__ void put(int p, uint32_t run, const Pieces& v) const {
    const int p_even = (int)from<0>(p), p_odd = (int)from<1>(p);
    const uint32_t even = from<0>(run), odd = from<1>(run);
    if (has(even)) *piece(p_even, lane & 1, lane & ~1) = v.even;
    if (has(odd)) *piece(p_odd, lane & 1, lane | 1) = v.odd;
  }
  __device__ __forceinline__ void put_back(uint32_t run, const Pieces& v) const {
    const uint32_t even = from<0>(run), odd = from<1>(run);
    if (has(even)) *global(even) = v.even;
    if (has(odd)) *global(odd) = v.odd;
  }
  __device__ __forceinline__ uint32_t codes_of(uint32_t name) const {
    uint16_t two;  // (4 actions: a byte to a cell, at any address)
    __builtin_memcpy(&two, codes + (codes_at + (name >> 1) * (A / 4)), 2);
    return two;
  }
  static __device__ __forceinline__ uint32_t pieces_of(uint32_t name) { return A == 4 ? 3u - (name & 1u) * 2u : 3u; }
};
__device__ __forceinline__ void wave_fence();

// All lanes of the wave call it; those without an env of their own do another's work once more, to the same effect.
// CODES: the move codes come along with the runs, else from `moves`.
template <int A, bool RICH, bool CODES, int PLACES, class Moves>
__device__ __forceinline__ void run_env_rows(const Rules& R, const Ptrs& P, const int env, const bool live, const uint64_t t0,
                                             const int n_steps, const Moves moves, const float* __restrict__ cr,
                                             const RowCache<A, CODES, PLACES> kept) {
  using Cache = RowCache<A, CODES, PLACES>;
  const int W = R.W, T = R.episode_len > 0 ? R.episode_len : 0x7fffffff;
  const float lr = R.lr, gamma = R.gamma;
  uint32_t explore_below = explore_threshold(R.eps0);
  float r_step = R.step_reward, r_goal = R.goal_reward, r_trap = R.trap_reward;
  if (RICH) asm volatile("" : "+v"(r_step), "+v"(r_goal), "+v"(r_trap));
  const bool cells = RICH && cr != nullptr;
  const bool base_cells = cells && (R.reward_flags & 2) != 0;
  const bool scheduled = RICH && R.eps_mode >= 2;
  const int start = P.start[env];
  int s = P.s[env];
  int ep_step = P.ep_step[env];
  int episode = P.episode[env];
  const int sx = start % W, sy = start / W;
  int x = s % W, y = s / W;
  float reward = 0.0f;
  int action = 0;
  bool hit = false;
  int place = Cache::place(x, y);
  typename Cache::Pieces run;
  const uint32_t name0 = kept.name(s, x), run0 = kept.run(name0, Cache::pieces_of(name0));
  kept.ask(run0, run);
  uint32_t codes = CODES ? kept.codes_of(name0) : 0u;
#pragma unroll
  for (int p = 0; p < Cache::kPlaces; ++p) kept.word(p) = Cache::kNone;
  uint32_t written = 0;  // two bits for each place: the pieces of its run
  if (scheduled) explore_below = explore_threshold(eps_of(R, P.eps_tab, t0, episode));
  uint64_t next_block = (t0 >> 1) + 1;
  Philox4 blk = explore_block(R.seed, (uint32_t)env, t0 >> 1);
  bool odd = (t0 & 1) != 0;
  kept.word(place) = (typename Cache::Word)(name0 | codes << 16);
  kept.put(place, run0, run);
  wave_fence();
  Row<A> row = kept.row(place, Cache::offset(x));
  uint32_t mv = CODES ? codes >> (8 * Cache::offset(x)) : moves.at(s, x, y);
  // (all of these have arrived: what is in flight at the loop's entry makes every step wait for all its stores)
  asm volatile("" : "+v"(ep_step), "+v"(episode), "+v"(mv), "+v"(explore_below));

  for (int k = 0; k < n_steps; ++k) {
    const uint32_t w0 = odd ? blk.w2 : blk.w0;
    const uint32_t w1 = odd ? blk.w3 : blk.w1;
    const int greedy = row_argmax(row);
    const int a = ((w0 >> 8) < explore_below) ? (int)below(w1, (uint32_t)A) : greedy;

    const uint32_t code = (mv >> (2 * a)) & 3u;
    const bool moved = code < (uint32_t)kTrap;
    int dx, dy;
    action_delta(a, A, dx, dy);
    hit = code == (uint32_t)kGoal;
    const bool trap = code == (uint32_t)kTrap;
    reward = hit ? r_goal : (trap ? r_trap : r_step);
    float by_cell = 0.0f;
    if (RICH && cells) {
      const int tgt = s + __mul24(dy, W) + dx;
      by_cell = cr[trap ? tgt : (moved ? tgt : s)];
    }
    dx = moved ? dx : 0;
    dy = moved ? dy : 0;
    const int s2 = s + __mul24(dy, W) + dx;
    const int x2 = x + dx, y2 = y + dy;
    ep_step += 1;
    const bool ends = hit || ep_step >= T;

    // the run of the cell to act from next: in its place, or asked for
    const int s_next = ends ? start : s2;
    const int off = Cache::offset(x);
    x = ends ? sx : x2;
    y = ends ? sy : y2;
    const int place_next = Cache::place(x, y);
    const uint32_t name_next = kept.name(s_next, x);
    const uint32_t there = kept.word(place_next);
    const bool miss = (there & 0xffffu) != name_next;
    const uint32_t wanted = miss ? kept.run(name_next, Cache::pieces_of(name_next)) : 0u;
    kept.ask(wanted, run);
    if (CODES) {
      codes = there >> 16;
      if (miss) codes = kept.codes_of(name_next);
    } else {
      mv = moves.at(s_next, x, y);
    }
    if (odd) blk = explore_block(R.seed, (uint32_t)env, next_block++);  // in the loads' shadow
    // Where the episode ends the update does not need that run: done first, because it may be the
    // run of this step's cell that makes place.  A truncated one needs the row of the cell that the move ends on, at
    // the goal the maximum is 0.
    const float q_old = row_get(row, a);
    float* const at = kept.value(place, off, a);
    float q_new = 0.0f;
    if (ends) {
      float m = 0.0f;
      if (!hit) {
        const int place2 = Cache::place(x2, y2);
        Row<A> row2 = kept.row(place2, Cache::offset(x2));
        row_opaque(row2);  // (one load through a selected address otherwise)
        if ((kept.word(place2) & 0xffffu) != kept.name(s2, x2))
          row2 = load_row<A>(reinterpret_cast<const float*>(kept.tables + (kept.table_at + (uint32_t)s2 * Cache::kRowBytes)));
        m = row_max(row2, false, R.max_mode);
      }
      if (RICH) reward = (cells && (hit || trap || base_cells)) ? by_cell : reward;
      q_new = td_value(q_old, reward, m, lr, gamma);
      *at = q_new;
    }
    written |= 1u << (place * 2 + Cache::piece_of(off, a));
    wave_fence();
    const typename Cache::Pieces old = kept.take(place_next);
    const uint32_t gone = (written >> (place_next * 2)) & 3u;
    const uint32_t leaves = miss ? kept.run(there & 0xffffu, gone) : 0u;
    written &= miss ? ~(3u << (place_next * 2)) : ~0u;
    if (miss) kept.word(place_next) = (typename Cache::Word)(name_next | codes << 16);
    wave_fence();
    kept.put(place_next, wanted, run);
    wave_fence();
    const Row<A> row_next = kept.row(place_next, Cache::offset(x));
    kept.put_back(leaves, old);
    if (!ends) {
      if (RICH) reward = (cells && (trap || base_cells)) ? by_cell : reward;
      q_new = td_value(q_old, reward, row_max(row_next, false, R.max_mode), lr, gamma);
      *at = q_new;
    }
    row = row_set(row_next, s_next == s ? a : -1, q_new);
    if (CODES) mv = codes >> (8 * Cache::offset(x));
    place = place_next;
    ep_step = ends ? 0 : ep_step;
    episode += ends ? 1 : 0;
    s = s_next;
    action = a;
    odd = !odd;
    if (RICH && scheduled && __builtin_amdgcn_ballot_w64(ends) != 0) {
      explore_below = explore_threshold(eps_of(R, P.eps_tab, t0, episode));
      asm volatile("" : "+v"(explore_below));
    }
  }

  wave_fence();
#pragma unroll
  for (int p = 0; p < Cache::kPlaces; ++p)
    kept.put_back(kept.run(kept.word(p) & 0xffffu, (written >> (p * 2)) & 3u), kept.take(p));
  if (!live) return;
  P.s[env] = s;
  P.ep_step[env] = ep_step;
  P.episode[env] = episode;
  P.reward[env] = reward;
  P.done[env] = hit ? 1 : 0;
  P.action[env] = (uint8_t)action;
}

// ---------------------------------------------------------------------------
// One env to A lanes of a wave, a lane to an action, for batches that leave lanes to spare.
// A lone wave issues an instruction every four cycles (measured: 2.4 GHz, dependent or not; a
// taken branch costs 25 to 40), an LDS read is back after 50 and an L2 hit after 220, so a step's
// time is mostly its number of instructions.  With an action to a lane the row is one register:
//   - the maximum over the row is two (A = 8: three) cross-lane operations, and so is the
//     choice of the first lane that holds it: every lane offers what its own action would do
//     - action, resulting cell, class of the target, one word - and the smallest word of
//     those that qualify wins, the action being its top bits;
//   - no value is looked up by a run-time action: the lane whose word won computes the
//     update on its own value, and all lanes write their values back;
//   - the row of the start cell is read only in the steps in which an episode of the wave ends.
// The exploration draws of the next steps are worked out ahead by all 64 lanes into a tape
// in LDS (a block of two draws is some 80 instructions, 40 of them Philox; with E envs to a wave a
// step's share is 80 E / 128).  A step with tables in LDS, episode statistics or none: one env to a
// wave 270 cycles, four 310, 16 400.
// ---------------------------------------------------------------------------

// A word of the tape: explore iff it is below the env's limit, and then the action is its low
// byte.  Epsilon by episode: the upper 24 bits are the draw's and the limit the threshold.
// Else whether to explore is settled when the word is written: the action, or kTapeGreedy.
constexpr uint32_t kTapeGreedy = 0xffffffffu, kTapeLimit = 0x80000000u;
__device__ __forceinline__ uint32_t tape_limit(float eps) {
  const uint32_t th = explore_threshold(eps);
  return th >= (1u << 24) ? 0xffffffffu : th << 8;  // (no word with the upper 24 bits set has all the lower ones)
}

// Where the draws' limits of the next tape come from: one for all steps, or (epsilon by step) the
// table's, asked for while the steps of the tape before are made.
struct TapeLimits {
  uint32_t below;
  float eps[2][2];  // of this lane's pairs of steps
  __device__ __forceinline__ void ask(const Rules& R, const Ptrs& P, const int log_envs, const uint64_t tb, const int lane) {
    if (R.eps_mode != 1) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint64_t t = tb + 2u * (unsigned)((lane + 64 * j) >> log_envs);
      eps[j][0] = eps_of(R, P.eps_tab, t, 0);
      eps[j][1] = eps_of(R, P.eps_tab, t + 1, 0);
    }
  }
};

// The tape of steps [tb, tb + steps) of a wave's 1 << log_envs envs from env0 on, a Philox
// block to a lane and pair of steps; tb and steps are even, and there are at most two blocks to
// a lane.  [step][env].
template <int A>
__device__ __forceinline__ void write_tape(const Rules& R, const int env0, const int log_envs, const uint64_t tb,
                                           const int steps, uint32_t* tape, const int lane, const TapeLimits& limits) {
  const int E = 1 << log_envs;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = lane + 64 * j;
    if (i >= (steps >> 1) << log_envs) break;
    const int e = i & (E - 1), b = i >> log_envs;
    const Philox4 blk = explore_block(R.seed, (uint32_t)(env0 + e), (tb >> 1) + (uint64_t)b);
    uint32_t w0 = below(blk.w1, (uint32_t)A), w1 = below(blk.w3, (uint32_t)A);
    if (R.eps_mode >= 2) {
      w0 |= blk.w0 & 0xffffff00u;
      w1 |= blk.w2 & 0xffffff00u;
    } else {
      const bool by_step = R.eps_mode == 1;
      w0 = (blk.w0 >> 8) < (by_step ? explore_threshold(limits.eps[j][0]) : limits.below) ? w0 : kTapeGreedy;
      w1 = (blk.w2 >> 8) < (by_step ? explore_threshold(limits.eps[j][1]) : limits.below) ? w1 : kTapeGreedy;
    }
    tape[((2 * b) << log_envs) + e] = w0;
    tape[((2 * b + 1) << log_envs) + e] = w1;
  }
}
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The cross-lane steps of run_lanes, written out.  v_max_f32 is fmaxf (a number beats none),
// but the compiler puts a v_max_f32 x, x in front of each operand and cannot fold the lane
// move into it then; and a lane move, like the use of a comparison's mask, has to stay two
// instructions away from the one that wrote its operand, which the compiler does not see
// inside an asm statement, so each block keeps that distance itself (also from what comes
// before it), with work that is due anyway where there is some.  A lone wave issues an
// instruction every four cycles (measured; runs of 8-byte encodings every five), s_nop 1 costs
// two of them.  Masks of comparisons go from vector instruction to vector instruction: a scalar
// instruction between them waits for 13 cycles, a branch on one for 28, a taken one for 25.
#define CRL_PAIRS "quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
#define CRL_HALVES "quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
#define CRL_EIGHT "row_half_mirror row_mask:0xf bank_mask:0xf\n\t"

// The update: top = the maximum of the row q2 over the env's lanes, but at least `floor` (no
// number: no floor), 0 in the lanes of `hit`; q_new = q after the update with that target in the
// lanes of `me`, elsewhere q; next = q_new in the lanes of `stays`, elsewhere q_next.  On the way,
// for the draw of the next step: named = c in the lane of its action (low byte) and all ones
// elsewhere, explore = the lanes whose draw is below their limit; word += next_word.
template <int A>
__device__ __forceinline__ float lanes_update(float q, float q2, float q_next, float reward, unsigned long long hit,
                                              unsigned long long me, unsigned long long stays, float lr, float gamma,
                                              float floor, uint32_t draw, uint32_t limit, uint32_t mine, uint32_t c,
                                              uint32_t& named, unsigned long long& explore, uint32_t& word,
                                              uint32_t next_word, float& q_new) {
  float m, next;
#define CRL_UPDATE(MORE)                                                              \
  asm("v_cmp_eq_u32_sdwa vcc, %[draw], %[mine] src0_sel:BYTE_0 src1_sel:DWORD\n\t"  \
      "v_cmp_lt_u32 %[explore], %[draw], %[limit]\n\t"                              \
      "v_max_f32_dpp %[m], %[q2], %[q2] " CRL_PAIRS                                   \
      "v_cndmask_b32 %[named], -1, %[c], vcc\n\t"                                   \
      "v_add_u32 %[word], %[next_word], %[word]\n\t"                                \
      "v_max_f32_dpp %[m], %[m], %[m] " CRL_HALVES MORE                               \
      "v_max_f32 %[m], %[m], %[floor]\n\t"                                          \
      "v_cndmask_b32 %[m], %[m], 0, %[hit]\n\t"                                     \
      "v_fma_f32 %[m], %[gamma], %[m], %[reward]\n\t"                               \
      "v_sub_f32 %[m], %[m], %[q]\n\t"                                              \
      "v_fma_f32 %[m], %[lr], %[m], %[q]\n\t"                                       \
      "v_cndmask_b32 %[q_new], %[q], %[m], %[me]\n\t"                               \
      "v_cndmask_b32 %[next], %[q_next], %[q_new], %[stays]"                          \
      : [m] "=&v"(m), [next] "=&v"(next), [named] "=&v"(named), [explore] "=&s"(explore), [word] "+v"(word),      \
        [q_new] "=&v"(q_new)                                                                                      \
      : [q] "v"(q), [q2] "v"(q2), [q_next] "v"(q_next), [reward] "v"(reward), [hit] "s"(hit), [me] "s"(me),       \
        [stays] "s"(stays), [lr] "s"(lr), [gamma] "s"(gamma), [floor] "v"(floor), [draw] "v"(draw),               \
        [limit] "v"(limit), [mine] "v"(mine), [c] "v"(c), [next_word] "s"(next_word)                              \
      : "vcc")
  if (A == 4) CRL_UPDATE("");
  else CRL_UPDATE("s_nop 1\n\tv_max_f32_dpp %[m], %[m], %[m] " CRL_EIGHT);
#undef CRL_UPDATE
  return next;
}

// Episode statistics of an env (in all its lanes).
struct LaneStats {
  float ret, ret_last, ret_sum;
  int len_last, len_sum;
};
// The choice: the smallest word of the lanes that qualify - those of `named` that are not all
// ones where the env explores, else those whose q no other beats, where `unless` is the value
// that a q that is no number counts as: in the first lane it stays one, and then nothing beats
// it (src/q_learning.cu:200-206: strict >, from action 0 on).  On the way: last = the lanes
// whose episode has no step left after this one.  TRACK: the step before had this reward, and in
// the lanes of `ends` an episode of `len` steps ended with it; the statistics take the places
// that are idle otherwise.
template <int A, bool TRACK>
__device__ __forceinline__ uint32_t lanes_choose(float q, float unless, uint32_t c, uint32_t named, unsigned long long explore,
                                                 int left, unsigned long long& last, LaneStats& stats, float reward,
                                                 unsigned long long ends, int len) {
  float v, m;
  uint32_t w;
#define CRL_CHOOSE(G1, G2, G3, G4, G5, MORE1, MORE2)                        \
  "v_max_f32 %[v], %[q], %[unless]\n\t"                                       \
  "v_cmp_ge_i32 %[last], 1, %[left]\n\t" G1                                   \
  "v_max_f32_dpp %[m], %[v], %[v] " CRL_PAIRS G2                                \
  "v_max_f32_dpp %[m], %[m], %[m] " CRL_HALVES MORE1                            \
  "v_cmp_nlt_f32 vcc, %[v], %[m]\n\t" G3                                      \
  "v_cndmask_b32 %[w], -1, %[c], vcc\n\t"                                     \
  "v_cndmask_b32 %[w], %[w], %[named], %[explore]\n\t" G4                     \
  "v_min_u32_dpp %[w], %[w], %[w] " CRL_PAIRS G5                                \
  "v_min_u32_dpp %[w], %[w], %[w] " CRL_HALVES MORE2
#define CRL_NOP "s_nop 0\n\t"
#define CRL_NOPS "s_nop 1\n\t"
#define CRL_CHOOSE_IN                                                                                                     \
  [q] "v"(q), [unless] "v"(unless), [c] "v"(c), [named] "v"(named), [explore] "s"(explore), [left] "v"(left)
#define CRL_MAX8 CRL_NOPS "v_max_f32_dpp %[m], %[m], %[m] " CRL_EIGHT
#define CRL_MIN8 CRL_NOPS "v_min_u32_dpp %[w], %[w], %[w] " CRL_EIGHT
  if constexpr (TRACK) {
    float sum;
#define CRL_TRACKED(MORE1, MORE2)                                                                                         \
  asm(CRL_CHOOSE("v_add_f32 %[ret], %[ret], %[reward]\n\t",                                                             \
                 "v_cndmask_b32 %[len_last], %[len_last], %[len], %[ends]\n\t"                                          \
                 "v_add_f32 %[sum], %[ret_sum], %[ret]\n\t",                                                            \
                 "v_cndmask_b32 %[ret_last], %[ret_last], %[ret], %[ends]\n\t"                                          \
                 "v_cndmask_b32 %[ret], %[ret], 0, %[ends]\n\t",                                                        \
                 "v_cndmask_b32 %[ret_sum], %[ret_sum], %[sum], %[ends]\n\t"                                            \
                 "v_cndmask_b32 %[sum], 0, %[len], %[ends]\n\t",                                                        \
                 "v_add_u32 %[len_sum], %[len_sum], %[sum]\n\t" CRL_NOP, MORE1, MORE2)                                \
      : [v] "=&v"(v), [m] "=&v"(m), [w] "=&v"(w), [last] "=&s"(last), [sum] "=&v"(sum), [ret] "+v"(stats.ret),            \
        [ret_last] "+v"(stats.ret_last), [ret_sum] "+v"(stats.ret_sum), [len_last] "+v"(stats.len_last),                  \
        [len_sum] "+v"(stats.len_sum)                                                                                     \
      : CRL_CHOOSE_IN, [reward] "v"(reward), [ends] "s"(ends), [len] "v"(len)                                             \
      : "vcc")
    if (A == 4) CRL_TRACKED("", "");
    else CRL_TRACKED(CRL_MAX8, CRL_MIN8);
#undef CRL_TRACKED
  } else {
#define CRL_PLAIN(MORE1, MORE2)                                                             \
  asm(CRL_CHOOSE(CRL_NOP, CRL_NOPS, CRL_NOPS, CRL_NOPS, CRL_NOPS, MORE1, MORE2)           \
      : [v] "=&v"(v), [m] "=&v"(m), [w] "=&v"(w), [last] "=&s"(last)                        \
      : CRL_CHOOSE_IN                                                                       \
      : "vcc")
    if (A == 4) CRL_PLAIN("", "");
    else CRL_PLAIN(CRL_MAX8, CRL_MIN8);
#undef CRL_PLAIN
  }
#undef CRL_CHOOSE
#undef CRL_CHOOSE_IN
#undef CRL_NOP
#undef CRL_NOPS
#undef CRL_MAX8
#undef CRL_MIN8
  return w;
}
#undef CRL_PAIRS
#undef CRL_HALVES
#undef CRL_EIGHT

// Where the env acts from next: where the move ends, `at2`, or the start cell in the lanes of
// `last` and where the target was the goal (hit).
__device__ __forceinline__ uint32_t lanes_next(uint32_t at2, uint32_t at_start, uint32_t cls, unsigned long long last,
                                               unsigned long long& hit) {
  uint32_t at;
  asm("v_cmp_eq_u32 %[hit], 4, %[cls]\n\t"
      "v_cndmask_b32 %[at], %[at2], %[start], %[last]\n\t"
      "s_nop 0\n\t"
      "v_cndmask_b32 %[at], %[at], %[start], %[hit]"
      : [at] "=&v"(at), [hit] "=&s"(hit)
      : [at2] "v"(at2), [start] "v"(at_start), [cls] "v"(cls), [last] "s"(last));
  return at;
}
// Steps left of the episode and episodes so far, after a step that ended one in the lanes returned.
__device__ __forceinline__ unsigned long long lanes_count(unsigned long long hit, unsigned long long last, int whole, int& left,
                                                          int& episode) {
  unsigned long long ends;
  asm("s_or_b64 %[ends], %[hit], %[last]\n\t"
      "v_add_u32 %[left], -1, %[left]\n\t"
      "v_cndmask_b32 %[left], %[left], %[whole], %[ends]\n\t"
      "v_addc_co_u32 %[episode], vcc, 0, %[episode], %[ends]"
      : [ends] "=&s"(ends), [left] "+v"(left), [episode] "+v"(episode)
      : [hit] "s"(hit), [last] "s"(last), [whole] "v"(whole)
      : "vcc", "scc");
  return ends;
}

// What an action does from a cell, as one word: the action in the top three bits, the
// resulting cell (where cell rewards count the target cell, whether the env gets there or not)
// as the byte offset of its row (a multiple of 16), the class of the target (kWall outside the
// grid) in bits 2 and 3.
constexpr uint32_t kMoveOffset = 0x1ffffff0u, kMoveClass = 0xcu;
__device__ __forceinline__ uint32_t move_word(uint32_t a, uint32_t offset, uint32_t cls) { return (a << 29) | offset | (cls << 2); }

// LDS by address
template <class T>
using LdsPtr = __attribute__((address_space(3))) T*;
template <class T>
__device__ __forceinline__ LdsPtr<T> lds_at(uint32_t address) { return reinterpret_cast<LdsPtr<T>>(address); }
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((LdsPtr<const void>)p);
}

// Table and move words of an env in LDS, cell by cell: A values, then A words - one
// instruction reads both of a lane's.  At most 2^29 bytes per table.
template <int A>
struct LaneLds {
  static constexpr uint32_t kRow = 8 * A;
  uint32_t first;  // LDS address of the lane's value of the env's first cell
  using At = uint32_t;
  __device__ __forceinline__ At at(uint32_t offset) const { return first + offset; }
  __device__ __forceinline__ At at_word(uint32_t word, At) const { return first + (word & kMoveOffset); }
  __device__ __forceinline__ uint32_t offset(At p) const { return p - first; }
  static __device__ __forceinline__ float value(At p) { return *lds_at<float>(p); }
  // asks for what `word` needs / the lane's move word from that, when it has arrived
  static __device__ __forceinline__ uint32_t code(At p) { return *lds_at<uint32_t>(p + 4 * A); }
  static __device__ __forceinline__ uint32_t word(At, uint32_t code) { return code; }
  static __device__ __forceinline__ void store(At p, float v) { *lds_at<float>(p) = v; }
};

// Values in LDS (QL) or in HBM and the caches, the cells' move codes in LDS (CL) or global
// memory, a byte per cell (two with 8 actions): the move word is worked out when the code
// has arrived, four or five instructions.
// TARGET: the words name the target cell.
template <int A, bool QL, bool CL, bool TARGET>
struct LaneCodes {
  static constexpr uint32_t kRow = 4 * A;
  unsigned char* values;       // QL: the lane's value of the env's first cell; else the wave's first table
  uint32_t values_at;          // QL: 0; else from there to the lane's value of its env's first cell
  const unsigned char* codes;  // CL: the env's codes; else the wave's first env's
  uint32_t codes_at;           // CL: 0; else from there to the env's
  uint32_t action;
  int step;                    // bytes from a row to the one the lane's action leads to
  using At = uint32_t;
  __device__ __forceinline__ At at(uint32_t offset) const { return offset; }
  __device__ __forceinline__ At at_word(uint32_t word, At at) const {
    const uint32_t there = word & kMoveOffset;
    return TARGET && (word & 8u) != 0u ? at : there;  // (classes from kTrap on leave the env where it is)
  }
  __device__ __forceinline__ uint32_t offset(At p) const { return p; }
  __device__ __forceinline__ float value(At p) const { return *reinterpret_cast<const float*>(values + (QL ? p : values_at + p)); }
  __device__ __forceinline__ uint32_t code(At p) const {
    const uint32_t i = codes_at + p / (A == 4 ? kRow : kRow / 2);
    return A == 4 ? (uint32_t)codes[i] : (uint32_t)*reinterpret_cast<const uint16_t*>(codes + i);
  }
  __device__ __forceinline__ uint32_t word(At p, uint32_t code) const {
    const uint32_t cls = __builtin_amdgcn_ubfe(code, 2 * action, 2u);
    if (TARGET) return ((p + (uint32_t)step) & kMoveOffset) | ((cls << 2) | (action << 29));
    // (a class's upper bit: the env stays where it is)
    const uint32_t there = p + (uint32_t)step + (action << 29);
    const uint32_t w = QL ? there - (uint32_t)__mul24((int)__builtin_amdgcn_ubfe(code, 2 * action + 1, 1u), step)  // (a table in LDS is small)
                          : there - ((uint32_t)__builtin_amdgcn_sbfe((int)code, 2 * action + 1, 1u) & (uint32_t)step);
    return w + (cls << 2);
  }
  __device__ __forceinline__ void store(At p, float v) const { *reinterpret_cast<float*>(values + (QL ? p : values_at + p)) = v; }
};

// Which of the wave's n_here envs (at most 1 << log_envs) a lane works for: env e is lanes
// e A ... e A + A - 1, and what lanes are left do the same once more, to the same effect.  Waves
// with up to 32 lanes switched off issue slower, and the slower the more of them a compute unit
// has (measured; vector instructions alone, 4 lanes, one wave to a SIMD: up to three times the
// cycles, 64 lanes: none): 1024 envs of 10x10, one to a wave, a step 616 -> 325 cycles;
// 1000 of 128x128 with 8 actions and cell rewards 0.57 -> 0.35 us.
template <int A>
__device__ __forceinline__ int lane_slot(const int lane, const int log_envs, const int n_here) {
  const int slot = (lane / A) & ((1 << log_envs) - 1);
  return slot < n_here ? slot : 0;
}

constexpr int kNoEvents = 0, kEpsilonEvents = 1, kAllEvents = 2;

// The steps.  Every lane of the wave calls it with its env's number in the wave (lane_slot).
// The rewards by class - step, goal, trap, step - lie
// at LDS address 0, where dynamic LDS starts in a kernel without any other; CELLS: `cell_rewards` of the cells of the wave's first env (or of the shared map) also count.  EVENTS: an
// episode's end changes more than where the env stands: epsilon by episode (kEpsilonEvents), or any of
// that, episode statistics and an episode budget (kAllEvents).  Epsilon alone needs one loop and none of
// the statistics' registers (43,662 envs of 10x10 with 8 actions, 300 steps, with a form of its own
// 278 -> 218 us; 4096 of 16x16 in LDS, with the look-up that has no branch, 94 -> 72).
// The row of the cell the move ends on (for the TD target) and that of the cell the env acts
// from next - another one only where its episode ended - are asked for together.
template <int A, bool CELLS, int EVENTS, class Mem>
__device__ __forceinline__ void run_lanes(const Rules& R, const Ptrs& P, const int env0, const int slot,
                                          const uint64_t t0, const int n_steps, const Mem mem, uint32_t* tape,
                                          const int log_envs, const int tape_steps,
                                          const float* __restrict__ cell_rewards) {
  const int lane = (int)__lane_id();
  const uint32_t mine = (uint32_t)lane & (A - 1);  // this lane's action
  const int env = env0 + slot;
  int whole = R.episode_len > 0 ? R.episode_len : 0x7fffffff;
  asm("" : "+v"(whole));
  const float lr = R.lr, gamma = R.gamma;
  const float nan = __uint_as_float(0x7fc00000u);
  const float floor = R.max_mode == 1 ? 0.0f : nan;
  const float unless = mine == 0 ? nan : -__builtin_inff();
  const typename Mem::At at_start = mem.at((uint32_t)P.start[env] * Mem::kRow);
  typename Mem::At at = mem.at((uint32_t)P.s[env] * Mem::kRow);
  int left = whole - P.ep_step[env];  // steps of the episode that are left
  int episode = P.episode[env];
  float reward = P.reward[env];
  uint32_t won = ((uint32_t)P.action[env] << 29) | (P.done[env] != 0 ? (uint32_t)kGoal << 2 : 0u);  // the last step's word
  constexpr bool kAll = EVENTS == kAllEvents;
  const bool by_episode = EVENTS == kEpsilonEvents || (kAll && R.eps_mode >= 2), track = kAll && P.ret_acc != nullptr;
  const bool base_cells = CELLS && (R.reward_flags & 2) != 0;
  const uint32_t rewards_at = CELLS && !P.map_shared ? (uint32_t)slot * (uint32_t)P.S * 4u : 0u;
  uint32_t limit = by_episode ? tape_limit(eps_of_episode(R, P.eps_tab, episode)) : kTapeLimit;
  float eps_next = by_episode ? eps_of_episode(R, P.eps_tab, episode + 1) : 0.0f;  // of the next episode: asked for ahead
  LaneStats stats{0.0f, 0.0f, 0.0f, 0, 0};
  if (track) stats = LaneStats{P.ret_acc[env], P.ret_last[env], P.ret_sum[env], P.len_last[env], P.len_sum[env]};
  const int budget = kAll && R.max_episodes > 0 ? R.max_episodes : 0x7fffffff;
  bool going = episode < budget;
  float q = mem.value(at);
  uint32_t c = mem.word(at, mem.code(at));
  // (arrived before the loop starts: a value that may be in flight there makes every round
  // wait for everything, the last store's answer included)
  asm volatile("" : "+v"(q), "+v"(c), "+v"(reward), "+v"(left), "+v"(episode), "+v"(won), "+v"(limit), "+v"(eps_next));
  if (kAll) asm volatile("" : "+v"(stats.ret), "+v"(stats.ret_last), "+v"(stats.ret_sum), "+v"(stats.len_last), "+v"(stats.len_sum));

  const uint64_t t_end = t0 + (uint64_t)n_steps;
  TapeLimits limits{explore_threshold(R.eps0), {}};
  limits.ask(R, P, log_envs, t0 & ~(uint64_t)1, lane);
  for (uint64_t tb = t0 & ~(uint64_t)1; tb < t_end; tb += (uint64_t)tape_steps) {
    wave_fence();
    write_tape<A>(R, env0, log_envs, tb, tape_steps, tape, lane, limits);
    wave_fence();
    limits.ask(R, P, log_envs, tb + (uint64_t)tape_steps, lane);
    const int k0 = tb < t0 ? 1 : 0;  // (the first block may start with a step of the launch before)
    const int k1 = (int)min((uint64_t)tape_steps, t_end - tb);
    // (whether an env can use up its budget in these steps)
    const bool close = kAll && __builtin_amdgcn_ballot_w64(episode >= budget - tape_steps) != 0ull;
    // (leaving the loop is the same for all lanes that are in it: an env that has used up its
    // budget ends the loop for its wave, and the others enter it again without it)
    for (int k = k0; k < k1;) {
      const unsigned long long who = __builtin_amdgcn_ballot_w64(going);
      if (who == 0ull) break;
      int kk = k;
      if (going) {
        uint32_t word = lds_address(tape) + 4u * (uint32_t)((kk << log_envs) + slot);
        const uint32_t first = *lds_at<uint32_t>(word);
        uint32_t named = (first & 0xffu) == mine ? c : 0xffffffffu;
        unsigned long long explore = __builtin_amdgcn_ballot_w64(first < limit), last;
        word += 4u << log_envs;
        int end = k1, len = 0;
        unsigned long long ends = 0ull;
        float paid = -0.0f;  // (nothing to add yet)
        auto step = [&](auto by_end, auto by_budget) __attribute__((always_inline)) {
          won = lanes_choose<A, kAll>(q, unless, c, named, explore, left, last, stats, paid, ends, len);
          const typename Mem::At at2 = mem.at_word(won, at);
          const uint32_t cls = won & kMoveClass;
          unsigned long long hit;
          const typename Mem::At at_next = lanes_next(at2, at_start, cls, last, hit);
          const uint32_t code = mem.code(at_next);
          const float q2 = mem.value(at2);
          float q_next = mem.value(at_next);
          reward = *lds_at<float>(cls);
          float by_cell = 0.0f;
          if (CELLS) {
            // the goal pays on the goal cell (where the move ends), a trap on the cell it
            // guards, anything else where the move ends: that is the target but for a wall
            const uint32_t pays = cls == kMoveClass ? mem.offset(at) : won & kMoveOffset;
            by_cell = *reinterpret_cast<const float*>(reinterpret_cast<const unsigned char*>(cell_rewards) +
                                                      (rewards_at + pays / (Mem::kRow / 4)));
          }
          const uint32_t draw = *lds_at<uint32_t>(word);  // (the one behind the tape's end is not used)
          const unsigned long long me = __builtin_amdgcn_ballot_w64(c == won), stays = __builtin_amdgcn_ballot_w64(at_next == at);
          if (kAll) len = whole - left + 1;
          ends = lanes_count(hit, last, whole, left, episode);
          // All of the above while the values are on their way.  (Without the barrier the move
          // word's arithmetic moves up and waits for its code before the other reads are asked
          // for: two trips to LDS in a row.  1M envs of 16x16 on LDS waves alone, with the codes
          // staged eight loads at a time as well: 3.18e10 -> 3.60e10 env-steps/s.)
          __builtin_amdgcn_sched_barrier(0);
          const uint32_t c_next = mem.word(at_next, code);
          if (CELLS) reward = (base_cells || (cls - 4u) < 8u) ? by_cell : reward;  // (goal or trap, or any)
          if constexpr (decltype(by_end)::value) {
            if (__builtin_expect(ends != 0ull, 0)) {
              if (by_episode) {
                limit = __builtin_amdgcn_inverse_ballot_w64(ends) ? tape_limit(eps_next) : limit;
                eps_next = eps_of_episode(R, P.eps_tab, episode + 1);
              }
              if (decltype(by_budget)::value && __builtin_amdgcn_ballot_w64(episode >= budget) != 0ull) end = kk + 1;
            }
          }
          float q_new;
          q = lanes_update<A>(q, q2, q_next, reward, hit, me, stays, lr, gamma, floor, draw, limit, mine, c_next, named,
                              explore, word, 4u << log_envs, q_new);
          mem.store(at, q_new);
          c = c_next;
          at = at_next;
          paid = reward;
          ++kk;
        };
        auto steps = [&](auto by_end) {  // (a taken branch and the moves before it are a tenth of a step)
          constexpr std::false_type no{};
          while (kk + 4 <= end) {
            step(by_end, no);
            step(by_end, no);
            step(by_end, no);
            step(by_end, no);
          }
          while (kk < end) step(by_end, no);
        };
        if constexpr (!kAll) {
          steps(std::integral_constant<bool, EVENTS == kEpsilonEvents>{});
        } else if (close) {
          do step(std::true_type{}, std::true_type{});
          while (kk < end);
        } else if (by_episode) {
          steps(std::true_type{});
        } else {
          steps(std::false_type{});
        }
        if (kAll) {  // (the last step's)
          const bool over = __builtin_amdgcn_inverse_ballot_w64(ends);
          stats.ret = stats.ret + paid;
          stats.ret_last = over ? stats.ret : stats.ret_last;
          stats.ret_sum = over ? stats.ret_sum + stats.ret : stats.ret_sum;
          stats.len_last = over ? len : stats.len_last;
          stats.len_sum += over ? len : 0;
          stats.ret = over ? 0.0f : stats.ret;
        }
        going = episode < budget;
      }
      k = __builtin_amdgcn_readlane(kk, __builtin_ctzll(who));
    }
  }

  if (lane == slot * A) {
    // (The addresses of the env's state worked out anew: kept over the steps they take 12 registers, and
    // of the 105 of kAllEvents in k_fused_lanes only four waves fit a SIMD - the last of 17 to 24 waves
    // to a compute unit wait.  34,816 envs of 9x8 with 8 actions, statistics, epsilon by episode, 13 / 100
    // steps 21.0 / 88.7 us with them.  Working the lane's places on the tape out anew as well makes it 75, six
    // waves, and costs 2 to 4 per cent of every launch.)
    int env = env0 + slot;
    if (kAll || (CELLS && EVENTS != kNoEvents)) asm volatile("" : "+v"(env));
    P.s[env] = (int)(mem.offset(at) / Mem::kRow);
    P.ep_step[env] = whole - left;
    P.episode[env] = episode;
    P.reward[env] = reward;
    P.done[env] = (won & kMoveClass) == (uint32_t)kGoal << 2 ? 1 : 0;
    P.action[env] = (uint8_t)(won >> 29);
    if (track) {
      P.ret_acc[env] = stats.ret;
      P.ret_last[env] = stats.ret_last;
      P.ret_sum[env] = stats.ret_sum;
      P.len_last[env] = stats.len_last;
      P.len_sum[env] = stats.len_sum;
    }
  }
}

// the form of run_lanes that a configuration needs
__host__ __device__ inline int lane_events(const Rules& R, const Ptrs& P) {
  return R.max_episodes > 0 || P.ret_acc != nullptr ? kAllEvents : R.eps_mode >= 2 ? kEpsilonEvents : kNoEvents;
}
// the rewards by class, where run_lanes looks them up; word i of n, by one wave
__device__ __forceinline__ void write_rewards(const Rules& R, float* rewards, int lane) {
  if (lane < 4) rewards[lane] = lane == kGoal ? R.goal_reward : lane == kTrap ? R.trap_reward : R.step_reward;
}
// n consecutive words into LDS by one wave, eight loads in flight per lane
__device__ __forceinline__ void copy_words(const uint32_t* __restrict__ src, const int n, uint32_t* dst, const int lane) {
  for (int i = lane; i < n; i += 64 * 8) {
    uint32_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + 64 * u < n) v[u] = src[i + 64 * u];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + 64 * u < n) dst[i + 64 * u] = v[u];
  }
}
// bytes from a row to the one that action `a` leads to
template <int A>
__device__ __forceinline__ int row_step(const Rules& R, uint32_t a, uint32_t row_bytes) {
  int dx, dy;
  action_delta((int)a, A, dx, dy);
  return (dy * R.W + dx) * (int)row_bytes;
}

// Batches whose tables all fit the chip's LDS: a wave of 1 << log_envs envs, alone in its
// workgroup, keeps them there for the whole launch.
// LDS: the rewards by class (at address 0: their index is their address), [env][env_bytes],
// the tape.  WORDS: an env is rows of values and move words side by side (8 bytes per
// key); else rows of values, then the move codes (4 bytes and a quarter; a shared map's
// codes only once, behind the tape).
template <int A, bool MAP_SHARED, bool WORDS, int EVENTS>
__device__ __forceinline__ void fused_lds(const Rules& R, const Ptrs& P, const uint64_t t0, const int n_steps,
                                          const int log_envs, const int env_bytes, const int tape_steps) {
  extern __shared__ __align__(16) unsigned char lds_bytes[];
  constexpr uint32_t kRow = WORDS ? LaneLds<A>::kRow : LaneCodes<A, true, true, false>::kRow;
  const int lane = threadIdx.x;
  const int E = 1 << log_envs;
  const int env0 = blockIdx.x << log_envs;
  const int n_here = min(E, P.N - env0);
  const int S = (int)P.S;
  float* rewards = reinterpret_cast<float*>(lds_bytes);
  unsigned char* envs = lds_bytes + 16;
  uint32_t* tape = reinterpret_cast<uint32_t*>(envs + (size_t)E * env_bytes);
  uint32_t* shared_codes = tape + ((tape_steps + 1) << log_envs);
  write_rewards(R, rewards, lane);
  if (!WORDS) {
    if (MAP_SHARED) {
      copy_words(P.moves, P.mv_words, shared_codes, lane);
    } else {
      for (int e = 0; e < n_here; ++e)
        copy_words(P.moves + (size_t)(env0 + e) * P.mv_words, P.mv_words,
                   reinterpret_cast<uint32_t*>(envs + (size_t)e * env_bytes + (size_t)S * kRow), lane);
    }
  }

  // a lane takes a cell at a time: its row (and its codes) in, its row (and its move words) out
  const float* Q = P.Q + (size_t)env0 * S * A;
  const int cells = n_here * S;
  int e = 0, cell = lane;
  for (int i0 = lane; i0 < cells; i0 += 64 * 4) {
    Row<A> row[4];
    uint32_t codes[4];
    int ee[4], cc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // (four rows in flight)
      while (cell >= S) {
        cell -= S;
        ++e;
      }
      ee[u] = e;
      cc[u] = cell;
      cell += 64;
      if (i0 + 64 * u < cells) {
        row[u] = load_row<A>(Q + (size_t)(i0 + 64 * u) * A);
        if (WORDS) {
          const unsigned char* map = reinterpret_cast<const unsigned char*>(P.moves + (MAP_SHARED ? 0 : (size_t)(env0 + ee[u]) * P.mv_words));
          codes[u] = A == 4 ? map[cc[u]] : reinterpret_cast<const uint16_t*>(map)[cc[u]];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i0 + 64 * u >= cells) break;
      unsigned char* to = envs + (size_t)ee[u] * env_bytes + (size_t)cc[u] * kRow;
      store_row(reinterpret_cast<float*>(to), row[u]);
      if (WORDS) {
        uint32_t w[A];
#pragma unroll
        for (int a = 0; a < A; ++a) {
          const uint32_t cls = (codes[u] >> (2 * a)) & 3u;
          const uint32_t from = (uint32_t)cc[u] * kRow;
          w[a] = move_word((uint32_t)a, cls < (uint32_t)kTrap ? from + (uint32_t)row_step<A>(R, a, kRow) : from, cls);
        }
#pragma unroll
        for (int a = 0; a < A; a += 4)
          *reinterpret_cast<uint4*>(to + 4 * A + 4 * a) = make_uint4(w[a], w[a + 1], w[a + 2], w[a + 3]);
      }
    }
  }
  wave_fence();
  const int slot = lane_slot<A>(lane, log_envs, n_here);
  const uint32_t action = (uint32_t)lane & (A - 1);
  unsigned char* mine = envs + (size_t)slot * env_bytes;
  if (WORDS) {
    run_lanes<A, false, EVENTS>(R, P, env0, slot, t0, n_steps, LaneLds<A>{lds_address(mine) + 4 * action}, tape, log_envs, tape_steps, nullptr);
  } else {
    const unsigned char* codes = MAP_SHARED ? reinterpret_cast<const unsigned char*>(shared_codes) : mine + (size_t)S * kRow;
    const LaneCodes<A, true, true, false> mem{mine + 4 * action, 0u, codes, 0u, action, row_step<A>(R, action, kRow)};
    run_lanes<A, false, EVENTS>(R, P, env0, slot, t0, n_steps, mem, tape, log_envs, tape_steps, nullptr);
  }
  wave_fence();
  float* out = P.Q + (size_t)env0 * S * A;
  e = 0;
  cell = lane;
  for (int i = lane; i < cells; i += 64, cell += 64) {
    while (cell >= S) {
      cell -= S;
      ++e;
    }
    store_row(out + (size_t)i * A, load_row<A>(reinterpret_cast<const float*>(envs + (size_t)e * env_bytes + (size_t)cell * kRow)));
  }
}
template <int A, bool WORDS, int EVENTS>
__global__ __launch_bounds__(64) void k_fused_tickets_lds(const Rules R, const Ptrs P, const uint64_t t0,
                                                           const int n_steps, const int log_envs,
                                                           const int env_bytes, const int tape_steps) {
  fused_lds<A, false, WORDS, EVENTS>(R, P, t0, n_steps, log_envs, env_bytes, tape_steps);
}
template <int A, bool WORDS, int EVENTS>
__global__ __launch_bounds__(64) void k_fused_per_env_lds(const Rules R, const Ptrs P, const uint64_t t0,
                                                           const int n_steps, const int log_envs,
                                                           const int env_bytes, const int tape_steps) {
  fused_lds<A, true, WORDS, EVENTS>(R, P, t0, n_steps, log_envs, env_bytes, tape_steps);
}

// Tables in HBM and the caches, an env to A lanes, a wave to 1 << log_envs envs from env0 on.
// `codes` are the move codes of the map (shared) or of the wave's first env, in LDS (CL) or
// global memory; `code_bytes` from one env's to the next (0: shared).
template <int A, bool CELLS, bool CL, int EVENTS>
__device__ __forceinline__ void fused_lanes_hbm(const Rules& R, const Ptrs& P, const int env0, const uint64_t t0,
                                                const int n_steps, const unsigned char* codes, const uint32_t code_bytes,
                                                uint32_t* tape, const int log_envs, const int tape_steps) {
  constexpr uint32_t kRow = LaneCodes<A, false, CL, CELLS>::kRow;
  const int lane = (int)__lane_id();
  const int slot = lane_slot<A>(lane, log_envs, P.N - env0);
  const uint32_t at = (uint32_t)slot, action = (uint32_t)lane & (A - 1);
  const LaneCodes<A, false, CL, CELLS> mem{reinterpret_cast<unsigned char*>(P.Q + (size_t)env0 * P.S * A),
                                    at * (uint32_t)P.S * kRow + 4u * action,
                                    CL ? codes + at * code_bytes : codes,
                                    CL ? 0u : at * code_bytes,
                                    action, row_step<A>(R, action, kRow)};
  const float* cr = CELLS ? P.cell_reward + (P.map_shared ? 0 : (size_t)env0 * P.S) : nullptr;  // of the wave's first env
  run_lanes<A, CELLS, EVENTS>(R, P, env0, slot, t0, n_steps, mem, tape, log_envs, tape_steps, cr);
}

// Per-env tables whose maps are shared (MAP = 1: the one map's move codes staged
// in LDS) or too large for LDS (MAP = 2: move codes read from global memory, one
// load per step).  A block takes chunks blockIdx, blockIdx + gridDim, ... and runs
// each for all n_steps.  MODE 0: the general loop, 1: the folded loop, 2: an env to A
// lanes, for batches that then still leave the chip at most a wave or two per SIMD
// (`log_envs` envs to a wave; LDS: rewards, a tape per wave, the shared map's codes).
template <int A, int MAP, int MODE>
__global__ __launch_bounds__(256) void k_fused_per_env(const Rules R, const Ptrs P,
                                                        const uint64_t t0, const int n_steps,
                                                        const int log_envs, const int tape_steps) {
  extern __shared__ __align__(16) uint32_t lds[];
  const int tid = threadIdx.x;
  const int bdim = blockDim.x;
  if constexpr (MODE == 2) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_waves = bdim >> 6;
    const int tape_words = (tape_steps + 1) << log_envs;
    float* rewards = reinterpret_cast<float*>(lds);
    uint32_t* codes = lds + 4 + n_waves * tape_words;
    write_rewards(R, rewards, tid);
    if (MAP == 1)
      for (int i = tid; i < P.mv_words; i += bdim) codes[i] = P.moves[i];
    __syncthreads();
    const int env0 = (blockIdx.x * n_waves + wave) << log_envs;
    if (env0 >= P.N) return;
    uint32_t* tape = lds + 4 + wave * tape_words;
    const uint32_t code_bytes = P.map_shared ? 0u : (uint32_t)P.mv_words * 4u;
    const unsigned char* from = reinterpret_cast<const unsigned char*>(
        MAP == 1 ? codes : P.moves + (P.map_shared ? 0 : (size_t)env0 * P.mv_words));
    auto run = [&](auto cells, auto events) __attribute__((always_inline)) {
      fused_lanes_hbm<A, decltype(cells)::value, MAP == 1, decltype(events)::value>(R, P, env0, t0, n_steps, from, code_bytes, tape,
                                                                                   log_envs, tape_steps);
    };
    auto with = [&](auto events) __attribute__((always_inline)) {
      if (P.cell_reward) run(std::true_type{}, events);
      else run(std::false_type{}, events);
    };
    const int events = lane_events(R, P);
    if (events == kNoEvents) with(std::integral_constant<int, kNoEvents>{});
    else if (events == kEpsilonEvents) with(std::integral_constant<int, kEpsilonEvents>{});
    else with(std::integral_constant<int, kAllEvents>{});
  } else {
    constexpr bool FAST = MODE == 1;
    const int n_chunks = (P.N + bdim - 1) / bdim;
    if (MAP == 1) {
      for (int i = tid; i < P.mv_words; i += bdim) lds[i] = P.moves[i];
      __syncthreads();
    }
    for (int chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
      const int env = chunk * bdim + tid;
      if (env >= P.N) continue;
      const float* cr =
          P.cell_reward ? P.cell_reward + (P.map_shared ? 0 : (size_t)env * P.S) : nullptr;
      const uint32_t* own_map = P.map + (P.map_shared ? 0 : (size_t)env * P.map_words);
      const GlobalTable<A> tab{P.Q + (size_t)env * P.S * A};
      if (MAP == 1) {
        if (FAST)
          run_env_fast<A, true>(R, P, env, t0, n_steps, MovesLds<A>{lds, 1}, cr, tab);
        else
          // (8 actions: the three-input xor has more scalars fetched back from lanes here - 26,086 envs of 32x25, epsilon
          // by step, statistics, 56 / 200 steps 95.6 / 318 us, 88.7 / 293; 4 actions 72.9, 74.4 at 56)
          run_env_steps<A, A == 4>(R, P, env, t0, n_steps, MovesLds<A>{lds, 1}, own_map, cr, tab);
      } else {
        const MovesGlobal<A> moves{P.moves + (P.map_shared ? 0 : (size_t)env * P.mv_words)};
        if (FAST)
          run_env_fast<A, true>(R, P, env, t0, n_steps, moves, cr, tab);
        else
          run_env_steps<A, true>(R, P, env, t0, n_steps, moves, own_map, cr, tab);
      }
    }
  }
}

// The same with per-env maps: one wave to a workgroup, which takes 1 << log_envs envs at a
// time, stages their move codes into its LDS and steps them for all n_steps, A lanes to an env.
// The first envs, and with `dealt` all of them, come by position; else the next ones by a draw from
// a counter, which waits 23 ns for each other wave that draws then.  `touch`: see below.
// What bounds it is the wave's dependent chain - 52 vector instructions a step, the tape's counted, and a trip to the row,
// 0.26 us per step of 4096 envs on 32x32 maps - of which a wave with 64 envs pays the slowest of 64
// trips and 150 instructions.
// LDS: the rewards by class, the tape, the codes env by env.
template <int A, bool CELLS, int EVENTS>
__global__ __launch_bounds__(64, EVENTS == kAllEvents ? 5 : 6) void k_fused_lanes(const Rules R, const Ptrs P, const uint64_t t0, const int n_steps,
                                                    unsigned* __restrict__ ticket, const int dealt, const int touch,
                                                    const int log_envs, const int tape_steps) {
  extern __shared__ __align__(16) uint32_t lds[];
  const int lane = threadIdx.x;
  const unsigned n_tickets = (unsigned)(((long)P.N + (1 << log_envs) - 1) >> log_envs);
  const size_t table = P.S * A;  // floats per table
  uint32_t* tape = lds + 4;
  uint32_t* words = tape + ((tape_steps + 1) << log_envs);
  write_rewards(R, reinterpret_cast<float*>(lds), lane);
  if (blockIdx.x == 0 && lane == 0) {
    ticket[1] = (unsigned)P.N;
    ticket[2] = 0u;
  }
  unsigned base = blockIdx.x;
  while (base < n_tickets) {  // every wave leaves: the number only grows
    const int env0 = (int)base << log_envs;
    const int n_here = min(1 << log_envs, P.N - env0);
    wave_fence();
    copy_words(P.moves + (size_t)env0 * P.mv_words, n_here * P.mv_words, words, lane);
    // (GlobalTable::touch for all of the wave's envs, whose tables are one run in HBM: where
    // they go through the chip in rounds, a launch meets most lines for the first time)
    if (touch) {
      const float* q = P.Q + (size_t)env0 * table;
      float acc = 0.0f;
      for (int i = lane * 32; i < n_here * (int)table; i += 64 * 32) acc += q[i];
      asm volatile("" ::"v"(acc));
    }
    wave_fence();
    fused_lanes_hbm<A, CELLS, true, EVENTS>(R, P, env0, t0, n_steps, reinterpret_cast<const unsigned char*>(words),
                                    (uint32_t)P.mv_words * 4u, tape, log_envs, tape_steps);
    if (dealt) {
      base += gridDim.x;
    } else {
      if (lane == 0) base = gridDim.x + atomicAdd(ticket, 1u);
      base = (unsigned)__builtin_amdgcn_readfirstlane((int)base);
    }
  }
}

// Per-env tables with per-env maps small enough for LDS: every wave is an
// independent worker that draws env ranges from one ticket counter (32 envs per
// ticket), stages its envs' maps into its own LDS slice ([word][lane]: conflict
// free) and steps them for all n_steps.  The grid size sets how many envs - and
// how many bytes of their tables - are live on the chip at once: few enough and
// the rows an env keeps returning to are still in the last-level cache.
//
// ROWS: a wave to a workgroup, its envs by position, rows kept in LDS (run_env_rows; MOVES: the move codes with them, no maps).
//
// All waves of a workgroup but the LDS waves step 64 envs each against tables in HBM / the
// caches, and spend most of their time waiting for one row per step.  With LDSW the last
// `lds_waves` waves use the idle issue slots and the LDS: they stage the WHOLE tables of their
// envs into LDS, step them there and write the tables back.  The split between the two kinds
// follows their speed; which worker steps an env does not change its results.
//
// MODE 0 is the general loop (LDSW: one LDS wave of 32 envs); 1 and 2 select the folded loop
// (run_env_fast; 2: its variant with per-cell rewards and per-episode epsilon), which works on
// move codes: with MOVES the table waves stage the pre-built codes, otherwise the (four times
// smaller) class maps, and derive the codes while their row loads are in flight.  MODE 1's LDS
// waves take 64 / A envs, A lanes to each (run_lanes; what bounds them is one env's dependent
// chain, 0.16 us per step where they are alone).  Three table waves and one LDS wave of 32 envs
// with two lanes each / two table waves and the LDS waves of 64 / A envs that fit, launch after
// launch: 1M envs of 16x16, 1000 steps 12.46 / 12.23 ms, of 8x8 8.83 / 8.26 ms.
constexpr int kTicketEnvs = 32;

// `count` envs' words (`wpe` per env, contiguous in HBM) into [word][lane]; eight
// loads in flight per lane (one at a time, a short launch is spent waiting here)
__device__ __forceinline__ void stage_words(const uint32_t* __restrict__ src, const int count,
                                            const int wpe, const int stride, uint32_t* dst,
                                            const int lane) {
  const int total = count * wpe;
  auto put = [&](int i, uint32_t v) {
    const int e = i / wpe, w = i - e * wpe;
    dst[w * stride + e] = v;
  };
  int i0 = 0;
  for (; i0 + 64 * 8 <= total; i0 += 64 * 8) {
    uint32_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(src + i0 + u * 64 + lane);  // read once per launch
#pragma unroll
    for (int u = 0; u < 8; ++u) put(i0 + u * 64 + lane, v[u]);
  }
  for (int i = i0 + lane; i < total; i += 64) put(i, __builtin_nontemporal_load(src + i));
}

// `per` pieces each of n consecutive envs - one contiguous run in HBM - into LDS, env_bytes
// apart, or out again, by one wave.  Read once and written once per launch: marked
// non-temporal so that they do not push the table waves' rows out of the L2.
__device__ __forceinline__ uint32_t stream_load(const uint32_t* p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ float4 stream_load(const float4* p) { return stream_load4(p); }
__device__ __forceinline__ void stream_store(const uint32_t v, uint32_t* p) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void stream_store(const float4 v, float4* p) { stream_store4(v, p); }
template <bool IN, class T>
__device__ __forceinline__ void strided_copy(T* __restrict__ g, const int per, const int n, unsigned char* envs,
                                             const int env_bytes, const int lane) {
  const int total = n * per;
  const int de = 64 / per, dp = 64 - de * per;  // 64 pieces on: that many envs and pieces
  int e = lane / per, piece = lane - e * per;
  constexpr int kFlight = 16;  // (1M envs of 16x16, 1000 steps: 8 / 16 / 32 10.71 / 10.59 / 11.05 ms)
  for (int i0 = lane; i0 < total; i0 += 64 * kFlight) {
    T v[kFlight];
    T* at[kFlight];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      at[u] = reinterpret_cast<T*>(envs + (size_t)e * env_bytes) + piece;
      if (i0 + 64 * u < total) v[u] = IN ? stream_load(g + i0 + 64 * u) : *at[u];
      e += de;
      piece += dp;
      const bool wrap = piece >= per;
      piece -= wrap ? per : 0;
      e += wrap ? 1 : 0;
    }
#pragma unroll
    for (int u = 0; u < kFlight; ++u)
      if (i0 + 64 * u < total) {
        if (IN) *at[u] = v[u];
        else stream_store(v[u], g + i0 + 64 * u);
      }
  }
}

template <int A, int MODE, bool LDSW, bool MOVES, int ROWS>
__global__ __launch_bounds__(LDSW ? 320 : ROWS ? 64 : 256) void k_fused_tickets(const Rules R, const Ptrs P,
                                                                     const uint64_t t0,
                                                                     const int n_steps,
                                                                     unsigned* __restrict__ ticket,
                                                                     const int tab_stride,
                                                                     const int fixed_tickets,
                                                                     const int tape_steps,
                                                                     const int lds_waves,
                                                                     const int env_bytes) {
  constexpr bool FAST = MODE >= 1;  // the folded loop ...
  constexpr bool RICH = MODE == 2;  // ... in its variant with per-cell rewards and per-episode epsilon
  constexpr bool kLaneTables = LDSW && FAST;  // the LDS waves give an env A lanes
  extern __shared__ __align__(16) uint32_t lds[];
  const int n_waves = (int)(blockDim.x >> 6);  // with LDSW the last `lds_waves` work on LDS tables
  const int lane = threadIdx.x & 63;
  const int wave = ROWS ? 0 : threadIdx.x >> 6;
  const bool lds_worker = LDSW && wave >= n_waves - lds_waves;
  // LDS: (kLaneTables) the rewards by class; one slice per table wave; then kLaneTables:
  // [LDS wave][its envs: rows, then move codes; its tape], else the LDS wave's slice, the tables
  constexpr bool kTableMoves = FAST && MOVES;
  const int slice = (kTableMoves ? P.mv_words : P.map_words) * 64;
  uint32_t* my_words = lds + (kLaneTables ? 4 : 0) + wave * slice;  // (the LDS waves are the last ones)
  float* tabs = reinterpret_cast<float*>(lds + (n_waves - 1) * slice + P.map_words * 64);
  // envs per ticket: 32, or what a wave that gives an env A lanes steps
  constexpr int unit = kLaneTables ? 64 / A : kTicketEnvs;
  const unsigned n_tickets = (unsigned)((P.N + unit - 1) / unit);
  const int cap = lds_worker ? unit : 64;
  const unsigned take = lds_worker ? 1u : 64u / (unsigned)unit;
  if (kLaneTables && lds_worker) write_rewards(R, reinterpret_cast<float*>(lds), lane);  // (every one of them, the same)
  const size_t table = P.S * A;  // floats per table

  // fixed_tickets: the tickets are dealt by position, wave after wave, round after round
  // (workers that all take the same time need no counter).  With a wave for every pair of tickets (a short launch with all
  // envs in flight) the tickets are dealt by position: tens of thousands of
  // atomic draws from one counter would take longer than the few steps.
  if (fixed_tickets && blockIdx.x == 0 && threadIdx.x == 0) {
    ticket[1] = (unsigned)P.N;
    ticket[2] = 0u;
  }
  unsigned stepped = 0;  // envs this worker has stepped
  for (unsigned round = 0;; ++round) {
    unsigned base = 0;
    if (fixed_tickets) {
      base = ((round * gridDim.x + blockIdx.x) * (unsigned)n_waves + (unsigned)wave) * take;
    } else {
      if (lane == 0) base = atomicAdd(ticket, take);
      base = __shfl(base, 0);
    }
    if (base >= n_tickets) break;  // every worker gets here: the counter only grows
    const int env0 = (int)base * unit;
    const int n_here = min(cap, P.N - env0);
    const int env = env0 + lane;
    const bool live = lane < n_here;
    stepped += (unsigned)n_here;

    // this worker's maps: contiguous in HBM, transposed into [word][lane]
    __builtin_amdgcn_wave_barrier();
    const bool codes = kTableMoves;
    if (kLaneTables && lds_worker) {
      constexpr int log_envs = A == 8 ? 3 : 4;
      unsigned char* envs = reinterpret_cast<unsigned char*>(lds + 4 + (n_waves - lds_waves) * slice) +
                            (size_t)(wave - (n_waves - lds_waves)) * (((size_t)env_bytes + 4u * (tape_steps + 1)) << log_envs);
      strided_copy<true>(reinterpret_cast<uint32_t*>(const_cast<uint32_t*>(P.moves)) + (size_t)env0 * P.mv_words, P.mv_words,
                         n_here, envs + table * 4, env_bytes, lane);
      float4* tables = reinterpret_cast<float4*>(P.Q + (size_t)env0 * table);
      strided_copy<true>(tables, (int)(table / 4), n_here, envs, env_bytes, lane);
      wave_fence();
      const int slot = lane_slot<A>(lane, log_envs, n_here);
      const uint32_t action = (uint32_t)lane & (A - 1);
      unsigned char* mine = envs + (size_t)slot * env_bytes;
      const LaneCodes<A, true, true, false> mem{mine + 4 * action, 0u, mine + table * 4, 0u, action, row_step<A>(R, action, 4 * A)};
      run_lanes<A, false, kNoEvents>(R, P, env0, slot, t0, n_steps, mem,
                                 reinterpret_cast<uint32_t*>(envs + ((size_t)env_bytes << log_envs)), log_envs, tape_steps, nullptr);
      wave_fence();
      strided_copy<false>(tables, (int)(table / 4), n_here, envs, env_bytes, lane);
      continue;
    }
    if (codes && !ROWS)
      stage_words(P.moves + (size_t)env0 * P.mv_words, n_here, P.mv_words, cap, my_words, lane);
    else if (!codes)
      stage_words(P.map + (size_t)env0 * P.map_words, n_here, P.map_words, 64, my_words, lane);
    const float* cr = P.cell_reward ? P.cell_reward + (size_t)env * P.S : nullptr;

    if constexpr (ROWS != 0) {
      using Cache = RowCache<A, MOVES, ROWS>;
      wave_fence();
      const int slot = min(lane, n_here - 1), first = __builtin_amdgcn_readfirstlane(env0);
      crl_f4* pieces = reinterpret_cast<crl_f4*>(lds + (MOVES ? 0 : slice));
      const Cache kept{pieces, reinterpret_cast<typename Cache::Word*>(pieces + 64 * Cache::kPlaces * 2) + lane,
                       reinterpret_cast<unsigned char*>(P.Q + (size_t)first * table),
                       reinterpret_cast<const unsigned char*>(P.moves + (size_t)first * P.mv_words),
                       (uint32_t)slot * (uint32_t)table * 4u, (uint32_t)slot * (uint32_t)P.mv_words * 4u, lane, R.W};
      run_env_rows<A, RICH, MOVES, ROWS>(R, P, env0 + slot, live, t0, n_steps, MovesFromMap<A>{my_words + slot, R.W, R.H},
                                   RICH && P.cell_reward ? P.cell_reward + (size_t)(env0 + slot) * P.S : nullptr, kept);
      continue;
    }
    if (!lds_worker) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (live) {
        const GlobalTable<A> tab{P.Q + (size_t)env * table};
        if (n_steps >= kTouchMinSteps) tab.touch((int)table);
        if (kTableMoves)
          run_env_fast<A, RICH>(R, P, env, t0, n_steps, MovesLds<A>{my_words + lane, 64}, RICH ? cr : nullptr, tab);
        else if (FAST)
          run_env_fast<A, RICH>(R, P, env, t0, n_steps, MovesFromMap<A>{my_words + lane, R.W, R.H}, RICH ? cr : nullptr, tab);
        else
          run_env_steps<A, false>(R, P, env, t0, n_steps, MovesFromMap<A>{my_words + lane, R.W, R.H},
                           P.map + (size_t)env * P.map_words, cr, tab);
      }
    } else {
      // tables in: n_here consecutive tables are one contiguous run in HBM
      const float4* g4 = reinterpret_cast<const float4*>(P.Q + (size_t)env0 * table);
      const int t4 = (int)(table / 4);
      const int total4 = n_here * t4;
      // streamed once in and once out: marked non-temporal so that they do not
      // push the table waves' rows out of the L2
      auto ld = [&](int i) -> float4 { return stream_load4(g4 + i); };
      auto put = [&](int i, const float4 v) {
        const int e = i / t4, o = i - e * t4;
        reinterpret_cast<float4*>(tabs + e * tab_stride)[o] = v;
      };
      int i0 = 0;
      for (; i0 + 64 * 8 <= total4; i0 += 64 * 8) {  // eight loads in flight per lane
        const int i = i0 + lane;
        const float4 v0 = ld(i), v1 = ld(i + 64), v2 = ld(i + 128), v3 = ld(i + 192);
        const float4 v4 = ld(i + 256), v5 = ld(i + 320), v6 = ld(i + 384), v7 = ld(i + 448);
        put(i, v0);
        put(i + 64, v1);
        put(i + 128, v2);
        put(i + 192, v3);
        put(i + 256, v4);
        put(i + 320, v5);
        put(i + 384, v6);
        put(i + 448, v7);
      }
      for (int i = i0 + lane; i < total4; i += 64) put(i, ld(i));
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (live) {
        const LdsTable<A> tab{tabs + lane * tab_stride};
        run_env_steps<A, false>(R, P, env, t0, n_steps, MovesFromMap<A>{my_words + lane, R.W, R.H},
                         P.map + (size_t)env * P.map_words, cr, tab);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      float4* o4 = reinterpret_cast<float4*>(P.Q + (size_t)env0 * table);
      auto get = [&](int i) -> float4 {
        const int e = i / t4, o = i - e * t4;
        return reinterpret_cast<const float4*>(tabs + e * tab_stride)[o];
      };
      int j0 = 0;
      for (; j0 + 64 * 4 <= total4; j0 += 64 * 4) {
        const int i = j0 + lane;
        const float4 v0 = get(i), v1 = get(i + 64), v2 = get(i + 128), v3 = get(i + 192);
        stream_store4(v0, o4 + i);
        stream_store4(v1, o4 + i + 64);
        stream_store4(v2, o4 + i + 128);
        stream_store4(v3, o4 + i + 192);
      }
      for (int i = j0 + lane; i < total4; i += 64) stream_store4(get(i), o4 + i);
    }
  }
  // who did how much: once per worker (a pair of atomics per ticket had every wave of a
  // short launch queue at the counters whenever a round of tickets ended)
  if (!fixed_tickets && lane == 0 && stepped != 0u) atomicAdd(ticket + (lds_worker ? 2 : 1), stepped);
}

// ---------------------------------------------------------------------------
// Stand-alone pieces: select, step, update.  They reproduce one fused step when
// called in that order and back the reference-shaped host classes.
// ---------------------------------------------------------------------------

// Epsilon-greedy select, one lane per env: the row is one 16-byte load (two with 8
// actions), the lowest index wins ties (src/q_learning.cu:200-206).  `host_out` (may be
// null): the actions also go to pinned host memory, 256 bytes in a row per wave - with A
// lanes per env only every A-th lane had one to store.
template <int A>
__global__ __launch_bounds__(256) void k_select(const Rules R, const Ptrs P, const uint64_t t,
                                                 int32_t* __restrict__ act_out,
                                                 int32_t* __restrict__ host_out, const HostSignal sig) {
  const int env = blockIdx.x * blockDim.x + threadIdx.x;
  if (env < P.N) {
    const int s = P.s[env];
    const int episode = P.episode[env];
    const float* Qe = P.Q + (P.table_shared ? 0 : (size_t)env * P.S * A);
    const int greedy = row_argmax(load_row<A>(Qe + (size_t)s * A));
    Draw d = pick_draw(explore_block(R.seed, (uint32_t)env, t >> 1), t, A);
    if (P.u_sup && t >= P.sup_t0 && t - P.sup_t0 < (uint64_t)P.sup_n) {
      const size_t o = (size_t)(t - P.sup_t0) * P.N + env;
      d.u = P.u_sup[o];
      d.a = P.a_sup[o];
    }
    const int a = (d.u < eps_of(R, P.eps_tab, t, episode)) ? d.a : greedy;
    act_out[env] = a;
    if (host_out) store_host(host_out + env, a);
  }
  signal_host(sig);
}

// The state arrays' copies in pinned host memory (all null: none is kept), laid out as the
// engine's own are.
struct StateMirror {
  int32_t* s;
  int32_t* ep_step;
  int32_t* episode;
  float* reward;
  uint8_t* done;
  uint8_t* action;
  __device__ __forceinline__ void put(int env, int s_, int ep_step_, int episode_, float reward_, int done_, int action_) const {
    if (!s) return;
    store_host(s + env, s_);
    store_host(ep_step + env, ep_step_);
    store_host(episode + env, episode_);
    store_host(reward + env, reward_);
    store_host(done + env, (uint8_t)done_);
    store_host(action + env, (uint8_t)action_);
  }
};

// One move for every env with supplied actions (src/environment.cu:113-125,
// rules of src/kernels.cu:13-66), then the restart of finished envs.
// `act` may be host memory the device can read; for a single env the action comes as `act0`
// (act null): one trip over the link less in a call of 6 us.
// The new state also goes to `mirror` (may be null).
__device__ __forceinline__ void step_env(const Rules& R, const Ptrs& P, const Transition& T,
                                         const int a, const StateMirror& M, const int env) {
  const uint32_t* gmap = P.map + (P.map_shared ? 0 : (size_t)env * P.map_words);
  auto cls = [&](int cell) -> int { return cell_class_of(gmap[cell >> 4], cell); };
  const float* cr = P.cell_reward ? P.cell_reward + (P.map_shared ? 0 : (size_t)env * P.S) : nullptr;
  // (everything that depends on nothing is asked for at once, before the first store)
  const int s0 = P.s[env], start = P.start[env], ep_step0 = P.ep_step[env];
  int episode = P.episode[env];
  const bool done0 = P.done[env] != 0;
  if (R.max_episodes > 0 && episode >= R.max_episodes) {
    T.s[env] = s0;  // budget used up: no move and, with action -1, no update
    T.a[env] = -1;
    T.r[env] = 0.0f;
    T.s2[env] = s0;
    T.done[env] = 0;
    trace_idle(P, env, P.trace_cursor, s0);
    M.put(env, s0, ep_step0, episode, P.reward[env], P.done[env], P.action[env]);
    return;
  }
  int x = s0 % R.W, y = s0 / R.W;
  float reward;
  bool hit;
  step_rule(R, ClassRewards{R.step_reward, R.goal_reward, R.trap_reward}, cls, cr, x, y, a, reward, hit);
  const int s2 = y * R.W + x;
  const bool done = hit || (!R.auto_reset && done0);
  int ep_step = ep_step0 + 1;
  const float ret = P.ret_acc ? P.ret_acc[env] + reward : 0.0f;
  T.s[env] = s0;
  T.a[env] = a;
  T.r[env] = reward;
  T.s2[env] = s2;
  T.done[env] = done ? 1 : 0;
  P.reward[env] = reward;
  P.done[env] = done ? 1 : 0;
  P.action[env] = (uint8_t)a;
  if (env < P.trace_n && P.trace_cursor < P.trace_cap) {
    const size_t o = (size_t)P.trace_cursor * P.trace_n + env;
    P.tr_s[o] = s2;
    P.tr_a[o] = (uint8_t)a;
    P.tr_r[o] = reward;
    P.tr_d[o] = done ? 1 : 0;
  }
  const bool ends = R.auto_reset && (done || (R.episode_len > 0 && ep_step >= R.episode_len));
  if (P.ret_acc) {
    if (ends) record_episode(P, env, ret, ep_step);
    P.ret_acc[env] = ends ? 0.0f : ret;
  }
  const int s_new = ends ? start : s2;
  ep_step = ends ? 0 : ep_step;
  P.s[env] = s_new;
  P.ep_step[env] = ep_step;
  if (ends) P.episode[env] = ++episode;
  M.put(env, s_new, ep_step, episode, reward, done ? 1 : 0, (uint8_t)a);
}
__global__ __launch_bounds__(256) void k_step(const Rules R, const Ptrs P, const Transition T,
                                               const int32_t* __restrict__ act, const int act0,
                                               const StateMirror M, const HostSignal sig) {
  const int env = blockIdx.x * blockDim.x + threadIdx.x;
  int a = act0;
  if (act && env < P.N) a = act[env];
  const bool kept = M.s != nullptr;
  if (!kept && sig.flag) {
    asm volatile("" : "+v"(a));  // arrived
    signal_read(sig);
  }
  if (env < P.N) step_env(R, P, T, a, M, env);
  if (kept) signal_host(sig);
}

// n16 16-byte words (at most 2 GB) from device memory to pinned host memory, and one word on its own
// (may be null)
__global__ __launch_bounds__(256) void k_export(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                 const size_t n16, const unsigned* __restrict__ word,
                                                 unsigned* __restrict__ word_out, const HostSignal sig) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const DevWindow to = dev_window(dst);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) store_host128(to, (uint32_t)i * 16u, src[i]);
  if (word && blockIdx.x == 0 && threadIdx.x == 0) store_host(word_out, *word);
  signal_host(sig);
}

// Environment::reset for envs [first, first+count) (src/environment.cu:6-14)
__global__ __launch_bounds__(256) void k_reset(const Ptrs P, const int first, const int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int env = first + i;
  P.s[env] = P.start[env];
  P.ep_step[env] = 0;
  P.reward[env] = 0.0f;
  P.done[env] = 0;
  P.action[env] = 0;
  if (P.ret_acc) P.ret_acc[env] = 0.0f;
}

// TD update of one recorded transition per env on the env's own table
// (src/gpu/kernels.cu:7-54, one thread per sample; tables are disjoint)
template <int A>
__global__ __launch_bounds__(256) void k_update_per_env(const Rules R, const Ptrs P,
                                                         const Transition T) {
  const int env = blockIdx.x * blockDim.x + threadIdx.x;
  if (env >= P.N) return;
  float* Qe = P.Q + (size_t)env * P.S * A;
  const int s = T.s[env], a = T.a[env], s2 = T.s2[env];
  if ((unsigned)a >= (unsigned)A) return;  // an invalid action has no table entry
  const Row<A> row2 = load_row<A>(Qe + (size_t)s2 * A);
  const float m = row_max(row2, T.done[env] != 0, R.max_mode);
  const size_t k = (size_t)s * A + a;
  Qe[k] = td_value(Qe[k], T.r[env], m, R.lr, R.gamma);
}

// (key, delta) of n samples against ONE table (K = S*A entries), all reads before any
// write, for the reduction that scans them.  `before`: see signal_reached.
template <int A, class Samples>
__global__ __launch_bounds__(256) void k_delta(const float* __restrict__ Q, const Samples X, const int n,
                                                const float lr, const float gamma, const int max_mode,
                                                int32_t* __restrict__ key, float* __restrict__ delta,
                                                const HostSignal before) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int k;
  float d;
  sample_delta<A>(X, i, n, Q, lr, gamma, max_mode, k, d);
  if (i < n) {
    key[i] = k;
    delta[i] = d;
  }
  signal_reached(before);
}

// Shared table, first half of a fused step: every env selects, moves and emits
// (key, delta) against the table as it stands; nothing is written to Q.  With
// REDUCE the workgroup (= one 256-sample block of the ordered reduction) also
// folds its own deltas and hands the block sums to the key owners.
// MAP = 1: shared map staged in LDS; MAP = 2: maps in global memory.
template <int A, int MAP, bool REDUCE>
__global__ __launch_bounds__(256) void k_shared_act(const Rules R, const Ptrs P, const uint64_t t,
                                                     const int trace_row,
                                                     int32_t* __restrict__ key,
                                                     float* __restrict__ delta, const ReduceGeom G,
                                                     unsigned long long* __restrict__ handoff) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  uint32_t* lds_map = reinterpret_cast<uint32_t*>(lds_raw + (REDUCE ? block_lds_bytes(G.own_shift) : 0));
  const int tid = threadIdx.x;
  const int env = blockIdx.x * blockDim.x + tid;
  bool live = env < P.N;
  // the env's cell is fetched while the map streams into LDS
  const int s_in = live ? P.s[env] : 0;
  if (REDUCE) block_lds_init(lds_raw, G);
  if (MAP == 1)
    for (int i = tid; i < P.map_words; i += blockDim.x) lds_map[i] = P.map[i];
  if (MAP == 1 || REDUCE) __syncthreads();
  int my_key = 0;
  float my_delta = 0.0f;
  if (live && R.max_episodes > 0 && P.episode[env] >= R.max_episodes) {
    live = false;  // budget used up: no move, no delta
    key[env] = -1;
    delta[env] = 0.0f;
    trace_idle(P, env, trace_row, s_in);
  }
  if (live) {
    const uint32_t* gmap = P.map + (P.map_shared ? 0 : (size_t)env * P.map_words);
    auto cls = [&](int cell) -> int {
      const uint32_t word = (MAP == 1) ? lds_map[cell >> 4] : gmap[cell >> 4];
      return cell_class_of(word, cell);
    };
    const float* cr =
        P.cell_reward ? P.cell_reward + (P.map_shared ? 0 : (size_t)env * P.S) : nullptr;
    const float* __restrict__ Q = P.Q;

    const int s0 = s_in;
    int x = s0 % R.W, y = s0 / R.W;
    const Row<A> row = load_row<A>(Q + (size_t)s0 * A);
    // The TD target needs the largest value of the row of the cell the move ends
    // on - one of the A neighbours, or this cell.  All of them are asked for now,
    // with the env's own row, instead of one more dependent round trip once the
    // action is known (the table is small and shared: these reads hit the caches).
    float nb_max[A];
#pragma unroll
    for (int i = 0; i < A; ++i) {
      int dx, dy;
      action_delta(i, A, dx, dy);
      const bool in = (unsigned)(x + dx) < (unsigned)R.W && (unsigned)(y + dy) < (unsigned)R.H;
      const int cell = in ? s0 + dy * R.W + dx : s0;
      nb_max[i] = row_max(load_row<A>(Q + (size_t)cell * A), false, 0);
    }
    Draw d = pick_draw(explore_block(R.seed, (uint32_t)env, t >> 1), t, A);
    if (P.u_sup && t >= P.sup_t0 && t - P.sup_t0 < (uint64_t)P.sup_n) {
      const size_t o = (size_t)(t - P.sup_t0) * P.N + env;
      d.u = P.u_sup[o];
      d.a = P.a_sup[o];
    }
    const int episode = P.episode[env];
    const float eps = eps_of(R, P.eps_tab, t, episode);
    const int a = (d.u < eps) ? d.a : row_argmax(row);
    float reward;
    bool hit;
    step_rule(R, ClassRewards{R.step_reward, R.goal_reward, R.trap_reward}, cls, cr, x, y, a, reward, hit);
    const int s2 = y * R.W + x;
    const bool done = hit || (!R.auto_reset && P.done[env] != 0);
    float m = row_max(row, false, 0);  // the env stayed where it was
#pragma unroll
    for (int i = 0; i < A; ++i) m = (s2 != s0 && a == i) ? nb_max[i] : m;
    if (R.max_mode == 1) m = fmaxf(0.0f, m);
    m = done ? 0.0f : m;
    my_key = s0 * A + a;
    my_delta = td_delta(row_get(row, a), reward, m, R.lr, R.gamma);
    key[env] = my_key;
    delta[env] = my_delta;

    const int ep_step = P.ep_step[env] + 1;
    P.reward[env] = reward;
    P.done[env] = done ? 1 : 0;
    P.action[env] = (uint8_t)a;
    if (env < P.trace_n && trace_row < P.trace_cap) {
      const size_t o = (size_t)trace_row * P.trace_n + env;
      P.tr_s[o] = s2;
      P.tr_a[o] = (uint8_t)a;
      P.tr_r[o] = reward;
      P.tr_d[o] = done ? 1 : 0;
    }
    const float ret = P.ret_acc ? P.ret_acc[env] + reward : 0.0f;
    if (R.auto_reset && (done || (R.episode_len > 0 && ep_step >= R.episode_len))) {
      if (P.ret_acc) {
        record_episode(P, env, ret, ep_step);
        P.ret_acc[env] = 0.0f;
      }
      P.s[env] = P.start[env];
      P.ep_step[env] = 0;
      P.episode[env] = episode + 1;
    } else {
      if (P.ret_acc) P.ret_acc[env] = ret;
      P.s[env] = s2;
      P.ep_step[env] = ep_step;
    }
  }
  if (REDUCE) reduce_block_wide(lds_raw, G, blockIdx.x, my_key, my_delta, live, handoff);
}

// Move codes of maps [first, first + count) from their class maps: one thread per
// word of codes.
template <int A>
__global__ __launch_bounds__(256) void k_build_moves(const uint32_t* __restrict__ map,
                                                      const int map_words, const int W, const int H,
                                                      const int mv_words, const int first,
                                                      const int count, uint32_t* __restrict__ moves) {
  constexpr int kCells = move_cells_per_word<A>();
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)count * mv_words) return;
  const int m = first + (int)(i / mv_words), w = (int)(i % mv_words);
  const uint32_t* g = map + (size_t)m * map_words;
  uint32_t out = 0;
#pragma unroll
  for (int j = 0; j < kCells; ++j) {
    const int c = w * kCells + j;
    if (c < W * H) {
      const uint32_t mv = moves_of_cell<A>([&](int word) -> uint32_t { return g[word]; }, W, H, c % W, c / W, c);
      out |= mv << (j * 2 * A);
    }
  }
  moves[(size_t)m * mv_words + w] = out;
}

__global__ void k_fill_u32(unsigned* p, const unsigned v, const size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
// n16 16-byte words, four to a thread of 256
__global__ __launch_bounds__(256) void k_clear16(uint4* __restrict__ p, const size_t n16) {
  const size_t i0 = (size_t)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (i0 + 256 * u < n16) p[i0 + 256 * u] = make_uint4(0u, 0u, 0u, 0u);
}
// (a launch instead of a device-to-device copy: a caller may record the call)
__global__ void k_copy3_u32(const unsigned* __restrict__ src, unsigned* __restrict__ dst) {
  if (threadIdx.x < 3) dst[threadIdx.x] = src[threadIdx.x];
}

// plain copy of n16 16-byte words: the known-size launch that calibrates the
// hardware traffic counters
__global__ __launch_bounds__(256) void k_probe_copy(const uint4* __restrict__ src,
                                                     uint4* __restrict__ dst, const size_t n16) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

}  // namespace crl
