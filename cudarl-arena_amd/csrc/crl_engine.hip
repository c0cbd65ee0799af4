// C ABI of the engine (include/crl.h): owns the device buffers, validates
// arguments on the host and launches the gfx950 kernels of crl_kernels.h.
// There is no CPU fallback anywhere in this file.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdarg>
#include <cstdio>
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/crl.h"
#include "crl_host.h"
#include "crl_kernels.h"
#include "crl_persist.h"
#include "crl_pinned.h"

namespace {

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  return crl::fail_with(code, buf);
}

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess)                                                               \
      return fail(_e == hipErrorOutOfMemory ? CRL_E_ALLOC : CRL_E_DEVICE, "%s: %s (%s:%d)", \
                  #expr, hipGetErrorString(_e), __FILE__, __LINE__);                    \
  } while (0)

// Runs the body of an entry point that allocates host memory or starts threads:
// nothing may throw across the C ABI.
template <class F>
int guarded(F&& body) {
  try {
    return body();
  } catch (const std::bad_alloc&) {
    return fail(CRL_E_ALLOC, "host allocation failed");
  } catch (const std::exception& x) {
    return fail(CRL_E_DEVICE, "%s", x.what());
  } catch (...) {
    return fail(CRL_E_DEVICE, "unknown failure");
  }
}

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  bool owned = false;
  hipError_t alloc(size_t count) {
    release();
    if (count == 0) return hipSuccess;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&p), count * sizeof(T));
    if (e == hipSuccess) {
      n = count;
    } else {
      p = nullptr;
      (void)hipGetLastError();  // reported here, not by the next launch's check
    }
    owned = p != nullptr;
    return e;
  }
  hipError_t ensure(size_t count) { return count <= n ? hipSuccess : alloc(count); }
  // `count` elements in a new allocation, the old one handed over to `keep` instead of freed (at
  // least twice as many as now, so that what is kept never exceeds what is in use)
  hipError_t replace(size_t count, std::vector<void*>& keep) {
    if (count <= n) return hipSuccess;
    count = std::max(count, 2 * n);
    if (owned) {
      try {
        keep.push_back(p);
      } catch (...) {
        return hipErrorOutOfMemory;
      }
      owned = false;
    }
    return alloc(count);
  }
  // a piece of somebody else's allocation
  void adopt(void* at, size_t count) {
    release();
    p = static_cast<T*>(at);
    n = count;
  }
  void release() {
    if (p && owned) (void)hipFree(p);
    p = nullptr;
    n = 0;
    owned = false;
  }
  ~DevBuf() { release(); }
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
};

// Scratch of crl_run_fused_noalloc: one array per GPU, part of the loaded code
// object, so the entry point never allocates.  Layout: 4 KB of counters (the ticket
// counters), then 10 MB for what the workgroups of a shared-table step exchange: the
// hand-off cells of the ordered reduction, or all exchange buffers of the one-launch
// kernel.  The array's name
// is a host-side stand-in, not a device address: host code only ever uses the
// address hipGetSymbolAddress returned for the device at hand.
constexpr size_t kScratchTicketBytes = 4096;
constexpr size_t kScratchExchangeBytes = (size_t)10 << 20;
constexpr size_t kScratchBytes = kScratchTicketBytes + kScratchExchangeBytes;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Address of `device`'s copy of the scratch array; looked up once per device, with
// that device current.  Called from crl_create, so that crl_run_fused_noalloc
// finds it there.
int scratch_of_device(int device, unsigned char** out) {
  if (device < 0 || device >= kMaxDevices) return fail(CRL_E_ARG, "device %d: at most %d devices", device, kMaxDevices);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch_ptr[device]) {
    HIP_TRY(hipSetDevice(device));
    void* p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(CRL_E_DEVICE, "hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_ptr[device] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch_ptr[device];
  return CRL_OK;
}

}  // namespace

// Keeps the pool of pinned blocks alive; the engine's first member, so the last one to go.
struct PoolUser {
  PoolUser() { crl::PinnedPool::get().add_user(); }
  ~PoolUser() { crl::PinnedPool::get().drop_user(); }
};

struct crl_engine {
  PoolUser pool_user;
  crl_config cfg{};
  int device = 0;
  hipStream_t stream = nullptr;
  int N = 0, W = 0, H = 0, A = 0;
  size_t S = 0, K = 0;
  int n_maps = 0, n_tables = 0, map_words = 0;
  int mv_words = 0;  // words of move codes per map; 0: no move codes are kept
  uint64_t t = 0;
  long resident_envs = 0;  // 0 = automatic
  int fused_variant = 0;   // 0 = automatic, 1 = plain, 2 = hybrid (when it fits)
  DevBuf<unsigned> ticket;
  DevBuf<unsigned> split;  // the engine's own copy of the last launch's ticket counters (crl_get_fused_split)
  bool hybrid_opt_in = false;
  // the scratch the call in progress works with: the engine's own allocations
  // (crl_run_fused, crl_update, crl_td_update) or the device's static array
  // (crl_run_fused_noalloc)
  bool no_alloc = false;
  unsigned char* static_scratch = nullptr;
  unsigned* tk = nullptr;  // ticket counters {next ticket, envs on HBM tables, envs on LDS tables}
  bool split_valid = false;  // the last fused launch drew tickets
  unsigned long long* ho = nullptr;  // hand-off cells of the ordered reduction
  // what the workgroups of a shared-table step exchange: the hand-off cells of the ordered
  // reduction, or all buffers of the one-launch kernel (the tagged views of the table's
  // cells, raw samples, hand-off cells)
  DevBuf<unsigned long long> exchange;
  // one-launch shared-table kernel: the engine's own give-up word followed by the phase
  // clocks, and whether a launch has not been checked for having given up yet
  DevBuf<unsigned long long> pdiag;  // [0] give-up word, [1..16] phase clocks; allocated at crl_create
  // The tags in `exchange` are at most this; 0: something else lies there, or may.  (Not kept once a
  // call has been recorded: a replay clears and counts from the start.)
  uint32_t exchange_tag = 0;
  bool persist_unchecked = false;
  bool persist_failed = false;   // a launch gave up: state and table are not valid until they are set again
  bool persist_refused = false;  // the device refused the co-resident launch once: not tried again
  bool persist_clocks = false;   // run the instantiation that keeps phase clocks
  int persist_spin_limit = crl::kPersistSpinLimit;  // polls a thread waits for its peers before it gives up

  // One allocation holds every array below that crl_create() makes, in the order it lists
  // them: what is read out together lies together (state_at: s, ep_step, episode, reward,
  // done, action; stats_at: the four statistics) and goes out in one piece.
  DevBuf<unsigned char> arena;
  unsigned char* state_at = nullptr;
  size_t state_bytes = 0;
  unsigned char* stats_at = nullptr;
  size_t stats_bytes = 0;

  // Pinned memory this engine and its kernels talk through.
  crl::PinBuf flag_page;        // word 0: number of the last signalled launch that is through; word 16: give-up word
  DevBuf<unsigned> flag_count;  // workgroups of a signalling launch that are through
  unsigned seq = 0;             // number of the last signalled launch
  crl::PinBuf out_page;         // what kernels hand to the host: state, statistics, actions, tables
  // What the host hands to kernels: one pinned block cut into pages that are taken in turn.
  crl::PinBuf in_block;
  struct InSlot {
    unsigned char* page = nullptr;
    unsigned last_seq = 0;  // the launch that reads it
  };
  static constexpr int kInSlots = 4;
  InSlot in_slot[kInSlots];
  int in_slots = 0, in_next = 0;  // pages there are, the one taken next
  size_t in_page_bytes = 0;
  // A call of this engine has been recorded into a graph: what its launches work on stays
  // allocated until the engine goes, also where a later call needs a larger buffer.
  bool recorded = false;
  struct Outgrown {
    std::vector<void*> p;
    ~Outgrown() {
      for (void* x : p) (void)hipFree(x);
    }
  } outgrown;
  template <class T>
  hipError_t grow(DevBuf<T>& buf, size_t count) {
    return recorded ? buf.replace(count, outgrown.p) : buf.ensure(count);
  }
  bool state_shared = false;    // the state may change between calls: device pointers to it are out,
                                // or a call that changes it has been recorded and may be replayed
  bool mirror_steps = false;    // crl_step's kernel also writes the state to out_page ...
  bool mirror_read = false;     // ... because the state was read after the step before
  bool stepped = false;         // crl_step was the last call that changed the state
  unsigned mirror_seq = 0;      // != 0: out_page holds the state as of this launch
  bool state_read = false;      // crl_get_state was called since the state last changed
  bool stats_follow = false;    // the statistics were read after the state the last time: they go out with it ...
  bool stats_here = false;      // ... and are in out_page, behind the state

  DevBuf<int32_t> s, ep_step, episode, start, act;
  DevBuf<float> reward;
  DevBuf<uint8_t> done, action;
  DevBuf<uint32_t> map;
  DevBuf<uint32_t> moves;  // move codes derived from map, for the folded fused loop
  DevBuf<float> cell_reward;
  DevBuf<float> Q;
  DevBuf<float> eps_tab;
  int eps_len = 1;
  // episode statistics (allocated when cfg.track_returns)
  DevBuf<float> ret_acc, ret_last, ret_sum;
  DevBuf<int32_t> len_last, len_sum;
  // transition of the last crl_step
  DevBuf<int32_t> tr_s, tr_a, tr_s2;
  DevBuf<float> tr_r;
  DevBuf<uint8_t> tr_done;
  bool have_transition = false, have_actions = false;
  // (key, delta) scratch of the ordered reduction
  DevBuf<int32_t> key;
  DevBuf<float> delta;
  bool lds_opt_in = false;
  // trace
  DevBuf<int32_t> trace_s;
  DevBuf<uint8_t> trace_a, trace_d;
  DevBuf<float> trace_r;
  int trace_n = 0, trace_cap = 0, trace_cursor = 0;
  // supplied exploration stream
  DevBuf<float> u_sup;
  DevBuf<int32_t> a_sup;
  uint64_t sup_t0 = 0;
  int sup_n = 0;

  crl::Rules rules() const {
    crl::Rules R{};
    R.W = W;
    R.H = H;
    R.A = A;
    R.goal_mode = cfg.goal_mode;
    R.reward_flags = cfg.reward_flags;
    R.auto_reset = cfg.auto_reset;
    R.episode_len = cfg.episode_len;
    R.max_mode = cfg.max_mode;
    R.eps_mode = cfg.eps_mode;
    R.eps_len = eps_len;
    R.max_episodes = cfg.max_episodes;
    R.lr = cfg.lr;
    R.gamma = cfg.gamma;
    R.step_reward = cfg.step_reward;
    R.goal_reward = cfg.goal_reward;
    R.trap_reward = cfg.trap_reward;
    R.eps0 = cfg.eps0;
    R.seed = cfg.seed;
    return R;
  }
  crl::Ptrs ptrs() const {
    crl::Ptrs P{};
    P.s = s.p;
    P.ep_step = ep_step.p;
    P.episode = episode.p;
    P.start = start.p;
    P.reward = reward.p;
    P.done = done.p;
    P.action = action.p;
    P.map = map.p;
    P.moves = moves.p;
    P.cell_reward = (cfg.reward_flags & CRL_REWARD_CELLS) ? cell_reward.p : nullptr;
    P.Q = Q.p;
    P.eps_tab = eps_tab.p;
    P.u_sup = sup_n > 0 ? u_sup.p : nullptr;
    P.a_sup = a_sup.p;
    P.sup_t0 = sup_t0;
    P.sup_n = sup_n;
    P.tr_s = trace_s.p;
    P.tr_a = trace_a.p;
    P.tr_r = trace_r.p;
    P.tr_d = trace_d.p;
    P.trace_n = trace_n;
    P.trace_cursor = trace_cursor;
    P.trace_cap = trace_cap;
    P.ret_acc = ret_acc.p;
    P.ret_last = ret_last.p;
    P.ret_sum = ret_sum.p;
    P.len_last = len_last.p;
    P.len_sum = len_sum.p;
    P.N = N;
    P.map_words = map_words;
    P.mv_words = mv_words;
    P.map_shared = cfg.map_mode == CRL_MAP_SHARED;
    P.table_shared = cfg.table_mode == CRL_TABLE_SHARED;
    P.S = S;
    return P;
  }
  crl::Transition transition() const {
    crl::Transition T{};
    T.s = tr_s.p;
    T.a = tr_a.p;
    T.r = tr_r.p;
    T.s2 = tr_s2.p;
    T.done = tr_done.p;
    return T;
  }
};

namespace {

constexpr int kLdsMapLimitBytes = 64 * 1024;
// Table bytes to keep in flight at once: three quarters of the MI355X Infinity
// Cache (256 MB).  Measured on 4 KB tables (table waves alone): 128 MB in flight 5.9e10 env-steps/s,
// 192 MB 6.3e10, 256 MB 5.2e10, 384 MB 3.9e10.
constexpr size_t kTableBytesInFlight = (size_t)192 << 20;
constexpr int kComputeUnits = 256;
constexpr long kMinEnvsInFlight = kComputeUnits * 3L * 64;  // three waves per compute unit
// Shorter launches have all envs in flight (all / as many as that, 2 / 4 / 6 / 8 / 12 steps: 1M envs of 16x16
// 107 / 176 / 251 / 332 / 503 us, 127 / 175 / 225 / 275 / 378; 100,000 of 32x32 27 / 34 / 41 / 48 / 66,
// 28 / 35 / 42 / 48 / 61; 200,000 of 16x16 with 8 actions 31 / 52 / 73 / 94 / 136, 31 / 46 / 60 / 74 / 104).
// The general loop on a shared map, 4 actions, loses by two shifts (20x20, 80,000 envs, statistics and epsilon by
// episode, 6 / 14 steps 21.0 / 42.7, 24.4 / 47.1; three shifts of 16x16, 14 steps 80.9, 69.5; with 8 actions, two of
// 20x20, 55.1, 51.0; two of 60x60, 9 steps 29.7, 28.5).
// Maps of their own and of some 1000 cells, whose tables' lines a few steps meet once, lose longer by three shifts
// and more, or two with 8 actions (105,108 envs of 43x23, 6 / 9 / 11 steps 43.1 / 56.0 / 66.9, 47.5 / 57.4 / 64.0; 200,000
// 66.0 / 87.9 / 105.0, 78.2 / 96.0 / 107.8; 105,000 of 32x32, epsilon by episode, 6 / 8 38.9 / 46.8, 44.6 / 51.2; 57,155 of 26x37
// with 8 actions, statistics, 6 / 7 34.5 / 38.3, 38.9 / 42.3; past 65,536 of these workgroups of four waves are one to a
// unit and some late: 67,524 of 24x44, 6 steps 46.2, 35.5).
constexpr int kInFlightMinSteps = 6, kInFlightMinStepsTwoShifts = 16, kInFlightMinStepsLargeMaps = 10;
constexpr size_t kInFlightLargeMap = 900;

// launch geometry of the fused per-env kernel
struct FusedPlan {
  int map_kind;  // 0 per-env LDS, 1 shared LDS, 2 global
  int block, grid;
  size_t lds;
  const char* name;
  bool tickets;    // per-env maps in LDS: waves draw env ranges from a ticket counter
  bool hybrid;     // ... whose last wave per workgroup steps envs whose tables it holds in LDS
  bool fast;       // the folded loop for the common configuration
  bool moves;      // ... whose table waves read pre-built move codes from LDS
  bool fixed;      // tickets dealt by position, round after round: no counter
  bool lanes;      // an env to A lanes, a wave to 2^log_envs envs, draws taped tape_steps ahead
  int log_envs, tape_steps;
  bool touch;      // ... whose tables are read ahead whole
  int rows;        // != 0: 64-env waves that keep their envs' rows in LDS, in so many places (moves: and not their maps)
  bool rich;       // ticket kernel: the folded loop's variant with per-cell rewards / per-episode epsilon
  int tab_stride;  // floats between two tables in LDS
  bool in_lds;     // ... with all tables in LDS
  bool words;      // ... beside their move words
  int env_bytes;   // ... bytes per env
  int lds_waves;   // hybrid: waves of a workgroup that work on LDS tables ...
};

constexpr size_t kLdsPerWorkgroup = 160 * 1024;  // gfx950
// static LDS of kernels that call the workgroup-wide "or" (the device library keeps a few
// words there), rounded up: their dynamic LDS can be at most the rest
constexpr size_t kStaticLdsReserve = 1024;
// How many workgroups that ask for `bytes` fit a compute unit: LDS is given out in pieces of 1280 bytes.
// (Counted in 1024, lane waves of 45x19 maps, 8 actions, 14,240 bytes, were put 11 to a unit where 10 fit, and the
// eleventh ran after the others: 131 steps, 10 / 11 to a unit 96 / 150 us; of 24x20, 8240 bytes, 17 / 18 / 19
// 132 / 142 / 190; of 28x25, 11,760 bytes, 12 / 13 105 / 157.)
constexpr size_t kLdsPiece = 1280;
constexpr long lds_fit(size_t bytes) { return (long)(kLdsPerWorkgroup / ((bytes + kLdsPiece - 1) / kLdsPiece * kLdsPiece)); }

// Where lane waves are no choice (rules they leave out, a caller that sets the envs in flight), launches shorter
// than this do not repay moving whole tables into LDS and back (beside lane waves: hybrid_pays in plan_fused).
// (1M envs of 16x16, steps per launch -> env-steps/s, 64-env waves / hybrid:
// 32: 2.4e10 / 2.1e10, 48: 2.8e10 / 2.75e10, 64: 3.0e10 / 3.3e10, 100: 3.6e10 / 4.2e10).
constexpr int kHybridMinSteps = 64;
constexpr int kStagedMovesMinSteps = 128;
constexpr int kLdsMinSteps = 16, kLdsAlwaysSteps = 144;
constexpr size_t kLdsBytesFree = 8192, kLdsBytesPerStep = 208, kLdsSmallWaveBytes = 5120, kLdsSmallMoved = 17000;
constexpr int kLongLaunchSteps = 4096;
constexpr int kLaneWavesMinSteps = 8;
constexpr int kLaneRoundsMinSteps = 64, kLaneRoundsManyMinSteps = 131;
constexpr int kLaneFewRoundsMinSteps = 48;
constexpr long kLaneRoundsManyEnvs = 65536;
constexpr int kLaneUnevenMinSteps = 384, kLaneUnevenManyRoundsMinSteps = 192;
constexpr int kLaneRoundsFourMinSteps = 64, kLaneRoundsFourLongSteps = 300;
constexpr int kLaneDrawnMinSteps = 256, kLaneDrawnManyMinSteps = 128;
constexpr int kLaneTouchMinSteps4 = 90, kLaneTouchMinSteps8 = 160, kLaneTouchFourRoundsMinSteps = 200;
// Hybrid workgroups in place of rounds of lane waves.
constexpr int kHybridFewRoundsMinSteps = 384, kHybridOneWaveMinSteps = 96;
constexpr long kHybridEnvStepsSmall = 18000000, kHybridEnvSteps4 = 24000000, kHybridEnvSteps8 = 28000000, kHybridEnvSteps8FewRounds = 20000000;
constexpr size_t kTableBytesAtOnce = (size_t)512 << 20;
// 64-env waves that keep rows in LDS, with the maps in LDS too where enough of them fit a compute unit, else the move codes
// come from HBM with the rows (20 steps, staged / not: 1M of 16x16 369 / 452 us, 100,000 of 22x22 with 8 actions 62 / 69, of
// 32x32, six staged to a unit, 73 / 55; 262,144 of 28x28, seven, 10 / 40 / 150 steps 77 / 208 / 701, 78 / 215 / 725; of 32x32 with 8
// actions, whose codes are twice as long, 96 / 214 / 658 at 10 / 30 / 100, 104 / 251 / 788).
// Six places for an env's rows in place of four, in longer calls: fewer rows asked for again, fewer waves to a unit (four / six,
// 1M of 16x16, nine waves fit, 3 / 20 / 40 / 150 / 400 steps 111 / 362 / 598 / 2262 / 5944, 114 / 355 / 570 / 1907 / 5027; of 8x8, 40 / 150
// 487 / 2012, 438 / 1410; 300,000 of 20x20, eight, 24 / 50 / 150 126 / 236 / 681, 136 / 245 / 664; of 28x28, six, 40 / 150 208 / 701,
// 210 / 672; of 32x32, five, 150 steps 721, 797; 300,000 of 16x16 with 8 actions, 60 / 300 392 / 1965, 390 / 1806; eight places, 300 steps of
// 1M of 16x16 3747 -> 3967.  With epsilon by episode, where envs explore, 1M of 16x16, 24 / 60 / 200 steps 414 / 956 / 3118, 436 / 1033 / 3255).
// (which of plan_fused's figures each line comes from)
constexpr int kRowsManyEnvs = 1 << 18;           // in place of every other plan, whatever the table ...
constexpr int kRowsManyLargerTables = 200000;    // ... of more than 256 values
constexpr int kRowsHybridSteps4 = 48, kRowsHybridSteps8 = 96;  // up to so many steps, and some for each key, before hybrid workgroups
constexpr int kRowsLanesSteps = 500;             // up to so many, 8 actions or epsilon by episode, before rounds of lane waves
constexpr int kRowsSomeEnvs = 6 * 64 * kComputeUnits, kRowsSomeEnvsRich = 1 << 17, kRowsSomeEnvsSteps = 88;  // fewer envs: in place of lane waves in two rounds and more
constexpr long kRowsRewardsSmallEnvs = 22L * 64 * kComputeUnits;  // with rewards of all cells
constexpr size_t kRowsRewardsSmallest = 25, kRowsRewardsSmaller = 26, kRowsRewardsSmall = 28, kRowsRewardsMiddle = 100, kRowsRewardsLarge = 256;  // cells: with rewards per cell ...
constexpr int kRowsRewardsMiddleSteps = 200, kRowsRewardsLargeSteps = 240;             // ... up to so many steps (cells_steps)
constexpr size_t kRowsSmallMap = 336;            // cells: eleven to a unit
constexpr int kRowsLargeMapMinSteps = 11, kRowsLargeMapMaxSteps = 130;  // larger maps, fewer envs: where plain 64-env waves are the other choice
constexpr long kRowsStagedWaves4 = 7, kRowsStagedWaves8 = 6;  // maps in LDS if so many waves then fit a unit (above)
constexpr long kRowsSixSoonWaves = 9, kRowsSixWaves = 6;      // six places if so many waves fit (above) ...
constexpr int kRowsSixSoonSteps = 32, kRowsSixSteps = 100;    // ... in calls of so many steps
// against plain waves (rows_pay):
constexpr long kRowsCells4 = 80, kRowsCells4Rich = 60, kRowsCells4Fixed = 40, kRowsCells8 = 96, kRowsCells8Rich = 80;  // cells to a step ...
constexpr long kRowsCells4Rewards = 32, kRowsCells8Rewards = 16;  // ... with rewards per cell and more than two waves to a unit
constexpr long kRowsRewardsEnvs = 10L * 16 * kComputeUnits;   // rewards per cell, large maps: 2.5 waves to a unit
constexpr long kRowsFixedEnvs = 11L * 16 * kComputeUnits;     // epsilon fixed, large maps: 2.75 waves to a unit ...
constexpr size_t kRowsFixedMap8 = 1300;                       // ... with 8 actions up to so many cells
constexpr int kRowsFixedMinSteps = 3;                         // epsilon fixed or rewards per cell, four waves to a unit
constexpr size_t kRowsTwoStepsMap = 600;                      // many envs, epsilon by episode: two steps are too few on more cells
// against lane waves with a floored maximum (rows_late):
constexpr int kRowsTwoRoundsSteps = 20, kRowsLateSteps = 240, kRowsSmallestTablesSteps = 64;
constexpr long kRowsTwoRoundsWaves = 27, kRowsLateWaves = 12;
constexpr size_t kRowsSmallestTables = 40;

// Configurations that run_lanes() steps: no goal test on the resulting cell, no sticky done,
// no trace and no supplied stream.
bool lanes_rules(const crl_engine* e) {
  const crl_config& c = e->cfg;
  return c.goal_mode == CRL_GOAL_ON_TARGET && c.auto_reset == 1 && e->trace_n == 0 && e->sup_n == 0;
}
// steps of a tape: enough that all 64 lanes have a Philox block to work out
int tape_steps_for(int log_envs) { return std::max(16, 128 >> log_envs); }
size_t tape_bytes(int log_envs) { return ((size_t)(tape_steps_for(log_envs) + 1) << log_envs) * 4; }
// as few envs to a wave as leaves no more than `waves` of them, and as many as it has lanes for
int lanes_log_envs(const crl_engine* e, long waves) {
  const int most = e->A == 8 ? 3 : 4;
  int log_envs = 0;
  while (log_envs < most && ((long)e->N + (1L << log_envs) - 1) >> log_envs > waves) ++log_envs;
  return log_envs;
}

// All tables in LDS, if they fit there with the envs spread over every SIMD of the chip.
// Not for launches so short that moving the tables in and out costs more than it saves.
bool plan_fused_lds(const crl_engine* e, int n_steps, FusedPlan* p) {
  const crl_config& c = e->cfg;
  if (!lanes_rules(e) || c.reward_flags != 0 || e->fused_variant != 0 || e->resident_envs != 0 || n_steps < kLdsMinSteps)
    return false;
  const bool shared = c.map_mode == CRL_MAP_SHARED;
  if (!shared && (size_t)e->map_words * 4 * 64 > (size_t)kLdsMapLimitBytes) return false;
  const int log_envs = lanes_log_envs(e, 4L * kComputeUnits);
  const long waves = ((long)e->N + (1L << log_envs) - 1) >> log_envs;
  const size_t per_unit = (size_t)((waves + kComputeUnits - 1) / kComputeUnits);
  // (an env's pieces in whole rows of 16 bytes, and a row more against bank conflicts)
  const size_t code_bytes = (size_t)e->mv_words * 4;
  const size_t env_bytes[2] = {((4 * e->K + (shared ? 0 : code_bytes) + 15) & ~(size_t)15) + 16, 8 * e->K + 16};
  for (int words = 1; words >= 0; --words) {
    const size_t bytes = 16 + (env_bytes[words] << log_envs) + tape_bytes(log_envs) + (shared && !words ? code_bytes : 0);
    // (pieces of 1024 bytes, not the 1280 of lds_fit: a unit's last wave may run after the others.  With the smallest
    // tables that is better than lane waves on HBM - 77,524 envs of 4x6, 160 / 500 steps 107 / 297 us, 120 / 357 - with
    // larger ones worse: 20,180 of 19x6 94 / 223, 54 / 153.)
    if (((bytes + 1023) & ~(size_t)1023) * per_unit > kLdsPerWorkgroup) continue;
    // What a wave's tables, or a quarter of a compute unit's, take to move in and out against the
    // steps' trips to HBM (tables in LDS / in HBM: 4096 envs of 16x16, 16 KB to a wave, 32 / 48 steps
    // 12.7 / 11.7, 14.9 / 15.5 us; 2000 of 32x32, 32 KB, 64 / 128 / 200 steps 22.0 / 18.9, 30.5 / 30.6,
    // 40.3 / 44.4; 30,000 of 8x8, eight waves of 16 KB to a unit, 64 / 128 steps 29.5 / 25.2, 42.9 / 43.3;
    // 100 of 48x48 with 8 actions, 72 KB, 128 / 200 steps 30.4 / 28.1, 39.6 / 41.4).
    // The smallest tables of 4 actions (up to 5 KB to a wave) cross sooner, beside their move words at
    // once (15.5 waves to a unit, 4x4, 16 / 32 steps: 13.1 / 17.6, 15.4 / 23.3 us; 12 waves, 5x4, 32 steps 16.4,
    // 20.2), beside move codes at some 40 steps (24 waves, 4x4, 32 / 64 steps 32.6 / 48.2, 34.9 / 62.6; 20 waves,
    // 5x4 29.9 / 43.3, 33.3 / 54.7).
    const size_t wave_bytes = (4 * e->K) << log_envs;
    size_t moved = std::max<size_t>(wave_bytes, wave_bytes * per_unit / 4);
    if (e->A == 4 && wave_bytes <= kLdsSmallWaveBytes) moved = words ? wave_bytes : std::min(moved, kLdsSmallMoved);
    if (n_steps < kLdsAlwaysSteps && (size_t)n_steps * kLdsBytesPerStep + kLdsBytesFree < moved) return false;
    p->in_lds = p->lanes = p->fast = true;
    p->words = words != 0;
    p->rich = c.eps_mode >= CRL_EPS_EPISODE_MULT;
    p->log_envs = log_envs;
    p->tape_steps = tape_steps_for(log_envs);
    p->env_bytes = (int)env_bytes[words];
    p->block = 64;
    p->grid = (int)waves;
    p->lds = bytes;
    p->map_kind = shared ? 1 : 0;
    static const char* names[2][2][2] = {
        {{"k_fused_tickets_lds<4,fast>", "k_fused_tickets_lds<4,fast+>"},
         {"k_fused_per_env_lds<4,fast>", "k_fused_per_env_lds<4,fast+>"}},
        {{"k_fused_tickets_lds<8,fast>", "k_fused_tickets_lds<8,fast+>"},
         {"k_fused_per_env_lds<8,fast>", "k_fused_per_env_lds<8,fast+>"}}};
    p->name = names[e->A == 8][shared][p->rich];
    return true;
  }
  return false;
}

FusedPlan plan_fused(const crl_engine* e, int n_steps) {
  FusedPlan p{};
  if (plan_fused_lds(e, n_steps, &p)) return p;
  // small batches spread over more compute units with one-wave blocks
  p.block = e->N >= 256 * 512 ? 256 : 64;
  if (e->cfg.map_mode == CRL_MAP_SHARED) {
    if ((size_t)e->mv_words * 4 <= (size_t)kLdsMapLimitBytes) {
      p.map_kind = 1;
      p.lds = (size_t)e->mv_words * 4;  // the shared map's move codes
    } else {
      p.map_kind = 2;
    }
  } else {
    if ((size_t)e->map_words * 4 * 64 <= (size_t)kLdsMapLimitBytes) {
      p.map_kind = 0;
      while ((size_t)e->map_words * 4 * p.block > (size_t)kLdsMapLimitBytes) p.block /= 2;
      p.lds = (size_t)e->map_words * 4 * p.block;
    } else {
      p.map_kind = 2;
    }
  }
  const crl_config& c = e->cfg;
  // what the folded loop leaves out altogether ...
  const bool foldable = c.goal_mode == CRL_GOAL_ON_TARGET && c.auto_reset == 1 && c.max_mode == CRL_MAX_TRUE &&
                        e->trace_n == 0 && e->sup_n == 0 && c.max_episodes == 0 && c.track_returns == 0 &&
                        e->mv_words > 0;
  // Envs live on the chip at once.  A worker steps its envs for all n steps
  // before it takes the next ones, so a smaller grid means fewer tables in
  // flight: when all tables together exceed what the last-level cache holds well,
  // keep that many bytes in flight (but never less than three waves per compute unit).
  long resident = e->resident_envs;
  if (resident <= 0) {
    const size_t table_bytes = e->K * sizeof(float);
    resident = e->N;
    // (a launch of a few steps re-uses no row often enough for that to matter: it
    // runs with every env in flight)
    const long fits = std::max<long>(kMinEnvsInFlight, (long)(kTableBytesInFlight / table_bytes));
    const bool general = !foldable || c.eps_mode == CRL_EPS_STEP_MULT;
    const bool two_shifts = p.map_kind == 1 && general && e->A == 4 && e->K < 4096 && e->N <= 2 * fits;
    const bool large_maps = p.map_kind == 0 && e->S >= kInFlightLargeMap && e->N > (e->A == 8 ? fits : 2 * fits) &&
                            (e->A == 4 || e->N <= 4 * 64 * kComputeUnits);
    const int min_steps = two_shifts ? kInFlightMinStepsTwoShifts : large_maps ? kInFlightMinStepsLargeMaps : kInFlightMinSteps;
    if ((size_t)e->N * table_bytes > kTableBytesInFlight && n_steps >= min_steps)
      resident = fits;
    // The batch goes through the chip in shifts of that many envs; a last shift that
    // fills a fraction of the chip costs a whole one.  Even the shifts out, in whole
    // waves per compute unit (65,536 envs with 32x32 maps: 3.5e10 env-steps/s as one
    // shift of 49,152 and one of 16,384, 4.4e10 as two of 32,768).
    if (resident < e->N) {
      const long shifts = (e->N + resident - 1) / resident;
      const long per_shift = (e->N + shifts - 1) / shifts;
      const long unit = 64L * kComputeUnits;
      resident = std::min(resident, (per_shift + unit - 1) / unit * unit);
    }
  }
  p.tickets = p.map_kind == 0;
  if (!p.tickets) {
    p.grid = (int)std::min<long>((e->N + p.block - 1) / p.block, std::max<long>(1, resident / p.block));
    // ... its variant for large or shared maps takes per-cell rewards and per-episode epsilon
    p.fast = foldable && c.eps_mode != CRL_EPS_STEP_MULT && c.table_mode != CRL_TABLE_SHARED;
    // An env to A lanes while that leaves the chip a wave or two per SIMD.
    const int log_envs = lanes_log_envs(e, 4L * kComputeUnits);
    const long waves = ((long)e->N + (1L << log_envs) - 1) >> log_envs;
    if (lanes_rules(e) && c.table_mode != CRL_TABLE_SHARED && (e->N + 63) / 64 <= kComputeUnits && resident >= e->N &&
        (e->K * sizeof(float)) << log_envs < (size_t)1 << 32) {
      p.fast = p.lanes = true;
      p.log_envs = log_envs;
      p.tape_steps = tape_steps_for(log_envs);
      const int per_block = waves > 2 * kComputeUnits ? 4 : waves > kComputeUnits ? 2 : 1;
      p.block = 64 * per_block;
      p.grid = (int)((waves + per_block - 1) / per_block);
      p.lds = 16 + per_block * tape_bytes(log_envs) + (p.map_kind == 1 ? (size_t)e->mv_words * 4 : 0);
    }
  } else {
    p.rich = foldable && c.eps_mode != CRL_EPS_STEP_MULT && !(c.eps_mode == CRL_EPS_FIXED && c.reward_flags == 0);
    p.fast = foldable && c.eps_mode != CRL_EPS_STEP_MULT;
    // Hybrid workgroups: some waves work on HBM tables, the others on whole tables in LDS.
    // One workgroup per compute unit (the LDS holds no second one).
    const size_t map_lds = (size_t)e->map_words * 64 * 4;
    const size_t mv_lds = (size_t)e->mv_words * 64 * 4;
    const int most_log_envs = e->A == 8 ? 3 : 4;  // an env to A lanes: the most that a wave has lanes for
    const long tickets = (e->N + crl::kTicketEnvs - 1) / crl::kTicketEnvs;
    // (not with per-cell rewards: they would stay in HBM, one request per step, and
    // a worker that waits for memory every step has no use for tables in LDS)
    bool fits = !p.rich;
    int hbm_waves = 0;
    if (p.fast) {
      // The folded loop's LDS waves give an env A lanes: two table waves, and beside them as
      // many LDS waves as there is room for up to three.  1M envs, 16x16 maps, table + LDS
      // waves: 1 + 2 7.6e10, 2 + 2 9.8e10, 3 + 2 9.4e10 (8x8, 2 + 3: 1.45e11);
      // 8 actions, 16x16: 2 + 1 4.2e10, 2 + 2 4.7e10, 3 + 2 4.2e10.
      hbm_waves = 2;
      p.log_envs = most_log_envs;
      p.tape_steps = tape_steps_for(p.log_envs);
      p.env_bytes = (int)(((4 * e->K + (size_t)e->mv_words * 4 + 15) & ~(size_t)15) + 16);
      const size_t wave_lds = ((size_t)p.env_bytes << p.log_envs) + tape_bytes(p.log_envs);
      p.lds_waves = 3;
      while (p.lds_waves > 0 && 16 + hbm_waves * map_lds + p.lds_waves * wave_lds > kLdsPerWorkgroup) --p.lds_waves;
      fits = fits && p.lds_waves > 0;
      // (no more than it uses: there is a compute unit for every workgroup, and LDS asked for so
      // that no second one fits beside it gains nothing - 1M envs of 8x8, 300 steps, 81 KB / 57 KB
      // 2.74 / 2.75 ms; 1M of 16x16, 1000 steps, 148.5 / 146.6 KB 11.75 / 11.75 ms)
      p.lds = 16 + hbm_waves * map_lds + p.lds_waves * wave_lds;
    } else {
      // The general loop's: 32 whole tables (padded by one row against bank conflicts), the
      // LDS wave's maps and at least one table wave's.
      p.tab_stride = (int)e->K + 4;
      p.lds_waves = 1;
      const size_t rest = map_lds + (size_t)crl::kTicketEnvs * p.tab_stride * 4;
      fits = fits && e->K % 4 == 0 && map_lds + rest <= kLdsPerWorkgroup;
      // at most three, so that the LDS wave has a SIMD to itself
      hbm_waves = (int)std::min<long>(3, std::max<long>(1, resident / (64L * kComputeUnits)));
      while (hbm_waves > 1 && hbm_waves * map_lds + rest > kLdsPerWorkgroup) --hbm_waves;
      p.lds = hbm_waves * map_lds + rest;
    }
    // Lane waves: an env to A lanes, one wave to a workgroup.
    // (one wave to a compute unit in long launches of small batches, whose rows are in the caches
    // most of the time; a wave to a SIMD in shorter ones, where most steps wait for a first use of
    // a line, and the fewer envs a wave has the less often: 4096 envs of 32x32, 256 steps 108 / 98 us)
    const long spread = n_steps > kLongLaunchSteps ? kComputeUnits : 4L * kComputeUnits;
    int lane_log_envs = most_log_envs;
    while (lane_log_envs > 0 && (e->N + (1L << lane_log_envs) - 1) >> lane_log_envs < spread) --lane_log_envs;
    const size_t lane_lds = 16 + tape_bytes(lane_log_envs) + ((size_t)e->mv_words * 4 << lane_log_envs);
    const long lane_fit = lds_fit(lane_lds);  // waves of a compute unit
    const long lane_units = (e->N + (1L << lane_log_envs) - 1) >> lane_log_envs;
    const bool lanes_can = lanes_rules(e) && (e->K * sizeof(float)) << lane_log_envs < (size_t)1 << 32;
    const size_t all_tables = (size_t)e->N * e->K * sizeof(float);
    const bool outgrown = all_tables > kTableBytesInFlight;
    // All envs at once: 24 waves to a compute unit are what the registers hold (80,000 envs of
    // 5x5 in one round 266 us, in two 361), 20 where the tables outgrow the caches - there 24
    // lose to the hybrid (98,000 envs of 16x16, 500 steps: 1294 / 650 us) and 15 to 20 win over
    // it and over 64-env waves (60,000 of 16x16, 64 / 500 steps: 143 / 566 hybrid, 86 / 420;
    // 40,000 of 20x20 with 8 actions, 130 steps: 212, 163) up to about 512 MB (65,536 of 32x32,
    // 1 GB, 300 steps: 503, 506).
    // With 4 actions rather fewer, in launches long enough that rows are used again: a full unit's waves
    // have less of the L2 each (waves to a unit; in one round / two, 31 / 130 / 300 / 800 steps: 17.1,
    // 70,000 envs of 6x6 28 / 95 / 208 / 625, 32 / 100 / 210 / 533 us; 19.5, 80,000 of 5x5 29 / 110 / 281 /
    // 769, 32 / 103 / 216 / 559; 19.8, 81,000 of 12x12 41 / 198 / 461 / 1214, 41 / 136 / 300 / 778; 22,
    // 90,000 of 7x7 130 steps 182, 117; epsilon by episode: 19.5 111 / 273, 129 / 280, 22 184 / 416, 138 /
    // 295; with 8 actions 43,662 of 10x10, 21.3, 29 / 90 / 186, 36 / 108 / 234).
    const bool by_episode = c.eps_mode >= CRL_EPS_EPISODE_MULT;
    const long at_once_waves = e->A == 4 && n_steps >= kLaneRoundsFourMinSteps
                                   ? (by_episode ? 20L : n_steps >= kLaneRoundsFourLongSteps ? 16L : 18L)
                                   : outgrown ? 20L : 24L;
    const bool lanes_at_once = lanes_can && lane_units <= kComputeUnits * std::min(lane_fit, at_once_waves) &&
                               all_tables <= kTableBytesAtOnce;
    // Lane waves in even rounds: as many waves as leave their rows in the caches most of the time
    // (16x16 maps, waves per compute unit: 4 actions, 524,288 envs 4: 4.8e10, 8: 6.2e10, 12: 5.7e10,
    // 16: 5.0e10; 8 actions, 262,144 envs 8: 3.7e10, 12: 4.2e10, 16: 4.0e10).
    const long per_round = kComputeUnits * (!outgrown ? 16L : e->A == 8 ? 12L : 8L);
    const long rounds = (lane_units + per_round - 1) / per_round;
    // Hybrid workgroups take a while to share out their envs, and their last table waves are late: they pay
    // over rounds of lane waves once a table's steps are worth its way into LDS and there is enough to step
    // (lane waves / hybrid, us; launch after launch, from the first on):
    //   8x8, 4 actions: 1M envs, 16 / 32 / 64 steps 433 / 703 / 938, 405 / 571 / 776; 200,000, 64 / 96 179 / 190, 249 / 236
    //   up to 6 KB, 4 actions: 150,000 of 12x12, 96 / 131 235 / 305, 247 / 294; 200,000, 64 / 96 273 / 380, 261 / 325;
    //     150,000 of 16x16, 96 / 131 329 / 440, 325 / 377; 140,000, 160 520, 420; 180,000, 96 / 131 409 / 498, 413 / 482;
    //     8 actions, six rounds and more: 130,000 of 8x8, 96 / 131 246 / 327, 262 / 321; 200,000 96 / 131 380 / 491, 362 /
    //     445; 150,000 of 12x12, 96 / 131 394 / 494, 388 / 462; five rounds: 110,000 of 12x12, 131 / 220 327 / 507, 394 / 552
    //   larger, 4 actions: 150,000 of 20x20, 131 / 170 485 / 652, 557 / 654; 110,000 of 25x20, 170 / 220 480 / 643, 547 / 642
    //   8 actions, two LDS waves: 150,000 of 16x16, 131 / 170 / 220 639 / 739 / 871, 657 / 752 / 872; 220,000, 131 / 170
    //     865 / 1141, 991 / 1138; one, five rounds and more: 100,000 of 24x12, 64 / 96 / 131 / 220 228 / 326 / 435 / 699,
    //     226 / 314 / 412 / 648; 150,000, 64 / 96 / 131 340 / 484 / 643, 370 / 459 / 592; 110,000 of 23x23, 96 / 131 / 300 380 /
    //     503 / 1075, 380 / 491 / 996; four rounds: 80,000 of 19x18, 131 / 200 362 / 534, 413 / 585
    //   four rounds of 8 actions from 20 million env-steps on: 94,000 of 19x12, 200 / 440 steps 546 / 1128, 520 / 892;
    //     98,000 of 9x9, 256 steps 420, 404
    // Where the lane waves have at most three rounds they are late by less, and the larger a table the sooner
    // hybrid workgroups pay: 95,000 of 12x12, 256 / 500 steps 322 / 546, 316 / 541, of 16x16 429, 375; 73,000 of 26x18, 256 /
    // 367 steps 465 / 657, 465 / 602; 80,000 of 20x20, 200 / 256 steps 379 / 477, 383 / 450; 8 actions, 73,000 of 12x12, 500 /
    // 1000 steps 644 / 1189, 722 / 1354, of 16x16 960 / 1729, 898 / 1574; 70,000 of 19x12, 440 steps 782, 745.
    const bool few_rounds = rounds <= 3;
    const int few_rounds_min_steps = e->A == 8 ? (e->K >= 1536 ? 400 : INT_MAX) : e->K >= 1024 ? 256 : kHybridFewRoundsMinSteps;
    const bool hybrid_pays =
        few_rounds ? n_steps >= few_rounds_min_steps
        : e->A == 8 && p.lds_waves == 1 && rounds > 4
            ? n_steps >= kHybridOneWaveMinSteps
            : 64L * n_steps >= 5L * (long)e->K &&
                  (long)e->N * n_steps >= (e->K < 512 || (e->K < 1536 && (e->A == 4 || rounds > 5)) ? kHybridEnvStepsSmall
                                           : e->A == 4                                              ? kHybridEnvSteps4
                                           : rounds > 4                                             ? kHybridEnvSteps8
                                                                                                    : kHybridEnvSteps8FewRounds);
    // 64-env waves that keep rows in LDS (run_env_rows), in place of all others (us, the other plan / these; launch after launch):
    //   64-env waves: 1M envs of 16x16, 3 / 6 / 10 / 20 / 32 steps 166 / 272 / 378 / 627 / 910, 108 / 178 / 245 / 369 / 500;
    //     262,144 of 32x32, 8 / 80 steps 93 / 628, 58 / 405; of 22x22 with 8 actions, 8 steps 105, 69; of 48x40 3 / 200 steps
    //     86 / 1477, 44 / 1011; 1M of 5x5, 1 / 8 steps 64 / 268, 63 / 133; 20,000 of 16x16, 1 / 4 steps 12.7 / 10.3, 7.9 / 9.8
    //   rounds of lane waves: 1M of 16x16, 64 steps 1571, 890; 262,144 of 32x32, 250 / 800 steps 1541 / 4450, 1185 / 3777; of 16x16 with 8
    //     actions, 150 steps 1183, 859; 300,000 of 4x4 with 8 actions, 8 / 60 steps 68 / 298, 40 / 172
    //     (floored maximum, however long with 4 actions: 90,000 of 16x16, 5 / 100 / 400 steps 28 / 175 / 625, 16 / 132 / 472; of 9x9 100 / 400
    //     112 / 402, 114 / 416; 130,000 of 12x12, 1000 steps 1604, 1125; 300,000 of 16x16, 200 / 1000 steps 1068 / 4350, 856 / 3913;
    //     8 actions: 130,000 of 14x14, 100 / 1000 steps 433 / 2636, 256 / 2266; 200,000 400 / 700 steps 1793 / 2849, 1679 / 2968, of 20x20 1000
    //     steps 5194, 4589; epsilon by episode, where envs explore, up to 500 steps: 300,000 of 16x16, 350 / 500 / 1000 1863 / 2575 /
    //     4949, 1722 / 2491 / 5315; 600,000 of 9x9, 300 / 1000 2696 / 7291, 2285 / 8516; 300,000 of 30x30, 1000 steps 6580, 6034;
    //     115,000 of 9x9, 20 / 60 steps 38 / 98, 41 / 104; 160,000 of 5x5 51 / 127, 45 / 110)
    //   hybrid workgroups, up to a length that grows with the table:
    //     1M of 8x8, 40 / 80 / 150 steps 697 / 939 / 1439, 438 / 780 / 1410; 400,000 of 12x12, 130 / 180 / 250 720 / 872 / 1127,
    //     621 / 852 / 1159; 1M of 16x16, 80 / 150 / 330 / 400 1892 / 2533 / 4227 / 4861, 1000 / 1907 / 4120 / 5027; 300,000 of 20x20,
    //     400 / 800 2156 / 3729, 1736 / 3506; 8 actions: 600,000 of 8x8, 100 / 170 1074 / 1575, 784 / 1283; 500,000 of 12x12, 160 / 200
    //     1616 / 1911, 1411 / 1744; 230,000 of 12x12 with 4, 150 / 180 451 / 508, 451 / 538; of 16x16, 250 / 300 869 / 975, 815 / 985; 300,000 of 16x16, 300 / 400 / 500 2011 / 2428 / 2854, 1806 / 2431 / 3091; 262,144 of 22x22, 600 4262, 3805
    //   fewer envs, lane waves in two rounds and more: 99,000 of 9x8, 16 / 50 / 80 steps 29 / 68 / 99, 27 / 62 / 91; of 12x12, 30 / 80
    //     69 / 151, 47 / 94; 200,000 of 5x4, 16 / 50 46 / 113, 37 / 110; of 15x15, 50 / 80 270 / 402, 175 / 261; 8 actions: 99,000 of 4x4,
    //     8 / 50 28 / 102, 18 / 71; 130,000 of 9x9, 30 / 80 120 / 232, 79 / 140; 260,000 of 7x7, 16 / 80 141 / 435, 83 / 279
    // With fewer envs still a step is as long as its slowest request and lane waves have fewer of those (50,000 of 16x16, 20 steps
    // 26.6, 33.3).  Not all of these lines lie where the two sides cross: 200,001 to 262,143 envs with tables of up to 256 values, up to
    // 200,000 on maps of up to 336 cells past 88 steps (at 80 steps rows are still 1.5 times as fast), and on larger ones below 11 and
    // above 130, keep the other plans although their neighbours in size are the faster ones with rows.
    const bool rows_can = lanes_rules(e) && c.max_episodes == 0 && c.track_returns == 0 && c.eps_mode != CRL_EPS_STEP_MULT &&
                          e->mv_words > 0 && e->resident_envs == 0 && e->fused_variant != 2;
    const size_t rows_lds4 = map_lds + crl::RowCache<4, false, 4>::kBytes;
    const bool rows_staged = lds_fit(rows_lds4) >= (e->A == 8 ? kRowsStagedWaves8 : kRowsStagedWaves4);
    const bool cells = c.reward_flags != 0, rows_rich = c.eps_mode != CRL_EPS_FIXED || cells;
    // (rewards per cell: lane waves, which take over from plain ones at 131 steps, are the faster ones then on most tables, the more so where
    // envs wander; lane waves / rows: rewards of goals and traps only, epsilon fixed, 357,632 of 4x12, 245 steps 1157, 2299; 910,400 of 4x17, 182
    // steps 2470, 4554; 247,808 of 24x5, 339 steps 1558, 2393; 8 actions, 278,651 of 10x33, 324 steps 2931, 3284; rewards of all cells, epsilon by
    // episode, 8 actions, 597,376 of 29x4, 197 steps 3306, 3499.  Rows go on on the smallest maps (974,336 of 5x3, 254 steps 3161, 1683; 682,624,
    // epsilon fixed, 308 steps 2040, 1310; 578,368 of 5x5 with 8 actions, 312 steps 2688, 2136); with 4 actions on 256 cells and more whose maps are staged (1.05 to 1.2
    // times as fast; not where codes come with the rows, 236,650 of 37x30, epsilon by episode, 532 steps 3837, 4715, unless lane waves have no even rounds
    // either, 104,006 of 61x33, floored maximum, 320 steps 1652 by the general loop, 1147; 8 actions, epsilon by episode, 296,064 of 13x30, 134 steps 1510, 1396, past 240 0.96 times); with rewards of all cells and
    // epsilon fixed (417,152 of 22x6, 363 steps 2197, 1597; 889,344 of 5x16 with 8 actions, 182 steps 3220, 2704; 896,384 of 15x3, 252 steps 2772,
    // 1980; not all of 30 to 100 cells, 229,376 of 4x20, 273 steps 823, 976); for a while with 4 actions, epsilon by episode, on 100 and more (861,017 of 30x8, 178 steps
    // 4179, 3594; 362,432 of 24x5, 230 steps 1860, 1676).)
    const bool base_cells = (c.reward_flags & CRL_REWARD_BASE_CELLS) != 0;
    // (the smallest maps with rewards of all cells, 4 actions, epsilon by episode, 20 to 300 steps, rows so many times as fast as lane waves: 26 cells,
    // 270,001 / 360,001 / 520,001 envs 0.98 to 1.06 / 1.09 to 1.17 / 1.3 and more; 27, 270,001 / 360,001 / 430,001 0.82 to 0.93 / 0.94 to 1.07 / 1.00 to
    // 1.15; 28, 0.90 to 1.07 / 1.00 to 1.14 / 1.08 to 1.28; 30 cells 0.77 to 0.85 / 0.90 to 1.00, 390,001 0.92 to 1.06.)
    const bool smallest = e->S <= kRowsRewardsSmallest ||
                          (e->A == 4 && base_cells && (e->S <= kRowsRewardsSmaller || (e->S <= kRowsRewardsSmall && (long)e->N > kRowsRewardsSmallEnvs)));
    const bool cells_long = smallest || (e->A == 4 && e->S >= kRowsRewardsLarge && rows_staged) || (base_cells && !by_episode) ||
                            kComputeUnits * lane_fit < per_round;  // (no even rounds)
    // (while the caches hold the tables lane waves take over from plain ones from 8 steps on, and are the faster ones then with 4 actions but on
    // the smallest maps; lane waves / rows, launches of 262,144 envs and more: rewards of goals and traps, 270,845 of 5x9, epsilon by episode,
    // 47 steps 217, 332; 274,286 of 5x9, 15 steps 78, 118; 298,062 of 2x20, by episode, 8 steps 50, 65; 422,354 of 3x9, 75 steps 425, 524;
    // 371,959 of 2x13, 96 steps 458, 559; but 408,508 of 3x4, by episode, 60 steps 290, 222; rewards of all cells, by episode, 336,159 of 4x8, 28
    // steps 152, 199; 274,212 of 6x7, 9 steps 53, 72; with epsilon fixed 281,012 of 6x6, 38 steps 149, 113; in calls that plain waves
    // would take, 312,999 of 3x9, 2 steps 33.7, 30.6.)
    const bool cells_cached = e->A == 4 && !outgrown && e->N >= kRowsManyEnvs && !smallest;
    const int cells_steps = cells_cached                                    ? kLaneWavesMinSteps - 1
                            : !by_episode || !rows_staged                   ? kLaneRoundsManyMinSteps - 1
                            : e->S >= kRowsRewardsLarge                     ? kRowsRewardsLargeSteps
                            : e->A == 4 && e->S >= kRowsRewardsMiddle       ? kRowsRewardsMiddleSteps
                                                                            : kLaneRoundsManyMinSteps - 1;
    const int rows_steps = fits && p.fast ? (e->A == 8 ? kRowsHybridSteps8 + (int)(e->K / 8) : kRowsHybridSteps4 + (int)(3 * e->K / 16))
                           : cells && !cells_long   ? cells_steps
                           : e->A == 8 || rows_rich ? std::max(kRowsLanesSteps, (int)(e->K / 3))
                                                    : INT_MAX;
    const bool rows_small = e->S <= kRowsSmallMap;
    const bool rows_many = e->N >= kRowsManyEnvs || (e->N > kRowsManyLargerTables && e->K > 256);
    const bool rows_some = foldable && !lanes_at_once && n_steps <= kRowsSomeEnvsSteps && (rows_small || n_steps >= kRowsLargeMapMinSteps) &&
                           (e->N > kRowsSomeEnvs ? e->N <= kRowsManyLargerTables && (!rows_rich || e->A == 8 || e->K >= 512 || e->N > kRowsSomeEnvsRich)
                                                 : (long)e->N > kLaneRoundsManyEnvs && e->K >= 640);
    const bool rows_floored = c.max_mode != CRL_MAX_TRUE && !lanes_at_once && (long)e->N > kLaneRoundsManyEnvs &&
                              e->K >= (e->N > kRowsSomeEnvs ? 257 : 640);
    // Up to three of them to a compute unit plain 64-env waves are faster (plain / rows: 40,960 of 8x8, 2 / 5 steps 7.1 / 9.0, 8.2 /
    // 11.1; 40,000 of 16x16 with 8 actions, 4 steps 12.0, 13.3; 40,960 of 32x32, 128 steps 141, 159; 24,576 of 40x40 with 8 actions 171,
    // 210; 44,866 of 4x38 with 8 actions, 43 steps 55, 68), and four in calls too short for a limit on the envs in flight (62,848 of
    // 4x4, 5 steps 9.9, 11.6; 49,984 of 8x8 with 8 actions, 6 steps 14.6, 16.6; 57,984 of 4x4, 3 steps 6.6, 8.0).  Rows are where
    //   plain waves go in shifts or their maps do not all fit LDS (56,000 envs and more, 16 steps and more 1.2 to 1.6 times as fast;
    //     35,968 of 64x64, 112 steps 203, 144);
    //   a map costs more to stage than the steps then save, some cells to a step: with two 64-env waves to a unit 80 (32,768 of 64x64, 20 /
    //     32 / 50 steps 41.3 / 52.1 / 70.2, 31.9 / 48.0 / 72.5; 30,000 of 48x48, 16 / 32 steps 30.5 / 45.0, 26.7 / 48.6), with three 60 while
    //     envs explore and 40 with epsilon fixed (40,960 of 32x32, 12 / 16 / 64 steps 24.1 / 28.0 / 83.1, 21.1 / 26.3 / 83.5); 8 actions 80
    //     and 96 (24,576 of 40x40, 16 / 20 steps 28.5 / 37.7, 27.9 / 36.5); not where the maps are staged for rows too (17,042 of 20x55
    //     with 8 actions, 11 steps 23.0, 27.0);
    //   epsilon is fixed: more than three, tables past the caches, from three steps on (65,536 of 16x16, 4 steps 14.2, 12.9; 61,803 of 42x7
    //     with 8 actions 15.5, 14.7); more than 2.75, large maps (48,000 of 32x32, 20 / 64 / 100 steps 35.5 / 99.5 / 136, 33.5 / 88.7 / 135; 8
    //     actions up to 1300 cells: 46,298 of 46x36, 125 steps 222, 253);
    //   cells have rewards, whatever epsilon: the same with more than three waves, on large maps with more than 2.5 (45,825 of 57x44 with 8
    //     actions, 32 steps 70, 52; 48,448 of 58x28, epsilon by episode, 74 steps 152, 126), and with more than two 32 and 16 cells to a step (41,216
    //     of 32x59, 64 steps 92.1, 82.5; 33,904 of 49x30 with 8 actions, 20 steps 38.2, 31.7).
    const bool two_waves = (long)e->N <= 2L * 64 * kComputeUnits;
    const long rows_cells = cells && !two_waves ? (e->A == 8 ? kRowsCells8Rewards : kRowsCells4Rewards)
                            : e->A == 8         ? (rows_rich ? kRowsCells8Rich : kRowsCells8)
                            : two_waves         ? kRowsCells4
                            : rows_rich         ? kRowsCells4Rich
                                                : kRowsCells4Fixed;
    // More envs than are at work at once, 4 actions, staged maps of more than 336 cells: not a call of one step (plain / rows: 262,144 of
    // 16x32 25.2, 27.9; 315,185 of 33x18 31.8, 38.0; 252,160 of 20x40 29.4, 34.4; 524,288 of 20x20 39.6, 39.4; 258,311 of 12x48, epsilon by
    // episode, 26.6, 30.5; with 8 actions 254,259 of 26x15 24.0, 24.1, 303,488 of 7x54 28.2, 27.0), on more than 600 while envs explore
    // nor one of two (274,538 of 24x26 39.4, 44.4; 339,243 of 16x46 48.4, 52.4; but 281,664 of 24x24 38.5, 37.1).  Where codes come with the
    // rows they pay at once (256,271 of 40x24, one step 38.8, 23.6), and in place of the general loop (505,664 of 29x13 39.6, 37.5).
    const int rows_from = e->A == 8 || cells || !foldable || !rows_staged || rows_small || e->N <= kRowsManyLargerTables ? 1
                          : rows_rich && e->S > kRowsTwoStepsMap                                                 ? 3
                                                                                                                 : 2;
    const bool rows_pay = n_steps >= rows_from && ((long)e->N > 4L * 64 * kComputeUnits || resident < e->N || ((long)e->N + 63) / 64 > kComputeUnits * lds_fit(map_lds) ||
                          (!rows_staged && n_steps >= kRowsLargeMapMinSteps && (long)e->S >= n_steps * rows_cells) ||
                          ((!rows_rich || cells) && outgrown && (long)e->N > kMinEnvsInFlight && n_steps >= kRowsFixedMinSteps) ||
                          ((!rows_rich || cells) && (long)e->N > (cells ? kRowsRewardsEnvs : kRowsFixedEnvs) && !rows_small &&
                           (e->A == 4 || cells || e->S <= kRowsFixedMap8)));
    // Floored maximum, 4 actions: rounds of lane waves stay (us, these / rows)
    //   epsilon by episode, tables that the caches hold and not two full rounds: 100,000 of 10x10, 100 / 400 steps 150 / 537, 157 / 580;
    //     102,577 of 17x4, 211 steps 254, 289; 106,471 of 6x12, 72 steps 103, 111; 117,792 of 13x8, 48 steps 100, 93;
    //   epsilon by episode, tables past them, long calls, where up to a quarter more waves with rows than are at work at once would begin
    //     when the others are through: 200,882 of 11x19 (12.3 to a unit, 12 fit), 315 steps 1175, 1317; 213,000 of 14x15, 358 steps 1317, 1421;
    //     172,032 of 22x20, 464 steps 1633, 1831; not with as many as fit (208,724 of 22x7, 265 steps 968, 778), smaller maps, of which
    //     more than twelve fit (305,000 of 20x4, 17.3 and 16 to a unit, 455 steps 1887, 1530) or shorter calls (240,442 of 17x11, 131 steps 652, 599);
    //   epsilon fixed, the smallest tables: 300,000 of 3x3, 20 / 100 / 400 / 1000 steps 66 / 250 / 935 / 2356, 55 / 254 / 977 / 2410; 376,832 of 2x3,
    //     197 steps 530, 584; of 4x4 400 steps 982, 991; 358,000 of 3x5, 151 steps 469, 436; 563,274 of 4x3, 850 steps 3816, 3357.
    const long rows_waves = ((long)e->N + 63) / 64, rows_at_once = kComputeUnits * lds_fit(rows_lds4);
    const bool rows_late = c.max_mode != CRL_MAX_TRUE && e->A == 4 &&
                           (!by_episode ? !outgrown && rounds <= 6 && e->K <= kRowsSmallestTables && n_steps >= kRowsSmallestTablesSteps
                            : outgrown  ? rows_staged && rows_at_once <= kRowsLateWaves * kComputeUnits && rows_waves > rows_at_once &&
                                             4 * rows_waves <= 5 * rows_at_once && n_steps >= kRowsLateSteps
                                        : lane_units <= kRowsTwoRoundsWaves * kComputeUnits && n_steps >= kRowsTwoRoundsSteps);
    const bool rows_first = rows_can && rows_pay && !rows_late && e->fused_variant == 0 && (((rows_many || rows_floored) && n_steps <= rows_steps) || rows_some);
    // ... hybrid workgroups (automatic) when the tables outgrow the caches: while they all fit, other plans are
    // faster (16x16 maps, 30,000 envs: 3.5e10 hybrid, 5.9e10 with lane waves); and where lane
    // waves could step what is left to the general loop, they are faster too (262,144 envs of
    // 16x16 with a zero-floored maximum: 5.1e10 general hybrid, 6.4e10)
    p.hybrid = fits && !rows_first && (e->fused_variant == 2 ||
                        (e->fused_variant == 0 && outgrown &&
                         (lanes_can && e->resident_envs == 0 ? p.fast && !lanes_at_once && hybrid_pays
                                                             : (!lanes_can || p.fast) && n_steps >= kHybridMinSteps)));
    if (p.hybrid) {
      p.grid = (int)std::min<long>(kComputeUnits, (tickets + 8) / 9);
      p.block = 64 * (hbm_waves + p.lds_waves);
    } else {
      long waves = 4, workers;  // waves per workgroup, 64-env workers in flight
      if (tickets / 2 < 4 * kComputeUnits) {
        // fewer 64-env workers than SIMDs on the chip: one-wave workgroups spread
        // them over the compute units instead of packing four per unit
        // (all envs in flight: a wave for the last, part-filled 64 as well.  Left over, these envs began when others were through:
        // 19,895 of 40x40 with 8 actions, one step 21.1 us, 12.4; 23,081 of 24x24, 5 steps 20.0, 12.6; 58,545 of 20x20, 3 steps 17.6, 12.5)
        waves = 1;
        workers = std::min<long>(std::max<long>(1, e->resident_envs > 0 ? resident / 64 : (resident + 63) / 64), (tickets + 1) / 2);
      } else if (resident <= 4L * 64 * kComputeUnits) {
        // at most four waves per compute unit: spread them over all units
        waves = std::max<long>(1, resident / (64L * kComputeUnits));
        workers = waves * std::min<long>(kComputeUnits, (tickets + 2 * waves - 1) / (2 * waves));
      } else {
        workers = 4 * std::min<long>(std::max<long>(1, resident / 256), (tickets + 7) / 8);
      }
      // every wave stages the maps of its 64 envs in its own LDS slice: large maps
      // leave room for fewer waves per workgroup (one always fits: map_kind 0
      // means 64 maps take at most 64 KB), the workers in flight stay the same
      while (waves > 1 && (size_t)waves * map_lds > kLdsPerWorkgroup) --waves;
      p.grid = (int)((workers + waves - 1) / waves);
      p.block = 64 * (int)waves;
      // staging the codes (four times the class map) pays off over a long launch only (1M envs of
      // 16x16, one step per launch 7.7e9 -> 1.4e10 with class maps, 48 steps 3.6e10 -> 3.7e10), and not
      // where fewer of the workgroups fit a compute unit for it (34,000 of 32x32, 128 steps: 193, 120 us)
      p.moves = p.fast && (size_t)((p.grid + kComputeUnits - 1) / kComputeUnits) * waves * mv_lds <= kLdsPerWorkgroup &&
                n_steps >= kStagedMovesMinSteps;
      // Few envs: A lanes to each, in as many waves as leave no more than two to a SIMD.  More:
      // all at once in lane waves, in place of the folded loop for launches of some steps (30,000
      // envs of 16x16, 4 / 8 / 16 steps: 23 / 28 / 35 us, 23 / 26 / 28), of the general loop always
      // (30,000 of 16x16, one step: 12.5 us, 8.9; in rounds 200,000, 2 / 6 steps: 34 / 75, 50 / 74).
      // Else lane waves in rounds (not with fewer of them because the codes take too much LDS:
      // 50,000 envs of 48x48, 4 waves: 643 / 700 us): always soon where the tables do not outgrow the
      // caches or the general loop is the other choice.  Where they do, 64-env / lane waves:
      //   tables that hybrid workgroups could take, 16 / 48 steps: 1M of 16x16 468 / 1246, 494 / 1177 us;
      //     70,000 with 8 actions 47.6 / 117, 47.9 / 103; the smaller the sooner: 130,000 of 12x12, 24
      //     steps 67.0, 64.8; 200,000 of 8x8, 8 / 16 steps 51.6 / 70.6, 44.1 / 64.3; with few rounds later:
      //     94,000 of 12x12, three, 32 / 48 steps 50.9 / 72.3, 53.6 / 72.7
      //   others, 32 / 64 / 96 steps: 52,000 of 32x32 61 / 114 / 160, 57 / 98 / 139; 40,000 of 24x24 with
      //     8 actions 49 / 100 / 142, 57 / 97 / 136; 100,000 of 32x32 123 / 229 / 333, 119 / 206 / 291 (the
      //     larger batches keep their 64-env waves up to 130 steps, a length that their tests hold them to)
      //   8 actions, not more than two waves of 64 envs to a compute unit: 64-env waves always, 25,161 of 28x46, 64 / 164 / 800
      //     steps 78 / 168 / 739, 96 / 211 / 922; 30,000 of 24x24 78 / 173 / 711, 87 / 191 / 856; 32,000 of 28x28 85 / 180 / 804, 94 /
      //     214 / 933; epsilon by episode, 400 steps 480 / 482 / 504, 501 / 473 / 512
      //   4 actions, not more than three waves of 64 envs to a compute unit: 64-env waves always, 34,000 of
      //     32x32, 128 / 1000 steps 120 / 727, 146 / 908; 49,000 176 / 1235, 174 / 1240
      const bool small = waves == 1 && tickets <= 2 * kComputeUnits;
      const long lane_waves = small || lanes_at_once ? lane_units : (lane_units + rounds - 1) / rounds;
      const int at_once_min_steps = p.fast ? kLaneWavesMinSteps : 1;
      const int rounds_min_steps = !(p.fast && outgrown)                             ? kLaneWavesMinSteps
                                   : fits && e->fused_variant == 0                   ? (few_rounds ? kLaneFewRoundsMinSteps : (int)std::min<size_t>(40, std::max<size_t>(kLaneWavesMinSteps, e->K / 24)))
                                   : e->A == 4 && (long)e->N <= kMinEnvsInFlight     ? INT_MAX
                                   : e->A == 8 && (long)e->N <= 2L * 64 * kComputeUnits ? INT_MAX
                                   : (long)e->N <= kLaneRoundsManyEnvs               ? kLaneRoundsMinSteps
                                                                                     : kLaneRoundsManyMinSteps;
      // Even rounds of one wave more to a compute unit than fits: as many as fit draw their envs instead (dealt by
      // position, the late ones run after all others; 67,000 envs of 45x19 with 8 actions, floored maximum, 64 / 131 / 200
      // / 425 steps late and dealt 264 / 495 / 721 / 1038, as many as fit 220 / 366 / 514 / 994; 100,000 of 40x40, 131 steps 652,
      // 441).  With up to three 64-env waves to a unit those are faster, also by the general loop (39,537 of 47x42, floored
      // maximum, 64 / 438 steps 101 / 492, 141 / 676; 45,000 of 45x19 with 8 actions 127 / 693, 162 / 743), and so they are in
      // short launches (67,045 of 40x47, 9 steps 57, 66).  In place of the folded loop in long launches only: 67,000 of 45x19, 131
      // steps 64-env / lane waves 374 / 366, 100,000 of 36x26 566 / 548, but 80,000 of 45x21 404 / 453 and at 200 601 / 641;
      // 45,000 of 45x19, fewer than three 64-env waves to a unit, 131 / 400 / 800 steps 227 / 594 / 1175, 261 / 720 / 1270;
      // 150,000, seven rounds, 131 / 200 / 425 752 / 1111 / 2231, 742 / 1065 / 2121.
      const bool uneven = !small && !lanes_at_once && lane_waves > kComputeUnits * lane_fit;
      const bool uneven_pay = !p.fast ? (long)e->N > kMinEnvsInFlight && n_steps >= kHybridMinSteps : (outgrown && (long)e->N > kLaneRoundsManyEnvs &&
                                          n_steps >= (rounds > 6 ? kLaneUnevenManyRoundsMinSteps : kLaneUnevenMinSteps));
      const bool rounds_ok = (!uneven || (uneven_pay && lane_waves <= kComputeUnits * (lane_fit + 1))) && n_steps >= rounds_min_steps;
      if (lanes_can && !rows_first && (small ? lane_fit > 0 : lanes_at_once ? n_steps >= at_once_min_steps : rounds_ok)) {
        p.fast = p.moves = p.lanes = true;
        p.rich = c.eps_mode >= CRL_EPS_EPISODE_MULT || c.reward_flags != 0;
        p.log_envs = lane_log_envs;
        p.tape_steps = tape_steps_for(lane_log_envs);
        const long most = e->resident_envs > 0 ? std::max<long>(1, resident >> lane_log_envs)
                          : uneven               ? kComputeUnits * lane_fit
                                                 : lane_waves;
        p.grid = (int)std::min<long>(lane_units, most);
        p.block = 64;
        const bool many_rounds = p.grid * 5L < lane_units;
        // (the tables' lines asked for ahead: 300,000 of 16x16, 64 / 96 / 200 / 1000 steps 531 / 682 /
        // 1196 / 4774 us with, 483 / 701 / 1346 / 5276 without; 200,000 with 8 actions, 128 / 200 steps 841 /
        // 1142, 808 / 1179; 198,000 of
        // 10x30, seven rounds, 757 steps 2375, 2740; 120,000 of 16x16, four rounds, 200 / 1000 steps 488 / 1910,
        // 373 / 1706.  In four or five rounds where envs explore for long, epsilon by episode, tables of 4 KB on, with /
        // without: 150,000 of 16x16, 131 / 200 / 329 / 700 steps 430 / 590 / 903 / 1804, 451 / 677 / 1075 / 2143; 149,286 of
        // 27x11, 700 steps 1831, 2165; 110,000 of 21x21, 131 / 200 / 329 413 / 546 / 803, 368 / 545 / 875; 90,000 of 16x16 with 8
        // actions 381 / 544 / 812, 384 / 569 / 901; not of 12x12: 4 actions 700 steps 1662, 1675, 8 actions 200 steps 472, 422)
        const bool explores = by_episode && e->K >= (e->A == 8 ? 1536 : 1024) && 8L * n_steps >= (long)e->K &&
                              n_steps >= kLaneTouchFourRoundsMinSteps && p.grid * 3L < lane_units;
        p.touch = outgrown && e->K <= (size_t)crl::kTouchFloats &&
                  (explores || (many_rounds && n_steps >= (e->A == 8 ? kLaneTouchMinSteps8 : kLaneTouchMinSteps4)));
        // (no more than it uses, also where there is a compute unit for every workgroup: 4096 envs
        // of 32x32, 10,000 steps, 17 / 64 / 81 KB 2.78 / 2.76 / 2.80 ms)
        p.lds = lane_lds;
      }
      // Envs dealt by position instead of drawn from a counter: 16,384 draws take 0.38 ms however short
      // the launch (1M envs: the whole of a 4-step launch, half of a 20-step one).  Lane waves, drawn /
      // dealt: 120,000 envs of 8x8, two rounds, 128 / 1000 steps 207 / 1315, 176 / 1268 us; 140,000 of 6x6
      // with 8 actions, five rounds, 128 / 300 / 1000 steps 290 / 563 / 1654, 279 / 609 / 1912; 300,000
      // of 16x16, ten rounds, 128 / 300 steps 868 / 1523, 879 / 1585; 891,000 of 20x14, 150 steps 2503, 2705.
      const bool drawn_lanes = uneven ? true
                               : n_steps >= kLaneDrawnMinSteps ? e->A == 8 || p.grid * 3L < lane_units
                                                             : n_steps >= kLaneDrawnManyMinSteps && p.grid * 5L < lane_units;
      p.fixed = p.lanes ? p.grid >= lane_units || !drawn_lanes : n_steps < kHybridMinSteps;
      if (!p.lanes) p.lds = waves * (p.moves ? mv_lds : map_lds);
      // No more of these than rows_first, or where they are the choice that is left: waves that keep rows instead (as many
      // as there are envs for, a workgroup each).
      if (rows_first || (!p.lanes && rows_can && foldable && rows_pay &&
                         (rows_small || (n_steps >= kRowsLargeMapMinSteps && n_steps <= kRowsLargeMapMaxSteps)))) {
        p.fast = p.fixed = true;
        p.rich = rows_rich;
        const size_t staged6 = map_lds + crl::RowCache<4, false, 6>::kBytes;
        const long fit6 = lds_fit(staged6);
        if (!p.rich && (fit6 >= kRowsSixSoonWaves ? n_steps >= kRowsSixSoonSteps : fit6 >= kRowsSixWaves && n_steps >= kRowsSixSteps)) {
          p.rows = 6;
          p.moves = false;
          p.lds = staged6;
        } else {
          p.rows = 4;
          p.moves = !rows_staged;
          p.lds = p.moves ? crl::RowCache<4, true, 4>::kBytes : rows_lds4;
        }
        p.block = 64;
        p.grid = (int)(((long)e->N + 63) / 64);
      }
    }
  }
  // (as launch_fused_a() picks the kernel)
  static const char* names[2][3][3] = {
      {{"k_fused_per_env<4,0>", "k_fused_per_env<4,1,general>", "k_fused_per_env<4,2,general>"},
       {"k_fused_per_env<4,0>", "k_fused_per_env<4,1,fast>", "k_fused_per_env<4,2,fast>"},
       {"k_fused_per_env<4,0>", "k_fused_per_env<4,1,fast,lanes>", "k_fused_per_env<4,2,fast,lanes>"}},
      {{"k_fused_per_env<8,0>", "k_fused_per_env<8,1,general>", "k_fused_per_env<8,2,general>"},
       {"k_fused_per_env<8,0>", "k_fused_per_env<8,1,fast>", "k_fused_per_env<8,2,fast>"},
       {"k_fused_per_env<8,0>", "k_fused_per_env<8,1,fast,lanes>", "k_fused_per_env<8,2,fast,lanes>"}}};
  p.name = names[e->A == 8][!p.fast ? 0 : p.lanes ? 2 : 1][p.map_kind];
  if (p.tickets) {
    static const char* tnames[2][3][2] = {
        {{"k_fused_tickets<4,general,hbm>", "k_fused_tickets<4,general,hbm+lds>"},
         {"k_fused_tickets<4,fast,hbm>", "k_fused_tickets<4,fast,hbm+lds>"},
         {"k_fused_tickets<4,fast+,hbm>", "k_fused_tickets<4,fast+,hbm>"}},
        {{"k_fused_tickets<8,general,hbm>", "k_fused_tickets<8,general,hbm+lds>"},
         {"k_fused_tickets<8,fast,hbm>", "k_fused_tickets<8,fast,hbm+lds>"},
         {"k_fused_tickets<8,fast+,hbm>", "k_fused_tickets<8,fast+,hbm>"}}};
    static const char* lnames[2][2] = {{"k_fused_lanes<4,fast>", "k_fused_lanes<4,fast,cells>"},
                                       {"k_fused_lanes<8,fast>", "k_fused_lanes<8,fast,cells>"}};
    p.name = p.lanes ? lnames[e->A == 8][(c.reward_flags & CRL_REWARD_CELLS) != 0]
                     : tnames[e->A == 8][p.rich ? 2 : p.fast ? 1 : 0][p.hybrid];
  }
  return p;
}

template <int A>
void launch_fused_a(const crl_engine* e, const FusedPlan& p, uint64_t t0, int n) {
  const crl::Rules R = e->rules();
  const crl::Ptrs P = e->ptrs();
  if (p.in_lds) {
    const int events = crl::lane_events(R, P);
#define CRL_LAUNCH_LDS(KERN)                                                                                              \
  do {                                                                                                                    \
    auto go = [&](auto kern) {                                                                                            \
      hipLaunchKernelGGL(kern, dim3(p.grid), dim3(64), p.lds, e->stream, R, P, t0, n, p.log_envs, p.env_bytes, p.tape_steps); \
    };                                                                                                                    \
    if (p.words) {                                                                                                        \
      if (events == crl::kNoEvents) go(crl::KERN<A, true, crl::kNoEvents>);                                               \
      else if (events == crl::kEpsilonEvents) go(crl::KERN<A, true, crl::kEpsilonEvents>);                                \
      else go(crl::KERN<A, true, crl::kAllEvents>);                                                                       \
    } else {                                                                                                              \
      if (events == crl::kNoEvents) go(crl::KERN<A, false, crl::kNoEvents>);                                              \
      else if (events == crl::kEpsilonEvents) go(crl::KERN<A, false, crl::kEpsilonEvents>);                               \
      else go(crl::KERN<A, false, crl::kAllEvents>);                                                                      \
    }                                                                                                                     \
  } while (0)
    if (p.map_kind == 1) CRL_LAUNCH_LDS(k_fused_per_env_lds);
    else CRL_LAUNCH_LDS(k_fused_tickets_lds);
#undef CRL_LAUNCH_LDS
    return;
  }
  if (p.tickets) {
    // (tickets dealt by position use no counter; the kernel itself notes who did how much, and
    // where it is kept: a launch to copy three words was 3 to 5 us of a call)
    if (!p.fixed) hipLaunchKernelGGL(crl::k_fill_u32, dim3(1), dim3(64), 0, e->stream, e->tk, 0u, 3);
    const dim3 g(p.grid), b(p.block);
    unsigned* tk = p.fixed ? e->split.p : e->tk;
#define CRL_LAUNCH_TICKETS(MODE, LDSW, MOVES)                                                       \
  hipLaunchKernelGGL((crl::k_fused_tickets<A, MODE, LDSW, MOVES, 0>), g, b, p.lds, e->stream, R, P, t0, n, \
                     tk, p.tab_stride, p.fixed ? 1 : 0, p.tape_steps, p.lds_waves, p.env_bytes)
#define CRL_LAUNCH_ROWS(MODE, MOVES, PLACES)                                                                                 \
  hipLaunchKernelGGL((crl::k_fused_tickets<A, MODE, false, MOVES, PLACES>), g, b, p.lds, e->stream, R, P, t0, n, tk, 0, 1, 0, 0, 0)
    const int events = crl::lane_events(R, P);
#define CRL_LAUNCH_LANES(CELLS)                                                                                            \
  do {                                                                                                                     \
    auto go = [&](auto kern) {                                                                                             \
      hipLaunchKernelGGL(kern, g, b, p.lds, e->stream, R, P, t0, n, tk, p.fixed ? 1 : 0, p.touch ? 1 : 0, p.log_envs, p.tape_steps); \
    };                                                                                                                     \
    if (events == crl::kNoEvents) go(crl::k_fused_lanes<A, CELLS, crl::kNoEvents>);                                        \
    else if (events == crl::kEpsilonEvents) go(crl::k_fused_lanes<A, CELLS, crl::kEpsilonEvents>);                         \
    else go(crl::k_fused_lanes<A, CELLS, crl::kAllEvents>);                                                                \
  } while (0)
    if (p.lanes && P.cell_reward)
      CRL_LAUNCH_LANES(true);
    else if (p.lanes)
      CRL_LAUNCH_LANES(false);
    else if (p.rows == 6)
      CRL_LAUNCH_ROWS(1, false, 6);
    else if (p.rows && p.rich && p.moves)
      CRL_LAUNCH_ROWS(2, true, 4);
    else if (p.rows && p.rich)
      CRL_LAUNCH_ROWS(2, false, 4);
    else if (p.rows && p.moves)
      CRL_LAUNCH_ROWS(1, true, 4);
    else if (p.rows)
      CRL_LAUNCH_ROWS(1, false, 4);
    else if (p.rich && p.moves)
      CRL_LAUNCH_TICKETS(2, false, true);
    else if (p.rich)
      CRL_LAUNCH_TICKETS(2, false, false);
    else if (p.fast && p.hybrid)
      CRL_LAUNCH_TICKETS(1, true, false);
    else if (p.fast && p.moves)
      CRL_LAUNCH_TICKETS(1, false, true);
    else if (p.fast)
      CRL_LAUNCH_TICKETS(1, false, false);
    else if (p.hybrid)
      CRL_LAUNCH_TICKETS(0, true, false);
    else
      CRL_LAUNCH_TICKETS(0, false, false);
#undef CRL_LAUNCH_TICKETS
#undef CRL_LAUNCH_ROWS
#undef CRL_LAUNCH_LANES
    return;
  }
#define CRL_LAUNCH_PER_ENV(MAP, MODE)                                                                 \
  hipLaunchKernelGGL((crl::k_fused_per_env<A, MAP, MODE>), dim3(p.grid), dim3(p.block),               \
                     MAP == 1 || MODE == 2 ? p.lds : 0, e->stream, R, P, t0, n, p.log_envs, p.tape_steps)
  const int mode = !p.fast ? 0 : p.lanes ? 2 : 1;
  if (p.map_kind == 1) {
    if (mode == 2) CRL_LAUNCH_PER_ENV(1, 2);
    else if (mode == 1) CRL_LAUNCH_PER_ENV(1, 1);
    else CRL_LAUNCH_PER_ENV(1, 0);
  } else {
    if (mode == 2) CRL_LAUNCH_PER_ENV(2, 2);
    else if (mode == 1) CRL_LAUNCH_PER_ENV(2, 1);
    else CRL_LAUNCH_PER_ENV(2, 0);
  }
#undef CRL_LAUNCH_PER_ENV
}

constexpr int kScanBlocks = 2;
// 8.4 million envs' cells for 256 owners, 524,288 envs' for 4096.  Two passes against the scan, us
// per step: 4 million envs of 16x16 310 / 36,300, 8 million 632 / 74,000, 140,000 envs of 1024x1024
// 179 / 5160, 500,000 668 / 18,000.
constexpr size_t kHandoffLimitBytes = (size_t)512 << 20;
constexpr size_t kNoAllocScanBytes = (size_t)128 << 20;

int ceil_log2(size_t v) {
  int b = 0;
  while (((size_t)1 << b) < v) ++b;
  return b;
}

int own_keys(const crl::ReduceGeom& G) {  // keys of the owner that has most
  const int rows = G.K >> G.a_shift;
  return ((rows + (1 << G.own_shift) - 1) >> G.own_shift) << G.a_shift;
}

// Owners of the two-launch reduction: 256, one per compute unit, also where the table has
// few keys for each (a block's 256 samples then fall into cells of a record or two, and the
// cells of 8 records are read 16 blocks at a time); more where an owner would have more keys
// than its LDS rows hold.
crl::ReduceGeom reduce_geom(const crl_engine* e, int n) {
  crl::ReduceGeom G{};
  G.K = (int)e->K;
  G.a_shift = e->A == 8 ? 3 : 2;
  G.n_blocks = (n + crl::kBlockSamples - 1) / crl::kBlockSamples;
  G.own_shift = crl::kPersistOwnShift;
  while (own_keys(G) > crl::kMaxOwnKeys) ++G.own_shift;
  G.cell_shift = crl::cell_shift_for(G.own_shift);
  G.main_shift = crl::main_shift_for(G.own_shift);
  return G;
}

size_t handoff_records(const crl::ReduceGeom& G) {
  return (((size_t)1 << G.own_shift) * (size_t)G.n_blocks) << G.cell_shift;
}

// Small tables need less room with as many owners as 64 keys each make: for a call whose
// hand-off cells have to fit into `limit` (4 million envs of 16x16: 581 us per step with 16 owners,
// 310 with 256).
crl::ReduceGeom reduce_geom_within(const crl_engine* e, int n, size_t limit) {
  crl::ReduceGeom G = reduce_geom(e, n);
  if (handoff_records(G) * sizeof(unsigned long long) <= limit || e->K > (size_t)crl::kDenseKeys) return G;
  G.own_shift = ceil_log2((e->K + crl::kOwnKeys - 1) / crl::kOwnKeys);
  G.cell_shift = crl::cell_shift_for(G.own_shift);
  G.main_shift = crl::main_shift_for(G.own_shift);
  return G;
}

// the two-pass reduction needs a bounded number of owners and a bounded hand-off buffer; and
// two blocks against a large table are scanned faster than their keys are handed over (10 steps
// of 256 / 512 / 1000 envs on 120x120 with 8 actions: 132 / 146 / 167 us, two passes 145 / 146 / 148)
bool reduce_fast(const crl::ReduceGeom& G) {
  if (G.n_blocks <= kScanBlocks && G.K > crl::kDenseKeys) return false;
  return 1 << G.own_shift <= crl::kMaxOwners && handoff_records(G) * sizeof(unsigned long long) <= kHandoffLimitBytes;
}

template <class Kern>
hipError_t allow_lds(Kern kern, size_t bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// kernels that use more than the default 64 KB of LDS per workgroup (gfx950 has 160 KB)
int opt_in_lds(crl_engine* e) {
  if (e->lds_opt_in) return CRL_OK;
  const size_t act = kLdsPerWorkgroup;  // what a launch asks for is checked against this
  HIP_TRY(allow_lds(crl::k_reduce_owners<false>, act));
  HIP_TRY(allow_lds(crl::k_reduce_owners<true>, act));
  HIP_TRY(allow_lds(crl::k_td_blocks<4, crl::PackedSamples>, act));
  HIP_TRY(allow_lds(crl::k_td_blocks<8, crl::PackedSamples>, act));
  HIP_TRY(allow_lds(crl::k_td_blocks<4, crl::Transition>, act));
  HIP_TRY(allow_lds(crl::k_td_blocks<8, crl::Transition>, act));
  HIP_TRY(allow_lds(crl::k_td_small<4, 4, crl::PackedSamples>, act));
  HIP_TRY(allow_lds(crl::k_td_small<8, 4, crl::PackedSamples>, act));
  HIP_TRY(allow_lds(crl::k_td_small<4, 4, crl::Transition>, act));
  HIP_TRY(allow_lds(crl::k_td_small<8, 4, crl::Transition>, act));
  HIP_TRY(allow_lds(crl::k_shared_act<4, 1, true>, act - kStaticLdsReserve));
  HIP_TRY(allow_lds(crl::k_shared_act<4, 2, true>, act - kStaticLdsReserve));
  HIP_TRY(allow_lds(crl::k_shared_act<8, 1, true>, act - kStaticLdsReserve));
  HIP_TRY(allow_lds(crl::k_shared_act<8, 2, true>, act - kStaticLdsReserve));
#define CRL_ALLOW_PERSIST(A, MAP)                                                                       \
  do {                                                                                                  \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, false, false, false>, act - kStaticLdsReserve));    \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, false, true, false>, act - kStaticLdsReserve));     \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, true, false, false>, act - kStaticLdsReserve));     \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, true, true, false>, act - kStaticLdsReserve));      \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, false, false, true>, act - kStaticLdsReserve));     \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, false, true, true>, act - kStaticLdsReserve));      \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, true, false, true>, act - kStaticLdsReserve));      \
    HIP_TRY(allow_lds(crl::k_shared_persist<A, MAP, true, true, true>, act - kStaticLdsReserve));       \
  } while (0)
  CRL_ALLOW_PERSIST(4, 1);
  CRL_ALLOW_PERSIST(4, 2);
  CRL_ALLOW_PERSIST(8, 1);
  CRL_ALLOW_PERSIST(8, 2);
#undef CRL_ALLOW_PERSIST
  e->lds_opt_in = true;
  return CRL_OK;
}

// the hand-off cells fit where this call may keep them
bool handoff_fits(const crl_engine* e, const crl::ReduceGeom& G) {
  return !e->no_alloc || handoff_records(G) * sizeof(unsigned long long) <= kScratchExchangeBytes;
}

// Is the engine's stream being captured, so that what is launched now is recorded?
int query_capture(const crl_engine* e, bool* active) {
  *active = false;
  if (!e->stream) return CRL_OK;  // (the null stream cannot be captured)
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  HIP_TRY(hipStreamIsCapturing(e->stream, &status));
  *active = status != hipStreamCaptureStatusNone;
  return CRL_OK;
}

// Does this call sum in two passes, or by the scan?  The scan also takes what has no room for its
// cells: in the static scratch tables of more than 16,384 keys and batches of millions (cells past
// kNoAllocScanBytes; what is between is refused by ensure_handoff), and the larger tables where the
// cells would have to be allocated now and the stream is being captured, which allows none.
int choose_passes(const crl_engine* e, const crl::ReduceGeom& G, bool* two) {
  const size_t bytes = handoff_records(G) * sizeof(unsigned long long);
  const bool large = G.K > crl::kDenseKeys;
  *two = reduce_fast(G);
  if (!*two) return CRL_OK;
  if (e->no_alloc) {
    *two = handoff_fits(e, G) || (!large && bytes <= kNoAllocScanBytes);
  } else if (large && handoff_records(G) > e->exchange.n) {
    bool recorded;
    const int rc = query_capture(e, &recorded);
    if (rc) return rc;
    *two = !recorded;
  }
  return CRL_OK;
}

// (`words`: the engine's own buffer gets at least that many 64-bit words)
int ensure_handoff(crl_engine* e, const crl::ReduceGeom& G, size_t words = 0) {
  const size_t recs = handoff_records(G);
  if (e->no_alloc) {
    if (!handoff_fits(e, G))
      return fail(CRL_E_RANGE, "the ordered reduction of this engine needs %zu bytes of hand-off cells, "
                  "the static scratch of crl_run_fused_noalloc holds %zu", recs * sizeof(unsigned long long),
                  kScratchExchangeBytes);
    e->ho = reinterpret_cast<unsigned long long*>(e->static_scratch + kScratchTicketBytes);
  } else {
    hipError_t h = e->grow(e->exchange, std::max(recs, words));
    if (h != hipSuccess) return fail(CRL_E_ALLOC, "hand-off buffer allocation failed: %s", hipGetErrorString(h));
    e->ho = e->exchange.p;
    e->exchange_tag = 0;
  }
  return opt_in_lds(e);
}

int reduce_owners(crl_engine* e, const crl::ReduceGeom& G, float* Q, int n, const crl::HostSignal& sig) {
  const int groups = (G.n_blocks + crl::kGroupBlocks - 1) / crl::kGroupBlocks;
  const int keys = own_keys(G), waves = std::min(groups, crl::kOwnerWaves);
  const dim3 grid(1 << G.own_shift), block(64 * waves);
  const size_t lds = crl::owners_lds_bytes(waves, keys);
  if (keys <= crl::kTileKeys)
    hipLaunchKernelGGL(crl::k_reduce_owners<true>, grid, block, lds, e->stream, G, keys, Q, e->key.p, e->delta.p, n, e->ho, sig);
  else
    hipLaunchKernelGGL(crl::k_reduce_owners<false>, grid, block, lds, e->stream, G, keys, Q, e->key.p, e->delta.p, n, e->ho, sig);
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// Q[k] += ordered sum of the deltas of the n samples with key k, on one table.
// Up to kSmallSamples in one launch; `changed`, `sig`: see k_td_small.
template <class Samples>
int td_small(crl_engine* e, float* Q, const Samples& X, int n, int2* changed, const crl::HostSignal& sig) {
  const int rc = opt_in_lds(e);
  if (rc) return rc;
#define CRL_TD_SMALL(A, NB)                                                                                        \
  hipLaunchKernelGGL((crl::k_td_small<A, NB, Samples>), dim3(1), dim3(crl::kBlockSamples * NB),                    \
                     sizeof(crl::SmallLds<NB>), e->stream, X, n, Q, e->cfg.lr, e->cfg.gamma, e->cfg.max_mode, changed, sig)
#define CRL_TD_SMALL_A(NB)              \
  do {                                  \
    if (e->A == 4) CRL_TD_SMALL(4, NB); \
    else CRL_TD_SMALL(8, NB);           \
  } while (0)
  if (n <= crl::kBlockSamples) CRL_TD_SMALL_A(1);
  else if (n <= 2 * crl::kBlockSamples) CRL_TD_SMALL_A(2);
  else CRL_TD_SMALL_A(4);
#undef CRL_TD_SMALL_A
#undef CRL_TD_SMALL
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// More: a begin, the samples in one piece or several (whole blocks but for the last), an end.
struct TdPlan {
  crl::ReduceGeom G;
  int n;
  bool two;  // two passes, or the scan
};

int td_begin(crl_engine* e, int n, TdPlan* p) {
  hipError_t h = e->grow(e->key, (size_t)n);
  if (h == hipSuccess) h = e->grow(e->delta, (size_t)n);
  if (h != hipSuccess) return fail(CRL_E_ALLOC, "scratch allocation failed: %s", hipGetErrorString(h));
  p->n = n;
  p->G = reduce_geom_within(e, n, kHandoffLimitBytes);
  e->no_alloc = false;  // crl_update / crl_td_update: the engine's own hand-off buffer
  const int rc = choose_passes(e, p->G, &p->two);
  if (rc) return rc;
  return p->two ? ensure_handoff(e, p->G) : opt_in_lds(e);
}

// samples [at, at + m), which are X's first; `before`: says that the pieces before have been read
template <class Samples>
int td_piece(crl_engine* e, const TdPlan& p, const float* Q, const Samples& X, size_t at, int m,
             const crl::HostSignal& before) {
  const float lr = e->cfg.lr, gamma = e->cfg.gamma;
  const int max_mode = e->cfg.max_mode;
  const size_t block = at / crl::kBlockSamples;
  const dim3 grid((m + crl::kBlockSamples - 1) / crl::kBlockSamples);
  int32_t* key = e->key.p + at;
  float* delta = e->delta.p + at;
  if (p.two) {
    unsigned long long* cells = e->ho + (block << p.G.cell_shift);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(crl::kBlockSamples), crl::block_lds_bytes(p.G.own_shift), e->stream, p.G, X, m, Q,
                         lr, gamma, max_mode, key, delta, cells, before);
    };
    if (e->A == 4) go(crl::k_td_blocks<4, Samples>);
    else go(crl::k_td_blocks<8, Samples>);
  } else {
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(256), 0, e->stream, Q, X, m, lr, gamma, max_mode, key, delta, before);
    };
    if (e->A == 4) go(crl::k_delta<4, Samples>);
    else go(crl::k_delta<8, Samples>);
  }
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// `read`: says that the samples have been read
int td_end(crl_engine* e, const TdPlan& p, float* Q, const crl::HostSignal& read) {
  if (p.two) return reduce_owners(e, p.G, Q, p.n, read);
  hipLaunchKernelGGL(crl::k_reduce_scan, dim3((unsigned)((e->K + crl::kOwnKeys - 1) / crl::kOwnKeys)), dim3(256), 0,
                     e->stream, Q, (int)e->K, e->key.p, e->delta.p, p.n, read);
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// one shared-table step of two launches
struct SharedPlan {
  crl::ReduceGeom G;
  bool two;      // block sums and key owners; else one scan of the samples
  bool lds_map;  // the map in LDS
  size_t lds;    // of the act kernel: reduction table (two passes), then the map
};

int plan_shared_step(const crl_engine* e, SharedPlan* p) {
  p->G = reduce_geom_within(e, e->N, e->no_alloc ? kScratchExchangeBytes : kHandoffLimitBytes);
  const int rc = choose_passes(e, p->G, &p->two);
  if (rc) return rc;
  // The shared table itself stays in L2: streaming its 64 KB into every workgroup's
  // LDS each step measured slower than the row reads it saves (12.4 against 12.05 us
  // per step on 65,536 envs, also against the five speculative reads per env).
  p->lds = p->two ? crl::block_lds_bytes(p->G.own_shift) : 0;
  const size_t limit = p->two ? kLdsPerWorkgroup - kStaticLdsReserve : (size_t)64 * 1024;
  const size_t map_bytes = (size_t)e->map_words * 4;
  p->lds_map = e->cfg.map_mode == CRL_MAP_SHARED && map_bytes <= (size_t)kLdsMapLimitBytes && p->lds + map_bytes <= limit;
  if (p->lds_map) p->lds += map_bytes;
  return CRL_OK;
}

template <int A, int MAP>
void launch_shared_act(crl_engine* e, const SharedPlan& p, uint64_t t, int trace_row) {
  const crl::Rules R = e->rules();
  const crl::Ptrs P = e->ptrs();
  const int block = 256, grid = (e->N + block - 1) / block;
  if (p.two)
    hipLaunchKernelGGL((crl::k_shared_act<A, MAP, true>), dim3(grid), dim3(block), p.lds, e->stream, R, P,
                       t, trace_row, e->key.p, e->delta.p, p.G, e->ho);
  else
    hipLaunchKernelGGL((crl::k_shared_act<A, MAP, false>), dim3(grid), dim3(block), p.lds, e->stream, R,
                       P, t, trace_row, e->key.p, e->delta.p, p.G, e->ho);
}

// act (select + move + delta + block sums), then the key owners or the scan; `words`: of the
// exchange buffer, at least
int shared_step(crl_engine* e, uint64_t t, int trace_row, size_t words) {
  SharedPlan p{};
  int rc = plan_shared_step(e, &p);
  if (rc == CRL_OK && p.two) rc = ensure_handoff(e, p.G, words);
  if (rc) return rc;
  if (e->A == 4) {
    if (p.lds_map) launch_shared_act<4, 1>(e, p, t, trace_row);
    else launch_shared_act<4, 2>(e, p, t, trace_row);
  } else {
    if (p.lds_map) launch_shared_act<8, 1>(e, p, t, trace_row);
    else launch_shared_act<8, 2>(e, p, t, trace_row);
  }
  HIP_TRY(hipGetLastError());
  if (p.two) return reduce_owners(e, p.G, e->Q.p, e->N, crl::HostSignal{});
  const int grid = (int)((e->K + crl::kOwnKeys - 1) / crl::kOwnKeys);
  hipLaunchKernelGGL(crl::k_reduce_scan, dim3(grid), dim3(256), 0, e->stream, e->Q.p, (int)e->K,
                     e->key.p, e->delta.p, e->N, crl::HostSignal{});
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// ---- shared table: all steps of a call in one launch ---------------------------------

struct PersistPlan {
  bool ok;
  int grid;
  bool lds_map;
  bool fold;  // the instantiation with the common configuration's rules folded in
  bool hashed;  // the form for more than 16,384 keys
  size_t lds;
  crl::ReduceGeom G;
  // what the workgroups exchange, in 64-bit words from the start of one buffer
  size_t at_table, at_raw, at_cells, words;
};

// The one-launch kernel needs every workgroup resident at once (one per compute unit), and an
// owner's keys in its LDS.
bool persist_shape(const crl_engine* e, PersistPlan* p) {
  const int n_blocks = (e->N + crl::kBlockSamples - 1) / crl::kBlockSamples;
  if (e->cfg.table_mode != CRL_TABLE_SHARED || n_blocks > crl::kPersistMaxGroups || crl::kPersistMaxGroups > kComputeUnits)
    return false;
  // always 256 workgroups, each a block (with or without envs) and an owner (with or
  // without keys): 16,384 keys at most are 64 to an owner, more up to 512 in the hashed form
  p->G = reduce_geom(e, e->N);
  p->G.own_shift = crl::kPersistOwnShift;
  p->hashed = e->K > (size_t)crl::kDenseKeys;
  if (p->hashed && own_keys(p->G) > crl::kOwnKeysHashed) return false;
  p->G.cell_shift = crl::cell_shift_for(p->G.own_shift);
  p->G.main_shift = crl::main_shift_for(p->G.own_shift);
  p->grid = crl::kPersistMaxGroups;
  p->G.n_blocks = p->grid;  // workgroups without envs hand over empty cells
  const int n_own = 1 << p->G.own_shift;
  auto pad = [](size_t words) { return (words + 31) & ~(size_t)31; };  // 256-byte pieces
  p->at_table = 0;
  p->at_raw = p->at_table + pad(2 * (size_t)e->K);  // a cell's view: its A values and A neighbours' maxima
  p->at_cells = p->at_raw + pad(2 * (size_t)e->N);  // raw samples and cells: two buffers each
  p->words = p->at_cells + 2 * (((size_t)n_own * p->grid) << p->G.cell_shift);
  return true;
}

// Shortest call worth the set-up of the one-launch kernel (one co-resident launch and its first
// values: 25 us) instead of two plain launches per step, which cost more the more envs there are.
// Where the two cross (us per call, one launch / two, at 8, 10, 12 and 14 steps): 3000 envs of 16x16
// 68/59, 80/74, 91/94, 102/112; 8000 of 32x32 70/61, 82/76, 94/91, 105/107; 16,000 of 32x32 70/65,
// 81/81, 94/97, 105/119; 32,768 of 64x64 73/71, 86/88, 99/106, 112/124; 65,536 of 64x64 80/85,
// 94/106, 109/128, 123/149.  The lines of the dense form lie two or three steps higher, where the two
// crossed while each call also cleared what is exchanged; callers read them from crl_fused_kernel_info,
// and they stay.
// With more than 16,384 keys two launches cost 9 to 11 us a step with 4 actions and 13 to 15 with 8
// (a row of the table is 32 bytes then, and a cell has nine of them to read), the hashed form 6.5 to
// 10; at 6, 8 and 10 steps: 20,000 envs of 101x99, 8 actions 74/75, 90/100, 106/125; 65,536 of 128x128,
// 8 actions 90/90, 112/120, 133/150; 3000 of 90x90 64/58, 77/77, 91/97; 20,000 of 128x128 72/62, 86/82,
// 102/103; 65,536 of 128x128 82/75, 103/100, 121/125.  Tables of up to 96 keys to an owner under few
// envs keep two launches, the plan that has always been reported for them (6000 envs of 72x72, 40
// steps: 307/401).
int persist_min_steps(const crl_engine* e, const PersistPlan& p) {
  const int n_envs = e->N;
  if (p.hashed && n_envs <= 8192 && own_keys(p.G) <= 96) return INT_MAX;
  if (p.hashed) return e->A == 8 ? 6 : 10;
  return n_envs <= 8192 ? 16 : n_envs <= 16384 ? 14 : n_envs <= 32768 ? 12 : n_envs <= 49152 ? 10 : 9;
}

// 64-bit words that the one-launch kernel's workgroups exchange through; 0: it cannot run
size_t persist_words(const crl_engine* e) {
  PersistPlan p{};
  return persist_shape(e, &p) ? p.words : 0;
}

PersistPlan plan_persist(const crl_engine* e, int n_steps) {
  PersistPlan p{};
  if (e->fused_variant == 1 || e->persist_refused) return p;
  if (!persist_shape(e, &p) || (e->fused_variant == 0 && n_steps < persist_min_steps(e, p))) return p;
  const crl_config& c = e->cfg;
  p.fold = c.goal_mode == CRL_GOAL_ON_TARGET && c.auto_reset == 1 && c.max_mode == CRL_MAX_TRUE && c.reward_flags == 0 &&
           e->trace_n == 0 && e->sup_n == 0 && c.max_episodes == 0 && c.track_returns == 0;
  const size_t map_bytes = (size_t)e->map_words * 4;
  const size_t lds = p.hashed ? sizeof(crl::PersistLdsHashed) : e->A == 8 ? sizeof(crl::PersistLds<8>) : sizeof(crl::PersistLds<4>);
  p.lds_map = e->cfg.map_mode == CRL_MAP_SHARED && lds + map_bytes <= kLdsPerWorkgroup - kStaticLdsReserve;
  p.lds = lds + (p.lds_map ? map_bytes : 0);
  if (e->no_alloc && p.words * sizeof(unsigned long long) > kScratchExchangeBytes) return p;
  p.ok = true;
  return p;
}

template <int A, int MAP, bool CLK, bool FOLD, bool HASHED>
hipError_t launch_persist_kernel(crl_engine* e, const PersistPlan& p, unsigned long long* buf, uint64_t t0,
                                 int n_steps, uint32_t tag0, int trace_row0) {
  crl::Rules R = e->rules();
  crl::Ptrs P = e->ptrs();
  int n_keys = p.G.K;
  crl::PersistBufs B{};
  B.table = buf + p.at_table;
  B.raw = buf + p.at_raw;
  B.cells = buf + p.at_cells;
  B.err = reinterpret_cast<unsigned*>(e->pdiag.p);
  B.clocks = e->pdiag.p + 1;
  int spin_limit = e->persist_spin_limit;
  void* args[] = {&R, &P, &t0, &n_steps, &tag0, &trace_row0, &n_keys, &B, &spin_limit};
  // a cooperative launch is refused unless all workgroups can be resident together,
  // which the kernel's waits rely on
  return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&crl::k_shared_persist<A, MAP, CLK, FOLD, HASHED>), dim3(p.grid),
                                    dim3(256), args, (unsigned)p.lds, e->stream);
}

static_assert(crl::kPersistClockWords == CRL_PERSIST_CLOCK_WORDS, "include/crl.h states the size of the diagnostics");

// -> CRL_OK and *launched = true, or *launched = false when the caller should take
// the two-launches-per-step path instead
int run_persist(crl_engine* e, int n_steps, bool* launched) {
  *launched = false;
  const PersistPlan p = plan_persist(e, n_steps);
  if (!p.ok) return CRL_OK;
  int rc;
  unsigned long long* buf;
  if (!e->no_alloc && p.words > e->exchange.n) {
    // (a stream being captured allows no allocation: two launches per step record such a call)
    bool recorded;
    rc = query_capture(e, &recorded);
    if (rc) return rc;
    if (recorded) return CRL_OK;
  }
  if (e->no_alloc) {
    buf = reinterpret_cast<unsigned long long*>(e->static_scratch + kScratchTicketBytes);
  } else {
    if (p.words > e->exchange.n) e->exchange_tag = 0;
    if (e->grow(e->exchange, p.words) != hipSuccess) return fail(CRL_E_ALLOC, "allocation of the exchange buffers failed");
    buf = e->exchange.p;
  }
  rc = opt_in_lds(e);
  if (rc) return rc;
  // A launch's tags go on from those of the launch before, so that what the workgroups exchange
  // need not be cleared for it (10 MB, a launch of 6 us and the gap behind it; 12
  // steps of 3000 envs on 16x16 97 -> 91 us).  It is cleared where the tags start again: in a buffer
  // that something else was in, in the scratch that all engines share, in a launch that is or has been
  // recorded (its replays bring its tags back) and when they have all been used; a call longer than
  // that goes out as several launches.  (A kernel, not a memset: a caller may record this.)
  const uint32_t max_tag = p.hashed ? crl::kPersistMaxTagHashed : crl::kPersistMaxTag;
  const bool keep = !e->no_alloc && !e->recorded;
  uint32_t tag = keep ? e->exchange_tag : 0;
  int done = 0;
  while (done < n_steps) {
    // (tags tag + 1 to tag + n + 1)
    const uint32_t left = (uint32_t)(n_steps - done);
    if (tag != 0 && (left >= max_tag || tag + left + 1 > max_tag)) tag = 0;
    const int n = (int)std::min(left, max_tag - 1);
    if (tag == 0) {
      const size_t n16 = p.words / 2;
      hipLaunchKernelGGL(crl::k_clear16, dim3((unsigned)((n16 + 1023) / 1024)), dim3(256), 0, e->stream,
                         reinterpret_cast<uint4*>(buf), n16);
    }
    const uint64_t t0 = e->t + (uint64_t)done;
    const int row0 = (int)std::min<long long>((long long)e->trace_cursor + done, e->trace_cap);
    hipError_t h;
#define CRL_PERSIST_FORM(A, MAP, HASHED)                                                                    \
  (e->persist_clocks ? (p.fold ? launch_persist_kernel<A, MAP, true, true, HASHED>(e, p, buf, t0, n, tag, row0)    \
                               : launch_persist_kernel<A, MAP, true, false, HASHED>(e, p, buf, t0, n, tag, row0))  \
                     : (p.fold ? launch_persist_kernel<A, MAP, false, true, HASHED>(e, p, buf, t0, n, tag, row0)   \
                               : launch_persist_kernel<A, MAP, false, false, HASHED>(e, p, buf, t0, n, tag, row0)))
#define CRL_PERSIST(A, MAP) (p.hashed ? CRL_PERSIST_FORM(A, MAP, true) : CRL_PERSIST_FORM(A, MAP, false))
    if (e->A == 4) h = p.lds_map ? CRL_PERSIST(4, 1) : CRL_PERSIST(4, 2);
    else h = p.lds_map ? CRL_PERSIST(8, 1) : CRL_PERSIST(8, 2);
#undef CRL_PERSIST
#undef CRL_PERSIST_FORM
    if (h != hipSuccess) {
      (void)hipGetLastError();
      if (done > 0) return fail(CRL_E_DEVICE, "the one-launch shared-table kernel was refused after %d steps: %s", done, hipGetErrorString(h));
      e->persist_refused = true;  // not resident all at once on this device: never mind, two launches per step
      return CRL_OK;
    }
    e->persist_unchecked = true;
    done += n;
    tag += (uint32_t)n + 1;
    if (!e->no_alloc) e->exchange_tag = keep ? tag : 0;
  }
  if (e->trace_n > 0) {
    const long long c = (long long)e->trace_cursor + n_steps;
    e->trace_cursor = c > e->trace_cap ? e->trace_cap : (int)c;
  }
  *launched = true;
  return CRL_OK;
}

// ---- pinned memory between host and kernels --------------------------------------------

constexpr size_t kLinkLimitBytes = (size_t)4 << 20;  // larger transfers: hipMemcpyAsync straight to and from the caller's memory
constexpr size_t kInPageBytesOfFour = (size_t)128 << 10;  // larger pages are two
// Transitions of a crl_td_update that go through one page.  Larger pieces cost more to pin, smaller
// ones more launches (one page of their own for all / pieces of 65,536 / 131,072 / 262,144, us per
// call among others: 200,000 58.8 / - / 62.8 / 58.8, 1 million 400 / 375 / 325 / 300, 2 million 935 /
// 1010 / 880 / 780; 6 million in a page of their own 39,000, in pieces 3000).
constexpr int kPieceSamples = 1 << 18;
constexpr int kFlagErrWord = 16;                     // of flag_page; in another 64-byte line than the flag

// the next launch that tells the host when it is through
crl::HostSignal next_signal(crl_engine* e) {
  if (++e->seq == 0) ++e->seq;
  crl::HostSignal sig;
  sig.flag = reinterpret_cast<unsigned*>(e->flag_page.p);
  sig.seq = e->seq;
  sig.count = e->flag_count.p;
  return sig;
}

bool seq_passed(const crl_engine* e, unsigned seq) {
  const volatile unsigned* flag = reinterpret_cast<const volatile unsigned*>(e->flag_page.p);
  return (int)(*flag - seq) >= 0;
}

// Waits until launch `seq` is through: looks at the flag for a while (a small call is over
// in microseconds), then leaves the waiting, and finding out about errors, to the runtime.
int wait_seq(crl_engine* e, unsigned seq) {
  if (!seq_passed(e, seq)) {
    const auto give_up = std::chrono::steady_clock::now() + std::chrono::microseconds(300);
    bool passed = false;
    do {
      for (int i = 0; i < 64 && !passed; ++i) {
        passed = seq_passed(e, seq);
        if (!passed) __builtin_ia32_pause();
      }
    } while (!passed && std::chrono::steady_clock::now() < give_up);
    if (!passed) {
      HIP_TRY(hipStreamSynchronize(e->stream));
      if (!seq_passed(e, seq)) return fail(CRL_E_DEVICE, "a launch ended without telling the host so");
    }
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return CRL_OK;
}

// out_page with room for `bytes`; what it held is no longer there
int claim_out_page(crl_engine* e, size_t bytes) {
  e->mirror_seq = 0;
  e->stats_here = false;
  if (bytes <= e->out_page.n) return CRL_OK;
  HIP_TRY(hipStreamSynchronize(e->stream));  // nobody may still be writing to the smaller one
  if (!e->out_page.ensure(bytes)) return fail(CRL_E_ALLOC, "pinned host memory: %zu bytes", bytes);
  return CRL_OK;
}

// The launch that reads this page is through.
int wait_slot(crl_engine* e, crl_engine::InSlot& slot) {
  if (slot.last_seq == 0) return CRL_OK;
  const int rc = wait_seq(e, slot.last_seq);
  if (rc == CRL_OK) slot.last_seq = 0;
  return rc;
}

// A page for `bytes` that no earlier launch still reads.  The pages grow together, and are two
// where they are large: what they cost is the first touch of their memory (0.37 ms per MB), paid
// by the first call that takes each of them.
int claim_in_slot(crl_engine* e, size_t bytes, crl_engine::InSlot** out) {
  if (bytes > e->in_page_bytes) {
    for (auto& slot : e->in_slot) {
      const int rc = wait_slot(e, slot);
      if (rc) return rc;
    }
    size_t page = 4096;
    while (page < bytes) page *= 2;
    const int slots = page > kInPageBytesOfFour ? 2 : crl_engine::kInSlots;
    e->in_page_bytes = 0;
    if (!e->in_block.ensure(page * slots)) return fail(CRL_E_ALLOC, "pinned host memory: %zu bytes", page * slots);
    e->in_page_bytes = page;
    e->in_slots = slots;
    e->in_next = 0;
    for (int i = 0; i < slots; ++i) e->in_slot[i].page = e->in_block.p + page * i;
  }
  crl_engine::InSlot& slot = e->in_slot[e->in_next];
  e->in_next = (e->in_next + 1) % e->in_slots;
  const int rc = wait_slot(e, slot);
  if (rc) return rc;
  *out = &slot;
  return CRL_OK;
}

int persist_result(crl_engine* e, unsigned gave_up);

// `bytes` of device memory (a multiple of 16, as all arrays of the arena are padded to) in
// out_page once this returns
int fetch_pinned(crl_engine* e, const void* src, size_t bytes) {
  int rc = claim_out_page(e, bytes);
  if (rc) return rc;
  const crl::HostSignal sig = next_signal(e);
  const size_t n16 = (bytes + 15) / 16;
  const int grid = (int)std::min<size_t>((n16 + 255) / 256, 256);
  const bool check = e->persist_unchecked;
  unsigned* flags = reinterpret_cast<unsigned*>(e->flag_page.p);
  hipLaunchKernelGGL(crl::k_export, dim3(grid), dim3(n16 < 256 ? 64 : 256), 0, e->stream,
                     static_cast<const uint4*>(src), reinterpret_cast<uint4*>(e->out_page.p), n16,
                     check ? reinterpret_cast<const unsigned*>(e->pdiag.p) : nullptr, flags + kFlagErrWord, sig);
  HIP_TRY(hipGetLastError());
  rc = wait_seq(e, sig.seq);
  if (rc) return rc;
  if (!check) return CRL_OK;
  e->persist_unchecked = false;
  return persist_result(e, static_cast<volatile unsigned*>(flags)[kFlagErrWord]);
}

// out_page as the engine's state arrays are laid out
crl::StateMirror state_mirror(const crl_engine* e) {
  crl::StateMirror M{};
  auto at = [&](const void* p) { return e->out_page.p + (static_cast<const unsigned char*>(p) - e->state_at); };
  M.s = reinterpret_cast<int32_t*>(at(e->s.p));
  M.ep_step = reinterpret_cast<int32_t*>(at(e->ep_step.p));
  M.episode = reinterpret_cast<int32_t*>(at(e->episode.p));
  M.reward = reinterpret_cast<float*>(at(e->reward.p));
  M.done = at(e->done.p);
  M.action = at(e->action.p);
  return M;
}

// Did a one-launch kernel give up waiting for its peers?  Called by the entry points
// that synchronise; reports a give-up once.  The give-up word stays set on the device
// (the kernel's later launches see it and return at once), and until the caller has set
// state or table again every call that works on them fails (require_valid).
int check_persist(crl_engine* e) {
  if (!e->persist_unchecked) return CRL_OK;
  e->persist_unchecked = false;
  unsigned gave_up = 0;
  HIP_TRY(hipMemcpyAsync(&gave_up, e->pdiag.p, sizeof gave_up, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return persist_result(e, gave_up);
}

int persist_result(crl_engine* e, unsigned gave_up) {
  if (!gave_up) return CRL_OK;
  e->persist_failed = true;
  return fail(CRL_E_DEVICE, "the one-launch shared-table kernel gave up waiting for its workgroups "
              "(were they all resident?); state and table are not valid: set them again (crl_reset, "
              "crl_set_state, crl_q_set) and use crl_set_fused_variant(e, 1)");
}

int require_valid(const crl_engine* e) {
  if (e->persist_failed)
    return fail(CRL_E_STATE, "a one-launch shared-table kernel gave up earlier: state and table are not valid "
                "until crl_reset, crl_set_state or crl_q_set");
  return CRL_OK;
}

// The caller sets state or table again.  A launch nobody has looked at yet is looked at
// first (and a give-up reported by this call); a give-up already reported is history.
int clear_persist_failure(crl_engine* e) {
  int rc = check_persist(e);
  if (rc) return rc;
  if (!e->persist_failed) return CRL_OK;
  HIP_TRY(hipMemsetAsync(e->pdiag.p, 0, sizeof(unsigned long long), e->stream));
  e->persist_failed = false;
  return CRL_OK;
}

// sizes that follow from the configuration alone
void set_geometry(crl_engine* e, const crl_config& cfg) {
  e->cfg = cfg;
  e->N = cfg.n_envs;
  e->W = cfg.width;
  e->H = cfg.height;
  e->A = cfg.n_actions;
  e->S = (size_t)cfg.width * cfg.height;
  e->K = e->S * e->A;
  e->n_maps = cfg.map_mode == CRL_MAP_SHARED ? 1 : e->N;
  e->n_tables = cfg.table_mode == CRL_TABLE_SHARED ? 1 : e->N;
  e->map_words = (int)((e->S + 15) / 16);
  const size_t cells_per_word = 16 / (size_t)e->A;
  e->mv_words = (int)((e->S + cells_per_word - 1) / cells_per_word);
}

// For calls that may be recorded: note it where this one is.
int note_recording(crl_engine* e) {
  bool active;
  const int rc = query_capture(e, &active);
  if (rc == CRL_OK && active) e->recorded = true;
  return rc;
}

// For calls that change the state: no copy of it that the host holds is good any more, and
// once such a call has been recorded none ever is, as its replays change the state unseen.
int state_changes(crl_engine* e) {
  const int rc = note_recording(e);
  if (rc) return rc;
  if (e->recorded) e->state_shared = true;
  e->mirror_seq = 0;
  e->state_read = e->stats_here = false;
  e->stepped = false;
  return CRL_OK;
}

int check_engine(const crl_engine* e) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  hipError_t err = hipSetDevice(e->device);
  if (err != hipSuccess) return fail(CRL_E_DEVICE, "hipSetDevice(%d): %s", e->device, hipGetErrorString(err));
  return CRL_OK;
}

int check_usable(const crl_engine* e) {
  int rc = check_engine(e);
  return rc ? rc : require_valid(e);
}

// move codes of maps [first, first + count) from the class maps on the device
int build_moves(crl_engine* e, int first, int count) {
  if (e->mv_words == 0 || count <= 0) return CRL_OK;
  const size_t threads = (size_t)count * e->mv_words;
  const dim3 g((unsigned)((threads + 255) / 256)), b(256);
  if (e->A == 4)
    hipLaunchKernelGGL(crl::k_build_moves<4>, g, b, 0, e->stream, e->map.p, e->map_words, e->W, e->H,
                       e->mv_words, first, count, e->moves.p);
  else
    hipLaunchKernelGGL(crl::k_build_moves<8>, g, b, 0, e->stream, e->map.p, e->map_words, e->W, e->H,
                       e->mv_words, first, count, e->moves.p);
  HIP_TRY(hipGetLastError());
  return CRL_OK;
}

// Packs the caller's class maps 2 bits to a cell and uploads them a slice of maps at a
// time (the engine keeps no host copy of maps or cell rewards: for 8192 maps of 256x256
// cells those would be 0.5 GB and 2 GB for the life of the engine).
int upload_maps(crl_engine* e, const uint8_t* cell_class, const float* cell_reward) {
  const size_t slice_maps = std::max<size_t>(1, ((size_t)16 << 20) / ((size_t)e->map_words * 4));
  std::vector<uint32_t> packed(std::min<size_t>(slice_maps, (size_t)e->n_maps) * e->map_words);
  for (size_t m0 = 0; m0 < (size_t)e->n_maps; m0 += slice_maps) {
    const size_t count = std::min(slice_maps, (size_t)e->n_maps - m0);
    std::fill(packed.begin(), packed.end(), 0u);
    for (size_t m = 0; m < count; ++m)
      crl::pack_classes(cell_class + (m0 + m) * e->S, e->S, packed.data() + m * e->map_words);
    HIP_TRY(hipMemcpyAsync(e->map.p + m0 * e->map_words, packed.data(), count * e->map_words * sizeof(uint32_t),
                           hipMemcpyHostToDevice, e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));  // the slice buffer is filled again next round
  }
  if (e->cfg.reward_flags & CRL_REWARD_CELLS)
    HIP_TRY(hipMemcpyAsync(e->cell_reward.p, cell_reward, (size_t)e->n_maps * e->S * sizeof(float),
                           hipMemcpyHostToDevice, e->stream));
  const int rc = build_moves(e, 0, e->n_maps);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(e->stream));
  return CRL_OK;
}

int opt_in_ticket_kernels(crl_engine* e);

int create_engine(const crl_config* cfg, int device, crl_engine** out) {
  if (!out) return fail(CRL_E_ARG, "out is null");
  *out = nullptr;
  int rc = crl::validate_config(cfg, crl::last_error());
  if (rc != CRL_OK) return rc;
  int ndev = 0;
  hipError_t herr = hipGetDeviceCount(&ndev);
  if (herr != hipSuccess || ndev <= 0)
    return fail(CRL_E_DEVICE, "no HIP device available (%s); this engine has no CPU path",
                herr != hipSuccess ? hipGetErrorString(herr) : "count is 0");
  if (device < 0 || device >= ndev) return fail(CRL_E_ARG, "device %d out of range [0,%d)", device, ndev);
  HIP_TRY(hipSetDevice(device));

  std::unique_ptr<crl_engine> own(new crl_engine());  // freed on every early return and on a throw
  crl_engine* e = own.get();
  set_geometry(e, *cfg);
  e->device = device;

  const size_t N = (size_t)e->N;
  std::vector<float> eps = crl::build_eps_table(*cfg);
  e->eps_len = (int)eps.size();
  const bool cells = (cfg->reward_flags & CRL_REWARD_CELLS) != 0;
  hipError_t a = hipSuccess;
  auto acc = [&](hipError_t x) {
    if (a == hipSuccess) a = x;
  };
  // One allocation and one clearing pass for everything (each hipMalloc and hipMemsetAsync
  // on its own costs microseconds to tens of them, and there are two dozen arrays).
  unsigned char* base = nullptr;
  size_t used = 0;
  auto carve = [&](auto& buf, size_t count) {
    if (base) buf.adopt(base + used, count);
    used += (count * sizeof(*buf.p) + 255) & ~(size_t)255;
  };
  size_t cleared = 0;  // what comes first is cleared
  auto lay_out = [&]() {
    used = 0;
    carve(e->s, N);
    carve(e->ep_step, N);
    carve(e->episode, N);
    carve(e->reward, N);
    carve(e->done, N);
    carve(e->action, N);
    e->state_at = base;
    e->state_bytes = used;
    if (cfg->track_returns) {
      e->stats_at = base + used;
      const size_t from = used;
      carve(e->ret_last, N);
      carve(e->len_last, N);
      carve(e->ret_sum, N);
      carve(e->len_sum, N);
      e->stats_bytes = used - from;
      carve(e->ret_acc, N);
    }
    carve(e->start, N);
    carve(e->act, N);
    carve(e->flag_count, 1);
    if (cfg->table_mode == CRL_TABLE_PER_ENV) {
      carve(e->ticket, 3);
      carve(e->split, 3);
    } else {
      carve(e->pdiag, 1 + crl::kPersistClockWords);
    }
    // (large arrays where an allocation of their own would start them: 1M tables of 4 KB that
    // start 256 bytes into a page each, 20 steps 631 -> 635 us, 1000 steps 12.17 -> 12.23 ms)
    auto page = [&](size_t bytes) {
      const size_t at = bytes >= (size_t)32 << 20 ? (size_t)2 << 20 : 256;
      used = (used + at - 1) & ~(at - 1);
    };
    page((size_t)e->n_maps * e->map_words * 4);
    carve(e->map, (size_t)e->n_maps * e->map_words);
    page((size_t)e->n_tables * e->K * 4);
    carve(e->Q, (size_t)e->n_tables * e->K);
    cleared = used;
    page((size_t)e->n_maps * e->mv_words * 4);
    carve(e->moves, (size_t)e->n_maps * e->mv_words + 1);  // move codes of every map, for the fused loops (and a word that is read, not used)
    if (cells) carve(e->cell_reward, (size_t)e->n_maps * e->S);
    carve(e->eps_tab, eps.size());
    carve(e->tr_s, N);
    carve(e->tr_a, N);
    carve(e->tr_s2, N);
    carve(e->tr_r, N);
    carve(e->tr_done, N);
    if (cfg->table_mode == CRL_TABLE_SHARED) {
      carve(e->key, N);
      carve(e->delta, N);
    }
  };
  lay_out();
  acc(e->arena.alloc(used));
  if (a == hipSuccess) {
    base = e->arena.p;
    lay_out();
  }
  if (a != hipSuccess) {
    const int code = a == hipErrorOutOfMemory ? CRL_E_ALLOC : CRL_E_DEVICE;
    return fail(code, "device allocation failed: %s", hipGetErrorString(a));
  }
  auto bail = [&](hipError_t x, const char* what) {
    return fail(CRL_E_DEVICE, "%s: %s", what, hipGetErrorString(x));
  };
  hipError_t h;
  if (!e->flag_page.ensure(128)) return fail(CRL_E_ALLOC, "pinned host memory for the engine's flag");
  std::memset(e->flag_page.p, 0, 128);
  if ((h = hipMemsetAsync(e->arena.p, 0, cleared, e->stream)) != hipSuccess) return bail(h, "clear the arena");
  if ((h = hipMemcpyAsync(e->eps_tab.p, eps.data(), eps.size() * sizeof(float), hipMemcpyHostToDevice,
                          e->stream)) != hipSuccess)
    return bail(h, "upload eps table");
  if (cells) {  // until crl_set_maps: every cell pays the step reward
    uint32_t bits;
    std::memcpy(&bits, &cfg->step_reward, 4);
    const size_t n = e->cell_reward.n;
    hipLaunchKernelGGL(crl::k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, e->stream,
                       reinterpret_cast<unsigned*>(e->cell_reward.p), bits, n);
    if ((h = hipGetLastError()) != hipSuccess) return bail(h, "fill cell rewards");
  }
  rc = build_moves(e, 0, e->n_maps);  // of the all-free maps that stand until crl_set_maps
  if (rc != CRL_OK) return rc;
  if ((h = hipStreamSynchronize(e->stream)) != hipSuccess) return bail(h, "sync");
  // set-up that crl_run_fused_noalloc must not have left to do: this device's copy
  // of the scratch array, and the kernels that may use the whole LDS
  rc = scratch_of_device(device, &e->static_scratch);
  if (rc == CRL_OK) rc = cfg->table_mode == CRL_TABLE_SHARED ? opt_in_lds(e) : opt_in_ticket_kernels(e);
  if (rc != CRL_OK) return rc;
  *out = own.release();
  return CRL_OK;
}

int reset_envs(crl_engine* e, int32_t first, int32_t count) {
  int rc = check_engine(e);
  if (rc) return rc;
  rc = clear_persist_failure(e);
  if (rc) return rc;
  if (first < 0 || count < 0 || (int64_t)first + count > e->N)
    return fail(CRL_E_RANGE, "env range [%d,%d) outside [0,%d)", first, first + count, e->N);
  if (count == 0) return CRL_OK;
  rc = state_changes(e);
  if (rc) return rc;
  hipLaunchKernelGGL(crl::k_reset, dim3((count + 255) / 256), dim3(256), 0, e->stream, e->ptrs(), first,
                     count);
  HIP_TRY(hipGetLastError());
  e->have_transition = false;
  return CRL_OK;
}

int set_maps(crl_engine* e, const uint8_t* cell_class, const int32_t* start,
                 const float* cell_reward) {
  int rc = check_engine(e);
  if (rc) return rc;
  if (!cell_class) return fail(CRL_E_ARG, "cell_class is null");
  const bool cells = (e->cfg.reward_flags & CRL_REWARD_CELLS) != 0;
  if (cells && !cell_reward) return fail(CRL_E_ARG, "reward_flags asks for cell rewards but none given");
  if (!cells && cell_reward) return fail(CRL_E_ARG, "cell rewards given but reward_flags has no CRL_REWARD_CELLS");
  const size_t total = (size_t)e->n_maps * e->S;
  for (size_t i = 0; i < total; ++i)
    if (cell_class[i] > CRL_CELL_WALL) return fail(CRL_E_ARG, "cell_class[%zu] = %d is not a cell class", i, (int)cell_class[i]);
  if (start)
    for (int i = 0; i < e->N; ++i)
      if (start[i] < 0 || (size_t)start[i] >= e->S)
        return fail(CRL_E_RANGE, "start[%d] = %d outside [0,%zu)", i, start[i], e->S);
  rc = upload_maps(e, cell_class, cell_reward);
  if (rc) return rc;
  if (start) {
    HIP_TRY(hipMemcpyAsync(e->start.p, start, (size_t)e->N * 4, hipMemcpyHostToDevice, e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));
  }
  return reset_envs(e, 0, e->N);
}

int set_cell(crl_engine* e, int32_t map_index, int32_t cell, int32_t cell_class,
                 float cell_reward) {
  int rc = check_engine(e);
  if (rc) return rc;
  if (map_index < 0 || map_index >= e->n_maps) return fail(CRL_E_RANGE, "map index %d outside [0,%d)", map_index, e->n_maps);
  if (cell < 0 || (size_t)cell >= e->S) return fail(CRL_E_RANGE, "cell %d outside [0,%zu)", cell, e->S);
  if (cell_class < CRL_CELL_FREE || cell_class > CRL_CELL_WALL) return fail(CRL_E_ARG, "%d is not a cell class", cell_class);
  const size_t at = (size_t)map_index * e->S + cell;
  // the word of 16 cells that holds this one: fetched, changed, put back
  const size_t word = (size_t)map_index * e->map_words + (cell >> 4);
  uint32_t packed = 0;
  HIP_TRY(hipMemcpyAsync(&packed, e->map.p + word, 4, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  const int shift = 2 * (cell & 15);
  packed = (packed & ~(3u << shift)) | ((uint32_t)cell_class << shift);
  HIP_TRY(hipMemcpyAsync(e->map.p + word, &packed, 4, hipMemcpyHostToDevice, e->stream));
  rc = build_moves(e, map_index, 1);  // the neighbours' codes name this cell
  if (rc) return rc;
  if (e->cfg.reward_flags & CRL_REWARD_CELLS)
    HIP_TRY(hipMemcpyAsync(e->cell_reward.p + at, &cell_reward, 4, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));  // `packed` and `cell_reward` are this call's
  return CRL_OK;
}

// every ticket-kernel instantiation launch_fused_a can pick may use the whole LDS:
// the plain ones, too, ask for more than the default 64 KB when large per-env
// maps share a workgroup (those that keep rows do not: six of them fit a compute
// unit where their maps are staged, 26,880 bytes at most)
int opt_in_ticket_kernels(crl_engine* e) {
  if (e->hybrid_opt_in) return CRL_OK;
  const void* fns[] = {
#define CRL_TICKET_KERNELS(A)                                                          \
  reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 0, false, false, 0>),            \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 1, false, false, 0>),        \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 2, false, false, 0>),        \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 0, true, false, 0>),         \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 1, true, false, 0>),         \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 1, false, true, 0>),         \
      reinterpret_cast<const void*>(&crl::k_fused_tickets<A, 2, false, true, 0>),         \
      CRL_LANE_KERNELS(A, false), CRL_LANE_KERNELS(A, true),                           \
      reinterpret_cast<const void*>(&crl::k_fused_per_env<A, 1, 2>),                   \
      CRL_LDS_KERNELS(A, false), CRL_LDS_KERNELS(A, true)
#define CRL_EVENTS(KERN, A, FLAG)                                                      \
  reinterpret_cast<const void*>(&crl::KERN<A, FLAG, crl::kNoEvents>),                  \
      reinterpret_cast<const void*>(&crl::KERN<A, FLAG, crl::kEpsilonEvents>),         \
      reinterpret_cast<const void*>(&crl::KERN<A, FLAG, crl::kAllEvents>)
#define CRL_LANE_KERNELS(A, CELLS) CRL_EVENTS(k_fused_lanes, A, CELLS)
#define CRL_LDS_KERNELS(A, WORDS) CRL_EVENTS(k_fused_tickets_lds, A, WORDS), CRL_EVENTS(k_fused_per_env_lds, A, WORDS)
      CRL_TICKET_KERNELS(4), CRL_TICKET_KERNELS(8)
#undef CRL_TICKET_KERNELS
#undef CRL_LDS_KERNELS
#undef CRL_LANE_KERNELS
#undef CRL_EVENTS
  };
  for (const void* fn : fns)
    HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsPerWorkgroup));
  e->hybrid_opt_in = true;
  return CRL_OK;
}

// For calls whose kernel reads what the host has just put down - in pages that are taken in
// turn, or as an argument: a replay of a recorded launch would read another call's.
int refuse_capture(const crl_engine* e) {
  bool active;
  const int rc = query_capture(e, &active);
  if (rc || !active) return rc;
  return fail(CRL_E_DEVICE, "a call that takes host data cannot be recorded: its stream is being captured");
}

// Bytes of a packed transition: the key, s' and done fit one word where a key has 16 bits and s' 15.
size_t sample_bytes(const crl_engine* e) { return e->K < 0xffffu ? 8 : 12; }

// Transitions [at, at + n) of a call packed into a page.
int pack_page(const crl_engine* e, size_t at, int n, const int32_t* s, const int32_t* a, const float* r,
              const int32_t* s_next, const uint8_t* done, unsigned char* page, crl::PackedSamples* X) {
  int32_t* key = reinterpret_cast<int32_t*>(page);
  const bool two_words = sample_bytes(e) == 8;
  uint32_t* s2d = two_words ? nullptr : reinterpret_cast<uint32_t*>(key + n);
  const bool fine = two_words ? crl::pack_transitions_short(n, (int)e->S, e->A, s + at, a + at, s_next + at, done + at,
                                                            reinterpret_cast<uint32_t*>(page))
                              : crl::pack_transitions(n, (int)e->S, e->A, s + at, a + at, s_next + at, done + at, key, s2d);
  if (!fine)
    for (size_t i = at; i < at + n; ++i) {
      if (s[i] < 0 || (size_t)s[i] >= e->S) return fail(CRL_E_RANGE, "s[%zu] = %d outside [0,%zu)", i, s[i], e->S);
      if (s_next[i] < 0 || (size_t)s_next[i] >= e->S)
        return fail(CRL_E_RANGE, "s_next[%zu] = %d outside [0,%zu)", i, s_next[i], e->S);
    }
  float* rewards = reinterpret_cast<float*>(key + (two_words ? n : 2 * (size_t)n));
  std::memcpy(rewards, r + at, (size_t)n * 4);
  X->key = key;
  X->s2d = s2d;
  X->r = rewards;
  return CRL_OK;
}

// Even pieces of at most kPieceSamples, each a page and a launch of the first pass of its own:
// a piece is packed while the kernels read the ones before.  A page is free again when the
// launch after the one that reads it starts.
int td_pieces(crl_engine* e, float* Q, int n, const int32_t* s, const int32_t* a, const float* r, const int32_t* s_next,
              const uint8_t* done) {
  TdPlan p;
  int rc = td_begin(e, n, &p);
  if (rc) return rc;
  const size_t pieces = ((size_t)n + kPieceSamples - 1) / kPieceSamples;
  const size_t even = ((n + pieces - 1) / pieces + crl::kBlockSamples - 1) & ~(size_t)(crl::kBlockSamples - 1);
  crl_engine::InSlot* unread = nullptr;  // the page of the last launch
  auto read = [&]() {
    crl::HostSignal sig{};
    if (unread) sig = next_signal(e);
    return sig;
  };
  for (size_t at = 0; at < (size_t)n; at += even) {
    const int m = (int)std::min(even, n - at);
    crl_engine::InSlot* slot;
    crl::PackedSamples X;
    rc = claim_in_slot(e, sample_bytes(e) * even, &slot);
    if (rc == CRL_OK) rc = pack_page(e, at, m, s, a, r, s_next, done, slot->page, &X);
    if (rc) return rc;
    const crl::HostSignal sig = read();
    rc = td_piece(e, p, Q, X, at, m, sig);
    if (rc) return rc;
    if (unread) unread->last_seq = sig.seq;
    unread = slot;
  }
  const crl::HostSignal sig = read();
  rc = td_end(e, p, Q, sig);
  if (rc == CRL_OK) unread->last_seq = sig.seq;
  return rc;
}

// crl_td_update and, with `keys`, crl_td_update_collect.  The transitions are packed into
// pinned memory, 8 or 12 bytes each, in the pass that checks them, and the kernel reads them
// there: the call returns without waiting for anything (65,536 transitions: five copies from
// pageable memory and a wait took 125 us).
int td_update(crl_engine* e, int32_t table, int32_t n, const int32_t* s, const int32_t* a, const float* r,
              const int32_t* s_next, const uint8_t* done, int32_t* keys, float* values) {
  int rc = check_usable(e);
  if (rc) return rc;
  if (table < 0 || table >= e->n_tables) return fail(CRL_E_RANGE, "table %d outside [0,%d)", table, e->n_tables);
  if (n < 0) return fail(CRL_E_ARG, "negative sample count");
  if (n == 0) return CRL_OK;
  if (!s || !a || !r || !s_next || !done) return fail(CRL_E_ARG, "null transition array");
  rc = refuse_capture(e);
  if (rc) return rc;
  float* Q = e->Q.p + (size_t)table * e->K;
  if (n > crl::kSmallSamples) {
    rc = td_pieces(e, Q, n, s, a, r, s_next, done);
    // nothing may be left that works on a page or waits for a number that never comes (nothing has
    // been applied: what is launched before the end only reads the table)
    if (rc) (void)hipStreamSynchronize(e->stream);
    return rc;
  }
  crl_engine::InSlot* slot;
  crl::PackedSamples X;
  rc = claim_in_slot(e, sample_bytes(e) * (size_t)n, &slot);
  if (rc == CRL_OK) rc = pack_page(e, 0, n, s, a, r, s_next, done, slot->page, &X);
  if (rc) return rc;
  int2* changed = nullptr;
  if (keys) {
    rc = claim_out_page(e, n * sizeof(int2));
    if (rc) return rc;
    changed = reinterpret_cast<int2*>(e->out_page.p);
  }
  const crl::HostSignal sig = next_signal(e);
  rc = td_small(e, Q, X, n, changed, sig);
  if (rc) {
    (void)hipStreamSynchronize(e->stream);
    return rc;
  }
  slot->last_seq = sig.seq;
  if (keys) {
    rc = wait_seq(e, sig.seq);
    if (rc) return rc;
    for (int i = 0; i < n; ++i) {
      keys[i] = changed[i].x;
      std::memcpy(values + i, &changed[i].y, 4);
    }
  }
  return CRL_OK;
}

// crl_run_fused and its allocation-free variant: with `no_alloc` the ticket
// counters and the hand-off cells live in the device's static scratch array and
// nothing below allocates or frees
int run_fused(crl_engine* e, int32_t n_steps, bool no_alloc) {
  int rc = check_engine(e);
  if (rc) return rc;
  if (n_steps < 0) return fail(CRL_E_ARG, "negative step count");
  if (n_steps == 0) return CRL_OK;
  if (no_alloc && !e->static_scratch) return fail(CRL_E_STATE, "the device's scratch array was not found at crl_create");
  rc = require_valid(e);
  if (rc) return rc;
  // whichever way this call ends, later calls work with the engine's own buffers again
  struct Restore {
    crl_engine* e;
    ~Restore() { e->no_alloc = false; }
  } restore{e};
  e->no_alloc = no_alloc;
  rc = state_changes(e);
  if (rc) return rc;
  if (e->cfg.table_mode == CRL_TABLE_PER_ENV) {
    const FusedPlan p = plan_fused(e, n_steps);
    if (p.lds > kLdsPerWorkgroup)
      return fail(CRL_E_STATE, "launch plan %s needs %zu bytes of LDS per workgroup, the device has %zu",
                  p.name, p.lds, kLdsPerWorkgroup);
    if (p.tickets) {
      if (no_alloc) {
        e->tk = reinterpret_cast<unsigned*>(e->static_scratch);
      } else {
        if (e->ticket.ensure(3) != hipSuccess) return fail(CRL_E_ALLOC, "ticket counter allocation failed");
        e->tk = e->ticket.p;
      }
      rc = opt_in_ticket_kernels(e);  // done at crl_create; a no-op here
      if (rc) return rc;
    }
    if (e->A == 4)
      launch_fused_a<4>(e, p, e->t, n_steps);
    else
      launch_fused_a<8>(e, p, e->t, n_steps);
    HIP_TRY(hipGetLastError());
    if (p.tickets && !p.fixed) {
      // the counters may sit in the scratch all engines of this GPU share: kept here
      hipLaunchKernelGGL(crl::k_copy3_u32, dim3(1), dim3(64), 0, e->stream, e->tk, e->split.p);
      HIP_TRY(hipGetLastError());
    }
    e->split_valid = p.tickets;
    if (e->trace_n > 0) {
      const long long c = (long long)e->trace_cursor + n_steps;
      e->trace_cursor = c > e->trace_cap ? e->trace_cap : (int)c;
    }
  } else {
    bool launched = false;
    rc = run_persist(e, n_steps, &launched);
    if (rc) return rc;
    // A call of a few steps takes two launches to a step and a longer one the one-launch kernel:
    // whichever comes first makes room for both, so that neither allocates later and both can be
    // recorded.  (Not calls of one to three steps: the larger allocation costs a first call 20 us,
    // 6 steps of 300 envs 66 / 85.  Not a call that is being recorded, which may allocate nothing: it
    // makes do with the cells that calls before it have left.)
    bool capturing = false;
    if (e->recorded) rc = query_capture(e, &capturing);  // (state_changes has noted this call)
    if (rc) return rc;
    const size_t words = n_steps > 3 && !capturing ? persist_words(e) : 0;
    for (int k = 0; !launched && k < n_steps; ++k) {
      rc = shared_step(e, e->t + (uint64_t)k, e->trace_cursor, words);
      if (rc) return rc;
      if (e->trace_n > 0 && e->trace_cursor < e->trace_cap) e->trace_cursor += 1;
    }
  }
  e->t += (uint64_t)n_steps;
  e->have_transition = false;
  e->have_actions = false;
  return CRL_OK;
}

}  // namespace

extern "C" {

const char* crl_last_error(void) { return crl::last_error().c_str(); }
const char* crl_version(void) { return CRL_VERSION; }

int crl_device_count(void) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) return fail(CRL_E_DEVICE, "hipGetDeviceCount: %s", hipGetErrorString(e));
  return n;
}

int crl_create(const crl_config* cfg, int device, crl_engine** out) {
  return guarded([&] { return create_engine(cfg, device, out); });
}

int crl_destroy(crl_engine* e) {
  if (!e) return CRL_OK;
  (void)hipSetDevice(e->device);
  (void)hipStreamSynchronize(e->stream);
  delete e;
  return CRL_OK;
}

int crl_set_stream(crl_engine* e, void* hip_stream) {
  int rc = check_engine(e);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(e->stream));
  e->stream = reinterpret_cast<hipStream_t>(hip_stream);
  return CRL_OK;
}

int crl_set_resident_envs(crl_engine* e, int32_t n_envs) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  if (n_envs < 0) return fail(CRL_E_ARG, "negative env count");
  e->resident_envs = n_envs;
  return CRL_OK;
}

int crl_set_fused_variant(crl_engine* e, int32_t variant) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  if (variant < 0 || variant > 2) return fail(CRL_E_ARG, "variant must be 0 (automatic), 1 or 2");
  e->fused_variant = variant;
  return CRL_OK;
}

int crl_get_fused_split(crl_engine* e, uint32_t* hbm_envs, uint32_t* lds_envs) {
  int rc = check_usable(e);
  if (rc) return rc;
  unsigned v[3] = {0, 0, 0};
  if (e->split_valid) {
    HIP_TRY(hipMemcpyAsync(v, e->split.p, sizeof v, hipMemcpyDeviceToHost, e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));
  }
  if (hbm_envs) *hbm_envs = v[1];
  if (lds_envs) *lds_envs = v[2];
  return CRL_OK;
}

int crl_sync(crl_engine* e) {
  int rc = check_engine(e);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(e->stream));
  return check_persist(e);
}

int crl_set_maps(crl_engine* e, const uint8_t* cell_class, const int32_t* start,
                 const float* cell_reward) {
  return guarded([&] { return set_maps(e, cell_class, start, cell_reward); });
}

int crl_set_cell(crl_engine* e, int32_t map_index, int32_t cell, int32_t cell_class,
                 float cell_reward) {
  return guarded([&] { return set_cell(e, map_index, cell, cell_class, cell_reward); });
}

int crl_reset(crl_engine* e, int32_t first, int32_t count) { return reset_envs(e, first, count); }

int crl_step(crl_engine* e, const int32_t* actions) {
  int rc = check_usable(e);
  if (rc == CRL_OK && actions) rc = refuse_capture(e);
  if (rc) return rc;
  const size_t bytes = (size_t)e->N * 4;
  const int32_t* act = e->act.p;
  int act0 = -1;
  crl::HostSignal sig{};
  crl::StateMirror mirror{};
  crl_engine::InSlot* slot = nullptr;
  if (!actions) {
    if (!e->have_actions) return fail(CRL_E_STATE, "crl_step(NULL) needs a preceding crl_select");
  } else if (e->N == 1) {
    act = nullptr;
    act0 = actions[0];
  } else if (bytes <= kLinkLimitBytes) {
    // the kernel reads the actions where they are put now, and the caller's buffer is free
    rc = claim_in_slot(e, bytes, &slot);
    if (rc) return rc;
    std::memcpy(slot->page, actions, bytes);
    act = reinterpret_cast<const int32_t*>(slot->page);
  } else {
    HIP_TRY(hipMemcpyAsync(e->act.p, actions, bytes, hipMemcpyHostToDevice, e->stream));
    // the host buffer may be reused as soon as we return
    HIP_TRY(hipStreamSynchronize(e->stream));
  }
  // A caller that looks at the state after every step gets it from the step's own kernel
  // instead of from a second launch: 6 us of launch and answer saved, 18 bytes per env
  // over the link added, so it stops with the first step whose state nobody asked for.
  // (Not in a call that a stream capture may record: a replay has no number of its own.)
  rc = state_changes(e);
  if (rc) return rc;
  if (!e->mirror_read) e->mirror_steps = false;
  e->mirror_read = false;
  const bool mirrors = actions && e->mirror_steps && !e->state_shared && e->state_bytes <= kLinkLimitBytes;
  if (mirrors) {
    rc = claim_out_page(e, e->state_bytes);
    if (rc) return rc;
    mirror = state_mirror(e);
  }
  if (slot || mirrors) sig = next_signal(e);
  const int block = e->N <= 64 ? 64 : 256;
  hipLaunchKernelGGL(crl::k_step, dim3((e->N + block - 1) / block), dim3(block), 0, e->stream, e->rules(),
                     e->ptrs(), e->transition(), act, act0, mirror, sig);
  HIP_TRY(hipGetLastError());
  if (slot) slot->last_seq = sig.seq;
  if (mirrors) e->mirror_seq = sig.seq;
  if (e->trace_n > 0 && e->trace_cursor < e->trace_cap) e->trace_cursor += 1;
  e->have_transition = true;
  e->have_actions = false;
  e->stepped = true;
  return CRL_OK;
}

int crl_select(crl_engine* e, int32_t* actions_out) {
  int rc = check_usable(e);
  if (rc == CRL_OK) rc = note_recording(e);
  if (rc) return rc;
  const size_t bytes = (size_t)e->N * 4;
  const bool direct = actions_out && bytes <= kLinkLimitBytes;
  int32_t* host_out = nullptr;
  crl::HostSignal sig{};
  if (direct) {
    rc = claim_out_page(e, bytes);
    if (rc) return rc;
    host_out = reinterpret_cast<int32_t*>(e->out_page.p);
    sig = next_signal(e);
  }
  const dim3 block(e->N <= 64 ? 64 : 256), grid((e->N + block.x - 1) / block.x);
  if (e->A == 4)
    hipLaunchKernelGGL((crl::k_select<4>), grid, block, 0, e->stream, e->rules(), e->ptrs(), e->t, e->act.p,
                       host_out, sig);
  else
    hipLaunchKernelGGL((crl::k_select<8>), grid, block, 0, e->stream, e->rules(), e->ptrs(), e->t, e->act.p,
                       host_out, sig);
  HIP_TRY(hipGetLastError());
  e->have_actions = true;
  if (direct) {
    rc = wait_seq(e, sig.seq);
    if (rc) return rc;
    std::memcpy(actions_out, host_out, bytes);
  } else if (actions_out) {
    HIP_TRY(hipMemcpyAsync(actions_out, e->act.p, bytes, hipMemcpyDeviceToHost, e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));
  }
  return CRL_OK;
}

int crl_update(crl_engine* e) {
  int rc = check_usable(e);
  if (rc) return rc;
  if (!e->have_transition) return fail(CRL_E_STATE, "crl_update needs a preceding crl_step");
  rc = note_recording(e);
  if (rc) return rc;
  const crl::Rules R = e->rules();
  const int grid = (e->N + 255) / 256;
  if (e->cfg.table_mode == CRL_TABLE_PER_ENV) {
    if (e->A == 4)
      hipLaunchKernelGGL((crl::k_update_per_env<4>), dim3(grid), dim3(256), 0, e->stream, R, e->ptrs(),
                         e->transition());
    else
      hipLaunchKernelGGL((crl::k_update_per_env<8>), dim3(grid), dim3(256), 0, e->stream, R, e->ptrs(),
                         e->transition());
    HIP_TRY(hipGetLastError());
  } else {
    const crl::Transition X = e->transition();
    if (e->N <= crl::kSmallSamples) {
      rc = td_small(e, e->Q.p, X, e->N, nullptr, crl::HostSignal{});
    } else {
      TdPlan p;
      rc = td_begin(e, e->N, &p);
      if (rc == CRL_OK) rc = td_piece(e, p, e->Q.p, X, 0, e->N, crl::HostSignal{});
      if (rc == CRL_OK) rc = td_end(e, p, e->Q.p, crl::HostSignal{});
    }
    if (rc) return rc;
  }
  e->have_transition = false;
  e->t += 1;
  return CRL_OK;
}

int crl_td_update(crl_engine* e, int32_t table, int32_t n, const int32_t* s, const int32_t* a,
                  const float* r, const int32_t* s_next, const uint8_t* done) {
  return td_update(e, table, n, s, a, r, s_next, done, nullptr, nullptr);
}

int crl_td_update_collect(crl_engine* e, int32_t table, int32_t n, const int32_t* s, const int32_t* a,
                          const float* r, const int32_t* s_next, const uint8_t* done, int32_t* keys,
                          float* values) {
  if (n > crl::kSmallSamples) return fail(CRL_E_RANGE, "%d samples, at most %d are collected", n, crl::kSmallSamples);
  if (n > 0 && (!keys || !values)) return fail(CRL_E_ARG, "null output array");
  return td_update(e, table, n, s, a, r, s_next, done, keys, values);
}

int crl_run_fused(crl_engine* e, int32_t n_steps) { return run_fused(e, n_steps, false); }

int crl_run_fused_noalloc(crl_engine* e, int32_t n_steps) { return run_fused(e, n_steps, true); }

int crl_get_state(crl_engine* e, int32_t* s, float* reward, uint8_t* done, uint8_t* action,
                  int32_t* ep_step, int32_t* episode) {
  int rc = check_usable(e);
  if (rc) return rc;
  const size_t N = (size_t)e->N;
  if (e->state_bytes <= kLinkLimitBytes) {
    if (e->mirror_seq != 0) {
      rc = wait_seq(e, e->mirror_seq);
      if (rc == CRL_OK) rc = check_persist(e);
    } else {
      // A caller that reads the statistics after the state (a training loop, chunk after chunk) gets both with one launch:
      // 7 us of a second launch and its answer saved, 16 bytes per env over the link added, so it stops with the first state
      // whose statistics nobody asked for.  (One env, 500 steps, state, statistics 77.5 -> 70.3 us; 4096 100.3 -> 92.6.)
      const size_t more = e->stats_follow && !e->state_shared && e->state_bytes + e->stats_bytes <= kLinkLimitBytes ? e->stats_bytes : 0;
      rc = fetch_pinned(e, e->state_at, e->state_bytes + more);
      e->stats_here = rc == CRL_OK && more != 0;
      if (rc == CRL_OK && e->stepped) e->mirror_steps = true;
    }
    if (rc) return rc;
    e->state_read = true;
    e->stats_follow = false;
    e->mirror_read = true;
    const crl::StateMirror M = state_mirror(e);
    if (s) std::memcpy(s, M.s, N * 4);
    if (reward) std::memcpy(reward, M.reward, N * 4);
    if (done) std::memcpy(done, M.done, N);
    if (action) std::memcpy(action, M.action, N);
    if (ep_step) std::memcpy(ep_step, M.ep_step, N * 4);
    if (episode) std::memcpy(episode, M.episode, N * 4);
    return CRL_OK;
  }
  if (s) HIP_TRY(hipMemcpyAsync(s, e->s.p, N * 4, hipMemcpyDeviceToHost, e->stream));
  if (reward) HIP_TRY(hipMemcpyAsync(reward, e->reward.p, N * 4, hipMemcpyDeviceToHost, e->stream));
  if (done) HIP_TRY(hipMemcpyAsync(done, e->done.p, N, hipMemcpyDeviceToHost, e->stream));
  if (action) HIP_TRY(hipMemcpyAsync(action, e->action.p, N, hipMemcpyDeviceToHost, e->stream));
  if (ep_step) HIP_TRY(hipMemcpyAsync(ep_step, e->ep_step.p, N * 4, hipMemcpyDeviceToHost, e->stream));
  if (episode) HIP_TRY(hipMemcpyAsync(episode, e->episode.p, N * 4, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return check_persist(e);
}

int crl_set_state(crl_engine* e, const int32_t* s, const int32_t* ep_step, const int32_t* episode) {
  int rc = check_engine(e);
  if (rc) return rc;
  rc = clear_persist_failure(e);
  if (rc) return rc;
  rc = state_changes(e);
  if (rc) return rc;
  const size_t N = (size_t)e->N;
  if (s) {
    for (int i = 0; i < e->N; ++i)
      if (s[i] < 0 || (size_t)s[i] >= e->S) return fail(CRL_E_RANGE, "s[%d] = %d outside [0,%zu)", i, s[i], e->S);
    HIP_TRY(hipMemcpyAsync(e->s.p, s, N * 4, hipMemcpyHostToDevice, e->stream));
  }
  if (ep_step) HIP_TRY(hipMemcpyAsync(e->ep_step.p, ep_step, N * 4, hipMemcpyHostToDevice, e->stream));
  if (episode) HIP_TRY(hipMemcpyAsync(e->episode.p, episode, N * 4, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  e->have_transition = false;
  e->have_actions = false;
  return CRL_OK;
}

int crl_get_episode_stats(crl_engine* e, float* last_return, int32_t* last_length, float* return_sum,
                          int32_t* length_sum) {
  int rc = check_usable(e);
  if (rc) return rc;
  if (!e->cfg.track_returns) return fail(CRL_E_STATE, "the engine was created without track_returns");
  const size_t b = (size_t)e->N * 4;
  if (e->stats_bytes <= kLinkLimitBytes) {
    const unsigned char* at = e->out_page.p + e->state_bytes;
    if (!e->stats_here) {
      rc = fetch_pinned(e, e->stats_at, e->stats_bytes);
      if (rc) return rc;
      at = e->out_page.p;
    }
    e->stats_here = false;
    e->stats_follow = e->state_read;
    auto out = [&](void* to, const void* from) {
      if (to) std::memcpy(to, at + (static_cast<const unsigned char*>(from) - e->stats_at), b);
    };
    out(last_return, e->ret_last.p);
    out(last_length, e->len_last.p);
    out(return_sum, e->ret_sum.p);
    out(length_sum, e->len_sum.p);
    return CRL_OK;
  }
  if (last_return) HIP_TRY(hipMemcpyAsync(last_return, e->ret_last.p, b, hipMemcpyDeviceToHost, e->stream));
  if (last_length) HIP_TRY(hipMemcpyAsync(last_length, e->len_last.p, b, hipMemcpyDeviceToHost, e->stream));
  if (return_sum) HIP_TRY(hipMemcpyAsync(return_sum, e->ret_sum.p, b, hipMemcpyDeviceToHost, e->stream));
  if (length_sum) HIP_TRY(hipMemcpyAsync(length_sum, e->len_sum.p, b, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return CRL_OK;
}

int crl_get_step_count(crl_engine* e, uint64_t* t) {
  if (!e || !t) return fail(CRL_E_ARG, "null argument");
  *t = e->t;
  return CRL_OK;
}

int crl_set_step_count(crl_engine* e, uint64_t t) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  e->t = t;
  return CRL_OK;
}

int crl_q_get_range(crl_engine* e, int32_t first_table, int32_t count, float* out) {
  int rc = check_usable(e);
  if (rc) return rc;
  if (!out) return fail(CRL_E_ARG, "out is null");
  if (first_table < 0 || count < 0 || (int64_t)first_table + count > e->n_tables)
    return fail(CRL_E_RANGE, "table range [%d,%d) outside [0,%d)", first_table, first_table + count, e->n_tables);
  const size_t bytes = (size_t)count * e->K * sizeof(float);
  if (bytes > 0 && bytes <= kLinkLimitBytes) {  // (K is a multiple of 4: 16-byte words)
    rc = fetch_pinned(e, e->Q.p + (size_t)first_table * e->K, bytes);
    if (rc) return rc;
    std::memcpy(out, e->out_page.p, bytes);
    return CRL_OK;
  }
  HIP_TRY(hipMemcpyAsync(out, e->Q.p + (size_t)first_table * e->K, bytes, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return check_persist(e);
}

int crl_q_get(crl_engine* e, int32_t table, float* out) { return crl_q_get_range(e, table, 1, out); }

int crl_q_set(crl_engine* e, int32_t table, const float* in) {
  int rc = check_engine(e);
  if (rc) return rc;
  rc = clear_persist_failure(e);
  if (rc) return rc;
  if (!in) return fail(CRL_E_ARG, "in is null");
  if (table < 0 || table >= e->n_tables) return fail(CRL_E_RANGE, "table %d outside [0,%d)", table, e->n_tables);
  HIP_TRY(hipMemcpyAsync(e->Q.p + (size_t)table * e->K, in, e->K * sizeof(float), hipMemcpyHostToDevice,
                         e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return CRL_OK;
}

int crl_set_trace(crl_engine* e, int32_t n_envs, int32_t max_steps) {
  int rc = check_engine(e);
  if (rc) return rc;
  if (n_envs < 0 || n_envs > e->N || max_steps < 0) return fail(CRL_E_ARG, "bad trace size");
  HIP_TRY(hipStreamSynchronize(e->stream));
  e->trace_n = 0;
  e->trace_cap = 0;
  e->trace_cursor = 0;
  if (n_envs == 0 || max_steps == 0) return CRL_OK;
  const size_t cells = (size_t)n_envs * max_steps;
  hipError_t h = hipSuccess;
  auto acc = [&](hipError_t x) {
    if (h == hipSuccess) h = x;
  };
  acc(e->grow(e->trace_s, cells));
  acc(e->grow(e->trace_a, cells));
  acc(e->grow(e->trace_r, cells));
  acc(e->grow(e->trace_d, cells));
  if (h != hipSuccess) return fail(CRL_E_ALLOC, "trace allocation failed: %s", hipGetErrorString(h));
  e->trace_n = n_envs;
  e->trace_cap = max_steps;
  return CRL_OK;
}

int crl_get_trace(crl_engine* e, int32_t n_steps, int32_t* s_next, uint8_t* action, float* reward,
                  uint8_t* done) {
  int rc = check_usable(e);
  if (rc) return rc;
  if (n_steps < 0 || n_steps > e->trace_cursor)
    return fail(CRL_E_RANGE, "%d steps asked, %d recorded", n_steps, e->trace_cursor);
  const size_t cells = (size_t)n_steps * e->trace_n;
  if (cells == 0) return CRL_OK;
  if (s_next) HIP_TRY(hipMemcpyAsync(s_next, e->trace_s.p, cells * 4, hipMemcpyDeviceToHost, e->stream));
  if (action) HIP_TRY(hipMemcpyAsync(action, e->trace_a.p, cells, hipMemcpyDeviceToHost, e->stream));
  if (reward) HIP_TRY(hipMemcpyAsync(reward, e->trace_r.p, cells * 4, hipMemcpyDeviceToHost, e->stream));
  if (done) HIP_TRY(hipMemcpyAsync(done, e->trace_d.p, cells, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  return check_persist(e);
}

int crl_set_persist_spin_limit(crl_engine* e, int32_t polls) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  if (polls < 1) return fail(CRL_E_ARG, "at least one poll");
  e->persist_spin_limit = polls;
  return CRL_OK;
}

int crl_set_exploration_stream(crl_engine* e, int32_t n_steps, const float* u, const int32_t* a_rand) {
  int rc = check_engine(e);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(e->stream));
  e->sup_n = 0;
  if (!u || n_steps <= 0) return CRL_OK;
  if (!a_rand) return fail(CRL_E_ARG, "a_rand is null");
  const size_t cells = (size_t)n_steps * e->N;
  for (size_t i = 0; i < cells; ++i)
    if (a_rand[i] < 0 || a_rand[i] >= e->A) return fail(CRL_E_RANGE, "a_rand[%zu] = %d outside [0,%d)", i, a_rand[i], e->A);
  hipError_t h = e->grow(e->u_sup, cells);
  if (h == hipSuccess) h = e->grow(e->a_sup, cells);
  if (h != hipSuccess) return fail(CRL_E_ALLOC, "stream allocation failed: %s", hipGetErrorString(h));
  HIP_TRY(hipMemcpyAsync(e->u_sup.p, u, cells * 4, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(hipMemcpyAsync(e->a_sup.p, a_rand, cells * 4, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(hipStreamSynchronize(e->stream));
  e->sup_t0 = e->t;
  e->sup_n = n_steps;
  return CRL_OK;
}

int crl_device_ptr(crl_engine* e, int32_t which, void** out) {
  if (!e || !out) return fail(CRL_E_ARG, "null argument");
  switch (which) {
    case CRL_PTR_S: *out = e->s.p; break;
    case CRL_PTR_EP_STEP: *out = e->ep_step.p; break;
    case CRL_PTR_EPISODE: *out = e->episode.p; break;
    case CRL_PTR_REWARD: *out = e->reward.p; break;
    case CRL_PTR_DONE: *out = e->done.p; break;
    case CRL_PTR_ACTION: *out = e->action.p; break;
    case CRL_PTR_Q: *out = e->Q.p; break;
    default: return fail(CRL_E_ARG, "unknown pointer id %d", which);
  }
  if (which != CRL_PTR_Q) {  // the caller may write through it from now on
    e->state_shared = true;
    e->mirror_seq = 0;
    e->stats_here = false;
  }
  return CRL_OK;
}

int crl_fused_kernel_info(crl_engine* e, int32_t n_steps, char* name, size_t name_len, int32_t* grid,
                          int32_t* block, int32_t* lds_bytes) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  if (e->cfg.table_mode == CRL_TABLE_PER_ENV) {
    const FusedPlan p = plan_fused(e, n_steps > 0 ? n_steps : 1 << 20);  // <= 0: a long launch
    if (name && name_len) snprintf(name, name_len, "%s", p.name);
    if (grid) *grid = p.grid;
    if (block) *block = p.block;
    if (lds_bytes) *lds_bytes = (int32_t)p.lds;
  } else {
    const PersistPlan pp = plan_persist(e, n_steps > 0 ? n_steps : 1 << 20);
    if (pp.ok) {
      if (name && name_len) snprintf(name, name_len, "k_shared_persist<%d,%d%s%s>", e->A, pp.lds_map ? 1 : 2,
                                      pp.fold ? ",folded" : "", pp.hashed ? ",hashed" : "");
      if (grid) *grid = pp.grid;
      if (block) *block = 256;
      if (lds_bytes) *lds_bytes = (int32_t)pp.lds;
      return CRL_OK;
    }
    SharedPlan sp{};
    const int rc = plan_shared_step(e, &sp);
    if (rc) return rc;
    if (name && name_len) snprintf(name, name_len, sp.two ? "k_shared_act+k_reduce_owners" : "k_shared_act+k_reduce_scan");
    if (grid) *grid = (e->N + 255) / 256;  // (of the first of the two)
    if (block) *block = 256;
    if (lds_bytes) *lds_bytes = (int32_t)sp.lds;
  }
  return CRL_OK;
}

static int plan_for_config(const crl_config* cfg, int32_t n_steps, FusedPlan* p) {
  int rc = crl::validate_config(cfg, crl::last_error());
  if (rc != CRL_OK) return rc;
  if (cfg->table_mode != CRL_TABLE_PER_ENV) return fail(CRL_E_ARG, "only per-env tables have a fused launch plan");
  crl_engine shell;  // sizes only: nothing is allocated and no device is touched
  set_geometry(&shell, *cfg);
  *p = plan_fused(&shell, n_steps > 0 ? n_steps : 1 << 20);
  return CRL_OK;
}

int crl_fused_plan_rows_for_config(const crl_config* cfg, int32_t n_steps, int32_t* rows, int32_t* codes) {
  FusedPlan p;
  int rc = plan_for_config(cfg, n_steps, &p);
  if (rc != CRL_OK) return rc;
  if (rows) *rows = p.rows;
  if (codes) *codes = p.moves ? 1 : 0;
  return CRL_OK;
}

int crl_fused_plan_for_config(const crl_config* cfg, int32_t n_steps, char* name, size_t name_len,
                              int32_t* grid, int32_t* block, int32_t* lds_bytes) {
  FusedPlan p;
  int rc = plan_for_config(cfg, n_steps, &p);
  if (rc != CRL_OK) return rc;
  if (name && name_len) snprintf(name, name_len, "%s", p.name);
  if (grid) *grid = p.grid;
  if (block) *block = p.block;
  if (lds_bytes) *lds_bytes = (int32_t)p.lds;
  if (p.grid < 1 || p.block < 64 || p.block > 1024 || p.lds > kLdsPerWorkgroup)
    return fail(CRL_E_STATE, "launch plan %s: grid %d, block %d, %zu bytes of LDS", p.name, p.grid, p.block, p.lds);
  return CRL_OK;
}

// Diagnostics: arms (or disarms) the phase clocks of the one-launch shared-table kernel.
// Armed, the instantiation that reads the shader clock eight times per step runs.
int crl_set_persist_clocks(crl_engine* e, int32_t on) {
  if (!e) return fail(CRL_E_ARG, "null engine");
  e->persist_clocks = on != 0;
  return CRL_OK;
}

// Diagnostics: what the last one-launch shared-table launch that ran with the clocks armed
// left behind (layout: include/crl.h); at most n_words 64-bit words are copied.
int crl_get_persist_clocks(crl_engine* e, uint64_t* out, size_t n_words) {
  int rc = check_engine(e);
  if (rc) return rc;
  if (!out) return fail(CRL_E_ARG, "out is null");
  if (!e->pdiag.p) return fail(CRL_E_STATE, "this engine has no shared table");
  HIP_TRY(hipStreamSynchronize(e->stream));
  rc = check_persist(e);
  if (rc) return rc;
  const size_t n = std::min<size_t>(n_words, crl::kPersistClockWords);
  HIP_TRY(hipMemcpy(out, e->pdiag.p + 1, n * sizeof(uint64_t), hipMemcpyDeviceToHost));
  return CRL_OK;
}

// Measurement helper: nanoseconds per barrier over `n_groups` co-resident workgroups
// built from device-scope loads and stores (pattern: see k_probe_barrier).
int crl_probe_barrier(int pattern, int n_groups, int rounds, double* ns_per_barrier) {
  if (pattern < 0 || pattern > 2 || n_groups < 1 || n_groups > crl::kPersistMaxGroups || rounds < 1 || !ns_per_barrier)
    return fail(CRL_E_ARG, "pattern 0..2, 1..%d workgroups, rounds >= 1", crl::kPersistMaxGroups);
  const size_t words = (size_t)(17 + crl::kPersistMaxGroups) * crl::kProbeLine;
  DevBuf<unsigned> mem;
  DevBuf<unsigned long long> out;
  if (mem.alloc(words) != hipSuccess || out.alloc(2) != hipSuccess) return fail(CRL_E_ALLOC, "probe allocation failed");
  HIP_TRY(hipMemset(mem.p, 0, words * sizeof(unsigned)));
  HIP_TRY(hipMemset(out.p, 0, 2 * sizeof(unsigned long long)));
  unsigned* m = mem.p;
  unsigned long long* o = out.p;
  void* args[] = {&m, &rounds, &o};
  const void* kern = pattern == 0   ? reinterpret_cast<const void*>(&crl::k_probe_barrier<0>)
                     : pattern == 1 ? reinterpret_cast<const void*>(&crl::k_probe_barrier<1>)
                                    : reinterpret_cast<const void*>(&crl::k_probe_barrier<2>);
  // co-resident or refused: the workgroups wait for each other
  HIP_TRY(hipLaunchCooperativeKernel(kern, dim3(n_groups), dim3(256), args, 0, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  unsigned long long h[2];
  HIP_TRY(hipMemcpy(h, out.p, sizeof h, hipMemcpyDeviceToHost));
  if (h[1]) return fail(CRL_E_DEVICE, "%llu workgroups gave up waiting", h[1]);
  *ns_per_barrier = (double)h[0] * 10.0 / rounds;  // 100 MHz ticks
  return CRL_OK;
}


int crl_probe_copy(size_t n_bytes, int repeats) {
  if (n_bytes == 0 || n_bytes % 16 != 0 || repeats < 1) return fail(CRL_E_ARG, "n_bytes must be a positive multiple of 16");
  DevBuf<uint8_t> src, dst;
  if (src.alloc(n_bytes) != hipSuccess || dst.alloc(n_bytes) != hipSuccess)
    return fail(CRL_E_ALLOC, "probe allocation failed");
  HIP_TRY(hipMemset(src.p, 1, n_bytes));
  HIP_TRY(hipMemset(dst.p, 0, n_bytes));
  const size_t n16 = n_bytes / 16;
  for (int i = 0; i < repeats; ++i)
    hipLaunchKernelGGL(crl::k_probe_copy, dim3(256 * 16), dim3(256), 0, nullptr,
                       reinterpret_cast<const uint4*>(src.p), reinterpret_cast<uint4*>(dst.p), n16);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipDeviceSynchronize());
  // the copy arrived: both ends of the destination hold the source's pattern
  uint8_t ends[2][256];
  const size_t tail = n_bytes >= sizeof ends[0] ? n_bytes - sizeof ends[0] : 0;
  const size_t len = n_bytes >= sizeof ends[0] ? sizeof ends[0] : n_bytes;
  HIP_TRY(hipMemcpy(ends[0], dst.p, len, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(ends[1], dst.p + tail, len, hipMemcpyDeviceToHost));
  for (size_t i = 0; i < len; ++i)
    if (ends[0][i] != 1 || ends[1][i] != 1) return fail(CRL_E_DEVICE, "copy kernel left byte %zu unwritten", i);
  return CRL_OK;
}

}  // extern "C"
