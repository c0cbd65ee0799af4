// Deterministic ordered reduction of TD deltas that hit the same (s,a) key of
// one table - the replacement for float atomics.  Samples (envs) are taken in
// index order through a fixed three-level tree:
//
//   block  = 256 consecutive samples, added left to right from +0.0f
//   group  = 16 consecutive blocks, block sums added left to right from +0.0f
//   total  = group sums added left to right from +0.0f;   Q[k] = Q[k] + total[k]
//
// Two passes over the chip:
//   1. one workgroup per block: the lowest thread that holds a key becomes the
//      key's leader (LDS atomic min on a table of keys), the other holders mark
//      themselves in the leader's 256-bit member set (LDS atomic or) and line
//      their deltas up by their place in it, and the leader adds them in that
//      order = thread order = sample order; every distinct key's block sum goes
//      to the workgroup that owns the key;
//   2. one workgroup per owner of keys adds the block sums it was handed, a wave
//      to a group, and then the groups.
// Up to 1024 samples (four blocks, one group) are one workgroup's work and one launch.
// Empty blocks add +0.0f, which changes nothing, so the result is a pure
// function of (keys, deltas) whatever the occupancy.
#pragma once
#include "crl_device.h"

namespace crl {

constexpr int kBlockSamples = 256;   // level 0
constexpr int kGroupBlocks = 16;     // level 1
constexpr int kOwnKeys = 64;         // one-launch kernel, dense form: keys per owner workgroup, 64 / A whole table rows
constexpr int kOwnKeysHashed = 512;  // ... hashed form
constexpr int kMaxOwnKeys = 1024;    // two launches: keys per owner at most
constexpr int kMaxOwners = 4096;     // ... and owners
constexpr int kSlotOverflow = 127;   // count value: more distinct keys than records, read the block's raw samples instead
constexpr int kStagePieces = 512;    // 16-byte pieces of the main halves of one block's cells in the one-launch kernel
constexpr int kDenseKeys = 16384;    // one-launch kernel, dense form: keys of its LDS table, one entry per key
constexpr int kHashSlots = 2048;     // hashed form, two launches: entries of the LDS table of the keys a block holds
constexpr int kTileBlocks = 256;     // blocks per LDS tile of pass 2
constexpr uint32_t kOwnerMix = 37;   // odd: spreads cells a power of two apart over owners
constexpr uint32_t kNoLead = 0xFFFFFFFFu;

// A hand-off record is 64 bits, written and read as one unit.  One-launch kernel, dense /
// hashed form (owners of up to 64 / 512 keys):
//   bits  0..5  / 0..8    slot of the key among its owner's
//   bits  6..12 / 9..15   record 0 of a cell only: how many records the cell holds
//                         (0: none, kSlotOverflow: more distinct keys than the cell has records)
//   bits 13..31 / 16..31  step tag (a record is valid once its tag is the step's)
//   bits 32..63           the block sum, fp32
template <bool HASHED>
struct Rec {
  static constexpr int kCountShift = HASHED ? 9 : 6, kTagShift = kCountShift + 7;
  static constexpr uint32_t kTagMask = (1u << (32 - kTagShift)) - 1u;
  static __device__ __forceinline__ unsigned long long make(uint32_t slot, uint32_t tag, float v) {
    return (unsigned long long)(slot | (tag << kTagShift)) | ((unsigned long long)__float_as_uint(v) << 32);
  }
  static __device__ __forceinline__ int slot(uint32_t meta) { return (int)(meta & ((1u << kCountShift) - 1u)); }
  static __device__ __forceinline__ int count(uint32_t meta) { return (int)((meta >> kCountShift) & 127u); }
};
static_assert(kOwnKeys == 1 << Rec<false>::kCountShift && kOwnKeysHashed == 1 << Rec<true>::kCountShift, "a record's slot");
// Two launches: slot in bits 0..15, count in bits 16..22, no tag.
__device__ __forceinline__ unsigned long long make_wide_rec(uint32_t slot, uint32_t count, float v) {
  return (unsigned long long)(slot | (count << 16)) | ((unsigned long long)__float_as_uint(v) << 32);
}
__device__ __forceinline__ int wide_slot(uint32_t meta) { return (int)(meta & 0xffffu); }
__device__ __forceinline__ int wide_count(uint32_t meta) { return (int)(meta >> 16); }
static_assert(kMaxOwnKeys <= 0x10000, "a record's slot has 16 bits");

struct ReduceGeom {
  int K;          // keys of the table, key = cell * A + action
  int a_shift;    // log2(A)
  int own_shift;  // log2(number of owners); an owner has (whole rows of) K >> own_shift keys or a row more
  int n_blocks;   // ceil(n / 256)
  int cell_shift; // log2(records of a hand-off cell), cell_shift_for(own_shift)
  int main_shift; // one-launch kernel: log2(records in the part of a cell that is written every step), main_shift_for()
};

// Records per hand-off cell.  A block's 256 samples spread over the owners, so a cell
// sees about 256 / owners distinct keys: eight records for 256 owners (more than eight
// keys once in a million cells), more where fewer owners share the samples, and all 64
// keys an owner has from 16 owners down, where a cell cannot overflow at all.  A block's
// cells together stay within 16 KB.
__host__ __device__ constexpr int cell_shift_for(int own_shift) {
  return own_shift >= 8 ? 3 : own_shift >= 6 ? 4 : own_shift == 5 ? 5 : 6;
}

// One-launch kernel: what a block's cell stores cost grows with their bytes (16 KB of
// cells of eight records for 256 owners, seven eighths of them padding, need 1.4 us to be
// acknowledged, 8 KB half of that).  So with more than 64 owners a cell is two halves:
// the main half, written whole every step with all the others of the block (8 KB), and
// an extension of as many records that only a block with more distinct keys for that
// owner than the main half holds writes into (one cell in 270 with 256 owners), record by
// record.  Record 0 of the main half says how many records there are in all.  The
// extensions lie [owner][block]: an owner asks for all of them with its main halves,
// 8 KB in one piece, and looks at those the counts point to.
__host__ __device__ constexpr int main_shift_for(int own_shift) {
  const int c = cell_shift_for(own_shift), m = 10 - own_shift;
  return m < c ? (m < 2 ? 2 : m) : c;
}

// key <-> (owner, slot among the owner's).  An owner holds whole table rows:
// hi = cell >> own_shift, owner = (cell + 37 * hi) mod owners, slot = hi * A + action
__device__ __forceinline__ int owner_of(int key, const ReduceGeom& G) {
  const uint32_t mask = (1u << G.own_shift) - 1u;
  const uint32_t cell = (uint32_t)key >> G.a_shift;
  return (int)((cell + kOwnerMix * (cell >> G.own_shift)) & mask);
}
__device__ __forceinline__ int slot_of(int key, const ReduceGeom& G) {
  const uint32_t cell = (uint32_t)key >> G.a_shift;
  return (int)(((cell >> G.own_shift) << G.a_shift) | ((uint32_t)key & ((1u << G.a_shift) - 1u)));
}
__device__ __forceinline__ int key_of(int owner, int slot, const ReduceGeom& G) {
  const uint32_t mask = (1u << G.own_shift) - 1u;
  const uint32_t hi = (uint32_t)slot >> G.a_shift;
  const uint32_t lo = ((uint32_t)owner - kOwnerMix * hi) & mask;
  const uint32_t cell = (hi << G.own_shift) | lo;
  return (int)((cell << G.a_shift) | ((uint32_t)slot & ((1u << G.a_shift) - 1u)));
}

// ---- device-scope accesses --------------------------------------------------------
// gfx950 has eight XCDs, each with its own L2; plain loads and stores are coherent
// inside one XCD only.  Relaxed atomic loads and stores at agent scope compile to
// accesses that carry the sc1 bit and are served past the L2: a value stored that
// way by one workgroup is seen by the next such load of any other, without the
// whole-L2 write-back / invalidate of a release / acquire fence.  64 bits is the
// unit: every exchanged datum carries its own step tag in the same 64 bits, so no
// ordering between two stores is ever relied on.
__device__ __forceinline__ void st_dev64(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_dev64(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev32(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ld_dev32(const unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Aligned 16-byte device-scope loads: a buffer load with the sc1 bit, through a window
// (buffer descriptor) that starts at `base` and spans 2 GB.  Each aligned 64-bit half is
// one of the tagged units above; nothing is assumed about the two halves of a load
// belonging together.  To the compiler this is an ordinary read of memory: a loop that
// asks again and again must call poll_fence() in every round, or the load is taken out
// of the loop as invariant.
typedef unsigned int crl_u4 __attribute__((ext_vector_type(4)));
using DevWindow = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ DevWindow dev_window(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ uint4 ld_dev128(DevWindow w, uint32_t byte_offset) {
  const crl_u4 v = __builtin_amdgcn_raw_buffer_load_b128(w, (int)byte_offset, 0, 16 /* sc1 */);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st_dev128(DevWindow w, uint32_t byte_offset, const uint4 v) {
  crl_u4 t;
  t.x = v.x;
  t.y = v.y;
  t.z = v.z;
  t.w = v.w;
  __builtin_amdgcn_raw_buffer_store_b128(t, w, (int)byte_offset, 0, 16 /* sc1 */);
}
// store_host() for 16 bytes
__device__ __forceinline__ void store_host128(DevWindow w, uint32_t byte_offset, const uint4 v) {
  crl_u4 t;
  t.x = v.x;
  t.y = v.y;
  t.z = v.z;
  t.w = v.w;
  __builtin_amdgcn_raw_buffer_store_b128(t, w, (int)byte_offset, 0, 17 /* sc0 sc1 */);
}
__device__ __forceinline__ void poll_fence() { asm volatile("" ::: "memory"); }

// `Entries` = entries of the table in which the leader of a key is found: one per key of
// the table, or (kHashSlots) one per distinct key of the block, found by hashing.
template <int Entries>
struct alignas(16) ReduceLdsT {  // (lead and members are also accessed 16 bytes at a time)
  alignas(16) uint32_t lead[Entries];                        // lowest thread of the block that holds the key; kNoLead between uses
  alignas(16) unsigned long long members[kBlockSamples][4];  // per leader: the threads that hold its key; zero between uses
  float delta[kBlockSamples];
  int handed[256];                               // block sums handed to each owner (one-launch kernel)
  int over;                                      // some owner was handed more than a cell holds
  int none;                                      // (written by the others; nobody reads it)
};

// The same where each key of the table has its place: a cell's lowest thread is found before the actions are
// chosen, while the step before is under way (cell_sums), and the holders of its A keys have a set each, by
// that thread's number.
template <int A>
struct alignas(16) CellReduceLds {
  static constexpr int kCells = kDenseKeys / A;
  alignas(16) uint32_t lead[kCells];                             // lowest thread of the block in the cell; kNoLead between uses
  alignas(16) unsigned long long members[kBlockSamples * A][4];  // [lead][action]; zero between uses
  float delta[kBlockSamples];
  int handed[256];
  int over;
  int none;
};

// Besides ReduceLds, reduce_block() needs kSortBytes of LDS for `sorted`: the deltas of a
// key's further holders, lined up for its leader ([place among the holders][leader]).
constexpr int kSortRows = 32;
constexpr size_t kSortBytes = (size_t)kSortRows * kBlockSamples * sizeof(float);

// Once per kernel, before the first reduce_block() and separated from it by a barrier.
template <int Entries>
__device__ __forceinline__ void reduce_block_init(ReduceLdsT<Entries>& L) {
  const int tid = threadIdx.x;
  uint4* lead4 = reinterpret_cast<uint4*>(L.lead);
  for (int i = tid; i < Entries / 4; i += kBlockSamples) lead4[i] = make_uint4(kNoLead, kNoLead, kNoLead, kNoLead);
  L.members[tid][0] = 0ull;
  L.members[tid][1] = 0ull;
  L.members[tid][2] = 0ull;
  L.members[tid][3] = 0ull;
  if (tid == 0) L.over = 0;
}

// acc and the deltas of a leader's further holders (those in mw), in thread order = sample order
__device__ __forceinline__ float add_holders(const float* delta, const float* sorted, const unsigned long long (&mw)[4], const int holders,
                                             float acc) {
  const int tid = threadIdx.x;
  const int lined = holders < kSortRows ? holders : kSortRows;
  for (int r0 = 0; r0 < lined; r0 += 4) {
    float d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = sorted[(r0 + i < kSortRows ? r0 + i : kSortRows - 1) * kBlockSamples + tid];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r0 + i < lined) acc = acc + d[i];
  }
  if (holders > kSortRows) {  // more holders than places: the rest one by one
    int seen = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      unsigned long long m = mw[w];
      while (m != 0ull) {
        const int j = __builtin_ctzll(m);
        if (seen >= kSortRows) acc = acc + delta[w * 64 + j];
        ++seen;
        m &= m - 1ull;
      }
    }
  }
  return acc;
}

// What both forms of pass 1 share: the ordered sum of each distinct key of a block, in its
// leader.  All 256 threads call it with their sample (valid = false: none); `at` is the
// key's entry of L.lead, where the caller has entered its thread with an atomic min.  On
// return (behind a barrier that only the last lines of the function follow) *sum is the
// leader's block sum.  L.lead[at] and the leader's member set are as they were used: who calls
// it again clears them first, when nobody waits for it.  -> whether this thread is a leader.
// (Written without branches: one wave to a SIMD has nothing to hide them behind.  A thread
// without a sample reads its own, empty member set; a thread that has nothing to line up
// writes its delta where it already is.)
template <int Entries, class Between>
__device__ __forceinline__ bool block_sums(ReduceLdsT<Entries>& L, const int at, const float delta, const bool valid,
                                           float* sorted, Between between, float* sum) {
  const int tid = threadIdx.x;
  L.delta[tid] = delta;
  __syncthreads();
  between();  // (what the last call left to its readers: they are past the barrier above)
  uint32_t ld = (uint32_t)tid;
  if (valid) {
    ld = L.lead[at];
    if (ld != (uint32_t)tid) atomicOr(&L.members[ld][tid >> 6], 1ull << (tid & 63));
  }
  __syncthreads();
  // A key's sum is its samples' deltas added in thread order, one after the other: the
  // leader has to walk through them.  Every further holder finds its place among them
  // (the set bits below its own) and puts its delta there, all at once, so that the
  // leader's walk is loads from known addresses, several in flight, instead of one bit
  // scan, load and add after the other (envs that crowd on a few cells: 14 holders of
  // one key in most blocks, 1 us of such a walk).
  const bool leader = valid && ld == (uint32_t)tid;
  unsigned long long mw[4];
  int holders;  // leader: the key's further holders
  {
    const ulonglong2 lo = *reinterpret_cast<const ulonglong2*>(&L.members[ld][0]);
    const ulonglong2 hi = *reinterpret_cast<const ulonglong2*>(&L.members[ld][2]);
    mw[0] = lo.x;
    mw[1] = lo.y;
    mw[2] = hi.x;
    mw[3] = hi.y;
    const int p0 = __popcll(mw[0]), p1 = __popcll(mw[1]), p2 = __popcll(mw[2]), p3 = __popcll(mw[3]);
    holders = leader ? p0 + p1 + p2 + p3 : 0;
    const int w = tid >> 6;
    const unsigned long long mine = w == 0 ? mw[0] : w == 1 ? mw[1] : w == 2 ? mw[2] : mw[3];
    const int place = (w > 0 ? p0 : 0) + (w > 1 ? p1 : 0) + (w > 2 ? p2 : 0) + __popcll(mine & ((1ull << (tid & 63)) - 1ull));
    const bool lines_up = valid && !leader && place < kSortRows;
    *(lines_up ? &sorted[place * kBlockSamples + (int)ld] : &L.delta[tid]) = delta;
  }
  __syncthreads();
  float acc = 0.0f;
  if (leader) {
    acc = acc + delta;  // the leader is the key's first sample; the other holders come after it
    if (holders != 0) acc = add_holders(L.delta, sorted, mw, holders, acc);
  }
  *sum = acc;
  return leader;
}

template <int A>
__device__ __forceinline__ void reduce_block_init(CellReduceLds<A>& L) {
  const int tid = threadIdx.x;
  uint4* lead4 = reinterpret_cast<uint4*>(L.lead);
  for (int i = tid; i < CellReduceLds<A>::kCells / 4; i += kBlockSamples) lead4[i] = make_uint4(kNoLead, kNoLead, kNoLead, kNoLead);
  for (int i = tid; i < kBlockSamples * A; i += kBlockSamples) {
    *reinterpret_cast<ulonglong2*>(&L.members[i][0]) = make_ulonglong2(0ull, 0ull);
    *reinterpret_cast<ulonglong2*>(&L.members[i][2]) = make_ulonglong2(0ull, 0ull);
  }
  if (tid == 0) L.over = 0;
}

// block_sums() where the threads of a cell know the lowest of them: all of a key's holders have entered themselves in
// `set` = lead * A + action, and a barrier later each of them sees its place, the first of them that it leads - one
// barrier and two trips to LDS fewer than finding the key's lowest thread first.  What makes it pay is that nothing else is done between
// the barriers: 65,536 envs, 200 steps, 64x64x4 / 32x32x4 1357 / 1267 us with keys' leaders, 1345 / 1242 with the next leads
// found and the sets cleared between the second barrier and the third, 1324 / 1228 behind the third; found in the same step,
// behind a barrier of their own, 1416 / 1316.
template <int A, class Between>
__device__ __forceinline__ bool cell_sums(CellReduceLds<A>& L, const int cell, const int set, const float delta, const bool valid, float* sorted,
                                          Between between, float* sum) {
  const int tid = threadIdx.x, w = tid >> 6;
  L.delta[tid] = delta;
  __syncthreads();
  between();
  unsigned long long mw[4];
  {
    const ulonglong2 lo = *reinterpret_cast<const ulonglong2*>(&L.members[set][0]);
    const ulonglong2 hi = *reinterpret_cast<const ulonglong2*>(&L.members[set][2]);
    mw[0] = lo.x;
    mw[1] = lo.y;
    mw[2] = hi.x;
    mw[3] = hi.y;
  }
  const int p0 = __popcll(mw[0]), p1 = __popcll(mw[1]), p2 = __popcll(mw[2]), p3 = __popcll(mw[3]);
  const unsigned long long mine = w == 0 ? mw[0] : w == 1 ? mw[1] : w == 2 ? mw[2] : mw[3];
  const int place = (w > 0 ? p0 : 0) + (w > 1 ? p1 : 0) + (w > 2 ? p2 : 0) + __popcll(mine & ((1ull << (tid & 63)) - 1ull));
  const bool leader = valid && place == 0;
  const int holders = leader ? p0 + p1 + p2 + p3 - 1 : 0;  // the key's further holders
  {
    const unsigned long long first = mw[0] != 0ull ? mw[0] : mw[1] != 0ull ? mw[1] : mw[2] != 0ull ? mw[2] : mw[3];
    const int ld = (mw[0] != 0ull ? 0 : mw[1] != 0ull ? 64 : mw[2] != 0ull ? 128 : 192) + __builtin_ctzll(first | (1ull << 63));
    const bool lines_up = valid && place > 0 && place <= kSortRows;
    *(lines_up ? &sorted[(place - 1) * kBlockSamples + ld] : &L.delta[tid]) = delta;
  }
  if (cell >= 0) L.lead[cell] = kNoLead;  // (read before the barrier above)
  __syncthreads();
  float acc = 0.0f;
  if (leader) {
    acc = acc + delta;
    if (holders != 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) mw[i] &= w == i ? ~(1ull << (tid & 63)) : ~0ull;
      acc = add_holders(L.delta, sorted, mw, holders, acc);
    }
  }
  *sum = acc;
  return leader;
}

// Before each reduce_block(), separated from it by a barrier (and from the
// one before by another): every record of every cell starts as "nothing, of this step".
// Thread t touches the 16-byte pieces t, t + 256, ... of `stage` here and on the way out
// of reduce_block(), and no others.
template <bool HASHED>
__device__ __forceinline__ void reduce_stage_init(unsigned long long* stage, const ReduceGeom G, const uint32_t tag) {
  const unsigned long long none = Rec<HASHED>::make(0u, tag, 0.0f);
  ulonglong2* stage2 = reinterpret_cast<ulonglong2*>(stage);
  for (int i = threadIdx.x; i < 1 << (G.main_shift - 1 + G.own_shift); i += kBlockSamples) stage2[i] = make_ulonglong2(none, none);
}

// One-launch kernel: pass 1 for one block.  All 256 threads of the workgroup call it with
// their sample (valid = false: no sample / no delta).  Hashed form: having entered their thread number in
// L.lead[at] with an atomic min, `at` the key's entry in `keys`, which is cleared again.  Dense form: in the set
// at = (lead of the cell) * A + action; cell and next_cell: where the env stands now and next, -1 without one.  The main halves of all cells of the
// block are put together in LDS (`stage`, owners << main_shift records, free again
// on return) and go out as whole lines (that of (block, owner) at (block * owners + owner)
// << main_shift behind `window_offset`), 16 bytes to a store and lane, every record
// carrying `tag`; a record beyond the main half goes straight to
// ext[(owner * blocks + block) << main_shift]:
// scattered 8-byte stores are partial line writes, and some 350 of them per workgroup
// took 1.6 us to be acknowledged.
// Returns (to every thread) whether some owner was handed more distinct keys than a
// cell has records: its cell then says kSlotOverflow and the owner needs the block's
// raw samples.
template <bool HASHED, class Lds>
__device__ __forceinline__ bool reduce_block(Lds& L, const ReduceGeom G, const int block, const int key, const int cell, const int next_cell,
                                             const int at, int* keys, const float delta,
                                             const bool valid, const uint32_t tag, float* sorted,
                                             unsigned long long* stage, const DevWindow window,
                                             const uint32_t window_offset, unsigned long long* ext) {
  const int tid = threadIdx.x;
  const int n_own = 1 << G.own_shift;
  const int cap = 1 << G.cell_shift;  // records of a cell
  const int cap_main = 1 << G.main_shift;  // of its main half
  float acc;
  auto clear = [&] {
    L.handed[tid] = 0;  // (256 owners)
    if (tid == 0) L.over = 0;
  };
  bool leader;
  if constexpr (HASHED) leader = block_sums(L, at, delta, valid, sorted, clear, &acc);
  else leader = cell_sums(L, cell, at, delta, valid, sorted, clear, &acc);
  int slot = 0, owner = 0;
  if (leader) {
    owner = owner_of(key, G);
    slot = atomicAdd(&L.handed[owner], 1);  // slot order is free: records carry the key
    *(slot >= cap ? &L.over : &L.none) = 1;
    // (record 0's count is added on the way out, when every leader has drawn its slot)
    if (slot < cap_main) stage[(owner << G.main_shift) + slot] = Rec<HASHED>::make((uint32_t)slot_of(key, G), tag, acc);
  }
  __syncthreads();
  const bool over = L.over != 0;
  // (behind the barrier: a barrier waits for the stores before it to be acknowledged)
  if (leader && slot >= cap_main && slot < cap)
    st_dev64(ext + ((((size_t)owner * G.n_blocks + block) << G.main_shift) + (slot - cap_main)),
             Rec<HASHED>::make((uint32_t)slot_of(key, G), tag, acc));

  // (the one-launch kernel always has 256 owners and main halves of 4 records: 512 pieces,
  // two to a thread, both asked for before the first is used)
  const ulonglong2* stage2 = reinterpret_cast<const ulonglong2*>(stage);
  const int piece_shift = G.main_shift - 1;  // log2(pieces of a cell's main half)
  const int pieces = n_own << piece_shift;
  constexpr int kPer = kStagePieces / kBlockSamples;
  static_assert(kPer == 2, "two pieces of the stage to a thread");
  ulonglong2 v[kPer];
  int c[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid + j * kBlockSamples;
    v[j] = i < pieces ? stage2[i] : make_ulonglong2(0ull, 0ull);
    c[j] = (i < pieces && (i & ((1 << piece_shift) - 1)) == 0) ? L.handed[i >> piece_shift] : 0;
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid + j * kBlockSamples;
    v[j].x |= (unsigned long long)(uint32_t)(c[j] > cap ? kSlotOverflow : c[j]) << Rec<HASHED>::kCountShift;
    if (i < pieces)
      st_dev128(window, window_offset + (uint32_t)((((size_t)block * n_own) << (G.main_shift + 3)) + (size_t)i * 16),
                make_uint4((uint32_t)v[j].x, (uint32_t)(v[j].x >> 32), (uint32_t)v[j].y, (uint32_t)(v[j].y >> 32)));
  }
  // For the next call, while the cells travel (the caller has a barrier before that): nobody waits for it here, where
  // between the barriers above it is in the way of the sums (hashed: 20,000 envs on 101x99x8, 50 steps 440 us there, 437 here).
  if (leader) {
    unsigned long long* set = L.members[HASHED ? tid : at];
    *reinterpret_cast<ulonglong2*>(set) = make_ulonglong2(0ull, 0ull);
    *reinterpret_cast<ulonglong2*>(set + 2) = make_ulonglong2(0ull, 0ull);
  }
  if constexpr (HASHED) {
    if (leader) {
      L.lead[at] = kNoLead;
      keys[at] = -1;
    }
  } else if (cell >= 0) {
    atomicMin(&L.lead[next_cell], (uint32_t)tid);
  }
  return over;
}

// ---- two launches: pass 1 ---------------------------------------------------------------

// Where the samples of an update come from: packed by the host (which has checked the
// states), or left behind by k_step.
struct PackedSamples {
  const int32_t* key;    // s * A + a, or -1: an action outside [0, A)
  const uint32_t* s2d;   // s' and, in the top bit, done; null: `key` holds the words of pack_transitions_short
  const float* r;
  template <int A>
  __device__ __forceinline__ void get(int i, int& k, int& s2, float& r_, bool& done) const {
    r_ = r[i];
    k = key[i];
    if (!s2d) {  // (8 bytes over the link instead of 12: 65,536 transitions 26.5 -> 23.9 us)
      const uint32_t v = (uint32_t)k;
      k = (v & 0xffffu) == 0xffffu ? -1 : (int)(v & 0xffffu);
      s2 = (int)((v >> 16) & 0x7fffu);
      done = (v >> 31) != 0u;
      return;
    }
    const uint32_t v = s2d[i];
    s2 = (int)(v & 0x7fffffffu);
    done = (v >> 31) != 0u;
  }
};
// transition left behind by k_step for k_update_* : (s, a, r, s', done)
struct Transition {
  int32_t* s;
  int32_t* a;
  float* r;
  int32_t* s2;
  uint8_t* done;
  template <int A>
  __device__ __forceinline__ void get(int i, int& k, int& s2_, float& r_, bool& done_) const {
    const int ai = a[i];
    k = (unsigned)ai < (unsigned)A ? s[i] * A + ai : -1;
    s2_ = s2[i];
    r_ = r[i];
    done_ = done[i] != 0;
  }
};

// (key, delta) of sample i of n against ONE table, all reads before any write; key = -1 and
// delta = 0 without a sample or for an invalid action.
template <int A, class Samples>
__device__ __forceinline__ void sample_delta(const Samples& X, const int i, const int n, const float* __restrict__ Q,
                                             const float lr, const float gamma, const int max_mode, int& k, float& d) {
  k = -1;
  d = 0.0f;
  int s2 = 0;
  float r = 0.0f;
  bool done = false;
  if (i < n) X.template get<A>(i, k, s2, r, done);
  if (k >= 0) {
    const float q = Q[k];
    const Row<A> row2 = load_row<A>(Q + (size_t)s2 * A);
    d = td_delta(q, r, row_max(row2, done, max_mode), lr, gamma);
  }
}

// The entry of `key` in a table of `mask` + 1 keys (-1: free) that has room for it.  In two
// halves: `found` is what a compare-and-swap of -1 for the key left at the first entry.
__device__ __forceinline__ int hash_start(const int mask, const int key) {
  return (int)(((unsigned)key * 0x9E3779B1u) >> 16) & mask;
}
__device__ __forceinline__ int hash_finish(int* keys, const int mask, const int key, int h, int found) {
  while (found != -1 && found != key) {
    h = (h + 1) & mask;
    found = atomicCAS(&keys[h], -1, key);
  }
  return h;
}
__device__ __forceinline__ int hash_enter(int* keys, const int mask, const int key) {
  const int h = hash_start(mask, key);
  return hash_finish(keys, mask, key, h, atomicCAS(&keys[h], -1, key));
}

// LDS of pass 1, then handed[owners] (block sums handed to each owner), then `sorted`.
// A block's 256 keys at most in a table of 2048: a probe or two, also for the unluckiest
// lane of a wave; tables of up to 2048 keys have an entry per key.
struct BlockLds {
  ReduceLdsT<kHashSlots> red;
  int keys[kHashSlots];
};
inline __host__ __device__ size_t block_lds_bytes(int own_shift) {
  return sizeof(BlockLds) + ((size_t)4 << own_shift) + kSortBytes;
}

// Before reduce_block_wide(), separated from it by a barrier.
__device__ __forceinline__ void block_lds_init(unsigned char* lds, const ReduceGeom G) {
  BlockLds& L = *reinterpret_cast<BlockLds*>(lds);
  int* handed = reinterpret_cast<int*>(lds + sizeof(BlockLds));
  reduce_block_init(L.red);
  for (int i = threadIdx.x; i < kHashSlots; i += kBlockSamples) L.keys[i] = -1;
  for (int i = threadIdx.x; i < 1 << G.own_shift; i += kBlockSamples) handed[i] = 0;
}

// Pass 1 for one block of 256 threads, once per launch.  The records go straight to memory,
// for a reader in a later launch; the cell of (owner, block) is at
// handoff[(owner * blocks + block) << cell_shift], so that an owner reads its cells side by side.
__device__ __forceinline__ void reduce_block_wide(unsigned char* lds, const ReduceGeom G, const int block,
                                                  const int key, const float delta, const bool valid,
                                                  unsigned long long* handoff) {
  BlockLds& L = *reinterpret_cast<BlockLds*>(lds);
  int* handed = reinterpret_cast<int*>(lds + sizeof(BlockLds));
  float* sorted = reinterpret_cast<float*>(lds + sizeof(BlockLds) + ((size_t)4 << G.own_shift));
  const int tid = threadIdx.x;
  const int cap = 1 << G.cell_shift;
  int at = 0;
  if (valid) {
    at = G.K <= kHashSlots ? key : hash_enter(L.keys, kHashSlots - 1, key);
    atomicMin(&L.red.lead[at], (uint32_t)tid);
  }
  float acc;
  const bool leader = block_sums(L.red, at, delta, valid, sorted, [] {}, &acc);
  int slot = 0, owner = 0;
  if (leader) {
    owner = owner_of(key, G);
    slot = atomicAdd(&handed[owner], 1);  // slot order is free: records carry the key
  }
  __syncthreads();
  if (leader && slot < cap) {
    uint32_t count = 0;
    if (slot == 0) {
      const int c = handed[owner];  // final: every leader has drawn its slot
      count = (uint32_t)(c > cap ? kSlotOverflow : c);
    }
    handoff[((((size_t)owner * G.n_blocks) + block) << G.cell_shift) + slot] =
        make_wide_rec((uint32_t)slot_of(key, G), count, acc);
  }
  for (int o = tid; o < 1 << G.own_shift; o += kBlockSamples)
    if (handed[o] == 0) handoff[(((size_t)o * G.n_blocks) + block) << G.cell_shift] = 0ull;
}

// Pass 1 over samples in memory (which may be the host's: each is read once).  `before`: see
// signal_reached.
template <int A, class Samples>
__global__ __launch_bounds__(kBlockSamples) void k_td_blocks(const ReduceGeom G, const Samples X, const int n,
                                                             const float* __restrict__ Q, const float lr,
                                                             const float gamma, const int max_mode,
                                                             int32_t* __restrict__ key, float* __restrict__ delta,
                                                             unsigned long long* __restrict__ handoff,
                                                             const HostSignal before) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int i = blockIdx.x * kBlockSamples + threadIdx.x;
  int k;
  float d;
  block_lds_init(lds_raw, G);
  sample_delta<A>(X, i, n, Q, lr, gamma, max_mode, k, d);
  if (i < n) {
    key[i] = k;
    delta[i] = d;
  }
  signal_reached(before);  // (not ahead of the samples: 262,144 of them 61.2 -> 60.6 us)
  __syncthreads();
  reduce_block_wide(lds_raw, G, blockIdx.x, k >= 0 ? k : 0, d, k >= 0, handoff);
}

// ---- two launches: pass 2 ---------------------------------------------------------------

constexpr int kOwnerWaves = 16;  // at most
constexpr int kTileKeys = 64;    // keys of an owner up to which a wave lays its group out as a tile
// 32-bit words of LDS per wave of k_reduce_owners besides its row of group sums: the tile,
// or the claims; and the list of 256 samples
inline __host__ __device__ int owner_wave_words(int own_keys) {
  return (own_keys <= kTileKeys ? kGroupBlocks * kTileKeys : own_keys) + kBlockSamples + kBlockSamples / 2;
}
inline __host__ __device__ size_t owners_lds_bytes(int waves, int own_keys) {
  return ((size_t)(waves + 1) * own_keys + (size_t)waves * owner_wave_words(own_keys)) * 4;
}

// One workgroup per owner, one wave per group of 16 blocks (in turn where there are more
// groups than waves): no barrier before the groups are added up.  With cells of 8 records a
// lane has the 16 bytes it needs of all 16 cells in one load.
// Owners with up to 64 keys (TILE): the wave lays the records out as a dense [block][key] tile
// of 4 KB and adds its columns, a lane to a key, 16 loads in flight - the same time whatever
// the records.  Owners with more keys: 16 blocks hand them some 20 records, so the work goes
// by the records.  All that are left enter their block number with a minimum under their
// key, the lowest block of each key adds its record to the key's sum and is done: as many
// rounds as the most crowded key of the group has blocks, two or three when the keys are
// spread, and never more than 16.
// Measured, both launches of a step of a shared table: 65,536 envs on 64x64x4 10.5 us (four
// waves of four groups each 12.5), 20,000 envs on 101x99x8 12.6 us and 65,536 on 128x128x8
// 15.0 us (every owner scanning all samples for its range of keys: 40-60 and 164 us).
// `sig`: tells the host that the launch before this one is through (block 0, at once).
template <bool TILE>
__global__ __launch_bounds__(kOwnerWaves * 64) void k_reduce_owners(const ReduceGeom G, const int own_keys,
                                                                    float* __restrict__ Q,
                                                                    const int32_t* __restrict__ key,
                                                                    const float* __restrict__ delta, const int n,
                                                                    const unsigned long long* __restrict__ handoff,
                                                                    const HostSignal sig) {
  extern __shared__ __align__(16) float sums[];  // [waves][own_keys] group sums, [own_keys] totals, the waves' own words
  const int tid = threadIdx.x, n_threads = blockDim.x;
  const int lane = tid & 63, wave = tid >> 6, n_waves = n_threads >> 6;
  const int owner = blockIdx.x;
  float* gs = sums + wave * own_keys;
  float* total = sums + n_waves * own_keys;
  float* own = total + own_keys + wave * owner_wave_words(own_keys);
  float* tile = own;                                       // TILE: [16 blocks][64 keys]
  uint32_t* claim = reinterpret_cast<uint32_t*>(own);      // else: [own_keys]
  float* list_v = own + (TILE ? kGroupBlocks * kTileKeys : own_keys);
  uint16_t* list_s = reinterpret_cast<uint16_t*>(list_v + kBlockSamples);
  signal_reached(sig);
  // the table entry this thread will update first: fetched now, needed last
  const int key0 = tid < own_keys ? key_of(owner, tid, G) : G.K;
  const float q0 = key0 < G.K ? Q[key0] : 0.0f;
  for (int k = tid; k < own_keys; k += n_threads) total[k] = 0.0f;
  auto wave_fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // block `blk` has more distinct keys for this owner than a cell holds: its part again,
  // from the samples, the first holder of a key adding up all of them in order
  auto from_samples = [&](int blk, auto put) {
    int m = 0;
    for (int j = 0; j < kBlockSamples; j += 64) {
      const int i = blk * kBlockSamples + j + lane;
      const int k = i < n ? key[i] : -1;
      const bool mine = k >= 0 && owner_of(k, G) == owner;
      const unsigned long long who = __builtin_amdgcn_ballot_w64(mine);
      if (mine) {
        const int at = m + __popcll(who & ((1ull << lane) - 1ull));
        list_s[at] = (uint16_t)slot_of(k, G);
        list_v[at] = delta[i];
      }
      m += __popcll(who);
    }
    wave_fence();
    for (int e = lane; e < m; e += 64) {
      const int slot = list_s[e];
      bool first = true;
      for (int f = 0; f < e; ++f) first = first && list_s[f] != slot;
      if (first) {
        float acc = 0.0f;
        for (int f = e; f < m; ++f)
          if (list_s[f] == slot) acc = acc + list_v[f];
        put(slot, acc);
      }
    }
    wave_fence();
  };

  const int n_groups = (G.n_blocks + kGroupBlocks - 1) / kGroupBlocks;
  for (int g0 = 0; g0 < n_groups; g0 += n_waves) {
    const int b0 = (g0 + wave) * kGroupBlocks;
    const unsigned long long* cells = handoff + (((size_t)owner * G.n_blocks + b0) << G.cell_shift);
    // lane l: records 2 (l & 3) and the next of block l >> 2
    const int b = lane >> 2, pair = lane & 3;
    uint4 rec = make_uint4(0, 0, 0, 0);
    if (G.cell_shift == 3 && b0 + b < G.n_blocks) rec = reinterpret_cast<const uint4*>(cells)[lane];
    if (TILE) {
      float4* tile4 = reinterpret_cast<float4*>(tile);
#pragma unroll
      for (int i = 0; i < kGroupBlocks * kTileKeys / 4 / 64; ++i) tile4[i * 64 + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
      for (int k = lane; k < own_keys; k += 64) {
        gs[k] = 0.0f;
        claim[k] = kNoLead;
      }
    }
    if (G.cell_shift == 3) {
      const int c = wide_count((uint32_t)__builtin_amdgcn_mov_dpp((int)rec.x, 0x00, 0xf, 0xf, true));  // of the quad's lane 0
      const bool over = c == kSlotOverflow;
      bool has0 = !over && 2 * pair < c, has1 = !over && 2 * pair + 1 < c;
      const int slot0 = wide_slot(rec.x), slot1 = wide_slot(rec.z);
      const float v0 = __uint_as_float(rec.y), v1 = __uint_as_float(rec.w);
      unsigned long long overs = __builtin_amdgcn_ballot_w64(over);
      if (TILE) {
        if (has0) tile[b * kTileKeys + slot0] = v0;
        if (has1) tile[b * kTileKeys + slot1] = v1;
        while (overs != 0ull) {
          const int bb = __builtin_ctzll(overs) >> 2;
          overs &= ~(0xfull << (4 * bb));
          from_samples(b0 + bb, [&](int slot, float acc) { tile[bb * kTileKeys + slot] = acc; });
        }
      } else if (overs != 0ull) {  // (rare) block after block
        for (int bb = 0; bb < kGroupBlocks; ++bb) {
          if ((overs >> (4 * bb)) & 1ull) {
            from_samples(b0 + bb, [&](int slot, float acc) { gs[slot] = gs[slot] + acc; });
          } else if (b == bb) {
            if (has0) gs[slot0] = gs[slot0] + v0;
            if (has1) gs[slot1] = gs[slot1] + v1;
          }
          wave_fence();
        }
      } else {
        while (__builtin_amdgcn_ballot_w64(has0 || has1) != 0ull) {  // (the lowest block of a key always gets through)
          if (has0) atomicMin(&claim[slot0], (uint32_t)b);
          if (has1) atomicMin(&claim[slot1], (uint32_t)b);
          wave_fence();
          const bool go0 = has0 && claim[slot0] == (uint32_t)b, go1 = has1 && claim[slot1] == (uint32_t)b;
          wave_fence();
          if (go0) {
            gs[slot0] = gs[slot0] + v0;
            claim[slot0] = kNoLead;
          }
          if (go1) {
            gs[slot1] = gs[slot1] + v1;
            claim[slot1] = kNoLead;
          }
          wave_fence();
          has0 = has0 && !go0;
          has1 = has1 && !go1;
        }
      }
    } else {  // few owners with large cells (and at most 64 keys each): lane l takes record l of one block after the other
      for (int bb = 0; bb < kGroupBlocks && b0 + bb < G.n_blocks; ++bb) {
        const unsigned long long r = lane < 1 << G.cell_shift ? cells[((size_t)bb << G.cell_shift) + lane] : 0ull;
        const int c = wide_count((uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)r));
        auto put = [&](int slot, float v) {
          if (TILE) tile[bb * kTileKeys + slot] = v;
          else gs[slot] = gs[slot] + v;
        };
        if (c == kSlotOverflow) from_samples(b0 + bb, put);
        else if (lane < c) put(wide_slot((uint32_t)r), __uint_as_float((uint32_t)(r >> 32)));
      }
    }
    if (TILE) {
      wave_fence();
      float v[kGroupBlocks];
#pragma unroll
      for (int bb = 0; bb < kGroupBlocks; ++bb) v[bb] = tile[bb * kTileKeys + lane];
      float acc = 0.0f;
#pragma unroll
      for (int bb = 0; bb < kGroupBlocks; ++bb) acc = acc + v[bb];
      if (lane < own_keys) gs[lane] = acc;
    }
    __syncthreads();
    const int here = min(n_waves, n_groups - g0);
    for (int k = tid; k < own_keys; k += n_threads) {
      float t = total[k];
      for (int w = 0; w < here; ++w) t = t + sums[w * own_keys + k];
      total[k] = t;
    }
    __syncthreads();
  }
  if (key0 < G.K) Q[key0] = q0 + total[tid];
  for (int k = tid + n_threads; k < own_keys; k += n_threads) {
    const int kk = key_of(owner, k, G);
    if (kk < G.K) Q[kk] = Q[kk] + total[k];
  }
}

// ---- up to 1024 samples: one launch --------------------------------------------------------

constexpr int kSmallSamples = 1024;
// One workgroup, 256 threads to a block of the tree.  A key has one entry in LDS with a
// leader per block; the leader of a key's first block adds the block sums (all in one
// group) and applies them.  Costs one launch and a trip for the samples instead of two
// launches with 256 owners, most of which are handed nothing.
// `changed` (host memory, may be null): per sample {key, new value} where its thread applied
// a total, {-1, 0} elsewhere.
template <int NB>
struct SmallLds {
  static constexpr int kSlots = 512 * NB;
  int keys[kSlots];
  uint32_t lead[NB][kSlots];
  unsigned long long members[NB * kBlockSamples][4];
  float delta[NB * kBlockSamples];
  float sum[NB * kBlockSamples];
};
template <int A, int NB, class Samples>
__global__ __launch_bounds__(kBlockSamples* NB) void k_td_small(const Samples X, const int n, float* __restrict__ Q,
                                                                const float lr, const float gamma, const int max_mode,
                                                                int2* __restrict__ changed, const HostSignal sig) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  using Lds = SmallLds<NB>;
  Lds& L = *reinterpret_cast<Lds*>(lds_raw);
  const int tid = threadIdx.x, blk = tid >> 8;
  int k;
  float d;
  sample_delta<A>(X, tid, n, Q, lr, gamma, max_mode, k, d);
  for (int i = tid; i < Lds::kSlots; i += kBlockSamples * NB) {
    L.keys[i] = -1;
#pragma unroll
    for (int b = 0; b < NB; ++b) L.lead[b][i] = kNoLead;
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) L.members[tid][w] = 0ull;
  L.delta[tid] = d;
  __syncthreads();
  const bool valid = k >= 0;
  int at = 0;
  if (valid) {
    at = hash_enter(L.keys, Lds::kSlots - 1, k);
    atomicMin(&L.lead[blk][at], (uint32_t)tid);
  }
  __syncthreads();
  uint32_t ld = kNoLead;
  if (valid) {
    ld = L.lead[blk][at];
    if (ld != (uint32_t)tid) atomicOr(&L.members[ld][(tid >> 6) & 3], 1ull << (tid & 63));
  }
  const bool leader = ld == (uint32_t)tid;
  __syncthreads();
  if (leader) {
    float acc = 0.0f + d;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      unsigned long long m = L.members[tid][w];
      const float* from = L.delta + blk * kBlockSamples + w * 64;
      while (m != 0ull) {  // thread order = sample order, four loads in flight
        float v[4];
        int have = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = m != 0ull ? from[__builtin_ctzll(m)] : 0.0f;
          have += m != 0ull ? 1 : 0;
          m &= m - 1ull;  // (0 stays 0)
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < have) acc = acc + v[j];
      }
    }
    L.sum[tid] = acc;
  }
  __syncthreads();  // (also: every thread has read the table)
  int2 out = make_int2(-1, 0);
  if (leader) {
    bool first = true;
#pragma unroll
    for (int b = 0; b < NB; ++b) first = first && (b >= blk || L.lead[b][at] == kNoLead);
    if (first) {
      float group = 0.0f;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t l = L.lead[b][at];
        if (l != kNoLead) group = group + L.sum[l];
      }
      const float q = Q[k] + (0.0f + group);
      Q[k] = q;
      out = make_int2(k, __float_as_int(q));
    }
  }
  if (changed && tid < n) store_host(reinterpret_cast<unsigned long long*>(changed) + tid, (unsigned long long)(uint32_t)out.x | (unsigned long long)(uint32_t)out.y << 32);
  signal_host(sig);
}

// Fallback for what needs too many owners or too large a hand-off buffer: one workgroup per 64 consecutive keys scans all samples,
// group by group (4096 samples), compacting its matches in order, and wave 0
// then folds them through the same tree.  Slow, same result.
__global__ __launch_bounds__(256) void k_reduce_scan(float* __restrict__ Q, const int K,
                                                      const int32_t* __restrict__ key,
                                                      const float* __restrict__ delta, const int n,
                                                      const HostSignal sig) {
  constexpr int kSpan = 1024;  // samples one wave scans per group: 4 blocks
  __shared__ float l_d[4][kSpan];
  __shared__ uint8_t l_k[4][kSpan];
  __shared__ uint16_t l_o[4][kSpan];  // sample offset inside the wave's span
  __shared__ int l_cnt[4];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int owner = blockIdx.x;
  float total = 0.0f;
  signal_reached(sig);

  for (int g0 = 0; g0 < n; g0 += 4 * kSpan) {
    int cnt = 0;
    const int base = g0 + wave * kSpan;
    for (int it = 0; it < kSpan / 64; ++it) {
      const int i = base + it * 64 + lane;
      const int k = (i < n) ? key[i] : -1;
      const bool match = (k >= 0) && ((k / kOwnKeys) == owner);
      const unsigned long long bal = __ballot(match);
      if (bal != 0ull) {
        if (match) {
          const int pos = cnt + __popcll(bal & ((1ull << lane) - 1ull));
          l_d[wave][pos] = delta[i];
          l_k[wave][pos] = (uint8_t)(k - owner * kOwnKeys);
          l_o[wave][pos] = (uint16_t)(it * 64 + lane);
        }
        cnt += __popcll(bal);
      }
    }
    if (lane == 0) l_cnt[wave] = cnt;
    __syncthreads();
    if (wave == 0) {
      float gs = 0.0f;
      for (int w = 0; w < 4; ++w) {
        const int c = l_cnt[w];
        float bs = 0.0f;
        int cur = 0;  // block inside the wave's span
        for (int e = 0; e < c; ++e) {
          const int blk = l_o[w][e] >> 8;
          if (blk != cur) {
            gs = gs + bs;
            bs = 0.0f;
            cur = blk;
          }
          const float dv = l_d[w][e];
          if (l_k[w][e] == lane) bs = bs + dv;
        }
        gs = gs + bs;
      }
      total = total + gs;
    }
    __syncthreads();
  }
  const int k = owner * kOwnKeys + lane;
  if (wave == 0 && k < K) Q[k] = Q[k] + total;
}

}  // namespace crl
