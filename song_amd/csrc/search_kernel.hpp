// Best-first graph search on gfx950: one query per 64-lane wavefront.
//
// Semantics follow the reference CPU search FixedDegreeGraph::astar_multi_start_search
// (graph.h:169-216): start at the entry vertex, repeatedly expand the (dist, id)-smallest
// unexpanded candidate, stop when the k-best expanded list is full and its largest distance
// is strictly below the next candidate's (graph.h:188), mark every discovered neighbour
// visited (graph.h:198-205), return the expanded list ascending by (dist, id).
//
// The CPU's unbounded queue is replaced by a bounded one that only ever drops entries that
// can never be expanded: an entry c is dropped when the pq-best expanded list is full with
// largest distance < c.d, or when the queue holds pq entries with distance < c.d.  Entries
// tied with the pq-th distance are kept (up to `slack`), so the expansion order -- and
// therefore the output -- equals the CPU's.  The queue is two-level: a sorted head of the
// (up to) 64 smallest entries, from which the minimum is popped, and an unsorted bag of the
// rest (every head entry <= T < every bag entry).  New candidates at most T are merged into
// the head, the others appended to the bag; the head's overflow moves to the bag; an empty
// head is refilled with the bag's 64 smallest (exact selection); the bag is bounded lazily
// (the drops above are applied when it nears its capacity).
//
// Per-wave LDS layout (bytes, in order):
//   visited  : H slots, no deletion: compact 16-bit entries in groups of 8 (vis16_insert) or
//              32-bit (id + 1) in groups of 4 (vis_insert), one 16-byte read per group; or,
//              approximate, a blocked Bloom filter of 2^hlog 32-bit words (bloom_insert)
//   best     : pq keys, the front of the pq-best expanded list, in any order; absent with
//              bglob, where the front lives in the wave slot's global region
//   cid      : 256 u32   candidate ids of the current expansion / radix-select bins
//   qv       : qld f32   the query, zero-padded to a multiple of 16
//   stage    : products of the exact sums done again (wide rows in exact mode, seq_stage)
// The queue head is one key per lane in registers, ascending over lanes [h, h + nq), nq <= 64,
// +inf in the others.
// The bag (qcap = pq + slack + 128 keys, unsorted, first bn live) is in global memory, one
// region per wave slot: it is written by plain stores as candidates arrive and read only when
// the head runs empty or the bag nears its capacity, so LDS holds only what every step
// touches and more waves fit on a CU.  The best list's 64 largest entries are one key per lane
// in registers; its front (the others, unsorted) is written once per entry and read only when
// 64 expansions have landed below the tail of a full list, and at the end, where the results
// are selected from it -- so with bglob it lives after the bag in the slot's global region (pq
// keys) and a large pq does not cost LDS.
//
// Each wave owns its LDS slice (one wave per workgroup in search_kernel; 1-4 waves, each
// on its own slice, in search_persistent).  LDS instructions of a wave execute in issue
// order, so lanes exchange data through LDS with only a compiler fence between the write
// and the read (lds_fence), and global loads stay in flight across those points.
//
// Per expansion the dependent global round trips are: adjacency row of the expanded
// vertex (prefetched one step ahead for the predicted next vertex, the queue head after
// the pop) and one gather of all new candidates' rows (all rows issued at once).
//
// Keys order by (distance, id) lexicographically:
//   KeyF (fp32 mode):  one u64 = (orderable float bits << 32) | id
//   KeyD (exact mode): orderable double bits + u32 id
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace song {

enum { M_L2 = 0, M_IP = 1, M_COS = 2 };

enum : uint32_t { F_VIS_OVF = 1u, F_Q_OVF = 2u, F_STEP_CAP = 4u, F_BAD_LAUNCH = 0x80000000u };

struct SearchParams {
    const float *data;      // n x ld
    const uint32_t *graph;  // n x gstride, [deg, ids...]
    const float *norms;     // cosine: per-vertex squared norm (fmaf chain), else null
    const float *queries;   // nq x dim
    const uint32_t *entry;  // nq x n_entry start vertices or null (vertex 0)
    int n_entry;            // entries per query (1..64)
    const int *steps_arr;   // per-query expansion cap or null
    const int *pq_arr;      // per-query pq or null
    const int *k_arr;       // per-query k or null
    const uint32_t *qidx;   // query index remap (retry pass) or null
    uint32_t *out_ids;      // nq x out_ld
    float *out_dist;        // nq x out_ld or null
    uint32_t *out_flags;    // nq or null
    uint32_t *out_stats;    // nq x 8 or null: expansions, distances, sum(1+deg), prefetch hits,
                            // settle step (last expansion that changed the first k), head
                            // refills from the bag, bag truncations, 0
    uint64_t n;
    int dim, ld, gstride;
    int qld;                // query floats in LDS: dim padded to 16
    int nq, pq, k, out_ld;
    int hlog, slack, max_steps, qcap;
    uint32_t *gvis;         // per-launch-slot spill tables (2^ghlog u32 each) or null
    int ghlog;
    int qbase;              // first query (or qidx entry) of this launch
    const uint8_t *data_lp; // low-precision rows (BF16 / FP8 kernels), lp_stride bytes each
    const float *scale;     // per-row scale of data_lp
    size_t lp_stride;
    int rerank;             // low-precision kernels: re-rank the final list in exact FP32
    // persistent kernel: waves take list positions t = (*work_next)++ while t < *work_count
    // and search query qidx[t] (t itself without a list)
    uint32_t *work_next;
    const uint32_t *work_count;
    uint32_t wave_lds;      // LDS bytes of one wave's slice (every launch; the layout must fit)
    int vis16;              // 1: compact visited table (16-bit slots, needs idbits - (hlog - 3) <= 13)
    int idbits;             // ids are below 2^idbits
    unsigned char *gbag;    // queue bags, one per launch slot / persistent wave, gbag_stride bytes
    size_t gbag_stride;     // >= qcap keys
    // queries whose visited set or queue overflowed are appended here for a re-run
    uint32_t *retry_list;
    uint32_t *retry_count;
    int wave_prio;          // persistent kernel: 1 = raise the waves' issue priority (s_setprio 2)
    int bloom_k;            // 0: exact visited table; 1..9: blocked Bloom filter of 2^hlog 32-bit words,
                            // bloom_k bits per id in one word (approximate: false positives skip vertices)
    int multiprobe;         // several-queries-per-wave kernel: expansions per step (1, or 2: the next
                            // queue head too; approximate)
    int seq_stage;          // 1: the slice has SEQ_STAGE floats after the query
    int int_rows;           // 1: every row value is an integer, in [row_min, row_max]
    float row_min, row_max;
};

// bytes of a slot's bag before the best-list front (bglob): qcap keys rounded to 256
template <class Key> __device__ __forceinline__ size_t bag_bytes(int qcap) {
    return ((size_t)qcap * sizeof(Key) + 255) & ~(size_t)255;
}

// ---------------------------------------------------------------- keys

__device__ __forceinline__ uint32_t ord32(float f) {
    uint32_t u = __float_as_uint(f);
    if (f == 0.0f) u = 0u;            // -0 and +0 compare equal on the CPU
    if (f != f) u = 0x7f800000u;      // NaN (zero-norm cosine) sorts as +inf
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float unord32(uint32_t o) {
    uint32_t u = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
    return __uint_as_float(u);
}
__device__ __forceinline__ uint64_t ord64(double d) {
    uint64_t u = (uint64_t)__double_as_longlong(d);
    if (d == 0.0) u = 0ull;
    if (d != d) u = 0x7ff0000000000000ull;
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double unord64(uint64_t o) {
    uint64_t u = (o & 0x8000000000000000ull) ? (o & 0x7fffffffffffffffull) : ~o;
    return __longlong_as_double((long long)u);
}

__device__ __forceinline__ uint32_t rl32(uint32_t v, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ uint64_t rl64(uint64_t v, int lane) {
    return ((uint64_t)rl32((uint32_t)(v >> 32), lane) << 32) | rl32((uint32_t)v, lane);
}

struct KeyF {
    static constexpr int DKBITS = 32;  // significant bits of dk()
    uint64_t v;
    __device__ static KeyF make_f(float d, uint32_t id) { return KeyF{((uint64_t)ord32(d) << 32) | id}; }
    __device__ static KeyF inf() { return KeyF{~0ull}; }
    __device__ uint32_t id() const { return (uint32_t)v; }
    __device__ uint64_t dk() const { return v >> 32; }
    __device__ float dist() const { return unord32((uint32_t)(v >> 32)); }
    __device__ KeyF rl(int lane) const { return KeyF{rl64(v, lane)}; }
};
__device__ __forceinline__ bool lt(const KeyF &a, const KeyF &b) { return a.v < b.v; }

struct KeyD {
    static constexpr int DKBITS = 64;
    uint64_t d;
    uint32_t i, pad;
    __device__ static KeyD make_d(double dist, uint32_t id) { return KeyD{ord64(dist), id, 0u}; }
    __device__ static KeyD inf() { return KeyD{~0ull, ~0u, 0u}; }
    __device__ uint32_t id() const { return i; }
    __device__ uint64_t dk() const { return d; }
    __device__ float dist() const { return (float)unord64(d); }
    __device__ KeyD rl(int lane) const { return KeyD{rl64(d, lane), rl32(i, lane), 0u}; }
};
__device__ __forceinline__ bool lt(const KeyD &a, const KeyD &b) {
    return a.d < b.d || (a.d == b.d && a.i < b.i);
}

__device__ __forceinline__ KeyF rl_key(const KeyF &k, int lane) { return k.rl(lane); }
__device__ __forceinline__ KeyD rl_key(const KeyD &k, int lane) { return k.rl(lane); }

// whole-wave lane shifts by one (DPP wave_shl:1 / wave_shr:1): shl1 gives lane i the value of
// lane i + 1 (lane 63 gets 0), shr1 the value of lane i - 1 (lane 0 gets 0).  The end lane's value is
// left to the instruction (zero), not to a copy made first; no caller uses it.
template <int CTRL> __device__ __forceinline__ uint32_t dpp32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, true);
}
constexpr int DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;
template <int CTRL> __device__ __forceinline__ uint64_t dpp64(uint64_t x) {
    return ((uint64_t)dpp32<CTRL>((uint32_t)(x >> 32)) << 32) | dpp32<CTRL>((uint32_t)x);
}
// c ? a : b field by field (a conditional over two key lvalues selects between their addresses,
// which puts the keys in scratch memory)
__device__ __forceinline__ KeyF ksel(bool c, const KeyF &a, const KeyF &b) { return KeyF{c ? a.v : b.v}; }
__device__ __forceinline__ KeyD ksel(bool c, const KeyD &a, const KeyD &b) {
    return KeyD{c ? a.d : b.d, c ? a.i : b.i, 0u};
}
__device__ __forceinline__ KeyF shl1(const KeyF &k) { return KeyF{dpp64<DPP_WAVE_SHL1>(k.v)}; }
__device__ __forceinline__ KeyF shr1(const KeyF &k) { return KeyF{dpp64<DPP_WAVE_SHR1>(k.v)}; }
__device__ __forceinline__ KeyD shl1(const KeyD &k) {
    return KeyD{dpp64<DPP_WAVE_SHL1>(k.d), dpp32<DPP_WAVE_SHL1>(k.i), 0u};
}
__device__ __forceinline__ KeyD shr1(const KeyD &k) {
    return KeyD{dpp64<DPP_WAVE_SHR1>(k.d), dpp32<DPP_WAVE_SHR1>(k.i), 0u};
}

template <bool EXACT> struct KeySel { using T = KeyF; };
template <> struct KeySel<true> { using T = KeyD; };

// ---------------------------------------------------------------- wave helpers

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63u); }
// The lane index as a value the compiler cannot see through, for the rare paths (refill,
// truncation, front insert): their lane masks -- (lane & j) == 0 of every bitonic step, lane < n of
// every block -- are then computed where they are used.  From the plain lane index they are loop
// invariants, which the compiler hoists out of the expansion loop into scalar register pairs; the
// loop has about 100 scalar registers, so 130-250 of them were spilled to vector lanes and read back
// on the common path.
__device__ __forceinline__ int rare_lane() {
    int l = lane_id();
    asm volatile("" : "+v"(l));
    return l;
}
// a wave-uniform 64-bit mask as a per-lane predicate (the mask is used as the condition register
// as it is: no shift or compare per lane)
__device__ __forceinline__ bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
// the lowest n bits, n in [0, 64]
__device__ __forceinline__ uint64_t low_bits(int n) { return n >= 64 ? ~0ull : (1ull << n) - 1ull; }
__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }
__device__ __forceinline__ int lanes_below(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// compiler-only fence for LDS traffic inside one wave (see the layout note above)
__device__ __forceinline__ void lds_fence() { __atomic_signal_fence(__ATOMIC_SEQ_CST); }
// wait for every vector-memory operation of this wave (s_waitcnt vmcnt(0)).  Placed at the end
// of the rare bag paths (refill, truncation): their loads land in registers that the common path
// reuses, and without a wait on the rare path itself the compiler has to wait for all memory
// operations -- the adjacency prefetch included -- at the top of every expansion.
__device__ __forceinline__ void vm_drain() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// before lanes read bag entries that other lanes of the wave stored to global memory: the
// stores complete first (workgroup scope: the wave's own CU)
__device__ __forceinline__ void bag_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); }

// lowest set bit exponent of a nonzero float (value = odd * 2^e); INT_MAX for 0
__device__ __forceinline__ int lsb_exp(float p) {
    uint32_t u = __float_as_uint(p) & 0x7fffffffu;
    if (u == 0u) return 0x3fffffff;
    int e = (int)(u >> 23);
    uint32_t m = u & 0x7fffffu;
    if (e) m |= 0x800000u;
    else e = 1;
    return e - 150 + __builtin_ctz(m);
}

// visited set: (id + 1) in an open-addressing table probed in aligned groups of 4 slots,
// one 16-byte LDS read per group.  An id goes to the first empty slot of the first group
// on its probe sequence that has one; with no deletions a lookup can therefore stop at the
// first group holding an empty slot.  Lanes inserting the same id race through
// compare-and-swap; exactly one of them sees the slot empty.  Returns true if id was absent.
__device__ __forceinline__ bool vis_insert(uint32_t *vis, uint32_t mask, int hlog, uint32_t id) {
    const uint32_t key = id + 1u;
    const uint32_t gmask = mask >> 2;
    uint32_t g = (id * 0x9E3779B1u) >> (34 - hlog);
    for (;;) {
        const uint4 v = *reinterpret_cast<const uint4 *>(vis + (g << 2));
        if (v.x == key || v.y == key || v.z == key || v.w == key) return false;
        const uint32_t e = v.x == 0u ? 0u : v.y == 0u ? 1u : v.z == 0u ? 2u : v.w == 0u ? 3u : 4u;
        if (e == 4u) {
            g = (g + 1u) & gmask;
            continue;
        }
        const uint32_t old = atomicCAS(&vis[(g << 2) + e], 0u, key);
        if (old == 0u) return true;
        if (old == key) return false;
        lds_fence();  // another id took the slot: read the group again
    }
}

// read-only lookup in the LDS table
__device__ __forceinline__ bool vis_test(const uint32_t *vis, uint32_t mask, int hlog, uint32_t id) {
    const uint32_t key = id + 1u;
    const uint32_t gmask = mask >> 2;
    uint32_t g = (id * 0x9E3779B1u) >> (34 - hlog);
    for (;;) {
        const uint4 v = *reinterpret_cast<const uint4 *>(vis + (g << 2));
        if (v.x == key || v.y == key || v.z == key || v.w == key) return true;
        if (v.x == 0u || v.y == 0u || v.z == 0u || v.w == 0u) return false;
        g = (g + 1u) & gmask;
    }
}

// Compact visited set (16-bit slots, half the LDS for the same slot count).  For ids below
// 2^idbits, h = id * 0x9E3779B1 mod 2^idbits is a bijection: its top gbits = hlog - 3 bits pick
// the home group of 8 slots (one 16-byte read), and a slot holds the other lob = idbits - gbits
// <= 13 bits as lo + 1 (never 0) with bits 14..15 = the displacement d <= 3 of the group that
// holds it.  Equal entries at equal displacement from equal homes mean equal h, hence equal ids,
// so the set is exact.  An id takes the first empty slot of the first group at d = 0..3 that has
// one (lookups stop there as in the 32-bit table); with none free in those 4 groups the insert
// reports an overflow and the caller continues in the global table.  Lanes inserting the same id
// read the same group state, choose the same slot and race through compare-and-swap on its word.
__device__ __forceinline__ void vis16_key(uint32_t id, int idbits, int gbits, uint32_t &home, uint32_t &lo1) {
    const uint32_t hm = idbits >= 32 ? 0xFFFFFFFFu : ((1u << idbits) - 1u);
    const uint32_t h = (id * 0x9E3779B1u) & hm;
    const int lob = idbits - gbits;
    home = h >> lob;
    lo1 = (h & ((1u << lob) - 1u)) + 1u;
}
// the zero 16-bit halves of x, flagged in bits 15 and 31: (x - 0x00010001) & ~x & 0x80008000.
// A zero low half is always flagged and a nonzero one never is; the high half's flag is exact
// unless the low half is zero (its borrow can flag a high half of 1).  So "some half is zero" and
// "the lowest zero half" read exactly from the flags.
__device__ __forceinline__ uint32_t zero_halves(uint32_t x) { return (x - 0x00010001u) & ~x & 0x80008000u; }
// some half of the group equals e (ee = e in both halves)
__device__ __forceinline__ bool group_has(const uint4 &v, uint32_t ee) {
    return (zero_halves(v.x ^ ee) | zero_halves(v.y ^ ee) | zero_halves(v.z ^ ee) | zero_halves(v.w ^ ee)) != 0u;
}
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_min16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
// 0: present, 1: inserted, 2: no room within 4 groups; every group from displacement d0 on
__device__ __forceinline__ int vis16_probe(uint32_t *vis, int gbits, uint32_t home, uint32_t lo1) {
    const uint32_t gmask = (1u << gbits) - 1u;
    for (uint32_t d = 0; d < 4u; ++d) {
        const uint32_t g = (home + d) & gmask;
        const uint32_t e = lo1 | (d << 14);
        for (;;) {
            const uint4 v = *reinterpret_cast<const uint4 *>(vis + (g << 2));
            if (group_has(v, e * 0x00010001u)) return 0;
            // the first empty slot: the first word with a zero half, then its lower zero half
            uint32_t old = v.x, z = zero_halves(v.x), wi = 0u;
            if (z == 0u) { old = v.y; z = zero_halves(v.y); wi = 1u; }
            if (z == 0u) { old = v.z; z = zero_halves(v.z); wi = 2u; }
            if (z == 0u) { old = v.w; z = zero_halves(v.w); wi = 3u; }
            if (z == 0u) break;  // group full: next displacement
            const uint32_t nw = old | (e << ((z & 0x8000u) ? 0 : 16));
            if (atomicCAS(&vis[(g << 2) + wi], old, nw) == old) return 1;
            lds_fence();  // the word changed: read the group again
        }
    }
    return 2;
}
// 0: present, 1: inserted, 2: no room within 4 groups.  The home group decides almost every id, so
// it is tested in straight line: the halves are compared by packed 16-bit minima, and, because a
// group fills its slots in order, it has room while its last half is zero and the first free word is
// the first one whose upper half is.  An id whose home group is full, or that lost the slot to
// another lane, takes the probe loop from the start.
__device__ __forceinline__ int vis16_insert(uint32_t *vis, int gbits, int idbits, uint32_t id) {
    uint32_t home, lo1;
    vis16_key(id, idbits, gbits, home, lo1);
    uint32_t *grp = vis + (home << 2);
    const uint4 v = *reinterpret_cast<const uint4 *>(grp);
    const uint32_t ee = lo1 * 0x00010001u;
    const uint32_t t = pk_min16(pk_min16(v.x ^ ee, v.y ^ ee), pk_min16(v.z ^ ee, v.w ^ ee));
    if ((t & 0xffffu) == 0u || t < 0x10000u) return 0;
    int r = 2;
    if (v.w < 0x10000u) {
        const bool fx = v.x >= 0x10000u, fy = v.y >= 0x10000u, fz = v.z >= 0x10000u;
        const uint32_t old = fz ? v.w : fy ? v.z : fx ? v.y : v.x;
        const uint32_t wi = fz ? 3u : fy ? 2u : fx ? 1u : 0u;
        const uint32_t nw = old == 0u ? lo1 : (old | (lo1 << 16));
        r = atomicCAS(&grp[wi], old, nw) == old ? 1 : 2;
        lds_fence();
    }
    if (r == 2) [[unlikely]] r = vis16_probe(vis, gbits, home, lo1);
    return r;
}
__device__ __forceinline__ bool vis16_test(const uint32_t *vis, int gbits, int idbits, uint32_t id) {
    uint32_t home, lo1;
    vis16_key(id, idbits, gbits, home, lo1);
    const uint32_t gmask = (1u << gbits) - 1u;
    for (uint32_t d = 0; d < 4u; ++d) {
        const uint32_t g = (home + d) & gmask;
        const uint32_t e = lo1 | (d << 14);
        const uint4 v = *reinterpret_cast<const uint4 *>(vis + (g << 2));
        if (group_has(v, e * 0x00010001u)) return true;
        if ((zero_halves(v.x) | zero_halves(v.y) | zero_halves(v.z) | zero_halves(v.w)) != 0u) return false;
    }
    return false;
}

// insert into a query's global spill table, one slot per probe (sub-groups of a wave, device-scope CAS)
__device__ __forceinline__ bool gvis_insert(uint32_t *g, uint32_t mask, int hlog, uint32_t id) {
    const uint32_t key = id + 1u;
    uint32_t s = (id * 0x9E3779B1u) >> (32 - hlog);
    for (;;) {
        const uint32_t old = atomicCAS(&g[s], 0u, key);
        if (old == 0u) return true;
        if (old == key) return false;
        s = (s + 1u) & mask;
    }
}

// The same table for a whole wave that owns it, without atomics: lanes with `want` insert their id and
// learn whether it was absent.  A lane reads its home group of four slots (16 bytes, one round trip);
// an id with a free slot there claims it through one LDS word per 64th of the slots (arb, 64 u32),
// so that lanes after the same slot -- the same id included -- take turns, and stores it without
// waiting.  An atomic compare-and-swap per probe, the other form, is a round trip to L2 for every
// lane and probe: the searches that outgrow their LDS table (the longest of a launch) spent most of
// their time on it.
__device__ __forceinline__ bool gvis_claim(uint32_t *g, int hlog, uint32_t id, bool want, uint32_t *arb) {
    const uint32_t key = id + 1u, gmask = (1u << (hlog - 2)) - 1u;
    const int lane = lane_id();
    uint32_t grp = (id * 0x9E3779B1u) >> (34 - hlog);
    bool fresh = false;
    bag_fence();
    while (ballot(want) != 0ull) {
        if (want) {
            const uint4 v = *reinterpret_cast<const uint4 *>(g + (grp << 2));
            const uint32_t e = v.x == 0u ? 0u : v.y == 0u ? 1u : v.z == 0u ? 2u : v.w == 0u ? 3u : 4u;
            if (v.x == key || v.y == key || v.z == key || v.w == key) {
                want = false;
            } else if (e == 4u) {
                grp = (grp + 1u) & gmask;
            } else {
                const uint32_t slot = (grp << 2) + e;
                arb[slot & 63u] = (uint32_t)lane;
                lds_fence();
                if (arb[slot & 63u] == (uint32_t)lane) {
                    g[slot] = key;
                    fresh = true;
                    want = false;
                }
            }
        }
        if (ballot(want) != 0ull) bag_fence();  // the stores above, before the groups are read again
    }
    return fresh;
}

// Blocked Bloom filter (the reference's BlockedBloomFilter, blocked_bloomfilter.h:9-82, with
// one 32-bit word per block): an id sets k bits of one word, all chosen by two murmur3
// finalizer mixes of the id -- the word from the top wlog bits of the first, the bit positions
// from 5-bit slices of the second (positions 7..9 from the first's low bits, below the word
// index for wlog <= 17).  Insert = one LDS atomic OR; the id counts as new unless all k bits
// were already set.  Lanes inserting the same id see exactly one "new" (the ORs serialise).
// No overflow and no deletion; a false positive skips a vertex that was never visited.
__device__ __forceinline__ uint32_t fmix32(uint32_t h) {
    h ^= h >> 16;
    h *= 0x85ebca6bu;
    h ^= h >> 13;
    h *= 0xc2b2ae35u;
    h ^= h >> 16;
    return h;
}
__device__ __forceinline__ uint32_t bloom_mask(uint32_t h1, uint32_t h2, int k) {
    uint32_t m = 0u;
#pragma unroll
    for (int i = 0; i < 6; ++i)
        if (i < k) m |= 1u << ((h2 >> (5 * i)) & 31u);
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (6 + i < k) m |= 1u << ((h1 >> (5 * i)) & 31u);
    return m;
}
__device__ __forceinline__ bool bloom_insert(uint32_t *bf, int wlog, int k, uint32_t id) {
    asm volatile("" : "+s"(k));  // its nine compares belong here, not hoisted out of the search loop
    const uint32_t h1 = fmix32(id * 2u + 1u), h2 = fmix32(id ^ 0x9E3779B9u);
    const uint32_t mask = bloom_mask(h1, h2, k);
    const uint32_t old = atomicOr(&bf[h1 >> (32 - wlog)], mask);
    return (old & mask) != mask;
}

// ---------------------------------------------------------------- distances

// Final distance from the accumulated dot/L2 sum, per reference data.h:28-62.
template <int METRIC>
__device__ __forceinline__ double finish_exact(double s, float lena, float lenv) {
    if (METRIC == M_L2) return s;
    if (METRIC == M_IP) return -s;
    int sign = s < 0 ? 1 : -1;
    return (double)sign * (s * s / (double)lena / (double)lenv);
}
template <int METRIC>
__device__ __forceinline__ float finish_f32(float s, float lena, float lenv) {
    if (METRIC == M_L2) return s;
    if (METRIC == M_IP) return -s;
    float sign = s < 0 ? 1.0f : -1.0f;
    return sign * (s * s / lena / lenv);
}

// One lane, sequential over the dimensions in the CPU's order (exact fallback).  Both operands are
// read in 16-byte units; the row and the query are zero past dim, and a zero product leaves the sum
// as it is.
template <int METRIC> __device__ __forceinline__ float product(float x, float q) {
    if (METRIC == M_L2) {
        const float d = x - q;
        return d * d;
    }
    return x * q;
}
template <int METRIC>
__device__ double seq_sum(const float *row, const float *qv, int dim) {
    const float4 *r4 = reinterpret_cast<const float4 *>(row);
    const float4 *q4 = reinterpret_cast<const float4 *>(qv);
    const int nu = (dim + 3) >> 2;
    double s = 0.0;
    float4 nx = r4[0];
    for (int j = 0; j < nu; ++j) {
        const float4 x = nx, q = q4[j];
        nx = r4[min(j + 1, nu - 1)];
        s += (double)product<METRIC>(x.x, q.x);
        s += (double)product<METRIC>(x.y, q.y);
        s += (double)product<METRIC>(x.z, q.z);
        s += (double)product<METRIC>(x.w, q.w);
    }
    return s;
}

// The same sums of 16 rows by a whole wave: lanes 4c .. 4c + 3 give row c's address, lane c returns
// its sum (c < 16).  What bounds the sum is its chain of double additions, one lane per row; the
// products of 64 dimensions at a time are made by all 64 lanes (4 per row, the next 64 dimensions'
// loads in flight) and handed over through LDS, so that the chain is a conversion and an addition per
// dimension.  With the loads, differences and products in the chain's own lane, 1,000 queries on rows of
// 960 dimensions took 9.31 ms and take 6.55 ms with the chain alone (242 -> 139 vector registers).
constexpr int SEQ_LD = 17;                      // float4s of a staged row: 16 and one to spread the banks
constexpr int SEQ_STAGE = 16 * SEQ_LD * 4;      // floats
template <int METRIC>
__device__ __forceinline__ double seq_sum16(const float *row, const float *qv, int dim, float *stage) {
    const int lane = lane_id(), c = lane >> 2, sub = lane & 3;
    const float4 *r4 = reinterpret_cast<const float4 *>(row);
    const float4 *q4 = reinterpret_cast<const float4 *>(qv);
    float4 *st = reinterpret_cast<float4 *>(stage);
    const int nu = (dim + 3) >> 2;
    double s = 0.0;
    float4 x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = r4[min(sub + 4 * i, nu - 1)];
    for (int u0 = 0; u0 < nu; u0 += 16) {
        lds_fence();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = u0 + sub + 4 * i;
            const float4 q = q4[min(u, nu - 1)];
            const bool in = u < nu;
            st[c * SEQ_LD + sub + 4 * i] =
                make_float4(in ? product<METRIC>(x[i].x, q.x) : 0.0f, in ? product<METRIC>(x[i].y, q.y) : 0.0f,
                            in ? product<METRIC>(x[i].z, q.z) : 0.0f, in ? product<METRIC>(x[i].w, q.w) : 0.0f);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = r4[min(u0 + 16 + sub + 4 * i, nu - 1)];
        lds_fence();
        if (lane < 16) {
#pragma unroll
            for (int h = 0; h < 16; h += 8) {
                float4 p[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) p[t] = st[lane * SEQ_LD + h + t];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    s += (double)p[t].x;
                    s += (double)p[t].y;
                    s += (double)p[t].z;
                    s += (double)p[t].w;
                }
            }
        }
    }
    lds_fence();
    return s;
}

// ---------------------------------------------------------------- row storage

// Base rows are read in 16-byte units.  ST_F32: the float32 rows (bfsg.data values,
// zero-padded); ST_BF16 / ST_FP8: a low-precision copy, value = code * scale[row], with a
// power-of-two scale for BF16 (lossless for integers up to 256) and max|x|/448 for FP8-E4M3.
enum { ST_F32 = 0, ST_BF16 = 1, ST_FP8 = 2 };
template <int STORE> struct Store;
template <> struct Store<ST_F32> { static constexpr int EPU = 4; };
template <> struct Store<ST_BF16> { static constexpr int EPU = 8; };
template <> struct Store<ST_FP8> { static constexpr int EPU = 16; };

template <int STORE>
__device__ __forceinline__ void decode_unit(const uint4 u, float (&x)[Store<STORE>::EPU]) {
    if constexpr (STORE == ST_F32) {
        x[0] = __uint_as_float(u.x); x[1] = __uint_as_float(u.y);
        x[2] = __uint_as_float(u.z); x[3] = __uint_as_float(u.w);
    } else if constexpr (STORE == ST_BF16) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            x[2 * t] = __uint_as_float(w[t] << 16);
            x[2 * t + 1] = __uint_as_float(w[t] & 0xffff0000u);
        }
    } else {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[t], false);
            const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[t], true);
            x[4 * t] = lo[0]; x[4 * t + 1] = lo[1]; x[4 * t + 2] = hi[0]; x[4 * t + 3] = hi[1];
        }
    }
}

// sum over the SUB lanes that share a row: xor steps SUB/2 .. 1, the last four as DPP moves inside a
// row of 16 lanes (a rotation by 4 stands for xor 4: after the xor 8 step lanes i and i ^ 8 agree)
template <int CTRL> __device__ __forceinline__ float dpp_f(float x) {
    return __uint_as_float(dpp32<CTRL>(__float_as_uint(x)));
}
template <int CTRL> __device__ __forceinline__ double dpp_d(double x) {
    return __longlong_as_double((long long)dpp64<CTRL>((uint64_t)__double_as_longlong(x)));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_ROR4 = 0x124, DPP_ROR8 = 0x128;
template <int SUB> __device__ __forceinline__ float sub_sum(float x) {
    if constexpr (SUB > 16)
        for (int o = SUB / 2; o > 8; o >>= 1) x += __shfl_xor(x, o);
    if constexpr (SUB > 8) x += dpp_f<DPP_ROR8>(x);
    if constexpr (SUB > 4) x += dpp_f<DPP_ROR4>(x);
    x += dpp_f<DPP_XOR2>(x);
    x += dpp_f<DPP_XOR1>(x);
    return x;
}
template <int SUB> __device__ __forceinline__ double sub_sum(double x) {
    if constexpr (SUB > 16)
        for (int o = SUB / 2; o > 8; o >>= 1) x += __shfl_xor(x, o);
    if constexpr (SUB > 8) x += dpp_d<DPP_ROR8>(x);
    if constexpr (SUB > 4) x += dpp_d<DPP_ROR4>(x);
    x += dpp_d<DPP_XOR2>(x);
    x += dpp_d<DPP_XOR1>(x);
    return x;
}
template <int SUB> __device__ __forceinline__ uint32_t sub_min(uint32_t x) {
    if constexpr (SUB > 16)
        for (int o = SUB / 2; o > 8; o >>= 1) x = min(x, (uint32_t)__shfl_xor((int)x, o));
    if constexpr (SUB > 8) x = min(x, dpp32<DPP_ROR8>(x));
    if constexpr (SUB > 4) x = min(x, dpp32<DPP_ROR4>(x));
    x = min(x, dpp32<DPP_XOR2>(x));
    x = min(x, dpp32<DPP_XOR1>(x));
    return x;
}

// the candidate whose key eval_candidates leaves in this lane: pass p = lane % SUB, group lane / SUB
template <int SUB> __device__ __forceinline__ int cand_of_lane() {
    return (lane_id() % SUB) * (64 / SUB) + lane_id() / SUB;
}

// Distances of the m candidates cid[0..m): lane l returns the key of candidate cand_of_lane<SUB>()
// (+inf when that is not below m).  SUB lanes share one row; each lane keeps its share of all rows of
// a pass in registers (up to NVU 16-byte units) so every row load of the pass is issued before the
// first use.  All SUB lanes of a row hold its sum, so the lane that keeps the key of pass p is
// simply the row's lane p: no key moves between lanes.  The units of a pass are processed in straight
// line (units past the row are clamped and their sum dropped by a select), so that the query's LDS
// reads and the row loads are all in flight together; with a branch per unit each unit waited for
// its own LDS reads.
// stage: LDS for the exact sums done again (SEQ_STAGE floats), or null.
template <int METRIC, bool EXACT, int STORE, int SUB, int NVU, class Key>
__device__ __forceinline__ Key eval_candidates(const SearchParams &P, int m, const uint32_t *cid, const float *qv,
                                               float lenv, float *stage = nullptr) {
    constexpr int EPU = Store<STORE>::EPU;
    const int lane = lane_id();
    constexpr int G = 64 / SUB;
    const int g = lane / SUB, sl = lane % SUB;
    const int nu = (STORE == ST_F32) ? (P.ld >> 2) : (int)(P.lp_stride >> 4);
    Key mine = Key::inf();
    bool redo = false;
    for (int base = 0; base < m; base += G) {
        const int c = base + g;
        if (c < m) {
            const uint32_t id = cid[c];
            const uint4 *row = (STORE == ST_F32)
                                   ? reinterpret_cast<const uint4 *>(P.data + (size_t)id * (size_t)P.ld)
                                   : reinterpret_cast<const uint4 *>(P.data_lp + (size_t)id * P.lp_stride);
            const float scale = (STORE != ST_F32) ? P.scale[id] : 1.0f;
            const float lena = (METRIC == M_COS) ? P.norms[id] : 0.0f;
            float facc = 0.0f;
            double dacc = 0.0, sab = 0.0;
            uint32_t umin = ~0u;
            // NVC units per lane from unit j0 on; MASKED: some may lie past the row
            const auto block = [&](int j0, auto masked, auto units) {
                constexpr bool MASKED = decltype(masked)::value;
                constexpr int NVC = decltype(units)::value;
                uint4 u[NVC];
#pragma unroll
                for (int v = 0; v < NVC; ++v) {
                    const int j = j0 + sl + v * SUB;
                    u[v] = row[MASKED ? min(j, nu - 1) : j];
                }
#pragma unroll
                for (int v = 0; v < NVC; ++v) {
                    const int j = j0 + sl + v * SUB;
                    const int jq = MASKED ? min(j, nu - 1) : j;
                    float x[EPU], q[EPU];
                    decode_unit<STORE>(u[v], x);
#pragma unroll
                    for (int t = 0; t < EPU; t += 4) {
                        const float4 q4 = *reinterpret_cast<const float4 *>(qv + jq * EPU + t);
                        q[t] = q4.x; q[t + 1] = q4.y; q[t + 2] = q4.z; q[t + 3] = q4.w;
                    }
                    const bool in = !MASKED || j < nu;
                    if constexpr (!EXACT) {
                        float f = facc;
#pragma unroll
                        for (int t = 0; t < EPU; ++t) {
                            const float xv = (STORE == ST_F32) ? x[t] : x[t] * scale;
                            if (METRIC == M_L2) {
                                const float d = xv - q[t];
                                f += d * d;
                            } else {
                                f += xv * q[t];
                            }
                        }
                        facc = in ? f : facc;
                    } else {
                        // float products (rounded), double accumulation; exact in any order when all
                        // products are multiples of 2^mn and sum |p| < 2^(mn+53).  2^mn from the
                        // smallest nonzero product's exponent (its last mantissa bit)
                        double f = dacc, sf = sab;
                        uint32_t um = umin;
#pragma unroll
                        for (int t = 0; t < EPU; ++t) {
                            float pr;
                            if (METRIC == M_L2) {
                                const float d = x[t] - q[t];
                                pr = d * d;
                            } else {
                                pr = x[t] * q[t];
                            }
                            f += (double)pr;
                            if (METRIC != M_L2) sf += (double)fabsf(pr);
                            um = min(um, (__float_as_uint(pr) & 0x7fffffffu) - 1u);
                        }
                        dacc = in ? f : dacc;
                        sab = in ? sf : sab;
                        umin = in ? um : umin;
                    }
                }
            };
            using T_ = std::true_type;
            using F_ = std::false_type;
            constexpr int CH = NVU * SUB;
            if (NVU == 2 && nu <= SUB) {
                block(0, T_{}, std::integral_constant<int, 1>{});
            } else {
                int j0 = 0;
                for (; j0 + CH <= nu; j0 += CH) block(j0, F_{}, std::integral_constant<int, NVU>{});
                if (j0 < nu) block(j0, T_{}, std::integral_constant<int, NVU>{});
            }
            Key k;
            bool seq = false;
            if constexpr (!EXACT) {
                k = Key::make_f(finish_f32<METRIC>(sub_sum<SUB>(facc), lena, lenv), id);
            } else {
                dacc = sub_sum<SUB>(dacc);
                const double tot = METRIC == M_L2 ? dacc : sub_sum<SUB>(sab);
                umin = sub_min<SUB>(umin);
                // every product zero (umin still all ones), or tot < 2^(mn + 53) with one bit to spare for
                // the rounding of tot itself: biased exponent of tot below mn + 53 + 1023 - 1
                const int mn = max((int)(umin >> 23), 1) - 150;
                const int te = (int)(((uint64_t)__double_as_longlong(tot) >> 52) & 2047u);
                seq = umin != ~0u && te - 1023 > mn + 51;
                k = Key::make_d(finish_exact<METRIC>(dacc, lena, lenv), id);
            }
            if (base == sl * G) {
                mine = k;
                redo = seq;
            }
        }
    }
    if constexpr (EXACT) {
        // sequential re-evaluation in the CPU's order of the flagged candidates: up to 16 at a time
        // through the stage, or one lane each
        const uint64_t todo = ballot(redo);
        if (todo != 0ull) {
            double s = 0.0;
            if (SUB * NVU > 64 && stage) {
                const int rank = lanes_below(todo), n = __popcll(todo);
                for (int c0 = 0; c0 < n; c0 += 16) {
                    const bool now = redo && rank >= c0 && rank < c0 + 16;
                    if (now) reinterpret_cast<uint32_t *>(stage)[rank - c0] = mine.id();
                    lds_fence();
                    const uint32_t id = reinterpret_cast<const uint32_t *>(stage)[min(lane >> 2, n - c0 - 1)];
                    const double t = seq_sum16<METRIC>(P.data + (size_t)id * (size_t)P.ld, qv, P.dim, stage);
                    const double got = __shfl(t, (rank - c0) & 63);
                    if (now) s = got;
                }
            } else if (redo) {
                s = seq_sum<METRIC>(P.data + (size_t)mine.id() * (size_t)P.ld, qv, P.dim);
            }
            if (redo) {
                const float lena = (METRIC == M_COS) ? P.norms[mine.id()] : 0.0f;
                mine = Key::make_d(finish_exact<METRIC>(s, lena, lenv), mine.id());
            }
        }
    }
    return mine;
}

// entries of arr[0..n), in any order, below x
template <class Key> __device__ __forceinline__ int count_below(const Key *arr, int n, const Key &x) {
    const int lane = rare_lane();
    int c = 0;
    for (int b0 = 0; b0 < n; b0 += 64) c += __popcll(ballot(b0 + lane < n && lt(arr[b0 + lane], x)));
    return c;
}

// ---------------------------------------------------------------- wave-wide key sets

__device__ __forceinline__ KeyF shfl_key(const KeyF &k, int src) {
    return KeyF{((uint64_t)(uint32_t)__shfl((int)(k.v >> 32), src) << 32) | (uint32_t)__shfl((int)k.v, src)};
}
__device__ __forceinline__ KeyD shfl_key(const KeyD &k, int src) {
    return KeyD{((uint64_t)(uint32_t)__shfl((int)(k.d >> 32), src) << 32) | (uint32_t)__shfl((int)k.d, src),
                (uint32_t)__shfl((int)k.i, src), 0u};
}
// the key order reversed (-> +inf, the largest key, only from the smallest possible one)
__device__ __forceinline__ KeyF flip(const KeyF &k) { return KeyF{~k.v}; }
__device__ __forceinline__ KeyD flip(const KeyD &k) { return KeyD{~k.d, ~k.i, 0u}; }
template <class Key> __device__ __forceinline__ Key kmin(const Key &a, const Key &b) { return lt(b, a) ? b : a; }
template <class Key> __device__ __forceinline__ Key kmax(const Key &a, const Key &b) { return lt(b, a) ? a : b; }

// Bitonic merge steps j = J/2 .. 1 over one key per lane: within blocks of K lanes the
// sequence ascends where (lane & K) == 0 and descends otherwise (K = 64: ascending).
template <class Key>
__device__ __forceinline__ Key bitonic_steps(Key v, int K, int J) {
    const int lane = rare_lane();
    const bool up = (lane & K) == 0;
    for (int j = J >> 1; j > 0; j >>= 1) {
        const Key o = shfl_key(v, lane ^ j);
        v = (((lane & j) == 0) == up) ? kmin(v, o) : kmax(v, o);
    }
    return v;
}

// The c = min(64, n) smallest keys of arr[0..n) (any order), ascending in lanes 0..c-1 with
// +inf above.  The first 64-key block is sorted (bitonic); each further block is compared with the
// running 64th smallest.  A block with no key below it is skipped, up to SEL_INSERT keys below it
// are inserted one at a time (rank by ballot, the lanes above shift up one), more are sorted and
// merged: min(best[i], block[63 - i]) holds the 64 smallest of both as a bitonic sequence.
// Bags are appended in nearly ascending order, so most blocks after the first are skipped or
// take a few insertions.
// FLIP: of the reversed order (the largest keys, reversed, the largest first).
constexpr int SEL_INSERT = 16;
template <bool FLIP = false, class Key>
__device__ __forceinline__ Key select64(const Key *arr, int n) {
    const int lane = rare_lane();
    const auto at = [&](int i) __attribute__((always_inline)) { return i < n ? (FLIP ? flip(arr[i]) : arr[i]) : Key::inf(); };
    Key best = at(lane);
    // two blocks' loads are in flight while one is sorted or scanned (two register slots, the
    // loop unrolled by two, so no slot is copied while its load is in flight)
    Key na = at(64 + lane);
    Key nb = at(128 + lane);
    for (int k = 2; k <= 64; k <<= 1) best = bitonic_steps(best, k, k);
    const auto take = [&](Key v) {
        uint64_t m = ballot(lt(v, best.rl(63)));
        if (__popcll(m) > SEL_INSERT) {
            for (int k = 2; k <= 64; k <<= 1) v = bitonic_steps(v, k, k);
            best = bitonic_steps(kmin(best, shfl_key(v, 63 - lane)), 64, 64);
        } else {
            for (; m != 0ull; m &= m - 1ull) {
                const Key x = v.rl(__builtin_ctzll(m));
                // rank 64 (x above the current 64th, lowered by earlier insertions): no change
                const int r = __popcll(ballot(lt(best, x)));
                const Key dn = shr1(best);  // (lane 0's is not used: it keeps its key or takes x)
                best = ksel(lane < r, best, ksel(lane == r, x, dn));
            }
        }
    };
    for (int b0 = 64; b0 < n; b0 += 128) {
        const Key va = na;
        if (b0 + 128 < n) na = at(b0 + 128 + lane);
        take(va);
        if (b0 + 64 < n) {
            const Key vb = nb;
            if (b0 + 192 < n) nb = at(b0 + 192 + lane);
            take(vb);
        }
    }
    return best;
}

// The r-th smallest (1-based, r <= n) distance key of arr[0..n), radix select on 8-bit digits
// from the top; hist: 256 u32 of this wave's LDS.
template <class Key>
__device__ uint64_t select_dk(const Key *arr, int n, int r, uint32_t *hist) {
    const int lane = rare_lane();
    uint64_t prefix = 0, pmask = 0;
    uint32_t need = (uint32_t)r;
    for (int shift = Key::DKBITS - 8; shift >= 0; shift -= 8) {
        for (int b = lane; b < 256; b += 64) hist[b] = 0u;
        lds_fence();
        for (int i = lane; i < n; i += 64) {
            const uint64_t d = arr[i].dk();
            if ((d & pmask) == prefix) atomicAdd(&hist[(uint32_t)(d >> shift) & 255u], 1u);
        }
        lds_fence();
        // lane l holds digits 4l..4l+3; an inclusive scan over the lanes finds the digit
        // where the count of smaller entries reaches `need`
        const uint32_t c0 = hist[4 * lane], c1 = hist[4 * lane + 1], c2 = hist[4 * lane + 2],
                       c3 = hist[4 * lane + 3];
        const uint32_t sum = c0 + c1 + c2 + c3;
        uint32_t incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = (uint32_t)__shfl_up((int)incl, o);
            if (lane >= o) incl += t;
        }
        const uint32_t excl = incl - sum;
        const int L = __builtin_ctzll(ballot(excl < need && incl >= need));
        uint32_t below = rl32(excl, L);
        int digit = 4 * L;
        const uint32_t d0 = rl32(c0, L), d1 = rl32(c1, L), d2 = rl32(c2, L);
        if (below + d0 < need) {
            below += d0;
            ++digit;
            if (below + d1 < need) {
                below += d1;
                ++digit;
                if (below + d2 < need) {
                    below += d2;
                    ++digit;
                }
            }
        }
        need -= below;
        prefix |= (uint64_t)digit << shift;
        pmask |= 255ull << shift;
        lds_fence();
    }
    return prefix;
}

// In-place compactions of arr[0..n) (order not kept); return the new count.  Entries only
// move left: the writes of block j land below the start of block j + 1, so they never touch
// the two blocks whose loads are in flight (issued two blocks ahead into two register slots,
// the loop unrolled by two), and block j's own slots are written only after its load is used.
template <class Key, class Keep>
__device__ __forceinline__ int compact(Key *arr, int n, Keep keep_fn) {
    const int lane = rare_lane();
    int out = 0;
    Key na = (lane < n) ? arr[lane] : Key::inf();
    Key nb = (64 + lane < n) ? arr[64 + lane] : Key::inf();
    const auto put = [&](int b0, const Key &e) {
        const bool keep = b0 + lane < n && keep_fn(e);
        const uint64_t km = ballot(keep);
        if (keep) arr[out + lanes_below(km)] = e;
        out += __popcll(km);
    };
    for (int b0 = 0; b0 < n; b0 += 128) {
        const Key ea = na;
        if (b0 + 128 < n) na = (b0 + 128 + lane < n) ? arr[b0 + 128 + lane] : Key::inf();
        put(b0, ea);
        if (b0 + 64 < n) {
            const Key eb = nb;
            if (b0 + 192 < n) nb = (b0 + 192 + lane < n) ? arr[b0 + 192 + lane] : Key::inf();
            put(b0 + 64, eb);
        }
    }
    return out;
}
template <class Key>
__device__ __forceinline__ int keep_dk_upto(Key *arr, int n, uint64_t dmax) {
    return compact(arr, n, [&](const Key &e) { return e.dk() <= dmax; });
}
template <class Key>
__device__ __forceinline__ int keep_above(Key *arr, int n, const Key &kx) {
    return compact(arr, n, [&](const Key &e) { return lt(kx, e); });
}

// shapes: (lanes per candidate row, 16-byte units per lane) by units per row
template <int SHAPE> struct Shape;
template <> struct Shape<0> { static constexpr int SUB = 4, NV = 2; };    // <= 8 units
template <> struct Shape<1> { static constexpr int SUB = 4, NV = 8; };    // <= 32 units
template <> struct Shape<2> { static constexpr int SUB = 4, NV = 16; };   // <= 64 units
template <> struct Shape<3> { static constexpr int SUB = 16, NV = 16; };  // <= 256 units
template <> struct Shape<4> { static constexpr int SUB = 64, NV = 16; };  // wider rows, chunked

// ---------------------------------------------------------------- two waves per query

// Two wavefronts per query (search_duo): the search wave runs search_query; the helper wave
// reads the search wave's predicted next expansion (the queue head it prefetches), and for that
// vertex's neighbours that are not yet visited computes the distances into a small LDS cache
// keyed by id, so that when the search wave expands that vertex its candidates' distances are
// usually there and the row gather leaves its dependent chain.  The helper only reads the
// search wave's visited table and never changes its state; a cache entry is the search key
// itself ((distance bits << 32) | id, one 64-bit LDS store), computed by the same code as the
// search wave's own, so results are unchanged whether or not an entry is used.
//
// Queries are separated by an epoch: at a new query the search wave bumps the epoch, waits
// (bounded) for the helper's acknowledgement -- given between two of its work units, after
// every store of the previous unit -- and only then clears and uses the cache; without the
// acknowledgement in time it searches that query without the cache.  The helper leaves when the
// search wave sets `done` after its last query.
struct DuoMail {
    uint32_t epoch, ack, tseq, tepoch, target, done, lenv_bits, pad[9];
};
constexpr int DUO_CACHE = 256;                 // cache entries (8 bytes each)
constexpr int DUO_ACK_SPINS = 4096;            // the search wave's bounded wait for the acknowledgement
constexpr int DUO_BYTES = (int)sizeof(DuoMail) + DUO_CACHE * 8 + 64 * 4;  // mailbox, cache, helper ids
__device__ __forceinline__ uint32_t duo_slot(uint32_t id) { return (id * 0x9E3779B1u) >> 24; }
__device__ __forceinline__ uint32_t lds_ld(const uint32_t *p) { return __atomic_load_n(p, __ATOMIC_ACQUIRE); }
__device__ __forceinline__ void lds_st(uint32_t *p, uint32_t v) { __atomic_store_n(p, v, __ATOMIC_RELEASE); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// ---------------------------------------------------------------- the search kernel

// What bounds it: the chain of one expansion (pop, visited probe, row gather, queue insert), most of
// it instruction and LDS latency, so its work is kept straight: probes and distances without
// branches per slot or unit, sums by DPP moves, keys inserted by lane shifts, no key moved between
// lanes through LDS.  Against the chain with LDS scatters, shuffles and per-unit branches (1M x 128
// L2 unless said; one launch): 10,000 queries at pq 704 13.75 -> 12.57 ms, 3,001 at pq 200 2.06 ->
// 1.79 ms, 48 at pq 128 816 -> 666 us; 5,000 cosine queries of 16 dimensions in exact arithmetic
// 1,005 -> 752 us; 1,000 queries on FP8 rows of 960 dimensions 2.16 -> 1.62 ms.
// One query on one wave: qi is the query, slot_q the wave's spill table, smem its LDS.
// BAGL: the queue's bag sits in the wave's LDS slice after the query (qcap keys) instead of in
// global memory -- for latency-bound launches with few waves per CU, where a refill or a
// truncation then scans LDS instead of waiting on global-memory round trips.
// HELP: the search wave of search_duo (float32 keys); duo = the mailbox and cache in LDS.
// BG: the best list's front in the slot's global region after the bag (float32 rows, bag in
// global memory); the launch sizes each slot's global region for it (bag_bytes + pq keys).
template <int METRIC, bool EXACT, int STORE, int SHAPE, bool BAGL = false, bool HELP = false, bool BG = false>
__device__ __forceinline__ void search_query(const SearchParams &P, const int qi, const int slot_q,
                                             unsigned char *smem, unsigned char *duo = nullptr) {
    using Key = typename KeySel<EXACT>::T;
    constexpr int SUB = Shape<SHAPE>::SUB, NV = Shape<SHAPE>::NV;
    constexpr int QH = 64;  // head entries: one per lane, ascending from lane h
    const int lane = lane_id();
    lds_fence();
    // per-query budgets are clamped to the launch's LDS sizing (pq) and output rows (out_ld)
    const int pq = P.pq_arr ? max(1, min(P.pq_arr[qi], P.pq)) : P.pq;
    const int k = max(0, min(min(P.k_arr ? P.k_arr[qi] : P.k, pq), P.out_ld));
    const uint32_t H = 1u << P.hlog;
    const uint32_t hmask = H - 1u;
    const uint32_t vis_limit = (H >> 2) * 3u;

    uint32_t *vis = reinterpret_cast<uint32_t *>(smem);
    const bool bloom = P.bloom_k > 0;
    const uint32_t vis_bytes = bloom ? (4u << P.hlog) : H * (P.vis16 ? 2u : 4u);
    const int gbits = P.hlog - 3;                               // compact table: groups of 8
    // the best list's front: LDS after the visited table, or (bglob: float32 rows, global bag) the
    // slot's global region after its bag
    static_assert(!BG || (STORE == ST_F32 && !BAGL), "the global front needs float32 rows and a global bag");
    constexpr bool bglob = BG;
    Key *B = reinterpret_cast<Key *>(smem + vis_bytes);
    // the front (computed where used, in rare paths, so that no registers hold a global
    // pointer through the loop)
    const auto Bf = [&]() -> Key * {
        if constexpr (BG)
            return reinterpret_cast<Key *>(P.gbag + (size_t)slot_q * P.gbag_stride + bag_bytes<Key>(P.qcap));
        else
            return B;
    };
    // global front: its stores are complete before it is read
    const auto front_fence = [&]() {
        if constexpr (BG) bag_fence();
    };
    uint32_t *cid = reinterpret_cast<uint32_t *>(B + (bglob ? 0 : ((P.pq + 1) & ~1)));  // 256 u32
    float *qv = reinterpret_cast<float *>(cid + 256);
    // bag, qcap keys: global memory (one region per slot), or this wave's LDS after the query
    float *stage = (EXACT && P.seq_stage) ? qv + P.qld : nullptr;  // SEQ_STAGE floats
    float *qv_end = qv + P.qld + ((EXACT && P.seq_stage) ? SEQ_STAGE : 0);
    Key *Bg = BAGL ? reinterpret_cast<Key *>(qv_end)
                   : reinterpret_cast<Key *>(P.gbag + (size_t)slot_q * P.gbag_stride);
    // the layout must fit the slice and the bag the launch allocated: otherwise flag the query
    // and touch neither (a host / kernel mismatch becomes an error, not out-of-range accesses)
    const unsigned char *lds_end = BAGL ? reinterpret_cast<unsigned char *>(Bg + P.qcap)
                                        : reinterpret_cast<unsigned char *>(qv_end);
    const size_t gneed = bglob ? bag_bytes<Key>(P.qcap) + (size_t)P.pq * sizeof(Key) : (size_t)P.qcap * sizeof(Key);
    if (lds_end - smem > (ptrdiff_t)P.wave_lds ||
        (!BAGL && (!P.gbag || gneed > P.gbag_stride))) {
        if (lane == 0 && P.out_flags) P.out_flags[qi] = F_BAD_LAUNCH;
        return;
    }

    for (uint32_t i = lane; i < (vis_bytes >> 4); i += 64) reinterpret_cast<uint4 *>(vis)[i] = make_uint4(0u, 0u, 0u, 0u);
    for (int i = lane; i < P.qld; i += 64) qv[i] = (i < P.dim) ? P.queries[(size_t)qi * P.dim + i] : 0.0f;
    lds_fence();

    float lenv = 0.0f;
    if (METRIC == M_COS) {
        // query norm in the CPU's order: lenv = fmaf(v[i], v[i], lenv) (data.h:55 under FMA contraction)
        if (lane == 0)
            for (int i = 0; i < P.dim; ++i) lenv = fmaf(qv[i], qv[i], lenv);
        lenv = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(lenv)));
    }

    // May a distance be summed in any order?  In exact mode always (a sum is exact in any order, or done
    // again in the CPU's); with float sums when rows and query are integers and every partial sum is
    // below 2^24.  Then up to 4 candidates take 16 lanes a row in place of Shape's 4: a quarter of the
    // row's serial work per lane, the same sums.
    constexpr bool WIDE = SUB == 4 && NV == 8 && STORE == ST_F32;
    bool any_order = WIDE && EXACT;
    if constexpr (WIDE && !EXACT && METRIC != M_COS) {
        if (P.int_rows) {
            float mn = INFINITY, mx = -INFINITY;
            bool whole = true;
            for (int i = lane; i < P.dim; i += 64) {
                const float v = qv[i];
                whole = whole && v == rintf(v);
                mn = fminf(mn, v);
                mx = fmaxf(mx, v);
            }
            for (int o = 32; o > 0; o >>= 1) {
                mn = fminf(mn, __shfl_xor(mn, o));
                mx = fmaxf(mx, __shfl_xor(mx, o));
            }
            const double a = METRIC == M_L2 ? (double)fmaxf(mx, P.row_max) - (double)fminf(mn, P.row_min)
                                            : (double)fmaxf(fabsf(P.row_max), fabsf(P.row_min));
            const double b = METRIC == M_L2 ? a : (double)fmaxf(fabsf(mx), fabsf(mn));
            any_order = ballot(!whole) == 0ull && (double)P.dim * a * b < 16777216.0;
        }
    }

    bool use_cache = false;
    uint32_t epoch = 0u, cache_hits = 0u;
    DuoMail *mail = nullptr;
    uint64_t *dcache = nullptr;
    if constexpr (HELP) {
        static_assert(!EXACT, "the helper's cache holds float32 keys");
        mail = reinterpret_cast<DuoMail *>(duo);
        dcache = reinterpret_cast<uint64_t *>(duo + sizeof(DuoMail));
        // new query (its vector and norm are in place): bump the epoch, wait for the helper to
        // acknowledge it, then clear the cache
        epoch = uni(lds_ld(&mail->epoch)) + 1u;
        if (lane == 0) {
            lds_st(&mail->lenv_bits, __float_as_uint(lenv));
            lds_st(&mail->epoch, epoch);
        }
        for (int s = 0; s < DUO_ACK_SPINS && !use_cache; ++s) {
            use_cache = uni(lds_ld(&mail->ack)) == epoch;
            if (!use_cache) __builtin_amdgcn_s_sleep(1);
        }
        if (use_cache)
            for (int i = lane; i < DUO_CACHE; i += 64) dcache[i] = ~0ull;
        lds_fence();
    }
    // the predicted next expansion, for the helper
    const auto publish = [&](uint32_t v) {
        if constexpr (HELP) {
            if (use_cache && lane == 0) {
                mail->target = v;
                mail->tepoch = epoch;
                lds_st(&mail->tseq, mail->tseq + 1u);
            }
        }
    };

    uint32_t flags = 0u;
    int steps = 0;
    uint32_t nvis = 0u;
    // statistics counters live in lane 0 of a vector register (read once at the end), which
    // keeps them out of the scalar registers the loop is short of
    uint32_t adj_words = 0u, pf_hits = 0u, refills = 0u, truncs = 0u;
    const uint32_t l0 = lane == 0 ? 1u : 0u;
    // visited spill: once the LDS table nears its load limit, new ids go to a global table
    // vmode: what an id is tested against -- the compact or the 32-bit LDS table, the Bloom filter, or
    // (after the switch) an LDS table and the global one
    enum { V_16 = 0, V_32 = 1, V_BLOOM = 2, V_SPILL = 3 };
    int vmode = bloom ? V_BLOOM : P.vis16 ? V_16 : V_32;
    uint32_t vstop = bloom ? ~0u : vis_limit - 64u;  // vertices beyond which the table switches
    uint32_t nglob = 0u;
    uint32_t *gv = nullptr;
    // the rest of this query's new ids go to the slot's global table, cleared here
    const auto to_spill = [&]() __attribute__((always_inline)) {
        vmode = V_SPILL;
        vstop = ~0u;
        gv = P.gvis + (size_t)slot_q * (1u << P.ghlog);
        for (uint32_t i = (uint32_t)rare_lane(); i < (1u << P.ghlog) / 4; i += 64)
            reinterpret_cast<uint4 *>(gv)[i] = make_uint4(0u, 0u, 0u, 0u);
    };
    const uint32_t glimit = ((1u << P.ghlog) >> 2) * 3u;
    int h = 0, nq = 0;
    // The best list (the pq smallest expanded keys): its largest nt <= 64 entries, the tail, ascending in
    // lanes [0, nt) of a register (+inf above), the other nf, the front, in memory in any order.  Only the
    // list's largest entry matters to the search, and expansions come out in nearly ascending order, so
    // almost all of them end in the tail; one below it is appended to the front.
    Key bt = Key::inf();
    int nt = 0, nf = 0;
    uint64_t bmax = ~0ull;  // distance key of the largest entry once the list is full
    // the queue head lives in registers: lanes [h, h + nq) hold its keys in ascending order
    Key hq = Key::inf();
    int bn = 0;          // bag entries: unsorted, all above T
    Key T = Key::inf();  // head entries <= T < bag entries (+inf while the bag is empty)

    // A wave-uniform key into the register head: a shift of the lanes below its rank into the consumed
    // lanes in front of the head, or, with none, of the lanes above it; then a full head gives its
    // largest key to the bag and lowers T.  Keys are distinct.  One key costs a compare, two lane
    // shifts and four selects and no LDS access; a merge that scattered head and new keys through LDS
    // took two dependent LDS round trips per expansion and the same work per new key.
    const auto push_head = [&](const Key &o) {
        const uint64_t below = ballot(lt(hq, o));  // (lanes outside [h, h + nq) hold +inf)
        const int r = __popcll(below);
        if (h > 0) [[likely]] {
            hq = ksel(in_mask(below >> 1), shl1(hq), hq);
            hq = ksel(in_mask(1ull << (h - 1 + r)), o, hq);
            --h;
            ++nq;
        } else {
            const bool full = nq == QH;
            if (full) {
                const Key top = hq.rl(QH - 1);
                if (lane == 0) Bg[bn] = ksel(r == QH, o, top);
                ++bn;
            }
            if (r < QH) {
                hq = ksel(in_mask(low_bits(r)), hq, shr1(hq));
                hq = ksel(in_mask(1ull << r), o, hq);
            }
            if (full) T = hq.rl(QH - 1);
            else ++nq;
        }
    };

    // start vertices (graph.h:175-181: vertex 0; the learned form passes its own), each
    // entered once through the visited set and placed in the queue in (dist, id) order
    {
        // entries >= n (0xFFFFFFFF pads shorter lists) are skipped; none left means vertex 0
        const int ne = P.entry ? P.n_entry : 1;
        uint32_t sid = (lane < ne) ? (P.entry ? P.entry[(size_t)qi * ne + lane] : 0u) : 0xFFFFFFFFu;
        bool use = lane < ne && (uint64_t)sid < P.n;
        if (ballot(use) == 0ull) {
            use = lane == 0;
            sid = 0u;
        }
        int ins = 0;
        if (use)
            ins = bloom ? (bloom_insert(vis, P.hlog, P.bloom_k, sid) ? 1 : 0)
                        : P.vis16 ? vis16_insert(vis, gbits, P.idbits, sid) : (vis_insert(vis, hmask, P.hlog, sid) ? 1 : 0);
        // no room for a start vertex (up to 64 in an empty table): the query is flagged and not
        // searched; the epilogue reports it for a re-run with a larger table
        if (ballot(ins == 2) != 0ull) flags |= F_VIS_OVF;
        const bool fresh = ins == 1;
        const uint64_t fm = ballot(fresh);
        const int m0 = __popcll(fm);
        if (fresh) cid[lanes_below(fm)] = sid;
        nvis = (uint32_t)m0;
        lds_fence();
        const Key k0 = eval_candidates<METRIC, EXACT, STORE, SUB, NV, Key>(P, m0, cid, qv, lenv, stage);
        for (uint64_t bits = ballot(cand_of_lane<SUB>() < m0); bits; bits &= bits - 1) push_head(k0.rl(__builtin_ctzll(bits)));
        lds_fence();
    }
    const int max_steps = P.steps_arr ? min(P.steps_arr[qi], P.max_steps) : P.max_steps;
    int settle = 0;  // lane 0 holds it

    // The adjacency row of the next expansion is asked for twice: `ahead`, of the predicted next vertex
    // right after the pop, a whole expansion early, which brings it into the caches; and `row`, of the
    // queue head when the expansion ends, which is the one used (nearly always the same row: a cache
    // hit that is there after the next pop).  Both loads are issued on every expansion and neither
    // register is written anywhere else on the common path, so no copy of a register whose load is in
    // flight -- which waits for that load, and for the bag's stores before it -- is ever needed.
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    uint32_t row_id = NONE, row = 0u, ahead = 0u;
    // all lanes load (lanes past the row read its last word and are never used: a row's
    // degree is below gstride), so the load needs no lane mask and no zero fill
    const int gshift = P.gstride == 32 ? 5 : 6;  // rows of 32 or 64 words
    const auto adj_row = [&](uint32_t v) -> uint32_t {
        return P.graph[((size_t)v << gshift) + (uint32_t)min(lane, P.gstride - 1)];
    };

    // one expansion; returns true to leave the loop
    const auto expand = [&]() -> bool {
        if (nq == 0 && bn == 0) [[unlikely]] return true;
        if (steps >= max_steps) [[unlikely]] {
            flags |= F_STEP_CAP;
            return true;
        }
        if (nq == 0) [[unlikely]] {
            // refill the head with the (up to) 64 smallest bag entries
            const int c = min(QH, bn);
            refills += l0;
            if constexpr (BAGL) lds_fence(); else bag_fence();
            const Key sel = select64(Bg, bn);
            hq = sel;  // +inf in lanes >= c
            const Key top = sel.rl(c - 1);
            h = 0;
            nq = c;
            bn = keep_above(Bg, bn, top);
            T = bn > 0 ? top : Key::inf();
            row_id = NONE;
            if constexpr (!BAGL) vm_drain();
        }
        const Key now = hq.rl(h);
        // stop rule, graph.h:188: |best| == pq and best.max.d < now.d (distance only, strict)
        if (nf + nt == pq && bmax < now.dk()) [[unlikely]] return true;
        ++steps;
        hq = ksel(in_mask(1ull << h), Key::inf(), hq);
        ++h;
        --nq;

        if (row_id == now.id()) [[likely]] {
            pf_hits += l0;
        } else {
            row = adj_row(now.id());
        }
        const uint32_t r = row;
        // (vertex 0's row when the head is empty: the load is issued on every expansion)
        const uint32_t next_id = nq > 0 ? hq.rl(h).id() : 0u;
        asm volatile("" ::"v"(ahead));  // the previous `ahead` has come in before `row` did
        ahead = adj_row(next_id);
        if (nq > 0) publish(next_id);

        // `now` into the pq-best list (push + pop-max of graph.h:193-195).  A sorted front cost a search
        // and a shift through memory for every expansion below the tail: 10,000 queries at pq 704 took
        // 12.57 ms with it and take 9.75 ms without (front in global memory; 14.1 and 12.8 ms in LDS).
        {
            // the tail's entries below `now` are its first c lanes, so the ballot itself is the mask of the
            // lanes that keep their entry
            const uint64_t below = ballot(lt(bt, now));
            const int c = __popcll(below);
            const bool full = nf + nt == pq;
            const bool in_tail = c > 0 || nf == 0;  // at or above the tail's smallest, or all is tail
            if (P.out_stats) [[unlikely]] {
                // the first k results change when fewer than k entries are smaller
                int p = nf + c;
                if (!in_tail) {
                    front_fence();
                    p = count_below(Bf(), nf, now);
                }
                if (p < k && lane == 0) settle = steps;
            }
            if (!full || c < nt) {
                if (in_tail && (full || nt < 64)) {
                    // lanes from c on move up one; of a full list the largest entry leaves
                    bt = ksel(in_mask(below), bt, shr1(bt));
                    bt = ksel(in_mask(1ull << c), now, bt);
                    if (!full) ++nt;
                    else if (nt < 64) bt = ksel(in_mask(1ull << nt), Key::inf(), bt);
                } else {
                    // a key joins the front: `now` if it is below the tail, else the tail's smallest, the
                    // lanes below c - 1 taking their upper neighbour's entry and `now` lane c - 1
                    if (lane == 0) Bf()[nf] = ksel(c == 0, now, bt);
                    ++nf;
                    if (c > 0) {
                        bt = ksel(in_mask(below >> 1), shl1(bt), bt);
                        bt = ksel(in_mask(1ull << (c - 1)), now, bt);
                    } else if (full) {
                        --nt;  // the largest entry leaves
                        bt = ksel(in_mask(1ull << nt), Key::inf(), bt);
                        if (nt == 0) [[unlikely]] {
                            // the front's largest entries become the tail
                            front_fence();
                            const Key sel = select64<true>(Bf(), nf);
                            nt = min(64, nf);
                            bt = flip(shfl_key(sel, (nt - 1 - lane) & 63));
                            bt = ksel(in_mask(low_bits(nt)), bt, Key::inf());
                            const Key low = bt.rl(0);
                            nf = compact(Bf(), nf, [&](const Key &e) { return lt(e, low); });
                            if constexpr (BG) vm_drain();
                        }
                    }
                }
                if (nf + nt == pq) bmax = bt.rl(nt - 1).dk();
                lds_fence();
            }
        }

        // neighbours of `now` in row order (graph.h:196-205)
        const int deg = (int)rl32(r, 0);
        adj_words += l0 * (1u + (uint32_t)deg);
        if (nvis > vstop) [[unlikely]] {
            if (!P.gvis) {
                flags |= F_VIS_OVF;
                return true;
            }
            to_spill();
        }
        bool fresh = false;
        const uint64_t nb = low_bits(deg + 1) & ~1ull;  // lanes 1..deg hold the neighbours
        if (vmode == V_16) [[likely]] {
            bool vovf = false;
            if (in_mask(nb)) {
                const int ins = vis16_insert(vis, gbits, P.idbits, r);
                fresh = ins == 1;
                vovf = ins == 2;
            }
            if (ballot(vovf) != 0ull) [[unlikely]] {
                // the compact table had no room near these ids: continue in the global table
                if (!P.gvis) {
                    flags |= F_VIS_OVF;
                    return true;
                }
                to_spill();
                if (gvis_claim(gv, P.ghlog, r, vovf, cid)) fresh = true;
            }
        } else if (vmode == V_32) {
            if (in_mask(nb)) fresh = vis_insert(vis, hmask, P.hlog, r);
        } else if (vmode == V_BLOOM) {
            if (in_mask(nb)) fresh = bloom_insert(vis, P.hlog, P.bloom_k, r);
        } else {
            bool in_lds = true;
            if (in_mask(nb)) in_lds = P.vis16 ? vis16_test(vis, gbits, P.idbits, r) : vis_test(vis, hmask, P.hlog, r);
            fresh = gvis_claim(gv, P.ghlog, r, !in_lds, cid);
        }
        const uint64_t fm = ballot(fresh);
        const int m = __popcll(fm);
        if (fresh) cid[lanes_below(fm)] = r;
        nvis += (uint32_t)m;
        if (vmode == V_SPILL) [[unlikely]] {
            nglob += (uint32_t)m;
            if (nglob + 64u > glimit) {
                flags |= F_VIS_OVF;
                return true;
            }
        }
        if (m == 0) return false;
        lds_fence();
        Key mine;
        bool have = cand_of_lane<SUB>() < m;
        bool cached = false;
        if constexpr (HELP) {
            if (use_cache) {
                // every candidate's distance in the helper's cache: no gather
                const uint64_t ce = fresh ? dcache[duo_slot(r)] : ~0ull;
                const bool hit = fresh && (uint32_t)ce == r;
                if (ballot(fresh && !hit) == 0ull) {
                    mine = KeyF{ce};
                    have = fresh;
                    cached = true;
                    cache_hits += l0;
                }
            }
        }
        if (!cached) {
            if (WIDE && any_order && m <= 4) {
                mine = eval_candidates<METRIC, EXACT, STORE, 16, 2, Key>(P, m, cid, qv, lenv, stage);
                have = cand_of_lane<16>() < m;
            } else {
                mine = eval_candidates<METRIC, EXACT, STORE, SUB, NV, Key>(P, m, cid, qv, lenv, stage);
            }
        }

        // ---- the candidates: at most T into the sorted head, above T into the bag
        const uint64_t cut = (nf + nt == pq) ? bmax : ~0ull;  // drop distance keys above cut
        const bool surv = have && mine.dk() <= cut;
        if (ballot(surv) == 0ull) return false;
        // (a row has at most 63 neighbours, each of which adds at most one key to the bag)
        if (bn + 63 > P.qcap) [[unlikely]] {
            // make room: drop bag entries beyond the pq-th smallest distance of head + bag
            // (ties kept) or beyond bmax; none of them can be expanded before the stop rule
            uint64_t dcut = (nf + nt == pq) ? bmax : ~0ull;
            truncs += l0;
            if constexpr (BAGL) lds_fence(); else bag_fence();
            if (pq <= nq) dcut = min(dcut, hq.rl(h + pq - 1).dk());
            else if (pq - nq <= bn) dcut = min(dcut, select_dk(Bg, bn, pq - nq, cid));
            bn = keep_dk_upto(Bg, bn, dcut);
            if constexpr (!BAGL) vm_drain();
            if (bn == 0) T = Key::inf();
            if (bn + 63 > P.qcap) {  // the tie group at the pq-th distance exceeds the slack
                flags |= F_Q_OVF;
                return true;
            }
        }
        const bool to_b = surv && lt(T, mine);
        const bool to_q = surv && !to_b;
        const uint64_t bm = ballot(to_b);
        if (to_b) Bg[bn + lanes_below(bm)] = mine;
        bn += __popcll(bm);
        for (uint64_t bits = ballot(to_q); bits; bits &= bits - 1) push_head(mine.rl(__builtin_ctzll(bits)));
        // the helper's target follows the queue head
        if constexpr (HELP)
            if (nq > 0 && hq.rl(h).id() != next_id) publish(hq.rl(h).id());
        return false;
    };
    while (flags == 0u && !expand()) {
        row_id = nq > 0 ? hq.rl(h).id() : NONE;
        row = adj_row(nq > 0 ? row_id : 0u);
    }
    // the whole best list in LDS (or, bglob, in the slot's global region) from here on
    if constexpr (BG) B = Bf();
    if (lane < nt) B[nf + lane] = bt;
    const int nbest = nf + nt;
    if constexpr (BG) bag_fence();
    else lds_fence();

    const int cnt = min(k, nbest);
    const size_t ob = (size_t)qi * (size_t)P.out_ld;
    if constexpr (STORE != ST_F32 && !EXACT) {
        if (P.rerank) {
            // exact FP32 distances for the whole pq-best list
            for (int base = 0; base < nbest; base += 64) {
                const int c = min(64, nbest - base);
                if (lane < c) cid[lane] = B[base + lane].id();
                lds_fence();
                const Key ex = eval_candidates<METRIC, false, ST_F32, 4, 8, Key>(P, c, cid, qv, lenv);
                if (cand_of_lane<4>() < c) B[base + cand_of_lane<4>()] = ex;
                lds_fence();
            }
        }
    }
    // output: the first k in ascending order (graph.h:209-215), 64 at a time
    for (int i0 = 0, n = nbest; i0 < k; i0 += 64) {
        Key e = Key::inf();
        if (i0 < cnt) {
            e = select64(B, n);
            if (i0 + 64 < cnt) {
                n = keep_above(B, n, e.rl(63));
                if constexpr (BG) bag_fence();
                else lds_fence();
            }
        }
        const int i = i0 + lane;
        if (i < k) {
            const bool ok = i < cnt;
            P.out_ids[ob + i] = ok ? e.id() : 0xFFFFFFFFu;
            if (P.out_dist) P.out_dist[ob + i] = ok ? e.dist() : __int_as_float(0x7f800000);
        }
    }
    if (lane == 0) {
        if (P.retry_list && (flags & (F_VIS_OVF | F_Q_OVF))) P.retry_list[atomicAdd(P.retry_count, 1u)] = (uint32_t)qi;
        if (P.out_flags) P.out_flags[qi] = flags;
        if (P.out_stats) {
            uint32_t *o = P.out_stats + 8 * (size_t)qi;
            o[0] = (uint32_t)steps;
            o[1] = nvis;
            o[2] = adj_words;
            o[3] = pf_hits;
            o[4] = (uint32_t)settle;
            o[5] = refills;
            o[6] = truncs;
            o[7] = cache_hits;
        }
    }
}

// One workgroup (one wave) per query of the launch.
template <int METRIC, bool EXACT, int STORE, int SHAPE, bool BG = false>
__global__ __launch_bounds__(64) void search_kernel(SearchParams P) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int slot_q = (int)blockIdx.x;
    const int qi = P.qidx ? (int)P.qidx[P.qbase + slot_q] : P.qbase + slot_q;
    search_query<METRIC, EXACT, STORE, SHAPE, false, false, BG>(P, qi, slot_q, smem);
}

// Persistent grid: every wave takes queries from the shared list until it is exhausted
// (each wave reaches the exit once *work_next passes *work_count).  A workgroup holds
// blockDim.x / 64 waves, each on its own wave_lds-byte slice of LDS and its own spill table.
template <int METRIC, bool EXACT, int STORE, int SHAPE, bool BAGL = false, bool BG = false>
__global__ __launch_bounds__(256) void search_persistent(SearchParams P) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int w = (int)(threadIdx.x >> 6);
    const int slot = (int)blockIdx.x * (int)(blockDim.x >> 6) + w;
    unsigned char *mine = smem + (size_t)w * P.wave_lds;
    const uint32_t count = *P.work_count;
    // a tier whose searches are the longest runs at raised issue priority, so that waves of
    // concurrently running tiers on the same SIMDs do not stretch its critical path
    if (P.wave_prio) __builtin_amdgcn_s_setprio(2);
    for (;;) {
        // Every lane issues the add (lane 0 adds 1, the others 0) and lane 0's old value is
        // broadcast.  No lane-0 branch here: the query's lane-0 epilogue ends the previous
        // iteration, and a second branch on the same predicate lets the compiler thread the
        // back edge so that lanes 1..63 start the next iteration without lane 0.
        const uint32_t v = atomicAdd(P.work_next, lane_id() == 0 ? 1u : 0u);
        const uint32_t t = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
        if (t >= count) break;
        const int qi = P.qidx ? (int)P.qidx[t] : (int)t;
        search_query<METRIC, EXACT, STORE, SHAPE, BAGL, false, BG>(P, qi, slot, mine);
    }
}

// The helper wave of search_duo (see DuoMail): slice = the search wave's LDS slice.
template <int METRIC, int STORE, int SHAPE, bool BG>
__device__ void duo_helper(const SearchParams &P, unsigned char *slice, unsigned char *duo) {
    constexpr int SUB = Shape<SHAPE>::SUB, NV = Shape<SHAPE>::NV;
    const int lane = lane_id();
    DuoMail *mail = reinterpret_cast<DuoMail *>(duo);
    uint64_t *dcache = reinterpret_cast<uint64_t *>(duo + sizeof(DuoMail));
    uint32_t *hid = reinterpret_cast<uint32_t *>(dcache + DUO_CACHE);
    // the search wave's layout (search_query): visited | pq keys (not with bglob) | 256 u32 | qv
    const uint32_t H = 1u << P.hlog;
    const uint32_t vis_bytes = H * (P.vis16 ? 2u : 4u);
    const uint32_t *vis = reinterpret_cast<const uint32_t *>(slice);
    const KeyF *B = reinterpret_cast<const KeyF *>(slice + vis_bytes);
    const uint32_t *cid = reinterpret_cast<const uint32_t *>(B + (BG ? 0 : ((P.pq + 1) & ~1)));
    const float *qv = reinterpret_cast<const float *>(cid + 256);
    uint32_t my_epoch = 0u, last_t = 0u;
    float lenv = 0.0f;
    for (;;) {
        uint32_t t = 0u;
        for (;;) {
            if (uni(lds_ld(&mail->done))) return;
            const uint32_t e = uni(lds_ld(&mail->epoch));
            if (e != my_epoch) {
                // everything this wave stored for the previous epoch is written: acknowledge
                my_epoch = e;
                lenv = __uint_as_float(uni(lds_ld(&mail->lenv_bits)));
                lds_fence();
                if (lane == 0) lds_st(&mail->ack, e);
            }
            t = uni(lds_ld(&mail->tseq));
            if (t != last_t) break;
            __builtin_amdgcn_s_sleep(2);
        }
        last_t = t;
        const uint32_t v = uni(mail->target), te = uni(mail->tepoch);
        if (te != my_epoch || (uint64_t)v >= P.n) continue;
        const uint32_t r = P.graph[(size_t)v * (size_t)P.gstride + (uint32_t)min(lane, P.gstride - 1)];
        const int deg = (int)rl32(r, 0);
        bool want = false;
        if (lane >= 1 && lane <= deg)
            want = !(P.vis16 ? vis16_test(vis, P.hlog - 3, P.idbits, r) : vis_test(vis, H - 1u, P.hlog, r));
        const uint64_t fm = ballot(want);
        const int m = __popcll(fm);
        if (m == 0) continue;
        if (want) hid[lanes_below(fm)] = r;
        lds_fence();
        const KeyF k = eval_candidates<METRIC, false, STORE, SUB, NV, KeyF>(P, m, hid, qv, lenv);
        if (cand_of_lane<SUB>() < m) dcache[duo_slot(k.id())] = k.v;
        lds_fence();
    }
}

// Two waves per query, one query per workgroup at a time: wave 0 searches (the persistent work
// loop of search_persistent), wave 1 helps (duo_helper).  LDS: the search wave's wave_lds slice,
// then DUO_BYTES of mailbox, cache and helper ids.
template <int METRIC, int STORE, int SHAPE, bool BG = false>
__global__ __launch_bounds__(128) void search_duo(SearchParams P) {
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *duo = smem + P.wave_lds;
    if (threadIdx.x < sizeof(DuoMail) / 4) reinterpret_cast<uint32_t *>(duo)[threadIdx.x] = 0u;
    __syncthreads();
    // both waves of a prioritised tier: the helper's distances are on the search wave's path
    if (P.wave_prio) __builtin_amdgcn_s_setprio(2);
    if (threadIdx.x >= 64) {
        duo_helper<METRIC, STORE, SHAPE, BG>(P, smem, duo);
        return;
    }
    const uint32_t count = *P.work_count;
    for (;;) {
        // every lane issues the add (see search_persistent)
        const uint32_t v = atomicAdd(P.work_next, lane_id() == 0 ? 1u : 0u);
        const uint32_t t = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
        if (t >= count) break;
        const int qi = P.qidx ? (int)P.qidx[t] : (int)t;
        search_query<METRIC, false, STORE, SHAPE, false, true, BG>(P, qi, (int)blockIdx.x, smem, duo);
    }
    lds_fence();
    if (lane_id() == 0) lds_st(&reinterpret_cast<DuoMail *>(duo)->done, 1u);
}

}  // namespace song
