// Differential weight cache resident in HBM.
//
// update = ONE kernel.  Every block (1024 threads) first replays the
// bookkeeping of WeightCache::update_active_weights
// (sparse_transformers/csrc/weight_cache.h:229-359) redundantly in its own LDS
// (integer work only, identical in every block):
//   diff      ascending added / removed lists     (weight_cache.h:84-110)
//   phase 1   i-th removed position <- i-th added  (:248-277)   parallel
//   phase 2   surplus additions appended           (:280-307)   parallel
//   phase 3   surplus removals, swap-with-last     (:310-353)   parallel: where
//             the entries of the tail go does not depend on the steps (surplus_ends)
// and then copies its share of the changed rows with 16-byte loads/stores.
// The plan only decides WHICH index ends up at WHICH position.  Because every
// active row is a bit-copy of a pool row, the data movement never has to
// follow the sequential order: each position whose index changed is rewritten
// straight from the pool (no reads of the active buffers, hence no hazards
// between copies).
//
// The bookkeeping (index list, remembered mask, count) is double-buffered:
// blocks read buffer `epoch`, one block writes buffer `epoch ^ 1`, and the
// block that arrives last (a ticket counter packed with the epoch in one word)
// flips the epoch.  Nothing ever waits: a block that starts late still reads
// the old buffer, because nobody writes it during this launch.
#include "st_common.h"

#include <atomic>
#include <chrono>

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <type_traits>

namespace st {

constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / kWave;
constexpr uint16_t kNone = 0xffffu;
// LDS per intermediate element: pos(2) + idx(2) + added/removed lists(2) + flags(1) + dirty(1/8)
constexpr int64_t kPlanMaxI = 22000;

// Block barrier that orders LDS traffic only.  __syncthreads() also waits for every outstanding global
// load, which would serialise loads that are meant to stay in flight across the bookkeeping phases.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, int lane)
{
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t o = __shfl_up(v, off, kWave);
        if (lane >= off) v += o;
    }
    return v;
}

// The same with DPP row shifts (no LDS crossbar traffic): four steps scan each row of 16 lanes, the row totals
// travel through scalar registers.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_shr_add(uint32_t v)
{
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);   // lanes shifted in from outside the row read 0
}
__device__ __forceinline__ uint32_t wave_incl_scan_dpp(uint32_t v, int lane)
{
    v = dpp_shr_add<0x111>(v);   // row_shr:1
    v = dpp_shr_add<0x112>(v);   // row_shr:2
    v = dpp_shr_add<0x114>(v);   // row_shr:4
    v = dpp_shr_add<0x118>(v);   // row_shr:8
    const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15), t1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31),
                   t2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
    const int row = lane >> 4;
    return v + (row >= 1 ? t0 : 0u) + (row >= 2 ? t1 : 0u) + (row >= 3 ? t2 : 0u);
}

// Exclusive scan of one uint32 per thread over WAVES waves; *total receives the sum.  `sync` is the
// barrier of exactly those waves.
template <int WAVES, typename S>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *wave_tot, uint32_t *total, int tid, S sync)
{
    const int lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t incl = wave_incl_scan(v, lane);
    sync();  // protect wave_tot from the previous use
    if (lane == kWave - 1) wave_tot[wave] = incl;
    sync();
    uint32_t prefix = 0, tot = 0;
    for (int w = 0; w < WAVES; ++w) {
        const uint32_t t = wave_tot[w];
        if (w < wave) prefix += t;
        tot += t;
    }
    *total = tot;
    return prefix + incl - v;
}

// Does any thread of the block see `v`?  (uniform)
template <int TPB, typename S>
__device__ __forceinline__ bool any_of_block(bool v, uint32_t *wave_tot, int tid, S sync)
{
    const bool w = __builtin_amdgcn_ballot_w64(v) != 0;
    sync();
    if ((tid & (kWave - 1)) == 0) wave_tot[tid >> 6] = w ? 1u : 0u;
    sync();
    uint32_t r = 0;
    for (int k = 0; k < TPB / kWave; ++k) r |= wave_tot[k];
    return r != 0;
}

struct CopyPlan {
    const unsigned char *pool[3];
    unsigned char *active[3];
    int nmat;
    int row_bytes;
};

// The same matrices for the fused update + MLP kernel, by name (no arrays: nothing for the compiler to index).
// Without a gate the gate members repeat the up members and are not used.
struct FusedRows {
    const unsigned char *pool_g, *pool_u, *pool_d;
    unsigned char *act_g, *act_u, *act_d;
    int row_bytes, has_gate;
};

__device__ __forceinline__ uint64_t nonzero_bytes(uint64_t x)
{
    x |= x >> 4; x |= x >> 2; x |= x >> 1;
    return x & 0x0101010101010101ull;
}

// 0x01-per-element bytes -> 8 bits (element k -> bit k)
__device__ __forceinline__ uint32_t pack_bits8(uint64_t ones)
{
    return (uint32_t)((ones * 0x0102040810204080ull) >> 56);
}

// Eight bytes of a mask and four entries of an index list.  AL: the size is a multiple of eight and the buffers are aligned for
// words.  Otherwise at any alignment: sizes that are no multiples of eight put the second half of the double buffers, and the
// masks of a stack's layers, anywhere.  (The loads are the same instructions.)  The last word of such a mask, or the last
// vector of a list, is the one that ends with it; mask_tail and list_tail shift its first elements down, at the place of use:
// shifted where it is loaded, the load would be waited for there.  I >= 8; what lies past I reads as zero in a mask and as
// anything in a list.  I 3405, H 896, bf16, eight rows, a stack of four layers: 86 us with the updates byte by byte, layer by
// layer; 70 so, in one launch.  One or two rows of x also get the fused kernel.  With one form for both, which is a tenth more
// code to fetch, aligned calls of that kernel were slower: H 896, I 2688, bf16, one / two rows 13.9 / 18.4 us, and
// 14.1 / 18.9 so.
template <bool AL> __device__ __forceinline__ uint64_t load_mask(const uint8_t *m, int e, int I)
{
    if constexpr (AL) return *reinterpret_cast<const uint64_t *>(m + e);
    uint64_t v;
    __builtin_memcpy(&v, m + (e < I - 8 ? e : I - 8), 8);
    return v;
}
template <bool AL> __device__ __forceinline__ uint64_t mask_tail(uint64_t v, int e, int I)
{
    if constexpr (AL) return v;
    const int over = e + 8 - I;   // (words past the end, all of whose elements are, come out as anything)
    return v >> (8 * (over > 0 ? over : 0) & 63);
}
template <bool AL> __device__ __forceinline__ void store_mask(uint8_t *m, int e, int I, uint64_t v)
{
    if constexpr (AL) {
        *reinterpret_cast<uint64_t *>(m + e) = v;
    } else if (e + 8 <= I) {
        __builtin_memcpy(m + e, &v, 8);
    } else {
        for (int k = 0; k < I - e; ++k) m[e + k] = (uint8_t)(v >> (8 * k));
    }
}
typedef int list4_t __attribute__((ext_vector_type(4), aligned(4)));
template <bool AL> __device__ __forceinline__ int4 load_list(const int32_t *l, int p, int I)
{
    if constexpr (AL) return *reinterpret_cast<const int4 *>(l + p);
    const list4_t v = *reinterpret_cast<const list4_t *>(l + (p < I - 4 ? p : I - 4));
    return make_int4(v.x, v.y, v.z, v.w);
}
template <bool AL> __device__ __forceinline__ int4 list_tail(int4 c, int p, int I)
{
    if constexpr (AL) return c;
    if (I & 3) {   // uniform
        const int over = p + 4 - I;
        const bool one = over > 0 && (over & 1), two = over > 0 && (over & 2);
        c.x = one ? c.y : c.x; c.y = one ? c.z : c.y; c.z = one ? c.w : c.z;
        c.x = two ? c.z : c.x; c.y = two ? c.w : c.y;
    }
    return c;
}

// The plan as every block computes it, and the LDS arrays that hold it.
struct PlanView {
    uint16_t *pos_l;    // index -> position (kNone when absent)
    uint16_t *idx_l;    // position -> index, after the update
    uint16_t *lists;    // positions to rewrite: [0, n_changed)
    uint32_t *dirty;    // bit per position whose index changed (complete only with MARK, or on the slow path)
    int ep;             // bookkeeping buffer this launch read
    bool writer;        // this block publishes
    bool arriver;       // this thread issued the block's arrival
    uint32_t arrival;   // arriver only: ticket word before this block's arrival (requested, not yet looked at)
    int next_epoch;     // epoch the last arrival leaves behind
    bool changed;       // false: the mask equals the remembered one, nothing was touched
    int n_old, n_new, na, nr;
    uint32_t n_changed;
};

constexpr size_t plan_lds_bytes(int I)
{
    return (size_t)((I + 7) & ~7) * 4 + (size_t)I * 2 + (size_t)(I & 1) * 2 + (size_t)((((I + 31) >> 5) + 1) & ~1) * 4 + (size_t)I + 16;
}

// Small block-wide scalars of the plan (static LDS, declared by the kernel so that waves which do not take
// part in the plan can read them).
struct PlanShared {
    uint32_t wave_tot[kPlanWaves];
    int n_new_s;   // count after the surplus removals
};

// Phase 3 (weight_cache.h:310-353): S surplus indices e_0 < e_1 < ... leave the list of n entries one by one, step k moving
// the entry that is last at the time (slot n-1-k, a "tail slot") to where e_k is at the time.  Every step depends on the
// list the previous one left, but the outcome does not need the steps: join tail slot n-1-k to the slot e_k starts in, for
// every k.  No two tail slots are joined to the same slot, so the joins form paths (and closed loops of tail slots, all of
// whose entries leave).  A step moves an entry only along its path, and a path begins at an entry of the tail that stays --
// nothing is joined to its slot -- and ends at a slot in front of the tail: the only slot of the path that is left in the
// end, so that is where the entry goes, whatever the order of the steps.  All paths are followed at once, a thread per tail
// slot, every slot pointing at least twice as far along after each round (usual churn has paths of one or two slots, which
// takes no round or one).
// H 3072, I 8192, an update of 2000 removals with its copies, between events: one path through all of them 15 us (chased in
// the order of the steps it took 1969 rounds, 1670 us), in random order 23 us (more rows to copy; 24 before).
//
// place(k): the position e_k starts at (kNone: not in the list, no step at all: only after an update that failed; the others
// move up).  Returns the count after the steps (in every thread); ends behind a barrier.
template <int TPB, typename P, typename S>
__device__ __forceinline__ int surplus_count(P place, int S_all, int n, uint32_t *wave_tot, int *shared_n, int tid, S sync)
{
    bool missing = false;
    for (int k = tid; k < S_all; k += TPB) missing = missing || place(k) == kNone;
    int S_ = S_all;
    if (any_of_block<TPB>(missing, wave_tot, tid, sync)) {
        if (tid == 0) {
            int m = 0;
            for (int k = 0; k < S_all; ++k)
                if (place(k) != kNone) { const uint16_t v = place(k); place(m) = v; ++m; }
            *shared_n = m;
        }
        sync();
        S_ = *shared_n;
    }
    return n - S_;
}

// Behind a barrier after surplus_count (base: its result): place(k) becomes the slot the path of tail slot n-1-k ends at,
// where stays(k): whether that slot's entry stays.
template <int TPB, typename P, typename Q, typename S>
__device__ __forceinline__ void surplus_ends(P place, Q stays, int base, int n, uint32_t *wave_tot, int tid, S sync)
{
    constexpr int kHops = 4, kRounds = 16;   // (2^16 slots; the bound is never met)
    bool open = false;
    for (int k = tid; k < n - base; k += TPB) open = open || (place(k) >= base && stays(k));
    for (int round = 0; any_of_block<TPB>(open, wave_tot, tid, sync) && round < kRounds; ++round) {
        open = false;
        for (int k = tid; k < n - base; k += TPB) {
            int q = place(k);
            if (q < base) continue;
            // (the others move on at the same time: whatever is read lies further along the same path)
            for (int hop = 0; hop < kHops && q >= base; ++hop) q = place(n - 1 - q);
            place(k) = (uint16_t)q;
            open = open || (q >= base && stays(k));
        }
    }
}

// Replays the bookkeeping of one update in LDS and publishes it (block 0 writes the other bookkeeping
// buffer, the last block to arrive flips the epoch).  Called by all PT threads of the block (tid = 0..PT-1);
// contains block barriers.  VEC (I >= 8): masks are read as 8-byte words and indices as 16-byte vectors; both bookkeeping
// buffers are requested together with the ticket, so the front costs one memory round trip.  MARK: the
// dirty bitmap is kept on the fast path too.
// NW: 8-element words per thread of the vector path (I <= 8 NW threads); the registers of the front loads follow from it.  AL: as above.
//
// Barrier sequence: 1 after the LDS fill; 2 in the diff scan;
// [unchanged mask: done]; 1 after the lists; 1 after phases 1 and 2; [surplus removals: those of surplus_count and surplus_ends and 1
// behind it, 2 in the compaction scan, 1 after the compaction].
template <bool VEC, int PT, int NW, bool MARK, bool AL>
__device__ __forceinline__ void cache_plan(PlanView &pv, unsigned char *smem, PlanShared *ps,
                                           const uint8_t *__restrict__ new_mask, uint8_t *__restrict__ cur_mask2,
                                           int32_t *__restrict__ indices2, int32_t *__restrict__ state, int I,
                                           const int tid)
{
    constexpr int TPB = PT;
    uint16_t *pos_l = reinterpret_cast<uint16_t *>(smem);  // index -> position
    const int span = AL ? I : (I + 7) & ~7;                // (the last words and vectors are written whole)
    uint16_t *idx_l = pos_l + span;                        // position -> index
    // added indices ascending from the front, removed indices ascending from the
    // back (k-th removed at lists[I-1-k]); the two never meet: na + nr <= I.
    // After the plan the same array holds the positions to rewrite.
    uint16_t *lists = idx_l + span;
    uint32_t *dirty = reinterpret_cast<uint32_t *>(lists + I + (I & 1));  // bit per position
    const int dirty_words = (I + 31) >> 5;
    uint8_t *flag_l = reinterpret_cast<uint8_t *>(dirty + ((dirty_words + 1) & ~1));  // bit0 new, bit1 old; 8-byte aligned
    uint32_t *wave_tot = ps->wave_tot;
    int &n_new_s = ps->n_new_s;
    auto sync = [&]() __attribute__((always_inline)) { lds_barrier(); };
    pv.pos_l = pos_l; pv.idx_l = idx_l; pv.lists = lists; pv.dirty = dirty;
    pv.arriver = tid == 0;

    ST_TL(0);
    // Elements per thread (a contiguous range, so the diff lists come out ascending).
    const int E = VEC ? ((I + 8 * TPB - 1) / (8 * TPB)) * 8 : (I + TPB - 1) / TPB;
    const int e0 = tid * E < I ? tid * E : I, e1 = e0 + E < I ? e0 + E : I;

    // The ticket word holds the epoch (bit 16: which buffer to read) and the arrivals so far.  Every thread
    // reads it with a plain load, together with the rest of the front; the epoch cannot flip before every
    // block has arrived, and a block arrives (one atomic, at the end of the plan) only after all its
    // threads have consumed this load, so they all see the same epoch.
    const uint32_t tword = __hip_atomic_load(reinterpret_cast<const uint32_t *>(&state[ST_STATE_TICKET]), __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);

    // (several small arrays rather than one big one: each has to stay below the size up to which the
    // compiler keeps a private array in registers)
    uint64_t v_new[NW], v_cur0[NW], v_cur1[NW];
    int4 v_i0a[NW], v_i0b[NW], v_i1a[NW], v_i1b[NW];
    int n_both[2];
    if constexpr (VEC) {
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int e = e0 + 8 * w;
            if (e < e1) {
                v_new[w] = load_mask<AL>(new_mask, e, I);
                v_cur0[w] = load_mask<AL>(cur_mask2, e, I);
                v_cur1[w] = load_mask<AL>(cur_mask2 + I, e, I);
                v_i0a[w] = load_list<AL>(indices2, e, I);
                v_i0b[w] = load_list<AL>(indices2, e + 4, I);
                v_i1a[w] = load_list<AL>(indices2 + I, e, I);
                v_i1b[w] = load_list<AL>(indices2 + I, e + 4, I);
            }
        }
        n_both[0] = state[ST_STATE_N_BUF0];
        n_both[1] = state[ST_STATE_N_BUF1];
    }
    for (int w = tid; w < dirty_words; w += TPB) dirty[w] = 0u;
    const int ep = (int)((tword >> 16) & 1u);
    const bool writer = blockIdx.x == 0;
    pv.ep = ep; pv.writer = writer;

    int n;
    // VEC: new / current mask words as 0x01 bytes, kept in registers for the diff and for publishing
    uint64_t w_new[NW], w_cur[NW];
    if constexpr (VEC) {
        n = ep ? n_both[1] : n_both[0];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int e = e0 + 8 * w;
            w_new[w] = w_cur[w] = 0;
            if (e < e1) {
                w_new[w] = nonzero_bytes(mask_tail<AL>(v_new[w], e, I));
                w_cur[w] = nonzero_bytes(mask_tail<AL>(ep ? v_cur1[w] : v_cur0[w], e, I));
                const int4 a = list_tail<AL>(ep ? v_i1a[w] : v_i0a[w], e, I), b4 = list_tail<AL>(ep ? v_i1b[w] : v_i0b[w], e + 4, I);
                uint4 packed;
                packed.x = (uint32_t)(a.x & 0xffff) | ((uint32_t)a.y << 16);
                packed.y = (uint32_t)(a.z & 0xffff) | ((uint32_t)a.w << 16);
                packed.z = (uint32_t)(b4.x & 0xffff) | ((uint32_t)b4.y << 16);
                packed.w = (uint32_t)(b4.z & 0xffff) | ((uint32_t)b4.w << 16);
                *reinterpret_cast<uint4 *>(idx_l + e) = packed;
                *reinterpret_cast<uint4 *>(pos_l + e) = make_uint4(0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu);
            }
        }
    } else {
        const uint8_t *cur_mask = cur_mask2 + (size_t)ep * I;
        const int32_t *indices = indices2 + (size_t)ep * I;
        n = state[ST_STATE_N_BUF0 + ep];
        for (int i = tid; i < I; i += TPB) {
            pos_l[i] = kNone;
            flag_l[i] = (new_mask[i] ? 1 : 0) | (cur_mask[i] ? 2 : 0);
            idx_l[i] = (uint16_t)indices[i];
        }
    }
    ST_TL(1);
    sync();
    ST_TL(2);
    for (int p = tid; p < n; p += TPB) pos_l[idx_l[p]] = (uint16_t)p;

    // ---- diff: contiguous element range per thread keeps the lists ascending
    uint32_t cnt = 0;  // added in the low half, removed in the high half
    if constexpr (VEC) {
#pragma unroll
        for (int w = 0; w < NW; ++w)
            cnt += (uint32_t)__popcll(w_new[w] & ~w_cur[w]) + ((uint32_t)__popcll(w_cur[w] & ~w_new[w]) << 16);
    } else {
        for (int i = e0; i < e1; ++i) {
            const uint8_t f = flag_l[i];
            cnt += (f == 1) ? 1u : 0u;
            cnt += (f == 2) ? 0x10000u : 0u;
        }
    }
    uint32_t total;
    const uint32_t off = block_excl_scan<TPB / kWave>(cnt, wave_tot, &total, tid, sync);  // contains __syncthreads
    ST_TL(3);
    const int na = (int)(total & 0xffffu), nr = (int)(total >> 16);
    if (na == 0 && nr == 0) {  // unchanged mask: nothing is touched (weight_cache.h:237-240)
        if (tid == 0 && writer) {
            state[ST_STATE_N_CHANGED] = 0;
            state[ST_STATE_N_ADDED] = 0;
            state[ST_STATE_N_REMOVED] = 0;
        }
        pv.next_epoch = ep;
        if (tid == 0) pv.arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
        pv.changed = false;
        pv.n_old = pv.n_new = n; pv.na = pv.nr = 0; pv.n_changed = 0;
        return;
    }
    {
        int oa = (int)(off & 0xffffu), orr = (int)(off >> 16);
        if constexpr (VEC) {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int e = e0 + 8 * w;
                uint64_t a = w_new[w] & ~w_cur[w], r = w_cur[w] & ~w_new[w];   // one 0x01 byte per element, ascending
                while (a) {
                    lists[oa++] = (uint16_t)(e + ((__ffsll((long long)a) - 1) >> 3));
                    a &= a - 1;
                }
                while (r) {
                    lists[I - 1 - (orr++)] = (uint16_t)(e + ((__ffsll((long long)r) - 1) >> 3));
                    r &= r - 1;
                }
            }
        } else {
            for (int i = e0; i < e1; ++i) {
                const uint8_t f = flag_l[i];
                if (f == 1) lists[oa++] = (uint16_t)i;
                if (f == 2) lists[I - 1 - (orr++)] = (uint16_t)i;
            }
        }
    }
    sync();

    const int pairs = na < nr ? na : nr;
    // Without surplus removals (nr <= na) the rewritten positions are known as soon as phases 1 and 2
    // have run: they replace the added indices in `lists` in place and no compaction is needed.
    const bool fast = nr <= na;
    // ---- phase 1: paired replacement
    for (int i = tid; i < pairs; i += TPB) {
        const int e = lists[I - 1 - i];
        const uint16_t p = pos_l[e];
        if (p != kNone) {
            const int a = lists[i];
            idx_l[p] = (uint16_t)a;
            pos_l[a] = p;
            pos_l[e] = kNone;
            if (MARK || !fast) atomicOr(&dirty[p >> 5], 1u << (p & 31));
        }
        if (fast) lists[i] = p;
    }
    // ---- phase 2: append surplus additions
    for (int i = pairs + tid; i < na; i += TPB) {
        const int p = n + (i - pairs);
        if (p < I) {
            const int a = lists[i];
            idx_l[p] = (uint16_t)a;
            pos_l[a] = (uint16_t)p;
        }
        lists[i] = p < I ? (uint16_t)p : kNone;
    }
    sync();

    int n_new;
    uint32_t n_changed;
    if (fast) {
        n_new = n + (na - pairs);
        if (n_new > I) n_new = I;
        n_changed = (uint32_t)na;
        ST_TL(4);
    } else {
        // (the places go over the removed indices, k-th surplus one at lists[I-1-pairs-k]; a surplus index is marked by
        // having no position any more)
        const int S_all = nr - pairs;
        auto place = [&](int k) __attribute__((always_inline)) -> uint16_t & { return lists[I - 1 - pairs - k]; };
        for (int k = tid; k < S_all; k += TPB) {
            const int e = place(k);
            place(k) = pos_l[e];
            pos_l[e] = kNone;
        }
        n_new = surplus_count<TPB>(place, S_all, n, wave_tot, &n_new_s, tid, sync);
        auto stays = [&](int k) __attribute__((always_inline)) { return pos_l[idx_l[n - 1 - k]] != kNone; };
        surplus_ends<TPB>(place, stays, n_new, n, wave_tot, tid, sync);
        for (int j = tid; j < n - n_new; j += TPB) {
            if (!stays(j)) continue;
            const int q = place(j);
            idx_l[q] = idx_l[n - 1 - j];
            atomicOr(&dirty[q >> 5], 1u << (q & 31));
        }
        sync();
        ST_TL(4);

        // ---- compact the dirty positions below n_new into the copy list (in LDS, over the dead lists)
        uint32_t word = 0;
        if (tid < dirty_words) {
            word = dirty[tid];
            const int lo = tid << 5;
            if (lo >= n_new) word = 0;
            else if (lo + 32 > n_new) word &= (1u << (n_new - lo)) - 1u;
        }
        uint32_t coff = block_excl_scan<TPB / kWave>((uint32_t)__popc(word), wave_tot, &n_changed, tid, sync);  // barrier: lists are dead now
        while (word) {
            const int bit = __ffs(word) - 1;
            word &= word - 1;
            lists[coff++] = (uint16_t)((tid << 5) + bit);
        }
        sync();
    }

    ST_TL(5);
    // ---- publish: one block writes the other bookkeeping buffer, the last arrival flips the epoch
    if (writer) {
        int32_t *idx_out = indices2 + (size_t)(ep ^ 1) * I;
        uint8_t *mask_out = cur_mask2 + (size_t)(ep ^ 1) * I;
        for (int p = tid; p < n_new; p += TPB) idx_out[p] = idx_l[p];
        // the reference stores the new mask only when the rebuild did not throw (n_new > 0)
        if constexpr (VEC) {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int e = e0 + 8 * w;
                if (e < e1) store_mask<AL>(mask_out, e, I, n_new > 0 ? w_new[w] : w_cur[w]);
            }
        } else {
            for (int i = tid; i < I; i += TPB) mask_out[i] = n_new > 0 ? (flag_l[i] & 1) : (flag_l[i] >> 1);
        }
        if (tid == 0) {
            state[ST_STATE_N_BUF0 + (ep ^ 1)] = n_new;
            state[ST_STATE_N_ACTIVE] = n_new;
            state[ST_STATE_N_CHANGED] = (int)n_changed;
            state[ST_STATE_N_ADDED] = na;
            state[ST_STATE_N_REMOVED] = nr;
            state[ST_STATE_SERIAL] += 1;
            state[ST_STATE_EPOCH] = ep ^ 1;
            if (n_new > 0) {
                state[ST_STATE_STATUS] = 0;
                state[ST_STATE_VALID] = 1;
            } else {
                state[ST_STATE_STATUS] = ST_ERR_NO_ACTIVE;
            }
        }
    }
    pv.next_epoch = ep ^ 1;
    if (tid == 0) pv.arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
    pv.changed = true;
    pv.n_old = n; pv.n_new = n_new; pv.na = na; pv.nr = nr; pv.n_changed = n_changed;
}


// Last step of a kernel that ran cache_plan: the block that arrived last resets the arrivals and sets the
// epoch.  Looking at the atomic's result only here keeps its round trip off the critical path.
__device__ __forceinline__ void plan_finish(const PlanView &pv, int32_t *__restrict__ state)
{
    if (pv.arriver) {
        uint32_t arrival = pv.arrival;
        asm volatile("" : "+v"(arrival));   // the result is first looked at here, not where it was requested
        if ((arrival & 0xffffu) == gridDim.x - 1)
            atomicExch(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), (uint32_t)pv.next_epoch << 16);
    }
}

// ---------------------------------------------------------------------------
// update kernel
// ---------------------------------------------------------------------------
// What the GPU tells the host on its own (pinned memory, written across the bus): the count, as a guess for later launches,
// from the publishing block of every update; and for a caller that waits the state words, each beside the number of the
// wait so that the host sees without ordered stores when all of them are its own.
struct HostWords {
    int32_t count;
    int32_t pad[15];
    uint64_t state[ST_STATE_WORDS];   // (number of the wait << 32) | value
};

__device__ __forceinline__ void tell_count(HostWords *hw, int n)
{
    __hip_atomic_store(&hw->count, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The state words to the host: a launch of its own behind the update, so that everything before it on the stream has ended
// once the host sees them -- every block's reads of the mask and of the module's weights, and its writes of the rows, not
// just the publishing block's plan.
__global__ __launch_bounds__(kWave) void cache_tell_kernel(const int32_t *__restrict__ state, HostWords *host, uint32_t number)
{
    const int k = threadIdx.x;
    if (k < ST_STATE_WORDS)
        __hip_atomic_store(&host->state[k], ((uint64_t)number << 32) | (uint32_t)state[k], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// The caches of one launch: several layers of equal shape (grid dimension y) or one.
struct UpdateLayer {
    const uint8_t *new_mask;
    uint8_t *cur_mask2;
    int32_t *indices2, *state;
    const unsigned char *pool[3];
    unsigned char *active[3];
    HostWords *host;
};
struct UpdateLayers {
    static constexpr bool kLayers = true;
    UpdateLayer l[kMaxLayers];
};

// A work item: position `pos` is rewritten with pool row `idx` (kNone or a position past the new count: nothing to do).
// This block's share of them, a wave per (item, matrix) with the whole row in flight (8 KB): at usual churn every wave has
// at most one, so the copies cost one round trip.  (A thread group of 512 per row and four rows in flight left a quarter of
// the lanes of a 6 KB row idle and took two dependent rounds from 1500 (item, matrix) pairs on: 11 us for 2600 of them.)
template <int TPB>
__device__ __forceinline__ void copy_items(const unsigned char *const (&pool)[3], unsigned char *const (&active)[3], int nmat,
                                           int row_bytes, int tid, int items, int n_new, const uint16_t *pos,
                                           const uint16_t *idx)
{
    constexpr int W = TPB / kWave;
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int chunks = row_bytes >> 4;
    const unsigned char *const pool0 = pool[0], *const pool1 = pool[1], *const pool2 = pool[2];
    unsigned char *const act0 = active[0], *const act1 = active[1], *const act2 = active[2];
    // the publishing block takes no copies when there are others to do them
    const bool solo = gridDim.x == 1;
    const int slots = (solo ? 1 : (int)gridDim.x - 1) * W;
    const int work = items * nmat;
    // (neighbouring items to different blocks: blocks own waves blk, blk + blocks, ...)
    for (int w = solo ? wave : blockIdx.x == 0 ? work : (int)blockIdx.x - 1 + ((int)gridDim.x - 1) * wave; w < work; w += slots) {
        const int j = w / nmat, m = w - j * nmat;
        const int p = __builtin_amdgcn_readfirstlane((int)pos[j]), e = __builtin_amdgcn_readfirstlane((int)idx[j]);
        if (p >= n_new) continue;
        const unsigned char *from = (m == 0 ? pool0 : m == 1 ? pool1 : pool2) + (size_t)e * row_bytes;
        unsigned char *to = (m == 0 ? act0 : m == 1 ? act1 : act2) + (size_t)p * row_bytes;
        constexpr int U = 8;
        for (int c0 = lane; c0 < chunks; c0 += U * kWave) {
            uint4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * kWave;
                v[u] = ld16_stream(from + ((size_t)(c < chunks ? c : chunks - 1) << 4));
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * kWave;
                if (c < chunks) st16(to + ((size_t)c << 4), v[u]);
            }
        }
    }
}

// LDS of the kernel below: two bytes per index for each of the items' indices, their positions and the surplus removals'
// places, and three per eight indices for the ranks of the removed ones.
constexpr size_t update_lds_bytes(int I)
{
    const size_t groups = (size_t)((I + 7) >> 3);
    return (size_t)((I + 7) & ~7) * 6 + ((groups * 2 + 15) & ~(size_t)15) + ((groups + 15) & ~(size_t)15);
}

// The update by POSITION.  Which index a position holds afterwards follows from the old list and the two masks without an
// index -> position map: a removed index has a rank among the removed ones (a prefix count per eight indices, and the
// bits below it), the i-th of them hands its position to the i-th added index (phase 1), the surplus additions follow at
// the end (phase 2), and a position of rank >= n_added is where a surplus removal starts (phase 3, surplus_ends).  So
// the plan is one scan, one pass over the list -- every thread keeps the positions it loaded in registers -- and two
// barriers when removals do not outnumber additions.  Every block plans for itself (as a launch of its own the plan would
// cost a kernel boundary) and copies its share of the items.
// Masks in 8-byte words, lists in 16-byte vectors, at any alignment (I >= 8); I <= 8 NW TPB.
template <int TPB, int NW, typename Tab, bool AL>
__global__ __launch_bounds__(TPB) void cache_update_kernel(const uint8_t *__restrict__ new_mask,
                                                           uint8_t *__restrict__ cur_mask2,
                                                           int32_t *__restrict__ indices2, int32_t *__restrict__ state,
                                                           int I, int idx_cap, CopyPlan cp, HostWords *host, Tab tab)
{
    if constexpr (Tab::kLayers) {
        const UpdateLayer &ly = tab.l[blockIdx.y];
        host = ly.host;
        new_mask = ly.new_mask;
        cur_mask2 = ly.cur_mask2;
        indices2 = ly.indices2;
        state = ly.state;
    }
    constexpr int NV = 2 * NW;                 // vectors of four positions per thread
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t wave_tot[TPB / kWave];
    __shared__ int shared_n;
    __shared__ uint32_t shared_changed;
    const int Ip = (I + 7) & ~7;
    uint16_t *const item_idx = reinterpret_cast<uint16_t *>(smem);   // added indices ascending; behind them the tail's entries
    uint16_t *const item_pos = item_idx + Ip;
    uint16_t *const place = item_pos + Ip;                           // k-th surplus index: where it starts; then the end of its tail slot's path
    uint16_t *const rem_before = place + Ip;                         // per eight indices: removed ones below
    uint8_t *const rem_bits = reinterpret_cast<uint8_t *>(rem_before) + ((((I + 7) >> 3) * 2 + 15) & ~15);
    const int tid = threadIdx.x;
    const bool writer = blockIdx.x == 0;
    auto sync = [&]() __attribute__((always_inline)) { lds_barrier(); };

    ST_TL(0);
    // ---- everything the plan reads, in one round trip: both halves of the double buffers are requested before the epoch
    // word has arrived.  (The epoch cannot flip before every block has arrived, and a block arrives -- one atomic, at the
    // end of its plan -- after all its threads have consumed this load.)
    const uint32_t tword = __hip_atomic_load(reinterpret_cast<const uint32_t *>(&state[ST_STATE_TICKET]), __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    const int words = (I + 8 * TPB - 1) / (8 * TPB);   // per thread: a contiguous range, so that lists come out ascending
    uint64_t v_new[NW], v_cur0[NW], v_cur1[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int e = !AL || (w < words && 8 * (tid * words + w) < I) ? 8 * (tid * words + w) : 0;
        v_new[w] = load_mask<AL>(new_mask, e, I);
        v_cur0[w] = load_mask<AL>(cur_mask2, e, I);
        v_cur1[w] = load_mask<AL>(cur_mask2 + I, e, I);
    }
    int4 v_i0[NV], v_i1[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const int p = 4 * (tid + TPB * q), pc = p < idx_cap ? p : 0;   // (idx_cap: a multiple of 8, or I)
        v_i0[q] = load_list<AL>(indices2, pc, I);
        v_i1[q] = load_list<AL>(indices2 + I, pc, I);
    }
    const int n_buf0 = state[ST_STATE_N_BUF0], n_buf1 = state[ST_STATE_N_BUF1];
    const int serial_old = state[ST_STATE_SERIAL], valid_old = state[ST_STATE_VALID];
    if (tid == 0) shared_changed = 0;
    const int ep = (int)((tword >> 16) & 1u);
    const int n = ep ? n_buf1 : n_buf0;

    // ---- diff: removed bits and their prefix counts per eight indices, added indices ascending
    uint64_t w_new[NW], w_cur[NW];
    uint32_t cnt = 0;   // added in the low half, removed in the high half
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int e = 8 * (tid * words + w);
        const bool in = w < words && e < I;
        w_new[w] = in ? nonzero_bytes(mask_tail<AL>(v_new[w], e, I)) : 0ull;
        w_cur[w] = in ? nonzero_bytes(mask_tail<AL>(ep ? v_cur1[w] : v_cur0[w], e, I)) : 0ull;
        cnt += (uint32_t)__popcll(w_new[w] & ~w_cur[w]) + ((uint32_t)__popcll(w_cur[w] & ~w_new[w]) << 16);
    }
    ST_TL(1);
    const int lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t incl = wave_incl_scan_dpp(cnt, lane);
    if (lane == kWave - 1) wave_tot[wave] = incl;
    sync();
    uint32_t prefix = incl - cnt, total = 0;
#pragma unroll
    for (int w = 0; w < TPB / kWave; ++w) {
        const uint32_t t = wave_tot[w];
        if (w < wave) prefix += t;
        total += t;
    }
    ST_TL(2);
    const int na = (int)(total & 0xffffu), nr = (int)(total >> 16);
    uint32_t arrival = 0;
    int next_epoch = ep ^ 1;
    if (na == 0 && nr == 0) {   // unchanged mask: nothing is touched (weight_cache.h:237-240)
        next_epoch = ep;
        if (tid == 0 && writer) {
            state[ST_STATE_N_CHANGED] = 0;
            state[ST_STATE_N_ADDED] = 0;
            state[ST_STATE_N_REMOVED] = 0;
            tell_count(host, n);
        }
        if (tid == 0) arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
    } else {
        const int pairs = na < nr ? na : nr, S_all = nr - pairs;
        {
            int oa = (int)(prefix & 0xffffu), orr = (int)(prefix >> 16);
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int g = tid * words + w;
                if (w < words && 8 * g < I) {
                    uint64_t a = w_new[w] & ~w_cur[w];   // one 0x01 byte per element, ascending
                    const uint64_t r = w_cur[w] & ~w_new[w];
                    rem_before[g] = (uint16_t)orr;
                    rem_bits[g] = (uint8_t)pack_bits8(r);
                    orr += __popcll(r);
                    while (a) {
                        item_idx[oa++] = (uint16_t)(8 * g + ((__ffsll((long long)a) - 1) >> 3));
                        a &= a - 1;
                    }
                }
            }
        }
        // (removed indices that are not in the list -- only after an update that failed -- leave these untouched)
        for (int i = tid; i < pairs; i += TPB) item_pos[i] = kNone;
        for (int i = tid; i < S_all; i += TPB) place[i] = kNone;
        for (int i = pairs + tid; i < na; i += TPB) {   // phase 2
            const int p = n + (i - pairs);
            item_pos[i] = p < I ? (uint16_t)p : kNone;
        }
        sync();
        ST_TL(3);
        // ---- the list: what every position holds after the paired replacements, in registers (kOut: a surplus index)
        constexpr int kOut = 0xffff;
        int32_t *const idx_out = indices2 + (size_t)(ep ^ 1) * I;
        int held[NV][4];
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int p0 = 4 * (tid + TPB * q);
            int4 c = ep ? v_i1[q] : v_i0[q];
            if (n > idx_cap && p0 >= idx_cap && p0 < n)   // more positions in use than the caller expected (one more round trip)
                c = load_list<AL>(indices2 + (size_t)ep * I, p0, I);
            c = list_tail<AL>(c, p0, I);
            const int e4[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int p = p0 + k, e = p < n ? e4[k] & 0xffff : 0;
                const uint32_t bits = rem_bits[e >> 3];
                int h = e;
                if (p < n && ((bits >> (e & 7)) & 1u)) {
                    const int rank = (int)rem_before[e >> 3] + __popc(bits & ((1u << (e & 7)) - 1u));
                    if (rank < na) {
                        h = item_idx[rank];
                        item_pos[rank] = (uint16_t)p;
                    } else {
                        h = kOut;
                        place[rank - na] = (uint16_t)p;
                    }
                }
                held[q][k] = h;
            }
        }
        int n_new = n + (na - pairs) < I ? n + (na - pairs) : I, items = na;
        if (S_all > 0) {
            sync();
            auto place_of = [&](int k) __attribute__((always_inline)) -> uint16_t & { return place[k]; };
            n_new = surplus_count<TPB>(place_of, S_all, n, wave_tot, &shared_n, tid, sync);
            // the entries of the tail, last first, behind the added indices: items like the others once their paths' ends are known
#pragma unroll
            for (int q = 0; q < NV; ++q)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int p = 4 * (tid + TPB * q) + k;
                    if (p >= n_new && p < n) item_idx[na + (n - 1 - p)] = (uint16_t)held[q][k];
                }
            sync();
            auto stays = [&](int j) __attribute__((always_inline)) { return item_idx[na + j] != kOut; };
            surplus_ends<TPB>(place_of, stays, n_new, n, wave_tot, tid, sync);
            const int S_ = n - n_new;
            items = na + S_;
            for (int j = tid; j < S_; j += TPB) {
                int to = kNone;
                if (stays(j)) {
                    to = place[j];
                    if (writer) idx_out[to] = item_idx[na + j];
                }
                item_pos[na + j] = (uint16_t)to;
            }
        }
        sync();
        ST_TL(4);
        // ---- publish: one block writes the other bookkeeping buffer, the last arrival flips the epoch
        if (writer) {
            uint8_t *mask_out = cur_mask2 + (size_t)(ep ^ 1) * I;
            const int kept = n < n_new ? n : n_new;
#pragma unroll
            for (int q = 0; q < NV; ++q)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int p = 4 * (tid + TPB * q) + k;
                    if (p < kept && held[q][k] != kOut) idx_out[p] = held[q][k];
                }
            for (int i = pairs + tid; i < na; i += TPB)
                if (item_pos[i] < n_new) idx_out[item_pos[i]] = item_idx[i];
            // the reference stores the new mask only when the rebuild did not throw (n_new > 0)
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int e = 8 * (tid * words + w);
                if (w < words && e < I) store_mask<AL>(mask_out, e, I, n_new > 0 ? w_new[w] : w_cur[w]);
            }
            uint32_t mine = 0;
            if (S_all > 0)
                for (int i = tid; i < items; i += TPB) mine += item_pos[i] < n_new ? 1u : 0u;
            if (mine) atomicAdd(&shared_changed, mine);
            sync();
            if (tid == 0) {
                state[ST_STATE_N_BUF0 + (ep ^ 1)] = n_new;
                state[ST_STATE_N_ACTIVE] = n_new;
                state[ST_STATE_N_CHANGED] = S_all > 0 ? (int)shared_changed : na;
                state[ST_STATE_N_ADDED] = na;
                state[ST_STATE_N_REMOVED] = nr;
                state[ST_STATE_SERIAL] = serial_old + 1;
                state[ST_STATE_EPOCH] = ep ^ 1;
                state[ST_STATE_STATUS] = n_new > 0 ? 0 : ST_ERR_NO_ACTIVE;
                state[ST_STATE_VALID] = n_new > 0 ? 1 : valid_old;
                tell_count(host, n_new);
            }
        }
        if (tid == 0) arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
        ST_TL(5);
        if constexpr (Tab::kLayers) {
            const UpdateLayer &ly = tab.l[blockIdx.y];
            copy_items<TPB>(ly.pool, ly.active, cp.nmat, cp.row_bytes, tid, items, n_new, item_pos, item_idx);
        } else {
            copy_items<TPB>(cp.pool, cp.active, cp.nmat, cp.row_bytes, tid, items, n_new, item_pos, item_idx);
        }
    }
    // the block that arrived last resets the arrivals and sets the epoch (the atomic's result is first looked at here)
    if (tid == 0) {
        asm volatile("" : "+v"(arrival));
        if ((arrival & 0xffffu) == gridDim.x - 1)
            atomicExch(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), (uint32_t)next_epoch << 16);
    }
    ST_TL(6);
}

// The same for masks of less than one 8-byte word: cache_plan above, then the copies.
template <int TPB>
__global__ __launch_bounds__(TPB) void cache_update_bytes_kernel(const uint8_t *__restrict__ new_mask,
                                                                 uint8_t *__restrict__ cur_mask2,
                                                                 int32_t *__restrict__ indices2,
                                                                 int32_t *__restrict__ state, int I, CopyPlan cp,
                                                                 HostWords *host)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ PlanShared ps;
    const int tid = threadIdx.x;
    PlanView pv;
    cache_plan<false, TPB, 1, false, true>(pv, smem, &ps, new_mask, cur_mask2, indices2, state, I, tid);
    if (tid == 0 && pv.writer) tell_count(host, pv.n_new);
    if (pv.changed) {
        // (the index of a rewritten position, beside the position: the map of the plan is not needed any more)
        for (int i = tid; i < (int)pv.n_changed; i += TPB) pv.pos_l[i] = pv.lists[i] != kNone ? pv.idx_l[pv.lists[i]] : 0;
        lds_barrier();
        copy_items<TPB>(cp.pool, cp.active, cp.nmat, cp.row_bytes, tid, (int)pv.n_changed, pv.n_new, pv.lists, pv.pos_l);
    }
    plan_finish(pv, state);
}

// ---------------------------------------------------------------------------
// update + sparse MLP in ONE kernel, with the plan worked out per POSITION
// instead of per index.
//
// A block only has to know, for each of the <= ceil(I / G) positions it owns,
// which row to read: position p held index e before the update; if e left the
// mask it is the i-th removed index (i = its rank among the removed, ascending)
// and the position receives the i-th added index (weight_cache.h:248-277);
// positions n_old .. n_new-1 receive the surplus additions in ascending order
// (:280-307).  Ranks come from bitmaps of the two masks and per-word prefix
// counts (one wave, no block-wide scans), the i-th added index from a binary
// search over those counts -- no index -> position map, no lists, no atomics,
// three LDS-only barriers, and straight-line code, so the rows a block requests
// on the caller's guess right after its (few) bookkeeping loads stay in flight
// through all of it.  Every block publishes its own positions of the new
// ordered list and a slice of the remembered mask into the other bookkeeping
// buffer; block 0 writes the state words; the last block to arrive flips the
// epoch (as in cache_plan).
// When removals outnumber additions, the surplus ones are taken out one by
// one in the reference (:310-353); their outcome is worked out in closed form
// (see the kernel), or, for very many of them, by cache_plan above for that
// launch only.
// ---------------------------------------------------------------------------
constexpr int kSparseMaxQ = 64;       // positions a block can own
constexpr int kSparseMaxW32 = 512;    // mask words: I <= 16384
constexpr int kSparseWords = 2;       // 8-byte mask words per thread, at most
constexpr int kSparseScan = 4;         // positions per thread whose old index is fetched up front for that replay
constexpr int kSrcPool = 0x40000000;  // src[]: bit 30 = read the pool row (low bits) and write it back; else active row

struct SparseShared {
    uint32_t newbits[kSparseMaxW32], oldbits[kSparseMaxW32];
    uint16_t pr[kSparseMaxW32];   // removed indices below each word
    int na, nr, n;
    int src[kSparseMaxQ];
    int found, paired_tail, replay_ok, fast_ok, nchg;   // surplus removals (removed > added)
};

template <typename T, int RB, int TPB, int NB, int NW, int SPECN, bool AL>
__global__ __launch_bounds__(TPB) void cache_sparse_decode_kernel(
    const uint8_t *__restrict__ new_mask, uint8_t *__restrict__ cur_mask2, int32_t *__restrict__ indices2,
    int32_t *__restrict__ state, int I, int launch_word, const T *__restrict__ x, int H, int n_hint,
    T *__restrict__ combined, long ldc, float *__restrict__ partials, int act, int plan_bytes, HostWords *host, FusedRows fr)
{
    constexpr int VEC = Elem<T>::kVec;
    // Slots of the first batch that are requested ahead of the plan, on the caller's guess of the count and from the
    // active buffers.  A slot whose row turns out to have changed is requested again into the same registers, which
    // has to wait until its first request has arrived; requests return in order, so for the last slots that wait
    // would be the whole stream plus one more round trip, and every row requested in vain is traffic.  The later
    // slots are therefore requested after the plan (first, so that they queue right behind the rows already
    // requested).  Half the batch ahead of the plan measured best (against a third, two thirds and all of it).
    constexpr int SPEC = SPECN;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[TPB / kWave][RB][NB][2];  // per-wave partial (g,u)
    __shared__ float hs[TPB / kWave][RB][NB];      // h of the rows being computed
    __shared__ SparseShared sh;
    __shared__ PlanShared plan_shared;

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    // (what the first loads need comes first in the argument list, the number of blocks included: the first 14 dwords
    // of the arguments are in scalar registers when the wave starts, anything else -- the launch dimensions too --
    // arrives by a load that the first instructions would wait for.  Four small numbers share one of those dwords.)
    const int blk = blockIdx.x;
    const int G = launch_word & 0xffff, gs_log2 = (launch_word >> 16) & 15, B = (launch_word >> 24) & 15;
    const int chunks = H / VEC;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    const int GS = 1 << gs_log2, ngrp = TPB >> gs_log2, wpg = GS >> 6;
    const int grp = tid >> gs_log2, cc = tid & (GS - 1);
    const bool valid = cc < chunks;
    const size_t coff = valid ? (size_t)cc * 16 : 0;
    const bool wave_live = __builtin_amdgcn_readfirstlane(cc & ~(kWave - 1)) < chunks;
    const bool has_gate = ((launch_word >> 20) & 1) != 0;
    const int row_bytes = H * (int)sizeof(T);
    const unsigned char *const pool_g = fr.pool_g, *const pool_u = fr.pool_u, *const pool_d = fr.pool_d;
    unsigned char *const act_g = fr.act_g, *const act_u = fr.act_u, *const act_d = fr.act_d;
    const int Q = (I + G - 1) / G;        // positions of this block: blk + G * q, q < Q (host: Q <= kSparseMaxQ)
    const int W32 = (I + 31) >> 5;

    ST_TL(0);
    // ---- bookkeeping loads: one round trip, all unconditional (clamped addresses).  The state words are read
    // through a lane offset the compiler cannot see through (always zero): as loads from one address for the whole
    // wave they would be moved to scalar registers at once, which means waiting for them before anything else
    // is requested.
    int lane_zero = 0;
    asm volatile("" : "+v"(lane_zero));
    const int32_t *state_v = state + lane_zero;
    const uint32_t tword = __hip_atomic_load(reinterpret_cast<const uint32_t *>(&state_v[ST_STATE_TICKET]),
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int n_buf0 = state_v[ST_STATE_N_BUF0], n_buf1 = state_v[ST_STATE_N_BUF1];
    const int serial_old = state_v[ST_STATE_SERIAL];
    constexpr int nw_rt = NW;   // 8-byte mask words per thread (host: I <= 8 * TPB * NW)
    uint64_t v_new[NW], v_c0[NW], v_c1[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int e = !AL || (tid * nw_rt + w) * 8 + 8 <= I ? (tid * nw_rt + w) * 8 : I - 8;
        v_new[w] = load_mask<AL>(new_mask, e, I);
        v_c0[w] = load_mask<AL>(cur_mask2, e, I);
        v_c1[w] = load_mask<AL>(cur_mask2 + I, e, I);
    }
    // The plan is worked out by ONE wave, the last of the block (with 6 KB rows a wave that owns no columns), while
    // the others already request rows; its lanes own the block's positions.
    constexpr int PW = TPB / kWave - 1;
    const bool plan_wave = wave == PW;
    static_assert(kSparseMaxQ == kWave, "one lane of the planning wave per position of the block");
    const int my_p = blk + G * lane;
    const int my_pc = my_p < I ? my_p : I - 1;
    const int i_old0 = indices2[my_pc], i_old1 = indices2[(size_t)I + my_pc];
    // The ordered list itself, four positions per thread, for the case that removals outnumber additions (the
    // surplus ones can sit at any position); only as far as the caller's guess of the count plus a quarter.
    const int n_spec = n_hint < I ? n_hint : I;
    int scan_cap = (n_spec + (n_spec >> 2) + 64) & ~3;
    if (scan_cap > kSparseScan * TPB) scan_cap = kSparseScan * TPB;
    if (scan_cap > I) scan_cap = I & ~3;
    const int scan_p = kSparseScan * tid;
    const bool scan_in = scan_p + kSparseScan <= scan_cap;
    const int scan_pc = scan_in ? scan_p : 0;
    static_assert(kSparseScan == 4, "one 16-byte load per bookkeeping buffer");
    const int4 sc0 = load_list<AL>(indices2, scan_pc, I);
    const int4 sc1 = load_list<AL>(indices2 + I, scan_pc, I);
    uint4 xr[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
        xr[b] = ld16(reinterpret_cast<const unsigned char *>(x) + (size_t)(b < B ? b : 0) * row_bytes + coff);

    // ---- the first batch of rows, on the caller's guess of the count, from the active buffers
    auto row_of = [&](int bat, int k) { return blk + G * (grp + ngrp * (bat * RB + k)); };
    uint4 wg[RB], wu[RB], wd[RB];
    // (every wave issues the same number of loads whatever its role: a wave without columns, and the gate loads
    // of an ungated cache, read one line of x instead -- with branches around the loads the compiler could no
    // longer tell how many requests are younger than the bookkeeping loads and would wait for all of them)
    // Addresses are a uniform base (scalar registers) plus a 32-bit lane offset, one offset per row for its three
    // matrices: with a 64-bit address per load the 18 requests alone would need 36 registers more.
    const uint32_t coff32 = (uint32_t)coff;
    const unsigned char *const dummy = reinterpret_cast<const unsigned char *>(x);
    const unsigned char *const sp_u = wave_live ? act_u : dummy, *const sp_d = wave_live ? act_d : dummy,
                        *const sp_g = wave_live && has_gate ? act_g : dummy;
    auto speculate = [&](auto lo_c, auto hi_c) __attribute__((always_inline)) {
        constexpr int LO = decltype(lo_c)::value, HI = decltype(hi_c)::value;
#pragma unroll
        for (int k = LO; k < HI; ++k) {
            const int p = row_of(0, k);
            // (a slot past the expected count reads one 16-byte piece for the whole wave: a single request instead of
            // a row's worth of traffic that nobody needs)
            const uint32_t off = wave_live && p < n_spec ? (uint32_t)p * (uint32_t)row_bytes + coff32 : 0u;
            wu[k] = ld16_stream(sp_u + off);
            wd[k] = ld16_stream(sp_d + off);
            wg[k] = ld16_stream(sp_g + (has_gate ? off : 0u));   // (the stand-in line of x has no rows to index)
        }
    };
    // Half of the rows that are requested ahead of the plan go out right behind the bookkeeping loads -- few enough
    // that the memory system is not yet saturated when those loads are served -- the other half once they have
    // arrived.  The barrier only orders the issue: every wave's bookkeeping loads are queued before any wave's rows.
    constexpr int SPEC_A = SPEC / 2;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    speculate(std::integral_constant<int, 0>{}, std::integral_constant<int, SPEC_A>{});
    __builtin_amdgcn_sched_barrier(0);
    ST_TL(1);

    // ---- masks -> bitmaps in LDS
    const int ep = (int)((tword >> 16) & 1u);
    const int n_old = ep ? n_buf1 : n_buf0;
    uint64_t w_new[NW], w_cur[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int bi = tid * nw_rt + w;            // byte of the bitmaps = elements [8 bi, 8 bi + 8)
        const bool in = w < nw_rt && bi * 8 < I;
        w_new[w] = in ? nonzero_bytes(mask_tail<AL>(v_new[w], bi * 8, I)) : 0ull;
        w_cur[w] = in ? nonzero_bytes(mask_tail<AL>(ep ? v_c1[w] : v_c0[w], bi * 8, I)) : 0ull;
        if (w < nw_rt && bi < W32 * 4) {
            reinterpret_cast<uint8_t *>(sh.newbits)[bi] = (uint8_t)pack_bits8(w_new[w]);
            reinterpret_cast<uint8_t *>(sh.oldbits)[bi] = (uint8_t)pack_bits8(w_cur[w]);
        }
    }
    // (behind the list of added indices, which holds I entries at most; the region of the per-index plan, six
    // bytes per index, is unused on this path)
    uint16_t *const scan_idx = reinterpret_cast<uint16_t *>(smem) + ((I + 7) & ~7);
    if (scan_in) {
        const int4 sc = ep ? sc1 : sc0;
        *reinterpret_cast<uint2 *>(scan_idx + scan_p) =
            make_uint2((uint32_t)(sc.x & 0xffff) | ((uint32_t)sc.y << 16), (uint32_t)(sc.z & 0xffff) | ((uint32_t)sc.w << 16));
    }
    lds_barrier();
    // ---- Rows are requested from here on, i.e. once every wave's bookkeeping loads have ARRIVED: loads issued into
    // a memory system that is already saturated with row requests take several times longer to come back (measured:
    // 5.7 us instead of under 2 when the rows were requested right behind them), and the plan hangs on them.  From
    // here on the plan needs LDS only.  It is one wave's work, so that it does not wait for the other waves either:
    // a wave's requests are accepted only as fast as the memory system takes them (the last wave of sixteen gets its
    // first batch out 3 us after the first), and a block barrier inside the plan would wait for all of that.
    ST_TL(2);
    int n = n_old;      // count after the update
    uint32_t arrival = 0;
    __builtin_amdgcn_sched_barrier(0);
    if (plan_wave) {
        // ---- per-word prefix counts of added / removed indices, eight words per lane at most
        const int wpl = (W32 + kWave - 1) >> 6;
        // (words per lane: at most 4 per 8-byte mask word a thread reads -- the host launches NW = 1 up to I = 8192 --
        // so that the unrolled loops below are no longer than this launch needs: the code of this branch is run by one
        // wave per block, once, and what it costs is mostly fetching it)
        constexpr int kWpl = 4 * NW;
        static_assert(kWpl * kWave * 32 >= 8 * TPB * NW, "the planning wave covers every mask word of the launch");
        uint32_t la[kWpl], lr[kWpl], aw[kWpl];
        uint32_t ca = 0, cr = 0;
        // (all reads of the bitmaps are issued together, from clamped addresses; the words stay in registers for the
        // second pass)
        uint32_t nwd[kWpl], owd[kWpl];
#pragma unroll
        for (int j = 0; j < kWpl; ++j) {
            const int t = lane * wpl + j;
            const int tc = t < W32 ? t : W32 - 1;
            nwd[j] = sh.newbits[tc];
            owd[j] = sh.oldbits[tc];
        }
#pragma unroll
        for (int j = 0; j < kWpl; ++j) {
            const int t = lane * wpl + j;
            const bool in = j < wpl && t < W32;
            const uint32_t nw = in ? nwd[j] : 0u, ow = in ? owd[j] : 0u;
            la[j] = ca; lr[j] = cr;
            aw[j] = nw & ~ow;
            ca += (uint32_t)__popc(aw[j]);
            cr += (uint32_t)__popc(ow & ~nw);
        }
        const uint32_t packed = ca | (cr << 16);
        const uint32_t incl = wave_incl_scan_dpp(packed, lane);
        const uint32_t excl = incl - packed;
        // removed: per-word prefix counts (a position looks its old index's rank up); added: the ascending list itself
        uint16_t *added_list = reinterpret_cast<uint16_t *>(smem);   // (the region of the per-index plan, unused on this path)
#pragma unroll
        for (int j = 0; j < kWpl; ++j) {
            const int t = lane * wpl + j;
            if (j < wpl && t < W32) {
                sh.pr[t] = (uint16_t)((excl >> 16) + lr[j]);
                // (a word rarely holds more than two added indices: the first two go out without a loop)
                uint32_t a = aw[j];
                int o = (int)((excl & 0xffffu) + la[j]);
                const uint32_t a2 = a & (a - 1u);
                if (a) added_list[o] = (uint16_t)(t * 32 + __ffs((int)a) - 1);
                if (a2) added_list[o + 1] = (uint16_t)(t * 32 + __ffs((int)a2) - 1);
                a = a2 & (a2 - 1u);
                o += 2;
                while (a) {
                    added_list[o++] = (uint16_t)(t * 32 + __ffs((int)a) - 1);
                    a &= a - 1u;
                }
            }
        }
        const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const int na_w = (int)(tot & 0xffffu), nr_w = (int)(tot >> 16);
        // (LDS operations of one wave execute in order: the lanes below read what other lanes of this wave wrote above)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        int s = -1;
        if (nr_w <= na_w) {
            // ---- every removed index is paired with an added one: the positions' sources follow per position
            int nn = n_old + (na_w - nr_w);
            if (nn > I) nn = I;
            if (lane < Q && my_p < nn) {
                int newidx;
                if (my_p < n_old) {
                    const int e = ep ? i_old1 : i_old0;
                    const int word = (e >> 5) & (kSparseMaxW32 - 1), bit = e & 31;
                    const uint32_t remw = sh.oldbits[word] & ~sh.newbits[word];
                    if ((remw >> bit) & 1u) {
                        const int rank = (int)sh.pr[word] + __popc(remw & ((1u << bit) - 1u));
                        newidx = (int)added_list[rank];
                        s = newidx | kSrcPool;
                    } else {
                        newidx = e;
                        s = my_p;
                    }
                } else {
                    newidx = (int)added_list[nr_w + (my_p - n_old)];
                    s = newidx | kSrcPool;
                }
                if ((na_w | nr_w) != 0) indices2[(size_t)(ep ^ 1) * I + my_p] = newidx;
            }
            if (lane == 0) sh.n = nn;
        } else {
            // ---- Removals outnumber additions: the surplus ones are taken out one by one, in ascending index order,
            // each by moving the last entry of the list into its place (weight_cache.h:310-353).  With S of them the list
            // ends as its first n_old - S positions ("base"); step k moves the entry that sits in tail slot S-1-k at
            // that time to where the k-th surplus index sits at that time.  Only the tail (S entries of the list, fetched
            // up front) has to be looked at: a surplus index that starts below the tail stays where it is until its own
            // step, so the lane that owns its position asks what step k moves ("land[k]"), and if that is another
            // surplus index (one that started in the tail and is taken out later), what that one's step moves, and
            // so on.  Inside the tail the moves depend on each other through the surplus indices that START there
            // (few: about S^2 / n_old): their slot at their own step is resolved first, one lane each, in rounds (a
            // lane whose chase runs into one that is not resolved yet tries again; the smallest always gets through);
            // then every entry of the tail follows the moves until a step takes it below the tail.  All of it is this
            // wave's work: the others keep streaming.  Used when S <= min(256, I/4), at most 64 surplus indices start
            // in the tail and the list was fetched far enough up front; else the whole block works it out behind the
            // barrier (below), or the per-index plan does.
            const int S = nr_w - na_w, base = n_old - S;   // uniform
            const int smax_w = (I >> 2) < TPB ? (I >> 2) : TPB;
            const int sm8 = (smax_w + 7) & ~7;
            constexpr int kMark = 0x8000, kNone = 0xffff, kOut = 0xfffe, kPop = 0xfffd, kUnres = 0xfffc;
            // (LDS behind the list of added indices: the fetched list, then five arrays of smax entries: 6.5 bytes per index at most)
            uint16_t *const loc = scan_idx + ((scan_cap + 7) & ~7);   // k -> tail slot the k-th surplus index starts in
            uint16_t *const tailv = loc + sm8;                        // tail slot -> entry after the paired replacements, or kMark | k
            uint16_t *const jres = tailv + sm8;                       // k (starting in the tail) -> its slot at step k
            uint16_t *const land = jres + sm8;                        // k -> what step k moves below the tail
            uint16_t *const jlist = land + sm8;                       // the surplus indices that start in the tail
            // (S <= 256: one wave walks the tail 64 slots at a time, and beyond four passes the whole block is faster)
            bool ok = S <= smax_w && S <= 4 * kWave && base >= 0 && n_old <= scan_cap && I >= 256;
            if (ok) {
#pragma unroll 1
                for (int c = lane; c < S; c += kWave) loc[c] = (uint16_t)kNone;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                int in_tail = 0, paired_tail = 0;
#pragma unroll 1
                for (int c = 0; c < S; c += kWave) {
                    const int j = c + lane;
                    const bool in = j < S;
                    const int e = (int)scan_idx[base + (in ? j : 0)];
                    const int word = (e >> 5) & (kSparseMaxW32 - 1), bit = e & 31;
                    const uint32_t remw = sh.oldbits[word] & ~sh.newbits[word];
                    const bool rem = in && ((remw >> bit) & 1u);
                    const int rank = (int)sh.pr[word] + __popc(remw & ((1u << bit) - 1u));
                    const bool paired = rem && rank < na_w, extra = rem && rank >= na_w;
                    const int k = extra ? rank - na_w : 0;
                    int v = e;
                    if (paired) v = (int)added_list[rank];
                    if (extra) v = kMark | k;
                    if (in) tailv[j] = (uint16_t)v;
                    const uint64_t mx = __builtin_amdgcn_ballot_w64(extra);
                    if (extra) {
                        const int jj = in_tail + __popcll(mx & ((1ull << lane) - 1ull));
                        loc[k] = (uint16_t)j;
                        jres[k] = (uint16_t)kUnres;
                        if (jj < kWave) jlist[jj] = (uint16_t)k;
                    }
                    in_tail += __popcll(mx);
                    paired_tail += __popcll(__builtin_amdgcn_ballot_w64(paired));
                }
                ok = in_tail <= kWave;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                if (ok) {
                    // ---- the surplus indices that start in the tail: where each sits at its own step
                    const int kk = lane < in_tail ? (int)jlist[lane] : -1;
                    bool open = kk >= 0;
#pragma unroll 1
                    for (int round = 0; round <= kWave && __builtin_amdgcn_ballot_w64(open) != 0; ++round) {
                        bool done = false;
                        int res = 0;
                        if (open) {
                            int pos = loc[kk];
#pragma unroll 1
                            for (int it = 0; it <= S; ++it) {
                                const int i = S - 1 - pos;   // the step that takes the entry of that slot
                                if (i > kk) { res = pos; done = true; break; }    // still there at its own step
                                if (i == kk) { res = kPop; done = true; break; }  // the last entry at its own step: nothing moves
                                const int li = loc[i], ji = jres[i];
                                if (li == kNone || ji == kOut) {   // step i moves it below the tail
                                    land[i] = (uint16_t)(kMark | kk);
                                    res = kOut; done = true; break;
                                }
                                if (ji == kUnres) break;   // next round
                                pos = ji;                  // step i moved it to that slot
                            }
                        }
                        if (open && done) jres[kk] = (uint16_t)res;
                        open = open && !done;
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                    }
                    // ---- every other entry of the tail follows the moves until one takes it below the tail
#pragma unroll 1
                    for (int c = lane; c < S; c += kWave) {
                        const int v = tailv[c];
                        if (v & kMark) continue;
                        int k = S - 1 - c;
#pragma unroll 1
                        for (int it = 0; it <= S; ++it) {
                            const int lk = loc[k], jk = jres[k];
                            if (lk == kNone || jk == kOut) { land[k] = (uint16_t)v; break; }
                            k = S - 1 - (jk < S ? jk : 0);
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                    if (lane < Q && my_p < base) {
                        const int e = ep ? i_old1 : i_old0;
                        const int word = (e >> 5) & (kSparseMaxW32 - 1), bit = e & 31;
                        const uint32_t remw = sh.oldbits[word] & ~sh.newbits[word];
                        int newidx = e;
                        if ((remw >> bit) & 1u) {
                            const int rank = (int)sh.pr[word] + __popc(remw & ((1u << bit) - 1u));
                            if (rank < na_w) {
                                newidx = (int)added_list[rank];
                            } else {
                                int v = land[(rank - na_w) < S ? rank - na_w : 0];
#pragma unroll 1
                                for (int it = 0; it < S && (v & kMark); ++it) v = land[(v & (kMark - 1)) < S ? (v & (kMark - 1)) : 0];
                                newidx = v < I ? v : e;   // (consistent bookkeeping always ends at an entry of the list)
                            }
                        }
                        s = newidx != e ? (newidx | kSrcPool) : my_p;
                        indices2[(size_t)(ep ^ 1) * I + my_p] = newidx;
                    }
                    if (lane == 0) {
                        sh.n = base;
                        // rewritten positions: the pairs' below the tail, and the places of the surplus indices below it
                        sh.nchg = na_w - paired_tail + (S - in_tail);
                    }
                }
            }
            if (lane == 0) sh.fast_ok = ok ? 1 : 0;
        }
        sh.src[lane] = s;
        if (lane == 0) { sh.na = na_w; sh.nr = nr_w; sh.found = 0; sh.paired_tail = 0; }
    }
    speculate(std::integral_constant<int, SPEC_A>{}, std::integral_constant<int, SPEC>{});
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    ST_TL(3);
    const int na = sh.na, nr = sh.nr;
    const bool changed = (na | nr) != 0;
    bool arriver = plan_wave && lane == 0;
    int next_epoch = ep;
    // Removals outnumber additions: the surplus ones are taken out one by one, in ascending index order, each by
    // moving the last entry of the list into its place (weight_cache.h:310-353).  With S of them the list ends as
    // its first n_old - S positions ("base"); the entries of the last S positions ("tail") that stay end up in the
    // places of the surplus indices below the tail.  Step k takes the entry at tail slot S-1-k and puts it where
    // the k-th surplus index sits at that time: its place in the list, unless that place is a tail slot whose own
    // step came earlier (then it has travelled on with that step's move, possibly again).  So the places follow
    // from the start positions by chasing through tail slots, which only surplus indices that START in the tail
    // need (few: about S^2 / n_old); they are resolved one after the other, then every surviving tail entry finds
    // its final place on its own.  This is the whole block's form of it, for the case that more than 64 surplus
    // indices start in the tail (the planning wave has done the others on its own, `fast`).  Used when
    // S <= min(1024, I/4) and the list was fetched far enough up front; else the per-index plan.
    const int surplus = nr - na, tail_base = n_old - surplus;
    const bool fast = surplus > 0 && sh.fast_ok != 0;
    const int smax = (I >> 2) < TPB ? (I >> 2) : TPB;
    // (LDS behind the list of added indices: the fetched list, then five arrays of smax entries: 6.5 bytes per index at most)
    bool replay = surplus > 0 && !fast && surplus <= smax && tail_base >= 0 && n_old <= scan_cap && I >= 256;
    constexpr uint16_t kGone = 0xffffu;   // hole[]: removed as the last entry, nothing moves; tailv[]: a surplus index
    uint16_t *const hole = scan_idx + ((scan_cap + 7) & ~7);   // start position of the k-th surplus index, then its place at step k
    uint16_t *const tailv = hole + ((smax + 7) & ~7);          // entry of tail slot j after the paired replacements
    if (replay) {
        const uint16_t *added_list = reinterpret_cast<const uint16_t *>(smem);
        // ---- every thread, four positions: paired replacements in place; where the surplus indices sit; the tail
        if (scan_in && scan_p < n_old) {
            uint2 pk = *reinterpret_cast<const uint2 *>(scan_idx + scan_p);
            uint32_t ent[kSparseScan] = {pk.x & 0xffffu, pk.x >> 16, pk.y & 0xffffu, pk.y >> 16};
            int found = 0, paired_tail = 0;
#pragma unroll
            for (int j = 0; j < kSparseScan; ++j) {
                const int p = scan_p + j;
                const int e = (int)ent[j];
                if (p < n_old) {
                    const int word = (e >> 5) & (kSparseMaxW32 - 1), bit = e & 31;
                    const uint32_t remw = sh.oldbits[word] & ~sh.newbits[word];
                    const bool rem = (remw >> bit) & 1u;
                    const int rank = rem ? (int)sh.pr[word] + __popc(remw & ((1u << bit) - 1u)) : 0;
                    const bool extra = rem && rank >= na;
                    if (rem && !extra) ent[j] = added_list[rank];
                    if (extra) { hole[rank - na] = (uint16_t)p; ++found; }
                    if (p >= tail_base) {
                        tailv[p - tail_base] = extra ? kGone : (uint16_t)ent[j];
                        if (rem && !extra) ++paired_tail;
                    }
                }
            }
            pk.x = ent[0] | (ent[1] << 16); pk.y = ent[2] | (ent[3] << 16);
            *reinterpret_cast<uint2 *>(scan_idx + scan_p) = pk;
            if (found) atomicAdd(&sh.found, found);
            if (paired_tail) atomicAdd(&sh.paired_tail, paired_tail);
        }
        lds_barrier();
        // ---- one wave: the places of the surplus indices that start in the tail.  An index's place depends on those
        // of smaller surplus indices only, and only on such that start in the tail themselves (the others stay where
        // they are), so they are resolved 64 at a time, one lane each, in rounds: a lane whose chase runs into an
        // index that is not resolved yet tries again in the next round (the smallest unresolved one always gets
        // through; two or three rounds as a rule).
        if (plan_wave) {
            const int S = __builtin_amdgcn_readfirstlane(surplus), base = __builtin_amdgcn_readfirstlane(tail_base);
            uint16_t *const jlist = tailv + ((smax + 7) & ~7);   // [S] the surplus indices (their rank k) that start in the tail
            uint16_t *const jrank = jlist + ((smax + 7) & ~7);   // [S] k -> position in jlist
            uint16_t *const jres = jrank + ((smax + 7) & ~7);    // [S] k -> resolved place
            int in_tail = 0;
            for (int c = 0; c < S; c += kWave) {
                const int k = c + lane;
                const bool is = k < S && (int)hole[k < S ? k : 0] >= base;
                const uint64_t m = __builtin_amdgcn_ballot_w64(is);
                if (is) {
                    const int j = in_tail + __popcll(m & ((1ull << lane) - 1ull));
                    jlist[j] = (uint16_t)k;
                    jrank[k] = (uint16_t)j;
                }
                in_tail += __popcll(m);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            for (int j0 = 0; j0 < in_tail; j0 += kWave) {
                const int kk = j0 + lane < in_tail ? (int)jlist[j0 + lane] : -1;
                bool open = kk >= 0;
                uint64_t resolved = 0;   // lanes of this group that are done (the same in every lane)
                int place = 0;
                for (int round = 0; round <= kWave && __builtin_amdgcn_ballot_w64(open) != 0; ++round) {
                    bool done = false;
                    if (open) {
                        int pos = hole[kk];
                        for (int it = 0; it <= S; ++it) {
                            const int i = S - 1 - (pos - base);   // the step that takes the entry of that tail slot
                            if (pos < base || pos == (int)kGone || i > kk || i < 0) { done = true; break; }   // stays there
                            if (i == kk) { pos = kGone; done = true; break; }   // it is the last entry at its own step
                            const int h = hole[i];
                            if (h < base) { pos = h; done = true; break; }      // travelled with an index that never moves
                            const int j = jrank[i];
                            if (j >= j0 && !((resolved >> (j - j0)) & 1ull)) break;   // not known yet: next round
                            pos = jres[i];
                        }
                        place = pos;
                    }
                    const uint64_t now = __builtin_amdgcn_ballot_w64(open && done);
                    if (open && done) jres[kk] = (uint16_t)place;
                    resolved |= now;
                    open = open && !done;
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                }
            }
            // (hole[] kept the start positions until here: the chase tells the two kinds of surplus index apart by them)
            for (int j = lane; j < in_tail; j += kWave) {
                const int kk = jlist[j];
                hole[kk] = jres[kk];
            }
            if (lane == 0) {
                // (a surplus index missing from the list would make the counts disagree: per-index plan then)
                sh.replay_ok = sh.found == S;
                sh.n = base;
                // rewritten positions: the pairs' below the tail, and the places of the surplus indices below it
                sh.nchg = na - sh.paired_tail + (S - in_tail);
            }
        }
        lds_barrier();
        replay = sh.replay_ok != 0;
        if (replay) {
            // ---- every surviving tail entry to its final place
            if (tid < surplus) {
                const uint16_t v = tailv[tid];
                if (v != kGone) {
                    int pos = hole[surplus - 1 - tid];
                    for (int it = 0; it < surplus && pos >= tail_base && pos < n_old; ++it)
                        pos = hole[surplus - 1 - (pos - tail_base)];
                    if (pos < tail_base) scan_idx[pos] = v;
                }
            }
            lds_barrier();
            if (plan_wave) {
                int s = -1;
                if (lane < Q && my_p < tail_base) {
                    const int newidx = scan_idx[my_p];
                    s = newidx != (ep ? i_old1 : i_old0) ? (newidx | kSrcPool) : my_p;
                    indices2[(size_t)(ep ^ 1) * I + my_p] = newidx;
                }
                sh.src[lane] = s;
            }
            lds_barrier();
        }
    }
    if (surplus <= 0 || fast || replay) {
        const int n_changed = fast || replay ? sh.nchg : na;
        n = sh.n;
        if (changed) {
            // the remembered mask: 8-byte words dealt to the blocks round-robin (the reference keeps the old
            // mask when the update leaves nothing active)
            uint8_t *mask_out = cur_mask2 + (size_t)(ep ^ 1) * I;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int bi = tid * nw_rt + w;
                if (w < nw_rt && bi * 8 < I && (bi % G) == blk)
                    store_mask<AL>(mask_out, bi * 8, I, n > 0 ? w_new[w] : w_cur[w]);
            }
            if (blk == 0 && arriver) {
                state[ST_STATE_N_BUF0 + (ep ^ 1)] = n;
                state[ST_STATE_N_ACTIVE] = n;
                state[ST_STATE_N_CHANGED] = n_changed;
                state[ST_STATE_N_ADDED] = na;
                state[ST_STATE_N_REMOVED] = nr;
                state[ST_STATE_SERIAL] = serial_old + 1;
                state[ST_STATE_EPOCH] = ep ^ 1;
                if (n > 0) {
                    state[ST_STATE_STATUS] = 0;
                    state[ST_STATE_VALID] = 1;
                } else {
                    state[ST_STATE_STATUS] = ST_ERR_NO_ACTIVE;
                }
            }
            next_epoch = ep ^ 1;
        } else if (blk == 0 && arriver) {
            state[ST_STATE_N_CHANGED] = 0;
            state[ST_STATE_N_ADDED] = 0;
            state[ST_STATE_N_REMOVED] = 0;
        }
        if (arriver) arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
    } else {
        // ---- too many surplus removals for the replay above: the per-index plan
        PlanView pv;
        cache_plan<true, TPB, NW, true, AL>(pv, smem, &plan_shared, new_mask, cur_mask2, indices2, state, I, tid);
        n = pv.n_new;
        if (plan_wave) {
            int s = -1;
            if (lane < Q && my_p < n) {
                const bool moved = my_p >= pv.n_old || ((pv.dirty[my_p >> 5] >> (my_p & 31)) & 1u);
                s = moved ? ((int)pv.idx_l[my_p] | kSrcPool) : my_p;
            }
            sh.src[lane] = s;
        }
        arriver = pv.arriver; arrival = pv.arrival; next_epoch = pv.next_epoch;
        // (requested again so that the first request's registers are free while the plan above runs)
        speculate(std::integral_constant<int, 0>{}, std::integral_constant<int, SPEC>{});
        lds_barrier();
    }
    if (blk == 0 && tid == 0) tell_count(host, n);
    ST_TL(4);

    float acc[NB][VEC];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[b][e] = 0.f;

    const int jcount = n > blk ? (n - blk + G - 1) / G : 0;      // rows of this block
    const int nbat = ((jcount + ngrp - 1) / ngrp + RB - 1) / RB;  // uniform over the block
    for (int bat = 0; bat < nbat; ++bat) {
        unsigned fresh = 0u;   // bit k: row of slot k comes from the pool and has to be written back
        auto request = [&](int k, bool speculated) __attribute__((always_inline)) {
            const int q = grp + ngrp * (bat * RB + k);
            const int p = blk + G * q;
            const int s = sh.src[q < kSparseMaxQ ? q : kSparseMaxQ - 1];
            const bool ok = q < Q && s >= 0;
            const bool pooled = ok && (s & kSrcPool) != 0;
            if (pooled) fresh |= 1u << k;
            if (speculated && !pooled && p < n_spec) return;
            const size_t ro = ok ? (size_t)(s & (kSrcPool - 1)) * row_bytes + coff : 0;   // no row: one piece for the whole wave
            wu[k] = ld16_stream((pooled ? pool_u : act_u) + ro);
            wd[k] = ld16_stream((pooled ? pool_d : act_d) + ro);
            wg[k] = has_gate ? ld16_stream((pooled ? pool_g : act_g) + ro) : zero4;
        };
        if (wave_live) {
            const bool spec = bat == 0 && n_spec > 0;
#pragma unroll
            for (int k = SPEC; k < RB; ++k) request(k, false);
#pragma unroll
            for (int k = 0; k < SPEC; ++k) request(k, spec);
            if (spec && !has_gate) {
#pragma unroll
                for (int k = 0; k < SPEC; ++k) wg[k] = zero4;
            }
        } else {
#pragma unroll
            for (int k = 0; k < RB; ++k) wg[k] = wu[k] = wd[k] = zero4;
        }
        ST_TL(6);

        // ---- phase 1: partial dot products on this thread's chunk
        uint4 xq[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) xq[b] = (valid && b < B) ? xr[b] : zero4;
#pragma unroll
        for (int k = 0; k < RB; ++k) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                float pg = 0.f, pu = 0.f;
                dot_chunk<T>(wg[k], wu[k], xq[b], pg, pu);
                const float sg = wave_sum_dpp(pg), su = wave_sum_dpp(pu);
                if (lane == 0) {
                    red[wave][k][b][0] = sg;
                    red[wave][k][b][1] = su;
                }
            }
        }
        // write the fresh rows back while the reductions settle
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            if (((fresh >> k) & 1u) && valid) {
                const size_t ro = (size_t)row_of(bat, k) * row_bytes + coff;
                st16(act_u + ro, wu[k]);
                st16(act_d + ro, wd[k]);
                if (has_gate) st16(act_g + ro, wg[k]);
            }
        }
        __syncthreads();
        if (tid < ngrp * RB * NB) {
            const int g_ = tid / (RB * NB), rem = tid - g_ * (RB * NB);
            const int k_ = rem / NB, b_ = rem - k_ * NB;
            const int row = blk + G * (g_ + ngrp * (bat * RB + k_));
            float sg = 0.f, su = 0.f;
            for (int wv = g_ * wpg; wv < (g_ + 1) * wpg; ++wv) {
                sg += red[wv][k_][b_][0];
                su += red[wv][k_][b_][1];
            }
            const float hv = has_gate ? activate(sg, act) * su : activate(su, act);
            const bool ok = row < n;
            hs[g_][k_][b_] = ok ? hv : 0.f;
            if (ok && combined && b_ < B) {
                combined[(size_t)b_ * ldc + row] = from_float<T>(hv);
                if (has_gate) combined[(size_t)b_ * ldc + n + row] = from_float<T>(su);
            }
        }
        __syncthreads();
        // ---- phase 2: down projection from the rows already in registers
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            const bool row_ok = row_of(bat, k) < n;
            const uint4 rd = row_ok ? wd[k] : zero4;
#pragma unroll
            for (int b = 0; b < NB; ++b) axpy_chunk<T>(hs[grp][k][b], rd, acc[b]);
        }
    }

    // ---- combine the thread groups through LDS (behind the plan arrays), one fp32 partial row per block
    if (ngrp > 1) {
        float *redc = reinterpret_cast<float *>(smem + plan_bytes);  // [ngrp-1][NB][H]
        if (grp > 0 && valid) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < VEC; e += 4)
                    *reinterpret_cast<float4 *>(redc + ((size_t)(grp - 1) * NB + b) * H + (size_t)cc * VEC + e) =
                        make_float4(acc[b][e], acc[b][e + 1], acc[b][e + 2], acc[b][e + 3]);
        }
        __syncthreads();
        if (grp == 0 && valid) {
            for (int gq = 1; gq < ngrp; ++gq)
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int e = 0; e < VEC; e += 4) {
                        const float4 v = *reinterpret_cast<const float4 *>(redc + ((size_t)(gq - 1) * NB + b) * H +
                                                                            (size_t)cc * VEC + e);
                        acc[b][e] += v.x; acc[b][e + 1] += v.y; acc[b][e + 2] += v.z; acc[b][e + 3] += v.w;
                    }
        }
    }
    if (grp == 0 && valid) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < VEC; e += 4)
                *reinterpret_cast<float4 *>(partials + ((size_t)blk * NB + b) * H + (size_t)cc * VEC + e) =
                    make_float4(acc[b][e], acc[b][e + 1], acc[b][e + 2], acc[b][e + 3]);
    }
    // the block that arrived last resets the arrivals and sets the epoch (the atomic's result is first looked at here)
    if (arriver) {
        asm volatile("" : "+v"(arrival));
        if ((arrival & 0xffffu) == (uint32_t)G - 1u)
            atomicExch(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), (uint32_t)next_epoch << 16);
    }
    ST_TL(7);
}

// ---------------------------------------------------------------------------
// update for intermediate sizes the kernels above cannot hold in LDS (kPlanMaxI < I <= kBigMaxI).
// The same replay of WeightCache::update_active_weights (weight_cache.h:229-359) in every block, with the
// masks as bitmaps and no added / removed lists: the i-th removed or added index is found through per-word
// prefix counts (rank of a set bit; i-th set bit by bisection), which leaves 4.5 bytes of LDS per element --
// the two index maps the sequential surplus removals (:310-353) need.  Blocks then copy the rows of the
// positions they own (position p belongs to block p mod (blocks - 1); block 0 publishes the bookkeeping).
// ---------------------------------------------------------------------------
constexpr int64_t kBigMaxI = 32768;
constexpr int kBigThreads = 1024;
constexpr int kBigWords = 4;   // 8-byte mask words per thread: I <= 8 * 1024 * 4

constexpr size_t big_lds_bytes(int I)
{
    const size_t w32 = (size_t)((I + 31) >> 5);
    return (size_t)I * 4 + w32 * 4 * 3 + w32 * 2 * 2 + 64;
}

struct BigShared {
    uint32_t wave_tot[kBigThreads / kWave];
    int n_new, na, nr;
};

// index of the i-th (from 0) set bit of bits[w] & ~mask_out[w] over all words, given the exclusive prefix counts
__device__ __forceinline__ int big_select(const uint32_t *bits, const uint32_t *notbits, const uint16_t *prefix, int W32, int i)
{
    int lo = 0;
    for (int step = 1024; step >= 1; step >>= 1) {
        const int c = lo + step;
        if (c < W32 && (int)prefix[c] <= i) lo = c;
    }
    uint32_t w = bits[lo] & ~notbits[lo];
    int j = i - (int)prefix[lo], pos = 0;
#pragma unroll
    for (int half = 16; half >= 1; half >>= 1) {
        const uint32_t lowmask = (1u << half) - 1u;
        const int c = __popc(w & lowmask);
        if (j >= c) { j -= c; pos += half; w >>= half; }
        w &= lowmask;
    }
    return lo * 32 + pos;
}

__global__ __launch_bounds__(kBigThreads) void cache_update_big_kernel(const uint8_t *__restrict__ new_mask,
                                                                      uint8_t *__restrict__ cur_mask2,
                                                                      int32_t *__restrict__ indices2,
                                                                      int32_t *__restrict__ state, int I, FusedRows fr,
                                                                      HostWords *host)
{
    constexpr int TPB = kBigThreads;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ BigShared bs;
    const int tid = threadIdx.x;
    const int W32 = (I + 31) >> 5;
    uint16_t *pos_l = reinterpret_cast<uint16_t *>(smem);   // index -> position (kNone when absent)
    uint16_t *idx_l = pos_l + I;                            // position -> index
    uint32_t *newbits = reinterpret_cast<uint32_t *>(idx_l + I + (I & 1));
    uint32_t *oldbits = newbits + W32, *dirty = oldbits + W32;
    uint16_t *pa = reinterpret_cast<uint16_t *>(dirty + W32), *pr = pa + W32 + (W32 & 1);
    auto sync = [&]() __attribute__((always_inline)) { lds_barrier(); };

    const uint32_t tword = __hip_atomic_load(reinterpret_cast<const uint32_t *>(&state[ST_STATE_TICKET]), __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    const int ep = (int)((tword >> 16) & 1u);
    const int n = state[ST_STATE_N_BUF0 + ep];
    const int serial_old = state[ST_STATE_SERIAL];
    const uint8_t *cur_mask = cur_mask2 + (size_t)ep * I;
    const int32_t *indices = indices2 + (size_t)ep * I;
    // masks -> bitmaps (8 elements per byte of the bitmaps), kept as 0x01 bytes in registers for publishing
    uint64_t w_new[kBigWords], w_cur[kBigWords];
#pragma unroll
    for (int w = 0; w < kBigWords; ++w) {
        const int bi = tid * kBigWords + w;
        const bool in = bi * 8 < I;
        const int ec = in ? bi * 8 : 0;
        w_new[w] = in ? nonzero_bytes(*reinterpret_cast<const uint64_t *>(new_mask + ec)) : 0ull;
        w_cur[w] = in ? nonzero_bytes(*reinterpret_cast<const uint64_t *>(cur_mask + ec)) : 0ull;
        if (bi < W32 * 4) {
            reinterpret_cast<uint8_t *>(newbits)[bi] = (uint8_t)pack_bits8(w_new[w]);
            reinterpret_cast<uint8_t *>(oldbits)[bi] = (uint8_t)pack_bits8(w_cur[w]);
        }
    }
    for (int i = tid; i < I; i += TPB) pos_l[i] = kNone;
    for (int w = tid; w < W32; w += TPB) dirty[w] = 0u;
    for (int p = tid; p < n; p += TPB) idx_l[p] = (uint16_t)indices[p];
    sync();
    for (int p = tid; p < n; p += TPB) pos_l[idx_l[p]] = (uint16_t)p;
    // per-word prefix counts of added / removed indices (one word per thread: W32 <= 1024)
    uint32_t addw = 0u, remw = 0u;
    if (tid < W32) { addw = newbits[tid] & ~oldbits[tid]; remw = oldbits[tid] & ~newbits[tid]; }
    uint32_t total;
    const uint32_t off = block_excl_scan<TPB / kWave>((uint32_t)__popc(addw) | ((uint32_t)__popc(remw) << 16), bs.wave_tot,
                                                      &total, tid, sync);
    if (tid < W32) { pa[tid] = (uint16_t)(off & 0xffffu); pr[tid] = (uint16_t)(off >> 16); }
    const int na = (int)(total & 0xffffu), nr = (int)(total >> 16);
    const bool writer = blockIdx.x == 0;
    uint32_t arrival = 0;
    if (na == 0 && nr == 0) {   // unchanged mask: nothing is touched (weight_cache.h:237-240)
        if (tid == 0 && writer) {
            state[ST_STATE_N_CHANGED] = 0;
            state[ST_STATE_N_ADDED] = 0;
            state[ST_STATE_N_REMOVED] = 0;
            tell_count(host, n);
        }
        if (tid == 0) {
            arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
            if ((arrival & 0xffffu) == gridDim.x - 1)
                atomicExch(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), (uint32_t)ep << 16);
        }
        return;
    }
    sync();   // pos_l, pa, pr complete
    const int pairs = na < nr ? na : nr;
    // ---- phase 1: the i-th removed index hands its position to the i-th added one; phase 2: surplus additions appended
    if (tid < W32) {
        uint32_t r = remw;
        int rank = (int)pr[tid];
        while (r && rank < pairs) {
            const int e = tid * 32 + __ffs((int)r) - 1;
            r &= r - 1u;
            const uint16_t p = pos_l[e];
            if (p != kNone) {
                const int a = big_select(newbits, oldbits, pa, W32, rank);
                idx_l[p] = (uint16_t)a;
                pos_l[a] = p;
                pos_l[e] = kNone;
                atomicOr(&dirty[p >> 5], 1u << (p & 31));
            }
            ++rank;
        }
        uint32_t a_bits = addw;
        int arank = (int)pa[tid];
        while (a_bits) {
            const int a = tid * 32 + __ffs((int)a_bits) - 1;
            a_bits &= a_bits - 1u;
            if (arank >= pairs) {
                const int p = n + (arank - pairs);
                if (p < I) {
                    idx_l[p] = (uint16_t)a;
                    pos_l[a] = (uint16_t)p;
                    atomicOr(&dirty[p >> 5], 1u << (p & 31));
                }
            }
            ++arank;
        }
    }
    sync();
    int n_new;
    if (nr <= na) {
        n_new = n + (na - pairs);
        if (n_new > I) n_new = I;
    } else {
        // ---- phase 3: surplus removals in ascending index order, sequential by construction
        if (tid == 0) {
            int m = n, k = 0;
            for (int w = 0; w < W32; ++w) {
                uint32_t r = oldbits[w] & ~newbits[w];
                while (r) {
                    const int e = w * 32 + __ffs((int)r) - 1;
                    r &= r - 1u;
                    if (k++ < pairs) continue;
                    const uint16_t p = pos_l[e];
                    if (p == kNone) continue;
                    if (m <= 0) { w = W32; break; }
                    const int last = m - 1;
                    if ((int)p != last) {
                        const uint16_t li = idx_l[last];
                        idx_l[p] = li;
                        pos_l[li] = p;
                        dirty[p >> 5] |= 1u << (p & 31);
                    }
                    --m;
                    pos_l[e] = kNone;
                }
            }
            bs.n_new = m;
        }
        sync();
        n_new = bs.n_new;
    }
    // rows rewritten: positions below the new count whose index changed
    uint32_t dcount = 0;
    for (int w = tid; w < W32; w += TPB) {
        uint32_t d = dirty[w];
        const int lo = w << 5;
        if (lo >= n_new) d = 0u;
        else if (lo + 32 > n_new) d &= (1u << (n_new - lo)) - 1u;
        dcount += (uint32_t)__popc(d);
    }
    uint32_t n_changed;
    (void)block_excl_scan<TPB / kWave>(dcount, bs.wave_tot, &n_changed, tid, sync);
    // ---- publish: block 0 writes the other bookkeeping buffer, the last arrival flips the epoch
    if (writer) {
        int32_t *idx_out = indices2 + (size_t)(ep ^ 1) * I;
        uint8_t *mask_out = cur_mask2 + (size_t)(ep ^ 1) * I;
        for (int p = tid; p < n_new; p += TPB) idx_out[p] = idx_l[p];
#pragma unroll
        for (int w = 0; w < kBigWords; ++w) {
            const int bi = tid * kBigWords + w;
            if (bi * 8 < I) *reinterpret_cast<uint64_t *>(mask_out + (size_t)bi * 8) = n_new > 0 ? w_new[w] : w_cur[w];
        }
        if (tid == 0) {
            state[ST_STATE_N_BUF0 + (ep ^ 1)] = n_new;
            state[ST_STATE_N_ACTIVE] = n_new;
            state[ST_STATE_N_CHANGED] = (int)n_changed;
            state[ST_STATE_N_ADDED] = na;
            state[ST_STATE_N_REMOVED] = nr;
            state[ST_STATE_SERIAL] = serial_old + 1;
            state[ST_STATE_EPOCH] = ep ^ 1;
            if (n_new > 0) {
                state[ST_STATE_STATUS] = 0;
                state[ST_STATE_VALID] = 1;
            } else {
                state[ST_STATE_STATUS] = ST_ERR_NO_ACTIVE;
            }
            tell_count(host, n_new);
        }
    }
    if (tid == 0) arrival = atomicAdd(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), 1u);
    // ---- copies: active[p] <- pool[index at p] for the dirty positions this block owns
    {
        const int row_bytes = fr.row_bytes, chunks = row_bytes >> 4;
        const bool has_gate = fr.has_gate != 0;
        const bool solo = gridDim.x == 1;
        const int owners = solo ? 1 : (int)gridDim.x - 1, me = solo ? 0 : (int)blockIdx.x - 1;
        if (solo || !writer) {
            for (int p = me; p < n_new; p += owners) {
                if (!((dirty[p >> 5] >> (p & 31)) & 1u)) continue;   // uniform over the block
                const size_t from = (size_t)idx_l[p] * row_bytes, to = (size_t)p * row_bytes;
                for (int c = tid; c < chunks; c += TPB) {
                    const size_t o = (size_t)c << 4;
                    const uint4 vu = ld16(fr.pool_u + from + o), vd = ld16(fr.pool_d + from + o);
                    uint4 vg = make_uint4(0u, 0u, 0u, 0u);
                    if (has_gate) vg = ld16(fr.pool_g + from + o);
                    st16(fr.act_u + to + o, vu);
                    st16(fr.act_d + to + o, vd);
                    if (has_gate) st16(fr.act_g + to + o, vg);
                }
            }
        }
    }
    if (tid == 0 && (arrival & 0xffffu) == gridDim.x - 1)
        atomicExch(reinterpret_cast<uint32_t *>(&state[ST_STATE_TICKET]), (uint32_t)(ep ^ 1) << 16);
}

// ---------------------------------------------------------------------------
// construction
// ---------------------------------------------------------------------------
// The module's matrices [gate,] up [I,H] and down [H,I], the pools and the packed buffers.
struct BuildMats {
    const unsigned char *src[2], *down;
    unsigned char *pool[2], *active[2], *downT_pool, *down_active;
    int nrow;          // matrices copied by row: 2 gated, 1 ungated
    int row_bytes;
    int down_vec;      // rows of `down` may be read in 16-byte vectors
};

// Elements e .. e + 7 of a mask as 0x01 bytes (0 past I and for a null mask).
__device__ __forceinline__ uint64_t mask8(const uint8_t *__restrict__ mask, int e, int I, bool vec)
{
    if (mask == nullptr || e >= I) return 0ull;
    if (vec && e + 8 <= I) return nonzero_bytes(*reinterpret_cast<const uint64_t *>(mask + e));
    uint64_t v = 0;
    for (int k = 0; k < 8; ++k)
        if (e + k < I && mask[e + k]) v |= 1ull << (8 * k);
    return v;
}

constexpr int kBuildThreads = 256, kBuildRows = kBuildThreads / kWave;   // a wave per row
template <int ESZ> struct BuildTile { static constexpr int rows = 256 / ESZ; };   // of a transposed tile, both ways: 256 bytes

// Everything a new cache holds, in one pass over the module's weights: pools, packed rows of the initial mask in ascending
// order (what the first update of an empty cache gives, weight_cache.h:199-226) and the bookkeeping of that update; with a
// null mask the pools and an empty cache.  Bound by memory: each weight is read once and written to the pool and the packed
// buffer from registers.  Block 0 does the bookkeeping, the next copy a row of gate or up per wave, the last transpose
// 256 x 256 byte tiles of `down`, 8 x 8 (4 x 4) elements per thread in registers, so that a wave's loads and stores are
// 128-byte lines on both sides and nothing goes through LDS.  A row's position is the number of set mask bytes before it,
// counted by every block while its rows are on the way.
// H 3072, I 8192, fp16, all rows (453 MB): 160 us as two copies, a transposing kernel (44 us), a reset and an update
// (69 us, reading the pools back), 79 us as one (5.7 TB/s).
template <int ESZ>
__global__ __launch_bounds__(kBuildThreads) void cache_build_kernel(const uint8_t *__restrict__ mask,
                                                                    uint8_t *__restrict__ cur_mask2,
                                                                    int32_t *__restrict__ indices2,
                                                                    int32_t *__restrict__ state, int I, int H, int mask_vec,
                                                                    HostWords *host, BuildMats a)
{
    constexpr int kTile = BuildTile<ESZ>::rows, V = 16 / ESZ;
    __shared__ uint32_t wave_tot[kBuildThreads / kWave];
    __shared__ int tile_pos[kTile];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto sync = [&]() __attribute__((always_inline)) { lds_barrier(); };
    // set mask bytes before element e0 (a multiple of 4); ends behind a barrier
    auto rank_of = [&](int e0) __attribute__((always_inline)) -> int {
        uint32_t c = 0;
#pragma unroll 4
        for (int e = 8 * tid; e < e0; e += 8 * kBuildThreads) {
            uint64_t m = mask8(mask, e, I, mask_vec);
            if (e + 8 > e0) m &= 0xffffffffull;
            c += (uint32_t)__popcll(m);
        }
        const uint32_t incl = wave_incl_scan_dpp(c, lane);
        if (lane == kWave - 1) wave_tot[wave] = incl;
        sync();
        uint32_t t = 0;
#pragma unroll
        for (int w = 0; w < kBuildThreads / kWave; ++w) t += wave_tot[w];
        return (int)t;
    };
    const int row_groups = (I + kBuildRows - 1) / kBuildRows;
    int unit = (int)blockIdx.x - 1;
    if (unit < 0) {   // ---- bookkeeping: every thread a contiguous range of the mask
        const int words = (I + 8 * kBuildThreads - 1) / (8 * kBuildThreads);
        uint32_t cnt = 0;
        for (int w = 0; w < words; ++w) cnt += (uint32_t)__popcll(mask8(mask, 8 * (tid * words + w), I, mask_vec));
        uint32_t total;
        int at = (int)block_excl_scan<kBuildThreads / kWave>(cnt, wave_tot, &total, tid, sync);
        const int n = (int)total;
        if (tid == 0) {
            // an empty initial mask equals the empty cache's: nothing changes and nothing is valid (weight_cache.h:237-240)
            const int some = n > 0 ? 1 : 0;
            int w[ST_STATE_WORDS] = {};
            w[ST_STATE_N_ACTIVE] = w[ST_STATE_N_CHANGED] = w[ST_STATE_N_ADDED] = w[ST_STATE_N_BUF1] = n;
            w[ST_STATE_VALID] = w[ST_STATE_SERIAL] = w[ST_STATE_EPOCH] = some;
            w[ST_STATE_TICKET] = some << 16;
            for (int k = 0; k < ST_STATE_WORDS; ++k) state[k] = w[k];
            tell_count(host, n);
        }
        for (int w = 0; w < words; ++w) {
            const int e0 = 8 * (tid * words + w);
            const uint64_t m = mask8(mask, e0, I, mask_vec);
            for (int k = 0; k < 8 && e0 + k < I; ++k) {
                const int e = e0 + k;
                const bool set = (m >> (8 * k)) & 1u;
                cur_mask2[e] = 0;
                cur_mask2[(size_t)I + e] = set ? 1 : 0;
                indices2[e] = -1;
                if (set) indices2[(size_t)I + at++] = e;
                if (e >= n) indices2[(size_t)I + e] = -1;
            }
        }
        return;
    }
    if (unit < a.nrow * row_groups) {   // ---- rows of gate and up
        const int m = unit >= row_groups ? 1 : 0, r0 = (unit - m * row_groups) * kBuildRows, r = r0 + wave;
        const bool in = r < I;
        const unsigned char *const from = (m ? a.src[1] : a.src[0]) + (size_t)(in ? r : r0) * a.row_bytes;
        unsigned char *const pool = (m ? a.pool[1] : a.pool[0]) + (size_t)r * a.row_bytes;
        const int chunks = a.row_bytes >> 4;
        constexpr int U = 8;
        uint4 v[U];
        auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * kWave;
                v[u] = ld16_stream(from + ((size_t)(c < chunks ? c : chunks - 1) << 4));
            }
        };
        load(lane);
        int pos = -1;
        if (mask != nullptr) {
            const int before = rank_of(r0);
            int mine = 0;
            for (int k = 0; k < wave; ++k) mine += r0 + k < I && mask[r0 + k] ? 1 : 0;
            if (in && mask[r]) pos = before + mine;
        }
        if (!in) return;
        unsigned char *const act = (m ? a.active[1] : a.active[0]) + (size_t)(pos < 0 ? 0 : pos) * a.row_bytes;
        for (int c0 = lane; c0 < chunks; c0 += U * kWave) {
            if (c0 != lane) load(c0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * kWave;
                if (c >= chunks) continue;
                st16(pool + ((size_t)c << 4), v[u]);
                if (pos >= 0) st16(act + ((size_t)c << 4), v[u]);
            }
        }
        return;
    }
    // ---- a tile of down: waves 2 x 2, lanes 8 x 8, V x V elements each
    unit -= a.nrow * row_groups;
    const int ht = (H + kTile - 1) / kTile;
    const int i0 = (unit / ht) * kTile, h0 = (unit % ht) * kTile;
    const int il = (wave & 1) * 8 * V + (lane & 7) * V, h = h0 + (wave >> 1) * 8 * V + (lane >> 3) * V, i = i0 + il;
    const bool in = h < H && i < I;   // (H is a multiple of V)
    uint4 v[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        v[k] = make_uint4(0u, 0u, 0u, 0u);
        if (!in) continue;
        const unsigned char *const p = a.down + ((size_t)(h + k) * I + i) * ESZ;
        if (a.down_vec) {
            v[k] = ld16_stream(p);
        } else {
            uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (i + e >= I) continue;
                if constexpr (ESZ == 2) d[e >> 1] |= (uint32_t)reinterpret_cast<const uint16_t *>(p)[e] << (16 * (e & 1));
                else d[e] = reinterpret_cast<const uint32_t *>(p)[e];
            }
            v[k] = make_uint4(d[0], d[1], d[2], d[3]);
        }
    }
    if (mask != nullptr) {
        const int before = rank_of(i0);
        const int e = i0 + tid;
        if (tid < kTile) {   // (whole waves)
            const bool set = e < I && mask[e] != 0;
            const uint64_t b = __ballot(set);
            int c = before + (int)__popcll(b & ((1ull << lane) - 1ull));
            if (wave == 1) {   // behind the first wave's elements
                const bool first = i0 + lane < I && mask[i0 + lane] != 0;
                c += (int)__popcll(__ballot(first));
            }
            tile_pos[tid] = set ? c : -1;
        }
        sync();
    }
    if (!in) return;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        if (i + k >= I) continue;
        uint32_t o[4];
        auto word = [&](const uint4 &q, int j) __attribute__((always_inline)) { return j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w; };
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (ESZ == 2)
                o[j] = __builtin_amdgcn_perm(word(v[2 * j + 1], k >> 1), word(v[2 * j], k >> 1), k & 1 ? 0x07060302u : 0x05040100u);
            else
                o[j] = word(v[j], k);
        }
        const uint4 q = make_uint4(o[0], o[1], o[2], o[3]);
        st16(a.downT_pool + (size_t)(i + k) * a.row_bytes + (size_t)h * ESZ, q);
        if (mask != nullptr) {
            const int p = tile_pos[il + k];
            if (p >= 0) st16(a.down_active + (size_t)p * a.row_bytes + (size_t)h * ESZ, q);
        }
    }
}

// ---------------------------------------------------------------------------
// the caches' pinned words
// ---------------------------------------------------------------------------
// A cache's copy of its state words and, behind them, what its updates write by themselves.
struct HostSlot {
    int32_t state[ST_STATE_WORDS];
    HostWords words;
};
static_assert(ST_STATE_WORDS * sizeof(int32_t) == 64 && sizeof(HostSlot) == 256, "cache lines of their own");

// Slots come from slabs that are kept between caches (allocating and freeing pinned memory waits for the device, and the
// words of a model's caches share pages).  At most one slab per GPU stays without a user.  A kernel still on its way when
// its cache is destroyed may write to the slot's next owner: its count is a guess there as everywhere, and the state words
// carry the number of their wait, which goes on from owner to owner.
struct HostSlab {
    static constexpr int kSlots = 64;
    HostSlab *next;
    int device;
    HostSlot *base;
    uint64_t used;
    uint32_t number[kSlots];
};
static std::mutex host_slab_mutex;
static HostSlab *host_slabs = nullptr;

// A free slot of the current device, zeroed; false if there is no memory.
static bool take_host_slot(HostSlab **slab, int *at)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(host_slab_mutex);
    HostSlab *s = host_slabs;
    while (s && (s->device != dev || s->used == ~0ull)) s = s->next;
    if (!s) {
        s = new (std::nothrow) HostSlab{};
        if (!s) return false;
        if (hipHostMalloc(reinterpret_cast<void **>(&s->base), HostSlab::kSlots * sizeof(HostSlot), hipHostMallocDefault) != hipSuccess) {
            delete s;
            return false;
        }
        s->device = dev;
        s->next = host_slabs;
        host_slabs = s;
    }
    *slab = s;
    *at = __builtin_ctzll(~s->used);
    s->used |= 1ull << *at;
    memset(&s->base[*at], 0, sizeof(HostSlot));
    return true;
}

static void give_host_slot_back(HostSlab *slab, int at, uint32_t number)
{
    std::lock_guard<std::mutex> lock(host_slab_mutex);
    slab->number[at] = number;
    slab->used &= ~(1ull << at);
    if (slab->used != 0) return;
    for (HostSlab **link = &host_slabs; *link; link = &(*link)->next) {   // another one without a user goes
        HostSlab *s = *link;
        if (s == slab || s->device != slab->device || s->used != 0) continue;
        *link = s->next;
        (void)hipHostFree(s->base);
        delete s;
        return;
    }
}

}  // namespace st

struct st_cache {
    st_cache_buffers b;
    int64_t I, H;
    int dtype, has_gate;
    int esz;
    st::HostSlab *slab;    // whose slot `slot` holds the next two
    int slot;
    int32_t *host_state;   // pinned: ST_STATE_WORDS words as st_cache_sync_state last read them
    st::HostWords *host;   // pinned, behind them: what updates write by themselves
    uint32_t number;       // of the last wait
};

extern "C" int64_t st_cache_max_intermediate(void) { return st::kBigMaxI; }

extern "C" st_cache *st_cache_create(const st_cache_buffers *bufs, int64_t I, int64_t H, int dtype, int has_gate)
{
    using namespace st;
    auto fail = [](const char *m) -> st_cache * { set_error("st_cache_create: %s", m); return nullptr; };
    if (!bufs) return fail("null buffers");
    if (dtype < ST_F32 || dtype > ST_BF16) return fail("unknown dtype");
    const int esz = dtype == ST_F32 ? 4 : 2;
    if (I < 1 || I > kBigMaxI) return fail("intermediate size out of range (see st_cache_max_intermediate)");
    if (I > kPlanMaxI && I % 8 != 0) return fail("intermediate sizes above 22000 must be multiples of 8");
    if (H < 1 || (H * esz) % 16 != 0) return fail("rows are not 16-byte multiples");
    if (!bufs->up_pool || !bufs->downT_pool || !bufs->up_active || !bufs->down_active || !bufs->indices ||
        !bufs->cur_mask || !bufs->state)
        return fail("null device buffer");
    if (has_gate && (!bufs->gate_pool || !bufs->gate_active)) return fail("has_gate set but gate buffers are null");
    const uintptr_t align = (uintptr_t)bufs->gate_pool | (uintptr_t)bufs->up_pool | (uintptr_t)bufs->downT_pool |
                            (uintptr_t)bufs->gate_active | (uintptr_t)bufs->up_active | (uintptr_t)bufs->down_active;
    if (align & 15) return fail("weight buffers must be 16-byte aligned");
    st_cache *c = new (std::nothrow) st_cache;
    if (!c) return fail("out of host memory");
    c->b = *bufs;
    c->I = I; c->H = H; c->dtype = dtype; c->has_gate = has_gate ? 1 : 0; c->esz = esz;
    if (!take_host_slot(&c->slab, &c->slot)) {
        delete c;
        return fail("hipHostMalloc failed");
    }
    c->host_state = c->slab->base[c->slot].state;
    c->host = &c->slab->base[c->slot].words;
    c->number = c->slab->number[c->slot];
    return c;
}

extern "C" void st_cache_destroy(st_cache *c)
{
    if (!c) return;
    st::give_host_slot_back(c->slab, c->slot, c->number);
    delete c;
}

// mask: of the rows that are active afterwards, in ascending order (null: none).
static int launch_build(st_cache *c, const void *gate, const void *up, const void *down, const uint8_t *mask, hipStream_t s)
{
    using namespace st;
    const size_t bytes = (size_t)c->I * c->H * c->esz;
    BuildMats a;
    a.row_bytes = (int)(c->H * c->esz);
    a.nrow = 0;
    auto rows = [&](const void *src, void *pool, void *active) -> int {
        if ((uintptr_t)src & 15) {   // rows that cannot be read in vectors: into the pool first, the kernel reads them there
            ST_HIP(hipMemcpyAsync(pool, src, bytes, hipMemcpyDeviceToDevice, s));
            src = pool;
        }
        a.src[a.nrow] = static_cast<const unsigned char *>(src);
        a.pool[a.nrow] = static_cast<unsigned char *>(pool);
        a.active[a.nrow++] = static_cast<unsigned char *>(active);
        return ST_OK;
    };
    int rc = c->has_gate ? rows(gate, c->b.gate_pool, c->b.gate_active) : ST_OK;
    if (rc == ST_OK) rc = rows(up, c->b.up_pool, c->b.up_active);
    if (rc != ST_OK) return rc;
    if (a.nrow == 1) { a.src[1] = a.src[0]; a.pool[1] = a.pool[0]; a.active[1] = a.active[0]; }
    a.down = static_cast<const unsigned char *>(down);
    a.downT_pool = static_cast<unsigned char *>(c->b.downT_pool);
    a.down_active = static_cast<unsigned char *>(c->b.down_active);
    a.down_vec = ((uintptr_t)down & 15) == 0 && (c->I * c->esz) % 16 == 0;
    const int tile = 256 / c->esz;
    const int64_t blocks = 1 + (int64_t)a.nrow * ((c->I + kBuildRows - 1) / kBuildRows) +
                           ((c->I + tile - 1) / tile) * ((c->H + tile - 1) / tile);
    ST_REQUIRE(blocks <= 0x7fffffff, "st_cache: hidden size %lld out of range", (long long)c->H);
    const int mask_vec = ((uintptr_t)mask & 7) == 0;
    if (c->esz == 4)
        hipLaunchKernelGGL(cache_build_kernel<4>, dim3((unsigned)blocks), dim3(kBuildThreads), 0, s, mask, c->b.cur_mask,
                           c->b.indices, c->b.state, (int)c->I, (int)c->H, mask_vec, c->host, a);
    else
        hipLaunchKernelGGL(cache_build_kernel<2>, dim3((unsigned)blocks), dim3(kBuildThreads), 0, s, mask, c->b.cur_mask,
                           c->b.indices, c->b.state, (int)c->I, (int)c->H, mask_vec, c->host, a);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

extern "C" int st_cache_load_weights(st_cache *c, const void *gate, const void *up, const void *down, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && up && down, "st_cache_load_weights: null pointer");
    ST_REQUIRE(!c->has_gate || gate, "st_cache_load_weights: gated cache needs gate weights");
    return launch_build(c, gate, up, down, nullptr, static_cast<hipStream_t>(stream));
}

// The pointers of one cache and the mask of its update.
static st::UpdateLayer update_layer(const st_cache *c, const uint8_t *mask)
{
    st::UpdateLayer y;
    y.new_mask = mask;
    y.cur_mask2 = c->b.cur_mask;
    y.indices2 = c->b.indices;
    y.state = c->b.state;
    int m = 0;
    if (c->has_gate) {
        y.pool[m] = static_cast<const unsigned char *>(c->b.gate_pool);
        y.active[m++] = static_cast<unsigned char *>(c->b.gate_active);
    }
    y.pool[m] = static_cast<const unsigned char *>(c->b.up_pool);
    y.active[m++] = static_cast<unsigned char *>(c->b.up_active);
    y.pool[m] = static_cast<const unsigned char *>(c->b.downT_pool);
    y.active[m++] = static_cast<unsigned char *>(c->b.down_active);
    for (; m < 3; ++m) { y.pool[m] = y.pool[0]; y.active[m] = y.active[0]; }
    y.host = c->host;
    return y;
}

// Masks as 8-byte words, index lists as 16-byte vectors, with no rest?
static bool update_is_aligned(const st_cache *c, const uint8_t *mask)
{
    return c->I % 8 == 0 && (uintptr_t)mask % 8 == 0 && (uintptr_t)c->b.cur_mask % 8 == 0 && (uintptr_t)c->b.indices % 16 == 0;
}

// The count an update last told the host, 0 if none has yet.  A guess: later updates may be on their way.
static int seen_count(const st_cache *c) { return *const_cast<const volatile int32_t *>(&c->host->count); }

// How much of the index list the plan fetches up front: a quarter more than the count the host saw last, everything when
// it has seen none.
static int update_idx_cap(const st_cache *c)
{
    const int I = (int)c->I, seen = seen_count(c);
    return seen > 0 && seen + seen / 4 + 64 < I ? (seen + seen / 4 + 64 + 7) & ~7 : I;
}

// One update, or those of L > 1 caches of equal shape in one launch (I <= kPlanMaxI; L > 1: I >= 8).
static int launch_update(st_cache *const *caches, const uint8_t *const *masks, int L, hipStream_t s)
{
    using namespace st;
    const st_cache *c = caches[0];
    const int I = (int)c->I;
    static const int blocks = [] {
        const char *v = getenv("ST_CACHE_BLOCKS");
        const int b = v ? atoi(v) : 0;
        return b >= 1 && b <= 1024 ? b : 0;
    }();
    static const int want_tpb = [] {
        const char *v = getenv("ST_CACHE_TPB");
        return v ? atoi(v) : 0;
    }();
    const bool words_fit = I >= 8;
    bool aligned = true;
    for (int l = 0; l < L; ++l) aligned = aligned && update_is_aligned(caches[l], masks[l]);
    // 512-thread blocks (ST_CACHE_TPB=512) leave room on the CU for a kernel of another stream, but
    // measure slower on their own; they cover I <= 12288.
    const bool small = L == 1 && want_tpb == 512 && words_fit && I <= 8 * 512 * 3;
    const int tpb = small ? 512 : kPlanThreads, words = (I + 8 * tpb - 1) / (8 * tpb);
    const UpdateLayer y = update_layer(c, masks[0]);
    CopyPlan cp;
    for (int m = 0; m < 3; ++m) { cp.pool[m] = y.pool[m]; cp.active[m] = y.active[m]; }
    cp.nmat = c->has_gate ? 3 : 2;
    cp.row_bytes = (int)(c->H * c->esz);
    ProfScope ps(ST_K_CACHE_UPDATE, s);
    auto launch = [&](auto kern, int grid, size_t lds, auto... rest) -> int {
        const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), 160 * 1024 - 256);
        if (rc != ST_OK) return rc;
        ST_LAUNCH(ps, kern, dim3(grid, L), dim3(tpb), lds, s, masks[0], c->b.cur_mask, c->b.indices, c->b.state, I,
                  rest...);
        return ST_OK;
    };
    int rc;
    if (L > 1) {
        UpdateLayers tab;
        int idx_cap = 0;
        for (int l = 0; l < kMaxLayers; ++l) {
            const int k = l < L ? l : 0;
            tab.l[l] = update_layer(caches[k], masks[k]);
            const int cap = update_idx_cap(caches[k]);
            idx_cap = cap > idx_cap ? cap : idx_cap;
        }
        // A block per CU: every one of them plans (4 us), then the copies run at the rate of the memory (28 caches at
        // H 3072, I 8192, 290 changed rows each: 300 MB in 55 us; two blocks per CU measured the same there, and 9 us
        // slower for two caches at I 14336)
        const size_t lds = update_lds_bytes(I);
        const int most = device_cu_count() * 3 / 4;
        int grid = blocks ? blocks : device_cu_count() / L;
        grid = grid < 4 ? 4 : grid > most ? most : grid;
        auto go = [&](auto al) -> int {
            constexpr bool AL = decltype(al)::value;
            return words == 1   ? launch(cache_update_kernel<1024, 1, UpdateLayers, AL>, grid, lds, idx_cap, cp, c->host, tab)
                   : words == 2 ? launch(cache_update_kernel<1024, 2, UpdateLayers, AL>, grid, lds, idx_cap, cp, c->host, tab)
                                : launch(cache_update_kernel<1024, 3, UpdateLayers, AL>, grid, lds, idx_cap, cp, c->host, tab);
        };
        rc = aligned ? go(std::true_type{}) : go(std::false_type{});
    } else {
        const int grid = blocks ? blocks : device_cu_count() * 3 / 4;   // (measured against 1/4, 3/8, 1/2 and all of the CUs)
        const size_t lds = update_lds_bytes(I);
        const int idx_cap = update_idx_cap(c);
        auto go = [&](auto al) -> int {
            constexpr bool AL = decltype(al)::value;
            return small        ? launch(cache_update_kernel<512, 3, NoLayers, AL>, grid, lds, idx_cap, cp, c->host, NoLayers{})
                   : words == 1 ? launch(cache_update_kernel<1024, 1, NoLayers, AL>, grid, lds, idx_cap, cp, c->host, NoLayers{})
                   : words == 2 ? launch(cache_update_kernel<1024, 2, NoLayers, AL>, grid, lds, idx_cap, cp, c->host, NoLayers{})
                                : launch(cache_update_kernel<1024, 3, NoLayers, AL>, grid, lds, idx_cap, cp, c->host, NoLayers{});
        };
        rc = !words_fit ? launch(cache_update_bytes_kernel<1024>, grid, plan_lds_bytes(I), cp, c->host)
             : aligned  ? go(std::true_type{})
                        : go(std::false_type{});
    }
    if (rc != ST_OK) return rc;
    ST_HIP(hipGetLastError());
    return ST_OK;
}

extern "C" int st_cache_update_async(st_cache *c, const uint8_t *mask, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && mask, "st_cache_update_async: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int I = (int)c->I;
    if (I > kPlanMaxI) {   // index maps of the other kernels do not fit the LDS: bitmap plan, rows by position
        ST_REQUIRE(I % 8 == 0 && (uintptr_t)mask % 8 == 0 && (uintptr_t)c->b.cur_mask % 8 == 0,
                   "st_cache_update_async: for I > %lld the masks must be 8-byte aligned", (long long)kPlanMaxI);
        FusedRows fr;
        fr.pool_u = static_cast<const unsigned char *>(c->b.up_pool);
        fr.act_u = static_cast<unsigned char *>(c->b.up_active);
        fr.pool_d = static_cast<const unsigned char *>(c->b.downT_pool);
        fr.act_d = static_cast<unsigned char *>(c->b.down_active);
        fr.pool_g = c->has_gate ? static_cast<const unsigned char *>(c->b.gate_pool) : fr.pool_u;
        fr.act_g = c->has_gate ? static_cast<unsigned char *>(c->b.gate_active) : fr.act_u;
        fr.row_bytes = (int)(c->H * c->esz);
        fr.has_gate = c->has_gate ? 1 : 0;
        const size_t lds_big = big_lds_bytes(I);
        static std::atomic<bool> big_attr{false};
        if (!big_attr.load(std::memory_order_acquire)) {
            ST_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(cache_update_big_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024));
            big_attr.store(true, std::memory_order_release);
        }
        ProfScope ps(ST_K_CACHE_UPDATE, s);
        ST_LAUNCH(ps, cache_update_big_kernel, dim3(device_cu_count()), dim3(kBigThreads), lds_big, s, mask,
                  c->b.cur_mask, c->b.indices, c->b.state, I, fr, c->host);
        ST_HIP(hipGetLastError());
        return ST_OK;
    }
    return launch_update(&c, &mask, 1, s);
}

extern "C" int st_cache_update_layers(st_cache *const *caches, const uint8_t *const *masks, int64_t L, void *stream)
{
    using namespace st;
    ST_REQUIRE(caches && masks && L >= 1, "st_cache_update_layers: null pointer or no layers");
    for (int64_t l = 0; l < L; ++l) {
        ST_REQUIRE(caches[l] && masks[l], "st_cache_update_layers: null pointer in layer %lld", (long long)l);
        for (int64_t k = 0; k < l; ++k)
            ST_REQUIRE(caches[k] != caches[l], "st_cache_update_layers: layers %lld and %lld are the same cache", (long long)k, (long long)l);
    }
    for (int64_t l0 = 0; l0 < L;) {
        // as many neighbours of one shape as a launch takes
        const st_cache *c = caches[l0];
        int nl = 1;
        while (nl < kMaxLayers && l0 + nl < L && caches[l0 + nl]->I == c->I && caches[l0 + nl]->H == c->H &&
               caches[l0 + nl]->dtype == c->dtype && caches[l0 + nl]->has_gate == c->has_gate)
            ++nl;
        if (nl == 1 || c->I < 8 || c->I > kPlanMaxI) {
            const int rc = st_cache_update_async(caches[l0], masks[l0], stream);
            if (rc != ST_OK) return rc;
            l0 += 1;
            continue;
        }
        const int rc = launch_update(caches + l0, masks + l0, nl, static_cast<hipStream_t>(stream));
        if (rc != ST_OK) return rc;
        l0 += nl;
    }
    return ST_OK;
}

extern "C" int st_cache_update_forward(st_cache *c, const uint8_t *mask, const void *x, int64_t B, int64_t n_hint,
                                       void *out, void *combined, int64_t ldc, void *workspace,
                                       int64_t workspace_bytes, int act, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && mask && x && out && workspace, "st_cache_update_forward: null pointer");
    ST_REQUIRE(B >= 1 && B <= 4096, "st_cache_update_forward: B=%lld out of range [1,4096]", (long long)B);
    ST_REQUIRE(act >= ST_ACT_RELU && act <= ST_ACT_IDENTITY, "st_cache_update_forward: unknown activation %d", act);
    ST_REQUIRE(workspace_bytes >= st_mlp_workspace_bytes(B, c->H, c->I),
               "st_cache_update_forward: workspace too small (%lld < %lld)", (long long)workspace_bytes,
               (long long)st_mlp_workspace_bytes(B, c->H, c->I));
    ST_REQUIRE((((uintptr_t)x | (uintptr_t)workspace) & 15) == 0, "st_cache_update_forward: pointers must be 16-byte aligned");
    // the count after the update is only known on the device: `combined` has to hold the largest possible one
    ST_REQUIRE(!combined || ldc >= (c->has_gate ? 2 : 1) * c->I,
               "st_cache_update_forward: ldc=%lld too small for %lld intermediate rows", (long long)ldc, (long long)c->I);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int I = (int)c->I, H = (int)c->H;
    const int row_bytes = (int)(c->H * c->esz), chunks = row_bytes >> 4;
    constexpr int TPB = 1024;
    int gs_log2 = 6;
    while ((1 << gs_log2) < chunks && (1 << gs_log2) < TPB) ++gs_log2;
    const int ngrp = TPB >> gs_log2;
    const size_t plan_bytes = (plan_lds_bytes(I) + 15) & ~(size_t)15;
    const int NBF = B == 2 ? 2 : 1;   // rows of x the fused kernel takes in one pass
    const size_t lds = plan_bytes + (size_t)(ngrp - 1) * NBF * H * 4;
    const int G = mlp_grid();
    static const bool fused_off = [] { const char *v = getenv("ST_CACHE_FUSED"); return v && atoi(v) == 0; }();
    const bool aligned = update_is_aligned(c, mask);
    // One kernel for one or two rows of x when a block owns at most kSparseMaxQ positions, the masks fit the
    // kernel's bitmaps and a row fits one pass of a thread group; everything else runs as two calls, as do two rows of small
    // matrices without alignment.  Replayed, us, one kernel / two calls: fp16, H 512, I 1537 19.0 / 17.5; H 896, 2689 19.0 / 17.8;
    // H 1536, 5001 19.3 / 19.0; H 1792, 5001 19.0 / 19.4; H 2048, 8189 20.9 / 22.2; fp32, H 1024, 4001 18.2 / 18.0; one after the
    // other from the host 0.2 to 1.6 us less for the calls up to H 2048, 5001.
    const bool fused = !fused_off && B <= 2 && I >= 8 && !(B == 2 && !aligned && (int64_t)I * row_bytes <= (int64_t)16 << 20) && G <= 0xffff && (I + G - 1) / G <= kSparseMaxQ &&
                       I <= 32 * kSparseMaxW32 && I <= 8 * TPB * kSparseWords && chunks <= TPB && row_bytes % 16 == 0 &&
                       lds <= (size_t)(148 * 1024);
    if (!fused) {   // two launches: update, then the forward that reads the count on the device
        if (n_hint < 0) n_hint = seen_count(c);
        const int rc = st_cache_update_async(c, mask, stream);
        if (rc != ST_OK) return rc;
        return st_mlp_forward(x, B, c->H, c->b.gate_active, c->b.up_active, c->b.down_active, c->I,
                              c->b.state + ST_STATE_N_ACTIVE, n_hint, out, combined, ldc, workspace, workspace_bytes, act,
                              c->dtype, c->has_gate, stream);
    }
    FusedRows fr;
    fr.pool_u = static_cast<const unsigned char *>(c->b.up_pool);
    fr.act_u = static_cast<unsigned char *>(c->b.up_active);
    fr.pool_d = static_cast<const unsigned char *>(c->b.downT_pool);
    fr.act_d = static_cast<unsigned char *>(c->b.down_active);
    fr.pool_g = c->has_gate ? static_cast<const unsigned char *>(c->b.gate_pool) : fr.pool_u;
    fr.act_g = c->has_gate ? static_cast<unsigned char *>(c->b.gate_active) : fr.act_u;
    fr.row_bytes = row_bytes;
    fr.has_gate = c->has_gate ? 1 : 0;
    float *partials = static_cast<float *>(workspace);
    if (n_hint < 0) n_hint = seen_count(c);
    const int hint = (int)(n_hint > c->I ? c->I : n_hint);
    {
        ProfScope ps(ST_K_CACHE_UPDATE_DECODE, s);
        auto launch = [&](auto kern, auto *xt, auto *ct) -> int {
            const int arc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), 148 * 1024);
            if (arc != ST_OK) return arc;
            // (blocks, log2 of the thread-group size, gated or not, rows of x: one argument, see the kernel)
            const int launch_word = G | (gs_log2 << 16) | (fr.has_gate << 20) | ((int)B << 24);
            ST_LAUNCH(ps, kern, dim3(G), dim3(TPB), lds, s, mask, c->b.cur_mask, c->b.indices, c->b.state, I,
                      launch_word, xt, H, hint, ct, (long)ldc, partials, act, (int)plan_bytes, c->host, fr);
            return ST_OK;
        };
        int rc;
        // Rows a thread group keeps in flight (it does not change which rows a group sums, or in which order): six;
        // seven where the caller's guess of the count gives a group 7, 13 or 14 rows (one batch less); three when
        // a group has at most three rows; two rows of x: six when that is one batch, else five.
        const int rpg = ((hint + G - 1) / G + ngrp - 1) / ngrp;   // rows per thread group on the caller's guess
        const bool seven = c->dtype != ST_F32 && B == 1 && (rpg + 6) / 7 < (rpg + 5) / 6;
#define ST_SPARSE_SPEC(TYPE, ROWS, NBX, SPEC)                                                                       \
    rc = aligned ? I <= 8 * TPB ? launch(cache_sparse_decode_kernel<TYPE, ROWS, TPB, NBX, 1, SPEC, true>, xt, ct)   \
                                : launch(cache_sparse_decode_kernel<TYPE, ROWS, TPB, NBX, 2, SPEC, true>, xt, ct)   \
         : I <= 8 * TPB         ? launch(cache_sparse_decode_kernel<TYPE, ROWS, TPB, NBX, 1, SPEC, false>, xt, ct)  \
                                : launch(cache_sparse_decode_kernel<TYPE, ROWS, TPB, NBX, 2, SPEC, false>, xt, ct)
#define ST_SPARSE_NW(TYPE, ROWS, NBX) ST_SPARSE_SPEC(TYPE, ROWS, NBX, ROWS / 2)
// (three rows in flight: two of them ahead of the plan -- with so few rows per block nearly everything waits for the plan
// otherwise; measured +4 % tok/s on the 10 %-active workloads against one, and against all three)
#define ST_SPARSE_NW3(TYPE) ST_SPARSE_SPEC(TYPE, 3, 1, 2)
#define ST_SPARSE_LAUNCH(TYPE)                                                                                      \
    do {                                                                                                            \
        const TYPE *xt = static_cast<const TYPE *>(x);                                                              \
        TYPE *ct = static_cast<TYPE *>(combined);                                                                   \
        if (B == 2 && rpg <= 6) ST_SPARSE_NW(TYPE, 6, 2);                                                           \
        else if (B == 2) ST_SPARSE_NW(TYPE, 5, 2);                                                                  \
        else if (seven) ST_SPARSE_NW(TYPE, 7, 1);                                                                   \
        else if (rpg >= 1 && rpg <= 3) ST_SPARSE_NW3(TYPE);                                                         \
        else ST_SPARSE_NW(TYPE, DecodeRows<TYPE>::value, 1);                                                        \
    } while (0)
        if (c->dtype == ST_F32) ST_SPARSE_LAUNCH(float);
        else if (c->dtype == ST_BF16) ST_SPARSE_LAUNCH(bf16_t);
        else ST_SPARSE_LAUNCH(f16_t);
#undef ST_SPARSE_LAUNCH
#undef ST_SPARSE_NW
#undef ST_SPARSE_NW3
#undef ST_SPARSE_SPEC
        if (rc != ST_OK) return rc;
    }
    ST_HIP(hipGetLastError());
    return launch_mlp_reduce(c->dtype, partials, G, NBF, (int)B, H, out, s);
}

extern "C" const volatile int32_t *st_cache_seen_count(const st_cache *c) { return c ? &c->host->count : nullptr; }

// The outcome of an update from the host's copy of the state words.
static int update_outcome(const st_cache *c)
{
    using namespace st;
    if (c->host_state[ST_STATE_FAULT] != 0) {
        set_error("st_cache: the fault word of the state is set; the cache contents are undefined");
        return ST_ERR_HIP;
    }
    if (c->host_state[ST_STATE_STATUS] == ST_ERR_NO_ACTIVE) {
        set_error("No active weights");
        return ST_ERR_NO_ACTIVE;
    }
    return ST_OK;
}

// A wait for what is on its way on `stream`, with the state words behind it in the host's copy and state_out, in two halves.
// A kernel behind the update writes the words to pinned memory: 17.0 us for an update of 400 rows at H 2048, I 8192, fp32,
// from call to return, against 21.8 with a copy of the state to the host and a wait for the stream.  (Words written by
// the update's publishing block itself were there 3.7 us earlier, while other blocks still read the mask and wrote rows.)
static int ask_for_state(st_cache *c, void *stream)
{
    using namespace st;
    if (++c->number == 0) c->number = 1;
    hipLaunchKernelGGL(cache_tell_kernel, dim3(1), dim3(kWave), 0, static_cast<hipStream_t>(stream), c->b.state, c->host, c->number);
    ST_HIP(hipGetLastError());
    return ST_OK;
}

static int await_state(st_cache *c, int32_t *state_out, void *stream)
{
    using namespace st;
    // Bounded: with much work ahead of it on the stream the wait is the stream's.
    const volatile uint64_t *w = c->host->state;
    const auto begun = std::chrono::steady_clock::now();
    for (int spins = 0;; ++spins) {
        bool all = true;
        int32_t v[ST_STATE_WORDS];
        for (int k = 0; k < ST_STATE_WORDS; ++k) {
            const uint64_t x = w[k];
            all = all && (uint32_t)(x >> 32) == c->number;
            v[k] = (int32_t)(uint32_t)x;
        }
        if (all) {
            std::atomic_thread_fence(std::memory_order_acquire);
            memcpy(c->host_state, v, sizeof v);
            if (state_out) memcpy(state_out, v, sizeof v);
            return update_outcome(c);
        }
        __builtin_ia32_pause();
        if ((spins & 63) == 63 && std::chrono::steady_clock::now() - begun > std::chrono::milliseconds(1)) break;
    }
    return st_cache_sync_state(c, state_out, stream);
}

static int wait_for_state(st_cache *c, int32_t *state_out, void *stream)
{
    const int rc = ask_for_state(c, stream);
    return rc != ST_OK ? rc : await_state(c, state_out, stream);
}

extern "C" int st_cache_update_sync(st_cache *c, const uint8_t *mask, int32_t *state_out, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && mask, "st_cache_update_sync: null pointer");
    const int rc = st_cache_update_async(c, mask, stream);
    return rc != ST_OK ? rc : wait_for_state(c, state_out, stream);
}

extern "C" int st_cache_load_weights_begin(st_cache *c, const void *gate, const void *up, const void *down,
                                           const uint8_t *mask, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && up && down && mask, "st_cache_load_weights_masked: null pointer");
    ST_REQUIRE(!c->has_gate || gate, "st_cache_load_weights_masked: gated cache needs gate weights");
    const int rc = launch_build(c, gate, up, down, mask, static_cast<hipStream_t>(stream));
    return rc != ST_OK ? rc : ask_for_state(c, stream);
}

extern "C" int st_cache_load_weights_end(st_cache *c, int32_t *state_out, void *stream)
{
    using namespace st;
    ST_REQUIRE(c, "st_cache_load_weights_end: null handle");
    return await_state(c, state_out, stream);
}

extern "C" int st_cache_load_weights_masked(st_cache *c, const void *gate, const void *up, const void *down,
                                            const uint8_t *mask, int32_t *state_out, void *stream)
{
    const int rc = st_cache_load_weights_begin(c, gate, up, down, mask, stream);
    return rc != ST_OK ? rc : await_state(c, state_out, stream);
}

extern "C" int st_cache_sync_state(st_cache *c, int32_t *state_out, void *stream)
{
    using namespace st;
    ST_REQUIRE(c, "st_cache_sync_state: null handle");
    hipStream_t s = static_cast<hipStream_t>(stream);
    ST_HIP(hipMemcpyAsync(c->host_state, c->b.state, ST_STATE_WORDS * sizeof(int32_t), hipMemcpyDeviceToHost, s));
    ST_HIP(hipStreamSynchronize(s));
    if (state_out)
        for (int i = 0; i < ST_STATE_WORDS; ++i) state_out[i] = c->host_state[i];
    return update_outcome(c);
}

extern "C" int st_cache_materialize_concat(st_cache *c, void *dst, int64_t n, void *stream)
{
    using namespace st;
    ST_REQUIRE(c && dst, "st_cache_materialize_concat: null pointer");
    ST_REQUIRE(n >= 1 && n <= c->I, "st_cache_materialize_concat: n=%lld out of range", (long long)n);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t blk = (size_t)n * c->H * c->esz;
    unsigned char *d = static_cast<unsigned char *>(dst);
    if (c->has_gate) {
        ST_HIP(hipMemcpyAsync(d, c->b.gate_active, blk, hipMemcpyDeviceToDevice, s));
        d += blk;
    }
    ST_HIP(hipMemcpyAsync(d, c->b.up_active, blk, hipMemcpyDeviceToDevice, s));
    return ST_OK;
}
