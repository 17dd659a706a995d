// spz_search.hip -- the IDA* hot path on CDNA4 (gfx950).
//
// One search = many instances (a batch of boards), each running its own
// threshold sequence h0, h0+2, ... (src/24puzzle.cc:146-152).  An iteration
// of an instance is:
//   * its top tree (root split, src/15puzzle_block_parallel.cu:150-187, done
//     once per solve by k_begin, or by k_split_level where duplicates are
//     pruned or the frontier is very large): the count of every top node whose
//     f fits the threshold is added from an f-histogram, and
//   * one work item per frontier node whose f fits the threshold; items are
//     searched depth-first by single lanes (k_round).  While a round runs, a
//     wave's idle lanes take the shallowest open nodes of its busy ones, and
//     waves without work are fed by others through mailboxes (the reference
//     shares only inside a block, src_horie/idas_dynamic.cu:199-247); the
//     queue holds frontier nodes and what overflows a stack.
// The count of iteration L is  sum_{top u: F(u)<=L} gen(u)
//                            + sum_{frontier v: F(v)<=L} subtree_count(v),
// where gen(u) counts every in-bounds non-reverse child of an expanded node
// before its f-test (src/24puzzle.cc:119-131) and F(u) is the largest f on
// u's path from the root.  IDA* expands a node in iteration L iff every node
// on its path has f <= L, i.e. F <= L; for Manhattan (consistent) F is the
// node's own f, the PDB max is not consistent, hence the path maximum.  So
// the counts are exact whatever the schedule.  With lookahead an instance
// runs its next iteration beside the current one; each keeps its own count
// and k_restart resolves them in order (k_spec, k_restart).
#include <hip/hip_ext.h>

#include "spz_board.h"

namespace spz {

// stack levels a lane may pop in one step: a wave runs the pop loop as often
// as its deepest popping lane needs, and each pop is a chain of dependent LDS
// reads, so more pops per step lengthen every lane's step (measured on
// MI355X: 2 beats 1, 3, 4, 6, 8 and 12 for both heuristics)
constexpr int kPops = 2;
// sibling-value cache of the PDB search: per lane, the deepest kSibLevels
// stack levels (ring, tagged with the level); see k_round
constexpr int kSibLevels = 8;
// steps between two looks of a wave at its idle lanes
constexpr int kShareSteps = 8;
// idle lanes of a wave that make sharing worth its cost
constexpr int kShareMin = 4;
// a node given to another lane of the wave, or to another wave, lies at least
// this many levels above the giver's own
constexpr int kGiveLevels = 2;
constexpr int kFeedLevels = 4;
// naps of a wave waiting for work in one round at most (a round has its own
// end; this bounds the wait whatever happens)
constexpr int kMaxNaps = 1 << 16;
// blocks of steps of a wave that starts late
constexpr int kLateBlocks = 64;



__device__ __forceinline__ uint64_t lanemask_lt() {
    uint32_t lo = __builtin_amdgcn_mbcnt_lo(~0u, 0u);
    uint32_t n = __builtin_amdgcn_mbcnt_hi(~0u, lo);
    return n == 0 ? 0ull : (~0ull >> (64 - n));
}

__device__ __forceinline__ unsigned long long shfl_u64(unsigned long long v, int src) {
    uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
    lo = __shfl(lo, src);
    hi = __shfl(hi, src);
    return ((unsigned long long)hi << 32) | lo;
}

__device__ __forceinline__ unsigned long long shfl_xor_u64(unsigned long long v, int off) {
    const uint32_t lo = __shfl_xor((uint32_t)v, off), hi = __shfl_xor((uint32_t)(v >> 32), off);
    return ((unsigned long long)hi << 32) | lo;
}

// Words that waves of other dies read or write while a round runs.  Relaxed
// agent-scope accesses: no cache is written back or invalidated, which would
// also drop the pattern-database lines.
template <class T> __device__ __forceinline__ T ld_agent(const T *a) {
    return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void st_agent(T *a, T v) {
    __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// what the wave stored so far has arrived before what it stores next
__device__ __forceinline__ void arrival_fence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0); // all counters: vector stores and atomics included
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ unsigned uniform(unsigned v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ unsigned long long uniform(unsigned long long v) {
    return ((unsigned long long)uniform((unsigned)(v >> 32)) << 32) | uniform((unsigned)v);
}

// The waves of a round form kGroups groups by workgroup number (workgroups go
// to the 8 dies in turn, so a group is a die's), each with words of its own
// for what every wave changes.
__device__ __forceinline__ unsigned group_of(unsigned block) { return block & (kGroups - 1); }
// Waves waiting for work are on kLists lists, by workgroup number too (so the
// waves of a list are a die's): a list's word is changed by compare-and-swap,
// of which one in the time of a look and a swap succeeds, a microsecond, and
// 8192 waves on 8 lists could not be fed at that rate.
__device__ __forceinline__ unsigned list_of(unsigned block) { return block & (kLists - 1); }
__device__ __forceinline__ unsigned list_waves(const KParams &p, unsigned x) {
    return ((unsigned)p.n_blocks + kLists - 1 - x) / kLists * (unsigned)p.block_waves;
}
// a list's waves: pushed onto it (high half) and not taken off it by a wave
// with work to give (low half)
__device__ __forceinline__ unsigned waiting(unsigned long long w) { return (unsigned)(w >> 32) - (unsigned)w; }
__device__ __forceinline__ unsigned wave_sum(unsigned n) {
    for (int off = 1; off < 64; off <<= 1) n += __shfl_xor(n, off);
    return uniform(n);
}
// both by a whole wave
__device__ __forceinline__ unsigned idle_waves(const KParams &p) {
    return wave_sum(waiting(ld_agent(&p.q_ctl[kQList + (threadIdx.x & 63u) * kLine])));
}
__device__ __forceinline__ unsigned started_waves(const KParams &p) {
    const unsigned lane = threadIdx.x & 63u;
    return wave_sum(lane < (unsigned)kGroups ? (unsigned)ld_agent(&p.q_ctl[kQStart + lane * kLine]) : 0u);
}

// Items and waves of slot isl not finished, and its node count: each group
// keeps its part (a group's part alone may be negative)
__device__ __forceinline__ unsigned slot_pend(const KParams &p, int isl) {
    unsigned n = 0;
    for (int x = 0; x < kGroups; ++x) n += p.pend[x * p.gstride + isl];
    return n;
}
__device__ __forceinline__ unsigned long long slot_count(const KParams &p, int isl) {
    unsigned long long n = 0;
    for (int x = 0; x < kGroups; ++x) n += p.cnt[x * p.gstride + isl];
    return n;
}

// A goal in slot isl makes a newer iteration in the other slot unnecessary
// (this one is the instance's last): mark that slot dead.  Lanes drop items
// of a dead slot unsearched.
__device__ __forceinline__ void kill_newer(const KParams &p, int isl) {
    const int o = isl ^ 1;
    if (p.itn[o] > p.itn[isl]) p.dead[o] = 1;
}

// The work queue is two rings of equal size: ring 0 holds work of the
// instances' current iterations, ring 1 that of lookahead iterations; idle
// lanes take from ring 0 first.  Slot of position pos of ring r:
__device__ __forceinline__ size_t q_slot(const KParams &p, int r, unsigned long long pos) {
    return (size_t)r * (size_t)(p.qmask + 1ull) + (size_t)(pos & p.qmask);
}

// Does the slot index isl belong to a lookahead iteration (newer than the
// instance's current one)?  Its work then goes to ring 1.
__device__ __forceinline__ int ahead_ring(const KParams &p, int isl) {
    return (p.lookahead && p.itn[isl] > p.it[isl >> 1]) ? 1 : 0;
}

// Append one item.  pos is a reserved position of ring r.
template <int W, int HEUR, class BD>
__device__ __forceinline__ void put_item(const KParams &p, int r, unsigned long long pos, const Pos<W, HEUR, BD> &s,
                                         int g, int prev, int inst, uint32_t origin) {
    Item it;
    s.bd.pack(it.b);
    it.meta = meta_pack(s.cell(), g, s.hs.h, prev);
    it.inst = (uint32_t)inst;
    it.x0 = 0;
    it.x1 = origin;
    p.q[q_slot(p, r, pos)] = it;
}

// Position i of a ring belongs to group i % kGroups, whose head word holds its
// next position not taken.  Reserve k positions at the tail of ring r; a tail
// more than the ring's capacity past the oldest item not taken would
// overwrite it, so that sets the error word (ctl[3]) and the host fails the
// solve with SPZ_E_CAPACITY rather than return counts from a corrupt queue.
template <int Unroll>
__device__ __forceinline__ unsigned long long q_reserve(const KParams &p, int r, unsigned long long k) {
    unsigned long long *c = p.q_ctl + kQTail + r * kQRing;
    const unsigned long long pos = atomicAdd(&c[0], k);
    unsigned long long oldest = c[1]; // the limit: taken positions end there
#pragma unroll Unroll
    for (int x = 0; x < kGroups; ++x) {
        const unsigned long long h = ld_agent(&p.q_ctl[kQHead + r * kQRing + x * kLine]);
        oldest = h < oldest ? h : oldest;
    }
    if (pos + k - oldest > p.qmask + 1ull) atomicOr(&p.ctl[3], 1u);
    return pos;
}

// Solution paths: move i of a path sits in bits 2(i%16) of word i/16; a
// path's words are `stride` apart (1 in the queue and solution arrays, the
// lane count in the per-lane array).  Bits past a path's length are zero, so
// a copied prefix needs no clearing.  The loops stay rolled: this code runs
// rarely, and unrolled it would hold a whole path in registers and cost the
// search kernel occupancy.
// Paths are addressed as base[off + word * stride] with 32-bit offsets
// (every path array holds fewer than 2^32 words), so the base stays scalar.
__device__ __forceinline__ void path_put(uint32_t *base, uint32_t off, uint32_t stride, int i, int d) {
    if (i >= kPathMax) return; // too long to record; no goal through it is recorded
    uint32_t &x = base[off + (uint32_t)(i >> 4) * stride];
    const int sh = 2 * (i & 15);
    x = (x & ~(3u << sh)) | ((uint32_t)d << sh);
}
__device__ __forceinline__ void path_copy(const uint32_t *sb, uint32_t so, uint32_t ss, uint32_t *db, uint32_t dof,
                                          uint32_t dstr) {
#pragma unroll 1
    for (uint32_t k = 0; k < (uint32_t)kPathWords; ++k) db[dof + k * dstr] = sb[so + k * ss];
}
// the same in a mail, which a wave of another die reads
__device__ __forceinline__ void path_put_agent(uint32_t *path, int i, int d) {
    if (i >= kPathMax) return;
    uint32_t *x = &path[i >> 4];
    const int sh = 2 * (i & 15);
    st_agent(x, (ld_agent(x) & ~(3u << sh)) | ((uint32_t)d << sh));
}
__device__ __forceinline__ void path_from_u64(unsigned long long v, uint32_t *db, uint32_t dof) {
    db[dof] = (uint32_t)v;
    db[dof + 1] = (uint32_t)(v >> 32);
#pragma unroll 1
    for (uint32_t k = 2; k < (uint32_t)kPathWords; ++k) db[dof + k] = 0u;
}

template <int W, int HEUR, class BD>
__device__ __forceinline__ void pos_from_item(Pos<W, HEUR, BD> &s, const uint32_t (&b)[4], uint32_t meta,
                                              const PdbCtx &P) {
    s.bd.unpack(b);
    s.set_cell(meta_blank(meta));
    init_heur<W, HEUR>(s, P, meta);
}

// The kernel's arguments, read again where they are used: held from the
// kernel's start they would not fit the scalar registers and be spilled to
// vector ones, which the search needs.
__device__ __forceinline__ const KParams &params_again() {
    auto *a = (const __attribute__((address_space(4))) KParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return *(const KParams *)a;
}

// ---------------------------------------------------------------------------
// k_round: a wave is a team of 64 depth-first search engines, one a lane.  A
// round runs wave-uniform steps; each step a lane pops up to kPops stack
// levels or makes one move down, and expands the node it stands on.  Every
// kShareSteps steps the wave settles what the steps left (items done, goals,
// full stacks) and evens out its work: its idle lanes take the shallowest
// open nodes of its busy ones, by lane exchange.  A wave without any work
// takes items of the queue, one where there are fewer items than waves, and
// where there are none it waits to be fed by a wave with work, through its
// mailbox.  The round ends after its time or steps, when every wave waits, or
// when so many wait that a new round is worth its cost (turn_ticks).  Busy
// lanes keep their state across rounds in the c_* context arrays.
//
// What bounds the sharing is that atomics on one address are served one after
// another, 12 ns each on MI355X whatever the die (83 M/s; loads of a line that
// atomics change are no faster, loads of an unchanged line 16 G/s).  A single
// search has one node count and one count of pending items, so both are kept
// by the wave: it counts as one pending unit of an instance however many of
// its lanes search it, and adds their node counts once, when that ends.
//
// The stack holds one byte per level (PDB: two): the move taken from that
// level (2 bits) and the moves still to try there (4-bit mask of children
// that passed the f-test).
// The 15-puzzle kernel is held to 64 VGPRs (8 waves per SIMD: its LDS use is
// small); the 24-puzzle kernels are bounded by their LDS (stack and boards)
// at 3 waves per SIMD.  PROF: with the lane-state counters (SPZ_PROFILE).
template <int W, int HEUR, bool PROF>
__global__ void __launch_bounds__(256, (W == 4 ? 8 : 3)) k_round(KParams p, const PdbGeo *geo_g) {
    if (p.ctl[1] == 0) return; // every instance is done: a round enqueued in advance
    // every wave of the grid starts within microseconds of the others
    const long long t_start = wall_clock64();
    const int MAXD = p.maxd;
    extern __shared__ uint8_t lds[];
    __shared__ PdbGeo geo_s;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const int gl = blockIdx.x * blockDim.x + threadIdx.x;
    const int NL = p.n_lanes;
    using SE = StackEntry<HEUR>;
    using ST = typename SE::T;
    // level k at stk[k * sstride]; an LDS-qualified pointer keeps the
    // address arithmetic in 32 bits
    __attribute__((address_space(3))) ST *stk = (__attribute__((address_space(3))) ST *)lds + wave * 64 + lane;
    ST *cstk = (ST *)p.c_stack;
    const int sstride = nw * 64;

    PdbCtx P{&geo_s, p.pdb};
    if constexpr (HEUR == 1) {
        const uint32_t *src = (const uint32_t *)geo_g;
        uint32_t *dst = (uint32_t *)&geo_s;
        for (int i = threadIdx.x; i < (int)(sizeof(PdbGeo) / 4); i += blockDim.x) dst[i] = src[i];
        __syncthreads();
    }

    const unsigned grp = group_of(blockIdx.x);
    const int wave_id = gl >> 6;
    if (lane == 0) atomicAdd(&p.q_ctl[kQStart + grp * kLine], 1ull);
    // a wave that starts when the round is already to end (the device did not
    // hold all workgroups at once) runs a while all the same
    const int least = uniform(ld_agent(p.stop)) ? kLateBlocks : 1;
    // per ring the groups whose part of the queue the wave has seen empty
    // (it stays empty for the round: heads only grow)
    unsigned empty0 = 0, empty1 = p.lookahead ? 0u : (1u << kGroups) - 1u;
    const int take_most = (int)p.ctl[4];
    int steps_left = (int)p.ctl[5];
    const int mode = p.mode;
    const unsigned n_waves = (unsigned)NL >> 6;

    const uint32_t stw = p.c_st[gl];
    int st = (int)(stw & 0xff);
    int sp = (int)(stw >> 8);
    // stack levels, then (width 5) the lanes' boards
    Pos<W, HEUR, typename HotBoard<W, HEUR>::T> s;
    // Sibling-value cache (PDB): when a lane enters the first passing child
    // of a node with at most two more, the values its f-test read for them
    // go into slot level % kSibLevels (tag = level in bits 24-31, 6+6 bits
    // per sibling); moving into such a sibling later then reads no table.
    // An entry overwritten by a deeper level (or from an earlier round: LDS
    // does not persist) fails its tag and the move reads the tables as
    // before.
    uint32_t *sibc = nullptr;
    if constexpr (HEUR == 1) {
        sibc = (uint32_t *)(lds + (size_t)MAXD * sstride * sizeof(ST) + (size_t)blockDim.x * kLdsBoardBytes) +
               threadIdx.x;
#pragma unroll
        for (int k = 0; k < kSibLevels; ++k) sibc[k * blockDim.x] = 0xffffffffu;
    }
    if constexpr (W == 5) {
        s.bd.p = lds + (size_t)MAXD * sstride * sizeof(ST) + threadIdx.x * kLdsBoardBytes;
    } else {
        s.bd.unpack({0u, 0u, 0u, 0u});
    }
    s.set_cell(0);
    s.hs.h = 0;
    // inst is the item's slot index (instance * 2 + iteration slot); an idle
    // lane keeps the one its node count belongs to
    int g = 0, prev = DIR_NONE, inst = 0, L = 0;
    uint32_t cnt = 0;

    // a saved GOAL is a goal node recorded already, to be expanded
    bool goal_seen = st == ST_GOAL;
    if (goal_seen) st = ST_FRESH;
    if (st == ST_FRESH || st == ST_POP) {
        uint32_t b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) b[k] = p.c_rows[k * NL + gl];
        s.bd.unpack(b);
        uint32_t m = p.c_meta[gl];
        inst = (int)p.c_inst[gl];
        cnt = p.c_cnt[gl];
        s.set_cell(meta_blank(m));
        g = meta_g(m);
        prev = meta_prev(m);
        s.hs.h = meta_h(m);
        if constexpr (HEUR == 1) {
            s.hs.i0 = p.c_pdb[0 * NL + gl];
            s.hs.i1 = p.c_pdb[1 * NL + gl];
            s.hs.i2 = p.c_pdb[2 * NL + gl];
            s.hs.i3 = p.c_pdb[3 * NL + gl];
            s.hs.j0 = p.c_pdb[4 * NL + gl];
            s.hs.j1 = p.c_pdb[5 * NL + gl];
            s.hs.j2 = p.c_pdb[6 * NL + gl];
            s.hs.j3 = p.c_pdb[7 * NL + gl];
            s.hs.v0 = p.c_pdb[8 * NL + gl];
            s.hs.v1 = p.c_pdb[9 * NL + gl];
            uint32_t v0 = s.hs.v0, v1 = s.hs.v1;
            s.hs.A = (int)((v0 & 0xff) + ((v0 >> 8) & 0xff) + ((v0 >> 16) & 0xff) + (v0 >> 24));
            s.hs.B = (int)((v1 & 0xff) + ((v1 >> 8) & 0xff) + ((v1 >> 16) & 0xff) + (v1 >> 24));
        }
        L = p.L[inst];
        // dropped: unwinds and finishes next step
        if (p.lookahead && p.dead[inst]) sp = 0, st = ST_POP, goal_seen = false;
        // eight levels' loads in flight at once (the tail re-reads the last one)
#pragma unroll 1
        for (int k = 0; k < sp; k += 8) {
            ST e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = cstk[(size_t)min(k + j, sp - 1) * NL + gl];
#pragma unroll
            for (int j = 0; j < 8; ++j) stk[min(k + j, sp - 1) * sstride] = e[j];
        }
    } else {
        st = ST_IDLE;
    }

    // the lane's node count stays with the instance it was counted for: on a
    // change of instance it is added there
    auto relabel = [&](int to) {
        const KParams &p = params_again();
        if (cnt && inst != to) {
            atomicAdd(&p.cnt[grp * p.gstride + inst], (unsigned long long)cnt);
            cnt = 0;
        }
        inst = to;
    };

    // an item becomes the lane's; the PDB lookups of its board are computed
    // for all lanes that start one together (init)
    bool init = false;
    auto start_item = [&](const Item &it) {
        const KParams &p = params_again();
        s.bd.unpack(it.b);
        s.set_cell(meta_blank(it.meta));
        s.hs.h = meta_h(it.meta);
        init = true;
        relabel((int)it.inst);
        if (p.want_load) p.c_origin[gl] = it.x1; // read when the item ends or is given away
        g = meta_g(it.meta);
        prev = meta_prev(it.meta);
        L = p.L[inst];
        sp = 0;
        goal_seen = false;
        st = ST_FRESH;
        if (mode == 1 && p.found[inst] != kNoGoal) st = ST_POP; // first-solution: abandon
        if (p.lookahead && p.dead[inst]) st = ST_POP;
    };

    // move down into child d (stack level sl, R = passing children still to
    // visit there); for the PDB the child's values are known or read
    uint32_t dpass = 0, dval = 0, dval2 = 0; // pending descent (ST_DESC)
    auto enter_child = [&](int d, uint32_t Rr, int sl, bool kn, uint32_t kvv) {
        uint32_t ov = 0;
        if constexpr (HEUR == 1)
            ov = move_pdb<W>(s, d, P, kn, kvv);
        else
            ov = move_md(s, d);
        stk[sl * sstride] = SE::make(d, Rr, ov);
        sp = sl + 1;
        ++g;
        prev = d;
        st = ST_FRESH;
    };
    // path of a new queue item: the item root's path, the moves of stack
    // levels 0..nst-1, then move last_d
    auto item_path = [&](int r, unsigned long long qpos, int nst, int last_d) {
        const KParams &p = params_again();
        const uint32_t qo = (uint32_t)q_slot(p, r, qpos) * kPathWords;
        path_copy(p.c_ipath, (uint32_t)gl, (uint32_t)NL, p.qpath, qo, 1);
        const int gr = g - sp; // depth of the item's root
        for (int k = 0; k < nst; ++k) path_put(p.qpath, qo, 1, gr + k, SE::dir(stk[k * sstride]));
        path_put(p.qpath, qo, 1, gr + nst, last_d);
    };
    // moves that give work away: the board, the blank and (Manhattan) h; for
    // the PDB the board alone, as the lane that takes the node computes its
    // lookups from the board
    auto step_down = [&](int d) -> uint32_t {
        if constexpr (HEUR == 1) {
            move_board_only(s, d);
            return 0u;
        } else {
            return move_md(s, d);
        }
    };
    auto step_back = [&](int d, uint32_t nearer) {
        if constexpr (HEUR == 1)
            move_board_only(s, 3 - d);
        else
            unmove_md(s, d, nearer);
    };
    // back up to the node whose child the lane's path enters at level lev
    auto go_back = [&](int lev) {
#pragma unroll 1
        for (int k = sp - 1; k >= lev; --k) {
            const uint32_t e = stk[k * sstride];
            step_back(SE::dir(e), SE::vals(e));
        }
    };
    // where the lane stands, kept while it goes back up its path: board, blank
    // and h (the PDB lookups do not move with step_back and step_down)
    struct Here {
        uint64_t b;
        uint32_t w[kLdsBoardBytes / 4];
        int c, h;
    };
    auto save_pos = [&](Here &o) {
        if constexpr (W == 4) {
            o.b = s.bd.b;
        } else {
#pragma unroll
            for (int k = 0; k < kLdsBoardBytes / 4; ++k) o.w[k] = ((const uint32_t *)s.bd.p)[k];
        }
        o.c = s.cell();
        if constexpr (HEUR == 0) o.h = s.hs.h;
    };
    auto load_pos = [&](const Here &o) {
        if constexpr (W == 4) {
            s.bd.b = o.b;
        } else {
#pragma unroll
            for (int k = 0; k < kLdsBoardBytes / 4; ++k) ((uint32_t *)s.bd.p)[k] = o.w[k];
        }
        s.set_cell(o.c);
        if constexpr (HEUR == 0) s.hs.h = o.h;
    };
    // the child in direction d of the node the lane stands on, at depth
    // `depth`, to position pos of ring r; the lane stays where it is
    auto queue_child = [&](int r, unsigned long long pos, int d, int depth) {
        const KParams &p = params_again();
        const uint32_t nearer = step_down(d);
        put_item<W, HEUR>(p, r, pos, s, depth, d, inst, p.want_load ? p.c_origin[gl] : 0u);
        step_back(d, nearer);
    };
    // a node of level k is given away: the level's cached sibling values no
    // longer match the children left there
    auto void_siblings = [&](int k) {
        if constexpr (HEUR == 1) {
            uint32_t &c = sibc[(k % kSibLevels) * blockDim.x];
            if ((c >> 24) == (uint32_t)k) c = 0xffffffffu;
        }
    };
    // the shallowest level with an open node, at least `above` levels above the
    // node the lane stands on (a smaller subtree is searched sooner than it
    // is handed over); 255: none
    auto give_level = [&](int above) -> int {
        int lev = 255;
        if (searching(st))
            for (int k = 0; k + above <= sp; ++k)
                if (SE::rest(stk[k * sstride])) {
                    lev = k;
                    break;
                }
        return lev;
    };
    // of the lanes in `from`, the `n` with the smallest 8-bit keys
    auto smallest = [&](uint64_t from, int key, int n) -> uint64_t {
        uint64_t chosen = 0;
#pragma unroll 1
        for (int bit = 7; bit >= 0; --bit) {
            const uint64_t zeros = __ballot(((key >> bit) & 1) == 0) & from;
            const int nz = __popcll(zeros);
            if (nz >= n) {
                from = zeros;
            } else {
                chosen |= zeros;
                n -= nz;
                from &= ~zeros;
            }
        }
        // equal keys: the lowest lanes
        const bool in = ((from >> lane) & 1ull) && __popcll(from & lanemask_lt()) < n;
        return chosen | __ballot(in);
    };

    // What the steps leave to be done between two blocks of them, so that
    // the steps hold no atomics and none of this code.
    auto settle = [&]() {
        const KParams &p = params_again();
        if (st == ST_GOAL) {
            atomicMin(&p.found[inst], g);
            if (p.lookahead) kill_newer(p, inst);
            // the first goal of the slot's iteration records its path (the
            // first iteration with a goal has threshold = optimum, and every
            // goal it finds has that depth)
            if (p.sol && g <= kPathMax && atomicCAS(&p.sol_len[inst], -1, g) == -1) {
                const uint32_t so = (uint32_t)inst * kPathWords;
                path_copy(p.c_ipath, (uint32_t)gl, (uint32_t)NL, p.sol, so, 1);
                for (int k = 0; k < sp; ++k) path_put(p.sol, so, 1, g - sp + k, SE::dir(stk[k * sstride]));
            }
            goal_seen = mode != 1;
            st = mode == 1 ? ST_POP : ST_FRESH;
        }
        if (st == ST_FULL) {
            // stack full: the passing children become queue items
            const int k = __builtin_popcount(dpass);
            atomicAdd(&p.pend[grp * p.gstride + inst], (unsigned)k);
            atomicAdd(&p.ctl[8], (unsigned)k);
            const int r = ahead_ring(p, inst);
            unsigned long long pos = q_reserve<1>(p, r, (unsigned long long)k);
#pragma unroll 1
            for (uint32_t pass = dpass; pass; pass &= pass - 1) {
                const int d = __builtin_ctz(pass);
                if (p.qpath) item_path(r, pos, sp, d);
                queue_child(r, pos++, d, g + 1);
            }
            st = ST_POP;
        }
        // items done: the wave's last one of an instance ends its pending
        // unit and adds the lanes' counts (read by the next kernel, so
        // nothing orders the two)
        if (p.want_load && st == ST_DONE && cnt) {
            atomicAdd(&p.cnt[grp * p.gstride + inst], (unsigned long long)cnt);
            atomicAdd(&p.load[(size_t)(inst >> 1) * p.capl + p.c_origin[gl]], (unsigned long long)cnt);
            cnt = 0;
        }
        uint64_t todo = __ballot(st == ST_DONE);
        while (todo) {
            const int lead = __ffsll((long long)todo) - 1;
            const int i = __builtin_amdgcn_readlane(inst, lead);
            const bool mine = inst == i;
            todo &= ~__ballot(mine);
            if (!__ballot(mine && st != ST_DONE && st != ST_IDLE)) {
                unsigned long long c = mine ? cnt : 0u;
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) c += shfl_xor_u64(c, off);
                if (mine) cnt = 0;
                if (lane == lead) {
                    if (c) atomicAdd(&p.cnt[grp * p.gstride + i], c);
                    atomicSub(&p.pend[grp * p.gstride + i], 1u);
                }
            }
        }
        if (st == ST_DONE) st = ST_IDLE;
    };

    // idle lanes get up to `most` queue items, of ring 0 first and of the
    // wave's own group first
    auto take_items = [&](int most, Item &it, bool &have) {
        const KParams &p = params_again();
#pragma unroll 1
        for (int t = 0; t < 2 * kGroups && most > 0; ++t) {
            const int r = t / kGroups;
            const unsigned x = (grp + t) & (kGroups - 1);
            if (((r ? empty1 : empty0) >> x) & 1u) continue;
            unsigned long long *c = p.q_ctl + kQHead + r * kQRing + x * kLine;
            const unsigned long long lim = p.q_ctl[kQTail + r * kQRing + 1];
            const uint64_t need = __ballot(st == ST_IDLE && !have);
            const int n = min(__popcll(need), most);
            if (n <= 0) break;
            const int leader = __ffsll((long long)need) - 1;
            unsigned long long base = 0;
            if (lane == leader) {
                base = ld_agent(c);
                if (base < lim) base = atomicAdd(c, (unsigned long long)n * kGroups);
            }
            base = shfl_u64(base, leader);
            const int rank = __popcll(need & lanemask_lt());
            const unsigned long long my = base + (unsigned long long)rank * kGroups;
            const bool took = st == ST_IDLE && !have && rank < n && my < lim;
            if (took) {
                it = p.q[q_slot(p, r, my)];
                have = true;
                if (p.qpath)
                    path_copy(p.qpath, (uint32_t)q_slot(p, r, my) * kPathWords, 1, p.c_ipath, (uint32_t)gl,
                              (uint32_t)NL);
            }
            if (base + (unsigned long long)n * kGroups >= lim) (r ? empty1 : empty0) |= 1u << x;
            // an item's pending unit becomes the wave's; more than one of an
            // instance are one
            uint64_t todo = __ballot(took);
            most -= __popcll(todo);
            while (todo) {
                const int lead = __ffsll((long long)todo) - 1;
                const int i = __builtin_amdgcn_readlane((int)it.inst, lead);
                const uint64_t got = __ballot(took && (int)it.inst == i);
                const uint64_t had = __ballot(!took && (have ? (int)it.inst == i : st != ST_IDLE && inst == i));
                todo &= ~got;
                const unsigned drop = (unsigned)__popcll(got) - (had ? 0u : 1u);
                if (drop && lane == lead) atomicSub(&p.pend[grp * p.gstride + i], drop);
            }
        }
    };

    // Inside the wave: each idle lane takes the shallowest open node of one
    // busy lane, by lane exchange (15-puzzle) or from its board in LDS.
    auto share = [&](uint64_t idle_mask) {
        const KParams &p = params_again();
        const int lev = give_level(kGiveLevels);
        const uint64_t donors = __ballot(lev < 255);
        if (!donors) return;
        const int n = min(__popcll(donors), __popcll(idle_mask));
        const uint64_t giving = smallest(donors, lev < 255 ? min(g - sp + lev, 255) : 255, n);
        const bool give = (giving >> lane) & 1ull;
        // the n-th giver hands to the n-th idle lane: givers push their lane
        // number to lane n, from where the takers read it
        const int grank = __popcll(giving & lanemask_lt()), trank = __popcll(idle_mask & lanemask_lt());
        const int slot = give ? grank : 63 - __popcll(~giving & lanemask_lt());
        const int at_rank = __builtin_amdgcn_ds_permute(slot << 2, lane);
        const int src = __shfl(at_rank, trank & 63);
        const bool take = ((idle_mask >> lane) & 1ull) && trank < n;
        // a giver goes back to its level and into the child it gives
        int d2 = 0;
        Here here;
        if (give) {
            save_pos(here);
            go_back(lev);
            const uint32_t e = stk[lev * sstride];
            const uint32_t R = SE::rest(e);
            d2 = __builtin_ctz(R);
            stk[lev * sstride] = SE::make(SE::dir(e), R & (R - 1), SE::vals(e));
            void_siblings(lev);
            (void)step_down(d2);
        }
        // the takers' copies.  The boards are read across lanes of the wave:
        // its LDS accesses complete in order, only the compiler must keep
        // them so
        const uint32_t m = meta_pack(s.cell(), give ? g - sp + lev + 1 : 0, s.hs.h, d2);
        const uint32_t m2 = (uint32_t)__shfl((int)m, src);
        const int i2 = __shfl(inst, src), L2 = __shfl(L, src);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (W == 4) {
            const unsigned long long b2 = shfl_u64(s.bd.b, src);
            if (take) s.bd.b = b2;
        } else {
            const uint32_t *from = (const uint32_t *)(s.bd.p + (src - lane) * kLdsBoardBytes);
            uint32_t w7[kLdsBoardBytes / 4];
#pragma unroll
            for (int k = 0; k < kLdsBoardBytes / 4; ++k) w7[k] = from[k];
            if (take) {
#pragma unroll
                for (int k = 0; k < kLdsBoardBytes / 4; ++k) ((uint32_t *)s.bd.p)[k] = w7[k];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int gsp = __shfl(g - sp, src), lev2 = __shfl(lev, src);
        if (take) {
            relabel(i2);
            L = L2;
            g = meta_g(m2);
            prev = meta_prev(m2);
            s.set_cell(meta_blank(m2));
            sp = 0;
            goal_seen = false;
            st = ST_FRESH;
            const int gsrc = gl + src - lane;
            if (p.want_load) p.c_origin[gl] = p.c_origin[gsrc];
            if (p.qpath) {
                // the giver's item path, its moves down to the level, the child
                path_copy(p.c_ipath, (uint32_t)gsrc, (uint32_t)NL, p.c_ipath, (uint32_t)gl, (uint32_t)NL);
                for (int k = 0; k < lev2; ++k)
                    path_put(p.c_ipath, (uint32_t)gl, (uint32_t)NL, gsp + k, SE::dir(stk[k * sstride + src - lane]));
                path_put(p.c_ipath, (uint32_t)gl, (uint32_t)NL, gsp + lev2, prev);
            }
            s.hs.h = meta_h(m2);
            init = true;
        }
        // the giver returns to where it stood
        if (give) load_pos(here);
    };

    // Between waves: a wave without work puts itself on its group's list and
    // waits at its own mailbox, a line nobody else polls; a wave with work
    // that sees somebody waiting takes one wave off the list and writes it
    // half of what it could give, the shallowest open nodes, one a lane.  So
    // the waiting cost no atomics but their entry and exit.  A mail is known
    // by the list position it answers; what a wave finds at its next round's
    // start was sent while it was leaving.
    unsigned ticket = (unsigned)uniform(p.ticket[wave_id]); // list position + 1 waited at, 0: none
    auto read_mail = [&](unsigned n, Item &it, bool &have) {
        const KParams &p = params_again();
        if ((unsigned)lane < n) {
            const unsigned long long *w = (const unsigned long long *)&p.mail[(size_t)wave_id * 64 + lane];
            const unsigned long long a = ld_agent(w), b = W == 5 ? ld_agent(w + 1) : 0ull;
            const unsigned long long m = ld_agent(w + 2), o = ld_agent(w + 3);
            it.b[0] = (uint32_t)a;
            it.b[1] = (uint32_t)(a >> 32);
            it.b[2] = (uint32_t)b;
            it.b[3] = (uint32_t)(b >> 32);
            it.meta = (uint32_t)m;
            it.inst = (uint32_t)(m >> 32);
            it.x0 = 0;
            it.x1 = (uint32_t)(o >> 32);
            have = true;
            if (p.qpath)
#pragma unroll 1
                for (uint32_t k = 0; k < (uint32_t)kPathWords; ++k)
                    p.c_ipath[(size_t)k * NL + gl] = ld_agent(&p.mail_path[((size_t)wave_id * 64 + lane) * kPathWords + k]);
        }
        ticket = 0;
    };
    // items of the mail that comes; 0: the round ends
    auto wait_for_mail = [&]() -> unsigned {
        const KParams &p = params_again();
        const unsigned x = list_of(blockIdx.x);
        unsigned long long *list = p.q_ctl + kQList + x * kLine;
        unsigned long long old = 0;
        if (lane == 0) old = atomicAdd(list, 1ull << 32);
        old = uniform(old);
        const unsigned pos = (unsigned)(old >> 32);
        ticket = pos + 1;
        if (lane == 0)
            st_agent(&p.list[(size_t)x * (p.list_mask + 1) + (pos & p.list_mask)],
                     ((unsigned long long)ticket << 32) | (unsigned)wave_id);
        // the last wave of the last list to run out of work ends the round
        if (waiting(old) + 1 == list_waves(p, x) && idle_waves(p) == (unsigned)NL >> 6) {
            if (lane == 0) st_agent(p.stop, 1u);
            return 0;
        }
#pragma unroll 1
        for (int nap = 0; nap < kMaxNaps; ++nap) {
            const unsigned long long h = uniform(ld_agent(&p.mail_head[(size_t)wave_id * kLine]));
            if ((unsigned)(h >> 32) == ticket) return (unsigned)h;
            if (uniform(ld_agent(p.stop))) return 0;
            // workgroups that have not started yet need the place
            if ((nap & 15) == 15 && started_waves(p) != (unsigned)NL >> 6) return 0;
            if (p.round_ticks && (unsigned long long)(wall_clock64() - t_start) >= p.round_ticks) return 0;
            for (int k = 0; k <= (nap < 3 ? nap : 3); ++k) __builtin_amdgcn_s_sleep(32);
        }
        return 0;
    };
    // for a waiting wave of list x
    auto feed = [&](unsigned x, uint32_t rnd) {
        const KParams &p = params_again();
        unsigned long long *list = p.q_ctl + kQList + x * kLine;
        unsigned long long w = uniform(ld_agent(list));
        const unsigned idle = waiting(w);
        if (idle == 0) return;
        // about as many tries in a look's time as waves waiting
        const unsigned all = list_waves(p, x), donors = all > idle ? all - idle : 1u;
        if (__umulhi(rnd, donors) >= idle) return;
        // who waits first is read before it is taken off the list: as long as
        // it is the first, its entry stays (a list has an entry for each of
        // its waves, and only waves that wait hold one), but once it is off,
        // the wave that comes a list's length after it overwrites that
        const unsigned pos = (unsigned)w;
        const unsigned long long entry = ld_agent(&p.list[(size_t)x * (p.list_mask + 1) + (pos & p.list_mask)]);
        const int lev = give_level(kFeedLevels);
        const uint64_t can = __ballot(lev < 255 && !ahead_ring(p, inst));
        const int n = (__popcll(can) + 1) / 2;
        if (n == 0) return;
        const unsigned long long e = uniform(entry);
        if ((unsigned)(e >> 32) != pos + 1) return; // not written yet, or taken off meanwhile
        bool got = false;
        if (lane == 0) {
            const unsigned long long seen = atomicCAS(list, w, w + 1);
            got = seen == w;
        }
        if (!__ballot(got)) return;
        const unsigned to = (unsigned)e;
        const uint64_t chosen = smallest(can, lev < 255 ? min(g - sp + lev, 255) : 255, n);
        const bool give = (chosen >> lane) & 1ull;
        // the receiving wave's pending unit of each instance
        uint64_t todo = chosen;
        while (todo) {
            const int lead = __ffsll((long long)todo) - 1;
            const int i = __builtin_amdgcn_readlane(inst, lead);
            todo &= ~__ballot(inst == i);
            if (lane == lead) atomicAdd(&p.pend[grp * p.gstride + i], 1u);
        }
        if (give) {
            const size_t slot = (size_t)to * 64 + (size_t)__popcll(chosen & lanemask_lt());
            const uint32_t e2 = stk[lev * sstride];
            const uint32_t R = SE::rest(e2);
            const int d2 = __builtin_ctz(R);
            if (p.qpath) {
                uint32_t *to_path = &p.mail_path[slot * kPathWords];
                for (uint32_t k = 0; k < (uint32_t)kPathWords; ++k)
                    st_agent(&to_path[k], p.c_ipath[(size_t)k * NL + gl]);
                for (int k = 0; k <= lev; ++k)
                    path_put_agent(to_path, g - sp + k, k < lev ? SE::dir(stk[k * sstride]) : d2);
            }
            Here here;
            save_pos(here);
            go_back(lev);
            stk[lev * sstride] = SE::make(SE::dir(e2), R & (R - 1), SE::vals(e2));
            void_siblings(lev);
            (void)step_down(d2);
            uint32_t b[4];
            s.bd.pack(b);
            unsigned long long *m = (unsigned long long *)&p.mail[slot];
            st_agent(m, ((unsigned long long)b[1] << 32) | b[0]);
            if constexpr (W == 5) st_agent(m + 1, ((unsigned long long)b[3] << 32) | b[2]);
            st_agent(m + 2, ((unsigned long long)(uint32_t)inst << 32) | meta_pack(s.cell(), g - sp + lev + 1, s.hs.h, d2));
            st_agent(m + 3, p.want_load ? (unsigned long long)p.c_origin[gl] << 32 : 0ull);
            load_pos(here);
        }
        arrival_fence();
        if (lane == 0) {
            st_agent(&p.mail_head[(size_t)to * kLine], ((unsigned long long)(pos + 1) << 32) | (unsigned)n);
            atomicAdd(&p.q_ctl[kQList + list_of(blockIdx.x) * kLine + 1], (unsigned long long)n); // statistics
        }
    };

    uint32_t pf_idle = 0, pf_exp = 0, pf_pop = 0, pf_steps = 0;
    uint32_t pf_sib = 0, pf_rd1 = 0, pf_rd2 = 0; // table reads: sibling moves, first, second partition
    // the restored context is complete before the loop, so the compiler's
    // wait tracking does not carry its loads into every iteration (where it
    // would wait on a move's table reads before issuing the f-test's)
    __builtin_amdgcn_s_waitcnt(0);
    const long long t_work = wall_clock64();
    bool left = false; // the wave ran out of work
    for (int blk = 0;; ++blk) {
        const KParams &p = params_again();
        settle();
        uint64_t idle_mask = __ballot(st == ST_IDLE);
        if (idle_mask == ~0ull || (take_most == 64 && __popcll(idle_mask) >= kShareMin)) {
            Item it;
            bool have = false;
            unsigned mail = 0;
            if (blk == 0 && ticket) {
                // sent while the wave was leaving the last round
                const unsigned long long h = uniform(p.mail_head[(size_t)wave_id * kLine]);
                if ((unsigned)(h >> 32) == ticket) mail = (unsigned)h;
                ticket = 0;
            }
            if (!mail) {
                take_items(take_most, it, have);
                if (idle_mask == ~0ull && !__ballot(have)) {
                    mail = wait_for_mail();
                    if (!mail) {
                        left = true;
                        break;
                    }
                }
            }
            if (mail) read_mail(mail, it, have);
            if (have) start_item(it);
            idle_mask = __ballot(st == ST_IDLE);
        }
        if (__popcll(idle_mask) >= kShareMin) share(idle_mask);
        if (init) {
            init_heur<W, HEUR>(s, P, meta_pack(0, 0, s.hs.h, 0));
            init = false;
        }
        // the time limit, the round's end as some wave saw it, and, every few
        // blocks, whether the waves waiting now, had they waited since this
        // wave began to work, would have waited long enough (never before a
        // wave's first block: every round makes progress)
        if (blk >= least) {
            const long long now = wall_clock64();
            bool stop = steps_left <= 0 || (p.round_ticks && (unsigned long long)(now - t_start) >= p.round_ticks);
            const bool over = uniform(ld_agent(p.stop)) != 0;
            if (!stop && !over && threadIdx.x < 64 && (blk & 7) == 0)
                stop = (unsigned long long)(now - t_work) * idle_waves(p) >= p.turn_ticks * n_waves;
            if (stop && !over && lane == 0) st_agent(p.stop, 1u);
            if (stop || over) break;
            if (((blk + wave_id) & 1) == 0) {
                // every other look at any list, not the wave's own
                uint32_t rnd = ((uint32_t)now ^ (uint32_t)wave_id * 0x9e3779b9u) * 0x85ebca6bu;
                rnd = (rnd ^ (rnd >> 15)) * 0xc2b2ae35u;
                feed(blk & 2 ? (rnd >> 7) & (kLists - 1) : list_of(blockIdx.x), rnd ^ (rnd << 13));
            }
        }
        if (mode == 1 && searching(st) && ld_agent(&p.found[inst]) != kNoGoal)
            sp = 0, st = ST_POP; // first-solution: the rest of the item is not wanted
        const int block = max(1, min(steps_left, kShareSteps));
        steps_left -= block;
        for (int step = 0; step < block; ++step) {
            if (!__ballot(searching(st))) break;
            // ---- pop: undo up to kPops moves, until a level with a passing
            // child not visited yet ----
            int down = -1;      // child entered this step (-1: none)
            int slot = 0;       // its stack level
            uint32_t R = 0;     // passing children still to visit at that level
            bool known = false; // its lookup values are known (PDB)
            uint32_t kv = 0;
#pragma unroll 1
            for (int pk = 0; pk < kPops && st == ST_POP; ++pk) {
                if (sp == 0) {
                    st = ST_DONE;
                    break;
                }
                uint32_t e = stk[(sp - 1) * sstride];
                int d = SE::dir(e);
                uint32_t Re = SE::rest(e);
                if constexpr (HEUR == 1)
                    do_move_known<W>(s, 3 - d, P, SE::vals(e));
                else
                    unmove_md(s, d, SE::vals(e));
                --g;
                if (Re) {
                    down = __builtin_ctz(Re);
                    R = Re & (Re - 1);
                    slot = sp - 1;
                    st = ST_FRESH;
                    if constexpr (HEUR == 1) {
                        uint32_t &c = sibc[(slot % kSibLevels) * blockDim.x];
                        const uint32_t cv = c;
                        if ((cv >> 24) == (uint32_t)slot) {
                            known = true;
                            kv = (cv & 63u) | (((cv >> 6) & 63u) << 8);
                            c = (cv & 0xff000000u) | ((cv >> 12) & 0xfffu); // the sibling after it moves up
                        }
                    }
                } else {
                    --sp;
                }
            }
            // ---- or enter the first passing child of last step's expansion ----
            if (st == ST_DESC) {
                down = __builtin_ctz(dpass);
                R = dpass & (dpass - 1);
                slot = sp;
                known = true;
                kv = (((down >= 2) ? dval2 : dval) >> (16 * (down & 1))) & 0xffffu;
                if constexpr (HEUR == 1) {
                    if (R) {
                        // values of the next two passing children, 6 + 6 bits
                        // each.  An entry holds two siblings: a node with three
                        // more (an item rooted at an instance's root, all four
                        // moves passing) voids its level's entry instead, so
                        // that none of them takes values left by an older node
                        // of this depth, or the zeros shifted in after two
                        uint32_t ent = 0xffffffffu;
                        if (__builtin_popcount(R) <= 2) {
                            const int s1 = __builtin_ctz(R);
                            const uint32_t R2 = R & (R - 1);
                            const int s2 = R2 ? __builtin_ctz(R2) : s1;
                            const uint32_t v1 = (((s1 >= 2) ? dval2 : dval) >> (16 * (s1 & 1))) & 0xffffu;
                            const uint32_t v2 = (((s2 >= 2) ? dval2 : dval) >> (16 * (s2 & 1))) & 0xffffu;
                            const uint32_t p1 = (v1 & 63u) | (((v1 >> 8) & 63u) << 6);
                            const uint32_t p2 = (v2 & 63u) | (((v2 >> 8) & 63u) << 6);
                            ent = ((uint32_t)slot << 24) | p1 | (p2 << 12);
                        }
                        sibc[(slot % kSibLevels) * blockDim.x] = ent;
                    }
                }
            }
            // ---- one move down per lane and step, both cases on one path.  For
            // the PDB the move's values are applied after the f-test's table
            // reads are issued, so both sets of reads are in flight together ----
            PendMove pm;
            bool pmv = false;
            if (down >= 0) {
                if constexpr (HEUR == 1) {
                    uint32_t ov;
                    if constexpr (PROF) pf_sib += known ? 0u : 1u;
                    pm = move_pdb_begin<W>(s, down, P, known, kv, ov);
                    pmv = true;
                    stk[slot * sstride] = SE::make(down, R, ov);
                    sp = slot + 1;
                    ++g;
                    prev = down;
                    st = ST_FRESH;
                } else {
                    enter_child(down, R, slot, known, kv);
                }
            }

            // ---- expand, first half (PDB): the children's lookup indices and
            // table reads; they need the node's indices, not its values ----
            uint32_t gen = 0;
            // per child slot: lookups kr/kf, the index of the second lookup, the
            // first and second values read, the direction
            int ckr[4], ckf[4], cv1[4], cv2[4], cdir[4];
            uint32_t cidx2[4];
            int ng = 0;
            bool regfirst = true; // read the regular lookup first (else the reflected)
            if (st == ST_FRESH) {
                gen = legal_moves(s) & ~back_move(prev);
                if constexpr (HEUR == 1) {
                    // lane-slot j reads the lane's j-th generated child, so the
                    // wave runs as many slots as its largest family (3 below the
                    // root), not one per direction.  Only one lookup per child
                    // is read here: that of the partition whose sum is larger at
                    // the node (before a pending move's values: a heuristic
                    // choice); the other is read only for children the first
                    // does not already cut off (the reference's early cut,
                    // src_horie/idas_pdb.cu:228-231, regular sum first).
                    ng = __builtin_popcount(gen);
                    regfirst = s.hs.A >= s.hs.B;
                    const int bl = s.cell();
                    const PdbGeo &G = *P.geo;
                    uint32_t rem = gen;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        ckr[j] = ckf[j] = cv1[j] = cv2[j] = cdir[j] = 0;
                        cidx2[j] = 0;
                        if (!__ballot(j < ng)) continue;
                        if (j < ng) {
                            const int d = __builtin_ctz(rem);
                            rem &= rem - 1;
                            const int from = bl + dir_cell<W>(d);
                            const int t = s.bd.tile(from);
                            const uint2 wa = G.w[t][from], wb = G.w[t][bl];
                            const int kr = (int)(wa.x >> 28), kf = (int)(wa.y >> 28);
                            const uint32_t ir = sel4(s.hs.i0, s.hs.i1, s.hs.i2, s.hs.i3, kr) + (wb.x - wa.x);
                            const uint32_t iff = sel4(s.hs.j0, s.hs.j1, s.hs.j2, s.hs.j3, kf) + (wb.y - wa.y);
                            cdir[j] = d;
                            ckr[j] = kr;
                            ckf[j] = kf;
                            cv1[j] = pdb_read(P, regfirst ? ir : iff);
                            cidx2[j] = regfirst ? iff : ir;
                        }
                    }
                }
            }
            if constexpr (HEUR == 1) {
                if (pmv) move_pdb_finish(s.hs, pm);
            }

            // ---- expand, second half: goal test, count, f-tests ----
            bool expanded = false;
            if (st == ST_FRESH) {
                const int h = s.hs.h;
                bool xp = true;
                if (h == 0) {
                    // recorded between two blocks of steps, then expanded
                    xp = goal_seen;
                    if (!goal_seen) st = ST_GOAL;
                    goal_seen = false;
                }
                if (xp) {
                    expanded = true;
                    cnt += (uint32_t)__builtin_popcount(gen);
                    uint32_t pass = gen;
                    uint32_t cvals = 0, cvals2 = 0; // PDB values of children 0,1 / 2,3 (16 bits each)
                    if constexpr (HEUR == 0) {
                        // Manhattan is consistent: h changes by exactly +-1 per
                        // move and f keeps the threshold's parity, so with slack
                        // >= 2 every child fits and with slack 0 only children
                        // with h-1 do.
                        const int slack = L - g - h;
                        if (slack <= 2) {
                            const uint32_t near = nearer_moves<W>(s.bd, s.cell(), s.row(), s.col());
                            if (slack < 2) pass = gen & near;
                            // A child at slack 0 (slack 0 and nearer, or slack 2
                            // and farther) whose own children all fail the
                            // f-test is a leaf: its children are counted here
                            // and it is not entered.  Its children's tiles are
                            // all on the current board (entering it would only
                            // move the blank there).  With h >= 2 no such child
                            // is a goal, and a leaf has no goal child (one would
                            // be nearer, and pass).  One child per expansion is
                            // tested, the first such: a wave would run the test
                            // as often as its lane with the most.
                            const uint32_t cand = h < 2 ? 0u : (slack < 2 ? pass : gen & ~near);
                            if (cand) {
                                const int d = __builtin_ctz(cand);
                                const int cc = s.cell() + dir_cell<W>(d);
                                int cr, ck;
                                uint32_t cgen = ~back_move(d);
                                if constexpr (W == 4) {
                                    cr = cc >> 2;
                                    ck = cc & 3;
                                    cgen &= legal_cell<W>(cc);
                                } else {
                                    cr = s.row() + dir_dr(d);
                                    ck = s.col() + dir_dc(d);
                                    cgen &= legal_moves<W>(cr, ck);
                                }
                                if (!(cgen & nearer_moves<W>(s.bd, cc, cr, ck))) {
                                    cnt += (uint32_t)__builtin_popcount(cgen);
                                    pass &= ~(1u << d);
                                }
                            }
                        }
                    } else {
                        // the PDB max is not consistent (lookups take the minimum
                        // over blank cells): h may jump by 3, so every generated
                        // child gets its own f-test
                        pass = 0;
                        const HState<1> &hs = s.hs;
                        // the first partition's sum of each child; the second
                        // lookup is read only where that sum fits
                        uint32_t need = 0;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if (j < ng) {
                                const int s1 = regfirst ? hs.A - byte_of(hs.v0, ckr[j]) + cv1[j]
                                                        : hs.B - byte_of(hs.v1, ckf[j]) + cv1[j];
                                if (g + 1 + s1 <= L) {
                                    need |= 1u << j;
                                    cv2[j] = pdb_read(P, cidx2[j]);
                                }
                                if constexpr (PROF) {
                                    pf_rd1 += 1u;
                                    pf_rd2 += (g + 1 + s1 <= L) ? 1u : 0u;
                                }
                            }
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            if ((need >> j) & 1u) {
                                const int d = cdir[j];
                                const int vr = regfirst ? cv1[j] : cv2[j];
                                const int vf = regfirst ? cv2[j] : cv1[j];
                                const int A = hs.A - byte_of(hs.v0, ckr[j]) + vr;
                                const int B = hs.B - byte_of(hs.v1, ckf[j]) + vf;
                                const int hc = A > B ? A : B;
                                pass |= (g + 1 + hc <= L) ? (1u << d) : 0u;
                                const uint32_t v = ((uint32_t)vr | ((uint32_t)vf << 8)) << (16u * (uint32_t)(d & 1));
                                if (d < 2)
                                    cvals |= v;
                                else
                                    cvals2 |= v;
                            }
                        }
                    }
                    if (!pass) {
                        st = ST_POP;
                    } else if (sp < MAXD) {
                        // enter the first passing child next step
                        st = ST_DESC;
                        dpass = pass;
                        dval = cvals;
                        dval2 = cvals2;
                    } else {
                        // stack full: the passing children become queue items
                        // between two blocks of steps
                        st = ST_FULL;
                        dpass = pass;
                    }
                }
            }

            if constexpr (PROF) {
                pf_steps += 1;
                pf_idle += (!expanded && (st == ST_IDLE || st >= ST_DONE)) ? 1u : 0u;
                pf_exp += expanded ? 1u : 0u;
                pf_pop += (!expanded && (st == ST_POP || st == ST_DESC)) ? 1u : 0u;
            }
        }
    }

    // a descent still pending is made now, so the saved context is a node
    if (st == ST_DESC) {
        const int dn = __builtin_ctz(dpass);
        enter_child(dn, dpass & (dpass - 1), sp, true, (((dn >= 2) ? dval2 : dval) >> (16 * (dn & 1))) & 0xffffu);
    }

    const bool busy = (st == ST_FRESH || st == ST_POP);
    if (lane == 0) p.ticket[wave_id] = left ? ticket : 0u;

    // node counts of idle lanes, and of lanes far on the way to wrapping
    uint64_t todo = __ballot(cnt != 0 && (!busy || cnt >= (1u << 30)));
    while (todo) {
        const int lead = __ffsll((long long)todo) - 1;
        const int i = __builtin_amdgcn_readlane(inst, lead);
        const bool mine = cnt != 0 && (!busy || cnt >= (1u << 30)) && inst == i;
        todo &= ~__ballot(mine);
        if (mine && p.want_load)
            atomicAdd(&p.load[(size_t)(inst >> 1) * p.capl + p.c_origin[gl]], (unsigned long long)cnt);
        unsigned long long c = mine ? cnt : 0u;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) c += shfl_xor_u64(c, off);
        if (mine) cnt = 0;
        if (lane == lead) atomicAdd(&p.cnt[grp * p.gstride + i], c);
    }
    if constexpr (PROF) {
        // wave sums of this round's lane-step states
        for (int off = 32; off > 0; off >>= 1) {
            pf_idle += __shfl_xor(pf_idle, off);
            pf_exp += __shfl_xor(pf_exp, off);
            pf_pop += __shfl_xor(pf_pop, off);
            pf_sib += __shfl_xor(pf_sib, off);
            pf_rd1 += __shfl_xor(pf_rd1, off);
            pf_rd2 += __shfl_xor(pf_rd2, off);
        }
        if (lane == 0) {
            unsigned long long *w = p.prof + (size_t)wave_id * 8; // the wave's own: one address for all would be a queue
            w[0] += pf_idle;
            w[1] += pf_exp;
            w[2] += pf_pop;
            w[3] += pf_steps;
            w[4] += pf_sib;
            w[5] += pf_rd1;
            w[6] += pf_rd2;
        }
    }
    if (p.wtime && lane == 0 && p.ctl[6] == p.wtime_round) {
        const int wg = gl >> 6; // global wave index
        p.wtime[2 * wg] = (unsigned long long)t_start;
        p.wtime[2 * wg + 1] = (unsigned long long)wall_clock64();
    }
    if (busy) {
        p.c_st[gl] = (uint32_t)(goal_seen && st == ST_FRESH ? ST_GOAL : st) | ((uint32_t)sp << 8);
        uint32_t b[4];
        s.bd.pack(b);
#pragma unroll
        for (int k = 0; k < 4; ++k) p.c_rows[k * NL + gl] = b[k];
        p.c_meta[gl] = meta_pack(s.cell(), g, s.hs.h, prev);
        p.c_inst[gl] = (uint32_t)inst;
        p.c_cnt[gl] = cnt;
        if constexpr (HEUR == 1) {
            p.c_pdb[0 * NL + gl] = s.hs.i0;
            p.c_pdb[1 * NL + gl] = s.hs.i1;
            p.c_pdb[2 * NL + gl] = s.hs.i2;
            p.c_pdb[3 * NL + gl] = s.hs.i3;
            p.c_pdb[4 * NL + gl] = s.hs.j0;
            p.c_pdb[5 * NL + gl] = s.hs.j1;
            p.c_pdb[6 * NL + gl] = s.hs.j2;
            p.c_pdb[7 * NL + gl] = s.hs.j3;
            p.c_pdb[8 * NL + gl] = s.hs.v0;
            p.c_pdb[9 * NL + gl] = s.hs.v1;
        }
        for (int k = 0; k < sp; ++k) cstk[(size_t)k * NL + gl] = stk[k * sstride];
    } else {
        p.c_st[gl] = ST_IDLE;
    }
}

// largest f on a frontier node's root path (its own f included)
__device__ __forceinline__ int path_f(const Item &it) {
    int f = meta_g(it.meta) + meta_h(it.meta);
    return (int)it.x0 > f ? (int)it.x0 : f;
}

// ---------------------------------------------------------------------------
// k_restart: between rounds, one block per instance; it acts where the current
// iteration has ended, none runs yet, or lookahead was asked for.  Thread 0
// resolves the instance's iterations in order: while the current iteration
// has drained, its count is recorded and it ends the instance (goal found,
// or iteration limit) or the next one becomes current -- already running if
// it was started as lookahead.  An iteration is started when the instance has
// none running, or as lookahead beside the current one when k_spec asked for
// it.  Starting iteration j (threshold Lbase + 2j) in slot j & 1:
//   1. logs (frontier node, previous threshold, nodes generated below it)
//      samples of the iteration that ended (learned-LB training data; only
//      without lookahead, where one iteration runs at a time),
//   2. sets the slot's count to the top-tree count of the threshold from the
//      f-histogram and notes a goal in the top tree,
//   3. queues the frontier nodes whose path-f fits, ordered by a key in
//      decreasing order (counting sort over 64 half-log2 buckets): frontier
//      order (uniform), last iteration's load (the reference's load-based
//      static LB, src/15puzzle_block_parallel.cu:490-563), or the learned
//      prediction -- longest expected subtree first.  With re-splitting
//      (resplit > 0, previous-load or learned policy), a node whose
//      estimate exceeds resplit x the mean of the nodes that fit is queued
//      as its children (two levels: grandchildren) instead, as the
//      reference re-splits heavy roots into ceil(load / mean) pieces,
//   4. clears the per-frontier-node loads (a split node's starts at the
//      children the split counted).
// An iteration with no frontier work is drained at once.  Lanes run no
// kernel meanwhile, so the resolution needs no atomics on instance state.

// Estimated subtree size of frontier node i in iteration it: the previous
// iteration's count below it (previous-load policy) or the learned
// prediction of log2(1 + size) (learned policy); 0 for frontier order.
__device__ __forceinline__ float lb_log2_est(const KParams &p, int inst, unsigned i, int it) {
    if (p.lb == 2) return it > 0 ? log2f((float)p.load[(size_t)inst * p.capl + i] + 1.f) : 0.f;
    if (p.lb == 1) return p.pred[((size_t)inst * p.capl + i) * kPredK + (it < kPredK ? it : kPredK - 1)];
    return 0.f;
}
// dispatch bucket of a key in half-log2 steps (64 buckets, largest first)
__device__ __forceinline__ int key_bucket(float key) {
    int b = (int)(key * 2.f);
    return b < 0 ? 0 : (b > 63 ? 63 : b);
}
// bucket of an item `level` split levels below a node of bucket b: each level
// divides the estimate by about 3 (the children of a node), 3 half-log2 steps
__device__ __forceinline__ int split_bucket(int b, int level) {
    int c = b - 3 * level;
    return c < 0 ? 0 : c;
}

// Re-split of a heavy frontier node (the reference's static load balancing,
// src/15puzzle_block_parallel.cu:490-563 with divide_root_set :325-375): the
// node is expanded here, its count of generated children added to the
// iteration (the lane that would take it counts the same children,
// src/24puzzle.cc:119-131), and its children whose f fits the threshold are
// queued in its place -- or, at two levels, their children.  A goal node is
// queued itself (its lane records the goal).  emit(pos, g, prev, level, d1,
// d2) receives each item; returns the generated-children count.
template <int W, int HEUR, class Emit>
__device__ unsigned split_node(const PdbCtx &P, const Item &x, int L, int levels, Emit &&emit) {
    Pos<W, HEUR> s;
    pos_from_item<W, HEUR>(s, x.b, x.meta, P);
    const int g = meta_g(x.meta), prev = meta_prev(x.meta);
    unsigned gen_total = 0;
    uint32_t gen = legal_moves(s);
    gen &= ~(prev < 4 ? (1u << (3 - prev)) : 0u);
    gen_total += (unsigned)__builtin_popcount(gen);
#pragma unroll 1
    while (gen) {
        const int d = __builtin_ctz(gen);
        gen &= gen - 1;
        Pos<W, HEUR> c = s;
        do_move<W, HEUR>(c, d, P);
        if (g + 1 + c.hs.h > L) continue;
        if (levels < 2 || c.hs.h == 0) {
            emit(c, g + 1, d, 1, d, 0);
            continue;
        }
        uint32_t gen2 = legal_moves(c);
        gen2 &= ~(1u << (3 - d));
        gen_total += (unsigned)__builtin_popcount(gen2);
#pragma unroll 1
        while (gen2) {
            const int d2 = __builtin_ctz(gen2);
            gen2 &= gen2 - 1;
            Pos<W, HEUR> c2 = c;
            do_move<W, HEUR>(c2, d2, P);
            if (g + 2 + c2.hs.h > L) continue;
            emit(c2, g + 2, d2, 2, d, d2);
        }
    }
    return gen_total;
}

// thread 0 of k_restart: resolve drained iterations; returns the index of an
// iteration to start, or -1
__device__ int resolve_instance(const KParams &p, int inst) {
    for (;;) {
        if (p.done[inst]) return -1;
        const int cur = p.it[inst];
        const int nl = p.nlive[inst];
        if (nl == 0) {
            p.nlive[inst] = 1;
            return cur;
        }
        const int isc = inst * 2 + (cur & 1);
        if (!p.drained[isc]) {
            if (p.want_next[inst] && nl == 1 && cur + 1 < p.max_iters && p.found[isc] == kNoGoal) {
                p.want_next[inst] = 0;
                p.nlive[inst] = 2;
                atomicAdd(&p.ctl[13], 1u);
                return cur + 1;
            }
            return -1;
        }
        p.iter_counts[(size_t)inst * p.max_iters + cur] = slot_count(p, isc);
        if (p.found[isc] != kNoGoal || cur + 1 >= p.max_iters) {
            p.opt[inst] = p.found[isc] != kNoGoal ? p.found[isc] : -1;
            p.done[inst] = 1;
            p.dead[inst * 2] = 1;
            p.dead[inst * 2 + 1] = 1;
            atomicSub(&p.ctl[1], 1u);
            return -1;
        }
        p.it[inst] = cur + 1;
        p.nlive[inst] = nl - 1;
    }
}

// threads of a restart block: four passes over the instance's frontier, its
// items' loads waited for in each (one instance, 2048 nodes: 18 us with 256
// threads, 16 us with 1024)
constexpr int kRestartThreads = 1024;

template <int W, int HEUR>
__device__ __forceinline__ void restart_instance(const KParams &p, const PdbGeo *geo_g, int inst) {
    __shared__ unsigned long long s_cnt;
    __shared__ unsigned s_bucket[64];
    __shared__ unsigned long long s_base;
    __shared__ int s_j, s_ring;
    __shared__ float s_est;
    __shared__ unsigned s_nfit, s_items;
    __shared__ PdbGeo geo_s;
    if (threadIdx.x == 0) {
        // nothing to do while the current iteration runs and no lookahead is
        // asked for
        const int live = p.nlive[inst], at = inst * 2 + (p.it[inst] & 1);
        const bool ended = live > 0 && slot_pend(p, at) == 0;
        s_j = !p.done[inst] && (live == 0 || ended || p.want_next[inst]) ? 1 : 0;
        if (live > 0) p.drained[at] = ended;
        if (live > 1) p.drained[at ^ 1] = slot_pend(p, at ^ 1) == 0;
    }
    __syncthreads();
    if (!s_j) return;
    __syncthreads();
    const unsigned nf = min(p.nfront[inst], (unsigned)p.capl);
    const Item *F = p.frontier + (size_t)inst * p.capl;
    unsigned long long *load = p.load + (size_t)inst * p.capl;
    // heavy-node re-split: only under a policy with estimates
    const bool resplit = p.resplit > 0 && p.lb != 0;
    PdbCtx P{&geo_s, p.pdb};
    if constexpr (HEUR == 1) {
        if (resplit) {
            const uint32_t *src = (const uint32_t *)geo_g;
            uint32_t *dst = (uint32_t *)&geo_s;
            for (int i = threadIdx.x; i < (int)(sizeof(PdbGeo) / 4); i += blockDim.x) dst[i] = src[i];
        }
    }

    for (;;) {
        if (threadIdx.x == 0) {
            s_j = resolve_instance(p, inst);
            s_ring = s_j > p.it[inst] ? 1 : 0; // a lookahead start goes to ring 1
        }
        __syncthreads();
        const int it = s_j;
        if (it < 0) break;
        const int isl = inst * 2 + (it & 1);
        const int L = p.Lbase[inst] + 2 * it;
        // 1. samples of the iteration that ended
        if (it > 0 && p.max_samples > 0 && !p.lookahead) {
            for (unsigned i = threadIdx.x; i < nf; i += blockDim.x) {
                if (path_f(F[i]) <= L - 2) {
                    unsigned k = atomicAdd(p.n_samples, 1u);
                    if (k < p.max_samples) {
                        Sample sm;
                        sm.item = F[i];
                        sm.thr = L - 2;
                        sm.pad = 0;
                        sm.load = load[i];
                        p.samples[k] = sm;
                    }
                }
            }
        }
        if (threadIdx.x == 0) {
            s_cnt = 0;
            s_est = 0.f;
            s_nfit = 0;
        }
        for (int b = threadIdx.x; b < 64; b += blockDim.x) s_bucket[b] = 0;
        __syncthreads();
        // 2. top tree: sum of gen over path-f <= L; with re-splitting, the
        // mean estimated subtree size of the frontier nodes that fit
        unsigned long long c = 0;
        for (int f = threadIdx.x; f < kFBins; f += blockDim.x)
            if (f <= L) c += p.topgen[(size_t)inst * kFBins + f];
        atomicAdd(&s_cnt, c);
        if (resplit) {
            float e = 0.f;
            unsigned k = 0;
            for (unsigned i = threadIdx.x; i < nf; i += blockDim.x)
                if (path_f(F[i]) <= L) {
                    e += exp2f(lb_log2_est(p, inst, i, it)) - 1.f;
                    ++k;
                }
            atomicAdd(&s_est, e);
            atomicAdd(&s_nfit, k);
        }
        __syncthreads();
        // a node is split one level when its estimate exceeds resplit x the
        // mean, two levels beyond 8 x that
        const float cut1 = resplit && s_nfit ? (float)p.resplit * s_est / (float)s_nfit : 3.4e38f;
        const float cut2 = 8.f * cut1;
        auto levels_of = [&](unsigned i, float key) -> int {
            if (!resplit) return 0;
            const float e = exp2f(key) - 1.f;
            return e > cut2 ? 2 : (e > cut1 ? 1 : 0);
        };
        // 3. bucket sizes of the items (frontier nodes that fit, or the items
        // a split node becomes); split nodes' generated children are counted
        for (unsigned i = threadIdx.x; i < nf; i += blockDim.x) {
            const Item x = F[i];
            if (path_f(x) > L) continue;
            const float key = lb_log2_est(p, inst, i, it);
            const int b = key_bucket(key);
            const int lv = levels_of(i, key);
            if (lv == 0 || meta_h(x.meta) == 0) {
                atomicAdd(&s_bucket[b], 1u);
                continue;
            }
            const unsigned gn = split_node<W, HEUR>(P, x, L, lv, [&](const Pos<W, HEUR> &, int, int, int level, int, int) {
                atomicAdd(&s_bucket[split_bucket(b, level)], 1u);
            });
            atomicAdd(&s_cnt, (unsigned long long)gn);
        }
        __syncthreads();
        static_assert(kRestartThreads >= 64, "a wave scans the buckets");
        if (threadIdx.x < 64) { // largest keys first
            const int b = 63 - (int)threadIdx.x;
            const unsigned n = s_bucket[b];
            unsigned upto = n;
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned v = __shfl_up(upto, o);
                if ((int)threadIdx.x >= o) upto += v;
            }
            s_bucket[b] = upto - n;
            if (threadIdx.x == 63) s_items = upto;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const unsigned off = s_items;
            s_base = off ? q_reserve<kGroups>(p, s_ring, (unsigned long long)off) : 0ull;
            p.L[isl] = L;
            p.itn[isl] = it;
            p.found[isl] = p.top_goal[inst] <= L ? p.top_goal[inst] : kNoGoal;
            for (int x = 0; x < kGroups; ++x) {
                p.cnt[x * p.gstride + isl] = x ? 0ull : s_cnt;
                p.pend[x * p.gstride + isl] = x ? 0u : off;
            }
            p.drained[isl] = off == 0 ? 1 : 0;
            p.dead[isl] = 0;
        }
        __syncthreads();
        // 4. the items to the queue; the per-node loads of the new iteration
        // start from zero, or from the children a split counted
        for (unsigned i = threadIdx.x; i < nf; i += blockDim.x) {
            Item x = F[i];
            unsigned long long ld = 0;
            if (path_f(x) <= L) {
                const float key = lb_log2_est(p, inst, i, it);
                const int b = key_bucket(key);
                const int lv = levels_of(i, key);
                if (lv == 0 || meta_h(x.meta) == 0) {
                    unsigned k = atomicAdd(&s_bucket[b], 1u);
                    x.inst = (uint32_t)isl;
                    x.x1 = i;
                    const size_t slot = q_slot(p, s_ring, s_base + k);
                    p.q[slot] = x;
                    if (p.qpath) path_from_u64(p.fpath[(size_t)inst * p.capl + i], p.qpath, (uint32_t)slot * kPathWords);
                } else {
                    const int g0 = meta_g(x.meta);
                    unsigned made = 0;
                    ld = split_node<W, HEUR>(P, x, L, lv, [&](const Pos<W, HEUR> &cp, int g, int prev, int level, int d1, int d2) {
                        ++made;
                        unsigned k = atomicAdd(&s_bucket[split_bucket(b, level)], 1u);
                        Item ci;
                        cp.bd.pack(ci.b);
                        ci.meta = meta_pack(cp.cell(), g, cp.hs.h, prev);
                        ci.inst = (uint32_t)isl;
                        ci.x0 = 0;
                        ci.x1 = i;
                        const size_t slot = q_slot(p, s_ring, s_base + k);
                        p.q[slot] = ci;
                        if (p.qpath) {
                            const uint32_t qo = (uint32_t)slot * kPathWords;
                            path_from_u64(p.fpath[(size_t)inst * p.capl + i], p.qpath, qo);
                            path_put(p.qpath, qo, 1, g0, d1);
                            if (level == 2) path_put(p.qpath, qo, 1, g0 + 1, d2);
                        }
                    });
                    atomicAdd(&p.ctl[14], 1u);
                    atomicAdd(&p.ctl[15], made);
                }
            }
            load[i] = ld;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) p.want_next[inst] = 0;
}

template <int W, int HEUR>
__global__ void __launch_bounds__(kRestartThreads) k_restart(KParams p, const PdbGeo *geo_g) {
    restart_instance<W, HEUR>(p, geo_g, (int)blockIdx.x);
}

// k_spec (lookahead): after a round, while the waves without work outnumber
// the queued items by more than 1/32 of the lanes, ask for lookahead for
// instances that run a single iteration (no goal yet, and a previous
// iteration, if any, of at least one node per lane), until their frontiers
// would fill them.  Instances are taken from a start that rotates with the
// round number.  Only the schedule changes: each iteration's count is its own,
// and the result is resolved in order.
// items of ring r not taken yet
__device__ __forceinline__ unsigned long long q_waiting(const KParams &p, int r) {
    const unsigned long long tail = p.q_ctl[kQTail + r * kQRing];
    unsigned long long n = 0;
    for (int x = 0; x < kGroups; ++x) {
        const unsigned long long h = p.q_ctl[kQHead + r * kQRing + x * kLine];
        if (h < tail) n += (tail - h + kGroups - 1) / kGroups;
    }
    return n;
}

__device__ __forceinline__ void ask_lookahead(const KParams &p) {
    __shared__ unsigned long long s_room, s_used;
    const unsigned idle = idle_waves(p);
    if (threadIdx.x == 0) {
        unsigned long long qlen = 0;
        for (int r = 0; r < 2; ++r) qlen += q_waiting(p, r);
        // a queued item feeds a wave
        const unsigned long long lanes = (unsigned long long)p.n_lanes;
        const unsigned long long taken = lanes - 64ull * idle + 64ull * qlen;
        s_room = (taken < lanes && lanes - taken >= lanes / 32) ? lanes - taken : 0ull;
        s_used = 0;
    }
    __syncthreads();
    if (s_room == 0) return;
    const int n = p.n_inst;
    const int start = (int)(p.ctl[6] % (unsigned)n);
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        int inst = start + k;
        if (inst >= n) inst -= n;
        if (p.done[inst] || p.nlive[inst] != 1) continue;
        const int cur = p.it[inst];
        const int isc = inst * 2 + (cur & 1);
        if (cur + 1 >= p.max_iters || p.found[isc] != kNoGoal || slot_pend(p, isc) == 0) continue;
        // an instance whose last finished iteration counted fewer nodes than
        // there are lanes has iterations that end within a round or two:
        // lookahead would mostly run work that its goal then drops (100
        // 40-move 15-puzzles: 3200 instances/s with it, 5300 without)
        if (cur > 0 && p.iter_counts[(size_t)inst * p.max_iters + cur - 1] < (unsigned long long)p.n_lanes) continue;
        const unsigned long long est = min(p.nfront[inst], (unsigned)p.capl);
        if (atomicAdd(&s_used, 8ull * est) >= s_room) continue;
        p.want_next[inst] = 1;
    }
}
__global__ void __launch_bounds__(256) k_spec(KParams p) { ask_lookahead(p); }

// k_control: between rounds.  Publishes the items appended to both rings
// during the last round, sets how many a wave takes at once (an even share of
// the queue, so that few items reach many waves), and clears the round's
// words: whoever still waits on a list waits no more.  One wave, a word a lane.
__device__ __forceinline__ void control(const KParams &p, int lane) {
    unsigned long long items = 0;
    if (lane < 2 * kGroups) {
        const int r = lane / kGroups, x = lane % kGroups;
        unsigned long long *head = p.q_ctl + kQHead + r * kQRing + x * kLine;
        const unsigned long long limit = p.q_ctl[kQTail + r * kQRing + 1], tail = p.q_ctl[kQTail + r * kQRing];
        unsigned long long h = *head;
        // a head past the limit goes back to the group's first position there
        if (h >= limit + kGroups) h = limit + ((unsigned)(x - (int)(limit % kGroups)) & (kGroups - 1));
        *head = h;
        if (h < tail) items = (tail - h + kGroups - 1) / kGroups;
    } else if (lane < 3 * kGroups) {
        p.q_ctl[kQStart + (lane - 2 * kGroups) * kLine] = 0;
    }
    static_assert(kLists == 64, "a list a lane");
    unsigned long long *list = p.q_ctl + kQList + lane * kLine;
    const unsigned long long w = list[0];
    unsigned idle = waiting(w);
    unsigned long long given = list[1];
    list[0] = (w & 0xffffffff00000000ull) | (w >> 32);
    list[1] = 0;
    for (int off = 32; off > 0; off >>= 1) {
        items += shfl_xor_u64(items, off);
        given += shfl_xor_u64(given, off);
        idle += __shfl_xor(idle, off);
    }
    arrival_fence(); // the limits are read
    if (lane < 2) {
        unsigned long long *c = p.q_ctl + kQTail + lane * kQRing;
        c[1] = c[0];
    }
    if (lane == 0) {
        const unsigned n_waves = (unsigned)p.n_lanes >> 6;
        *p.stop = 0;
        p.ctl[7] += (unsigned)given;
        p.ctl[12] = n_waves - idle;  // waves with work at the round's end, for the host
        p.ctl[20] = items > 0xffffffffull ? 0xffffffffu : (unsigned)items;
        const unsigned long long share = (items + n_waves - 1) / n_waves;
        p.ctl[4] = share < 1 ? 1u : share > 64 ? 64u : (unsigned)share;
        p.ctl[6] += 1;
    }
}

__global__ void __launch_bounds__(64) k_control(KParams p) { control(p, (int)threadIdx.x); }

// k_turn: the three between the rounds of a single instance, in its one
// workgroup.  As launches of their own k_spec and k_control take 4.6 and 4.9 us
// a round, most of it the launch (one 15-puzzle of 8 to 16 rounds: 2.42 -> 2.23
// and 4.25 -> 4.03 ms, the graph made later among it).
template <int W, int HEUR>
__global__ void __launch_bounds__(kRestartThreads) k_turn(KParams p, const PdbGeo *geo_g, int spec) {
    if (spec) {
        ask_lookahead(p);
        __syncthreads();
    }
    restart_instance<W, HEUR>(p, geo_g, 0);
    __syncthreads();
    if (threadIdx.x < 64) control(p, (int)threadIdx.x);
}

// ---------------------------------------------------------------------------
// Root split: one node of a level.  It is expanded without pruning: its
// generated children are counted under its f (hist), and they form the next
// level, from position reserve(children) of `out` on.  lp_in/lp_out: the
// levels' paths, or null.  F = largest f on the path from the root (x0 carries
// the parent's F): the node is expanded in iteration L iff F <= L, heuristic
// consistent or not.
template <int W, int HEUR, class Reserve, class Hist, class Goal>
__device__ __forceinline__ void split_expand(const KParams &p, const PdbCtx &P, int inst, const Item &it, Item *out,
                                             const unsigned long long *lp_in, unsigned long long *lp_out,
                                             Reserve &&reserve, Hist &&hist, Goal &&goal) {
    Pos<W, HEUR> s;
    pos_from_item<W, HEUR>(s, it.b, it.meta, P);
    const int g = meta_g(it.meta), prev = meta_prev(it.meta);
    int f = g + s.hs.h;
    if ((int)it.x0 > f) f = (int)it.x0;
    if (s.hs.h == 0) {
        goal(f);
        // levels run in depth order, so the first goal recorded is a
        // shallowest one; it goes to both iteration slots (the iteration that
        // ends the instance, in either slot, finds no shallower goal)
        if (p.sol)
            for (int sl = inst * 2; sl < inst * 2 + 2; ++sl)
                if (atomicCAS(&p.sol_len[sl], -1, g) == -1) path_from_u64(*lp_in, p.sol, (uint32_t)sl * kPathWords);
    }
    uint32_t gen = legal_moves(s) & ~back_move(prev);
    const unsigned n = (unsigned)__builtin_popcount(gen);
    hist(f < kFBins ? f : kFBins - 1, n);
    unsigned k = reserve(n);
    while (gen) {
        const int d = __builtin_ctz(gen);
        gen &= gen - 1;
        Pos<W, HEUR> c = s;
        do_move<W, HEUR>(c, d, P);
        Item ci;
        c.bd.pack(ci.b);
        ci.meta = meta_pack(c.cell(), g + 1, c.hs.h, d);
        ci.inst = (uint32_t)inst;
        ci.x0 = (uint32_t)f;
        ci.x1 = 0;
        if (k < (unsigned)p.capl) {
            out[k] = ci;
            // split depth <= 32 when paths are recorded: move g fits the u64
            if (lp_out) lp_out[k] = *lp_in | ((unsigned long long)d << (2 * g));
        }
        ++k;
    }
}

template <int HEUR> __device__ __forceinline__ void load_geo(PdbGeo &geo_s, const PdbGeo *geo_g) {
    if constexpr (HEUR == 1) {
        const uint32_t *src = (const uint32_t *)geo_g;
        uint32_t *dst = (uint32_t *)&geo_s;
        for (int i = threadIdx.x; i < (int)(sizeof(PdbGeo) / 4); i += blockDim.x) dst[i] = src[i];
        __syncthreads();
    }
}

// k_split_level: one level of the root split, all instances at once.  A level
// that already holds >= target nodes (or is at max depth) becomes the
// instance's frontier; otherwise every node is expanded.
template <int W, int HEUR>
__global__ void __launch_bounds__(256) k_split_level(KParams p, const PdbGeo *geo_g, const Item *lvl_in,
                                                     const unsigned *n_in, Item *lvl_out, unsigned *n_out,
                                                     int *frozen, int depth, int max_depth, unsigned target,
                                                     const unsigned long long *lp_in, unsigned long long *lp_out) {
    __shared__ PdbGeo geo_s;
    PdbCtx P{&geo_s, p.pdb};
    load_geo<HEUR>(geo_s, geo_g);
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int inst = (int)(gid / (size_t)p.capl);
    const unsigned j = (unsigned)(gid % (size_t)p.capl);
    if (inst >= p.n_inst) return;
    // frozen[inst] = 1 + the depth at which the instance froze; it is written
    // during that launch, so this launch only honours earlier freezes
    const int fz = frozen[inst];
    if (fz != 0 && fz - 1 < depth) return;
    const unsigned n = min(n_in[inst], (unsigned)p.capl);
    const bool freeze = (n >= target) || (depth >= max_depth);
    const size_t at = (size_t)inst * p.capl;
    if (freeze) {
        if (j < n) {
            ((Item *)p.frontier)[at + j] = lvl_in[at + j];
            if (lp_in) ((unsigned long long *)p.fpath)[at + j] = lp_in[at + j];
        }
        if (j == 0) {
            ((unsigned *)p.nfront)[inst] = n;
            frozen[inst] = depth + 1;
        }
        return;
    }
    if (j >= n) return;
    split_expand<W, HEUR>(
        p, P, inst, lvl_in[at + j], lvl_out + at, lp_in ? lp_in + at + j : nullptr, lp_out ? lp_out + at : nullptr,
        [&](unsigned k) { return atomicAdd(&n_out[inst], k); },
        [&](int f, unsigned k) { atomicAdd((unsigned *)&p.topgen[(size_t)inst * kFBins + f], k); },
        [&](int f) { atomicMin((int *)&p.top_goal[inst], f); });
}

// k_begin: one workgroup per instance starts it: the root's heuristic, the
// per-instance state, and (split) the whole root split, level by level in the
// instance's region of the two level buffers, sizes and f-histogram in LDS.
// A launch a level over all instances' regions costs 4 us a level however
// small, and where there are many instances mostly looks at empty slots (100
// instances, 2048 nodes each: 25 launches, 2.1 ms; so 0.05 ms).  One workgroup
// falls behind the grid on a very large frontier (kOneBlockSplit).
constexpr int kBeginThreads = 1024;
template <int W, int HEUR>
__global__ void __launch_bounds__(kBeginThreads) k_begin(KParams p, const PdbGeo *geo_g, Item *lvl0, Item *lvl1,
                                                         unsigned *nlvl0, int *frozen, int max_depth, unsigned target,
                                                         unsigned long long *lp0, unsigned long long *lp1, int split) {
    __shared__ PdbGeo geo_s;
    __shared__ unsigned s_n[2], s_hist[kFBins];
    __shared__ int s_goal;
    PdbCtx P{&geo_s, p.pdb};
    load_geo<HEUR>(geo_s, geo_g);
    const int inst = (int)blockIdx.x, t = threadIdx.x;
    const size_t at = (size_t)inst * p.capl;
    if (t == 0) {
        Item it = p.roots[inst];
        Board<W> bd;
        bd.unpack(it.b);
        int h = 0;
        if constexpr (HEUR == 0) {
            for (int c = 0; c < W * W; ++c) {
                const int x = bd.tile(c);
                if (x) h += abs(c / W - trow<W>(x)) + abs(c % W - tcol<W>(x));
            }
        } else {
            HState<1> hs;
            pdb_init(P, hs, bd);
            h = hs.h;
        }
        it.meta = (it.meta & 0xff00ffffu) | ((uint32_t)h << 16);
        ((Item *)p.roots)[inst] = it;
        lvl0[at] = it;
        if (lp0) lp0[at] = 0ull; // the root's empty path
        s_n[0] = 1;
        s_n[1] = 0;
        s_goal = kNoGoal;
        p.it[inst] = 0;
        p.nlive[inst] = 0;
        p.want_next[inst] = 0;
        p.done[inst] = 0;
        p.opt[inst] = -1;
        ((int *)p.Lbase)[inst] = h;
        if (!split) {
            nlvl0[inst] = 1;
            frozen[inst] = 0;
            ((int *)p.top_goal)[inst] = kNoGoal;
        }
    }
    if (t < 2) {
        const int isl = inst * 2 + t;
        p.L[isl] = 0;
        p.itn[isl] = 0;
        p.found[isl] = kNoGoal;
        p.drained[isl] = 0;
        p.dead[isl] = 0;
        if (p.sol_len) p.sol_len[isl] = -1; // none yet
    }
    for (int i = t; i < p.max_iters; i += kBeginThreads) p.iter_counts[(size_t)inst * p.max_iters + i] = 0;
    for (int f = t; f < kFBins; f += kBeginThreads) {
        s_hist[f] = 0;
        if (!split) ((unsigned *)p.topgen)[(size_t)inst * kFBins + f] = 0;
    }
    if (!split) return;
    for (int depth = 0;; ++depth) {
        __syncthreads();
        const int a = depth & 1;
        const unsigned n = min(s_n[a], (unsigned)p.capl);
        const Item *in = (a ? lvl1 : lvl0) + at;
        Item *out = (a ? lvl0 : lvl1) + at;
        unsigned long long *li = a ? lp1 : lp0, *lo = a ? lp0 : lp1;
        __syncthreads(); // s_n is read
        if (t == 0) s_n[a] = 0;
        if (n >= target || depth >= max_depth) {
            for (unsigned j = t; j < n; j += kBeginThreads) {
                ((Item *)p.frontier)[at + j] = in[j];
                if (li) ((unsigned long long *)p.fpath)[at + j] = li[at + j];
            }
            if (t == 0) {
                ((unsigned *)p.nfront)[inst] = n;
                ((int *)p.top_goal)[inst] = s_goal;
            }
            for (int f = t; f < kFBins; f += kBeginThreads) ((unsigned *)p.topgen)[(size_t)inst * kFBins + f] = s_hist[f];
            return;
        }
        for (unsigned j = t; j < n; j += kBeginThreads)
            split_expand<W, HEUR>(
                p, P, inst, in[j], out, li ? li + at + j : nullptr, lo ? lo + at : nullptr,
                [&](unsigned k) { return atomicAdd(&s_n[a ^ 1], k); },
                [&](int f, unsigned k) { atomicAdd(&s_hist[f], k); }, [&](int f) { atomicMin(&s_goal, f); });
    }
}

// The words of a solve's waves: no lane has a context, no wave waits.
__global__ void __launch_bounds__(256) k_clear_waves(KParams p, unsigned n_list) {
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i < (unsigned)p.n_lanes) p.c_st[i] = ST_IDLE;
    if (i < (unsigned)p.n_lanes >> 6) {
        p.ticket[i] = 0;
        p.mail_head[(size_t)i * kLine] = 0;
    }
    if (i < n_list) p.list[i] = 0;
}

// Boards given as bytes (row-major, W*W per board, `bytes` 16-byte aligned and
// readable up to a multiple of 16): each is checked -- a permutation, and one
// that moves reach from the goal: its inversions and the blank's row + column
// have the same parity -- and its heuristic goes to h[i], or the packed board
// with it to items[i]; thr and tgt (null: none) are copied along.  A bad board
// sets *bad and stands as the goal board.  The input may be host memory: a
// block reads its bytes once, 16 at a time, into LDS.  Bound by that transfer
// (40,003 boards, 1.0 MB: 20 us; the host's check and packing of them took
// 3 ms).
template <int W, int HEUR>
__global__ void __launch_bounds__(256) k_boards(const uint8_t *bytes, int n, const PdbGeo *geo_g, const uint8_t *pdb,
                                                const int *thr, const float *tgt, Item *items, int *thr_d,
                                                float *tgt_d, int *h, unsigned *bad) {
    constexpr int N2 = W * W;
    __shared__ PdbGeo geo_s;
    __shared__ uint4 raw[256 * N2 / 16];
    PdbCtx P{&geo_s, pdb};
    load_geo<HEUR>(geo_s, geo_g);
    const int t = threadIdx.x, i = (int)blockIdx.x * 256 + t;
    const int here = min(256, n - (int)blockIdx.x * 256);
    const uint4 *src = (const uint4 *)(bytes + (size_t)blockIdx.x * (256 * N2));
    for (int k = t; k < (here * N2 + 15) / 16; k += 256) raw[k] = src[k];
    const int th = thr && t < here ? thr[i] : 0;
    const float tg = tgt && t < here ? tgt[i] : 0.f;
    __syncthreads();
    if (t >= here) return;
    const uint8_t *b = (const uint8_t *)raw + t * N2;
    uint32_t seen = 0;
    int inv = 0, blank = 0;
    bool ok = true;
    uint64_t lo = 0, hi = 0; // cells 0-11 and 12-23 of width 5; width 4 in lo
#pragma unroll
    for (int c = 0; c < N2; ++c) {
        const uint32_t v = b[c];
        ok &= v < (uint32_t)N2 && !((seen >> (v & 31u)) & 1u);
        inv += __popc(seen >> (v & 31u)); // the greater ones before it
        seen |= 1u << (v & 31u);
        blank = v ? blank : c;
        if constexpr (W == 4)
            lo |= (uint64_t)(v & 15u) << (4 * c);
        else if (c < 24)
            (c < 12 ? lo : hi) |= (uint64_t)(v & 31u) << (5 * (c % 12));
    }
    ok &= ((inv ^ (blank / W + blank % W)) & 1) == 0;
    Board<W> bd;
    if constexpr (W == 4) {
        bd.b = lo;
    } else {
        bd.lo = lo;
        bd.hi = hi;
        bd.top = b[24];
    }
    if (!ok) {
        *bad = 1u;
        if constexpr (W == 4) {
            bd.b = 0xfedcba9876543210ull;
        } else {
            bd.lo = bd.hi = 0;
            bd.top = 24;
            for (int c = 0; c < 24; ++c) (c < 12 ? bd.lo : bd.hi) |= (uint64_t)c << (5 * (c % 12));
        }
        blank = 0;
    }
    int v = 0;
    if constexpr (HEUR == 0) {
        for (int c = 0; c < N2; ++c) {
            const int x = bd.tile(c);
            if (x) v += abs(c / W - trow<W>(x)) + abs(c % W - tcol<W>(x));
        }
    } else {
        HState<1> hs;
        pdb_init(P, hs, bd);
        v = hs.h;
    }
    if (h) h[i] = v;
    if (items) {
        Item it;
        bd.pack(it.b);
        it.meta = meta_pack(blank, 0, v, DIR_NONE);
        it.inst = it.x0 = it.x1 = 0;
        items[i] = it;
    }
    if (thr) thr_d[i] = th;
    if (tgt) tgt_d[i] = tg;
}

hipError_t launch_boards(int width, int heur, const uint8_t *bytes, int n, const PdbGeo *geo, const uint8_t *pdb,
                         const int *thr, const float *tgt, Item *items, int *thr_d, float *tgt_d, int *h,
                         unsigned *bad, hipStream_t s) {
    auto *const k = width == 4 ? &k_boards<4, 0> : heur == 0 ? &k_boards<5, 0> : &k_boards<5, 1>;
    hipLaunchKernelGGL(k, dim3((unsigned)(((size_t)n + 255) / 256)), dim3(256), 0, s, bytes, n, geo, pdb, thr, tgt,
                       items, thr_d, tgt_d, h, bad);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// host-side launchers
size_t round_lds_bytes(int width, int maxd, int wg, int heur);

template <int W, int HEUR>
// With t0/t1 the runtime records the two events with the dispatch itself, so
// their interval is the kernel's own duration (no launch gap before it).
static hipError_t launch_round_t(const KParams &p, const PdbGeo *geo, int wg, hipStream_t s, hipEvent_t t0,
                                 hipEvent_t t1) {
    size_t lds = round_lds_bytes(W, p.maxd, wg, HEUR);
    auto *const k = p.prof ? &k_round<W, HEUR, true> : &k_round<W, HEUR, false>;
    if (t0 && t1)
        hipExtLaunchKernelGGL(k, dim3(p.n_lanes / wg), dim3(wg), (uint32_t)lds, s, t0, t1, 0u, p, geo);
    else
        hipLaunchKernelGGL(k, dim3(p.n_lanes / wg), dim3(wg), lds, s, p, geo);
    return hipGetLastError();
}

hipError_t launch_round(int width, int heur, const KParams &p, const PdbGeo *geo, int wg, hipStream_t s,
                        hipEvent_t t0, hipEvent_t t1) {
    if (width == 4) return launch_round_t<4, 0>(p, geo, wg, s, t0, t1);
    if (heur == 0) return launch_round_t<5, 0>(p, geo, wg, s, t0, t1);
    return launch_round_t<5, 1>(p, geo, wg, s, t0, t1);
}

// dynamic LDS of k_round: the stack levels, then (width 5) the boards, then
// (PDB) the sibling-value cache
size_t round_lds_bytes(int width, int maxd, int wg, int heur) {
    return (size_t)maxd * wg * (heur == 1 ? 2 : 1) + (width == 5 ? (size_t)kLdsBoardBytes * wg + kLdsBoardPad : 0) +
           (heur == 1 ? (size_t)kSibLevels * 4 * wg : 0);
}

const void *round_kernel_ptr(int width, int heur) {
    if (width == 4) return (const void *)&k_round<4, 0, false>;
    if (heur == 0) return (const void *)&k_round<5, 0, false>;
    return (const void *)&k_round<5, 1, false>;
}

hipError_t launch_turn(int width, int heur, const KParams &p, const PdbGeo *geo, bool spec, hipStream_t s) {
    if (p.n_inst == 1) {
        auto *const k = width == 4 ? &k_turn<4, 0> : heur == 0 ? &k_turn<5, 0> : &k_turn<5, 1>;
        hipLaunchKernelGGL(k, dim3(1), dim3(kRestartThreads), 0, s, p, geo, spec ? 1 : 0);
        return hipGetLastError();
    }
    if (spec) hipLaunchKernelGGL(k_spec, dim3(1), dim3(256), 0, s, p);
    auto *const k = width == 4 ? &k_restart<4, 0> : heur == 0 ? &k_restart<5, 0> : &k_restart<5, 1>;
    hipLaunchKernelGGL(k, dim3(p.n_inst), dim3(kRestartThreads), 0, s, p, geo);
    hipLaunchKernelGGL(k_control, dim3(1), dim3(64), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_split_level(int width, int heur, const KParams &p, const PdbGeo *geo, const Item *lvl_in,
                              const unsigned *n_in, Item *lvl_out, unsigned *n_out, int *frozen, int depth,
                              int max_depth, unsigned target, const unsigned long long *lp_in,
                              unsigned long long *lp_out, hipStream_t s) {
    const size_t total = (size_t)p.n_inst * p.capl;
    auto *const k = width == 4 ? &k_split_level<4, 0> : heur == 0 ? &k_split_level<5, 0> : &k_split_level<5, 1>;
    hipLaunchKernelGGL(k, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, p, geo, lvl_in, n_in, lvl_out, n_out,
                       frozen, depth, max_depth, target, lp_in, lp_out);
    return hipGetLastError();
}

hipError_t launch_begin(int width, int heur, const KParams &p, const PdbGeo *geo, Item *lvl0, Item *lvl1,
                        unsigned *nlvl0, int *frozen, int max_depth, unsigned target, unsigned long long *lp0,
                        unsigned long long *lp1, bool split, unsigned n_list, hipStream_t s) {
    const unsigned most = (unsigned)p.n_lanes > n_list ? (unsigned)p.n_lanes : n_list;
    hipLaunchKernelGGL(k_clear_waves, dim3((most + 255) / 256), dim3(256), 0, s, p, n_list);
    auto *const k = width == 4 ? &k_begin<4, 0> : heur == 0 ? &k_begin<5, 0> : &k_begin<5, 1>;
    hipLaunchKernelGGL(k, dim3(p.n_inst), dim3(kBeginThreads), 0, s, p, geo, lvl0, lvl1, nlvl0, frozen, max_depth,
                       target, lp0, lp1, split ? 1 : 0);
    return hipGetLastError();
}

} // namespace spz
