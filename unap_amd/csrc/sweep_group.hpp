// sweep_group.hpp -- whole DIC / DILU and Gauss-Seidel sweeps in one launch,
// run by a group of workgroups that step through the level schedule together.
//
// A level-scheduled sweep launched level by level costs about 5 us a level
// (launch, drain, cold start) whatever the level holds, and the one-workgroup
// tail has one CU's gather rate.  Here a group of resident workgroups walks
// all levels (and all sweeps of a smoothing call) behind a barrier of its own.
// On one XCD that barrier is a store and a poll in the L2 that its CUs share:
// 0.2 us a hop and 0.3 us in all, against 0.4 us a hop across XCDs and 0.25 us
// for one returning atomic (11 ns apart on one address, so counting arrivals
// or handing out rows by atomics would cost more than the levels).
//
// Joining.  A launch holds more workgroups than take part.  Each one that
// starts reads the XCD it runs on and registers there (on one XCD: the first
// to arrive elects its own, and the others leave); the first closes the list
// when all expected are in, or a few microseconds later.  Only registered, and
// therefore running, workgroups take part, so no barrier ever waits for a
// workgroup that has no place on the device, and the work is split by the
// number that registered.  A wait that never ends all the same (a fault in
// this scheme) gives up after some seconds.  That is reported to the host, and
// from then on nothing waits long: the workgroup that gave up goes through its
// remaining steps with a poll a wait, the others see the failure in theirs, and
// the launches queued behind leave at once, until the host has reported the
// error.
//
// Visibility.  Values that cross workgroups (the swept vector, the flags) are
// read with agent-scope loads, which pass the CU's own cache; the group on one
// XCD stores them to the L2 those loads are answered from, a wider group
// through it (agent scope).  A wavefront waits for its stores' acknowledgement
// before its workgroup raises its flag.
#pragma once

#include "group_steps.hpp"
#include "ops.hpp"

namespace unap_hip {

constexpr int kXcds = 8;
constexpr int kGroupPerXcd = 32;         // workgroups of one XCD that may take part
constexpr unsigned kGroupClosed = 1u << 31;
constexpr int kWaitLimit = 1 << 23;      // polls before a wait gives up (seconds)
constexpr int kWaitLook = 1 << 14;       // polls between looks at the failure word (milliseconds)

// Words written by different workgroups at different times lie on lines of
// their own; words polled together share one.  The words of the list are zero
// between launches.  The steps are never reset: they count on from launch to
// launch (epoch), because an XCD's own flags stay dirty in its L2, and a reset
// from another XCD would be undone when they are written back.  What a word
// left from earlier launches may hold: group_steps.hpp.
template <typename W>
struct GroupWords {
    W flag[kXcds][kGroupPerXcd];    // step reached, by workgroup
    W xflag[32];                    // step reached, by XCD
    W go[kXcds][128 / sizeof(W)];   // step the XCD's workgroups may start
};
struct GroupSync {
    unsigned elect[32];
    unsigned exits[32];
    unsigned reg[kXcds][32];             // registered workgroups
    unsigned count[32];                  // 1 + the number that takes part, by XCD
    GroupStep epoch[16];                 // steps of all launches before; top bit: a wait gave up
    GroupWords<unsigned> next;           // for a launch's steps (group_steps.hpp)
    GroupWords<GroupStep> first;         // for the meeting before them, or the first
};

struct GroupCtl {
    GroupSync* s;
    int* fail;   // host word: a wait gave up
    int expect;  // workgroups the group is meant to have
    int limit;   // polls before a wait gives up
};

// A workgroup's place: ranks run through the XCDs in turn, so that neighbouring
// ranks share an L2.  rank < 0: it takes no part.
struct Group {
    int rank, size;
    int xcd, local, localSize;
    unsigned xcds;    // bit x: XCD x takes part
    GroupStep epoch;  // this launch's steps count from here
};

template <typename T>
__device__ __forceinline__ T groupPeek(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T gld(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Stores of a group on one XCD stop at its L2; a wider group's go through it.
template <bool One, typename T>
__device__ __forceinline__ void gst(T* p, T v) {
    if constexpr (One)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A workgroup's waits on others, by one wavefront (all lanes together).  What
// lies between two polls and after the last is part of a step's chain: one
// counter runs through all waits, and what decides about giving up stands
// apart.  (With a count and a state a wait, the sweeps on all XCDs took 3%
// longer; with four polls a turn of the loop, 6%.)
struct Waits {
    int limit;          // polls before a wait gives up
    GroupStep* failed;  // device (top bit) and host words of that
    int* fail;
    int polls;          // until the next look
    int left = 0;       // of the limit, for the wait at step `at`
    unsigned at = ~0u;
    bool over = false;  // a wait has given up
    __device__ __forceinline__ Waits(int l, GroupStep* d, int* h)
        : limit(l), failed(d), fail(h), polls(min(l, kWaitLook)) {}
    // Until done(), or given up; s: the step waited for.
    template <class Done>
    __device__ __forceinline__ void until(unsigned s, Done&& done) {
        while (!done()) {
            if (__builtin_expect(--polls >= 0, 1)) continue;
            look(s);
            if (over) return;
        }
    }
    __device__ void look(unsigned s) {
        polls = 0;  // once it is over, a wait's first poll looks and returns
        if (s != at) {
            at = s;
            left = limit;
        }
        left -= kWaitLook;
        over = groupBroken(groupPeek(failed));
        if (over) return;
        if (left >= 0) {
            polls = kWaitLook;
            return;
        }
        over = true;
        __hip_atomic_fetch_or(failed, kGroupBroken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *fail = 1;
    }
};

template <bool One>
__device__ __forceinline__ Group groupJoin(const GroupCtl& c) {
    __shared__ Group sg;
    if (threadIdx.x < 64) {  // the first wavefront, all lanes together
        GroupSync* S = c.s;
        const int lane = (int)threadIdx.x;
        const unsigned xcd = __builtin_amdgcn_s_getreg((31 << 11) | 20) & (kXcds - 1);  // HW_REG_XCC_ID
        unsigned mine = kGroupClosed;
        bool leader = false;
        if (lane == 0) {
            // one XCD: the first arrival's; all: the first arrival closes the list
            unsigned old = 0u;
            const unsigned me = One ? 1u + xcd : 1u;
            __hip_atomic_compare_exchange_strong(&S->elect[0], &old, me, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            if (!One || old == 0u || old == me)
                mine = __hip_atomic_fetch_add(&S->reg[xcd][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            leader = old == 0u;
        }
        mine = __builtin_amdgcn_readfirstlane(mine);
        leader = __builtin_amdgcn_readfirstlane((int)leader) != 0;
        bool in = !(mine & kGroupClosed) && mine < (unsigned)kGroupPerXcd;
        unsigned count = 0u;  // lane x < 8: 1 + XCD x's workgroups
        if (leader) {
            const long long t0 = wall_clock64();  // 100 MHz
            for (;;) {
                unsigned r = lane < kXcds ? groupPeek(&S->reg[lane][0]) : 0u;
#pragma unroll
                for (int o = kXcds / 2; o >= 1; o >>= 1) r += __shfl_xor(r, o, 64);
                if (__builtin_amdgcn_readfirstlane(r) >= (unsigned)c.expect || wall_clock64() - t0 >= 400) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (lane < kXcds) {
                const unsigned r = __hip_atomic_fetch_or(&S->reg[lane][0], kGroupClosed, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT);
                count = 1u + (r < (unsigned)kGroupPerXcd ? r : (unsigned)kGroupPerXcd);
                __hip_atomic_store(&S->count[lane], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if (in) {
            Waits w(c.limit, &S->epoch[0], c.fail);
            w.until(0u, [&] {
                count = groupPeek(&S->count[lane & (kXcds - 1)]);
                if (!__any(count == 0u)) return true;
                __builtin_amdgcn_s_sleep(1);
                return false;
            });
            in = !w.over;
        }
        Group g{-1, 0, (int)xcd, (int)mine, 0, 0u, 0};
        if (in) {
            int before = 0;
#pragma unroll
            for (int x = 0; x < kXcds; ++x) {
                const int k = (int)__builtin_amdgcn_readlane(count, x) - 1;
                if (x < (int)xcd) before += k;
                if (x == (int)xcd) g.localSize = k;
                g.size += k;
                if (k > 0) g.xcds |= 1u << x;
            }
            g.epoch = groupPeek(&S->epoch[0]);  // but for the top bit, changed by the launch's last workgroup only
            if (g.local < g.localSize && !groupBroken(g.epoch)) g.rank = before + g.local;
        }
        if (lane == 0) sg = g;
    }
    __syncthreads();
    return sg;
}

// The end of a workgroup's part in a launch of `steps` steps, participant or
// not: the last workgroup of the launch clears the list and moves the epoch.
__device__ __forceinline__ void groupLeave(const GroupCtl& c, GroupStep steps) {
    __syncthreads();
    if (threadIdx.x != 0) return;
    GroupSync* S = c.s;
    if (__hip_atomic_fetch_add(&S->exits[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1u) return;
    auto put = [](auto* p, auto v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    put(&S->epoch[0], groupPeek(&S->epoch[0]) + steps);
    for (int x = 0; x < kXcds; ++x) {
        put(&S->reg[x][0], 0u);
        put(&S->count[x], 0u);
    }
    put(&S->elect[0], 0u);
    put(&S->exits[0], 0u);
}

// Waits until the word this lane watches is at least s, for every lane (lanes
// with none to watch take the workgroup's or XCD's own).
template <typename W>
__device__ __forceinline__ void groupAwait(Waits& wait, const W* p, W s) {
    wait.until((unsigned)s, [&] { return !__any(!groupReached(groupPeek(p), s)); });
}
// Step s of the group's barrier, by one wavefront of each workgroup.  Across
// XCDs it goes by XCD: their first workgroups meet for the others, so that a
// step's traffic between L2s is eight words rather than every flag to every L2.
template <bool One, typename W>
__device__ __forceinline__ void groupMeet(Waits& wait, const Group& g, GroupWords<W>& w, W s) {
    const int lane = (int)threadIdx.x & 63;
    if (lane == 0) gst<true>(&w.flag[g.xcd][g.local], s);
    const W* flag = &w.flag[g.xcd][lane < g.localSize ? lane : g.local];
    if constexpr (One) {
        groupAwait<W>(wait, flag, s);
        return;
    }
    if (g.local != 0) {
        groupAwait<W>(wait, &w.go[g.xcd][0], s);
        return;
    }
    groupAwait<W>(wait, flag, s);
    if (lane == 0) gst<false>(&w.xflag[g.xcd], s);
    groupAwait<W>(wait, &w.xflag[lane < kXcds && (g.xcds >> lane & 1u) ? lane : g.xcd], s);
    if (lane == 0) gst<true>(&w.go[g.xcd][0], s);
}

// Roles of a workgroup's wavefronts.  The watcher raises the workgroup's flag
// and polls the others'.  The sweepers compute.  The loaders copy what the
// sweepers will need besides the swept values from the packed table into an
// LDS ring, two items ahead, by direct loads (no registers, no arithmetic).
// A step's length is the chain flag -> gather -> arithmetic -> store -> flag,
// in which a lone wavefront's every instruction counts: so the table holds
// each lane's data ready to use, and what a sweeper can prepare falls between
// the two barriers of a step, while the watcher polls.
//
// Items.  A level's rows go to the workgroups in runs of whole groups (the
// rows of one wavefront); a workgroup takes its run kSweepers groups at a
// time, one such round being an item.  The group's barrier follows the last
// item of a level, the workgroup's own follows every item.
constexpr int kGroupLevels = 512;  // levels of a launch (bounds kept in LDS)
constexpr int kRing = 2;

struct GroupLevel {
    int first, count;  // this workgroup's groups in the table
    int row;           // first row (schedule position) of them
    int passes;        // items of the level, the same for every workgroup
};

// Fills this workgroup's runs for levels [0, nl) of start / grp0 (schedule
// bounds and table groups).
template <int RW, int NS>
__device__ __forceinline__ void groupRuns(const Group& g, GroupLevel* lev, int* end, const int* start, const int* grp0,
                                          int nl) {
    for (int k = (int)threadIdx.x; k < nl; k += (int)blockDim.x) {
        const int g0 = grp0[k], ng = grp0[k + 1] - g0;
        const int chunk = (ng + g.size - 1) / g.size;
        const int f = min(g.rank * chunk, ng);
        lev[k] = {g0 + f, min(chunk, ng - f), start[k] + f * RW, (chunk + NS - 1) / NS};
        end[k] = start[k + 1];
    }
}

// Level k's run in scalar registers (k is the same for the whole wavefront).
__device__ __forceinline__ GroupLevel groupLevel(const GroupLevel* lev, int k) {
    const GroupLevel L = lev[k];
    return {__builtin_amdgcn_readfirstlane(L.first), __builtin_amdgcn_readfirstlane(L.count),
            __builtin_amdgcn_readfirstlane(L.row), __builtin_amdgcn_readfirstlane(L.passes)};
}
__device__ __forceinline__ int groupWave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// Walks the items of a launch: the nl levels of the list, `rounds` times over
// (Gauss-Seidel sweeps).  Uniform over the wavefront.
struct GroupWalk {
    const GroupLevel* lev;
    const int* end;
    int nl;
    int k, ps, left;  // level of the list, item of the level, levels still to come (< 0: past the end)
    GroupLevel L;     // level k
    int stop;         // its last row + 1
    __device__ __forceinline__ void level() {
        L = groupLevel(lev, k);
        stop = __builtin_amdgcn_readfirstlane(end[k]);
    }
    __device__ __forceinline__ GroupWalk(const GroupLevel* l, const int* e, int n, int rounds)
        : lev(l), end(e), nl(n), k(0), ps(0), left(n * rounds - 1) {
        level();
    }
    __device__ __forceinline__ bool done() const { return left < 0; }
    __device__ __forceinline__ bool lastOfLevel() const { return ps + 1 >= L.passes; }
    __device__ __forceinline__ void next() {
        if (left < 0) return;
        if (!lastOfLevel()) {
            ++ps;
            return;
        }
        ps = 0;
        k = k + 1 == nl ? 0 : k + 1;
        if (--left >= 0) level();
    }
    // Sweeper tw's row (schedule position) for its lane-row wr of RW, or -1.
    template <int RW, int NS>
    __device__ __forceinline__ int row(int tw, int wr) const {
        const int at = tw + ps * NS;
        const int q = L.row + at * RW + wr;
        return left >= 0 && at < L.count && q < stop ? q : -1;
    }
};

// Sets a workgroup's words of the launch's steps (by its first wavefront,
// which then has other loads to wait for).
__device__ __forceinline__ void groupWords(const GroupCtl& c, const Group& g) {
    if (threadIdx.x != 0) return;
    const unsigned e = (unsigned)g.epoch;
    GroupWords<unsigned>& w = c.s->next;
    gst<true>(&w.flag[g.xcd][g.local], e);
    if (g.local != 0) return;
    gst<false>(&w.xflag[g.xcd], e);
    gst<true>(&w.go[g.xcd][0], e);
}
// The watcher's part.  On one XCD the group meets on the 64-bit words before
// the first step, while the loaders fill the ring.  Across XCDs a meeting takes
// longer than that (4 us more a launch), so it is the first step's own.
template <bool One>
__device__ __forceinline__ void groupWatch(const GroupCtl& c, const Group& g, GroupWalk t) {
    Waits wait(c.limit, &c.s->epoch[0], c.fail);
    unsigned s = (unsigned)g.epoch;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the words are set before the others know
    if constexpr (One) groupMeet<One>(wait, g, c.s->first, g.epoch + 1);
    __syncthreads();
    __syncthreads();
    for (;;) {
        const bool last = t.lastOfLevel();
        t.next();
        if (t.done()) return;
        __builtin_amdgcn_s_barrier();
        if (last) {
            if (!One && s == (unsigned)g.epoch)
                groupMeet<One>(wait, g, c.s->first, g.epoch + 1);
            else
                groupMeet<One>(wait, g, c.s->next, s + 1u);
            ++s;
        }
        __syncthreads();
    }
}

// A loader's part: wavefront j of NL copies its share of the P pieces (64
// lanes x 16 bytes) of the sweepers' groups.
template <int NS, int NL, int P>
__device__ __forceinline__ void groupLoad(const uint4* tab, uint4 (&ring)[kRing][NS][P][64], GroupWalk t, int j) {
    const int lane = (int)threadIdx.x & 63;
    int slot = 0;
    auto copy = [&]() __attribute__((always_inline)) {
        const int left = t.L.count - t.ps * NS;  // groups of this item that exist
        const uint4* src = tab + (size_t)(t.L.first + t.ps * NS) * P * 64 + lane;
        for (int pc = j; pc < min(left, NS) * P; pc += NL)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(src + (size_t)pc * 64),
                (__attribute__((address_space(3))) void*)(&ring[slot][0][0][0] + pc * 64), 16, 0, 0);
        slot = slot + 1 == kRing ? 0 : slot + 1;
    };
    GroupWalk u = t;
    copy();
    t.next();
    if (!t.done()) copy();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // items 0 and 1 are in the ring
    __syncthreads();  // the sweepers have taken item 0
    for (;;) {
        // while item u runs: item u + 2.  The copies of item u + 1, issued an
        // item ago, are waited for here, before the barrier they must precede.
        // Bare barriers: __syncthreads would wait for the new copies too.
        u.next();
        if (u.done()) return;
        t.next();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (!t.done()) copy();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
    }
}

// ----------------------------------------------------------- packed tables
// What a lane needs of a matrix row, 16 bytes a piece, piece p of group g at
// tab[(g P + p) 64 + lane]: written once for the matrix's values, read
// straight into LDS.
template <typename T>
struct GroupPack;
template <>
struct GroupPack<double> {
    static constexpr int kGs = 4, kOvf = 3, kLu = 5;
};
template <>
struct GroupPack<float> {
    static constexpr int kGs = 3, kOvf = 2, kLu = 4;
};
__device__ __forceinline__ uint4 pack2(double a, double b) {
    uint4 u;
    double d[2] = {a, b};
    __builtin_memcpy(&u, d, 16);
    return u;
}
__device__ __forceinline__ void unpack2(const uint4& u, double& a, double& b) {
    double d[2];
    __builtin_memcpy(d, &u, 16);
    a = d[0];
    b = d[1];
}
__device__ __forceinline__ unsigned bitsOf(float f) { return __float_as_uint(f); }

constexpr int kGsS = 4;  // Gauss-Seidel entries a lane and chunk
// One chunk of a row's entries: columns, then coefficients.
template <typename T>
__device__ __forceinline__ void packEntries(const int (&c)[kGsS], const T (&v)[kGsS], uint4* out) {
    out[0] = make_uint4((unsigned)c[0], (unsigned)c[1], (unsigned)c[2], (unsigned)c[3]);
    if constexpr (sizeof(T) == 8) {
        out[64] = pack2(v[0], v[1]);
        out[128] = pack2(v[2], v[3]);
    } else {
        out[64] = make_uint4(bitsOf(v[0]), bitsOf(v[1]), bitsOf(v[2]), bitsOf(v[3]));
    }
}
template <typename T>
__device__ __forceinline__ void unpackEntries(const uint4* in, unsigned (&o)[kGsS], T (&v)[kGsS]) {
    const uint4 c = in[0];
    o[0] = c.x;
    o[1] = c.y;
    o[2] = c.z;
    o[3] = c.w;
    if constexpr (sizeof(T) == 8) {
        unpack2(in[64], v[0], v[1]);
        unpack2(in[128], v[2], v[3]);
    } else {
        const uint4 q = in[64];
        v[0] = __uint_as_float(q.x);
        v[1] = __uint_as_float(q.y);
        v[2] = __uint_as_float(q.z);
        v[3] = __uint_as_float(q.w);
    }
}

// Gauss-Seidel table: lane i of a row's LPR lanes holds entries i, i + LPR,
// ...; the last piece holds the diagonal, the entry count and where the row's
// further entries start in the overflow table (chunks of LPR kGsS entries).
// grp: first row and row count of every group; grpOvf: its first overflow chunk.
template <int LPR, typename T>
__global__ void __launch_bounds__(256) kPackGs(DMat<T> A, const int2* __restrict__ grp, const int* __restrict__ grpOvf,
                                               int ng, uint4* __restrict__ tab, uint4* __restrict__ ovf) {
    const int g = blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    if (g >= ng) return;
    constexpr int P = GroupPack<T>::kGs, PO = GroupPack<T>::kOvf;
    const int i = lane % LPR, wr = lane / LPR;
    const bool on = wr < grp[g].y;
    const int r = grp[g].x + (on ? wr : 0);
    const int n = on ? (int)(A.rowInfo[r] & 0xffffu) : 0;
    const long long base = A.sliceStart[r >> kSliceShift] + (r & (kSliceRows - 1));
    const T diag = on ? A.diag[r] : (T)1;
    auto chunk = [&](int t0, uint4* out) __attribute__((always_inline)) {
        int c[kGsS];
        T v[kGsS];
#pragma unroll
        for (int m = 0; m < kGsS; ++m) {
            const int t = t0 + i + LPR * m;
            const long long p = base + ((long long)(t < n ? t : 0) << kSliceShift);
            c[m] = t < n ? A.col[p] : r;  // an absent entry reads the row's own value: no address is read by all
            v[m] = t < n ? A.val[p] : (T)0;
        }
        packEntries<T>(c, v, out);
    };
    uint4* out = tab + (size_t)g * P * 64 + lane;
    chunk(0, out);
    if constexpr (sizeof(T) == 8) {
        uint4 u = pack2(diag, 0.0);
        u.z = (unsigned)n;
        u.w = (unsigned)grpOvf[g];
        out[(P - 1) * 64] = u;
    } else {
        out[(P - 1) * 64] = make_uint4(bitsOf(diag), 0u, (unsigned)n, (unsigned)grpOvf[g]);
    }
    for (int ch = 0; __any(n > (ch + 1) * LPR * kGsS); ++ch)
        chunk((ch + 1) * LPR * kGsS, ovf + ((size_t)(grpOvf[g] + ch) * PO) * 64 + lane);
}

// DIC / DILU table, one lane a row: columns and coefficients of the first
// kLuS entries of the sweep's side, the entry count and the row.  rows null:
// position = row.  Forward entries are the row's first `mid`; the backward
// copy holds all its entries in sweep order.
constexpr int kLuS = 6;
template <typename T>
__global__ void __launch_bounds__(256) kPackLu(DMat<T> M, const int* __restrict__ rows, int fwd,
                                               const int2* __restrict__ grp, int ng, uint4* __restrict__ tab) {
    const int g = blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    if (g >= ng) return;
    constexpr int P = GroupPack<T>::kLu;
    const bool on = lane < grp[g].y;
    const int q = grp[g].x + (on ? lane : 0);
    const int r = rows ? rows[q] : q;
    const int at = fwd ? r : q;
    const uint32_t info = M.rowInfo[at];
    const int n = !on ? 0 : (fwd ? (int)(info >> 16) : (int)(info & 0xffffu));
    const long long base = M.sliceStart[at >> kSliceShift] + (at & (kSliceRows - 1));
    int c[kLuS];
    T v[kLuS];
#pragma unroll
    for (int j = 0; j < kLuS; ++j) {
        const long long p = base + ((long long)(j < n ? j : 0) << kSliceShift);
        c[j] = j < n ? M.col[p] : r;
        v[j] = j < n ? M.val[p] : (T)0;
    }
    uint4* out = tab + (size_t)g * P * 64 + lane;
    out[0] = make_uint4((unsigned)c[0], (unsigned)c[1], (unsigned)c[2], (unsigned)c[3]);
    out[64] = make_uint4((unsigned)c[4], (unsigned)c[5], (unsigned)n, (unsigned)r);
    if constexpr (sizeof(T) == 8) {
        out[128] = pack2(v[0], v[1]);
        out[192] = pack2(v[2], v[3]);
        out[256] = pack2(v[4], v[5]);
    } else {
        out[128] = make_uint4(bitsOf(v[0]), bitsOf(v[1]), bitsOf(v[2]), bitsOf(v[3]));
        out[192] = make_uint4(bitsOf(v[4]), bitsOf(v[5]), 0u, 0u);
    }
}

// ------------------------------------------------------------- DIC / DILU
// The levels are the forward ones, then the backward ones.  The arithmetic of
// a row is fwdRow's / bwdRow's: its first value is rD r (forward) or its
// forward value, gathered (backward); then (rD coef) w is subtracted entry by
// entry.
constexpr int kLuSweepers = 8, kLuLoaders = 5;
constexpr int kLuThreads = 64 * (1 + kLuSweepers + kLuLoaders);
template <typename T>
struct GroupLu {
    DMat<T> F, B;  // entries past the packed ones: forward by row, backward by position
    const uint4* tab;
    const int* grp0;      // groups before each level, forward then backward (one list of nFwd + nBwd + 1)
    const int* fwdStart;
    const int* bwdStart;
    int nFwd, nBwd;
    const T* r;
    const T* rD;
    const T* rDpos;  // rD by backward position
    T* w;
};

template <bool One, typename T>
__global__ void __launch_bounds__(kLuThreads) kGroupLu(GroupLu<T> a, GroupCtl c, Skip sk) {
    if (sk.on()) return;
    constexpr int P = GroupPack<T>::kLu, NS = kLuSweepers;
    __shared__ uint4 ring[kRing][NS][P][64];
    __shared__ GroupLevel lev[kGroupLevels];
    __shared__ int end[kGroupLevels];
    const Group g = groupJoin<One>(c);
    if (g.rank >= 0) {
        const int nl = a.nFwd + a.nBwd;
        groupWords(c, g);
        groupRuns<64, NS>(g, lev, end, a.fwdStart, a.grp0, a.nFwd);
        groupRuns<64, NS>(g, lev + a.nFwd, end + a.nFwd, a.bwdStart, a.grp0 + a.nFwd, a.nBwd);
        __syncthreads();
        const int wave = groupWave(), lane = (int)threadIdx.x & 63;
        GroupWalk t(lev, end, nl, 1);
        if (wave == 0) {
            groupWatch<One>(c, g, t);
        } else if (wave <= NS) {
            const int tw = wave - 1;
            // an item's position in the schedule and the factors of its first value, two items ahead
            struct Lead {
                int q;
                bool bwd;
                T rd, in;
            };
            auto ahead = [&]() __attribute__((always_inline)) {
                Lead v{t.row<64, NS>(tw, lane), t.k >= a.nFwd, (T)0, (T)0};
                const T* d = v.bwd ? a.rDpos : a.rD;
                if (v.q >= 0) {
                    v.rd = d[v.q];
                    if (!v.bwd) v.in = a.r[v.q];
                }
                t.next();
                return v;
            };
            unsigned o[kLuS];
            T f[kLuS], init = (T)0;
            int n = 0, r = 0, slot = 0;
            bool longer = false, active = false;
            Lead cur, n1 = ahead(), n2 = ahead();
            auto take = [&]() __attribute__((always_inline)) {
                cur = n1;
                n1 = n2;
                const uint4* in = &ring[slot][tw][0][lane];
                slot = slot + 1 == kRing ? 0 : slot + 1;
                const uint4 c0 = in[0], c1 = in[64];
                o[0] = c0.x;
                o[1] = c0.y;
                o[2] = c0.z;
                o[3] = c0.w;
                o[4] = c1.x;
                o[5] = c1.y;
                if constexpr (sizeof(T) == 8) {
                    unpack2(in[128], f[0], f[1]);
                    unpack2(in[192], f[2], f[3]);
                    unpack2(in[256], f[4], f[5]);
                } else {
                    const uint4 v0 = in[128], v1 = in[192];
                    f[0] = __uint_as_float(v0.x);
                    f[1] = __uint_as_float(v0.y);
                    f[2] = __uint_as_float(v0.z);
                    f[3] = __uint_as_float(v0.w);
                    f[4] = __uint_as_float(v1.x);
                    f[5] = __uint_as_float(v1.y);
                }
                n = (int)c1.z;
                r = (int)c1.w;
#pragma unroll
                for (int j = 0; j < kLuS; ++j) f[j] = cur.rd * f[j];
                init = cur.rd * cur.in;
                active = __any(cur.q >= 0);
                longer = active && __any(n > kLuS);
                n2 = ahead();
            };
            __syncthreads();  // items 0 and 1 are in the ring
            take();
            __syncthreads();
            GroupWalk u(lev, end, nl, 1);
            u.next();
            for (;;) {
                if (active) {
                    // absent entries subtract +0, which leaves any value as it is
                    T x[kLuS];
#pragma unroll
                    for (int j = 0; j < kLuS; ++j) x[j] = gld(a.w + o[j]);
                    const T own = gld(a.w + (unsigned)r);
                    T acc = cur.bwd ? own : init;
#pragma unroll
                    for (int j = 0; j < kLuS; ++j) acc = acc - (j < n ? f[j] * x[j] : (T)0);
                    if (longer && n > kLuS) {
                        const DMat<T>& M = cur.bwd ? a.B : a.F;
                        const int at = cur.bwd ? cur.q : r;
                        const long long base = M.sliceStart[at >> kSliceShift] + (at & (kSliceRows - 1));
                        for (int k = kLuS; k < n; ++k) {
                            const long long p = base + ((long long)k << kSliceShift);
                            acc = acc - (cur.rd * M.val[p]) * gld(a.w + M.col[p]);
                        }
                    }
                    if (cur.q >= 0) gst<One>(a.w + (unsigned)r, acc);
                }
                if (u.done()) break;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stored, before the flag
                __syncthreads();
                take();
                u.next();
                __syncthreads();
            }
        } else {
            groupLoad<NS, kLuLoaders, P>(a.tab, ring, t, wave - 1 - NS);
        }
    }
    groupLeave(c, (GroupStep)(a.nFwd + a.nBwd));
}

// ------------------------------------------------------------ Gauss-Seidel
// LPR lanes a row.  Lane i multiplies its entries; the products are exchanged
// through LDS and subtracted in entry order (gsRow's arithmetic).
constexpr int kGsSweepers = 10, kGsLoaders = 5;
constexpr int kGsThreads = 64 * (1 + kGsSweepers + kGsLoaders);
template <typename T>
struct GroupGs {
    const uint4* tab;
    const uint4* ovf;
    const int* grp0;
    const int* start;
    int nl, nSweeps;
    T* x;
    const T* b;
};

// Subtracts a chunk's products from acc in entry order; absent entries
// subtract +0, which leaves every value as it is.
template <int LPR, typename T>
__device__ __forceinline__ T groupGsSub(const T (&v)[kGsS], const T (&x)[kGsS], int left, int i, T acc, T* mine,
                                        const T* group) {
#pragma unroll
    for (int m = 0; m < kGsS; ++m) mine[m * 64] = i + LPR * m < left ? v[m] * x[m] : (T)0;
    __builtin_amdgcn_wave_barrier();
    // entry LPR m + j is slot m of lane j of the row
#pragma unroll
    for (int m = 0; m < kGsS; ++m) {
        if (m > 0 && !__any(LPR * m < left)) break;
#pragma unroll
        for (int j = 0; j < LPR; ++j) acc = acc - group[m * 64 + j];
    }
    __builtin_amdgcn_wave_barrier();
    return acc;
}

template <bool One, int LPR, typename T>
__global__ void __launch_bounds__(kGsThreads) kGroupGs(GroupGs<T> a, GroupCtl c, Skip sk) {
    if (sk.on()) return;
    constexpr int RW = 64 / LPR, NS = kGsSweepers, P = GroupPack<T>::kGs, PO = GroupPack<T>::kOvf;
    __shared__ uint4 ring[kRing][NS][P][64];
    __shared__ T buf[NS * 64 * kGsS];
    __shared__ GroupLevel lev[kGroupLevels];
    __shared__ int end[kGroupLevels];
    const Group g = groupJoin<One>(c);
    if (g.rank >= 0) {
        groupWords(c, g);
        groupRuns<RW, NS>(g, lev, end, a.start, a.grp0, a.nl);
        __syncthreads();
        const int wave = groupWave(), lane = (int)threadIdx.x & 63;
        GroupWalk t(lev, end, a.nl, a.nSweeps);
        if (wave == 0) {
            groupWatch<One>(c, g, t);
        } else if (wave <= NS) {
            const int tw = wave - 1, i = lane % LPR, wr = lane / LPR;
            T* mine = buf + tw * 64 * kGsS + lane;
            const T* group = buf + tw * 64 * kGsS + (lane - i);
            struct Lead {  // an item's row and right-hand side, two items ahead
                int r;
                T b;
            };
            auto ahead = [&]() __attribute__((always_inline)) {
                Lead v{t.row<RW, NS>(tw, wr), (T)0};
                if (v.r >= 0) v.b = a.b[v.r];
                t.next();
                return v;
            };
            unsigned o[kGsS], oo[kGsS];
            T v[kGsS], vv[kGsS], diag = (T)1;
            int n = 0, slot = 0, chunk = 0;
            bool longer = false, active = false;
            Lead cur, n1 = ahead(), n2 = ahead();
            auto more = [&](int ch) __attribute__((always_inline)) {
                unpackEntries<T>(a.ovf + ((size_t)(chunk + ch) * PO) * 64 + lane, oo, vv);
            };
            auto take = [&]() __attribute__((always_inline)) {
                cur = n1;
                n1 = n2;
                const uint4* in = &ring[slot][tw][0][lane];
                slot = slot + 1 == kRing ? 0 : slot + 1;
                unpackEntries<T>(in, o, v);
                const uint4 d = in[(P - 1) * 64];
                if constexpr (sizeof(T) == 8) {
                    double unused;
                    unpack2(d, diag, unused);
                } else {
                    diag = __uint_as_float(d.x);
                }
                n = (int)d.z;
                chunk = (int)d.w;
                active = __any(cur.r >= 0);  // a slot without a group holds anything
                longer = active && __any(n > LPR * kGsS);
                if (longer) more(0);  // the first further chunk, on its way while the watcher polls
                n2 = ahead();
            };
            __syncthreads();  // items 0 and 1 are in the ring
            take();
            __syncthreads();
            GroupWalk u(lev, end, a.nl, a.nSweeps);
            u.next();
            for (;;) {
                if (active) {
                    T x[kGsS], xx[kGsS];
#pragma unroll
                    for (int m = 0; m < kGsS; ++m) x[m] = gld(a.x + o[m]);
                    if (longer) {
#pragma unroll
                        for (int m = 0; m < kGsS; ++m) xx[m] = gld(a.x + oo[m]);
                    }
                    T acc = groupGsSub<LPR>(v, x, n, i, cur.b, mine, group);
                    if (longer) {
                        acc = groupGsSub<LPR>(vv, xx, n - LPR * kGsS, i, acc, mine, group);
                        for (int ch = 1; __any(n > (ch + 1) * LPR * kGsS); ++ch) {
                            more(ch);
#pragma unroll
                            for (int m = 0; m < kGsS; ++m) xx[m] = gld(a.x + oo[m]);
                            acc = groupGsSub<LPR>(vv, xx, n - (ch + 1) * LPR * kGsS, i, acc, mine, group);
                        }
                    }
                    if (cur.r >= 0 && i == 0) gst<One>(a.x + (unsigned)cur.r, acc / diag);
                }
                if (u.done()) break;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stored, before the flag
                __syncthreads();
                take();
                u.next();
                __syncthreads();
            }
        } else {
            groupLoad<NS, kGsLoaders, P>(a.tab, ring, t, wave - 1 - NS);
        }
    }
    groupLeave(c, (GroupStep)a.nl * (GroupStep)a.nSweeps);
}

}  // namespace unap_hip
