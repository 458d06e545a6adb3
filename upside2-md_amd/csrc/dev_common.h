// Device helpers shared by the engine kernels: block reductions, the B-spline
// and sigmoid primitives of the reference (src/spline.h, src/vector_math.h),
// and the fixed-order gather that replaces scatter-with-atomics.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include "engine_dev.h"

namespace upside {

// Address-space-typed pointers.  Arena and table pointers reach the device
// code through descriptors, so the compiler sees them as generic (flat)
// pointers: every flat load is counted against both the vector-memory and
// the LDS counters and waits serialise.  Device code therefore holds them as
// global (gp, global_load) or LDS (lp, ds_read) pointers.  Descriptors and
// programs are constant while a kernel runs: they are read through the
// constant address space (cp), so that a record at a workgroup-uniform address
// arrives in scalar registers through the scalar cache, which the team
// barriers do not invalidate.
#define UPS_GLOBAL __attribute__((address_space(1)))
#define UPS_LDS __attribute__((address_space(3)))
#define UPS_CONST __attribute__((address_space(4)))
template <class T> using gp = UPS_GLOBAL T*;
template <class T> using lp = UPS_LDS T*;
template <class T> using cp = UPS_CONST const T*;
template <class T> __device__ __forceinline__ gp<T> gmem(T* p) { return (gp<T>)p; }
template <class T> __device__ __forceinline__ cp<T> cmem(const T* p) { return (cp<T>)p; }
using OpC = UPS_CONST const OpRec;
using GraphC = UPS_CONST const PairGraph;
using RotC = UPS_CONST const RotamerDev;
using SysC = UPS_CONST const SysDesc;

// Arena pointers.  What one workgroup of a team writes to the system's arenas,
// the others read after the next team barrier.  Every load from an arena goes
// past the CU's L1 to the L2 of its XCD (buffer loads with sc1, agent scope:
// 90 ns against 52 for an L1 hit and the same as an L1 miss, measured by a
// pointer chase), so a barrier does not have to invalidate L1 (see team_sync).
// A pointer is a buffer resource that starts at its array (so that only one
// array, not an arena, has to be smaller than 4 GB; as fast as one resource an
// arena with a scalar offset) and a lane's offset.
constexpr int AUX_SC1 = 16;                   // cache policy bits of a buffer access
constexpr int RSRC_FLAGS = 0x00027000;        // raw buffer of 32-bit data
template <class T> struct Unconst { using type = T; };
template <class T> struct Unconst<const T> { using type = T; };
template <class T> struct ap {
    using V = typename Unconst<T>::type;
    gp<V> p;
    __amdgpu_buffer_rsrc_t r;
    int o;
    __device__ __forceinline__ V load() const {
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, o * 4, 0, AUX_SC1));
    }
    struct Ref {
        ap a;
        __device__ __forceinline__ operator V() const { return a.load(); }
        __device__ __forceinline__ V operator=(V v) const { *a.ptr() = v; return v; }
        __device__ __forceinline__ V operator=(const Ref& b) const { return *this = (V)b; }
        __device__ __forceinline__ V operator+=(V v) const { return *this = a.load() + v; }
    };
    // for atomics and stores
    __device__ __forceinline__ gp<V> ptr() const { return p + o; }
    __device__ __forceinline__ ap operator+(int k) const { ap q = *this; q.o += k; return q; }
    __device__ __forceinline__ Ref operator[](int k) const { return Ref{*this + k}; }
    __device__ __forceinline__ operator ap<const V>() const { return ap<const V>{p, r, o}; }
    // N consecutive elements, and added to.  (A load is not moved across a store
    // to an arena, so elements are loaded together before any is stored.)
    template <int N> __device__ __forceinline__ void get(V* v) const {
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = (*this + k).load();
    }
    template <int N> __device__ __forceinline__ void add(const V* v) const {
        V x[N];
        get<N>(x);
#pragma unroll
        for (int k = 0; k < N; ++k) (*this)[k] = x[k] + v[k];
    }
};
// Read only: an element is its value.
template <class T> struct ap<const T> {
    gp<T> p;
    __amdgpu_buffer_rsrc_t r;
    int o;
    __device__ __forceinline__ ap operator+(int k) const { ap q = *this; q.o += k; return q; }
    __device__ __forceinline__ T operator[](int k) const {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (o + k) * 4, 0, AUX_SC1));
    }
    template <int N> __device__ __forceinline__ void get(T* v) const {
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = (*this)[k];
    }
};
// A whole arena; offsets added to it are uniform.
template <class T> struct Arena {
    gp<T> p;
    __device__ __forceinline__ ap<T> operator+(int k) const {
        return ap<T>{p + k, __builtin_amdgcn_make_buffer_rsrc((T*)(p + k), 0, -1, RSRC_FLAGS), 0};
    }
    __device__ __forceinline__ typename ap<T>::Ref operator[](int k) const { return (*this + k)[0]; }
    // Data at k that nobody writes while it is read, through L1: only after
    // l1_drop.  For records of a few cache lines read piece by piece (an edge's
    // matrix): past L1 every 16-byte piece is a request to L2 of its own.
    __device__ __forceinline__ gp<const T> cached(int k) const { return p + k; }
};

// A value every lane holds alike, as a scalar.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float unif(float v) { return __int_as_float(uni(__float_as_int(v))); }
__device__ __forceinline__ unsigned long long uni64(unsigned long long v) {
    const unsigned lo = (unsigned)uni((int)(unsigned)v), hi = (unsigned)uni((int)(unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// The team that runs the current ops: G workgroups with a common arrival
// counter (G = 1: one workgroup, no grid barriers).  Data-parallel loops
// stride over the team's threads (gtid, gsize); team_sync separates phases
// whose data cross workgroups.
struct Team {
    unsigned long long bar_next;  // count that opens this workgroup's next barrier on `bar`
    int tpar;          // buffer parity of the next reduction
    int rank, G;       // workgroup rank in the team, team size (rank is the fourth word: sync_store)
    int gsize;         // team threads
    int err;           // int arena offset of the error word this team sets
    lp<int> lost;      // LDS word of the workgroup: a wait of its ended without the others (team_sync)
    gp<unsigned long long> bar;   // arrival counter
    gp<float> tred;    // reduction scratch, 2 buffers of G floats
    unsigned long long* prof;  // wall-clock accumulators (null: profiling off)
};

// Execution context of one workgroup.  Everything here is uniform over the
// workgroup except tid and gtid.  Functions that take a Ctx are inlined into
// the few outlined phase functions of the kernel (PHASE), and within one a
// context is a set of scalar registers: ctx_load reads it from LDS at the
// phase's start.  (Passed by reference it lives in private memory, and every
// phase began by reloading it from L2, when a team barrier still dropped L1.
// Measured with the program records in scalar registers, ms per step: 0.55 ->
// 0.47 for 67 residues on 8 workgroups, 1.03 -> 0.95 for 500 on 32.)
struct Ctx : Team {
    Arena<float> A;        // per-system float arena
    Arena<int> I;          // per-system int arena
    gp<const float> CF;    // constant float arena
    gp<const int> CI;      // constant int arena
    cp<SysDesc> S;         // the system
    cp<RunArgs> args;      // the launch's arguments
    gp<unsigned> bar_flag; // team barrier spin-timeout flag
    lp<float> red;         // LDS reduction scratch [NWAVE]
    lp<int> ired;          // LDS reduction scratch [NWAVE] (ints)
    lp<float> lds;         // LDS staging area [LDS_FLOATS]
    int pbase;             // first fixed profile slot
    int cur_op;            // program op being run (team barriers are counted per op while profiling)
    int local;             // the whole team runs on one XCD (shares one L2)
    int bp_layout;         // where rotamer solves run (see bp_on_one_wg)
    unsigned spin_limit;   // RunArgs::spin_limit
    int tid, gtid;         // thread in the workgroup, in the team (not kept in LDS)
};

// Threads of a team are numbered wave by wave across its workgroups, so that a
// phase with fewer elements than threads still runs on every CU (numbered
// workgroup by workgroup, 1000 residues' 3000 angles of a part of 8 workgroups
// are 47 waves on 6 CUs; 300 residues with warm solves 0.700 -> 0.677 ms per
// step, an evaluation of 101 residues 1432 -> 1371 us).
__device__ __forceinline__ int team_tid(int rank, int G, int tid) { return ((tid >> 6) * G + rank) * 64 + (tid & 63); }

// sync_store keeps the words that barriers advance as the first four.
static_assert(__builtin_offsetof(Team, bar_next) == 0 && __builtin_offsetof(Team, tpar) == 8 &&
              __builtin_offsetof(Team, rank) == 12, "first 16 bytes of a context");

// The context in LDS, one copy per wave (no wave waits for another's): the
// current one, the whole team's while the current one is narrowed to a part of
// it, and the next barrier counts of the parts this workgroup belongs to.
constexpr int CTX_BYTES = sizeof(Ctx) - 2 * sizeof(int);
constexpr int CTX_WORDS = (CTX_BYTES + 15) / 16 * 4;
constexpr int CTX_ROOT = CTX_WORDS, CTX_NEXT = 2 * CTX_WORDS;
constexpr int CTX_WAVE = 2 * CTX_WORDS + 8;
constexpr int CTX_LOST = NWAVE * CTX_WAVE;  // Team::lost, after the waves' copies
constexpr int CTX_TOTAL = CTX_LOST + 4;
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lp<int> ctx_wave(lp<int> mem) { return mem + (int)(threadIdx.x >> 6) * CTX_WAVE; }
__device__ __forceinline__ void ctx_store(lp<int> mem, const Ctx& c, int at = 0) {
    int w[CTX_WORDS] = {};
    __builtin_memcpy(w, &c, CTX_BYTES);
    lp<i32x4> m = (lp<i32x4>)(ctx_wave(mem) + at);
#pragma unroll
    for (int k = 0; k < CTX_WORDS / 4; ++k) m[k] = i32x4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
}
// A workgroup whose team cannot meet ends here (all its waves: the word is set
// between two workgroup barriers, and every wave reads it at the same places).
__device__ __forceinline__ void leave_if(int lost) {
    if (uni(lost)) __builtin_amdgcn_endpgm();
}
__device__ __forceinline__ Ctx ctx_load(lp<int> mem, int at = 0) {
    int w[CTX_WORDS];
    lp<i32x4> m = (lp<i32x4>)(ctx_wave(mem) + at);
#pragma unroll
    for (int k = 0; k < CTX_WORDS / 4; ++k) {
        const i32x4 v = m[k];
#pragma unroll
        for (int q = 0; q < 4; ++q) w[4 * k + q] = uni(v[q]);
    }
    Ctx c;
    __builtin_memcpy(&c, w, CTX_BYTES);
    c.tid = (int)threadIdx.x;
    c.gtid = team_tid(c.rank, c.G, c.tid);
    return c;
}
// After barriers and reductions: the words they advance.
__device__ __forceinline__ void sync_store(lp<int> mem, const Ctx& c) {
    *(lp<i32x4>)ctx_wave(mem) = i32x4{(int)(unsigned)c.bar_next, (int)(unsigned)(c.bar_next >> 32), c.tpar, c.rank};
}
// End of a phase function: leaves the barrier state in LDS, gives back a result.
__device__ __forceinline__ int phase_ret(lp<int> mem, const Ctx& c, int value) {
    sync_store(mem, c);
    return value;
}

__device__ __forceinline__ unsigned long long ptick(const Ctx& c) { return c.prof ? wall_clock64() : 0ull; }
__device__ __forceinline__ void pacc(const Ctx& c, int slot, unsigned long long t0) {
    // a no-return atomic: the thread does not wait for the accumulator's line
    if (c.prof && c.gtid == 0)
        __hip_atomic_fetch_add(c.prof + c.pbase + slot, wall_clock64() - t0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Team barrier on a monotonic 64-bit arrival counter: arrival n of a team of
// G falls in barrier n / G, which opens when the counter reaches the next
// multiple of G.  Nothing is reset between barriers, and the counter is a
// multiple of G between launches (the host zeroes it when the team size
// changes).  Every workgroup keeps the count that opens its next barrier
// (bar_first at the start, then + G per barrier), so its arrival is a
// no-return atomic: it does not wait for the counter's old value before it
// starts polling.  A stale poll can only prolong a wait.
//   Memory ordering: a team spread over XCDs (separate L2s) needs
// device-scope fences (write back L2 before arriving, invalidate after the
// wait).  A team on one XCD shares its L2, and loads of what others wrote go to
// L2 (ap).  Either way every wave waits for its stores to be acknowledged by L2
// before the workgroup barrier, which does not wait for them.  On one XCD
// nothing is invalidated: a device-scope invalidate of L1 after the wait, with
// plain loads, is served by the shared L2 one CU after the other (a barrier of
// 2, 8, 16, 32 workgroups and reads of three others' data: 1.07, 1.38, 1.82,
// 2.92 us with it; 0.95, 0.92, 0.93, 1.12 without).
//   The wait is bounded (RunArgs::spin_limit): a workgroup that has polled that
// often, or sees that another of its team gave up, records a timeout and closes
// the counter for good (BAR_CLOSED), and so any other that it comes to
// (enter_sub, leave_sub): nobody passes a barrier on account of what it does
// without the others.  It goes on, waiting for nobody, to the next place where
// it reads `lost`, and ends there: where integers that others should have
// written would be taken as an index, an offset or a count (the pair lists,
// ahead of the edges, and the edges of a solve: list_sync, team_or,
// team_exscan; the exchange), and at the start of an evaluation.  In between it
// may compute floats from what others had not finished, which become an index
// nowhere there but through a clamp.  So a launch always drains, inside of its
// arrays; the host then reports the run as failed.  (Reading the word at every
// barrier, or at the start of every phase, costs up to 6 % of an evaluation of
// 10 residues or a step of 67.)

// s_waitcnt immediate: vmcnt(0), expcnt and lgkmcnt not waited on.
constexpr int WAIT_VMEM = 0x0F70;

// Set in a counter: as a signed number it is below every count (counts are
// compared signed), whoever still arrives.
constexpr unsigned long long BAR_CLOSED = 1ull << 63;

// Count that opens the first barrier of a team of G on counter `bar`, read
// before this workgroup's first arrival: fewer than G arrivals of that
// barrier can precede it (it cannot open without this workgroup), so the
// count rounded down to a multiple of G is the base.  (A closed counter: any
// count that it cannot reach.)
__device__ __forceinline__ unsigned long long bar_first(gp<unsigned long long> bar, int G) {
    const unsigned long long v = uni64(__hip_atomic_load(bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) & ~BAR_CLOSED;
    return (v / (unsigned long long)G + 1ull) * (unsigned long long)G;
}

__device__ __forceinline__ void close_bar(Ctx& c) {
    (void)__hip_atomic_fetch_or(c.bar, BAR_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void team_sync(Ctx& c) {
    // every wave's stores acknowledged by L2 before the team can observe the arrival
    if (c.G > 1) __builtin_amdgcn_s_waitcnt(WAIT_VMEM);
    __syncthreads();
    if (c.G > 1) {
        const unsigned long long target = c.bar_next;
        c.bar_next = target + (unsigned long long)c.G;
        if (c.tid == 0) {
            if (!c.local) __threadfence();
            (void)__hip_atomic_fetch_add(c.bar, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            unsigned spins = 0;
            while ((long long)__hip_atomic_load(c.bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (long long)target) {
                __builtin_amdgcn_s_sleep(2);
                // after one timeout anywhere in the team no barrier waits long,
                // so the launch drains quickly (a poll takes 241 ns with a look
                // at the flag, 190 without)
                if (__builtin_expect(++spins > c.spin_limit || (spins % 16 == 0 &&
                    __hip_atomic_load(c.bar_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u), 0)) {
                    __hip_atomic_store(c.bar_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    close_bar(c);
                    *c.lost = 1;
                    break;
                }
            }
            if (!c.local) __threadfence();
        }
        __syncthreads();
        asm volatile("" ::: "memory");  // no load of an arena is moved up or reused across
        // profiling: team barriers per op, after the fixed slots
        if (c.prof && c.tid == 0)
            __hip_atomic_fetch_add(c.prof + c.pbase + PROF_EXTRA + c.cur_op, 1ull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
}

// A barrier after which offsets or counts that others wrote are read.
__device__ __forceinline__ void list_sync(Ctx& c) {
    team_sync(c);
    if (c.G > 1) leave_if(*c.lost);
}

// Barrier over every workgroup of the launch that takes part in replica
// exchange (teams on different XCDs: device-scope fences on both sides), on a
// monotonic arrival counter as team_sync.  Bounded: a timeout sets the flag,
// which the host turns into an error, and the workgroups leave.
__device__ __forceinline__ void grid_sync(Ctx& c, UPS_CONST const RexDev& x) {
    __builtin_amdgcn_s_waitcnt(WAIT_VMEM);  // every wave's: thread 0's fence waits for its own wave's stores
    __syncthreads();
    leave_if(*c.lost);
    if (c.tid == 0) {
        __threadfence();
        unsigned long long old = __hip_atomic_fetch_add(x.grid_bar, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long long target = (old / (unsigned long long)x.n_wg + 1ull) * (unsigned long long)x.n_wg;
        unsigned spins = 0;
        while (__hip_atomic_load(x.grid_bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            __builtin_amdgcn_s_sleep(2);
            if (++spins > c.spin_limit ||
                __hip_atomic_load(x.grid_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
                __hip_atomic_store(x.grid_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                *c.lost = 1;
                break;
            }
        }
        __threadfence();
    }
    __syncthreads();
    leave_if(*c.lost);
}

// Drop the CU's L1, which may hold lines of the arenas from before other
// workgroups wrote them, ahead of cached reads.  All threads of the workgroup.
__device__ __forceinline__ void l1_drop(Ctx& c) {
    if (c.G == 1) return;  // nobody else writes this system's arenas
    if (c.tid == 0) asm volatile("buffer_inv sc1" ::: "memory");
    __syncthreads();
}

// Sub-teams: parts of a team that run beside each other, each with an arrival
// counter and reduction scratch of its own.  A workgroup belongs to the same
// part of each kind for a whole launch, so it keeps the kind's barrier count
// (two words at CTX_NEXT) from one use to the next.
enum SubTeam : int {
    SUB_REST = 0,   // ranks 1..G-1, beside rank 0's rotamer solve
    SUB_HALF = 1,   // ranks [0, G/2) and [G/2, G)
    SUB_QUARTER = 2 // ranks [j*G/4, (j+1)*G/4)
};
struct SubPart { int first, size, word, buf; };  // ranks, counter word, reduction buffer
__device__ __forceinline__ SubPart sub_part(int kind, int rank, int G) {
    if (kind == SUB_REST) return SubPart{1, G - 1, BAR_SUB1, 1};
    if (kind == SUB_HALF) return rank < G / 2 ? SubPart{0, G / 2, BAR_LO, 2} : SubPart{G / 2, G - G / 2, BAR_HI, 3};
    int j = 0;
    while (j + 1 < 4 && rank >= (j + 1) * G / 4) ++j;
    return SubPart{j * G / 4, (j + 1) * G / 4 - j * G / 4, BAR_Q + 2 * j, 4 + j};
}
__device__ __forceinline__ void sub_next_put(lp<int> mem, int kind, unsigned long long v) {
    lp<int> m = ctx_wave(mem) + CTX_NEXT + 2 * kind;
    m[0] = (int)(unsigned)v;
    m[1] = (int)(unsigned)(v >> 32);
}

// Narrow the context from the whole team to this workgroup's part of kind
// `kind`.  Each part's first workgroup keeps the profile accumulators `prof`,
// so that each part's ops are timed.
__device__ __forceinline__ void enter_sub(lp<int> mem, Ctx& c, int kind, gp<int> words, unsigned long long* prof) {
    ctx_store(mem, c, CTX_ROOT);
    const SubPart p = sub_part(kind, c.rank, c.G);
    lp<int> m = ctx_wave(mem) + CTX_NEXT + 2 * kind;
    c.bar_next = ((unsigned long long)(unsigned)uni(m[1]) << 32) | (unsigned)uni(m[0]);
    c.G = p.size;
    c.rank -= p.first;
    c.gtid = team_tid(c.rank, c.G, c.tid);
    c.gsize = p.size * NT;
    c.bar = (gp<unsigned long long>)(words + p.word);
    c.tred += p.buf * 2 * MAX_TEAM;
    c.tpar = 0;
    c.prof = c.rank == 0 ? prof : nullptr;
    if (uni(*c.lost) && c.tid == 0) close_bar(c);
}
// Back to the whole team.
__device__ __forceinline__ void leave_sub(lp<int> mem, Ctx& c, int kind) {
    sub_next_put(mem, kind, c.bar_next);
    c = ctx_load(mem, CTX_ROOT);
    ctx_store(mem, c);
    if (uni(*c.lost) && c.tid == 0) close_bar(c);
}

// XCD of the calling workgroup (hardware register XCC_ID).
__device__ __forceinline__ unsigned xcd_id() { return __builtin_amdgcn_s_getreg((15 << 11) | (0 << 6) | 20); }

// At launch start of a team: every workgroup records its XCD; the team uses
// L2-local barriers only if all agree.  All threads of the team.
__device__ __forceinline__ void team_place(Ctx& c, gp<int> xtab) {
    c.local = 0;
    if (c.G == 1) return;
    if (c.tid == 0) __hip_atomic_store(&xtab[c.rank], (int)xcd_id(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    team_sync(c);
    int same = 1;
    int x0 = __hip_atomic_load(&xtab[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int r = 1; r < c.G; ++r) same &= __hip_atomic_load(&xtab[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == x0;
    team_sync(c);  // every workgroup has read the table before it is rewritten
    c.local = uni(same);
    if (c.rank == 0 && c.tid == 0) xtab[-1] = same;  // reported to the host (barrier word 3)
}

__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Block sum in a fixed order (lane tree, then waves in index order): the
// result is the same on every run.  All threads must call it.
__device__ __forceinline__ float block_sum(Ctx& c, float v) {
    v = wave_sum(v);
    __syncthreads();  // the previous reduction has been read
    if ((c.tid & 63) == 0) c.red[c.tid >> 6] = v;
    __syncthreads();
    float t = 0.f;
    for (int w = 0; w < NWAVE; ++w) t += c.red[w];
    return unif(t);
}
__device__ __forceinline__ float block_max(Ctx& c, float v) {
    v = wave_max(v);
    __syncthreads();
    if ((c.tid & 63) == 0) c.red[c.tid >> 6] = v;
    __syncthreads();
    float t = c.red[0];
    for (int w = 1; w < NWAVE; ++w) t = fmaxf(t, c.red[w]);
    return unif(t);
}

// Team reductions: workgroup partials combined in rank order (fixed order, so
// the result is the same on every run).  All threads of the team.  The
// partials of all ranks (at most MAX_TEAM, one per lane) are read in one
// memory trip and combined from registers; a loop over them in memory pays a
// trip per unrolled group of ranks.
static_assert(MAX_TEAM <= 64, "one lane per rank");
// The partial of rank min(lane, G - 1), after all ranks have stored theirs.
__device__ __forceinline__ float team_partial(Ctx& c, float t) {
    gp<float> buf = c.tred + c.tpar * c.G;
    c.tpar ^= 1;
    if (c.tid == 0) buf[c.rank] = t;
    team_sync(c);
    return __hip_atomic_load(buf + min(c.tid & 63, c.G - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ float team_sum(Ctx& c, float v) {
    float t = block_sum(c, v);
    if (c.G == 1) return t;
    const float x = team_partial(c, t);
    float s = 0.f;
    for (int r = 0; r < c.G; ++r) s += lane_value(x, r);
    return unif(s);
}
__device__ __forceinline__ float team_max(Ctx& c, float v) {
    float t = block_max(c, v);
    if (c.G == 1) return t;
    return unif(wave_max(team_partial(c, t)));
}
__device__ __forceinline__ int team_or(Ctx& c, int v) {
    int t = uni(__syncthreads_or(v));
    if (c.G == 1) return t;
    const float x = team_partial(c, t ? 1.f : 0.f);
    leave_if(*c.lost);  // the answer decides whether lists are built
    return __any(x > 0.f) ? 1 : 0;
}

// In-place exclusive scan of the ints a[0..n) (any memory); returns the
// total.  Each thread scans a contiguous chunk, chunk totals are scanned
// across the block.  All threads must call it.
template <class P>
__device__ __forceinline__ int block_exscan(Ctx& c, P a, int n) {
    int per = (n + NT - 1) / NT;
    int b = c.tid * per, e = min(b + per, n);
    int s = 0;
    for (int i = b; i < e; ++i) s += a[i];
    int lane = c.tid & 63, w = c.tid >> 6;
    int v = s;
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    __syncthreads();
    if (lane == 63) c.ired[w] = v;
    __syncthreads();
    int before = 0, tot = 0;
    for (int k = 0; k < NWAVE; ++k) {
        int x = c.ired[k];
        if (k < w) before += x;
        tot += x;
    }
    int run = before + v - s;
    for (int i = b; i < e; ++i) {
        int x = a[i];
        a[i] = run;
        run += x;
    }
    __syncthreads();
    return tot;
}

// Team-wide in-place exclusive scan of the ints a[0..n) in global memory;
// returns the total.  Each workgroup scans a contiguous chunk, chunk totals
// are added in rank order.  All threads of the team.
template <class P>
__device__ __forceinline__ int team_exscan(Ctx& c, P a, int n) {
    int per = (n + c.G - 1) / c.G;
    int b = min(c.rank * per, n), e = min(b + per, n);
    int tot = uni(block_exscan(c, a + b, e - b));
    if (c.G == 1) return tot;
    const int lane = c.tid & 63;
    const int part = __float_as_int(team_partial(c, __int_as_float(tot)));
    leave_if(*c.lost);
    const int x = lane < c.G ? part : 0;
    int v = x;  // inclusive scan over the ranks
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    const int all = __builtin_amdgcn_readlane(v, 63);
    const int before = __builtin_amdgcn_readlane(v - x, c.rank);
    for (int i = b + c.tid; i < e; i += NT) a[i] += before;
    list_sync(c);
    return all;
}

// Sum over aligned groups of G lanes (G a power of two <= 64), fixed order;
// every lane of the group receives the group total.
template <int G>
__device__ __forceinline__ float group_sum(float v) {
    for (int o = G >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ---- splines (src/spline.h) -------------------------------------------------
// Uniform cubic B-spline with coefficient window p[xb-1 .. xb+2] at x>=1
// (first spline centred at -1, src/spline.h:98-127,242-256): value, derivative.
template <class P>
__device__ __forceinline__ void deboor(P p, float x, float& v, float& d) {
    int xb = (int)x;
    float y = x - (float)xb;
    P c = p + xb - 1;
    float c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
    float omy = 1.f - y, y2 = y * y, y3 = y2 * y;
    float w0 = omy * omy * omy * (1.f / 6.f);
    float w1 = (3.f * y3 - 6.f * y2 + 4.f) * (1.f / 6.f);
    float w2 = (-3.f * y3 + 3.f * y2 + 3.f * y + 1.f) * (1.f / 6.f);
    float w3 = y3 * (1.f / 6.f);
    v = w0 * c0 + w1 * c1 + w2 * c2 + w3 * c3;
    float e0 = -0.5f * omy * omy;
    float e1 = 1.5f * y2 - 2.f * y;
    float e2 = -1.5f * y2 + y + 0.5f;
    float e3 = 0.5f * y2;
    d = e0 * c0 + e1 * c1 + e2 * c2 + e3 * c3;
}

// Clamped variant (src/spline.h:326-358): constant outside [1, n_knot-2).
template <class P>
__device__ __forceinline__ void clamped_deboor(P p, float x, int n_knot, float& v, float& d) {
    if (!(x >= 1.f)) {  // also catches NaN, which must never index the table
        v = p[0] * (1.f / 6.f) + p[1] * (2.f / 3.f) + p[2] * (1.f / 6.f);
        d = 0.f;
    } else if (x >= (float)(n_knot - 2)) {
        v = p[n_knot - 3] * (1.f / 6.f) + p[n_knot - 2] * (2.f / 3.f) + p[n_knot - 1] * (1.f / 6.f);
        d = 0.f;
    } else {
        deboor(p, x, v, d);
    }
}

// 1/(1+exp(x)) and its derivative exp(x)/(1+exp(x))^2 (src/vector_math.h:683-690).
__device__ __forceinline__ void sigmoid(float x, float& v, float& d) {
    float z = expf(-x);
    float w = 1.f / (1.f + z);
    v = w;
    d = z * w * w;
}

// Compact sigmoid 0.25(y+2)(y-1)^2 with y = x*sharpness, 1 below -1, 0 above 1
// (src/vector_math.h:701-720).
template <typename S>
__device__ __forceinline__ void compact_sigmoid(S x, S sharp, S& v, S& d) {
    S y = x * sharp;
    v = S(0.25) * (y + S(2)) * (y - S(1)) * (y - S(1));
    d = (sharp * S(0.75)) * (y * y - S(1));
    if (y < S(-1)) { v = S(1); d = S(0); }
    if (y > S(1)) { v = S(0); d = S(0); }
}

// Periodic bicubic patch c[16] (value, d/dfx, d/dfy), src/spline.h:63-82.
template <class P>
__device__ __forceinline__ void bicubic(P c, float fx, float fy, float& v, float& dx, float& dy) {
    float fx2 = fx * fx, fx3 = fx * fx2, fy2 = fy * fy;
    float vx0 = c[0] + fy * (c[1] + fy * (c[2] + fy * c[3]));
    float vx1 = c[4] + fy * (c[5] + fy * (c[6] + fy * c[7]));
    float vx2 = c[8] + fy * (c[9] + fy * (c[10] + fy * c[11]));
    float vx3 = c[12] + fy * (c[13] + fy * (c[14] + fy * c[15]));
    float vy1 = c[1] + fx * (c[5] + fx * (c[9] + fx * c[13]));
    float vy2 = c[2] + fx * (c[6] + fx * (c[10] + fx * c[14]));
    float vy3 = c[3] + fx * (c[7] + fx * (c[11] + fx * c[15]));
    dx = vx1 + 2.f * fx * vx2 + 3.f * fx2 * vx3;
    dy = vy1 + 2.f * fy * vy2 + 3.f * fy2 * vy3;
    v = vx0 + fx * vx1 + fx2 * vx2 + fx3 * vx3;
}

template <class P>
__device__ __forceinline__ void quat_to_rot(P q, float* U) {
    float a = q[0], b = q[1], c = q[2], d = q[3];
    U[0] = a * a + b * b - c * c - d * d; U[1] = 2.f * b * c - 2.f * a * d; U[2] = 2.f * b * d + 2.f * a * c;
    U[3] = 2.f * b * c + 2.f * a * d; U[4] = a * a - b * b + c * c - d * d; U[5] = 2.f * c * d - 2.f * a * b;
    U[6] = 2.f * b * d - 2.f * a * c; U[7] = 2.f * c * d + 2.f * a * b; U[8] = a * a - b * b - c * c + d * d;
}

// Fixed-order gather (see engine_dev.h): each target row adds the sum of its
// contributions, in plan order.  A thread loads each contribution's index
// once and all its components with it (per component the terms are summed in
// plan order, as one component at a time would).  Called by all threads of
// the team; no barrier at the end.
template <int CW>
__device__ __forceinline__ void plan_gather_w(Ctx& c, gp<const int> off, gp<const int> idx, ap<float> sens,
                                              ap<const float> con, int nt, int ss, int col, int cs) {
    for (int t = c.gtid; t < nt; t += c.gsize) {
        const int b = off[t], e = off[t + 1];
        if (b == e) continue;
        float acc[CW];
#pragma unroll
        for (int k = 0; k < CW; ++k) acc[k] = 0.f;
#pragma unroll 2
        for (int j = b; j < e; ++j) {
            ap<const float> q = con + idx[j] * cs;
#pragma unroll
            for (int k = 0; k < CW; ++k) acc[k] += q[k];
        }
        (sens + (t * ss + col)).template add<CW>(acc);
    }
}

__device__ __forceinline__ void plan_gather(Ctx& c, int plan) {
    cp<int> h = (cp<int>)(c.CI + plan);  // the header is uniform: scalar loads
    int nt = h[0], cw = h[1], so = h[2], ss = h[3], col = h[4], cb = h[5], cs = h[6];
    gp<const int> off = c.CI + plan + PLAN_HDR;
    gp<const int> idx = off + nt + 1;
    ap<float> sens = c.A + so;
    ap<const float> con = c.A + cb;
    switch (cw) {
    case 1: plan_gather_w<1>(c, off, idx, sens, con, nt, ss, col, cs); break;
    case 2: plan_gather_w<2>(c, off, idx, sens, con, nt, ss, col, cs); break;
    case 3: plan_gather_w<3>(c, off, idx, sens, con, nt, ss, col, cs); break;
    case 6: plan_gather_w<6>(c, off, idx, sens, con, nt, ss, col, cs); break;
    default:
        for (int t = c.gtid; t < nt; t += c.gsize) {
            int b = off[t], e = off[t + 1];
            if (b == e) continue;
            for (int k = 0; k < cw; ++k) {
                float acc = 0.f;
                for (int j = b; j < e; ++j) acc += con[idx[j] * cs + k];
                sens[t * ss + col + k] += acc;
            }
        }
    }
}

}  // namespace upside
