// persist.hpp -- matrix-resident kernels: a square block matrix cut into
// parts of rows, one workgroup per part and at most one part per CU, all
// parts resident at once, so that a sequence of products runs in one launch
// with the matrix held in registers.
//
// The parts are balls of the node graph (grown breadth first on the host,
// once per pattern): a part of 104 rows of the 200k-tet cylinder has a halo
// of about 250 nodes, against 470 to 800 for 104 consecutive rows.  A row has
// a group of 4 to 64 lanes, each holding U of its blocks.
//
// Between products the parts exchange the entries of the vector that their
// neighbours' blocks touch (the halo) through global memory.  On eight XCDs
// an ordinary store stays in the writer's L2, so the exchange uses agent-scope
// relaxed atomics (write-through stores, loads that miss the L2s), and every
// 8-byte word carries half a value and half a tag, the epoch it belongs to: a
// reader polls the words it needs until their tags match, one trip through
// memory, with no flag, no fence and no grid-wide barrier.  (Measured, 256
// workgroups: a barrier on one counter 3.9 us, on eight counters under a
// master 2.25 us; a product step with drained stores and per-part flags 6.0
// us, with tagged words 3.6 us,
// start and end of the kernel included.)
//
// Two buffers alternate.  A part writes step s + 2 over step s only after it
// has read its neighbours' step s + 1, which they write after reading all of
// step s: the pattern must be structurally symmetric, so that whoever reads a
// part is also read by it.
//
// Every wait is bounded: a lane that has polled for kWaitTicks raises the
// abort flag, its workgroup ends, and all others end at their next wait; the
// caller then takes the path of one launch per product, and so do some solves
// after it (Parts::rest).  A workgroup that
// gives up also sets the solver's own flag (stop, done) for the launches
// already queued, and leaving frees its CU for one that had to wait: a
// workgroup may start while the flags change, so one lane reads them for all
// (leave_at_start).  Giving up happens only
// when the parts are not resident together (another kernel that itself waits
// holds CUs); ResidentTurn keeps two such kernels of one process apart.
#pragma once

#include "internal.hpp"

#include <mutex>

namespace svfsi {

// Device view of a partition.  Row r of part b (in lane order) is node
// rowId[rowOff[b] + r], and rowOff[b] + r is its position in the exchange
// buffer.  lane: per lane of the part its row | log2(lanes of the row) << 16,
// -1 for none; a row's lanes are consecutive and aligned to their number.
struct PartsDev {
    const int* rowOff;          // G+1
    const int* rowId;           // nNo
    const int* laneOff;         // G+1
    const int* lane;
    const int* hOff;            // G+1 offsets into hPos
    const int* hPos;            // halo: positions in the exchange buffer
    const unsigned short* lcol; // per block: local index of its column, own rows first, then the halo
    unsigned long long* xb;     // 16 tagged words per node
    unsigned long long* red;    // partials of two sums over all parts, 2 G words each
    unsigned long long wait;    // ticks before a waiting lane gives up
    int G;
};

constexpr unsigned long long kWaitTicks = 100000000ull; // 1 s of the 100 MHz wall clock

template <typename T>
__device__ __forceinline__ T ld_agent(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// At a kernel's entry, by all lanes: whether the workgroup leaves, the flag set
// by an earlier launch or, when parts give up, by this one.  The lanes must
// agree, since those that stay index with LDS that all of them fill.  Clears
// *bad, the workgroup's own give-up flag.
__device__ __forceinline__ bool leave_at_start(const int* flag, int* bad)
{
    __shared__ int leave;
    if (threadIdx.x == 0) {
        leave = ld_agent(flag);
        *bad = 0;
    }
    __syncthreads();
    return leave != 0;
}

// 32 bits of payload under a tag
__device__ __forceinline__ void put_word(unsigned long long* p, unsigned v, unsigned tag)
{
    st_agent(p, ((unsigned long long)tag << 32) | v);
}

// Polls the N words p[m] (null: skipped) until each carries tag, payloads to
// v.  false: gave up, or another workgroup has.
template <int N>
__device__ __forceinline__ bool get_words(const unsigned long long* const (&p)[N], unsigned tag, unsigned (&v)[N],
                                          unsigned long long wait, int* abortFlag)
{
    unsigned long long t0 = 0;
    for (int n = 1;; ++n) {
        unsigned long long w[N];
#pragma unroll
        for (int m = 0; m < N; ++m) w[m] = p[m] ? ld_agent(p[m]) : ((unsigned long long)tag << 32);
        bool all = true;
#pragma unroll
        for (int m = 0; m < N; ++m) {
            all = all && (unsigned)(w[m] >> 32) == tag;
            v[m] = (unsigned)w[m];
        }
        if (all) return true;
        if ((n & 63) == 0 || wait == 0) {
            if (ld_agent(abortFlag)) return false;
            const unsigned long long t = wall_clock64();
            if (!t0) t0 = t;
            if (t - t0 >= wait) {
                st_agent(abortFlag, 1);
                return false;
            }
        }
    }
}

// A partition of a pattern for kernels that hold U blocks per lane.
struct Parts {
    int G = 0, U = 0, maxOwn = 0, maxHalo = 0, maxLanes = 0;
    unsigned epoch = 0; // the last tag used; xb starts out with tag 0
    long long launches = 0, giveUps = 0; // svfsi_resident_stats
    // After a give-up the next `rest` solves go without; 16, and four times as
    // many after each give-up in a row, up to 65,536: a passing contention costs
    // a second and 16 slower solves, a lasting one a few seconds in an hour
    int rest = 0, row = 0;
    void gave_up()
    {
        ++giveUps;
        rest = 16 << 2 * row;
        if (row < 6) ++row;
    }
    void solved() { row = 0; }
    unsigned long long wait = kWaitTicks;
    size_t ldsMax = 0;
    DBuf tab, xb;
    size_t at[7] = {}; // of rowOff, rowId, laneOff, lane, hOff, hPos, lcol in tab
    size_t red = 0;    // of the sums' words in xb, 2 G per sum
    PartsDev dev() const
    {
        const int* t = tab.as<int>();
        unsigned long long* x = xb.as<unsigned long long>();
        return {t + at[0], t + at[1], t + at[2], t + at[3], t + at[4], t + at[5],
                reinterpret_cast<const unsigned short*>(t + at[6]), x, x + red, wait, G};
    }
};

// Partitions L if its pattern fits the chip (at the end of FSILS_LHS_CREATE).
void persist_build(Lhs& L);
// The partition of L for a solve, asked for once by it; nullptr when there is
// none, the path is off or resting after a give-up, or (pcg) the kernels of
// pcg.hip do not fit it.
Parts* persist_parts(Lhs& L, bool pcg);

// A solve that launches matrix-resident kernels, from enter to leave (or its
// end).  Kernels of two such solves on different streams would wait for each
// other's CUs, so each launch is put behind what the other solves of the device
// and process have queued so far, by events on the device: the solves' other
// kernels overlap, no host thread waits, and a solve that is alone pays a
// mutex.  Streams named by hipStreamPerThread, which another thread cannot
// name, take turns solve by solve instead.
struct ResidentTurn {
    int dev = -1;
    hipStream_t s = nullptr;
    ResidentTurn *prev = nullptr, *next = nullptr;
    ResidentTurn() = default;
    ResidentTurn(const ResidentTurn&) = delete;
    ResidentTurn& operator=(const ResidentTurn&) = delete;
    ~ResidentTurn() { leave(); }
    bool enter(hipStream_t stream);
    void leave();
    // launch() with no other resident launch of the device between the events
    // and it
    template <class F>
    int launch(F&& f)
    {
        std::lock_guard<std::mutex> g(mutex());
        SV_TRY(follow_others());
        return f();
    }

private:
    std::mutex& mutex() const;
    int follow_others();
};

// z = p(B) D^-1 q, all factors of the polynomial preconditioner in one
// launch (ppoly.hip).  ops: nOps pairs (mode, factor) of SpMV steps as
// launch_poly's; lastLin: the closing linear factor without a product, or -1.
int ppoly_launch(Lhs& L, Parts& P, int dof, const float* B, const float* dinv, const double* q, float* z, double* z64,
                 const double* coef, const int* ops, int nOps, int lastLin, int* stop, int* abortFlag,
                 hipStream_t s);
size_t ppoly_lds(const Parts& P); // its dynamic LDS

// `its` iterations of CGRADV (dof 3) and of CGRAD_SCHUR in one launch
// (pcg.hip), from X, R, Pv and *st on to them; Parts with U = 3.
struct CgState;
int pcg3_launch(Lhs& L, Parts& P, const double* K, double* X, double* R, double* Pv, CgState* st, int its,
                hipStream_t s);
int pcgs_launch(Lhs& L, Parts& P, const double* Lm, const double* G, const double* Gt, double* X, double* R,
                double* Pv, CgState* st, int its, hipStream_t s);
size_t pcg_lds(const Parts& P); // their dynamic LDS
// whether they fit: their static LDS is below 512 bytes, and the sums were
// measured with at most 256 partials
inline bool pcg_fits(const Parts& P)
{
    return P.U == 3 && P.G <= 256 && pcg_lds(P) + 512 <= P.ldsMax;
}
// iterations per launch: about 2 ms, with the matrix read once
constexpr int kPcgChunk = 256;

} // namespace svfsi
