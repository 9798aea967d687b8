// persist.cpp -- host side of the matrix-resident kernels (persist.hpp).
#include "persist.hpp"

#include <algorithm>
#include <atomic>
#include <climits>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>

namespace svfsi {

namespace {
struct Device {
    std::mutex mu;
    std::condition_variable cv;   // a solve has left
    ResidentTurn* turns = nullptr; // the solves between enter and leave
    hipEvent_t ev = nullptr;
};
constexpr int kDevices = 64;
Device g_dev[kDevices];
} // namespace

std::mutex& ResidentTurn::mutex() const { return g_dev[dev].mu; }

bool ResidentTurn::enter(hipStream_t stream)
{
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= kDevices) return false;
    Device& D = g_dev[d];
    std::unique_lock<std::mutex> g(D.mu);
    // nobody inside waits for anybody here, so this ends with their solves
    D.cv.wait(g, [&] {
        for (ResidentTurn* t = D.turns; t; t = t->next)
            if (stream == hipStreamPerThread || t->s == hipStreamPerThread) return false;
        return true;
    });
    dev = d;
    s = stream;
    prev = nullptr;
    next = D.turns;
    if (next) next->prev = this;
    D.turns = this;
    return true;
}

void ResidentTurn::leave()
{
    if (dev < 0) return;
    Device& D = g_dev[dev];
    {
        std::lock_guard<std::mutex> g(D.mu);
        (prev ? prev->next : D.turns) = next;
        if (next) next->prev = prev;
    }
    D.cv.notify_all();
    dev = -1;
}

// The device's event, made with its first partition: solves allocate nothing.
static int make_event()
{
    int d = 0;
    SV_HIP(hipGetDevice(&d));
    if (d < 0 || d >= kDevices) return SVFSI_OK; // no solve enters there
    std::lock_guard<std::mutex> g(g_dev[d].mu);
    if (!g_dev[d].ev) SV_HIP(hipEventCreateWithFlags(&g_dev[d].ev, hipEventDisableTiming));
    return SVFSI_OK;
}

// The streams of the others are alive: their solves are inside.  An event may be
// recorded again once a stream was told to wait for it.
int ResidentTurn::follow_others()
{
    Device& D = g_dev[dev];
    for (ResidentTurn* t = D.turns; t; t = t->next) {
        if (t == this || t->s == s) continue;
        SV_HIP(hipEventRecord(D.ev, t->s));
        SV_HIP(hipStreamWaitEvent(s, D.ev, 0));
    }
    return SVFSI_OK;
}

// LDS of k_ppoly: two exchange tables, halo positions
size_t ppoly_lds(const Parts& P)
{
    return (size_t)(P.maxOwn + P.maxHalo) * 32 + (size_t)P.maxHalo * 4;
}

// lanes of a row of n blocks: the smallest power of two from gMin on that
// holds them U each; 0: none up to 64
static int row_lanes(int n, int U, int gMin)
{
    int g = gMin;
    while (g <= 64 && g * U < n) g <<= 1;
    return g <= 64 ? g : 0;
}

// U blocks per lane and rows of at least gMin lanes; P.G stays 0 when the
// pattern does not fit.
//
// Part of FSILS_LHS_CREATE, so that every solve of a pattern takes the same
// path: about 3.5 ms for the 200k-tet cylinder (8.5 with the halos found by one
// thread).
static int build(Lhs& L, Parts& P, int U, int gMin, int cus, size_t ldsMax)
{
    const std::vector<int>& rp = L.hRowPtr;
    const std::vector<int>& cp = L.hColPtr;
    const int n = L.nNo;
    long long total = 0;
    for (int i = 0; i < n; ++i) {
        const int g = row_lanes(rp[i + 1] - rp[i], U, gMin);
        if (!g) return SVFSI_OK;
        total += g;
    }
    // half a workgroup's lanes per part until every CU has one
    long long G = (total + 511) / 512;
    if (G > cus) G = cus;
    const int target = (int)((total + G - 1) / G);
    if (target > 1024) return SVFSI_OK;
    // balls of the node graph: breadth first from a node that the last part
    // reached and left, a part closed once it has its share of the lanes.
    // stamp: 1 + the part that queued a node last, INT_MAX once it is taken
    std::vector<unsigned char> lg(n);
    for (int i = 0; i < n; ++i) lg[i] = (unsigned char)__builtin_ctz((unsigned)row_lanes(rp[i + 1] - rp[i], U, gMin));
    std::vector<int> rowOff(1, 0), rowId(n), queue((size_t)n + 1), stamp(n, 0);
    int nr = 0, seed = 0, lanes = 0, p = 1, head = 0, tail = 0;
    while (nr < n) {
        if (head == tail) {
            while (stamp[seed] == INT_MAX) ++seed;
            queue[0] = seed;
            stamp[seed] = p;
            head = 0;
            tail = 1;
        }
        const int v = queue[head];
        if (lanes >= target || lanes + (1 << lg[v]) > 1024) {
            rowOff.push_back(nr);
            lanes = 0;
            ++p;
            queue[0] = v;
            stamp[v] = p;
            head = 0;
            tail = 1;
            continue;
        }
        ++head;
        stamp[v] = INT_MAX;
        rowId[nr++] = v;
        lanes += 1 << lg[v];
        for (int k = rp[v]; k < rp[v + 1]; ++k) { // no branch: half the tests would be mispredicted
            const int c = cp[k];
            queue[tail] = c;
            tail += stamp[c] < p;
            stamp[c] = std::max(stamp[c], p);
        }
    }
    rowOff.push_back(n);
    G = (long long)rowOff.size() - 1;
    if (G > cus || G >= 0xffff) return SVFSI_OK;
    // rows by descending lane count, so that every group is aligned
    std::vector<int> laneOff(1, 0), lane, pos(n), ball;
    lane.reserve((size_t)total + 64 * (size_t)G);
    P.maxOwn = P.maxHalo = P.maxLanes = 0;
    for (int b = 0; b < (int)G; ++b) {
        ball.assign(rowId.begin() + rowOff[b], rowId.begin() + rowOff[b + 1]);
        int at = rowOff[b];
        for (int q = 6; q >= 0; --q)
            for (int v : ball)
                if (lg[v] == q) {
                    rowId[at] = v;
                    pos[v] = at;
                    lane.insert(lane.end(), (size_t)1 << q, (at - rowOff[b]) | q << 16);
                    ++at;
                }
        while (lane.size() % 64) lane.push_back(-1);
        laneOff.push_back((int)lane.size());
        P.maxLanes = std::max(P.maxLanes, laneOff[b + 1] - laneOff[b]);
        P.maxOwn = std::max(P.maxOwn, rowOff[b + 1] - rowOff[b]);
    }
    if (P.maxLanes > 1024) return SVFSI_OK;
    // halos and local columns, the parts shared out over a few threads
    std::vector<std::vector<int>> halo((size_t)G);
    std::vector<unsigned short> lcol(L.nnz);
    std::atomic<int> nextPart{0}, failed{0};
    auto halos = [&]() {
        try {
            std::vector<unsigned> slot(n, 0xffffffffu); // by position: part << 16 | index in its halo
            std::vector<unsigned long long> key;
            std::vector<unsigned short> rank;
            for (int b; (b = nextPart.fetch_add(1)) < (int)G;) {
                const int o0 = rowOff[b], own = rowOff[b + 1] - o0;
                std::vector<int>& h = halo[b];
                for (int i = o0; i < o0 + own; ++i)
                    for (int k = rp[rowId[i]]; k < rp[rowId[i] + 1]; ++k) {
                        const int q = pos[cp[k]], d = q - o0;
                        if ((unsigned)d < (unsigned)own) {
                            lcol[k] = (unsigned short)d;
                            continue;
                        }
                        if (slot[q] >> 16 != (unsigned)b) {
                            if (own + h.size() >= 65536) {
                                failed = 1;
                                return;
                            }
                            slot[q] = (unsigned)b << 16 | (unsigned)h.size();
                            h.push_back(q);
                        }
                        lcol[k] = (unsigned short)(own + (slot[q] & 0xffff));
                    }
                // ascending positions: neighbouring lanes poll neighbouring words
                const int nh = (int)h.size();
                key.resize(nh);
                rank.resize(nh);
                for (int i = 0; i < nh; ++i) key[i] = (unsigned long long)h[i] << 16 | (unsigned)i;
                std::sort(key.begin(), key.end());
                for (int i = 0; i < nh; ++i) {
                    h[i] = (int)(key[i] >> 16);
                    rank[key[i] & 0xffff] = (unsigned short)(own + i);
                }
                for (int i = o0; i < o0 + own; ++i)
                    for (int k = rp[rowId[i]]; k < rp[rowId[i] + 1]; ++k)
                        if ((int)lcol[k] >= own) lcol[k] = rank[lcol[k] - own];
            }
        } catch (...) {
            failed = 1;
        }
    };
    {
        std::vector<std::thread> crew;
        try {
            crew.reserve(6);
            if (L.nnz > 50000) // below, starting threads costs what they save
                for (int i = 0; i < 6; ++i) crew.emplace_back(halos);
        } catch (...) { // this thread does it with those that started
        }
        halos();
        for (std::thread& t : crew) t.join();
    }
    if (failed) return SVFSI_OK;
    std::vector<int> hOff(1, 0), hPos;
    for (const std::vector<int>& h : halo) {
        hPos.insert(hPos.end(), h.begin(), h.end());
        hOff.push_back((int)hPos.size());
        P.maxHalo = std::max(P.maxHalo, (int)h.size());
    }
    if (ppoly_lds(P) + 64 > ldsMax) return SVFSI_OK;
    // one array for all tables
    const std::vector<int>* tabs[6] = {&rowOff, &rowId, &laneOff, &lane, &hOff, &hPos};
    size_t ints = 0;
    for (int i = 0; i < 6; ++i) {
        P.at[i] = ints;
        ints += tabs[i]->size();
    }
    P.at[6] = ints;
    std::vector<int> all(ints + (lcol.size() + 1) / 2);
    for (int i = 0; i < 6; ++i) std::copy(tabs[i]->begin(), tabs[i]->end(), all.begin() + P.at[i]);
    std::memcpy(all.data() + ints, lcol.data(), lcol.size() * sizeof(unsigned short));
    SV_TRY(P.tab.ensure(all.size() * sizeof(int)));
    SV_HIP(hipMemcpy(P.tab.p, all.data(), all.size() * sizeof(int), hipMemcpyHostToDevice));
    // the exchange buffer and the partials of two sums over all parts, tag 0;
    // cleared before this returns: the first solve may be on a stream that does
    // not wait for the null stream, and what a freed pattern left in the memory
    // may carry the tags that it starts with
    P.red = (size_t)n * 16;
    const size_t words = P.red + (size_t)G * 4;
    SV_TRY(P.xb.ensure(words * sizeof(unsigned long long)));
    SV_HIP(hipMemset(P.xb.p, 0, words * sizeof(unsigned long long)));
    SV_HIP(hipStreamSynchronize(nullptr));
    P.ldsMax = ldsMax;
    P.U = U;
    P.G = (int)G;
    return SVFSI_OK;
}

static int choose(Lhs& L, Parts& P)
{
    int d = 0, cus = 0, lds = 0;
    SV_HIP(hipGetDevice(&d));
    SV_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d));
    SV_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, d));
    // 8 lanes and 3 blocks a lane suit tet4 rows (15 to 24 blocks); where
    // that needs more lanes than the chip has, 4 lanes and 5 blocks.  Mixed
    // solve, with them / with one launch per factor, ms: 3 blocks, elasticity
    // cube 28^3 2.99 / 4.47; 5 blocks, cubes 32^3 3.75 / 5.86 and 37^3 5.14 /
    // 9.68, fluid cylinders of 35,306, 40,381 and 47,392 nodes 4.69 / 8.66,
    // 4.72 / 9.09 and 5.72 / 11.2.  CG has no form with 5 blocks.
    SV_TRY(build(L, P, 3, 8, cus, (size_t)lds));
    if (!P.G) SV_TRY(build(L, P, 5, 4, cus, (size_t)lds));
    return SVFSI_OK;
}

void persist_build(Lhs& L)
{
    // the exchange needs a structurally symmetric pattern (persist.hpp)
    if (!L.symmetric) return;
    try {
        std::shared_ptr<Parts> P = std::make_shared<Parts>();
        if (choose(L, *P) != SVFSI_OK || (P->G > 0 && make_event() != SVFSI_OK)) (void)hipGetLastError();
        else if (P->G > 0) L.parts = P;
    } catch (...) { // out of host memory: no parts
    }
}

Parts* persist_parts(Lhs& L, bool pcg)
{
    // SVFSI_PERSIST=0: one launch per product throughout (read at each call)
    const char* e = getenv("SVFSI_PERSIST");
    if (!L.parts || (pcg && !pcg_fits(*L.parts)) || (e && e[0] == '0')) return nullptr;
    if (L.parts->rest > 0) {
        --L.parts->rest;
        return nullptr;
    }
    // SVFSI_PERSIST_WAIT: ticks of 10 ns a lane waits before it gives up; 0:
    // at the first word that is not there yet (tests of that path)
    const char* w = getenv("SVFSI_PERSIST_WAIT");
    L.parts->wait = w ? strtoull(w, nullptr, 10) : kWaitTicks;
    return L.parts.get();
}

} // namespace svfsi
