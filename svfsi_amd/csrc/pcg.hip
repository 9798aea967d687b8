// pcg.hip -- matrix-resident conjugate gradients (persist.hpp): CGRADV on dof 3
// and the NS solver's CGRAD_SCHUR, FP64, a chunk of iterations per launch.
//
// One workgroup per part keeps its blocks and its rows of X, R and P in
// registers and P of its rows and halo in LDS.  An iteration is the product
// from LDS, the two sums <P, K P> and |R|^2 over all parts, and one exchange of
// R: the halo's new P is formed where it is used, from the neighbours' R and
// the part's own copy of their P, with the arithmetic of the row that owns it.
// Every part forms the same scalars from the same sums, in the same order, so
// all leave the loop in the same iteration.  The scalar and vector steps are
// those of k_cg_update / k_cg_pupdate.
//
// What bounds it: latency.  A sum over all parts is one trip through memory
// (every part reads all partials; two levels of 16 took 1.1 us more), the
// exchange of R travels with the second and that of G P with the first, and
// sums over a wavefront go by DPP (shuffles: 1 us more per iteration).  Per
// iteration, 9,261-node elasticity cube: 12.4 us with three launches, 6.2 here
// (step 5.4 -> 2.8 ms); 26,667-node cylinder, Schur complement: 18.6 us, here
// 10.3 (NS step 8.3 -> 4.8 ms).  The tables are 16-byte aligned: behind static
// LDS of an odd number of doubles the steps took 3.2 and 5.0 ms.
#include "persist.hpp"
#include "devutil.hpp"
#include "stream.hpp"
#include "cgstate.hpp"

namespace svfsi {

namespace {

typedef unsigned long long u64;

__device__ __forceinline__ void put_double(u64* p, double v, unsigned tag)
{
    put_word(p, (unsigned)__double2loint(v), tag);
    put_word(p + 1, (unsigned)__double2hiint(v), tag);
}

// v of another lane of the row of 16, by a DPP control
template <int C>
__device__ __forceinline__ double dpp(double v)
{
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), C, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), C, 0xf, 0xf, true));
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kMirror16 = 0x140;

// Sum over each row of 16 lanes and over the wavefront, in every lane: DPP
// moves, where a butterfly of shuffles goes through the LDS unit six times
// (three sums over a wavefront stand in each sum over the parts).
__device__ __forceinline__ double sum16(double v)
{
    v += dpp<kXor1>(v);
    v += dpp<kXor2>(v);
    v += dpp<kMirror8>(v); // quads hold their sums: the other quad's
    v += dpp<kMirror16>(v);
    return v;
}
__device__ __forceinline__ double lane_value(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ double sum64(double v)
{
    v = sum16(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// sum of v[] over the row's gs >= 8 lanes (wide: the widest row of the wave)
template <int N>
__device__ __forceinline__ void row_sum(double (&v)[N], int gs, int wide)
{
#pragma unroll
    for (int m = 0; m < N; ++m) {
        v[m] += dpp<kXor1>(v[m]);
        v[m] += dpp<kXor2>(v[m]);
        v[m] += dpp<kMirror8>(v[m]);
    }
    if (wide > 8)
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const double t = dpp<kMirror16>(v[m]);
            if (gs > 8) v[m] += t;
        }
    if (wide > 16)
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const double t = __shfl_xor(v[m], 16, kWave);
            if (gs > 16) v[m] += t;
        }
    if (wide > 32)
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const double t = __shfl_xor(v[m], 32, kWave);
            if (gs > 32) v[m] += t;
        }
}

struct ReduceLds {
    double w[16], r[16];
    int bad;
};

// waves that read the partials, the first ones: a partial per lane
__device__ __forceinline__ int sum_waves(const PartsDev& P)
{
    return min((int)blockDim.x >> 6, (P.G + 63) >> 6);
}

// Sum of v over all lanes of all parts, the same bits everywhere: a part
// writes its partial and reads those of all (red: 2 G words).  The waves that
// have none to read run meanwhile(), all of them after reading if there are
// no others (false: gave up).  Returns false, in every lane, when a wait of
// this workgroup gave up.
template <class F>
__device__ __forceinline__ bool sum_parts(const PartsDev& P, int part, u64* red, unsigned tag, double v,
                                          ReduceLds& L, int* abortFlag, double& out, F&& meanwhile)
{
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, nw = blockDim.x >> 6, nr = sum_waves(P);
    v = sum64(v);
    if (l == 0) L.w[wave] = v;
    __syncthreads();
    if (wave == 0) {
        const double s = sum16(l < nw ? L.w[l] : 0.0); // lanes 0 to 15
        if (l < 2) put_word(red + 2 * part + l, (unsigned)(l ? __double2hiint(s) : __double2loint(s)), tag);
    }
    bool ok = true;
    if (wave < nr) {
        double s = 0.0;
        for (int q = threadIdx.x; q < P.G && ok; q += 64 * nr) {
            const u64* p[2] = {red + 2 * q, red + 2 * q + 1};
            unsigned w[2];
            ok = get_words<2>(p, tag, w, P.wait, abortFlag);
            s += __hiloint2double((int)w[1], (int)w[0]);
        }
        s = sum64(s);
        if (l == 0) L.r[wave] = s;
    }
    if ((wave >= nr || nw == nr) && !meanwhile()) ok = false;
    if (!ok) L.bad = 1;
    __syncthreads();
    double s = L.r[0];
    for (int w = 1; w < nr; ++w) s += L.r[w];
    out = s;
    return !L.bad;
}

// The lanes' share of a part, as in k_ppoly.
struct Lane {
    int o0, nr, nh, lr, gs, l, row, wide;
    bool has;
};
__device__ __forceinline__ Lane lane_of(const PartsDev& P, int b)
{
    Lane t;
    const int tid = threadIdx.x;
    t.o0 = P.rowOff[b];
    t.nr = P.rowOff[b + 1] - t.o0;
    t.nh = P.hOff[b + 1] - P.hOff[b];
    const int li = P.laneOff[b] + tid;
    const int info = li < P.laneOff[b + 1] ? P.lane[li] : -1;
    t.has = info >= 0;
    t.lr = info & 0xffff;
    t.gs = t.has ? 1 << (info >> 16) : 0;
    t.l = tid & (t.gs - 1);
    t.row = t.has ? P.rowId[t.o0 + t.lr] : 0;
    t.wide = __any(t.gs > 32) ? 64 : (__any(t.gs > 16) ? 32 : (__any(t.gs > 8) ? 16 : 8));
    return t;
}

constexpr int kXbNode = 16; // exchange words per node: two buffers of eight

// NV doubles per halo node, at word w0 of its buffer, to dst (stride ds), by
// nl lanes from first on.
template <int NV>
__device__ __forceinline__ bool get_halo(const PartsDev& P, const int* sH, int nh, int first, int nl, size_t buf, int w0,
                                         unsigned tag, double* dst, int ds, int* abortFlag)
{
    bool ok = true;
    for (int t0 = (int)threadIdx.x - first; t0 < NV * nh && ok; t0 += 2 * nl) {
        const u64* src[4];
        unsigned v[4];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int t = t0 + m * nl, h = t / NV;
            const u64* p = t < NV * nh ? P.xb + (size_t)sH[h] * kXbNode + buf + w0 + 2 * (t - h * NV) : nullptr;
            src[2 * m] = p;
            src[2 * m + 1] = p ? p + 1 : nullptr;
        }
        ok = get_words<4>(src, tag, v, P.wait, abortFlag);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int t = t0 + m * nl, h = t / NV;
            if (t < NV * nh) dst[(size_t)h * ds + t - h * NV] = __hiloint2double((int)v[2 * m + 1], (int)v[2 * m]);
        }
    }
    return ok;
}

} // namespace

// CGRADV, dof 3.
template <int U>
__global__ __launch_bounds__(1024) void k_pcg3(PartsDev P, int tabN, int maxHalo, const int* __restrict__ rowPtr,
                                               const double* __restrict__ val, double* __restrict__ X,
                                               double* __restrict__ R, double* __restrict__ Pv, CgState* st,
                                               int its, unsigned base)
{
    __shared__ ReduceLds L;
    if (leave_at_start(&st->done, &L.bad)) return;
    extern __shared__ __align__(16) double ldsd[]; // four doubles a node, read together
    double* tp = ldsd;                // P: own rows, then the halo, 4 per node
    double* tr = tp + 4 * tabN;       // R of the halo, 3 per node
    int* sH = reinterpret_cast<int*>(tr + 3 * maxHalo);
    const int tid = threadIdx.x, NT = blockDim.x, b = blockIdx.x;
    const int w1 = NT > 64 * sum_waves(P) ? 64 * sum_waves(P) : 0; // the others fetch the halo
    const Lane t = lane_of(P, b);
    const int nr = t.nr, nh = t.nh;
    double a[U][9];
    int lc[U];
    {
        const int k0 = t.has ? rowPtr[t.row] : 0, k1 = t.has ? rowPtr[t.row + 1] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + t.l + u * t.gs;
            const bool in = t.has && k < k1;
            lc[u] = in ? (int)P.lcol[k] : -1;
            if (in) load9<false>(val + (size_t)k * 9, a[u]);
            else
#pragma unroll
                for (int m = 0; m < 9; ++m) a[u][m] = 0.0;
        }
    }
    const bool own = t.has && t.l < 3;
    const size_t vi = (size_t)t.row * 3 + t.l;
    double x = 0.0, r = 0.0, p = 0.0;
    if (own) {
        x = X[vi];
        r = R[vi];
        p = Pv[vi];
        tp[4 * t.lr + t.l] = p;
    }
    for (int i = tid; i < nh; i += NT) sH[i] = P.hPos[P.hOff[b] + i];
    __syncthreads();
    for (int q = tid; q < 3 * nh; q += NT) {
        const int h = q / 3, c = q - 3 * h;
        tp[4 * (nr + h) + c] = Pv[(size_t)P.rowId[sH[h]] * 3 + c];
    }
    double err = st->err, errO = st->errO, alpha = st->alpha;
    const double eps = st->eps;
    int itr = st->itr, done = 0, suc = 0;
    const int mItr = st->mItr;
    __syncthreads();
    for (int it = 0; it < its && !done; ++it) {
        const unsigned tag = base + it;
        double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (lc[u] >= 0) {
                const double* xv = tp + 4 * lc[u];
                const double x0 = xv[0], x1 = xv[1], x2 = xv[2];
#pragma unroll
                for (int i = 0; i < 3; ++i) s[i] += a[u][3 * i] * x0 + a[u][3 * i + 1] * x1 + a[u][3 * i + 2] * x2;
            }
        row_sum<3>(s, t.gs, t.wide);
        const double kp = t.l == 0 ? s[0] : (t.l == 1 ? s[1] : s[2]);
        double pkp, rr;
        if (!sum_parts(P, b, P.red, tag, own ? p * kp : 0.0, L, &st->abort, pkp, [] { return true; })) break;
        alpha = err / pkp;
        if (own) {
            x = x + alpha * p;
            r = r + (-alpha) * kp;
            put_double(P.xb + (size_t)(t.o0 + t.lr) * kXbNode + 8 * (it & 1) + 2 * t.l, r, tag);
        }
        const bool ok = sum_parts(P, b, P.red + 2 * P.G, tag, own ? r * r : 0.0, L, &st->abort, rr, [&] {
            return get_halo<3>(P, sH, nh, w1, NT - w1, 8 * (it & 1), 0, tag, tr, 3, &st->abort);
        });
        if (!ok) break;
        const double nrm = sqrt(rr);
        errO = err;
        err = nrm * nrm;
        const double r1 = errO / err, r2 = err / errO;
        if (own) {
            p = (p + r1 * r) * r2;
            tp[4 * t.lr + t.l] = p;
        }
        for (int q = tid; q < 3 * nh; q += NT) {
            const int h = q / 3;
            double* ph = tp + 4 * (nr + h) + q - 3 * h;
            *ph = (*ph + r1 * tr[q]) * r2;
        }
        ++itr;
        if (itr >= mItr) done = 1;
        else if (err < eps) done = suc = 1;
        __syncthreads();
    }
    if (L.bad) { // some part gave up: the caller starts over
        if (tid == 0) st_agent(&st->done, 1);
        return;
    }
    if (own) {
        X[vi] = x;
        R[vi] = r;
        Pv[vi] = p;
    }
    if (b == 0 && tid == 0) {
        st->alpha = alpha;
        st->err = err;
        st->errO = errO;
        st->itr = itr;
        if (done) {
            st->suc = suc;
            st->done = 1;
        }
    }
}

// CGRAD_SCHUR: S P = L P - Gt (G P), one unknown per node.
template <int U>
__global__ __launch_bounds__(1024) void k_pcgs(PartsDev P, int tabN, int maxHalo, const int* __restrict__ rowPtr,
                                               const double* __restrict__ Lm, const double* __restrict__ G,
                                               const double* __restrict__ Gt, double* __restrict__ X,
                                               double* __restrict__ R, double* __restrict__ Pv, CgState* st,
                                               int its, unsigned base)
{
    __shared__ ReduceLds L;
    if (leave_at_start(&st->done, &L.bad)) return;
    extern __shared__ __align__(16) double ldsd[]; // four doubles a node, read together
    double* tg = ldsd;                // G P: own rows, then the halo, 4 per node
    double* tp = tg + 4 * tabN;       // P: own rows, then the halo
    double* tr = tp + tabN;           // R of the halo
    int* sH = reinterpret_cast<int*>(tr + maxHalo);
    const int tid = threadIdx.x, NT = blockDim.x, b = blockIdx.x;
    const int w1 = NT > 64 * sum_waves(P) ? 64 * sum_waves(P) : 0; // the others fetch the halo
    const Lane t = lane_of(P, b);
    const int nr = t.nr, nh = t.nh;
    double gl[U], g[U][3], gt[U][3];
    int lc[U];
    {
        const int k0 = t.has ? rowPtr[t.row] : 0, k1 = t.has ? rowPtr[t.row + 1] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + t.l + u * t.gs;
            const bool in = t.has && k < k1;
            lc[u] = in ? (int)P.lcol[k] : -1;
            gl[u] = in ? Lm[k] : 0.0;
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                g[u][m] = in ? G[(size_t)k * 3 + m] : 0.0;
                gt[u][m] = in ? Gt[(size_t)k * 3 + m] : 0.0;
            }
        }
    }
    const bool own = t.has && t.l == 0, own3 = t.has && t.l < 3;
    double x = 0.0, r = 0.0, p = 0.0;
    if (own) {
        x = X[t.row];
        r = R[t.row];
        p = Pv[t.row];
        tp[t.lr] = p;
    }
    for (int i = tid; i < nh; i += NT) sH[i] = P.hPos[P.hOff[b] + i];
    __syncthreads();
    for (int h = tid; h < nh; h += NT) tp[nr + h] = Pv[P.rowId[sH[h]]];
    double err = st->err, errO = st->errO, alpha = st->alpha;
    const double eps = st->eps;
    int itr = st->itr, done = 0, suc = 0;
    const int mItr = st->mItr;
    u64* mine = P.xb + (size_t)(t.o0 + t.lr) * kXbNode;
    __syncthreads();
    for (int it = 0; it < its && !done; ++it) {
        const unsigned tag = base + it;
        const int buf = 8 * (it & 1);
        double s[4] = {0.0, 0.0, 0.0, 0.0}; // G P and L P
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (lc[u] >= 0) {
                const double pv = tp[lc[u]];
#pragma unroll
                for (int m = 0; m < 3; ++m) s[m] += g[u][m] * pv;
                s[3] += gl[u] * pv;
            }
        row_sum<4>(s, t.gs, t.wide);
        const double gp = t.l == 0 ? s[0] : (t.l == 1 ? s[1] : s[2]);
        if (own3) {
            tg[4 * t.lr + t.l] = gp;
            put_double(mine + buf + 2 * t.l, gp, tag);
        }
        // Gt = -G^T: <P, S P> = <P, L P> + |G P|^2, summed while G P travels
        double psp, rr;
        if (!sum_parts(P, b, P.red, tag, (own ? p * s[3] : 0.0) + (own3 ? gp * gp : 0.0), L, &st->abort, psp, [&] {
                return get_halo<3>(P, sH, nh, w1, NT - w1, buf, 0, tag, tg + 4 * nr, 4, &st->abort);
            }))
            break;
        double d[1] = {0.0};
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (lc[u] >= 0) {
                const double* v = tg + 4 * lc[u];
                d[0] += gt[u][0] * v[0] + gt[u][1] * v[1] + gt[u][2] * v[2];
            }
        row_sum<1>(d, t.gs, t.wide);
        const double sp = s[3] + (-1.0) * d[0];
        alpha = err / psp;
        if (own) {
            x = x + alpha * p;
            r = r + (-alpha) * sp;
            put_double(mine + buf + 6, r, tag);
        }
        const bool ok = sum_parts(P, b, P.red + 2 * P.G, tag, own ? r * r : 0.0, L, &st->abort, rr, [&] {
            return get_halo<1>(P, sH, nh, w1, NT - w1, buf, 6, tag, tr, 1, &st->abort);
        });
        if (!ok) break;
        const double nrm = sqrt(rr);
        errO = err;
        err = nrm * nrm;
        const double r1 = errO / err, r2 = err / errO;
        if (own) {
            p = (p + r1 * r) * r2;
            tp[t.lr] = p;
        }
        for (int h = tid; h < nh; h += NT) tp[nr + h] = (tp[nr + h] + r1 * tr[h]) * r2;
        ++itr;
        if (itr >= mItr) done = 1;
        else if (err < eps) done = suc = 1;
        __syncthreads();
    }
    if (L.bad) {
        if (tid == 0) st_agent(&st->done, 1);
        return;
    }
    if (own) {
        X[t.row] = x;
        R[t.row] = r;
        Pv[t.row] = p;
    }
    if (b == 0 && tid == 0) {
        st->alpha = alpha;
        st->err = err;
        st->errO = errO;
        st->itr = itr;
        if (done) {
            st->suc = suc;
            st->done = 1;
        }
    }
}

size_t pcg_lds(const Parts& P)
{
    const size_t tab = (size_t)(P.maxOwn + P.maxHalo);
    const size_t cg = 4 * tab + 3 * (size_t)P.maxHalo, cgs = 5 * tab + (size_t)P.maxHalo;
    return (cg > cgs ? cg : cgs) * sizeof(double) + (size_t)P.maxHalo * sizeof(int);
}

template <class K>
static int lds_limit(K kernel, size_t lds)
{
    if (lds > ((size_t)64 << 10))
        SV_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
    return SVFSI_OK;
}

int pcg3_launch(Lhs& L, Parts& P, const double* K, double* X, double* R, double* Pv, CgState* st, int its,
                hipStream_t s)
{
    const size_t lds = pcg_lds(P);
    SV_TRY(lds_limit(&k_pcg3<3>, lds));
    // algorithmic bytes: the matrix and its indices once, X, R and P in and out
    ProfScope ps(7, (double)L.nnz * (9.0 * 8.0 + 2.0) + 6.0 * 24.0 * L.nNo);
    SV_LAUNCH(ps, k_pcg3<3>, dim3((unsigned)P.G), dim3((unsigned)P.maxLanes), lds, s, P.dev(),
              P.maxOwn + P.maxHalo, P.maxHalo, L.rowPtr.as<int>(), K, X, R, Pv, st, its, P.epoch + 1);
    SV_HIP(hipGetLastError());
    P.epoch += (unsigned)its + 1u;
    ++P.launches;
    return SVFSI_OK;
}

int pcgs_launch(Lhs& L, Parts& P, const double* Lm, const double* G, const double* Gt, double* X, double* R,
                double* Pv, CgState* st, int its, hipStream_t s)
{
    const size_t lds = pcg_lds(P);
    SV_TRY(lds_limit(&k_pcgs<3>, lds));
    ProfScope ps(7, (double)L.nnz * (7.0 * 8.0 + 2.0) + 6.0 * 8.0 * L.nNo);
    SV_LAUNCH(ps, k_pcgs<3>, dim3((unsigned)P.G), dim3((unsigned)P.maxLanes), lds, s, P.dev(),
              P.maxOwn + P.maxHalo, P.maxHalo, L.rowPtr.as<int>(), Lm, G, Gt, X, R, Pv, st, its, P.epoch + 1);
    SV_HIP(hipGetLastError());
    P.epoch += (unsigned)its + 1u;
    ++P.launches;
    return SVFSI_OK;
}

} // namespace svfsi
