// ppoly.hip -- the polynomial preconditioner as one matrix-resident kernel
// (persist.hpp): z = p(B) D^-1 q, FP32, dof 3 and 4.
//
// One workgroup per part holds its blocks of B in registers (U per lane) for
// all factors.  Per factor its lanes poll the halo of the current vector into
// LDS, and then every row's lanes form and sum the products of their blocks
// (lane l: blocks l, l + lanes, ...), meet by shuffles, and the first DOF of
// them make the factor's update (launch_poly's modes) with the row's vectors
// in registers and publish the new entry: one workgroup barrier per factor.
//
// What bounds it: the launches this replaces move the matrix (31 MB on the
// 200k-tet cylinder) from L2 and the Infinity Cache for each of the 24 factor
// steps, 8.1 us each, 200 us per application with the launches around them;
// here a step is one trip of the halo through memory and a few hundred ns of
// LDS gathers, shuffles and FP64 updates, and the matrix is read once per
// application: 80 us, the mixed step of that mesh 6.05 -> 3.77 ms (LELAS 20^3
// 2.95 -> 2.12 ms).  The table is 16-byte aligned and indexed from its own
// name, so that a gather is one ds_read_b128; through a pointer array it was a
// flat load (93 us, step 4.04 ms).
// With dof 4 and five blocks a lane 4 of the 128 registers spill (20 bytes of
// scratch a lane).  Tried before: parts of consecutive rows (160 us: twice the
// halo), products through LDS with a second barrier (3.2 us of the 6.5 us per
// step).
#include "persist.hpp"
#include "devutil.hpp"
#include "stream.hpp"

namespace svfsi {

typedef float f4_t __attribute__((ext_vector_type(4)));

// v of lane ^ O (O < 32)
template <int O>
__device__ __forceinline__ float lane_xor(float v)
{
    const int i = __float_as_int(v);
    if constexpr (O == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0xB1, 0xf, 0xf, true));
    else if constexpr (O == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x4E, 0xf, 0xf, true));
    else return __int_as_float(__builtin_amdgcn_ds_swizzle(i, (O << 10) | 0x1f));
}

template <int DOF, int U>
__global__ __launch_bounds__(1024) void k_ppoly(PartsDev P, int nNo, int tabN, const int* __restrict__ rowPtr,
                                                const float* __restrict__ val, const float* __restrict__ dinv,
                                                const double* __restrict__ q, float* __restrict__ z,
                                                double* __restrict__ z64, const double* __restrict__ coef,
                                                const int* __restrict__ ops, int nOps, int lastLin, unsigned base,
                                                int* stop, int* abortFlag)
{
    __shared__ int bad[2]; // by step parity: a wave may give up at a step while another still reads the last one's
    if (threadIdx.x == 0) bad[1] = 0;
    if (leave_at_start(stop, &bad[0])) return;
    constexpr int DD = DOF * DOF;
    extern __shared__ __align__(16) float lds[]; // read as f4_t
    auto tab = [&](int s) { return lds + (s & 1) * 4 * tabN; }; // the current vector, own rows then halo
    int* sH = reinterpret_cast<int*>(lds + 8 * tabN);
    const int tid = threadIdx.x, NT = blockDim.x;
    const int b = blockIdx.x;
    const int o0 = P.rowOff[b], nr = P.rowOff[b + 1] - o0;
    const int h0 = P.hOff[b], nh = P.hOff[b + 1] - h0, nw = nh * DOF; // halo nodes, words
    const size_t xbN = (size_t)nNo * 4;

    const int li = P.laneOff[b] + tid;
    const int info = li < P.laneOff[b + 1] ? P.lane[li] : -1;
    const int lr = info & 0xffff, gs = info >= 0 ? 1 << (info >> 16) : 0, l = tid & (gs - 1);
    const bool has = info >= 0;
    const int row = has ? P.rowId[o0 + lr] : 0;
    float a[U][DD];
    int lc[U];
    {
        const int k0 = has ? rowPtr[row] : 0, k1 = has ? rowPtr[row + 1] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + l + u * gs;
            if (has && k < k1) {
                lc[u] = (int)P.lcol[k];
                load_block<DOF, false>(val + (size_t)k * DD, a[u]);
            } else {
                lc[u] = -1;
#pragma unroll
                for (int m = 0; m < DD; ++m) a[u][m] = 0.f;
            }
        }
    }
    for (int i = tid; i < nh; i += NT) sH[i] = P.hPos[h0 + i];
    // the row's entry c = l of the vectors: x the current one, y the result,
    // o the one before a quadratic factor's first half
    const bool own = has && l < DOF;
    float x = 0.f, y = 0.f, o = 0.f;
    if (own) { // x = D^-1 q (k_fg_start's arithmetic)
        const double* qi = q + (size_t)row * DOF;
        if (dinv) {
            const float* d = dinv + (size_t)row * DD + l * DOF;
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < DOF; ++m) s += (double)d[m] * (double)(float)qi[m];
            x = (float)s;
        } else {
            x = (float)qi[l];
        }
        tab(0)[4 * lr + l] = x;
        put_word(P.xb + (size_t)(o0 + lr) * 4 + l, __float_as_uint(x), base);
    }
    __syncthreads(); // sH

    // lanes of the widest row in this wave: how far the sums must reach
    const int wide = __any(gs > 32) ? 64 : (__any(gs > 16) ? 32 : (__any(gs > 8) ? 16 : 8));
    for (int s = 0; s < nOps; ++s) {
        const int mode = ops[2 * s], f = ops[2 * s + 1];
        const double c1 = coef[2 * f], c2 = coef[2 * f + 1];
        float* xt = tab(s);
        // the halo of the current vector, up to four words a lane at a time
        const unsigned long long* xin = P.xb + (size_t)(s & 1) * xbN;
        for (int t0 = tid; t0 < nw; t0 += 4 * NT) {
            const unsigned long long* src[4];
            unsigned v[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int t = t0 + m * NT, h = t / DOF;
                src[m] = t < nw ? xin + (size_t)sH[h] * 4 + (t - h * DOF) : nullptr;
            }
            if (!get_words<4>(src, base + s, v, P.wait, abortFlag)) {
                bad[s & 1] = 1;
                break;
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int t = t0 + m * NT, h = t / DOF;
                if (t < nw) xt[4 * (nr + h) + t - h * DOF] = __uint_as_float(v[m]);
            }
        }
        __syncthreads();
        if (bad[s & 1]) {
            if (tid == 0) st_agent(stop, 1);
            return;
        }
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
        if (!(mode == 2 && c2 == 0.0)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (lc[u] >= 0) {
                    const f4_t xv = *reinterpret_cast<const f4_t*>(xt + 4 * lc[u]);
                    float p[DOF];
#pragma unroll
                    for (int i = 0; i < DOF; ++i) {
                        p[i] = a[u][i * DOF] * xv[0];
#pragma unroll
                        for (int m = 1; m < DOF; ++m) p[i] += a[u][i * DOF + m] * xv[m];
                    }
                    s0 += p[0];
                    s1 += p[1];
                    s2 += p[2];
                    if constexpr (DOF == 4) s3 += p[3];
                }
            }
            // sums over the row's gs lanes
            auto meet = [&](auto shuffle, int d) {
                const float t0 = shuffle(s0), t1 = shuffle(s1), t2 = shuffle(s2);
                if (d < gs) {
                    s0 += t0;
                    s1 += t1;
                    s2 += t2;
                }
                if constexpr (DOF == 4) {
                    const float t3 = shuffle(s3);
                    if (d < gs) s3 += t3;
                }
            };
            if (wide > 32) meet([](float v) { return __shfl_xor(v, 32, kWave); }, 32);
            if (wide > 16) meet([](float v) { return lane_xor<16>(v); }, 16);
            if (wide > 8) meet([](float v) { return lane_xor<8>(v); }, 8);
            meet([](float v) { return lane_xor<4>(v); }, 4);
            meet([](float v) { return lane_xor<2>(v); }, 2);
            meet([](float v) { return lane_xor<1>(v); }, 1);
        }
        if (own) {
            const float acc = l == 0 ? s0 : (l == 1 ? s1 : (l == 2 ? s2 : s3));
            const double pv = (double)x;
            if (mode == 0) {
                y = (float)((double)y + c1 * pv);
                x = (float)(pv - c1 * acc);
            } else if (mode == 1) {
                o = x;
                y = (float)((double)y + c1 * pv - c2 * acc);
                x = acc;
            } else {
                x = (float)((double)o - c1 * pv + c2 * acc);
            }
            if (s + 1 < nOps) {
                put_word(P.xb + (size_t)((s + 1) & 1) * xbN + (size_t)(o0 + lr) * 4 + l, __float_as_uint(x),
                         base + s + 1);
                tab(s + 1)[4 * lr + l] = x;
            }
        }
    }
    if (own) {
        if (lastLin >= 0) y = (float)((double)y + coef[2 * lastLin] * (double)x);
        const size_t m = (size_t)row * DOF + l;
        z[m] = y;
        z64[m] = (double)y;
    }
}

template <int DOF, int U>
static int launch(Lhs& L, Parts& P, const float* B, const float* dinv, const double* q, float* z, double* z64,
                  const double* coef, const int* ops, int nOps, int lastLin, int* stop, int* abortFlag, hipStream_t s)
{
    const size_t lds = ppoly_lds(P);
    const unsigned base = P.epoch + 1; // tags base .. base + nOps
    if (lds > ((size_t)64 << 10))
        SV_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_ppoly<DOF, U>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // algorithmic bytes: the matrix and its indices once, q, z and z64, per
    // step one vector written and read
    const double vec = (double)L.nNo * DOF * 4.0;
    ProfScope ps(6, (double)L.nnz * DOF * DOF * 4.0 + 2.0 * L.nnz + 5.0 * vec + 2.0 * nOps * vec);
    SV_LAUNCH(ps, (k_ppoly<DOF, U>), dim3((unsigned)P.G), dim3((unsigned)P.maxLanes), lds, s, P.dev(), L.nNo,
              P.maxOwn + P.maxHalo, L.rowPtr.as<int>(), B, dinv, q, z, z64, coef, ops, nOps, lastLin, base, stop,
              abortFlag);
    SV_HIP(hipGetLastError());
    P.epoch += (unsigned)nOps + 1u;
    ++P.launches;
    return SVFSI_OK;
}

int ppoly_launch(Lhs& L, Parts& P, int dof, const float* B, const float* dinv, const double* q, float* z, double* z64,
                 const double* coef, const int* ops, int nOps, int lastLin, int* stop, int* abortFlag, hipStream_t s)
{
#define SV_PP(D, UU) return launch<D, UU>(L, P, B, dinv, q, z, z64, coef, ops, nOps, lastLin, stop, abortFlag, s)
    if (dof == 4) {
        if (P.U == 3) SV_PP(4, 3);
        SV_PP(4, 5);
    }
    if (P.U == 3) SV_PP(3, 3);
    SV_PP(3, 5);
#undef SV_PP
}

} // namespace svfsi
