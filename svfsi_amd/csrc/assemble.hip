// assemble.hip -- element tangent/residual construction and DOASSEM scatter
// for gfx950.
//
// By default one launch over all elements writes what the elements contribute
// (tet4: a record of 128 or 320 bytes per element; tet10: its blocks) and a
// second one sums, for each block of Val or row of a node, its elements'
// contributions in element-id order, the order of DOASSEM's loop
// (svFSI/LHSA.f:266-298): deterministic bit for bit, and no two lanes write one
// place.
//
// The coloured kernels (SVFSI_ASM_GATHER=0, STRUCT's kernel selectors, and
// STRUCT where rows are too long for LDS or the scratch cannot be had) process
// elements colour by colour: no two elements of a colour share a node, so a
// launch adds at most one contribution to a block or row, again in a fixed
// order.  There one thread owns one (a,b) node pair of one element, recomputes
// the geometry and the Gauss-point kinematics, accumulates its block over the
// points as the reference routine does, and adds it to Val through the scatter
// map (the bisection of LHSA.f:282-292, done once at mesh creation); the thread
// with b = 0 also builds the residual rows of node a.
#include "internal.hpp"
#include "devutil.hpp"
#include "assemble.hpp"

#include <cmath>

// The element routines are evaluated without contracting multiply-adds into
// FMAs, in the oracle's operation order: Delaunay meshes contain sliver
// elements whose Jacobian inversion amplifies any difference in rounding, and
// the FP64 assembly is to reproduce the CPU restatement to ~1e-12 on them too.
// What comes behind the inversion (sums over points, blocks from records) is
// contracted, by a pragma where it is.
#pragma clang fp contract(off)

namespace svfsi {



// GNN for an affine tet4 (svFSI/NN.f:1469-1565): Nxi of TET4 are constant
// (NN.f:663-671): dN1 = e1, dN2 = e2, dN3 = e3, dN4 = -(1,1,1).
__device__ __forceinline__ void gnn_tet4(const double xl[4][3], double Nx[4][3], double& Jac,
                                         double ks[3][3])
{
    double A[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        A[i][0] = xl[0][i] - xl[3][i];
        A[i][1] = xl[1][i] - xl[3][i];
        A[i][2] = xl[2][i] - xl[3][i];
    }
    // the reference sums x_a * Nxi_a over a; for tet4 that is x_j - x_4
    const double J = A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0]
                   + A[0][2] * A[1][0] * A[2][1] - A[0][0] * A[1][2] * A[2][1]
                   - A[0][1] * A[1][0] * A[2][2] - A[0][2] * A[1][1] * A[2][0];
    double B[3][3];
    B[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) / J;
    B[0][1] = (A[2][1] * A[0][2] - A[2][2] * A[0][1]) / J;
    B[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) / J;
    B[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) / J;
    B[1][1] = (A[2][2] * A[0][0] - A[2][0] * A[0][2]) / J;
    B[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) / J;
    B[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) / J;
    B[2][1] = (A[2][0] * A[0][1] - A[2][1] * A[0][0]) / J;
    B[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) / J;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) ks[i][j] = B[0][i] * B[0][j] + B[1][i] * B[1][j] + B[2][i] * B[2][j];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        Nx[0][j] = B[0][j];
        Nx[1][j] = B[1][j];
        Nx[2][j] = B[2][j];
        Nx[3][j] = -B[0][j] - B[1][j] - B[2][j];
    }
    Jac = J;
}

typedef double d2_t __attribute__((ext_vector_type(2)));

// v of the lane ^1 / ^2 in the same group of four lanes
template <int X>
__device__ __forceinline__ double quad_xor(double v)
{
    constexpr int ctrl = X == 1 ? 0xB1 : 0x4E; // quad_perm [1,0,3,2] / [2,3,0,1]
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// v of lane K of the group of four lanes
template <int K>
__device__ __forceinline__ double quad_get(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), K * 0x55, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), K * 0x55, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double quad_sum(double v)
{
    v += quad_xor<2>(v);
    v += quad_xor<1>(v);
    return v;
}
// ---------------------------------------------------------------------------
// The record gathers: Val(:, j) += the element blocks of nnz entry j, in
// element-id order (DOASSEM's element loop, LHSA.f:266-298), the blocks formed
// from the elements' records.  gSrc[k] = 16 e + 4 a + b names contribution k,
// gPtr the contributions of each entry.  One workgroup takes a tile of whole
// entries with at most kGatherTile contributions (Mesh::gTile); four lanes
// form a contribution, every lane kGatherTile / 64 of them with all loads
// issued first (row(): the lane's row of the block), and leave its rows in
// LDS; then DD lanes per entry add them in order.  An entry with more
// contributions than a tile holds has a tile of its own and goes through it
// in passes.
//
// Bound by latency: a contribution is the chain gPtr -> gSrc -> record ->
// Val, so what counts is how many chains are in flight.  16 lanes per entry
// walking its list, four chains at a time, took 94 us (fluid, 197,696 tets)
// and 90 us (LELAS, 215,622), with most lanes waiting on short lists and the
// 24 contributions of the diagonal entries; the tiles take 80 and 59
// us (with multiply-adds contracted here, where no Jacobian is inverted).
// Tiles go in XCD-contiguous order: the entries of neighbouring rows read the
// same records.  Val may be only 8-byte aligned.
// ---------------------------------------------------------------------------
template <int DD, class ROW>
__device__ __forceinline__ void gather_tile(unsigned b, const int* __restrict__ tile, const int* __restrict__ gPtr,
                                            const int* __restrict__ gSrc, double* __restrict__ val, ROW&& row)
{
    constexpr int T = kGatherTile, U = T / 64, RW = DD == 16 ? 4 : 3, EPP = 256 / DD; // entries per pass of the sum
    __shared__ double sB[T][DD];
    __shared__ int sP[T + 1];
    const int tid = threadIdx.x, r = tid & 3;
    const int j0 = tile[b], nj = tile[b + 1] - j0;
    for (int i = tid; i <= nj; i += 256) sP[i] = gPtr[j0 + i];
    const int k0 = gPtr[j0], k1 = gPtr[j0 + nj];
    // the old values of the entries this lane will write, loaded early
    double old[U];
    const int se = tid / DD, sq = tid - se * DD;
#pragma unroll
    for (int m = 0; m < U; ++m) {
        const int e = se + m * EPP;
        old[m] = (se < EPP && e < nj) ? val[(size_t)(j0 + e) * DD + sq] : 0.0;
    }
    double sum = 0.0; // an entry larger than the tile (nj = 1): the passes' running sum
    for (int kb = k0; kb < k1; kb += T) {
        unsigned src[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = kb + u * 64 + (tid >> 2);
            src[u] = k < k1 ? (unsigned)gSrc[k] : 0u;
        }
        double v[U][RW];
#pragma unroll
        for (int u = 0; u < U; ++u) row(src[u], r, v[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (r < RW)
#pragma unroll
                for (int c = 0; c < RW; ++c) sB[u * 64 + (tid >> 2)][r * RW + c] = v[u][c];
        __syncthreads();
        if (se < EPP) {
#pragma unroll
            for (int m = 0; m < U; ++m) {
                const int e = se + m * EPP;
                if (e >= nj) break;
                const int ke = min(sP[e + 1], kb + T);
                double s = nj == 1 ? sum : 0.0;
#pragma unroll 4
                for (int k = max(sP[e], kb); k < ke; ++k) s += sB[k - kb][sq];
                if (nj == 1) sum = s;
                if (sP[e + 1] <= kb + T) val[(size_t)(j0 + e) * DD + sq] = old[m] + s;
            }
            for (int e = se + U * EPP; e < nj; e += EPP) { // many short entries
                const int ke = sP[e + 1];
                double s = 0.0;
                for (int k = sP[e]; k < ke; ++k) s += sB[k - kb][sq];
                val[(size_t)(j0 + e) * DD + sq] += s;
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// LELAS3D (svFSI/LELAS.f:130-242) in CONSTRUCT_LELAS (LELAS.f:38-128), tet4.
// ---------------------------------------------------------------------------
// The coloured scatter path (SVFSI_ASM_GATHER=0).
__global__ __launch_bounds__(256) void k_asm_lelas(int begin, int count, const int* __restrict__ ien,
                                                   const int* __restrict__ elemId,
                                                   const int* __restrict__ emap,
                                                   const double* __restrict__ x, int tDof,
                                                   const double* __restrict__ Ag,
                                                   const double* __restrict__ Dg,
                                                   const double* __restrict__ Eel, AsmParams P,
                                                   Tet4Rule rule, double* __restrict__ val,
                                                   double* __restrict__ R)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count * 16) return;
    const int p = elemId[begin + (t >> 4)];
    const int ab = t & 15;
    const int a = ab >> 2, b = ab & 3;
    int nd[4];
    double xl[4][3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        nd[q] = ien[(size_t)p * 4 + q];
#pragma unroll
        for (int i = 0; i < 3; ++i) xl[q][i] = x[(size_t)nd[q] * 3 + i];
    }
    double Nx[4][3], ks[3][3], Jac;
    gnn_tet4(xl, Nx, Jac, ks);
    const double E = Eel ? Eel[p] : P.E;
    const double nu = P.nu, rho = P.rho;
    const double lambda = E * nu / (1.0 + nu) / (1.0 - 2.0 * nu);
    const double mu = E * 0.5 / (1.0 + nu);
    const double lDm = lambda / mu;
    const double T1 = P.af * P.beta * P.dt * P.dt;
    const double amd = P.am / T1 * rho;
    double k[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const double NxdNx = Nx[a][0] * Nx[b][0] + Nx[a][1] * Nx[b][1] + Nx[a][2] * Nx[b][2];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const double w = rule.w[g] * Jac;
        const double wl = w * T1 * mu;
        const double Tm = amd * rule.N[g][a] * rule.N[g][b] / mu + NxdNx;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double v = (i == j) ? Tm + (1.0 + lDm) * Nx[a][i] * Nx[b][i]
                                          : lDm * Nx[a][i] * Nx[b][j] + Nx[a][j] * Nx[b][i];
                k[i * 3 + j] += wl * v;
            }
    }
    double* vb = val + (size_t)emap[(size_t)p * 16 + ab] * 9;
#pragma unroll
    for (int q = 0; q < 9; ++q) vb[q] += k[q];

    if (b != 0) return;
    // residual row a (LELAS.f:161-205 and 208-215)
    double ed[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const double* D = Dg + (size_t)nd[q] * tDof;
        ed[0] += Nx[q][0] * D[0];
        ed[1] += Nx[q][1] * D[1];
        ed[2] += Nx[q][2] * D[2];
        ed[3] += Nx[q][1] * D[0] + Nx[q][0] * D[1];
        ed[4] += Nx[q][2] * D[1] + Nx[q][1] * D[2];
        ed[5] += Nx[q][0] * D[2] + Nx[q][2] * D[0];
    }
    const double divD = lambda * (ed[0] + ed[1] + ed[2]);
    double S[6];
    S[0] = divD + 2.0 * mu * ed[0];
    S[1] = divD + 2.0 * mu * ed[1];
    S[2] = divD + 2.0 * mu * ed[2];
    S[3] = mu * ed[3];
    S[4] = mu * ed[4];
    S[5] = mu * ed[5];
    double r[3] = {0, 0, 0};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const double w = rule.w[g] * Jac;
        double ud[3] = {-P.fb[0], -P.fb[1], -P.fb[2]};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double* A = Ag + (size_t)nd[q] * tDof;
#pragma unroll
            for (int i = 0; i < 3; ++i) ud[i] += rule.N[g][q] * A[i];
        }
        const double Na = rule.N[g][a];
        r[0] += w * (rho * Na * ud[0] + Nx[a][0] * S[0] + Nx[a][1] * S[3] + Nx[a][2] * S[5]);
        r[1] += w * (rho * Na * ud[1] + Nx[a][0] * S[3] + Nx[a][1] * S[1] + Nx[a][2] * S[4]);
        r[2] += w * (rho * Na * ud[2] + Nx[a][0] * S[5] + Nx[a][1] * S[4] + Nx[a][2] * S[2]);
    }
    double* Rr = R + (size_t)ien[(size_t)p * 4 + a] * 3;
    Rr[0] += r[0];
    Rr[1] += r[1];
    Rr[2] += r[2];
}

// ---------------------------------------------------------------------------
// LELAS gather assembly, two launches (the scheme of the fluid's records
// below).  Summed over the Gauss points, the (a,b) block of an element is
//   c0 Nx_a Nx_b^T + c1 Nx_b Nx_a^T + (c1 Nx_a.Nx_b + m_ab) I
// with c0 = V af beta dt^2 lambda, c1 = V af beta dt^2 mu and the consistent
// mass m_ab = am rho Jac sum_g w_g N_a N_b, which takes one value on the
// diagonal (c2) and one off it (c3): 16 numbers, one 128-byte line, against
// 1152 bytes of element blocks.  On the 215,622-tet cube the element kernel
// takes 22 us and the gather 59, against 195 us for 16 lanes per element
// storing their blocks and 81 + 8 us for summing those.
// ---------------------------------------------------------------------------
constexpr int LR_C = 12, LR_SZ = 16;

// Four lanes per element: lane a reads node a and forms row a of the
// residual (LELAS.f:161-215).
__global__ __launch_bounds__(256) void k_lelas_rec(int nEl, const int* __restrict__ ien, const double* __restrict__ x,
                                                   int tDof, const double* __restrict__ Ag,
                                                   const double* __restrict__ Dg, const double* __restrict__ Eel,
                                                   AsmParams P, Tet4Rule rule, double* __restrict__ rec,
                                                   double* __restrict__ re, const int* __restrict__ rslot)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nEl * 4) return; // whole quads
    const int p = t >> 2, a = t & 3;
    const int nd = ien[t];
    double xa[3], Da[3], Aa[3], xl[4][3], D[4][3], As[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xa[i] = x[(size_t)nd * 3 + i];
        Da[i] = Dg[(size_t)nd * tDof + i];
        Aa[i] = Ag[(size_t)nd * tDof + i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xl[0][i] = quad_get<0>(xa[i]);
        xl[1][i] = quad_get<1>(xa[i]);
        xl[2][i] = quad_get<2>(xa[i]);
        xl[3][i] = quad_get<3>(xa[i]);
        D[0][i] = quad_get<0>(Da[i]);
        D[1][i] = quad_get<1>(Da[i]);
        D[2][i] = quad_get<2>(Da[i]);
        D[3][i] = quad_get<3>(Da[i]);
        As[i] = quad_sum(Aa[i]);
    }
    double Nx[4][3], ks[3][3], Jac;
    gnn_tet4(xl, Nx, Jac, ks);
    double Nxa[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (q == a) {
#pragma unroll
            for (int i = 0; i < 3; ++i) Nxa[i] = Nx[q][i];
        }
    const double E = Eel ? Eel[p] : P.E;
    const double nu = P.nu, rho = P.rho;
    const double lambda = E * nu / (1.0 + nu) / (1.0 - 2.0 * nu);
    const double mu = E * 0.5 / (1.0 + nu);
    const double T1 = P.af * P.beta * P.dt * P.dt;
    // sum_g w_g, w_g N_a, w_g N_a^2 and w_g N_a N_b (a symmetric rule)
    double w0 = 0.0, w1 = 0.0, md = 0.0, mo = 0.0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        w0 += rule.w[g];
        w1 += rule.w[g] * rule.N[g][0];
        md += rule.w[g] * rule.N[g][0] * rule.N[g][0];
        mo += rule.w[g] * rule.N[g][0] * rule.N[g][1];
    }
    const double V = w0 * Jac;
    const double c = a == 0 ? V * T1 * lambda : (a == 1 ? V * T1 * mu : P.am * rho * Jac * (a == 2 ? md : mo));
    double* rc = rec + (size_t)p * LR_SZ;
#pragma unroll
    for (int i = 0; i < 3; ++i) rc[3 * a + i] = Nxa[i];
    rc[LR_C + a] = c;
    double ed[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        ed[0] += Nx[q][0] * D[q][0];
        ed[1] += Nx[q][1] * D[q][1];
        ed[2] += Nx[q][2] * D[q][2];
        ed[3] += Nx[q][1] * D[q][0] + Nx[q][0] * D[q][1];
        ed[4] += Nx[q][2] * D[q][1] + Nx[q][1] * D[q][2];
        ed[5] += Nx[q][0] * D[q][2] + Nx[q][2] * D[q][0];
    }
    const double divD = lambda * (ed[0] + ed[1] + ed[2]);
    const double S0 = divD + 2.0 * mu * ed[0], S1 = divD + 2.0 * mu * ed[1], S2 = divD + 2.0 * mu * ed[2];
    const double S3 = mu * ed[3], S4 = mu * ed[4], S5 = mu * ed[5];
    const double rJ = rho * Jac;
    double* rr = re + (size_t)rslot[t] * 3;
    rr[0] = rJ * (mo * As[0] + (md - mo) * Aa[0] - w1 * P.fb[0]) + V * (Nxa[0] * S0 + Nxa[1] * S3 + Nxa[2] * S5);
    rr[1] = rJ * (mo * As[1] + (md - mo) * Aa[1] - w1 * P.fb[1]) + V * (Nxa[0] * S3 + Nxa[1] * S1 + Nxa[2] * S4);
    rr[2] = rJ * (mo * As[2] + (md - mo) * Aa[2] - w1 * P.fb[2]) + V * (Nxa[0] * S5 + Nxa[1] * S4 + Nxa[2] * S2);
}

// Val from the records (gather_tile; the fourth lane of a quad only loads)
// and, in the workgroups from nbVal on, the R rows.
__global__ __launch_bounds__(256) void k_lelas_gather(int nNo, unsigned nbVal, const int* __restrict__ tile,
                                                      const int* __restrict__ gPtr, const int* __restrict__ gSrc,
                                                      const double* __restrict__ rec, double* __restrict__ val,
                                                      const int* __restrict__ rPtr, const double* __restrict__ re,
                                                      double* __restrict__ R)
{
    if (blockIdx.x >= nbVal) {
        const unsigned t = (blockIdx.x - nbVal) * 256 + threadIdx.x;
        const int i = (int)(t / 3), c = (int)(t - 3 * (t / 3));
        if (i >= nNo) return;
        const int k1 = rPtr[i + 1];
        double s = 0.0;
#pragma unroll 4
        for (int k = rPtr[i]; k < k1; ++k) s += re[(size_t)k * 3 + c];
        R[(size_t)i * 3 + c] += s;
        return;
    }
    gather_tile<9>(xcd_part(blockIdx.x, nbVal), tile, gPtr, gSrc, val, [&](unsigned src, int r, double (&v)[3]) {
#pragma clang fp contract(fast) // no Jacobian here: see the top of the file
        const int a = (int)(src >> 2) & 3, b = (int)src & 3;
        const double* rc = rec + (size_t)(src >> 4) * LR_SZ;
        const d2_a8 m = *reinterpret_cast<const d2_a8*>(rc + (r == 0 ? 3 * a : (r == 1 ? 3 * b : LR_C + 2 * (r - 2))));
        const double n = rc[r == 0 ? 3 * a + 2 : (r == 1 ? 3 * b + 2 : 0)];
        const double a0 = quad_get<0>(m.x), a1 = quad_get<0>(m.y), a2 = quad_get<0>(n);
        const double b0 = quad_get<1>(m.x), b1 = quad_get<1>(m.y), b2 = quad_get<1>(n);
        const double c0 = quad_get<2>(m.x), c1 = quad_get<2>(m.y), c2 = quad_get<3>(m.x), c3 = quad_get<3>(m.y);
        const double d = c1 * (a0 * b0 + a1 * b1 + a2 * b2) + (a == b ? c2 : c3);
        const double fb = c0 * (r == 0 ? a0 : (r == 1 ? a1 : a2)); // factor of Nx_b
        const double fa = c1 * (r == 0 ? b0 : (r == 1 ? b1 : b2)); // factor of Nx_a
        v[0] = fb * b0 + fa * a0 + (r == 0 ? d : 0.0);
        v[1] = fb * b1 + fa * a1 + (r == 1 ? d : 0.0);
        v[2] = fb * b2 + fa * a2 + (r == 2 ? d : 0.0);
    });
}

// ---------------------------------------------------------------------------
// FLUID3D_M + FLUID3D_C (svFSI/FLUID.f:192-560, 813-1084) in CONSTRUCT_FLUID
// (FLUID.f:40-190), tet4 VMS (nFs = 1), Newtonian viscosity: GNNxx of an
// affine tet is zero, so uxx = d2u2 = 0, and mu_x = mu_g = 0 (GETVISCOSITY
// viscType_Const, FLUID.f:1700-1703).  The momentum blocks (1..12) and the
// continuity blocks (13..16) are disjoint, so one Gauss loop builds both in
// the same per-entry order as the reference's two loops.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool iszero_d(double a)
{
    const double eps = 2.220446049250313e-16;
    const double aa = fabs(a);
    const double nrm = aa > eps ? aa : eps;
    return (aa / nrm) < 10.0 * eps;
}

// Forward-mode dual number: value and derivative with respect to one
// parameter.  The fluid element routine below is written once over a
// scalar type T; T = double assembles, T = Dual with mu = (mu_e, 1) gives the
// exact derivative of the element tangent and residual with respect to the
// element viscosity.
struct Dual {
    double v, d;
};
__device__ __forceinline__ Dual mkd(double v) { return {v, 0.0}; }
__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ Dual operator+(Dual a, double b) { return {a.v + b, a.d}; }
__device__ __forceinline__ Dual operator+(double a, Dual b) { return {a + b.v, b.d}; }
__device__ __forceinline__ Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ Dual operator-(Dual a, double b) { return {a.v - b, a.d}; }
__device__ __forceinline__ Dual operator-(double a, Dual b) { return {a - b.v, -b.d}; }
__device__ __forceinline__ Dual operator-(Dual a) { return {-a.v, -a.d}; }
__device__ __forceinline__ Dual operator*(Dual a, Dual b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ __forceinline__ Dual operator*(Dual a, double b) { return {a.v * b, a.d * b}; }
__device__ __forceinline__ Dual operator*(double a, Dual b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ Dual operator/(Dual a, Dual b)
{
    const double q = a.v / b.v;
    return {q, (a.d - q * b.d) / b.v};
}
__device__ __forceinline__ Dual operator/(Dual a, double b) { return {a.v / b, a.d / b}; }
__device__ __forceinline__ Dual operator/(double a, Dual b)
{
    const double q = a / b.v;
    return {q, -q * b.d / b.v};
}
__device__ __forceinline__ Dual dsqrt(Dual a)
{
    const double r = sqrt(a.v);
    return {r, 0.5 * a.d / r};
}
__device__ __forceinline__ double dsqrt(double a) { return sqrt(a); }
__device__ __forceinline__ double val_of(double a) { return a; }
__device__ __forceinline__ double val_of(Dual a) { return a.v; }
template <typename T> __device__ __forceinline__ T scal(double v);
template <> __device__ __forceinline__ double scal<double>(double v) { return v; }
template <> __device__ __forceinline__ Dual scal<Dual>(double v) { return mkd(v); }

// Element data of one tet4 shared by the 16 (a,b) threads of an element.
struct FluidElem {
    int nd[4];
    double Nx[4][3], ks[3][3], Jac;
    double yl[4][4], al[4][3];
    double ux[3][3], px[3], divU;
};

__device__ __forceinline__ void fluid_elem(int p, const int* __restrict__ ien, const double* __restrict__ x,
                                           int tDof, const double* __restrict__ Ag,
                                           const double* __restrict__ Yg, FluidElem& E)
{
    double xl[4][3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        E.nd[q] = ien[(size_t)p * 4 + q];
#pragma unroll
        for (int i = 0; i < 3; ++i) xl[q][i] = x[(size_t)E.nd[q] * 3 + i];
    }
    gnn_tet4(xl, E.Nx, E.Jac, E.ks);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int c = 0; c < 4; ++c) E.yl[q][c] = Yg[(size_t)E.nd[q] * tDof + c];
#pragma unroll
        for (int c = 0; c < 3; ++c) E.al[q][c] = Ag[(size_t)E.nd[q] * tDof + c];
    }
    // element-constant kinematics: ux(i,c) = sum Nx(i,q) y(c,q), px, divU
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int c = 0; c < 3; ++c) E.ux[i][c] = 0.0;
        E.px[i] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int c = 0; c < 3; ++c) E.ux[i][c] += E.Nx[q][i] * E.yl[q][c];
        }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 3; ++i) E.px[i] += E.Nx[q][i] * E.yl[q][3];
    E.divU = E.ux[0][0] + E.ux[1][1] + E.ux[2][2];
}

// Gauss-point quantities of FLUID3D_M/C shared by all (a,b) blocks of a
// tet4 element: u, u_dot (with body force), p, the VMS parameters tau_M,
// tau_C, tau_B and the fine-scale velocity u' (svFSI/FLUID.f:220-412).
template <typename T> struct FluidGP {
    double u[3], ud[3], pp;
    T tauM, tauC, tauB, up[3];
};

template <typename T>
__device__ __forceinline__ void fluid_gp_n(const FluidElem& E, T mu, const AsmParams& P, const double N[4],
                                           FluidGP<T>& G)
{
    const double rho = P.rho;
    const double ctM = 1.0, ctC = 36.0;
    double kS0 = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) kS0 += E.ks[i][j] * E.ks[i][j];
    const T kS = ctC * kS0 * (mu / rho) * (mu / rho);
    const double kT = 4.0 * (ctM / P.dt) * (ctM / P.dt);
    const double trK = E.ks[0][0] + E.ks[1][1] + E.ks[2][2];
    double ud[3] = {-P.fb[0], -P.fb[1], -P.fb[2]};
    double u[3] = {0, 0, 0};
    double pp = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const double Nq = N[q];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            ud[c] += Nq * E.al[q][c];
            u[c] += Nq * E.yl[q][c];
        }
        pp += Nq * E.yl[q][3];
    }
    double kU = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) kU += u[i] * u[j] * E.ks[i][j];
    const T tauM = 1.0 / (rho * dsqrt(kT + kU + kS));
    T up[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double rV = ud[c] + u[0] * E.ux[0][c] + u[1] * E.ux[1][c] + u[2] * E.ux[2][c];
        up[c] = -tauM * (rho * rV + E.px[c] - mu * 0.0);
    }
    const T tauC = 1.0 / (tauM * trK);
    T tauB = scal<T>(0.0);
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) tauB = tauB + up[i] * up[j] * E.ks[i][j];
    if (iszero_d(val_of(tauB))) tauB = scal<T>(2.220446049250313e-16);
    tauB = rho / dsqrt(tauB);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        G.u[c] = u[c];
        G.ud[c] = ud[c];
        G.up[c] = up[c];
    }
    G.pp = pp;
    G.tauM = tauM;
    G.tauC = tauC;
    G.tauB = tauB;
}

// Viscosity of a tet4 element (GETVISCOSITY, svFSI/FLUID.f:1690-1739, at
// the shear rate gamma = sqrt(es:es / 2) of FLUID.f:359-373): the velocity
// gradient of a linear tet is constant, so mu and mu_g = (d mu / d gamma) /
// gamma are element constants.  mu_i is the element's (or the equation's)
// viscosity; the constant model returns it with mu_g = 0.  Casson raises
// gamma to its threshold lam below it, as the reference does.
__device__ __forceinline__ void fluid_visc(const FluidElem& E, const AsmParams& P, double mu_i, double& mu,
                                           double& mu_g)
{
    mu = mu_i;
    mu_g = 0.0;
    if (P.viscType != 697 && P.viscType != 696) return;
    double gam = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double es = E.ux[i][j] + E.ux[j][i];
            gam += es * es;
        }
    gam = sqrt(0.5 * gam);
    double mux;
    if (P.viscType == 697) {
        double T1 = 1.0 + pow(P.lam * gam, P.va);
        double T2 = pow(T1, (P.vn - 1.0) / P.va);
        mu = mu_i + (P.mu_o - mu_i) * T2;
        T1 = T2 / T1;
        T2 = pow(P.lam, P.va) * pow(gam, P.va - 1.0) * T1;
        mux = (P.mu_o - mu_i) * (P.vn - 1.0) * T2;
    } else {
        double mu_o = P.mu_o;
        if (gam < P.lam) {
            mu_o = mu_o / sqrt(P.lam);
            gam = P.lam;
        } else {
            mu_o = mu_o / sqrt(gam);
        }
        mu = (mu_i + mu_o) * (mu_i + mu_o);
        mux = 2.0 * mu_o * (mu_o + mu_i) / gam;
    }
    mu_g = iszero_d(gam) ? 0.0 : mux / gam;
}

// FLUID3D_M + FLUID3D_C (svFSI/FLUID.f:192-560, 813-1084), the Gauss point
// g contribution to the (a,b) block of one tet4 element, Newtonian
// viscosity mu, second derivatives zero: k (4x4 block, row-major) and, when
// want_r, the residual of node a.
// Rows a and b of the element arrays, selected without dynamic indexing
// (which would place the element record in scratch memory).
struct FluidAB {
    double Nxa[3], Nxb[3];
    double Na[4], Nb[4]; // N_a, N_b at the four Gauss points
    double esNxa[3], esNxb[3]; // esNx(c,a) = sum_j es(j,c) Nx(j,a) (FLUID.f:321-328)
};

__device__ __forceinline__ void fluid_ab(const FluidElem& E, const Tet4Rule& rule, int a, int b, FluidAB& S)
{
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        S.Nxa[i] = 0.0;
        S.Nxb[i] = 0.0;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        S.Na[g] = 0.0;
        S.Nb[g] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (q == a) S.Nxa[i] = E.Nx[q][i];
            if (q == b) S.Nxb[i] = E.Nx[q][i];
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (q == a) S.Na[g] = rule.N[g][q];
            if (q == b) S.Nb[g] = rule.N[g][q];
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double e0 = E.ux[0][c] + E.ux[c][0], e1 = E.ux[1][c] + E.ux[c][1], e2 = E.ux[2][c] + E.ux[c][2];
        S.esNxa[c] = e0 * S.Nxa[0] + e1 * S.Nxa[1] + e2 * S.Nxa[2];
        S.esNxb[c] = e0 * S.Nxb[0] + e1 * S.Nxb[1] + e2 * S.Nxb[2];
    }
}

template <typename T>
__device__ __forceinline__ void fluid_pair_gp(const FluidElem& E, T mu, double mug, const AsmParams& P,
                                              const Tet4Rule& rule, int g, const FluidGP<T>& G, const FluidAB& S,
                                              bool want_r, T k[16], T r[4])
{
    const double* Nxa = S.Nxa;
    const double* Nxb = S.Nxb;
    const double rho = P.rho;
    const double T1c = P.af * P.gam * P.dt;
    const double amd = P.am / T1c;
    const double NxNx = Nxa[0] * Nxb[0] + Nxa[1] * Nxb[1] + Nxa[2] * Nxb[2];
    const double w = rule.w[g] * E.Jac;
    const double wl = w * T1c;
    const double wr = w * rho;
    const double* u = G.u;
    const double* ud = G.ud;
    const T tauM = G.tauM, tauC = G.tauC, tauB = G.tauB;
    const T* up = G.up;
    const T ua[3] = {u[0] + up[0], u[1] + up[1], u[2] + up[2]};

    const double Na = S.Na[g], Nb = S.Nb[g];
    const double uNxa = u[0] * Nxa[0] + u[1] * Nxa[1] + u[2] * Nxa[2];
    const double uNxb = u[0] * Nxb[0] + u[1] * Nxb[1] + u[2] * Nxb[2];
    const T upNxa = up[0] * Nxa[0] + up[1] * Nxa[1] + up[2] * Nxa[2];
    const T upNxb = up[0] * Nxb[0] + up[1] * Nxb[1] + up[2] * Nxb[2];
    const T uaNxa = uNxa + upNxa;
    const double T1b = -rho * uNxb;   // updu(i,c,b) = delta_ic T1b

    // momentum u-u blocks (FLUID.f:494-545)
    const T T1 = mu * NxNx + rho * amd * Nb * (Na + rho * tauM * uaNxa) + rho * Na * (uNxb + upNxb)
               + tauB * upNxa * upNxb;
#pragma unroll
    for (int rr = 0; rr < 3; ++rr)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double updu = (rr == c) ? T1b : 0.0;
            const T T2 = mu * Nxa[c] * Nxb[rr] + tauC * Nxa[rr] * Nxb[c] + S.esNxa[rr] * mug * S.esNxb[c]
                       - rho * tauM * uaNxa * updu;
            k[rr * 4 + c] = k[rr * 4 + c] + wl * ((rr == c) ? T2 + T1 : T2);
        }
    // momentum u-p blocks (FLUID.f:548-557)
    {
        const T T1p = rho * tauM * uaNxa;
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) k[rr * 4 + 3] = k[rr * 4 + 3] - wl * (Nxa[rr] * Nb - Nxb[rr] * T1p);
    }
    // continuity p-u and p-p blocks (FLUID.f:1052-1081)
    {
        const double T1q = rho * amd * Nb;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double T2 = Nxa[c] * (T1b - T1q);
            k[12 + c] = k[12 + c] + wl * (Na * Nxb[c] - tauM * T2);
        }
        k[15] = k[15] + wl * tauM * NxNx;
    }
    if (want_r) {
        // momentum residual (FLUID.f:429-465) and continuity (1046-1049)
        const T pa = G.pp - tauC * E.divU;
        T rVb[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            rVb[c] = tauB * (up[0] * E.ux[0][c] + up[1] * E.ux[1][c] + up[2] * E.ux[2][c]);
        T rM[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double es = E.ux[i][c] + E.ux[c][i];
                rM[i][c] = mu * es - rho * up[c] * ua[i] + rVb[c] * up[i] - (i == c ? pa : scal<T>(0.0));
            }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T rV = ud[c] + ua[0] * E.ux[0][c] + ua[1] * E.ux[1][c] + ua[2] * E.ux[2][c];
            r[c] = r[c] + (wr * Na * rV
                           + w * (Nxa[0] * rM[0][c] + Nxa[1] * rM[1][c] + Nxa[2] * rM[2][c]));
        }
        r[3] = r[3] + w * (Na * E.divU - upNxa);
    }
}

// The coloured scatter path (SVFSI_ASM_GATHER=0): 16 lanes per element, one
// per (a,b) block, read-modify-write of Val.
__global__ __launch_bounds__(256) void k_asm_fluid(int begin, int count, const int* __restrict__ ien,
                                                   const int* __restrict__ elemId,
                                                   const int* __restrict__ emap,
                                                   const double* __restrict__ x, int tDof,
                                                   const double* __restrict__ Ag,
                                                   const double* __restrict__ Yg,
                                                   const double* __restrict__ muEl, AsmParams P,
                                                   Tet4Rule rule, double* __restrict__ val,
                                                   double* __restrict__ R)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count * 16) return;
    const int p = elemId[begin + (t >> 4)];
    const int ab = t & 15;
    const int a = ab >> 2, b = ab & 3;
    FluidElem E;
    fluid_elem(p, ien, x, tDof, Ag, Yg, E);
    double mu, mug;
    fluid_visc(E, P, muEl ? muEl[p] : P.mu, mu, mug);
    double k[16], r[4];
    // the 16 lanes of an element (consecutive lanes of one wave; count * 16
    // threads, so a group is active or inactive as a whole) evaluate the
    // Gauss-point quantities once per point, lane (ab & 3) for point ab & 3,
    // and fetch each point's values from its lane
    FluidGP<double> mine;
    {
        // the point this lane evaluates, selected without dynamic indexing
        FluidGP<double> G;
#pragma unroll
        for (int g = 0; g < 4; ++g)
            if (g == (ab & 3)) fluid_gp_n<double>(E, mu, P, rule.N[g], mine);
        (void)G;
    }
    FluidAB S;
    fluid_ab(E, rule, a, b, S);
    const int base = (threadIdx.x & (kWave - 1)) & ~15;
#pragma unroll
    for (int q = 0; q < 16; ++q) k[q] = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = 0.0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        FluidGP<double> G;
        const int src = base + g;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            G.u[c] = __shfl(mine.u[c], src, kWave);
            G.ud[c] = __shfl(mine.ud[c], src, kWave);
            G.up[c] = __shfl(mine.up[c], src, kWave);
        }
        G.pp = __shfl(mine.pp, src, kWave);
        G.tauM = __shfl(mine.tauM, src, kWave);
        G.tauC = __shfl(mine.tauC, src, kWave);
        G.tauB = __shfl(mine.tauB, src, kWave);
        fluid_pair_gp<double>(E, mu, mug, P, rule, g, G, S, b == 0, k, r);
    }
    double* vb = val + (size_t)emap[(size_t)p * 16 + ab] * 16;
#pragma unroll
    for (int q = 0; q < 16; ++q) vb[q] += k[q];
    if (b == 0) {
        // the node index reloaded from ien: indexing the per-thread E.nd with
        // the lane-dependent a would place the whole element record in
        // scratch memory
        double* Rr = R + (size_t)ien[(size_t)p * 4 + a] * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c) Rr[c] += r[c];
    }
}

// ---------------------------------------------------------------------------
// FLUID gather assembly, two launches.
//
// The (a,b) block of an element, summed over its Gauss points g, needs only
//   u-u  T_ab I + c0 Nx_b Nx_a^T + c1 Nx_a Nx_b^T
//        (+ c4 esNx_a esNx_b^T with a shear-rate dependent viscosity)
//   u-p  Nx_b A_a - c2 Nx_a        p-u  c2 Nx_b + B_b Nx_a
//   p-p  c3 Nx_a.Nx_b
// with wl_g = w_g Jac af gam dt and
//   T_ab = sum_g wl_g [rho am/(af gam dt) N_b (N_a + rho tauM ua.Nx_a) + rho N_a ua.Nx_b
//                      + tauB (u'.Nx_a)(u'.Nx_b) + rho^2 tauM (ua.Nx_a)(u.Nx_b)] + c0 Nx_a.Nx_b
//   A_a = sum_g wl_g rho tauM ua.Nx_a,   B_b = sum_g wl_g tauM rho (u.Nx_b + am/(af gam dt) N_b)
//   c0 = sum_g wl_g mu, c1 = sum_g wl_g tauC, c2 = sum_g wl_g N_b, c3 = sum_g wl_g tauM
// (FLUID.f:494-557, 1052-1081).  k_fluid_rec evaluates these 40 numbers (56
// with esNx) per element, four lanes each, a lane per Gauss point, the sums
// over g by exchanges inside the quad; k_fluid_gather forms and sums the
// blocks of each Val entry from the records of its elements.
//
// What bounds it: the element blocks themselves (2 KB per element) would be
// written and read back, 810 MB on the 197,696-tet cylinder, against 320 B
// per element of record, which the gather mostly finds in L2.  And the
// element arithmetic: geometry and point quantities are evaluated 4 times
// per element instead of 16, and the sum over g is taken once per element
// instead of inside every entry.  FLUID assembly of that mesh: k_fluid_rec 45
// us and k_fluid_gather 80 us, where the element blocks took 315 us (16 lanes
// per element, each its block with the geometry repeated) and their gather
// 119 + 12 us.
// ---------------------------------------------------------------------------
constexpr int FR_T = 0, FR_N = 16, FR_B = 32, FR_C = 36, FR_ES = 40;
template <bool NN> struct FluidRec { static constexpr int SZ = NN ? 56 : 40; };

// Sum over the four lanes of a quad of v[4][W], lane g keeping row g.
template <int W>
__device__ __forceinline__ void quad_rows(int g, const double (&v)[4][W], double (&o)[W])
{
    const bool hi = g & 2, lo = g & 1;
    double m[2][W];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int b = 0; b < W; ++b)
            m[i][b] = (hi ? v[2 + i][b] : v[i][b]) + quad_xor<2>(hi ? v[i][b] : v[2 + i][b]);
#pragma unroll
    for (int b = 0; b < W; ++b) o[b] = (lo ? m[1][b] : m[0][b]) + quad_xor<1>(lo ? m[0][b] : m[1][b]);
}

template <bool NN>
__global__ __launch_bounds__(256) void k_fluid_rec(int nEl, const int* __restrict__ ien,
                                                   const double* __restrict__ x, int tDof,
                                                   const double* __restrict__ Ag, const double* __restrict__ Yg,
                                                   const double* __restrict__ muEl, AsmParams P, Tet4Rule rule,
                                                   double* __restrict__ rec,
                                                   double* __restrict__ re, const int* __restrict__ rslot)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nEl * 4) return;
    const int p = t >> 2, g = t & 3;
    FluidElem E;
    fluid_elem(p, ien, x, tDof, Ag, Yg, E);
    double mu, mug;
    fluid_visc(E, P, muEl ? muEl[p] : P.mu, mu, mug);
    FluidGP<double> G;
    double N[4], wg = 0.0, Nxg[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) N[q] = 0.0;
#pragma unroll
    for (int m = 0; m < 4; ++m)
        if (m == g) {
            wg = rule.w[m];
#pragma unroll
            for (int q = 0; q < 4; ++q) N[q] = rule.N[m][q];
#pragma unroll
            for (int i = 0; i < 3; ++i) Nxg[i] = E.Nx[m][i];
        }
    fluid_gp_n<double>(E, mu, P, N, G);
    const double rho = P.rho;
    const double T1c = P.af * P.gam * P.dt;
    const double amd = P.am / T1c;
    const double w = wg * E.Jac;
    const double wl = w * T1c;
    const double tauM = G.tauM;
    double uN[4], upN[4], uaN[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        uN[a] = G.u[0] * E.Nx[a][0] + G.u[1] * E.Nx[a][1] + G.u[2] * E.Nx[a][2];
        upN[a] = G.up[0] * E.Nx[a][0] + G.up[1] * E.Nx[a][1] + G.up[2] * E.Nx[a][2];
        uaN[a] = uN[a] + upN[a];
    }
    double v[4][6], o[6];
    {
#pragma clang fp contract(fast) // the Jacobian is behind: see the top of the file
        const double ra = rho * amd;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const double adv = rho * tauM * uaN[a];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                v[a][b] = wl * (ra * N[b] * (N[a] + adv) + rho * (N[a] * uaN[b] + adv * uN[b])
                                + G.tauB * upN[a] * upN[b]);
            v[a][4] = wl * adv;
            v[a][5] = wl * tauM * (rho * uN[a] + ra * N[a]);
        }
    }
    quad_rows<6>(g, v, o);
    const double W = quad_sum(wl);
    const double c0 = W * mu, c1 = quad_sum(wl * G.tauC), c2 = quad_sum(wl * N[0]), c3 = quad_sum(wl * tauM);
#pragma unroll
    for (int b = 0; b < 4; ++b)
        o[b] += c0 * (Nxg[0] * E.Nx[b][0] + Nxg[1] * E.Nx[b][1] + Nxg[2] * E.Nx[b][2]);
    double* rc = rec + (size_t)p * FluidRec<NN>::SZ;
    *reinterpret_cast<d2_t*>(rc + FR_T + 4 * g) = d2_t{o[0], o[1]};
    *reinterpret_cast<d2_t*>(rc + FR_T + 4 * g + 2) = d2_t{o[2], o[3]};
    *reinterpret_cast<d2_t*>(rc + FR_N + 4 * g) = d2_t{Nxg[0], Nxg[1]};
    *reinterpret_cast<d2_t*>(rc + FR_N + 4 * g + 2) = d2_t{Nxg[2], o[4]};
    rc[FR_B + g] = o[5];
    rc[FR_C + g] = g == 0 ? c0 : (g == 1 ? c1 : (g == 2 ? c2 : c3));
    if constexpr (NN) {
        double es[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            es[c] = (E.ux[0][c] + E.ux[c][0]) * Nxg[0] + (E.ux[1][c] + E.ux[c][1]) * Nxg[1]
                  + (E.ux[2][c] + E.ux[c][2]) * Nxg[2];
        *reinterpret_cast<d2_t*>(rc + FR_ES + 4 * g) = d2_t{es[0], es[1]};
        *reinterpret_cast<d2_t*>(rc + FR_ES + 4 * g + 2) = d2_t{es[2], W * mug};
    }
    // residual rows (FLUID.f:429-465, 1046-1049)
    const double ua[3] = {G.u[0] + G.up[0], G.u[1] + G.up[1], G.u[2] + G.up[2]};
    const double pa = G.pp - G.tauC * E.divU;
    double rV[3], rVb[3], rM[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        rV[c] = G.ud[c] + ua[0] * E.ux[0][c] + ua[1] * E.ux[1][c] + ua[2] * E.ux[2][c];
        rVb[c] = G.tauB * (G.up[0] * E.ux[0][c] + G.up[1] * E.ux[1][c] + G.up[2] * E.ux[2][c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int i = 0; i < 3; ++i)
            rM[i][c] = mu * (E.ux[i][c] + E.ux[c][i]) - rho * G.up[c] * ua[i] + rVb[c] * G.up[i]
                     - (i == c ? pa : 0.0);
    double rv[4][4], ro[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            rv[a][c] = w * rho * N[a] * rV[c]
                     + w * (E.Nx[a][0] * rM[0][c] + E.Nx[a][1] * rM[1][c] + E.Nx[a][2] * rM[2][c]);
        rv[a][3] = w * (N[a] * E.divU - upN[a]);
    }
    quad_rows<4>(g, rv, ro);
    double* rr = re + (size_t)rslot[t] * 4;
    *reinterpret_cast<d2_t*>(rr) = d2_t{ro[0], ro[1]};
    *reinterpret_cast<d2_t*>(rr + 2) = d2_t{ro[2], ro[3]};
}

// Val from the records (gather_tile) and, in the workgroups from nbVal on, the
// R rows.  The four lanes of a quad load a quarter of a contribution's 112 B
// each and pass it on: two load instructions instead of eight (122 -> 94 us
// before the tiles).
template <bool NN>
__global__ __launch_bounds__(256) void k_fluid_gather(int nNo, unsigned nbVal, const int* __restrict__ tile,
                                                      const int* __restrict__ gPtr, const int* __restrict__ gSrc,
                                                      const double* __restrict__ rec, double* __restrict__ val,
                                                      const int* __restrict__ rPtr, const double* __restrict__ re,
                                                      double* __restrict__ R)
{
    if (blockIdx.x >= nbVal) {
        const unsigned t = (blockIdx.x - nbVal) * 256 + threadIdx.x;
        const int i = (int)(t >> 2), c = (int)(t & 3);
        if (i >= nNo) return;
        const int k1 = rPtr[i + 1];
        double s = 0.0;
#pragma unroll 4
        for (int k = rPtr[i]; k < k1; ++k) s += re[(size_t)k * 4 + c];
        R[(size_t)i * 4 + c] += s;
        return;
    }
    gather_tile<16>(xcd_part(blockIdx.x, nbVal), tile, gPtr, gSrc, val, [&](unsigned src, int r, double (&v)[4]) {
#pragma clang fp contract(fast) // no Jacobian here: see the top of the file
        const bool mom = r < 3;
        const int a = (int)(src >> 2) & 3, b = (int)src & 3;
        const double* rc = rec + (size_t)(src >> 4) * FluidRec<NN>::SZ;
        const d2_t m = *reinterpret_cast<const d2_t*>(rc + FR_N + 4 * (r < 2 ? a : b) + 2 * (r & 1));
        const d2_a8 n = *reinterpret_cast<const d2_a8*>(
            rc + (r == 0 ? FR_C : (r == 1 ? FR_C + 2 : (r == 2 ? FR_T + 4 * a + b : FR_B + b))));
        const d2_t a0 = {quad_get<0>(m.x), quad_get<0>(m.y)}, a1 = {quad_get<1>(m.x), quad_get<1>(m.y)};
        const d2_t b0 = {quad_get<2>(m.x), quad_get<2>(m.y)}, b1 = {quad_get<3>(m.x), quad_get<3>(m.y)};
        const d2_t c01 = {quad_get<0>(n.x), quad_get<0>(n.y)}, c23 = {quad_get<1>(n.x), quad_get<1>(n.y)};
        const double T = quad_get<2>(n.x), Bb = quad_get<3>(n.x);
        const double ar = r == 0 ? a0.x : (r == 1 ? a0.y : a1.x);
        const double br = r == 0 ? b0.x : (r == 1 ? b0.y : b1.x);
        const double fx = mom ? c01.x * br : Bb;     // factor of Nx_a
        const double fy = mom ? c01.y * ar : c23.x;  // factor of Nx_b
        double v0 = fx * a0.x + fy * b0.x;
        double v1 = fx * a0.y + fy * b0.y;
        double v2 = fx * a1.x + fy * b1.x;
        if constexpr (NN) {
            const double ea = rc[FR_ES + 4 * a + r], eb = rc[FR_ES + 4 * b + r]; // lane 3: c4
            const double c4 = quad_get<3>(ea); // by all four lanes, before the choice below
            const double er = mom ? c4 * ea : 0.0;
            v0 += er * quad_get<0>(eb);
            v1 += er * quad_get<1>(eb);
            v2 += er * quad_get<2>(eb);
        }
        v[0] = v0 + (r == 0 ? T : 0.0);
        v[1] = v1 + (r == 1 ? T : 0.0);
        v[2] = v2 + (r == 2 ? T : 0.0);
        v[3] = mom ? br * a1.y - c23.x * ar : c23.y * (a0.x * b0.x + a0.y * b0.y + a1.x * b1.x);
    });
}

// Viscosity sensitivity of the fluid element (no reference counterpart):
// g_e = lam_e^T (dR_e/dmu_e - dK_e/dmu_e du_e), the element term of
// dL/dmu_e when K du = R and K^T lam = dL/du.  Four lanes per element, one
// per Gauss point.  The element matrix is never formed: lam_e^T K_e du_e
// needs the block sums of FLUID3D_M/C only through the values and gradients
// of the two nodal fields at the point (l, lp and Lx, Lpx of lam; D, Dp and
// Dx, Dpx of du), so a lane gathers those with the state's while it reads
// the nodes and evaluates the bilinear form once in dual numbers (mu_e, 1).
// Bound by FP64 arithmetic: the geometry and stabilisation parameters, about
// 700 flops per lane.  One lane per (a, b) block, each repeating the
// geometry and all four points in dual numbers, took 432 us on the
// 197,696-tet cylinder; this takes about 40 us (adjoint terms of one gradient: 454 -> 96 us).
__global__ __launch_bounds__(256) void k_fluid_dmu(int nEl, const int* __restrict__ ien,
                                                   const double* __restrict__ x, int tDof,
                                                   const double* __restrict__ Ag, const double* __restrict__ Yg,
                                                   const double* __restrict__ muEl, AsmParams P, Tet4Rule rule,
                                                   const double* __restrict__ lam,
                                                   const double* __restrict__ du, double* __restrict__ g)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nEl * 4) return;
    const int p = t >> 2, gp = t & 3;
    int nd[4];
    double xl[4][3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        nd[q] = ien[(size_t)p * 4 + q];
#pragma unroll
        for (int i = 0; i < 3; ++i) xl[q][i] = x[(size_t)nd[q] * 3 + i];
    }
    double Nx[4][3], ks[3][3], Jac;
    gnn_tet4(xl, Nx, Jac, ks);
    // N and the weight of this lane's point, without a lane-dependent index
    double N[4], w = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        N[q] = 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m)
            if (m == gp) N[q] = rule.N[m][q];
        if (q == gp) w = rule.w[q] * Jac;
    }
    double u[3] = {0, 0, 0}, ud[3] = {-P.fb[0], -P.fb[1], -P.fb[2]}, pp = 0.0;
    double ux[3][3] = {}, px[3] = {0, 0, 0};
    double l[3] = {0, 0, 0}, lp = 0.0, Lx[3][3] = {}, Lpx[3] = {0, 0, 0};
    double D[3] = {0, 0, 0}, Dp = 0.0, Dx[3][3] = {}, Dpx[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const double* yq = Yg + (size_t)nd[q] * tDof;
        const double* aq = Ag + (size_t)nd[q] * tDof;
        const double* lq = lam + (size_t)nd[q] * 4;
        const double* dq = du + (size_t)nd[q] * 4;
        const double y3 = yq[3], l3 = lq[3], d3 = dq[3];
        pp += N[q] * y3;
        lp += N[q] * l3;
        Dp += N[q] * d3;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            px[i] += Nx[q][i] * y3;
            Lpx[i] += Nx[q][i] * l3;
            Dpx[i] += Nx[q][i] * d3;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double yc = yq[c], lc = lq[c], dc = dq[c];
            u[c] += N[q] * yc;
            ud[c] += N[q] * aq[c];
            l[c] += N[q] * lc;
            D[c] += N[q] * dc;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                ux[i][c] += Nx[q][i] * yc;
                Lx[i][c] += Nx[q][i] * lc;
                Dx[i][c] += Nx[q][i] * dc;
            }
        }
    }
    const double rho = P.rho;
    const Dual mu = {muEl ? muEl[p] : P.mu, 1.0};
    const double divU = ux[0][0] + ux[1][1] + ux[2][2];
    const double divL = Lx[0][0] + Lx[1][1] + Lx[2][2];
    const double divD = Dx[0][0] + Dx[1][1] + Dx[2][2];
    // stabilisation parameters and fine-scale velocity (fluid_gp)
    double kS0 = 0.0, kU = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            kS0 += ks[i][j] * ks[i][j];
            kU += u[i] * u[j] * ks[i][j];
        }
    const Dual kS = 36.0 * kS0 * (mu / rho) * (mu / rho);
    const double kT = 4.0 * (1.0 / P.dt) * (1.0 / P.dt);
    const double trK = ks[0][0] + ks[1][1] + ks[2][2];
    const Dual tauM = 1.0 / (rho * dsqrt(kT + kU + kS));
    const Dual tauC = 1.0 / (tauM * trK);
    Dual up[3], ua[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double rV = ud[c] + u[0] * ux[0][c] + u[1] * ux[1][c] + u[2] * ux[2][c];
        up[c] = -tauM * (rho * rV + px[c]);
        ua[c] = u[c] + up[c];
    }
    Dual tauB = mkd(0.0);
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) tauB = tauB + up[i] * up[j] * ks[i][j];
    if (iszero_d(tauB.v)) tauB = mkd(2.220446049250313e-16);
    tauB = rho / dsqrt(tauB);

    const double T1c = P.af * P.gam * P.dt;
    const double amd = P.am / T1c;
    // lam^T K du (fluid_pair_gp's blocks summed over a and b), over w T1c
    double mm = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int c = 0; c < 3; ++c) mm += Lx[i][c] * (Dx[i][c] + Dx[c][i]);
    Dual k = mu * mm + tauC * (divL * divD) - divL * Dp + lp * divD
           + tauM * (Lpx[0] * Dpx[0] + Lpx[1] * Dpx[1] + Lpx[2] * Dpx[2]);
    // lam^T R: w times the gradient terms, w rho times the inertia
    const Dual pa = pp - tauC * divU;
    Dual r = mkd(lp * divU) - up[0] * Lpx[0] - up[1] * Lpx[1] - up[2] * Lpx[2] - pa * divL;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double uD = u[0] * Dx[0][c] + u[1] * Dx[1][c] + u[2] * Dx[2][c];
        const Dual upL = up[0] * Lx[0][c] + up[1] * Lx[1][c] + up[2] * Lx[2][c];
        const Dual upD = up[0] * Dx[0][c] + up[1] * Dx[1][c] + up[2] * Dx[2][c];
        const Dual uaL = (u[0] * Lx[0][c] + u[1] * Lx[1][c] + u[2] * Lx[2][c]) + upL;
        const Dual upU = up[0] * ux[0][c] + up[1] * ux[1][c] + up[2] * ux[2][c];
        const double uU = u[0] * ux[0][c] + u[1] * ux[1][c] + u[2] * ux[2][c];
        const Dual tL = rho * tauM * uaL;
        const double acc = rho * (amd * D[c] + uD);
        k = k + tL * (acc + Dpx[c]) + (rho * l[c]) * (amd * D[c] + uD + upD) + tauB * upL * upD
          + (tauM * acc) * Lpx[c];
        // rM[i][c] = mu es - rho up_c ua_i + rVb_c up_i, contracted with Lx
        double es = 0.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) es += Lx[i][c] * (ux[i][c] + ux[c][i]);
        r = r + mu * es - rho * up[c] * uaL + tauB * upU * upL + (rho * l[c]) * (ud[c] + uU + upU);
    }
    double s = w * (r.d - T1c * k.d);
    s += __shfl_xor(s, 1, 4);
    s += __shfl_xor(s, 2, 4);
    if (gp == 0) g[p] = s;
}

// ---------------------------------------------------------------------------
// Face terms on tri3 faces (GNNB, svFSI/NN.f:1856-1996).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void gnnb_tri3(const double* x, int n0, int n1, int n2, int inner,
                                          double n[3])
{
    double t1[3], t2[3], v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        t1[i] = x[(size_t)n0 * 3 + i] - x[(size_t)n2 * 3 + i];
        t2[i] = x[(size_t)n1 * 3 + i] - x[(size_t)n2 * 3 + i];
        v[i] = x[(size_t)n0 * 3 + i] - x[(size_t)inner * 3 + i];
    }
    n[0] = t1[1] * t2[2] - t1[2] * t2[1];
    n[1] = t1[2] * t2[0] - t1[0] * t2[2];
    n[2] = t1[0] * t2[1] - t1[1] * t2[0];
    if (n[0] * v[0] + n[1] * v[1] + n[2] * v[2] < 0.0) {
        n[0] = -n[0];
        n[1] = -n[1];
        n[2] = -n[2];
    }
}

// The face terms are gathered like the elements': eight lanes per node (or
// Val block) share its faces, in face order, and meet by shuffles, so a face
// set is one launch whatever its colouring (FaceSet::nPtr, bPtr).  At these
// sizes (a few hundred faces) a launch is all there is to time: one per
// colour took 7 x 1.9 us (36 faces) to 10 x 4.8 us (the outlet of the
// 197,696-tet cylinder), one for the whole set 4-5 us.
constexpr int kFaceLanes = 8;

__device__ __forceinline__ double face_lanes_sum(double v)
{
#pragma unroll
    for (int o = kFaceLanes / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kFaceLanes);
    return v;
}

// SETBCTRACL (svFSI/SETBC.f:319-416): lR(:,a) -= w N_a h.
__global__ __launch_bounds__(256) void k_face_traction(int nNodes, const int* __restrict__ nPtr,
                                                       const int* __restrict__ nSrc, const int* __restrict__ nDst,
                                                       const int* __restrict__ fien, const int* __restrict__ inner,
                                                       const double* __restrict__ x, int dof, double h0, double h1,
                                                       double h2, Tri3Rule rule, double* __restrict__ R)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int i = t / kFaceLanes, l = t % kFaceLanes;
    if (i >= nNodes) return; // whole groups
    const double h[3] = {h0, h1, h2};
    double r[3] = {0, 0, 0};
    for (int k = nPtr[i] + l; k < nPtr[i + 1]; k += kFaceLanes) {
        const int f = nSrc[k] / 3, a = nSrc[k] % 3;
        double n[3];
        gnnb_tri3(x, fien[f * 3], fien[f * 3 + 1], fien[f * 3 + 2], inner[f], n);
        const double Jac = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            const double w = rule.w[g] * Jac;
            const double Na = a == 0 ? rule.N[g][0] : (a == 1 ? rule.N[g][1] : rule.N[g][2]);
#pragma unroll
            for (int c = 0; c < 3; ++c) r[c] -= w * Na * h[c];
        }
    }
    double* Rr = R + (size_t)nDst[i] * dof;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double s = face_lanes_sum(r[c]);
        if (l == c) Rr[c] += s;
    }
}

// BFLUID with h = 0 (svFSI/FLUID.f:1280-1336): the nBlk Val blocks of the
// face set first, then its nodes' rows of R.
__global__ __launch_bounds__(256) void k_face_backflow(int nBlk, const int* __restrict__ bPtr,
                                                       const int* __restrict__ bSrc, const int* __restrict__ bDst,
                                                       int nNodes, const int* __restrict__ nPtr,
                                                       const int* __restrict__ nSrc, const int* __restrict__ nDst,
                                                       const int* __restrict__ fien, const int* __restrict__ inner,
                                                       const double* __restrict__ x, int tDof,
                                                       const double* __restrict__ Yg, AsmParams P, Tri3Rule rule,
                                                       double* __restrict__ val, double* __restrict__ R)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int item = t / kFaceLanes, l = t % kFaceLanes;
    if (item >= nBlk + nNodes) return; // whole groups
    const bool blk = item < nBlk;
    const int i = blk ? item : item - nBlk;
    const int* ptr = blk ? bPtr : nPtr;
    const int* src = blk ? bSrc : nSrc;
    double s[3] = {0, 0, 0}; // a block's diagonal in s[0], or a node's three rows
    for (int k = ptr[i] + l; k < ptr[i + 1]; k += kFaceLanes) {
        const int q = src[k];
        const int f = blk ? q / 9 : q / 3;
        const int a = blk ? (q % 9) / 3 : q % 3, b = q % 3;
        const int nd[3] = {fien[f * 3], fien[f * 3 + 1], fien[f * 3 + 2]};
        double n[3];
        gnnb_tri3(x, nd[0], nd[1], nd[2], inner[f], n);
        const double Jac = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
        const double nV[3] = {n[0] / Jac, n[1] / Jac, n[2] / Jac};
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            const double w = rule.w[g] * Jac;
            double y[3] = {0, 0, 0};
#pragma unroll
            for (int m = 0; m < 3; ++m)
#pragma unroll
                for (int c = 0; c < 3; ++c) y[c] += rule.N[g][m] * Yg[(size_t)nd[m] * tDof + c];
            const double wl = w * P.af * P.gam * P.dt;
            double udn = y[0] * nV[0] + y[1] * nV[1] + y[2] * nV[2];
            udn = 0.5 * P.bstab * P.rho * (udn - fabs(udn));
            const double Na = a == 0 ? rule.N[g][0] : (a == 1 ? rule.N[g][1] : rule.N[g][2]);
            const double Nb = b == 0 ? rule.N[g][0] : (b == 1 ? rule.N[g][1] : rule.N[g][2]);
            if (blk) {
                s[0] -= wl * Na * Nb * udn;
            } else {
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] -= w * Na * (udn * y[c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) s[c] = face_lanes_sum(s[c]);
    if (l >= 3) return;
    if (blk)
        val[(size_t)bDst[i] * 16 + 5 * l] += s[0];
    else
        R[(size_t)nDst[i] * 4 + l] += l == 0 ? s[0] : (l == 1 ? s[1] : s[2]);
}

// LSALLOC's zeroing of both arrays in one launch (16-byte stores where the
// arrays allow).
template <bool V>
__global__ __launch_bounds__(256) void k_zero2(size_t n1, double* __restrict__ a, size_t n2, double* __restrict__ b,
                                               unsigned nb1)
{
    const bool first = blockIdx.x < nb1;
    double* p = first ? a : b;
    const size_t n = first ? n1 : n2;
    const size_t q0 = (size_t)(first ? blockIdx.x : blockIdx.x - nb1) * 2048 + (size_t)threadIdx.x * (V ? 2 : 1);
#pragma unroll
    for (int m = 0; m < (V ? 4 : 8); ++m) {
        const size_t q = q0 + (size_t)m * (V ? 512 : 256);
        if constexpr (V) {
            if (q + 1 < n) *reinterpret_cast<d2_t*>(p + q) = d2_t{0.0, 0.0};
            else if (q < n) p[q] = 0.0;
        } else {
            if (q < n) p[q] = 0.0;
        }
    }
}

int launch_zero2(size_t n1, double* a, size_t n2, double* b, hipStream_t s)
{
    const unsigned nb1 = (unsigned)((n1 + 2047) / 2048), nb2 = (unsigned)((n2 + 2047) / 2048);
    if (nb1 + nb2 == 0) return SVFSI_OK;
    if ((((uintptr_t)a | (uintptr_t)b) & 15) == 0)
        hipLaunchKernelGGL(k_zero2<true>, dim3(nb1 + nb2), dim3(256), 0, s, n1, a, n2, b, nb1);
    else
        hipLaunchKernelGGL(k_zero2<false>, dim3(nb1 + nb2), dim3(256), 0, s, n1, a, n2, b, nb1);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

// ---------------------------------------------------------------------------
// Adjoint: g_e = -lam_e^T (dK_e/dE_e) u_e for the LELAS tet4 tangent.  The
// stiffness part of LELAS3D is proportional to E (lambda, mu ~ E) and the
// mass part does not depend on E, so dK_e/dE_e is the stiffness tangent at
// unit modulus.  One thread per element; element matrices are recomputed,
// never stored.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_lelas_dkde(int nEl, const int* __restrict__ ien,
                                                    const double* __restrict__ x, AsmParams P,
                                                    Tet4Rule rule, const double* __restrict__ lam,
                                                    const double* __restrict__ u,
                                                    double* __restrict__ g)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nEl) return;
    int nd[4];
    double xl[4][3], la[4][3], ub[4][3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        nd[q] = ien[(size_t)p * 4 + q];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            xl[q][i] = x[(size_t)nd[q] * 3 + i];
            la[q][i] = lam[(size_t)nd[q] * 3 + i];
            ub[q][i] = u[(size_t)nd[q] * 3 + i];
        }
    }
    double Nx[4][3], ks[3][3], Jac;
    gnn_tet4(xl, Nx, Jac, ks);
    const double nu = P.nu;
    const double lambda = nu / (1.0 + nu) / (1.0 - 2.0 * nu);
    const double mu = 0.5 / (1.0 + nu);
    const double lDm = lambda / mu;
    const double T1 = P.af * P.beta * P.dt * P.dt;
    double wsum = 0.0;
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) wsum += rule.w[gq] * Jac * T1 * mu;
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const double NxdNx = Nx[a][0] * Nx[b][0] + Nx[a][1] * Nx[b][1] + Nx[a][2] * Nx[b][2];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double v = (i == j) ? NxdNx + (1.0 + lDm) * Nx[a][i] * Nx[b][i]
                                              : lDm * Nx[a][i] * Nx[b][j] + Nx[a][j] * Nx[b][i];
                    s += la[a][i] * (wsum * v) * ub[b][j];
                }
        }
    g[p] = -s;
}

// ---------------------------------------------------------------------------
// STRUCT3D + GETPK2CC nHK (svFSI/STRUCT.f:164-496, MATMODELS.f:41-150,
// 539-564, 1588-1647) in CONSTRUCT_dSOLID (STRUCT.f:39-162), TET10, solid
// viscosity 0, no damping, prestress or fibres.  One wavefront handles EPW
// elements of one colour.  Phase 1: a lane per (element, Gauss point)
// evaluates GNN, F, the neo-Hookean S and Voigt Dm, P = F S and the inertia
// term into an LDS record.  Phase 2: lanes stride over the (element, a, b)
// node pairs, accumulate the 3x3 block over the Gauss points as the
// reference does for that block, and add it to Val through the scatter map;
// the b = 0 lane also builds the residual row of node a.
// ---------------------------------------------------------------------------
// Gauss-point record layout (doubles).  The shape functions come last: the
// material-point records kept in HBM (SR_HBM doubles each) leave them out,
// since N depends only on the rule.
constexpr int SR_W = 0, SR_NX = 1, SR_S = 31, SR_DM = 40, SR_P = 76, SR_UD = 85, SR_F = 88, SR_HBM = 97,
              SR_N = 97, SR_SZ = 107;

__device__ __forceinline__ double det3d(const double A[3][3])
{
    return A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1])
         - A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0])
         + A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
}

// Material point (element e, Gauss point with rule record rg) of STRUCT3D:
// GNN, F, the neo-Hookean S and Voigt Dm (GETPK2CC), P = F S and the inertia
// term, written to the record rc (layout SR_*; N only when WITH_N).
template <bool WITH_N>
__device__ __forceinline__ void struct_point(int e, const int* __restrict__ ien, const double* __restrict__ x,
                                             int tDof, const double* __restrict__ Ag,
                                             const double* __restrict__ Dg, const AsmParams& P,
                                             const double* __restrict__ rg, double* rc)
{
    // GNN (NN.f:1469-1565), streaming the nodes to keep registers low
    double A[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll 2
    for (int a = 0; a < 10; ++a) {
        const int na = ien[(size_t)e * 10 + a];
        double xa[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) xa[i] = x[(size_t)na * 3 + i];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) A[i][j] += xa[i] * rg[11 + a * 3 + j];
    }
    const double J = A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0]
                   + A[0][2] * A[1][0] * A[2][1] - A[0][0] * A[1][2] * A[2][1]
                   - A[0][1] * A[1][0] * A[2][2] - A[0][2] * A[1][1] * A[2][0];
    double B[3][3];
    B[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) / J;
    B[0][1] = (A[2][1] * A[0][2] - A[2][2] * A[0][1]) / J;
    B[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) / J;
    B[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) / J;
    B[1][1] = (A[2][2] * A[0][0] - A[2][0] * A[0][2]) / J;
    B[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) / J;
    B[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) / J;
    B[2][1] = (A[2][0] * A[0][1] - A[2][1] * A[0][0]) / J;
    B[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) / J;
    // Nx (to LDS), F and inertia (STRUCT.f:195-235)
    double F[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    double ud[3] = {-P.rho * P.fb[0], -P.rho * P.fb[1], -P.rho * P.fb[2]};
#pragma unroll 2
    for (int a = 0; a < 10; ++a) {
        const int na = ien[(size_t)e * 10 + a];
        double Nxa[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            Nxa[j] = rg[11 + a * 3] * B[0][j] + rg[11 + a * 3 + 1] * B[1][j] + rg[11 + a * 3 + 2] * B[2][j];
            rc[SR_NX + a * 3 + j] = Nxa[j];
        }
        const double Na = rg[1 + a];
        if constexpr (WITH_N) rc[SR_N + a] = Na;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double Dai = Dg[(size_t)na * tDof + i];
            ud[i] += Na * (P.rho * Ag[(size_t)na * tDof + i]);
#pragma unroll
            for (int j = 0; j < 3; ++j) F[i][j] += Nxa[j] * Dai;
        }
    }
    // GETPK2CC, neo-Hookean + GETSVOLP
    const double nd3 = 3.0;
    const double Jf = det3d(F);
    const double J2d = pow(Jf, -2.0 / nd3);
    double C[3][3], Ci[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) C[i][j] = F[0][i] * F[0][j] + F[1][i] * F[1][j] + F[2][i] * F[2][j];
    {
        const double d = det3d(C);
        Ci[0][0] = (C[1][1] * C[2][2] - C[1][2] * C[2][1]) / d;
        Ci[0][1] = (C[0][2] * C[2][1] - C[0][1] * C[2][2]) / d;
        Ci[0][2] = (C[0][1] * C[1][2] - C[0][2] * C[1][1]) / d;
        Ci[1][0] = (C[1][2] * C[2][0] - C[1][0] * C[2][2]) / d;
        Ci[1][1] = (C[0][0] * C[2][2] - C[0][2] * C[2][0]) / d;
        Ci[1][2] = (C[0][2] * C[1][0] - C[0][0] * C[1][2]) / d;
        Ci[2][0] = (C[1][0] * C[2][1] - C[1][1] * C[2][0]) / d;
        Ci[2][1] = (C[0][1] * C[2][0] - C[0][0] * C[2][1]) / d;
        Ci[2][2] = (C[0][0] * C[1][1] - C[0][1] * C[1][0]) / d;
    }
    double p = 0.0, pl = 0.0;
    const double Kp = P.Kpen;
    if (!iszero_d(Kp)) {
        if (P.volType == 1) { p = Kp * (Jf - 1.0); pl = Kp * (2.0 * Jf - 1.0); }
        else if (P.volType == 3) { p = Kp * (1.0 - 1.0 / Jf); pl = Kp; }
        else { p = 0.5 * Kp * (Jf - 1.0 / Jf); pl = Kp * Jf; }
    }
    const double g1 = 2.0 * P.C10;
    double CSb = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) CSb += C[i][j] * (i == j ? g1 : 0.0);
    const double r1 = J2d * CSb / nd3;
    double Sd[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Sd[i][j] = J2d * (i == j ? g1 : 0.0) - r1 * Ci[i][j];
    const int vi[6][2] = {{0, 0}, {1, 1}, {2, 2}, {0, 1}, {1, 2}, {2, 0}};
#pragma unroll
    for (int aa = 0; aa < 6; ++aa)
#pragma unroll
        for (int bb = 0; bb < 6; ++bb) {
            const int i = vi[aa][0], j = vi[aa][1], kk = vi[bb][0], l = vi[bb][1];
            const double dy1 = Ci[i][j] * Sd[kk][l] + Sd[i][j] * Ci[kk][l];
            const double sym = 0.5 * (Ci[i][kk] * Ci[j][l] + Ci[i][l] * Ci[j][kk]);
            const double dyc = Ci[i][j] * Ci[kk][l];
            rc[SR_DM + aa * 6 + bb] = (-2.0 / nd3) * dy1 + 2.0 * (r1 - p * Jf) * sym + (pl * Jf - 2.0 * r1 / nd3) * dyc;
        }
    double S[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            S[i][j] = Sd[i][j] + p * Jf * Ci[i][j];
            rc[SR_S + i * 3 + j] = S[i][j];
            rc[SR_F + i * 3 + j] = F[i][j];
        }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) rc[SR_P + i * 3 + j] = F[i][0] * S[0][j] + F[i][1] * S[1][j] + F[i][2] * S[2][j];
    rc[SR_W] = rg[0] * J;
#pragma unroll
    for (int i = 0; i < 3; ++i) rc[SR_UD + i] = ud[i];
}

template <int NG, int EPW>
__global__ __launch_bounds__(256) void k_asm_struct(int begin, int count, const int* __restrict__ ien,
                                                   const int* __restrict__ emap, const double* __restrict__ x,
                                                   int tDof, const double* __restrict__ Ag,
                                                   const double* __restrict__ Dg, AsmParams P,
                                                   const double* __restrict__ rule, double* __restrict__ val,
                                                   double* __restrict__ R)
{
    __shared__ double rec[EPW * NG][SR_SZ];
    __shared__ double dbm[EPW * NG][10][18]; // Dm B_b per (element, Gauss point, node b)
    const int lane = threadIdx.x;
    const int e0 = begin + blockIdx.x * EPW;
    const int eEnd = begin + count;
    if (lane < EPW * NG) {
        const int k = lane / NG, g = lane - (lane / NG) * NG;
        const int e = e0 + k;
        double* rc = rec[lane];
        if (e < eEnd) struct_point<true>(e, ien, x, tDof, Ag, Dg, P, rule + g * kTet10Rec, rc);
    }
    __syncthreads();
    // Dm B_b, shared by the ten blocks (a, b) of column b
    for (int idx = lane; idx < EPW * NG * 10; idx += 256) {
        const int kg = idx / 10, b = idx - (idx / 10) * 10;
        if (e0 + kg / NG >= eEnd) continue;
        const double* rc = rec[kg];
        const double* Nxb = rc + SR_NX + b * 3;
        const double* Fg = rc + SR_F;
        double Bb[6][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            Bb[0][c] = Nxb[0] * Fg[c * 3 + 0];
            Bb[1][c] = Nxb[1] * Fg[c * 3 + 1];
            Bb[2][c] = Nxb[2] * Fg[c * 3 + 2];
            Bb[3][c] = Nxb[0] * Fg[c * 3 + 1] + Fg[c * 3 + 0] * Nxb[1];
            Bb[4][c] = Nxb[1] * Fg[c * 3 + 2] + Fg[c * 3 + 1] * Nxb[2];
            Bb[5][c] = Nxb[2] * Fg[c * 3 + 0] + Fg[c * 3 + 2] * Nxb[0];
        }
#pragma unroll
        for (int rr = 0; rr < 6; ++rr)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double sacc = 0.0;
#pragma unroll
                for (int q = 0; q < 6; ++q) sacc += rc[SR_DM + rr * 6 + q] * Bb[q][c];
                dbm[kg][b][rr * 3 + c] = sacc;
            }
    }
    __syncthreads();
    const double afu = P.af * P.beta * P.dt * P.dt;
    const double amd = P.am * P.rho;
    for (int pidx = lane; pidx < EPW * 100; pidx += 256) {
        const int k = pidx / 100, ab = pidx - (pidx / 100) * 100;
        const int a = ab / 10, b = ab - (ab / 10) * 10;
        const int e = e0 + k;
        if (e >= eEnd) continue;
        double kk[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        double r[3] = {0, 0, 0};
#pragma unroll 1
        for (int g = 0; g < NG; ++g) {
            const double* rc = rec[k * NG + g];
            const double w = rc[SR_W];
            const double* Nxa = rc + SR_NX + a * 3;
            const double* Nxb = rc + SR_NX + b * 3;
            const double* Sg = rc + SR_S;
            const double* Fg = rc + SR_F;
            double NxSNx = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int i = 0; i < 3; ++i) NxSNx += Nxa[i] * Sg[i * 3 + j] * Nxb[j];
            const double T1 = amd * rc[SR_N + a] * rc[SR_N + b] + afu * NxSNx;
            double Ba[6][3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Ba[0][c] = Nxa[0] * Fg[c * 3 + 0];
                Ba[1][c] = Nxa[1] * Fg[c * 3 + 1];
                Ba[2][c] = Nxa[2] * Fg[c * 3 + 2];
                Ba[3][c] = Nxa[0] * Fg[c * 3 + 1] + Fg[c * 3 + 0] * Nxa[1];
                Ba[4][c] = Nxa[1] * Fg[c * 3 + 2] + Fg[c * 3 + 1] * Nxa[2];
                Ba[5][c] = Nxa[2] * Fg[c * 3 + 0] + Fg[c * 3 + 2] * Nxa[0];
            }
            const double* DBm = dbm[k * NG + g][b];
#pragma unroll
            for (int rr = 0; rr < 3; ++rr)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double BmDBm = 0.0;
#pragma unroll
                    for (int q = 0; q < 6; ++q) BmDBm += Ba[q][rr] * DBm[q * 3 + c];
                    kk[rr * 3 + c] += w * ((rr == c ? T1 : 0.0) + afu * BmDBm);
                }
            if (b == 0) {
                const double Na = rc[SR_N + a];
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    r[i] += w * (Na * rc[SR_UD + i] + Nxa[0] * rc[SR_P + i * 3] + Nxa[1] * rc[SR_P + i * 3 + 1]
                                 + Nxa[2] * rc[SR_P + i * 3 + 2]);
            }
        }
        double* vb = val + (size_t)emap[(size_t)e * 100 + ab] * 9;
#pragma unroll
        for (int q = 0; q < 9; ++q) vb[q] += kk[q];
        if (b == 0) {
            double* Rr = R + (size_t)ien[(size_t)e * 10 + a] * 3;
#pragma unroll
            for (int i = 0; i < 3; ++i) Rr[i] += r[i];
        }
    }
}

// ---------------------------------------------------------------------------
// STRUCT3D with the B^T Dm B contraction on the matrix cores.
//
// k_struct_points evaluates every material point (element, Gauss point) of
// the mesh in one launch, a lane each, and stores the record (SR_HBM doubles,
// colour-sorted element order) in HBM.  k_asm_struct_mfma then assembles one
// colour: per element the material stiffness
//   K_mat[(a,i),(b,j)] = afu sum_g w_g (B_a,g^T Dm_g B_b,g)_ij
// is the product A^T C of two (6 nG) x 30 matrices, A[(g,q),(a,i)] =
// B_a,g[q][i] and C[(g,q),(b,j)] = afu w_g (Dm_g B_b,g)[q][j] (STRUCT.f:
// 295-319, 348-493), padded to 32 columns and a multiple of 4 rows.  Each
// of its four 16 x 16 output tiles is a chain of 16x16x4 MFMA steps (FP64,
// or FP32 with FP32 accumulation).  The geometric and inertia term
// delta_ij w_g (amd N_a N_b + afu Nx_a.S.Nx_b) and the residual stay on the
// FP64 vector units in the scatter pass.
// ---------------------------------------------------------------------------
template <int NG>
__global__ __launch_bounds__(256) void k_struct_points(int nEl, const int* __restrict__ ien,
                                                      const double* __restrict__ x, int tDof,
                                                      const double* __restrict__ Ag,
                                                      const double* __restrict__ Dg, AsmParams P,
                                                      const double* __restrict__ rule, double* __restrict__ rec)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (size_t)nEl * NG) return;
    const int e = (int)(t / NG), g = (int)(t - (size_t)e * NG);
    struct_point<false>(e, ien, x, tDof, Ag, Dg, P, rule + g * kTet10Rec, rec + t * SR_HBM);
}

// One 16x16x4 MFMA step.  Operands: lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16].  The output item r of lane l is D[row(l, r)][l % 16];
// the row order differs between the FP64 and FP32 instructions (measured
// on gfx950 with random operands).
template <typename MT> struct MfmaTile;
template <> struct MfmaTile<double> {
    typedef double V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V step(double a, double b, V c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return (l >> 4) + 4 * r; }
};
template <> struct MfmaTile<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V step(float a, float b, V c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return 4 * (l >> 4) + r; }
};

template <int NG, typename MT, int EPW>
__global__ __launch_bounds__(256) void k_asm_struct_mfma(int begin, int count, const int* __restrict__ ien,
                                                        const int* __restrict__ emap, AsmParams P,
                                                        const double* __restrict__ rule,
                                                        const double* __restrict__ rec, double* __restrict__ val,
                                                        double* __restrict__ R, double* __restrict__ ke,
                                                        double* __restrict__ re, const int* __restrict__ gslot,
                                                        const int* __restrict__ rslot)
{
    constexpr int KP = (6 * NG + 3) / 4 * 4;   // contraction length, padded to the MFMA depth
    constexpr int OPN = 2 * EPW * KP * 32 > EPW * 1024 ? 2 * EPW * KP * 32 : EPW * 1024;
    constexpr int NTASK = EPW * 4;             // (element, output tile) pairs
    constexpr int TPW = (NTASK + 3) / 4;       // per wave
    typedef typename MfmaTile<MT>::V Acc;
    __shared__ double rs[EPW * NG * SR_HBM];
    __shared__ MT op[OPN];
    MT* Aop = op;                    // [EPW][KP][32]
    MT* Cop = op + EPW * KP * 32;    // [EPW][KP][32]
    MT* Kout = op;                   // [EPW][32][32], after the products
    const int tid = threadIdx.x;
    const int e0 = begin + blockIdx.x * EPW;
    const int nE = min(EPW, begin + count - e0);
    {
        const double* src = rec + (size_t)e0 * NG * SR_HBM;
        for (int i = tid; i < nE * NG * SR_HBM; i += 256) rs[i] = src[i];
    }
    // zero padding: columns 30, 31 of every row, and rows 6 NG .. KP-1
    for (int i = tid; i < EPW * KP * 2; i += 256) {
        const int row = i >> 1, c = 30 + (i & 1);
        Aop[row * 32 + c] = (MT)0;
        Cop[row * 32 + c] = (MT)0;
    }
    if constexpr (KP > 6 * NG) {
        for (int i = tid; i < EPW * (KP - 6 * NG) * 32; i += 256) {
            const int e = i / ((KP - 6 * NG) * 32), r = i - e * ((KP - 6 * NG) * 32);
            Aop[((size_t)e * KP + 6 * NG) * 32 + r] = (MT)0;
            Cop[((size_t)e * KP + 6 * NG) * 32 + r] = (MT)0;
        }
    }
    __syncthreads();
    const double afu = P.af * P.beta * P.dt * P.dt;
    // operands: B_b (rows (g, q), columns (b, j)) and afu w Dm B_b
    for (int t = tid; t < nE * NG * 10; t += 256) {
        const int e = t / (NG * 10), r = t - e * (NG * 10);
        const int g = r / 10, b = r - g * 10;
        const double* rc = rs + (e * NG + g) * SR_HBM;
        const double* Nxb = rc + SR_NX + b * 3;
        const double* Fg = rc + SR_F;
        double Bb[6][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            Bb[0][c] = Nxb[0] * Fg[c * 3 + 0];
            Bb[1][c] = Nxb[1] * Fg[c * 3 + 1];
            Bb[2][c] = Nxb[2] * Fg[c * 3 + 2];
            Bb[3][c] = Nxb[0] * Fg[c * 3 + 1] + Fg[c * 3 + 0] * Nxb[1];
            Bb[4][c] = Nxb[1] * Fg[c * 3 + 2] + Fg[c * 3 + 1] * Nxb[2];
            Bb[5][c] = Nxb[2] * Fg[c * 3 + 0] + Fg[c * 3 + 2] * Nxb[0];
        }
        const double sc = afu * rc[SR_W];
        MT* Ar = Aop + ((size_t)e * KP + g * 6) * 32 + b * 3;
        MT* Cr = Cop + ((size_t)e * KP + g * 6) * 32 + b * 3;
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double d = 0.0;
#pragma unroll
                for (int m = 0; m < 6; ++m) d += rc[SR_DM + q * 6 + m] * Bb[m][c];
                Ar[q * 32 + c] = (MT)Bb[q][c];
                Cr[q * 32 + c] = (MT)(sc * d);
            }
    }
    __syncthreads();
    // products: wave w takes the (element, tile) tasks w, w + 4, ...
    const int wave = tid >> 6, l = tid & 63;
    Acc acc[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
        acc[u] = Acc{0, 0, 0, 0};
        const int task = wave + 4 * u;
        const int e = task >> 2;
        if (task < NTASK && e < nE) { // uniform across the wave
            const int ti = (task >> 1) & 1, tj = task & 1;
            const MT* Ab = Aop + (size_t)e * KP * 32 + (l >> 4) * 32 + 16 * ti + (l & 15);
            const MT* Cb = Cop + (size_t)e * KP * 32 + (l >> 4) * 32 + 16 * tj + (l & 15);
#pragma unroll 6
            for (int s = 0; s < KP / 4; ++s) acc[u] = MfmaTile<MT>::step(Ab[s * 128], Cb[s * 128], acc[u]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
        const int task = wave + 4 * u;
        const int e = task >> 2;
        if (task < NTASK && e < nE) {
            const int ti = (task >> 1) & 1, tj = task & 1;
            MT* Kt = Kout + e * 1024 + 16 * ti * 32 + 16 * tj + (l & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) Kt[MfmaTile<MT>::row(l, r) * 32] = acc[u][r];
        }
    }
    __syncthreads();
    // scatter: geometric + inertia term and the residual in FP64, then Val
    const double amd = P.am * P.rho;
    for (int t = tid; t < nE * 100; t += 256) {
        const int e = t / 100, ab = t - (t / 100) * 100;
        const int a = ab / 10, b = ab - (ab / 10) * 10;
        double T1 = 0.0;
        double r[3] = {0, 0, 0};
#pragma unroll 1
        for (int g = 0; g < NG; ++g) {
            const double* rc = rs + (e * NG + g) * SR_HBM;
            const double* rg = rule + g * kTet10Rec;
            const double w = rc[SR_W];
            const double* Nxa = rc + SR_NX + a * 3;
            const double* Nxb = rc + SR_NX + b * 3;
            const double* Sg = rc + SR_S;
            double NxSNx = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int i = 0; i < 3; ++i) NxSNx += Nxa[i] * Sg[i * 3 + j] * Nxb[j];
            const double Na = rg[1 + a];
            T1 += w * (amd * Na * rg[1 + b] + afu * NxSNx);
            if (b == 0) {
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    r[i] += w * (Na * rc[SR_UD + i] + Nxa[0] * rc[SR_P + i * 3] + Nxa[1] * rc[SR_P + i * 3 + 1]
                                 + Nxa[2] * rc[SR_P + i * 3 + 2]);
            }
        }
        const MT* Kb = Kout + e * 1024 + (3 * a) * 32 + 3 * b;
        if (ke) {
            double* kb = ke + (size_t)gslot[(size_t)(e0 + e) * 100 + ab] * 9;
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) kb[i * 3 + j] = (double)Kb[i * 32 + j] + (i == j ? T1 : 0.0);
            if (b == 0) {
                double* rr = re + (size_t)rslot[(size_t)(e0 + e) * 10 + a] * 3;
#pragma unroll
                for (int i = 0; i < 3; ++i) rr[i] = r[i];
            }
            continue;
        }
        double* vb = val + (size_t)emap[(size_t)(e0 + e) * 100 + ab] * 9;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) vb[i * 3 + j] += (double)Kb[i * 32 + j] + (i == j ? T1 : 0.0);
        if (b == 0) {
            double* Rr = R + (size_t)ien[(size_t)(e0 + e) * 10 + a] * 3;
#pragma unroll
            for (int i = 0; i < 3; ++i) Rr[i] += r[i];
        }
    }
}

// ---------------------------------------------------------------------------
// STRUCT3D, the default kernels: the neo-Hookean tangent as outer products,
// and a row gather.
//
// GETPK2CC's tangent is Dm = -2/3 (Ci x Sd + Sd x Ci) + 2 (r1 - p J) (Ci o Ci)
// + (pl J - 2 r1/3) Ci x Ci with Sd = s I - r1 Ci (s = 2 C10 J^(-2/3), r1 = s
// tr(C)/3), and the strain operator turns a symmetric tensor X into
// B_a^T X = F X Nx_a.  With m_a = F Nx_a and n_a = F Ci Nx_a = F^-T Nx_a
// (F Ci F^T = I) the material and geometric parts of block (a,b) are, at a
// point,
//   -2/3 s (n_a m_b^T + m_a n_b^T) + (pl J + 2 r1/3) n_a n_b^T
//   + (r1 - p J) n_b n_a^T + s (Nx_a.Nx_b) I
// (the (r1 - p J) n_a.n_b of the material part and of Nx_a.S.Nx_b cancel), and
// the residual's F S Nx_a = s m_a - (r1 - p J) n_a.  That is 38 multiply-adds
// per block and point, where the 6x6 contraction B_a^T Dm B_b takes 54 and
// Dm B_b another 108 per node: the vector units need 30 us for the 82,944
// elements of the 24^3 cube at the 4-point rule, less than staging the
// operands for the matrix cores.
//
// k_struct_rec (4 points): a lane per (element, point) writes the point's
// record, with the Jacobian's inverse B (Nx_a = B^T xi_a, xi_a the reference
// gradients): F^-T B^T, F B^T, B B^T and scalars, 30 doubles.
// k_struct_elem: a lane per point and node writes C xi_a, n_a and m_a to LDS
// (15 points: a lane per point, from the mesh), then 50 lanes per element each sum two neighbouring blocks of a row over
// the points and store them, element blocks contiguous (7.2 KB).
// k_struct_rows: a wavefront per node adds the 720-byte strips of its
// elements into the node's row of Val, in LDS, in element-id order.
//
// What bounds it: the element blocks, 600 MB written and read on the 24^3
// cube (82,944 elements), and the latency of the records' node gathers.  There
// 661 us, against 1412 with B^T Dm B on the matrix cores and a coloured
// scatter (30 launches, each a read-modify-write of scattered 72-byte blocks,
// 1.22 ms); 4,374 elements with 15 points: 559 -> 67 us.  Strips formed in the
// row kernel from the records, without the blocks' trip through memory, took
// 660 and 130 us (two or three wavefronts per SIMD, a serial chain each).
// ---------------------------------------------------------------------------
constexpr int SP_N = 0, SP_M = 9, SP_C = 18, SP_K = 24, SP_UD = 27, SP_SZ = 30; // point record
constexpr int SN_SZ = 10;        // per node: C xi (without records Nx), n, m (scaled), pad
constexpr int SQ_C = 10 * SN_SZ; // then kap, gam, w, w times the inertia
constexpr int SQ_WS = SQ_C + 6;  // then, without records, w s
template <bool REC> struct StructLds { static constexpr int SZ = REC ? SQ_WS : SQ_WS + 2; };

// Kinematics and neo-Hookean scalars of a point: the Jacobian's inverse B, F,
// F^-T, the inertia ud, w, w s, -2/3 w s, w (pl J + 2 r1/3) and w (r1 - p J).
struct StructPoint {
    double B[3][3], F[3][3], Fi[3][3], ud[3], w, ws, cm, kap, gam;
};

// nx(a, Nx_a) is called for each node on the way.
template <class NX>
__device__ __forceinline__ void struct_point(int e, const int* __restrict__ ien, const double* __restrict__ x, int tDof,
                                             const double* __restrict__ Ag, const double* __restrict__ Dg,
                                             const AsmParams& P, const double* __restrict__ rg, StructPoint& S, NX&& nx)
{
    double (&B)[3][3] = S.B;
    double (&F)[3][3] = S.F;
    double (&Fi)[3][3] = S.Fi;
    double (&ud)[3] = S.ud;
    double A[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll 5
    for (int a = 0; a < 10; ++a) {
        const int na = ien[(size_t)e * 10 + a];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double xi = x[(size_t)na * 3 + i];
#pragma unroll
            for (int j = 0; j < 3; ++j) A[i][j] += xi * rg[11 + a * 3 + j];
        }
    }
    const double J = A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0]
                   + A[0][2] * A[1][0] * A[2][1] - A[0][0] * A[1][2] * A[2][1]
                   - A[0][1] * A[1][0] * A[2][2] - A[0][2] * A[1][1] * A[2][0];
    B[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) / J;
    B[0][1] = (A[2][1] * A[0][2] - A[2][2] * A[0][1]) / J;
    B[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) / J;
    B[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) / J;
    B[1][1] = (A[2][2] * A[0][0] - A[2][0] * A[0][2]) / J;
    B[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) / J;
    B[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) / J;
    B[2][1] = (A[2][0] * A[0][1] - A[2][1] * A[0][0]) / J;
    B[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) / J;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        ud[i] = -P.rho * P.fb[i];
#pragma unroll
        for (int j = 0; j < 3; ++j) F[i][j] = i == j ? 1.0 : 0.0;
    }
#pragma unroll 5
    for (int a = 0; a < 10; ++a) {
        const int na = ien[(size_t)e * 10 + a];
        double Nxa[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            Nxa[j] = rg[11 + a * 3] * B[0][j] + rg[11 + a * 3 + 1] * B[1][j] + rg[11 + a * 3 + 2] * B[2][j];
        }
        nx(a, Nxa);
        const double Na = rg[1 + a];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double Dai = Dg[(size_t)na * tDof + i];
            ud[i] += Na * (P.rho * Ag[(size_t)na * tDof + i]);
#pragma unroll
            for (int j = 0; j < 3; ++j) F[i][j] += Nxa[j] * Dai;
        }
    }
    const double Jf = det3d(F);
    Fi[0][0] = (F[1][1] * F[2][2] - F[1][2] * F[2][1]) / Jf;
    Fi[0][1] = (F[1][2] * F[2][0] - F[1][0] * F[2][2]) / Jf;
    Fi[0][2] = (F[1][0] * F[2][1] - F[1][1] * F[2][0]) / Jf;
    Fi[1][0] = (F[0][2] * F[2][1] - F[0][1] * F[2][2]) / Jf;
    Fi[1][1] = (F[0][0] * F[2][2] - F[0][2] * F[2][0]) / Jf;
    Fi[1][2] = (F[0][1] * F[2][0] - F[0][0] * F[2][1]) / Jf;
    Fi[2][0] = (F[0][1] * F[1][2] - F[0][2] * F[1][1]) / Jf;
    Fi[2][1] = (F[0][2] * F[1][0] - F[0][0] * F[1][2]) / Jf;
    Fi[2][2] = (F[0][0] * F[1][1] - F[0][1] * F[1][0]) / Jf;
    double p = 0.0, pl = 0.0, trC = 0.0;
    const double Kp = P.Kpen;
    if (!iszero_d(Kp)) {
        if (P.volType == 1) { p = Kp * (Jf - 1.0); pl = Kp * (2.0 * Jf - 1.0); }
        else if (P.volType == 3) { p = Kp * (1.0 - 1.0 / Jf); pl = Kp; }
        else { p = 0.5 * Kp * (Jf - 1.0 / Jf); pl = Kp * Jf; }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) trC += F[i][j] * F[i][j];
    const double s = pow(Jf, -2.0 / 3.0) * (2.0 * P.C10);
    const double r1 = s * trC / 3.0;
    S.w = rg[0] * J;
    S.ws = S.w * s;
    S.cm = -2.0 / 3.0 * S.ws;
    S.kap = S.w * (pl * Jf + 2.0 * r1 / 3.0);
    S.gam = S.w * (r1 - p * Jf);
}

// Record of point g of element e: F^-T B^T, w (-2/3 s) F B^T, w s B B^T (00, 11,
// 22, 01, 02, 12), w (pl J + 2 r1/3), w (r1 - p J), w and w times the inertia.
__device__ __forceinline__ void struct_point_rec(int e, const int* __restrict__ ien, const double* __restrict__ x,
                                                 int tDof, const double* __restrict__ Ag,
                                                 const double* __restrict__ Dg, const AsmParams& P,
                                                 const double* __restrict__ rg, double* out)
{
    StructPoint S;
    struct_point(e, ien, x, tDof, Ag, Dg, P, rg, S, [](int, const double (&)[3]) {});
    const double (&B)[3][3] = S.B;
    const double (&F)[3][3] = S.F;
    const double (&Fi)[3][3] = S.Fi;
    const double ws = S.ws, cm = S.cm;
    double o[SP_SZ];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            o[SP_N + 3 * i + k] = Fi[i][0] * B[k][0] + Fi[i][1] * B[k][1] + Fi[i][2] * B[k][2];
            o[SP_M + 3 * i + k] = cm * (F[i][0] * B[k][0] + F[i][1] * B[k][1] + F[i][2] * B[k][2]);
        }
    auto bb = [&](int k, int m) { return ws * (B[k][0] * B[m][0] + B[k][1] * B[m][1] + B[k][2] * B[m][2]); };
    o[SP_C] = bb(0, 0);
    o[SP_C + 1] = bb(1, 1);
    o[SP_C + 2] = bb(2, 2);
    o[SP_C + 3] = bb(0, 1);
    o[SP_C + 4] = bb(0, 2);
    o[SP_C + 5] = bb(1, 2);
    o[SP_K] = S.kap;
    o[SP_K + 1] = S.gam;
    o[SP_K + 2] = S.w;
#pragma unroll
    for (int i = 0; i < 3; ++i) o[SP_UD + i] = S.w * S.ud[i];
    // 240 bytes: 16-byte aligned
#pragma unroll
    for (int q = 0; q < SP_SZ / 2; ++q) *reinterpret_cast<d2_t*>(out + 2 * q) = d2_t{o[2 * q], o[2 * q + 1]};
}

// The same point's node vectors, straight to LDS (SN_SZ doubles a node): Nx_a,
// n_a and w (-2/3 s) m_a; then the scalars of SQ_C and w s.
__device__ __forceinline__ void struct_point_vec(int e, const int* __restrict__ ien, const double* __restrict__ x,
                                                 int tDof, const double* __restrict__ Ag,
                                                 const double* __restrict__ Dg, const AsmParams& P,
                                                 const double* __restrict__ rg, double* rc)
{
    StructPoint S;
    struct_point(e, ien, x, tDof, Ag, Dg, P, rg, S, [rc](int a, const double (&Nxa)[3]) {
#pragma unroll
        for (int j = 0; j < 3; ++j) rc[a * SN_SZ + j] = Nxa[j];
    });
    rc[SQ_C] = S.kap;
    rc[SQ_C + 1] = S.gam;
    rc[SQ_C + 2] = S.w;
#pragma unroll
    for (int i = 0; i < 3; ++i) rc[SQ_C + 3 + i] = S.w * S.ud[i];
    rc[SQ_WS] = S.ws;
#pragma unroll 5
    for (int a = 0; a < 10; ++a) {
        double* na = rc + a * SN_SZ;
        const double n0 = na[0], n1 = na[1], n2 = na[2];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            na[3 + i] = S.Fi[i][0] * n0 + S.Fi[i][1] * n1 + S.Fi[i][2] * n2;
            na[6 + i] = S.cm * (S.F[i][0] * n0 + S.F[i][1] * n1 + S.F[i][2] * n2);
        }
    }
}

__global__ __launch_bounds__(256) void k_struct_rec(int nEl, int nG, const int* __restrict__ ien,
                                                    const double* __restrict__ x, int tDof,
                                                    const double* __restrict__ Ag, const double* __restrict__ Dg,
                                                    AsmParams P, const double* __restrict__ rule,
                                                    double* __restrict__ rec)
{
    const int id = blockIdx.x * 256 + threadIdx.x, e = id / nG;
    if (e < nEl)
        struct_point_rec(e, ien, x, tDof, Ag, Dg, P, rule + (id - e * nG) * kTet10Rec, rec + (size_t)id * SP_SZ);
}

// Element blocks.  With 15 points 75 lanes of a workgroup take a point each,
// from the mesh to its node vectors, for five elements: 67 us per call at 4,374
// elements and 183 at 16,464, against 79 and 214 for two elements in 128 lanes
// that left point records in LDS first (a launch of its own for the records
// takes 18 us alone).  With 4 points, where 20 lanes would be busy, the records
// come from k_struct_rec (REC; 82,944 elements: 62 + 281 us against 430).
template <int NG, int EPW, int NT, bool REC>
__global__ __launch_bounds__(NT) void k_struct_elem(int nEl, const int* __restrict__ ien,
                                                    const double* __restrict__ x, int tDof,
                                                    const double* __restrict__ Ag, const double* __restrict__ Dg,
                                                    AsmParams P, const double* __restrict__ rule,
                                                    const double* __restrict__ recs, double* __restrict__ ke,
                                                    double* __restrict__ re)
{
#pragma clang fp contract(fast) // the Jacobians are behind: see the top of the file
    static_assert(EPW * 50 <= NT, "one pass of lanes in the second phase");
    __shared__ __align__(16) double pt[EPW * NG][StructLds<REC>::SZ];
    constexpr int XN = REC ? 3 : 0;
    __shared__ __align__(16) double sX[NG * 10][XN + 1]; // reference gradient (with records) and N
    const int tid = threadIdx.x;
    const int e0 = blockIdx.x * EPW;
    for (int q = tid; q < NG * 10 * (XN + 1); q += NT) {
        const int n = q / (XN + 1), c = q - n * (XN + 1), g = n / 10, a = n - 10 * g;
        sX[n][c] = rule[g * kTet10Rec + (c < XN ? 11 + 3 * a + c : 1 + a)];
    }
    const int nPt = min(EPW, nEl - e0) * NG;
    if constexpr (REC) {
        for (int q = tid; q < nPt * 10; q += NT) {
            const int p = q / 10, a = q - 10 * p, g = p % NG;
            const d2_t* rc = reinterpret_cast<const d2_t*>(recs + ((size_t)e0 * NG + p) * SP_SZ);
            double o[SP_SZ];
#pragma unroll
            for (int u = 0; u < SP_SZ / 2; ++u) {
                const d2_t v = rc[u];
                o[2 * u] = v.x;
                o[2 * u + 1] = v.y;
            }
            const double* xi = rule + g * kTet10Rec + 11 + 3 * a;
            const double x0 = xi[0], x1 = xi[1], x2 = xi[2];
            double* n = pt[p] + a * SN_SZ;
            n[0] = o[SP_C] * x0 + o[SP_C + 3] * x1 + o[SP_C + 4] * x2;
            n[1] = o[SP_C + 3] * x0 + o[SP_C + 1] * x1 + o[SP_C + 5] * x2;
            n[2] = o[SP_C + 4] * x0 + o[SP_C + 5] * x1 + o[SP_C + 2] * x2;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                n[3 + c] = o[SP_N + 3 * c] * x0 + o[SP_N + 3 * c + 1] * x1 + o[SP_N + 3 * c + 2] * x2;
                n[6 + c] = o[SP_M + 3 * c] * x0 + o[SP_M + 3 * c + 1] * x1 + o[SP_M + 3 * c + 2] * x2;
            }
            if (a < 6) pt[p][SQ_C + a] = a == 0 ? o[SP_K] : a == 1 ? o[SP_K + 1] : a == 2 ? o[SP_K + 2]
                                         : a == 3 ? o[SP_UD] : a == 4 ? o[SP_UD + 1] : o[SP_UD + 2];
        }
    } else {
        static_assert(EPW * NG <= NT, "a lane per point");
        if (tid < nPt)
            struct_point_vec(e0 + tid / NG, ien, x, tDof, Ag, Dg, P, rule + tid % NG * kTet10Rec, pt[tid]);
    }
    __syncthreads();
    const int k = tid / 50, r = tid - k * 50, e = e0 + k;
    if (k >= EPW || e >= nEl) return;
    {
#pragma clang fp contract(fast) // the Jacobians are behind: see the top of the file
        const int a = r / 5, b0 = 2 * (r - 5 * a);
        double K[2][9], T[2] = {0, 0}, M[2] = {0, 0}, R[3] = {0, 0, 0};
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 9; ++q) K[h][q] = 0.0;
#pragma unroll 1
        for (int g = 0; g < NG; ++g) {
            const double* rc = pt[k * NG + g];
            double na[SN_SZ];
#pragma unroll
            for (int q = 0; q < SN_SZ / 2; ++q) {
                const d2_t v = *reinterpret_cast<const d2_t*>(rc + a * SN_SZ + 2 * q);
                na[2 * q] = v.x;
                na[2 * q + 1] = v.y;
            }
            const double kap = rc[SQ_C], gam = rc[SQ_C + 1], w = rc[SQ_C + 2];
            const double Na = sX[g * 10 + a][XN];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                double nb[SN_SZ];
#pragma unroll
                for (int q = REC ? 1 : 0; q < SN_SZ / 2; ++q) {
                    const d2_t v = *reinterpret_cast<const d2_t*>(rc + (b0 + h) * SN_SZ + 2 * q);
                    nb[2 * q] = v.x;
                    nb[2 * q + 1] = v.y;
                }
                const double* xb = sX[g * 10 + b0 + h];
                if constexpr (REC) T[h] += na[0] * xb[0] + na[1] * xb[1] + na[2] * xb[2];
                else T[h] += rc[SQ_WS] * (na[0] * nb[0] + na[1] * nb[1] + na[2] * nb[2]);
                M[h] += w * (Na * xb[XN]);
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double eb = kap * nb[3 + j] + nb[6 + j]; // n_a's partner
                    const double ga = gam * na[3 + j];             // n_b's, transposed
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        K[h][i * 3 + j] += na[3 + i] * eb + na[6 + i] * nb[3 + j] + nb[3 + i] * ga;
                }
            }
            if (b0 == 0) {
#pragma unroll
                for (int i = 0; i < 3; ++i) R[i] += Na * rc[SQ_C + 3 + i] - 1.5 * na[6 + i] - gam * na[3 + i];
            }
        }
        const double afu = P.af * P.beta * P.dt * P.dt, amd = P.am * P.rho;
        double* o = ke + ((size_t)e * 100 + a * 10 + b0) * 9; // two blocks: 144 B, 16-byte aligned
        double v[18];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 9; ++q) v[9 * h + q] = afu * K[h][q] + (q % 4 == 0 ? amd * M[h] + afu * T[h] : 0.0);
#pragma unroll
        for (int q = 0; q < 9; ++q) *reinterpret_cast<d2_t*>(o + 2 * q) = d2_t{v[2 * q], v[2 * q + 1]};
        if (b0 == 0) {
            double* rr = re + ((size_t)e * 10 + a) * 3;
#pragma unroll
            for (int i = 0; i < 3; ++i) rr[i] = R[i];
        }
    }
}

// Row of Val and of R of node i: a wavefront adds the strips ke[(e, a)][0..89]
// of the node's elements (rSrc = 10 e + a, in element-id order) into LDS.  Its
// LDS additions are issued strip by strip and complete in that order, and a
// strip's 90 values go to 90 places, so the sums are in element order; four
// strips' loads are in flight.
__global__ __launch_bounds__(256) void k_struct_rows(int nNo, int maxRow, const int* __restrict__ rowPtr,
                                                     const int* __restrict__ rPtr, const int* __restrict__ rSrc,
                                                     const int* __restrict__ emap, const double* __restrict__ ke,
                                                     const double* __restrict__ re, double* __restrict__ val,
                                                     double* __restrict__ R)
{
    extern __shared__ double accs[];
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int i = (int)xcd_part(blockIdx.x, gridDim.x) * 4 + wave;
    if (i >= nNo) return;
    double* acc = accs + (size_t)wave * maxRow * 9;
    const int k0 = rowPtr[i], nv = (rowPtr[i + 1] - k0) * 9;
    for (int q = l; q < nv; q += 64) acc[q] = 0.0;
    // the additions below are by other lanes than the zeroing
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int b1 = l / 9, q1 = l - 9 * b1;               // value l of a strip
    const int b2 = (l + 64) / 9, q2 = l + 64 - 9 * b2;   // value l + 64, l < 26
    const int s1 = rPtr[i + 1];
    double r = 0.0;
    for (int s = rPtr[i]; s < s1; s += 4) {
        double u[4], v[4], rv[4];
        int m[4], n[4];
#pragma unroll
        for (int h = 0; h < 4; ++h)
            if (s + h < s1) {
                const size_t src = (size_t)rSrc[s + h];
                m[h] = emap[src * 10 + b1];
                u[h] = ke[src * 90 + l];
                n[h] = l < 26 ? emap[src * 10 + b2] : 0;
                v[h] = l < 26 ? ke[src * 90 + l + 64] : 0.0;
                rv[h] = l < 3 ? re[src * 3 + l] : 0.0;
            }
#pragma unroll
        for (int h = 0; h < 4; ++h)
            if (s + h < s1) {
                __hip_atomic_fetch_add(acc + (size_t)(m[h] - k0) * 9 + q1, u[h], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
                if (l < 26)
                    __hip_atomic_fetch_add(acc + (size_t)(n[h] - k0) * 9 + q2, v[h], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                r += rv[h];
            }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    double* o = val + (size_t)k0 * 9;
    for (int q = l; q < nv; q += 64) o[q] += acc[q];
    if (l < 3) R[(size_t)i * 3 + l] += r;
}

// ---------------------------------------------------------------------------
// Gather assembly: Val(:, j) += the sum of the element blocks that land on
// nnz block j, R(:, i) += the sum of node i's element residual rows.  The
// element kernels stored those contributions contiguously, in element-id
// order (DOASSEM's element loop, LHSA.f:266-298), so each sum is a streaming
// read, deterministic, and associates like the reference's.  DD consecutive
// lanes share one block.
// ---------------------------------------------------------------------------
template <int DD>
__global__ __launch_bounds__(256) void k_gather(size_t nItems, const int* __restrict__ ptr,
                                               const double* __restrict__ src, double* __restrict__ dst)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t j = t / DD;
    if (j >= nItems) return;
    const int q = (int)(t - j * DD);
    const int k1 = ptr[j + 1];
    double sum = 0.0;
    int k = ptr[j];
    // four loads in flight, added in element order (the sums associate as
    // DOASSEM's element loop does)
    for (; k + 4 <= k1; k += 4) {
        const double a0 = src[(size_t)k * DD + q], a1 = src[(size_t)(k + 1) * DD + q];
        const double a2 = src[(size_t)(k + 2) * DD + q], a3 = src[(size_t)(k + 3) * DD + q];
        sum += a0;
        sum += a1;
        sum += a2;
        sum += a3;
    }
    for (; k < k1; ++k) sum += src[(size_t)k * DD + q];
    dst[j * DD + q] += sum;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Whether tet4 assembly goes through records and a gather, and whether STRUCT's
// matrix-core kernels, when selected, store their blocks for k_gather instead of
// scattering them colour by colour.  Not by default there: 5.8 ms against 5.0
// on the 40^3 tet10 cube, since 72-byte blocks straddle cache lines (the default
// STRUCT kernels are others, launch_asm_struct).  SVFSI_ASM_GATHER = 0 / 1
// overrides.
static bool gather_enabled(int eNoN)
{
    const char* v = getenv("SVFSI_ASM_GATHER");
    if (v && (v[0] == '0' || v[0] == '1')) return v[0] == '1';
    return eNoN == 4;
}

int launch_gather(Mesh& M, int dof, double* val, double* R, hipStream_t s)
{
    const size_t nb = (size_t)M.lhs->nnz, nr = (size_t)M.nNo;
    const double* ke = M.ke.as<double>();
    const double* re = M.re.as<double>();
    auto grid = [](size_t items, int dd) { return dim3((unsigned)((items * dd + 255) / 256)); };
    if (dof == 3) {
        hipLaunchKernelGGL(k_gather<9>, grid(nb, 9), dim3(256), 0, s, nb, M.gPtr.as<int>(), ke, val);
        hipLaunchKernelGGL(k_gather<3>, grid(nr, 3), dim3(256), 0, s, nr, M.rPtr.as<int>(), re, R);
    } else {
        hipLaunchKernelGGL(k_gather<16>, grid(nb, 16), dim3(256), 0, s, nb, M.gPtr.as<int>(), ke, val);
        hipLaunchKernelGGL(k_gather<4>, grid(nr, 4), dim3(256), 0, s, nr, M.rPtr.as<int>(), re, R);
    }
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

template <bool NN>
static int launch_fluid_rec(Mesh& M, const AsmParams& P, const Tet4Rule& rule, int tDof, const double* Ag,
                            const double* Yg, const double* muEl, double* val, double* R, hipStream_t s)
{
    SV_TRY(M.ke.ensure((size_t)M.nEl * FluidRec<NN>::SZ * sizeof(double)));
    double* rec = M.ke.as<double>();
    double* re = M.re.as<double>();
    hipLaunchKernelGGL(k_fluid_rec<NN>, dim3((unsigned)(((size_t)M.nEl * 4 + 255) / 256)), dim3(256), 0, s, M.nEl,
                       M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Yg, muEl, P, rule, rec, re,
                       M.rSlot.as<int>());
    const unsigned nbVal = (unsigned)M.nGTile;
    const unsigned nbR = (unsigned)(((size_t)M.nNo * 4 + 255) / 256);
    hipLaunchKernelGGL(k_fluid_gather<NN>, dim3(nbVal + nbR), dim3(256), 0, s, M.nNo, nbVal, M.gTile.as<int>(),
                       M.gPtr.as<int>(), M.gSrc.as<int>(), (const double*)rec, val, M.rPtr.as<int>(),
                       (const double*)re, R);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

int launch_asm_tet4(Mesh& M, int phys, const AsmParams& P, const Tet4Rule& rule, int tDof, const double* Ag,
                    const double* Yg, const double* Dg, const double* prop, double* val, double* R, hipStream_t s)
{
    const int dof = phys == SVFSI_PHYS_LELAS ? 3 : 4;
    if (gather_enabled(M.eNoN)) {
        SV_TRY(M.re.ensure((size_t)M.nEl * 4 * dof * sizeof(double)));
        if (phys == SVFSI_PHYS_LELAS) {
            SV_TRY(M.ke.ensure((size_t)M.nEl * LR_SZ * sizeof(double)));
            double* rec = M.ke.as<double>();
            double* re = M.re.as<double>();
            hipLaunchKernelGGL(k_lelas_rec, dim3((unsigned)(((size_t)M.nEl * 4 + 255) / 256)), dim3(256), 0, s, M.nEl,
                               M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Dg, prop, P, rule, rec, re,
                               M.rSlot.as<int>());
            const unsigned nbVal = (unsigned)M.nGTile;
            const unsigned nbR = (unsigned)(((size_t)M.nNo * 3 + 255) / 256);
            hipLaunchKernelGGL(k_lelas_gather, dim3(nbVal + nbR), dim3(256), 0, s, M.nNo, nbVal, M.gTile.as<int>(),
                               M.gPtr.as<int>(), M.gSrc.as<int>(), (const double*)rec, val, M.rPtr.as<int>(),
                               (const double*)re, R);
            SV_HIP(hipGetLastError());
            return SVFSI_OK;
        }
        // mu_g is zero with the constant viscosity, whose record leaves esNx out
        if (P.viscType == SVFSI_VISC_CONST) return launch_fluid_rec<false>(M, P, rule, tDof, Ag, Yg, prop, val, R, s);
        return launch_fluid_rec<true>(M, P, rule, tDof, Ag, Yg, prop, val, R, s);
    }
    const int nC = (int)M.colorOff.size() - 1;
    for (int c = 0; c < nC; ++c) {
        const int begin = M.colorOff[c], count = M.colorOff[c + 1] - begin;
        if (count == 0) continue;
        const unsigned grid = (unsigned)((count * 16 + 255) / 256);
        if (phys == SVFSI_PHYS_LELAS)
            hipLaunchKernelGGL(k_asm_lelas, dim3(grid), dim3(256), 0, s, begin, count, M.ien.as<int>(),
                               M.elemId.as<int>(), M.emap.as<int>(), M.x.as<double>(), tDof, Ag, Dg, prop,
                               P, rule, val, R);
        else
            hipLaunchKernelGGL(k_asm_fluid, dim3(grid), dim3(256), 0, s, begin, count, M.ien.as<int>(),
                               M.elemId.as<int>(), M.emap.as<int>(), M.x.as<double>(), tDof, Ag, Yg, prop,
                               P, rule, val, R);
    }
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

static dim3 face_grid(int items) { return dim3((unsigned)(((size_t)items * kFaceLanes + 255) / 256)); }

int launch_face_traction(const Mesh& M, const Mesh::FaceSet& F, int dof, const double* h,
                         const Tri3Rule& rule, double* R, hipStream_t s)
{
    if (F.nNodes == 0) return SVFSI_OK;
    hipLaunchKernelGGL(k_face_traction, face_grid(F.nNodes), dim3(256), 0, s, F.nNodes, F.nPtr.as<int>(),
                       F.nSrc.as<int>(), F.nDst.as<int>(), F.fien.as<int>(), F.inner.as<int>(), M.x.as<double>(), dof,
                       h[0], h[1], h[2], rule, R);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

int launch_face_backflow(const Mesh& M, const Mesh::FaceSet& F, const AsmParams& P, int tDof,
                         const double* Yg, const Tri3Rule& rule, double* val, double* R, hipStream_t s)
{
    if (F.nNodes == 0) return SVFSI_OK;
    hipLaunchKernelGGL(k_face_backflow, face_grid(F.nBlk + F.nNodes), dim3(256), 0, s, F.nBlk, F.bPtr.as<int>(),
                       F.bSrc.as<int>(), F.bDst.as<int>(), F.nNodes, F.nPtr.as<int>(), F.nSrc.as<int>(),
                       F.nDst.as<int>(), F.fien.as<int>(), F.inner.as<int>(), M.x.as<double>(), tDof, Yg, P, rule,
                       val, R);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

int launch_fluid_dmu(const Mesh& M, const AsmParams& P, const Tet4Rule& rule, int tDof, const double* Ag,
                     const double* Yg, const double* muEl, const double* lam, const double* du, double* g,
                     hipStream_t s)
{
    if (M.nEl == 0) return SVFSI_OK;
    const unsigned grid = (unsigned)(((size_t)M.nEl * 4 + 255) / 256);
    hipLaunchKernelGGL(k_fluid_dmu, dim3(grid), dim3(256), 0, s, M.nEl, M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Yg, muEl, P, rule, lam, du, g);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

int launch_lelas_dkde(const Mesh& M, const AsmParams& P, const Tet4Rule& rule, const double* lam,
                      const double* u, double* g, hipStream_t s)
{
    if (M.nEl == 0) return SVFSI_OK;
    hipLaunchKernelGGL(k_lelas_dkde, dim3((M.nEl + 255) / 256), dim3(256), 0, s, M.nEl, M.ien.as<int>(),
                       M.x.as<double>(), P, rule, lam, u, g);
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

// Scratch of the outer-product kernels: 7.44 KB per element, and 960 B of point
// records with four points.  false: not to be had, or more than
// SVFSI_ASM_SCRATCH_MB allows; what was taken is given back to the coloured
// kernels that run instead, whose points take 3.1 KB per element with four
// points (11.6 KB with 15).
static bool struct_scratch(Mesh& M, int nG)
{
    const size_t ke = (size_t)M.nEl * 100 * 9 * sizeof(double), re = (size_t)M.nEl * 10 * 3 * sizeof(double);
    const size_t rec = nG == 4 ? (size_t)M.nEl * nG * SP_SZ * sizeof(double) : 0;
    const char* v = getenv("SVFSI_ASM_SCRATCH_MB");
    if (v && ke + re + rec > (size_t)strtoull(v, nullptr, 10) << 20) return false;
    if (M.ke.ensure(ke) == SVFSI_OK && M.re.ensure(re) == SVFSI_OK && (!rec || M.srec.ensure(rec) == SVFSI_OK))
        return true;
    (void)hipGetLastError();
    M.ke.release();
    M.re.release();
    M.srec.release();
    return false;
}

int launch_asm_struct(Mesh& M, const AsmParams& P, int nG, const double* rule, int tDof, const double* Ag,
                      const double* Dg, double* val, double* R, int kern, hipStream_t s)
{
    if (nG != 4 && nG != 15) {
        set_error("STRUCT: nG %d not supported", nG);
        return SVFSI_ERR_NOTSUP;
    }
    if (kern == SVFSI_STRUCT_AUTO) {
        // the outer-product kernels and their row gather, unless a row of Val
        // is too long for four of them in LDS, the coloured scatter is asked
        // for (SVFSI_ASM_GATHER=0) or the scratch cannot be had
        const char* v = getenv("SVFSI_ASM_GATHER");
        const size_t lds = (size_t)M.maxRow * 9 * 4 * sizeof(double);
        if (lds <= ((size_t)64 << 10) && !(v && v[0] == '0') && struct_scratch(M, nG)) {
            double* ke = M.ke.as<double>();
            double* re = M.re.as<double>();
            constexpr int E4 = 5, E15 = 5;
            if (nG == 4) {
                const size_t nPts = (size_t)M.nEl * nG;
                double* rec = M.srec.as<double>();
                hipLaunchKernelGGL(k_struct_rec, dim3((unsigned)((nPts + 255) / 256)), dim3(256), 0, s, M.nEl, nG,
                                   M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Dg, P, rule, rec);
                hipLaunchKernelGGL((k_struct_elem<4, E4, 256, true>), dim3((unsigned)((M.nEl + E4 - 1) / E4)),
                                   dim3(256), 0, s, M.nEl, M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Dg, P, rule,
                                   (const double*)rec, ke, re);
            } else {
                hipLaunchKernelGGL((k_struct_elem<15, E15, 256, false>), dim3((unsigned)((M.nEl + E15 - 1) / E15)),
                                   dim3(256), 0, s, M.nEl, M.ien.as<int>(), M.x.as<double>(), tDof, Ag, Dg, P, rule,
                                   (const double*)nullptr, ke, re);
            }
            hipLaunchKernelGGL(k_struct_rows, dim3((unsigned)((M.nNo + 3) / 4)), dim3(256), lds, s, M.nNo, M.maxRow,
                               M.lhs->rowPtr.as<int>(), M.rPtr.as<int>(), M.rSrc.as<int>(), M.emap.as<int>(),
                               (const double*)ke, (const double*)re, val, R);
            SV_HIP(hipGetLastError());
            return SVFSI_OK;
        }
        kern = SVFSI_STRUCT_MFMA64;
    }
    if (kern != SVFSI_STRUCT_VALU && kern != SVFSI_STRUCT_MFMA64 && kern != SVFSI_STRUCT_MFMA32) {
        set_error("STRUCT: unknown kernel selector %d", kern);
        return SVFSI_ERR_ARG;
    }
    const int nC = (int)M.colorOff.size() - 1;
    if (kern != SVFSI_STRUCT_VALU) {
        const size_t nPts = (size_t)M.nEl * nG;
        SV_TRY(M.srec.ensure(nPts * SR_HBM * sizeof(double)));
        double* rec = M.srec.as<double>();
        const unsigned gp = (unsigned)((nPts + 255) / 256);
        {
            ProfScope ps(3, (double)nPts * SR_HBM * 8.0);
            if (nG == 4)
                SV_LAUNCH(ps, (k_struct_points<4>), dim3(gp), dim3(256), 0, s, M.nEl, M.ien.as<int>(),
                          M.x.as<double>(), tDof, Ag, Dg, P, rule, rec);
            else
                SV_LAUNCH(ps, (k_struct_points<15>), dim3(gp), dim3(256), 0, s, M.nEl, M.ien.as<int>(),
                          M.x.as<double>(), tDof, Ag, Dg, P, rule, rec);
        }
        SV_HIP(hipGetLastError());
        constexpr int EPW4 = 4, EPW15 = 2;
        const bool gather = gather_enabled(M.eNoN);
        double* ke = nullptr;
        double* re = nullptr;
        if (gather) {
            SV_TRY(M.ke.ensure((size_t)M.nEl * 100 * 9 * sizeof(double)));
            SV_TRY(M.re.ensure((size_t)M.nEl * 10 * 3 * sizeof(double)));
            ke = M.ke.as<double>();
            re = M.re.as<double>();
        }
        // gather: one launch over all elements; scatter: one per colour
        const int nL = gather ? 1 : nC;
        for (int c = 0; c < nL; ++c) {
            const int begin = gather ? 0 : M.colorOff[c];
            const int count = gather ? M.nEl : M.colorOff[c + 1] - begin;
            if (count == 0) continue;
            const int epw = nG == 4 ? EPW4 : EPW15;
            const dim3 grid((count + epw - 1) / epw);
            ProfScope ps(2, 2.0 * 30 * 30 * 6 * nG * (double)count);
#define SV_SMFMA(NGV, MT, EPWV)                                                                                     \
    SV_LAUNCH(ps, (k_asm_struct_mfma<NGV, MT, EPWV>), grid, dim3(256), 0, s, begin, count, M.ien.as<int>(),   \
              M.emap.as<int>(), P, rule, rec, val, R, ke, re, M.gSlot.as<int>(), M.rSlot.as<int>())
            if (nG == 4) {
                if (kern == SVFSI_STRUCT_MFMA64) SV_SMFMA(4, double, EPW4);
                else SV_SMFMA(4, float, EPW4);
            } else {
                if (kern == SVFSI_STRUCT_MFMA64) SV_SMFMA(15, double, EPW15);
                else SV_SMFMA(15, float, EPW15);
            }
#undef SV_SMFMA
        }
        SV_HIP(hipGetLastError());
        return gather ? launch_gather(M, 3, val, R, s) : SVFSI_OK;
    }
    for (int c = 0; c < nC; ++c) {
        const int begin = M.colorOff[c], count = M.colorOff[c + 1] - begin;
        if (count == 0) continue;
        ProfScope ps(2, 2.0 * 30 * 30 * 6 * nG * (double)count);
        if (nG == 4) {
            constexpr int EPW = 8;
            SV_LAUNCH(ps, (k_asm_struct<4, EPW>), dim3((count + EPW - 1) / EPW), dim3(256), 0, s, begin, count,
                      M.ien.as<int>(), M.emap.as<int>(), M.x.as<double>(), tDof, Ag, Dg, P, rule, val, R);
        } else {
            constexpr int EPW = 2;
            SV_LAUNCH(ps, (k_asm_struct<15, EPW>), dim3((count + EPW - 1) / EPW), dim3(256), 0, s, begin, count,
                      M.ien.as<int>(), M.emap.as<int>(), M.x.as<double>(), tDof, Ag, Dg, P, rule, val, R);
        }
    }
    SV_HIP(hipGetLastError());
    return SVFSI_OK;
}

} // namespace svfsi
