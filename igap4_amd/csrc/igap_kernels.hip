// igap_kernels.hip -- CDNA4 (gfx950) kernels of the IGA residual/tangent assembly.
//
//   k_residual_gen, k_residual_sep, k_residual_sep_t  per-element residual vectors R_e[81]
//                     (volume loop of Residual_iga, src/assmcore_iga.c:118-259)
//   k_residual_gather deterministic per-dof sum of R_e + Neumann load +
//                     Dirichlet rows R_d = U_d - g_d (:258, :273-497)
//   k_tangent_sep, k_tangent_sep_t, k_tangent_gen, k_tangent_elem
//                     per-element tangents K_e[81x81] (volume loop of Tangent_iga,
//                     :607-764): separable patches, static and transient; equal weights
//                     and any geometry, static; everything else, on the matrix cores
//   k_tangent_gather_rows  deterministic per-nonzero sum of K_e into the CSR values
//                     with MatZeroRowsColumns(diag=1) fused (:763, :844)
//   k_csr_cols        column indices of the CSR pattern
//
// Element numbering e = (ex*ny + ey)*nz + ez (the reference's x->y->z loop
// order); local basis b = 9*bx + 3*by + bz; local dof 3*b + i.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <stdint.h>

#include "igap_device.h"
#include "igap_sep_pipeline.h"

namespace igap {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// ============================================================================
// Element e's Gauss-point fields for the density integral
// (256 threads): the control points and 1-D tables to LDS, then by sum
// factorisation the physical u-jets of every history level
// (sJet[q][h][k][a], par_periodic added) and the weight, G^-1, d2x/dxi2
// and W jets (sGeo[q][38]).  Ends with a block barrier.
// z and y passes of the Gauss-point field sum factorisation:
//   sA[f][bx*3+by][qz][dz] = sum_bz c_f(b) tz[qz][dz][bz]
//   sB[f][bx][qy][qz][s6]  = sum_by sA[f][bx*3+by][qz][dz(s6)] ty[qy][dy(s6)][by]
// with c = w, w X, w U (per field f) and the y-z jet slots s6 = (00, 10, 01,
// 20, 11, 02) in (dy, dz).  One thread per (f, bx*3+by) for z and per (f, bx,
// qz) for y: the inputs of a thread are loaded once and all its outputs
// (12 and 24) follow, with the reference's summation order per output.
// The NF fields are F0 .. F0 + NF - 1 of that list, stored from field 0 on.
template <int NF, int STR, int F0 = 0>
__device__ __forceinline__ void sf_zy(const double (*sT)[4][3][3], const double *sCP, double *sA, double *sB)
{
    static_assert(NF * 12 <= 256, "one thread per (field, bx, qz) in a 256-thread workgroup");
    const int tid = threadIdx.x;
    if (tid < NF * 9) {
        const int f = tid / 9, bxy = tid - 9 * f, fg = F0 + f;
        double cf[3];
#pragma unroll
        for (int bz = 0; bz < 3; bz++) {
            const double *c = sCP + STR * (3 * bxy + bz);
            cf[bz] = (fg == 0) ? c[3] : c[3] * ((fg < 4) ? c[fg - 1] : c[fg]);
        }
        double *o = sA + 108 * f + 12 * bxy;
#pragma unroll
        for (int qz = 0; qz < 4; qz++)
#pragma unroll
            for (int dz = 0; dz < 3; dz++) {
                const double *tz = &sT[2][qz][dz][0];
                double acc = 0.0;
#pragma unroll
                for (int bz = 0; bz < 3; bz++) acc += cf[bz] * tz[bz];
                o[3 * qz + dz] = acc;
            }
    }
    __syncthreads();
    if (tid < NF * 12) {
        const int f = tid / 12, r = tid - 12 * f, bx = r >> 2, qz = r & 3;
        const double *a = sA + 108 * f + 36 * bx + 3 * qz;   // a[12 by + dz]
        double av[3][3];
#pragma unroll
        for (int by = 0; by < 3; by++)
#pragma unroll
            for (int dz = 0; dz < 3; dz++) av[by][dz] = a[12 * by + dz];
        double *o = sB + 288 * f + 96 * bx + 6 * qz;         // o[24 qy + s6]
#pragma unroll
        for (int qy = 0; qy < 4; qy++)
#pragma unroll
            for (int s6 = 0; s6 < 6; s6++) {
                const int dy = (s6 == 1 || s6 == 4) ? 1 : (s6 == 3 ? 2 : 0);
                const int dz = (s6 == 2 || s6 == 4) ? 1 : (s6 == 5 ? 2 : 0);
                const double *ty = &sT[1][qy][dy][0];
                o[24 * qy + s6] = av[0][dz] * ty[0] + av[1][dz] * ty[1] + av[2][dz] * ty[2];
            }
    }
    __syncthreads();
}

// fields per sum-factorisation pass of gp_fields: static all 7 at once;
// transient the 9 history fields after the 4 geometry fields
template <int NH>
constexpr int gp_fields_per_pass() { return NH == 1 ? 4 + 3 * NH : 3 * NH; }

template <int NH>
__device__ __forceinline__ void gp_fields(const MeshK &M, const double *__restrict__ Uh, int64_t ndof, int e,
                                          double (*sT)[4][3][3], double *sCP, double *sWork, double *sJet, double *sGeo)
{
    constexpr int STR = 4 + 3 * NH;
    constexpr int NF = 4 + 3 * NH;
    constexpr int NFP = gp_fields_per_pass<NH>();
    constexpr int GEO_R = 38;
    const int tid = threadIdx.x;
    const int nz = M.nelem[2], ny = M.nelem[1];
    const int ex = e / (ny * nz), ey = (e / nz) % ny, ez = e % nz;
    const int ed[3] = {ex, ey, ez};
    if (tid < 27) {
        int bx = tid / 9, by = (tid / 3) % 3, bz = tid % 3;
        int ax = ex + bx, ay = ey + by, az = ez + bz;
        int64_t id = ((int64_t)M.na[1] * M.na[2]) * ax + (int64_t)M.na[2] * ay + az;
        sCP[STR * tid + 0] = M.X[3 * id + 0];
        sCP[STR * tid + 1] = M.X[3 * id + 1];
        sCP[STR * tid + 2] = M.X[3 * id + 2];
        sCP[STR * tid + 3] = M.w[id];
        int64_t oc = ((int64_t)M.nb[1] * M.nb[2]) * own1(ax, M.nb[0], M.periodic[0])
                   + (int64_t)M.nb[2] * own1(ay, M.nb[1], M.periodic[1]) + own1(az, M.nb[2], M.periodic[2]);
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int k = 0; k < 3; k++) sCP[STR * tid + 4 + 3 * h + k] = Uh[h * ndof + 3 * oc + k];
    } else if (tid >= 64 && tid < 64 + 12) {
        int d = (tid - 64) / 4, q = (tid - 64) % 4;
        const double *kV = M.knot[d] + ed[d];
        double c = M.gq[q];
        double x = (-c + 1.0) * kV[2] + c * kV[3];
        bspline1d(kV, x, sT[d][q][0], sT[d][q][1], sT[d][q][2]);
    }
    __syncthreads();

    // fields at the Gauss points (z, then y, then x).  Transient: two passes,
    // geometry (w, w X) then the history levels (w U), so that the buffers
    // hold 9 fields instead of 13
    {
        double *sA = sWork, *sB = sWork + NFP * 108;
        sf_zy<(NH == 1 ? NF : 4), STR>(sT, sCP, sA, sB);

        const int q = tid >> 2, part = tid & 3, lq = (tid & 63) & ~3;
        const int qd[3] = {q >> 4, (q >> 2) & 3, q & 3};
        const double *tx = &sT[0][qd[0]][0][0];
        const int boff = (4 * qd[1] + qd[2]) * 6;
        double W[10], Jg[3][10];
        sf_jet(sB + boff, tx, W);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int f = (part == 0) ? 1 + j : 4 + 3 * j + part - 1;
            if (part == 0 || (NH == 1 && j < NH)) {
                double Pj[10];
                sf_jet(sB + 288 * f + boff, tx, Pj);
                nurbs_param(Pj, 1.0, W, Jg[j]);
            } else {
#pragma unroll
                for (int a = 0; a < 10; a++) Jg[j][a] = (a >= 1 && a <= 3 && a - 1 == j) ? 1.0 : 0.0;
            }
        }
        double G[9], Gi[9], X2[18];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) G[3 * i + j] = Jg[i][1 + j];
        const double detG = inv3(G, Gi);
#pragma unroll
        for (int i = 0; i < 9; i++) Gi[i] = __shfl(Gi[i], lq, 64);
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int s2 = 0; s2 < 6; s2++) X2[6 * d + s2] = __shfl(Jg[d][4 + s2], lq, 64);
        if (NH != 1) {
            __syncthreads();
            sf_zy<3 * NH, STR, 4>(sT, sCP, sA, sB);
            if (part > 0) {
#pragma unroll
                for (int h = 0; h < NH; h++) {
                    double Pj[10];
                    sf_jet(sB + 288 * (3 * h + part - 1) + boff, tx, Pj);
                    nurbs_param(Pj, 1.0, W, Jg[h]);
                }
            }
        }
        if (part > 0) {
            const int k = part - 1;
            double xq[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double *kV = M.knot[d] + ed[d];
                const double c = M.gq[qd[d]];
                xq[d] = (-c + 1.0) * kV[2] + c * kV[3];
            }
#pragma unroll
            for (int h = 0; h < NH; h++) {
                phys_jet(Jg[h], Gi, X2);
                add_periodic1(M, xq, k, Jg[h]);
#pragma unroll
                for (int a = 0; a < 10; a++) sJet[q * 30 * NH + 30 * h + 10 * k + a] = Jg[h][a];
            }
        }
        // sGeo may share memory with the field buffers read above
        __syncthreads();
        if (part == 0) {
            double *g = sGeo + q * GEO_R;
            double dX[3];
#pragma unroll
            for (int d = 0; d < 3; d++) dX[d] = M.knot[d][ed[d] + 3] - M.knot[d][ed[d] + 2];
            g[0] = M.gw[qd[0]] * M.gw[qd[1]] * M.gw[qd[2]] * dX[0] * dX[1] * dX[2] * detG;
#pragma unroll
            for (int i = 0; i < 9; i++) g[1 + i] = Gi[i];
#pragma unroll
            for (int i = 0; i < 18; i++) g[10 + i] = X2[i];
#pragma unroll
            for (int i = 0; i < 10; i++) g[28 + i] = W[i];
        }
    }
    __syncthreads();
}

// ============================================================================
// density integral (iga_intdensity volume part, src/postcore_iga.c:84-234):
// per element sum_q w_q hh(u_q) -> Hd[e][ND]; lane = Gauss point, butterfly
// sums over the 64 lanes
// ============================================================================
template <int NH>
__global__ __launch_bounds__(256, (NH == 1 ? 1 : 2)) void k_density_elem(MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof,
                                                      double *__restrict__ Hd, int nel)
{
    constexpr int STR = 4 + 3 * NH;
    constexpr int GEO_R = 38;
    constexpr int ND = (NH == 1) ? ND_STATIC : ND_TRANSIENT;
    __shared__ double sT[3][4][3][3];
    __shared__ double sCP[27 * STR];
    constexpr int WA = gp_fields_per_pass<NH>() * (108 + 288), WG = 64 * GEO_R;
    __shared__ double sWork[WA > WG ? WA : WG];   // stage A, then sGeo
    __shared__ double sJet[64 * 30 * NH];
    double *sGeo = sWork;
    const int e = blockIdx.x;
    gp_fields<NH>(M, Uh, ndof, e, sT, sCP, sWork, sJet, sGeo);
    if (threadIdx.x < 64) {
        const int q = threadIdx.x;
        double hh[ND];
        if (NH == 1) phys_density_static(sJet + q * 30, P, hh);
        else phys_density_transient(sJet + q * 90, P, hh);
        const double w = sGeo[q * GEO_R];
#pragma unroll
        for (int i = 0; i < ND; i++) {
            double v = w * hh[i];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            if (q == 0) Hd[(int64_t)e * ND + i] = v;
        }
    }
}

// H[i] = sum over elements of Hd[e][i], in a fixed order (one block per density)
__global__ __launch_bounds__(256) void k_density_reduce(int nel, int nd, const double *__restrict__ Hd, double *__restrict__ H)
{
    __shared__ double red[256];
    const int i = blockIdx.x;
    double s = 0.0;
    for (int e = threadIdx.x; e < nel; e += 256) s += Hd[(int64_t)e * nd + i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) H[i] = red[0];
}

// The elements of owned control point a along one direction, ascending (the
// reference accumulates in element order): element e[j] with a its local
// point l[j], where ok[j].  A periodic direction has at least five elements.
struct ElemRow {
    int e[3], l[3];
    bool ok[3];
    __device__ __forceinline__ ElemRow(int a, int nelem, int periodic)
    {
#pragma unroll
        for (int j = 0; j < 3; j++) {
            // wrapped elements come last: locals 0, 2, 1 at a = 0 and 1, 0, 2 at a = 1
            const int lp = a == 0 ? (j == 0 ? 0 : 3 - j) : a == 1 ? (j == 2 ? 2 : 1 - j) : 2 - j;
            l[j] = periodic ? lp : 2 - j;
            e[j] = a - l[j];
            if (periodic && e[j] < 0) e[j] += nelem;
            ok[j] = e[j] >= 0 && e[j] < nelem;
        }
    }
};

// One thread per dof, its loads (27 at most) in flight together.  As one thread
// per control point looping over run-time index lists (in scratch memory) it took 14.6 us at
// 64x16x16, now 5.3.  Ucopy (may be null): where the iterate U is kept.
__global__ __launch_bounds__(256) void k_residual_gather(MeshK M, const double *__restrict__ Re, const double *U, double *Ucopy,
                                                         const double *__restrict__ Fneu, const int32_t *__restrict__ mask,
                                                         const double *__restrict__ g, double *R, int64_t ncp)
{
    const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= 3 * ncp) return;
    // control-point and dof indices fit in 32 bits (the CSR columns are int32)
    const int a = (int)((uint32_t)d / 3u), k = (int)d - 3 * a;
    const int nb1 = M.nb[1], nb2 = M.nb[2], az = a % nb2, axy = a / nb2, ay = axy % nb1, ax = axy / nb1;
    const ElemRow X(ax, M.nelem[0], M.periodic[0]), Y(ay, M.nelem[1], M.periodic[1]), Z(az, M.nelem[2], M.periodic[2]);
    const int m = mask[d];
    const double u = U[d], f = m ? g[d] : Fneu[d];
    double v[27];
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3; y++)
#pragma unroll
            for (int z = 0; z < 3; z++) {
                const bool ok = X.ok[x] && Y.ok[y] && Z.ok[z];
                const int64_t e = ((int64_t)X.e[x] * M.nelem[1] + Y.e[y]) * M.nelem[2] + Z.e[z];
                v[9 * x + 3 * y + z] = Re[ok ? e * 81 + 27 * X.l[x] + 9 * Y.l[y] + 3 * Z.l[z] + k : 0];
            }
    double s = 0.0;
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3; y++)
#pragma unroll
            for (int z = 0; z < 3; z++)
                if (X.ok[x] && Y.ok[y] && Z.ok[z]) s += v[9 * x + 3 * y + z];
    if (Ucopy) Ucopy[d] = u;
    R[d] = m ? u - f : s + f;
}

// ============================================================================
// tangent: one workgroup (4 waves) per element.
//   stage A  (once)      geometry and u-jets of the 64 Gauss points, 4 lanes
//                        per point splitting the 27 basis functions
//   stage B  (16 chunks of QC = 4 Gauss points)
//     B1  physical basis jets R_q[10][27] -> LDS
//     B2  pointwise tangent D_q = w_q C_q (30x30, the blocks i <= j) -> LDS
//     B3  K^{ij} += sum_{q,a} R_q[a][b] * (sum_b' D_q[(i,a),(j,b')] R_q[b'][c])
//         for the six blocks i <= j (K_e is symmetric; K^{ji} = K^{ij}^T is
//         written by mirroring) on V_MFMA_{F64,F32}_16X16X4: M = b, N = c
//         (27 -> 32), K = (q,a).  Wave w owns column tile w>>1 and blocks
//         3(w&1)..3(w&1)+2 for both row tiles, so each B operand it forms on
//         the VALU from D and R feeds two matrix-core products.  For the
//         static physics the value slot a = 0 of D is zero and is skipped.
// ============================================================================
constexpr int QC = 4;
constexpr int GEO = 38;   // per Gauss point: wgt, Gi[9], X2[18], W[10]
// Operands of the 16x16x4 products: lane l supplies A[l&15][l>>4] and
// B[l>>4][l&15].  Result register r of lane l holds D[row(l>>4, r)][l&15];
// the row map of each instruction is pinned by igap_gpu_selftest_mfma.
template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef double4_t acc_t;
    static __device__ __forceinline__ acc_t run(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kr, int r) { return 4 * r + kr; }
};
template <> struct Mfma<float> {
    typedef float4_t acc_t;
    static __device__ __forceinline__ acc_t run(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kr, int r) { return 4 * kr + r; }
};

__constant__ const int kBlkI[6] = {0, 0, 0, 1, 1, 2};
__constant__ const int kBlkJ[6] = {0, 1, 2, 1, 2, 2};


// Stage A of the element tangent (256 threads): the Gauss-point fields by
// sum factorisation from the control points in sCP and the 1-D tables in sT.
// Static physics: the strain-measure state of all 64 points -> sSt[q][STW];
// transient: the physical u-jets of Um and Ud -> sJet[q][h][k][a].  Per point
// sGeo[q][GEOK] = wgt (= Gauss weight x span lengths x det G), then, when
// GEOK allows, G^-1 (9), d2x/dxi2 (18) and the weight jet W (10).  sWork
// holds the field buffers.  Ends with a block barrier.
template <int NH, int GEOK>
__device__ __forceinline__ void tangent_fields(const MeshK &M, const PhysK &P, const int *ed, double (*sT)[4][3][3],
                                               const double *sCP, double *sWork, double *sGeo, double *sJet, double *sSt)
{
    constexpr int NL = (NH == 1) ? 1 : 2;
    constexpr int STR = 4 + 3 * NL;
    constexpr int NF = 4 + 3 * NL;             // fields w, w X (3), w U (3 per held level)
    constexpr int NFP = (NH == 1) ? NF : 6;    // fields per sum-factorisation pass
    const int tid = threadIdx.x;
    // ---- stage A: fields at the 64 Gauss points by sum factorisation.
    //      The fields P_f = sum_b c_{b,f} N_b with c = w, w X (3), w U (3 per
    //      level) are contracted one direction at a time (z, then y, then x:
    //      27 -> 108 -> 288 -> 640 values per field); the rational jets follow
    //      by the quotient rule on P_f / W and the physical jets by the chain
    //      rule, both linear in the basis, so the result is the reference's
    //      sum over b of c_b R_b in another order of summation.
    {
        double *sA = sWork, *sB = sA + NFP * 108;
        sf_zy<(NH == 1 ? NF : 4), STR>(sT, sCP, sA, sB);

        const int q = tid >> 2, part = tid & 3, lq = (tid & 63) & ~3;
        const int qd[3] = {q >> 4, (q >> 2) & 3, q & 3};
        const double *tx = &sT[0][qd[0]][0][0];
        const int boff = (4 * qd[1] + qd[2]) * 6;
        double W[10], Jg[3][10];
        sf_jet(sB + boff, tx, W);
        // part 0: the three geometry fields; part 1 + k: displacement
        // component k of every held level (transient: second pass below)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int f = (part == 0) ? 1 + j : 4 + 3 * j + part - 1;
            if (part == 0 || (NH == 1 && j < NL)) {
                double Pj[10];
                sf_jet(sB + 288 * f + boff, tx, Pj);
                nurbs_param(Pj, 1.0, W, Jg[j]);
            } else {
#pragma unroll
                for (int a = 0; a < 10; a++) Jg[j][a] = (a >= 1 && a <= 3 && a - 1 == j) ? 1.0 : 0.0;
            }
        }
        double G[9], Gi[9], X2[18];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) G[3 * i + j] = Jg[i][1 + j];
        const double detG = inv3(G, Gi);
#pragma unroll
        for (int i = 0; i < 9; i++) Gi[i] = __shfl(Gi[i], lq, 64);
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int s2 = 0; s2 < 6; s2++) X2[6 * d + s2] = __shfl(Jg[d][4 + s2], lq, 64);
        double xq[3], dX[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double *kV = M.knot[d] + ed[d];
            const double c = M.gq[qd[d]];
            xq[d] = (-c + 1.0) * kV[2] + c * kV[3];
            dX[d] = kV[3] - kV[2];
        }
        if (NH != 1) {
            // second pass: the fields w Um (3) and w Ud (3)
            __syncthreads();
            sf_zy<6, STR, 4>(sT, sCP, sA, sB);
            if (part > 0) {
#pragma unroll
                for (int h = 0; h < NL; h++) {
                    double Pj[10];
                    sf_jet(sB + 288 * (3 * h + part - 1) + boff, tx, Pj);
                    nurbs_param(Pj, 1.0, W, Jg[h]);
                }
            }
        }
        if (part > 0) {
            const int k = part - 1;
#pragma unroll
            for (int h = 0; h < NL; h++) {
                phys_jet(Jg[h], Gi, X2);
                // the periodic macro-field shifts every level alike: Um takes
                // it, the difference Ud does not
                if (h == 0) add_periodic1(M, xq, k, Jg[h]);
                if (NH != 1) {
#pragma unroll
                    for (int a = 0; a < 10; a++) sJet[q * 30 * NL + 30 * h + 10 * k + a] = Jg[h][a];
                }
            }
        }
        if (NH == 1) {
            double u[30];
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int a = 0; a < 10; a++) u[10 * k + a] = __shfl(Jg[0][a], lq + 1 + k, 64);
            if (part == 0) {
                State st;
                phys_state(u, P, st);
                double *sp = sSt + q * STW;
#pragma unroll
                for (int i = 0; i < 9; i++) sp[ST_F + i] = st.F[i];
#pragma unroll
                for (int i = 0; i < 27; i++) sp[ST_H + i] = st.H[i];
#pragma unroll
                for (int i = 0; i < 9; i++) { sp[ST_S + i] = st.S[i]; sp[ST_G + i] = st.G[i]; sp[ST_N + i] = st.N[i]; }
            }
        }
        if (part == 0) {
            double *g = sGeo + q * GEOK;
            g[0] = M.gw[qd[0]] * M.gw[qd[1]] * M.gw[qd[2]] * dX[0] * dX[1] * dX[2] * detG;
            if (GEOK > 1) {
#pragma unroll
                for (int i = 0; i < 9; i++) g[1 + i] = Gi[i];
#pragma unroll
                for (int i = 0; i < 18; i++) g[10 + i] = X2[i];
            }
            if (GEOK > 28) {
#pragma unroll
                for (int i = 0; i < 10; i++) g[28 + i] = W[i];
            }
        }
    }
    __syncthreads();
}

// Where k_tangent_elem<..., DIRECT = true> adds its element matrix: the
// elements of one of the 27 colours (ex, ey, ez) = (cx, cy, cz) + 3 (i, j, k)
// of a non-periodic patch -- no two of them share a control point, so none
// share a CSR row -- straight into the CSR values, skipping the entries of
// Dirichlet rows and columns (MatZeroRowsColumns, whose unit diagonal
// k_dirichlet_diag writes afterwards).
struct Scatter {
    const int64_t *rowptr;
    const int32_t *mask;
    int c[3];    // colour
    int nc[3];   // elements of the colour per direction
};

// CSR position of column 3C + j in the row of control point B that starts at
// row_start, for control points B, C within +-2 of each other on a
// non-periodic patch: the column block's slot in the row's sorted stencil
__device__ __forceinline__ int64_t stencil_pos(const MeshK &M, int64_t row_start, int Bx, int By, int Bz, int Cx, int Cy, int Cz,
                                               int j)
{
    const int lx = Bx - 2 < 0 ? 0 : Bx - 2, ly = By - 2 < 0 ? 0 : By - 2, lz = Bz - 2 < 0 ? 0 : Bz - 2;
    const int hy = By + 2 > M.nb[1] - 1 ? M.nb[1] - 1 : By + 2, hz = Bz + 2 > M.nb[2] - 1 ? M.nb[2] - 1 : Bz + 2;
    const int nsy = hy - ly + 1, nsz = hz - lz + 1;
    return row_start + 3 * (((Cx - lx) * nsy + (Cy - ly)) * nsz + (Cz - lz)) + j;
}

// the same position for row 3B + i looked up in rowptr
__device__ __forceinline__ int64_t csr_pos(const MeshK &M, const int64_t *__restrict__ rowptr, int Bx, int By, int Bz, int i,
                                           int Cx, int Cy, int Cz, int j)
{
    const int64_t row = 3 * (((int64_t)M.nb[1] * M.nb[2]) * Bx + (int64_t)M.nb[2] * By + Bz) + i;
    return stencil_pos(M, rowptr[row], Bx, By, Bz, Cx, Cy, Cz, j);
}

template <typename T, int NH, bool DIRECT>
__global__ __launch_bounds__(256, 2) void k_tangent_elem(MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof,
                                                         T *__restrict__ Ke, int nel, Scatter S)
{
    // field levels held per control point: static U; transient the two
    // combinations the rule evaluates, Um = (U^1 + U^0)/2 and Ud = (U - U^0)/2
    // (rule node j: Um + s_j Ud)
    constexpr int NL = (NH == 1) ? 1 : 2;
    constexpr int STR = 4 + 3 * NL;
    constexpr int NNODE = (NH == 1) ? 1 : 8;
    constexpr int A0 = (NH == 1) ? 1 : 0;     // first jet slot in the contraction
    constexpr int NA = 10 - A0;               // jet slots per Gauss point in K
    // rows of D are padded to whole 16-byte LDS vectors so that B3 reads them
    // with 128-bit loads at compile-time offsets
    constexpr int VN = 16 / (int)sizeof(T);
    constexpr int RS = (NA + VN - 1) / VN * VN;   // row stride of D
    constexpr int NN = NA * RS;                   // stride of one (i,j) block of D
    static_assert(QC == 4, "the MFMA k-row is the Gauss point of a 4-point chunk");
    // static: the strain-measure state of all 64 Gauss points is built once in
    // stage A; transient: the u-jets of Um and Ud are kept and the eight
    // rule-node states are built per chunk.  Two workgroups share a CU, so
    // the transient keeps its LDS under 80 KB: the field sum factorisation
    // runs in two passes (geometry, then Um/Ud) and the weight jet W is
    // rebuilt per chunk from the basis instead of being stored.
    constexpr int SST = (NH == 1) ? 64 * STW : QC * MW;   // static: states; transient: moment states
    constexpr int GEOK = (NH == 1) ? GEO : GEO - 10;     // per Gauss point: wgt, Gi[9], X2[18] (+ W[10] static)
    __shared__ double sT[3][4][3][3];          // 1-D tables [d][q_d][order][i]
    __shared__ double sCP[27 * STR];
    __shared__ double sGeo[64 * GEOK];
    __shared__ double sJet[(NH == 1) ? 1 : 64 * 30 * NL];
    __shared__ double sSt[SST];
    // stage A's sum-factorisation buffers share memory with stage B's R and D
    constexpr int NF = 4 + 3 * NL;             // fields w, w X (3), w U (3 per held level)
    constexpr int NFP = (NH == 1) ? NF : 6;    // fields per sum-factorisation pass
    constexpr int WORK_A = NFP * (108 + 288) * (int)sizeof(double);
    constexpr int WORK_B = QC * (10 * 32 + 6 * NN) * (int)sizeof(T);
    __shared__ __attribute__((aligned(16))) char sWork[WORK_A > WORK_B ? WORK_A : WORK_B];
    T(*sR)[10][32] = reinterpret_cast<T(*)[10][32]>(sWork);
    T(*sD)[6 * NN] = reinterpret_cast<T(*)[6 * NN]>(sWork + QC * 10 * 32 * sizeof(T));   // blocks i <= j, slots A0..9

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int e = blockIdx.x;
    int ex, ey, ez;
    if (DIRECT) {
        // element (i, j, k) of the colour's lattice
        const int k = e % S.nc[2], j = (e / S.nc[2]) % S.nc[1], i = e / (S.nc[1] * S.nc[2]);
        ex = S.c[0] + 3 * i;
        ey = S.c[1] + 3 * j;
        ez = S.c[2] + 3 * k;
    } else {
        const int nz = M.nelem[2], ny = M.nelem[1];
        ex = e / (ny * nz);
        ey = (e / nz) % ny;
        ez = e % nz;
    }
    const int ed[3] = {ex, ey, ez};

    // ---- element data, 1-D tables
    if (tid < 27) {
        int bx = tid / 9, by = (tid / 3) % 3, bz = tid % 3;
        int ax = ex + bx, ay = ey + by, az = ez + bz;
        int64_t id = ((int64_t)M.na[1] * M.na[2]) * ax + (int64_t)M.na[2] * ay + az;
        sCP[STR * tid + 0] = M.X[3 * id + 0];
        sCP[STR * tid + 1] = M.X[3 * id + 1];
        sCP[STR * tid + 2] = M.X[3 * id + 2];
        sCP[STR * tid + 3] = M.w[id];
        int64_t oc = ((int64_t)M.nb[1] * M.nb[2]) * own1(ax, M.nb[0], M.periodic[0])
                   + (int64_t)M.nb[2] * own1(ay, M.nb[1], M.periodic[1]) + own1(az, M.nb[2], M.periodic[2]);
        if (NH == 1) {
#pragma unroll
            for (int k = 0; k < 3; k++) sCP[STR * tid + 4 + k] = Uh[3 * oc + k];
        } else {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double u0 = Uh[3 * oc + k], u1 = Uh[ndof + 3 * oc + k], u2 = Uh[2 * ndof + 3 * oc + k];
                sCP[STR * tid + 4 + k] = 0.5 * (u1 + u2);
                sCP[STR * tid + 7 + k] = 0.5 * (u0 - u2);
            }
        }
    } else if (tid >= 64 && tid < 64 + 12) {
        int d = (tid - 64) / 4, q = (tid - 64) % 4;
        const double *kV = M.knot[d] + ed[d];
        double c = M.gq[q];
        double x = (-c + 1.0) * kV[2] + c * kV[3];
        bspline1d(kV, x, sT[d][q][0], sT[d][q][1], sT[d][q][2]);
    }
    __syncthreads();

    tangent_fields<NH, GEOK>(M, P, ed, sT, sCP, reinterpret_cast<double *>(sWork), sGeo, sJet, sSt);

    typedef typename Mfma<T>::acc_t acc_t;
    acc_t acc[3][2];
#pragma unroll
    for (int t = 0; t < 3; t++) { acc[t][0] = (acc_t){0, 0, 0, 0}; acc[t][1] = (acc_t){0, 0, 0, 0}; }
    const int ctile = wv >> 1, blk0 = 3 * (wv & 1), m = lane & 15, kr = lane >> 4;
    int bi[3], bj[3];
#pragma unroll
    for (int t = 0; t < 3; t++) { bi[t] = kBlkI[blk0 + t]; bj[t] = kBlkJ[blk0 + t]; }

    Mom mu = {0.0, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0};
    if (NH != 1) {
#pragma unroll
        for (int j = 0; j < NNODE; j++) {
            mu.m0 += P.ct[j];
            mu.m1 += P.ct[j] * P.s[j];
            mu.m2 += P.ct[j] * P.s[j] * P.s[j];
        }
        mu.factor();
    }
    T Rn[10];   // static: basis jets of the next chunk's point, built by lanes 32..58 on even chunks
    for (int chunk = 0; chunk < 64 / QC; chunk++) {
        const int q0 = chunk * QC;
        // ---- B1 (transient: + the rule-node states): wave wv builds the basis
        //      jets of Gauss point q0 + wv.  Static: lanes 32..58 are otherwise
        //      idle here, so on even chunks they build the jets of point
        //      q0 + 4 + wv (the next chunk's) and store them on the odd chunk:
        //      one B1 pass per two chunks.
        if (NH == 1) {
            const int ql = wv;
            if ((chunk & 1) == 0) {
                const int hi = lane >> 5, b = lane & 31, q = q0 + ql + 4 * hi;
                if (b < 27) {
                    const int qd[3] = {q >> 4, (q >> 2) & 3, q & 3};
                    const double *t0 = &sT[0][qd[0]][0][0], *t1 = &sT[1][qd[1]][0][0], *t2 = &sT[2][qd[2]][0][0];
                    const double *g = sGeo + q * GEOK;
                    double N[10], R[10];
                    tensor_jet(t0, t1, t2, b, N);
                    nurbs_param(N, sCP[STR * b + 3], g + 28, R);
                    phys_jet(R, g + 1, g + 10);
                    if (hi == 0) {
#pragma unroll
                        for (int a = 0; a < 10; a++) sR[ql][a][b] = (T)R[a];
                    } else {
#pragma unroll
                        for (int a = 0; a < 10; a++) Rn[a] = (T)R[a];
                    }
                } else if (hi == 0) {
#pragma unroll
                    for (int a = 0; a < 10; a++) sR[ql][a][b] = (T)0;
                }
            } else {
                const int b = lane - 32;
                if (b >= 0 && b < 27) {
#pragma unroll
                    for (int a = 0; a < 10; a++) sR[ql][a][b] = Rn[a];
                } else if (lane >= 27 && lane < 32) {
#pragma unroll
                    for (int a = 0; a < 10; a++) sR[ql][a][lane] = (T)0;
                }
            }
        } else {
            const int ql = wv, q = q0 + ql, b = lane;
            if (b < 32) {
                // basis jets; the weight jet W = sum_b w_b N_b is summed over
                // lanes 0..31 (27..31 add zero)
                const int qd[3] = {q >> 4, (q >> 2) & 3, q & 3};
                const double *t0 = &sT[0][qd[0]][0][0], *t1 = &sT[1][qd[1]][0][0], *t2 = &sT[2][qd[2]][0][0];
                const double *g = sGeo + q * GEOK;
                double N[10], W[10], R[10];
                const double wb = (b < 27) ? sCP[STR * b + 3] : 0.0;
                if (b < 27) {
                    tensor_jet(t0, t1, t2, b, N);
                } else {
#pragma unroll
                    for (int a = 0; a < 10; a++) N[a] = 0.0;
                }
#pragma unroll
                for (int a = 0; a < 10; a++) W[a] = wb * N[a];
#pragma unroll
                for (int a = 0; a < 10; a++) {
                    W[a] = sum16(W[a]);
                    W[a] += __shfl_xor(W[a], 16, 64);
                }
                if (b < 27) {
                    nurbs_param(N, wb, W, R);
                    phys_jet(R, g + 1, g + 10);
#pragma unroll
                    for (int a = 0; a < 10; a++) sR[ql][a][b] = (T)R[a];
                } else {
#pragma unroll
                    for (int a = 0; a < 10; a++) sR[ql][a][b] = (T)0;
                }
            } else if (NH != 1 && b < 32 + NNODE) {
                // rule node j: S, G and N at us_j, weighted and summed over
                // the eight lanes 32..39 into the moment state
                const int j = b - 32;
                const double *u = sJet + q * 30 * NL;
                double us[30];
#pragma unroll
                for (int i = 0; i < 30; i++) us[i] = u[i] + P.s[j] * u[30 + i];
                State st;
                phys_state(us, P, st);
                const double w0 = P.ct[j], w1 = w0 * P.s[j], w2 = w1 * P.s[j];
                // node sums over lanes 32..39, one entry at a time (few live
                // registers); lane 32 stores Sb, Gb and the N sums as L^-1 Nm L^-T
                double *ms = sSt + ql * MW;
                const double c12 = 1.0 / (mu.a11 * mu.a22), c22 = 1.0 / mu.d2;
#pragma unroll
                for (int i = 0; i < 9; i++) {
                    double sv = w0 * st.S[i], gv = w0 * st.G[i];
                    double n0 = w0 * st.N[i], n1 = w1 * st.N[i], n2 = w2 * st.N[i];
                    sv = sum8(sv);
                    gv = sum8(gv);
                    n0 = sum8(n0);
                    n1 = sum8(n1);
                    n2 = sum8(n2);
                    if (j == 0) {
                        ms[MS + i] = sv;
                        ms[MG + i] = gv;
                        ms[MN11 + i] = n0 / mu.m0;
                        ms[MN12 + i] = (n1 - mu.lf * n0) * c12;
                        ms[MN22 + i] = ((mu.lf * n0 - n1) * mu.lf + (n2 - mu.lf * n1)) * c22;
                    }
                }
            } else if (NH != 1 && b >= 40) {
                // F^ and H^ (two components each) of the midpoint m0 = (u1+u0)/2
                // and the increment d = (u-u0)/2: X^_1 = a11 (X0 + lf Xd),
                // X^_2 = a22 Xd, for the 9 entries of F and the 27 of H
                const double *u = sJet + q * 30 * NL;
                double *ms = sSt + ql * MW;
                for (int i = b - 40; i < 36; i += 24) {
                    const bool isF = i < 9;
                    const int r = isF ? i : i - 9;
                    int slot;
                    if (isF) slot = 10 * (r / 3) + 1 + (r % 3);
                    else slot = 10 * (r / 9) + sidx((r % 9) / 3, r % 3);
                    double x0 = u[slot];
                    const double xd = u[30 + slot];
                    if (isF && (r / 3) == (r % 3)) x0 += 1.0;
                    const double x1 = mu.a11 * (x0 + mu.lf * xd), x2 = mu.a22 * xd;
                    if (isF) { ms[MF1 + r] = x1; ms[MF2 + r] = x2; }
                    else { ms[MH1 + r] = x1; ms[MH2 + r] = x2; }
                }
            }
        }
        if (NH != 1) __syncthreads();   // node states are read by the whole wave below
        // ---- B2: D_q = w_q C_q on the blocks i <= j for the chunk's points.
        //      Static: the chunk's 216 rows sorted by kind across the waves
        //      (tasks 0..71 first-gradient rows: point t / 18, block
        //      (t % 18) / 3, row t % 3 + 1; 72..215 second-gradient rows:
        //      point u / 36, block (u % 36) / 6, row u % 6 + 4, u = t - 72),
        //      so that three waves run one branch of the one-hot rows.
        //      Transient: likewise with the value rows first.
        if (NH == 1) {
            if (tid < 216) {
                int ql, p, ar;
                if (tid < 72) {
                    ql = tid / 18;
                    const int r = tid - 18 * ql;
                    p = r / 3;
                    ar = r - 3 * p;
                } else {
                    const int u = tid - 72;
                    ql = u / 36;
                    const int r = u - 36 * ql;
                    p = r / 6;
                    ar = 3 + r - 6 * p;
                }
                const int q = q0 + ql;
                const double wgt = sGeo[q * GEOK];
                double row[NA];
                c_row_onehot(sSt + q * STW, P, kBlkI[p], ar + A0, kBlkJ[p], row);
                T *D = sD[ql] + p * NN + ar * RS;
#pragma unroll
                for (int bb = 0; bb < NA; bb++) D[bb] = (T)(wgt * row[bb]);
            }
        } else if (tid < 240) {
            // the chunk's 240 rows sorted by kind: 0..23 value rows (the
            // inertia alone; point t / 6, block t % 6), 24..95 first-gradient
            // rows, 96..239 second-gradient rows
            int ql, p, ar;
            if (tid < 24) {
                ql = tid / 6;
                p = tid - 6 * ql;
                ar = 0;
            } else if (tid < 96) {
                const int u = tid - 24;
                ql = u / 18;
                const int r = u - 18 * ql;
                p = r / 3;
                ar = 1 + r - 3 * p;
            } else {
                const int u = tid - 96;
                ql = u / 36;
                const int r = u - 36 * ql;
                p = r / 6;
                ar = 4 + r - 6 * p;
            }
            const int q = q0 + ql, k = kBlkI[p], l = kBlkJ[p];
            const double wgt = sGeo[q * GEOK];
            double row[NA];
            row[0] = 0.0;   // value column: the inertia alone
            if (ar == 0) {
#pragma unroll
                for (int bb = 1; bb < NA; bb++) row[bb] = 0.0;
                if (k == l) row[0] = P.cii / (2. * P.dt) + P.rho / (P.dt * P.dt);
            } else {
                c_row_mom_onehot(sSt + ql * MW, P, k, ar, l, row + 1);
            }
            T *D = sD[ql] + p * NN + ar * RS;
#pragma unroll
            for (int bb = 0; bb < NA; bb++) D[bb] = (T)(wgt * row[bb]);
        }
        __syncthreads();
        // ---- B3: matrix-core contraction over (q, a) of this chunk.  The
        //      4-deep k-row of each MFMA is the chunk's Gauss point (kr) and
        //      the k-step is the jet slot, so every LDS address is a lane base
        //      plus a compile-time offset and the lane's basis column Rc is
        //      read once per chunk.
        {
            const T *Rq = &sR[kr][A0][0];
            const T *Dq = sD[kr] + blk0 * NN;
            T Rc[NA];
#pragma unroll
            for (int bb = 0; bb < NA; bb++) Rc[bb] = Rq[32 * bb + 16 * ctile + m];
#pragma unroll
            for (int a = 0; a < NA; a++) {
                const T Av0 = Rq[32 * a + m], Av1 = Rq[32 * a + 16 + m];
#pragma unroll
                for (int t = 0; t < 3; t++) {
                    typedef T vec_t __attribute__((ext_vector_type(VN)));
                    const vec_t *dv = reinterpret_cast<const vec_t *>(Dq + t * NN + a * RS);
                    T d[RS];
#pragma unroll
                    for (int v = 0; v < RS / VN; v++) {
                        const vec_t x = dv[v];
#pragma unroll
                        for (int c = 0; c < VN; c++) d[VN * v + c] = x[c];
                    }
                    T y = d[0] * Rc[0];
#pragma unroll
                    for (int bb = 1; bb < NA; bb++) y += d[bb] * Rc[bb];
                    acc[t][0] = Mfma<T>::run(Av0, y, acc[t][0]);
                    acc[t][1] = Mfma<T>::run(Av1, y, acc[t][1]);
                }
            }
        }
        __syncthreads();
    }

    const int c = 16 * ctile + m;
    if (DIRECT) {
        // ---- add (row 3b+i, column 3c+j) and the mirrored entry into the CSR
        //      values, Dirichlet rows and columns left at zero.  The elements
        //      of one colour share no row, so no other workgroup of the launch
        //      touches these entries.  The row starts and masks of the
        //      element's 81 rows are staged in LDS (the geometry buffer is
        //      free after the last chunk); then every load of the lane is
        //      issued before its first store, so the epilogue waits for one
        //      round trip.
        int64_t *sRow = reinterpret_cast<int64_t *>(sGeo);
        int32_t *sMsk = reinterpret_cast<int32_t *>(sGeo + 81);
        if (tid < 81) {
            const int b = tid / 3, i = tid - 3 * (tid / 3);
            const int64_t cp = ((int64_t)M.nb[1] * M.nb[2]) * (ex + b / 9) + (int64_t)M.nb[2] * (ey + (b / 3) % 3) + (ez + b % 3);
            sRow[tid] = S.rowptr[3 * cp + i];
            sMsk[tid] = S.mask[3 * cp + i];
        }
        __syncthreads();
        if (c < 27) {
            const int Cx = ex + c / 9, Cy = ey + (c / 3) % 3, Cz = ez + c % 3;
            T vp[3][8], vq[3][8];
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const int b = 16 * (k >> 2) + Mfma<T>::row(kr, k & 3);
                    vp[t][k] = vq[t][k] = (T)0;
                    if (b < 27 && sMsk[3 * c + bj[t]] == 0 && sMsk[3 * b + bi[t]] == 0) {
                        const int Bx = ex + b / 9, By = ey + (b / 3) % 3, Bz = ez + b % 3;
                        vp[t][k] = Ke[stencil_pos(M, sRow[3 * b + bi[t]], Bx, By, Bz, Cx, Cy, Cz, bj[t])];
                        if (bi[t] != bj[t]) vq[t][k] = Ke[stencil_pos(M, sRow[3 * c + bj[t]], Cx, Cy, Cz, Bx, By, Bz, bi[t])];
                    }
                }
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const int b = 16 * (k >> 2) + Mfma<T>::row(kr, k & 3);
                    if (b < 27 && sMsk[3 * c + bj[t]] == 0 && sMsk[3 * b + bi[t]] == 0) {
                        const int Bx = ex + b / 9, By = ey + (b / 3) % 3, Bz = ez + b % 3;
                        const T v = acc[t][k >> 2][k & 3];
                        Ke[stencil_pos(M, sRow[3 * b + bi[t]], Bx, By, Bz, Cx, Cy, Cz, bj[t])] = vp[t][k] + v;
                        if (bi[t] != bj[t])
                            Ke[stencil_pos(M, sRow[3 * c + bj[t]], Cx, Cy, Cz, Bx, By, Bz, bi[t])] = vq[t][k] + v;
                    }
                }
        }
        return;
    }
    // ---- write K_e (row 3b+i, column 3c+j) and the mirrored block (3c+j, 3b+i)
    T *out = Ke + (int64_t)e * 6561;
    if (c < 27) {
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int bt = 0; bt < 2; bt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int b = 16 * bt + Mfma<T>::row(kr, r);
                    if (b < 27) {
                        T v = acc[t][bt][r];
                        out[(3 * b + bi[t]) * 81 + 3 * c + bj[t]] = v;
                        if (bi[t] != bj[t]) out[(3 * c + bj[t]) * 81 + 3 * b + bi[t]] = v;
                    }
                }
    }
}

// ============================================================================
// Tangent on a separable patch (k_tangent_sep, static physics): every
// coordinate of the geometry depends on its own parametric direction only,
// x_d = f_d(xi_d), and all control weights are equal, as on the igabeam
// patches (mesh/igabeam.c).  Then G = diag(f_x', f_y', f_z'), the rational
// basis is the B-spline basis, and the physical jet of basis b at Gauss point
// q is a product of three 1-D tables of physical derivatives,
//   R_q[a][b] = Px[qx][dx(a)][bx] Py[qy][dy(a)][by] Pz[qz][dz(a)][bz],
//   P_d[q][0] = N,  P_d[q][1] = N' / g,  P_d[q][2] = (N'' - (g'/g) N') / g^2
// (g = f_d', g' = f_d'' at the point; the chain rule of src/assmcore_iga.c:
// 179-208 with a diagonal G).  The contraction of Tangent_iga
// (src/assmcore_iga.c:723-749),
//   K^ij[b][c] = sum_q sum_{a,a'} R_q[a][b] D_q[(i,a),(j,a')] R_q[a'][c],
// then factors direction by direction (sum factorisation), with s = (dx, dy)
// the x-y part of a jet slot:
//   E1[(s,bz),(s',cz)] = sum_qz sum_{dz,dz'} Pz[qz][dz][bz] D_q[(s,dz)][(s',dz')] Pz[qz][dz'][cz]  per (qx, qy) pencil
//   E2[(dx,by,bz),(dx',cy,cz)] += sum_{dy,dy'} Py[qy][dy][by] Py[qy][dy'][cy] E1[((dx,dy),bz),((dx',dy'),cz)]
//   K[(bx,by,bz),(cx,cy,cz)]   += sum_{dx,dx'} Px[qx][dx][bx] Px[qx][dx'][cx] E2   after the fourth qy
// ~0.7 MFLOP per element on the vector ALUs instead of the 27x27 product per
// point and jet slot.  The displacement jets come from the same tables by sum
// factorisation (no quotient or chain rule left to apply); the element matrix
// is written in k_tangent_elem's layout (row 3b+i, column 3c+j).
// ============================================================================
// The 1-D tables of a separable patch, one block per element of a direction
// (blockIdx.y = direction), lane q < 4 its 1-D Gauss point: the rational basis
// rho_i = N_i / S (S = sum_i N_i) and its derivatives made physical with
// g = dx_d/dxi_d and g' = d2x_d/dxi_d^2 from the element's three control
// coordinates along d (x_d depends on the index along d alone):
//   [q][0][i] = rho_i,  [q][1][i] = rho_i' / g,  [q][2][i] = (rho_i'' - (g'/g) rho_i') / g^2,
// then the point weight gw_q dX g.  Built once per context, as the knots and
// control points are: evaluating them in every element's workgroup is a chain of
// dependent loads and divisions (k_residual_sep at 128x32x32 0.99 -> 0.84 ms).
__global__ __launch_bounds__(64) void k_sep_tables(MeshK M, double *__restrict__ tab, float *__restrict__ tabf)
{
    const int d = blockIdx.y, e = blockIdx.x, q = threadIdx.x;
    if (e >= M.nelem[d] || q >= 4) return;
    const int first = (d > 0 ? M.nelem[0] : 0) + (d > 1 ? M.nelem[1] : 0);
    const double *kV = M.knot[d] + e;
    const double c = M.gq[q];
    const double x = (-c + 1.0) * kV[2] + c * kV[3];
    double t[9];
    bspline1d(kV, x, t, t + 3, t + 6);
    // the rational basis of equal weights is N_b / W with W = S_x S_y S_z,
    // S = sum_i N_i (1 up to the MTOL guard of the B-spline formulas):
    // a product of the 1-D quotients rho_i = N_i / S, whose derivatives
    // follow from the 1-D quotient rule
    const double S0 = t[0] + t[1] + t[2], S1 = t[3] + t[4] + t[5], S2 = t[6] + t[7] + t[8];
    const double iS = 1.0 / S0;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        t[b] *= iS;
        t[3 + b] = (t[3 + b] - t[b] * S1) * iS;
        t[6 + b] = (t[6 + b] - 2.0 * t[3 + b] * S1 - t[b] * S2) * iS;
    }
    double xc[3];
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const int64_t id = d == 0 ? (int64_t)M.na[1] * M.na[2] * (e + b) : d == 1 ? (int64_t)M.na[2] * (e + b) : e + b;
        xc[b] = M.X[3 * id + d];
    }
    // (parametric tables of a patch that is not separable: g = 1, g' = 0)
    const double g = M.separable ? t[3] * xc[0] + t[4] * xc[1] + t[5] * xc[2] : 1.0;
    const double gp = M.separable ? t[6] * xc[0] + t[7] * xc[1] + t[8] * xc[2] : 0.0;
    const double ig = 1.0 / g, r = gp * ig;
    double *o = tab + (int64_t)(first + e) * TAB_STRIDE;
    float *of = tabf + (int64_t)(first + e) * TAB_STRIDE;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const double v[3] = {t[b], t[3 + b] * ig, (t[6 + b] - r * t[3 + b]) * (ig * ig)};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            o[9 * q + 3 * a + b] = v[a];
            of[9 * q + 3 * a + b] = (float)v[a];
        }
    }
    const double w = M.gw[q] * (kV[3] - kV[2]) * g;
    o[36 + q] = w;
    of[36 + q] = (float)w;
}

// Per-element set-up on a separable patch (at least 256 threads, no barrier):
// the 27 control displacements -> sU[27][STR], the tables of the element's three
// 1-D elements -> sPd[d][q][order][i] and their point weights -> sW[d][q].
template <int NH = 1, int STR = 3>
__device__ __forceinline__ void sep_element(const MeshK &M, const double *__restrict__ Uh, const int *ed, double *sU,
                                            double (*sPd)[4][3][3], double (*sW)[4], int64_t ndof = 0,
                                            double *sUd = nullptr)
{
    const int tid = threadIdx.x;
    if (tid < 27) {
        const int bx = tid / 9, by = (tid / 3) % 3, bz = tid % 3;
        const int64_t oc = ((int64_t)M.nb[1] * M.nb[2]) * own1(ed[0] + bx, M.nb[0], M.periodic[0])
                         + (int64_t)M.nb[2] * own1(ed[1] + by, M.nb[1], M.periodic[1]) + own1(ed[2] + bz, M.nb[2], M.periodic[2]);
        if (NH == 1) {
#pragma unroll
            for (int k = 0; k < 3; k++) sU[STR * tid + k] = Uh[3 * oc + k];
        } else {
            // the transient rule's two fields: Um = (U^1 + U^2)/2 -> sU and
            // Ud = (U - U^2)/2 -> sUd (rule node j: Um + s_j Ud)
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double u0 = Uh[3 * oc + k], u1 = Uh[ndof + 3 * oc + k], u2 = Uh[2 * ndof + 3 * oc + k];
                sU[STR * tid + k] = 0.5 * (u1 + u2);
                sUd[STR * tid + k] = 0.5 * (u0 - u2);
            }
        }
    } else if (tid >= 64 && tid < 64 + 3 * TAB_STRIDE) {
        const int d = (tid - 64) / TAB_STRIDE, i = (tid - 64) - TAB_STRIDE * d;
        const double v = M.tab[d][(int64_t)ed[d] * TAB_STRIDE + i];
        if (i < 36) (&sPd[d][0][0][0])[i] = v;
        else sW[d][i - 36] = v;
    }
}

// the periodic macro-field at point q added to the jet of component k
__device__ __forceinline__ void sep_macro(const MeshK &M, const int *ed, int q, int k, double *J)
{
    const int qd[3] = {q >> 4, (q >> 2) & 3, q & 3};
    double xq[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double *kV = M.knot[d] + ed[d];
        const double c = M.gq[qd[d]];
        xq[d] = (-c + 1.0) * kV[2] + c * kV[3];
    }
    add_periodic1(M, xq, k, J);
}

// Physical displacement jets at the 64 Gauss points of a separable element by
// sum factorisation over the physical tables (z, y, then x; sWork holds 1188
// doubles), after sep_element and a barrier; at least 192 threads, all of which
// call it.  Lane q of wave k < 3 returns in J the jet of component k at point q
// (par_periodic's macro-field added).  The passes are
// short and serial, so each takes as many threads as it has independent groups
// of outputs (108, 144 and 192).
__device__ __forceinline__ void sep_fields(const MeshK &M, const int *ed, const double *sU, const double (*sPd)[4][3][3],
                                           double *sWork, double *J)
{
    const int tid = threadIdx.x;
    double *sA = sWork, *sB = sA + 3 * 108;
    // z: sA[k][bx*3+by][qz][dz] = sum_bz U_k(b) Pz[qz][dz][bz]
    if (tid < 108) {
        const int qz = tid & 3, g = tid >> 2, k = g / 9, bxy = g - 9 * k;
        const double c0 = sU[3 * (3 * bxy) + k], c1 = sU[3 * (3 * bxy + 1) + k], c2 = sU[3 * (3 * bxy + 2) + k];
        double *o = sA + 108 * k + 12 * bxy + 3 * qz;
#pragma unroll
        for (int dz = 0; dz < 3; dz++) {
            const double *tz = &sPd[2][qz][dz][0];
            o[dz] = c0 * tz[0] + c1 * tz[1] + c2 * tz[2];
        }
    }
    __syncthreads();
    // y: sB[k][bx][qy][qz][s6] = sum_by sA[k][bx*3+by][qz][dz(s6)] Py[qy][dy(s6)][by],
    //    s6 = (dy, dz) in the order (0,0) (1,0) (0,1) (2,0) (1,1) (0,2)
    if (tid < 144) {
        const int qz = tid & 3, qy = (tid >> 2) & 3, g = tid >> 4, k = g / 3, bx = g - 3 * k;
        const double *a = sA + 108 * k + 36 * bx + 3 * qz;   // a[12 by + dz]
        double *o = sB + 288 * k + 96 * bx + 24 * qy + 6 * qz;
#pragma unroll
        for (int s6 = 0; s6 < 6; s6++) {
            const int dy = (s6 == 1 || s6 == 4) ? 1 : (s6 == 3 ? 2 : 0);
            const int dz = (s6 == 2 || s6 == 4) ? 1 : (s6 == 5 ? 2 : 0);
            const double *ty = &sPd[1][qy][dy][0];
            o[s6] = a[dz] * ty[0] + a[12 + dz] * ty[1] + a[24 + dz] * ty[2];
        }
    }
    __syncthreads();
    // x
    if (tid < 192) {
        const int q = tid & 63, k = tid >> 6;
        sf_jet(sB + 288 * k + (q & 15) * 6, &sPd[0][q >> 4][0][0], J);
        sep_macro(M, ed, q, k, J);
    }
}

// Field passes of six nodal fields c[b][f] at once (two of sep_fields' sets, or
// coordinates and displacements), sWork 6 * (108 + 288) doubles: the z and y
// passes; six_jet then is the x pass of one field at one point.  One pass of
// six has half the barriers of two passes of three.
__device__ __forceinline__ void six_fields(const double (*c)[6], const double (*sPd)[4][3][3], double *sWork)
{
    double *sA = sWork, *sB = sA + 6 * 108;
    for (int i = threadIdx.x; i < 216; i += blockDim.x) {
        const int qz = i & 3, g = i >> 2, f = g / 9, bxy = g - 9 * f;
        const double c0 = c[3 * bxy][f], c1 = c[3 * bxy + 1][f], c2 = c[3 * bxy + 2][f];
        double *o = sA + 108 * f + 12 * bxy + 3 * qz;
#pragma unroll
        for (int dz = 0; dz < 3; dz++) {
            const double *tz = &sPd[2][qz][dz][0];
            o[dz] = c0 * tz[0] + c1 * tz[1] + c2 * tz[2];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 288; i += blockDim.x) {
        const int qz = i & 3, qy = (i >> 2) & 3, g = i >> 4, f = g / 3, bx = g - 3 * f;
        const double *a = sA + 108 * f + 36 * bx + 3 * qz;   // a[12 by + dz]
        double *o = sB + 288 * f + 96 * bx + 24 * qy + 6 * qz;
#pragma unroll
        for (int s6 = 0; s6 < 6; s6++) {
            const int dy = (s6 == 1 || s6 == 4) ? 1 : (s6 == 3 ? 2 : 0);
            const int dz = (s6 == 2 || s6 == 4) ? 1 : (s6 == 5 ? 2 : 0);
            const double *ty = &sPd[1][qy][dy][0];
            o[s6] = a[dz] * ty[0] + a[12 + dz] * ty[1] + a[24 + dz] * ty[2];
        }
    }
    __syncthreads();
}
__device__ __forceinline__ void six_jet(const double *sWork, const double (*sPd)[4][3][3], int f, int q, double *J)
{
    sf_jet(sWork + 6 * 108 + 288 * f + (q & 15) * 6, &sPd[0][q >> 4][0][0], J);
}
// Gauss weight x span lengths x det G at point q of a separable element
__device__ __forceinline__ double sep_weight(int q, const double (*sW)[4]) { return sW[0][q >> 4] * sW[1][(q >> 2) & 3] * sW[2][q & 3]; }

// Strain-measure states of the 64 points for StaticIn, from the jets of
// sep_fields (lane q of wave k < 3 holds component k; 256 threads take part):
// F and H as they come; then wave K < 3 takes column K of the strain gradients
// and wave 3 the strains.  Ends with a block barrier.
__device__ __forceinline__ void sep_states(const PhysK &P, const double *J, const double (*sW)[4], double *sSt)
{
    constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
    const int tid = threadIdx.x, q = tid & 63, part = tid >> 6;
    double *sp = sSt + q * SST_W;
    if (tid < 192) {
#pragma unroll
        for (int i = 0; i < 3; i++) sp[10 * part + i] = J[1 + i] + (part == i ? 1.0 : 0.0);
#pragma unroll
        for (int t = 0; t < 6; t++) sp[10 * part + 4 + t] = J[4 + t];
    }
    __syncthreads();
    if (tid < 256) {
        double F[9];
#pragma unroll
        for (int i = 0; i < 9; i++) F[i] = sp[10 * (i / 3) + i % 3];
        const double w = sep_weight(q, sW);
        if (part < 3) {
            // G_IK = 2 le^2 (E_II,K - their mean), column K = part
            const int h[3] = {part, part == 0 ? 1 : part + 2, part == 0 ? 2 : part + 3};   // slot of (I, K)
            double EK[3];
#pragma unroll
            for (int I = 0; I < 3; I++) EK[I] = F[I] * sp[4 + h[I]] + F[3 + I] * sp[14 + h[I]] + F[6 + I] * sp[24 + h[I]];
            const double tr = (EK[0] + EK[1] + EK[2]) / 3.0, g = w * 2 * P.le * P.le;
#pragma unroll
            for (int I = 0; I < 3; I++) sp[SST_G + 3 * I + part] = g * (EK[I] - tr);
        } else {
            double S[9], N[9];
            phys_strain(F, P, S, N);
#pragma unroll
            for (int I = 0; I < 3; I++)
#pragma unroll
                for (int K = I; K < 3; K++) {
                    sp[SST_S + SY[I][K]] = w * S[3 * I + K];
                    sp[SST_N + SY[I][K]] = w * N[3 * I + K];
                }
            sp[SST_WGT] = w;
        }
    }
    __syncthreads();
}

// Write-out of the separable tangents: a y lane of the pipeline holds the
// entries K[(3 bx + cx) * 3 + by] of block p = (i, j) for its cy and bc = 3 bz + cz.  DIRECT: sRow and sMsk hold the row starts and Dirichlet flags
// of the element's 81 rows.
template <typename T, bool DIRECT>
__device__ __forceinline__ void sep_write(const MeshK &M, T *__restrict__ Ke, int e, int ex, int ey, int ez, int p, int bc, int cy, const T *K,
                                          const int64_t *sRow, const int32_t *sMsk)
{
    // (the lane's place is hidden from the loop around the call: its addresses,
    // hoisted out of it, would fill the registers)
    asm volatile("" : "+v"(p), "+v"(bc));
    const int bz = bc / 3, cz = bc % 3;
    const int i = blk_k(p), j = blk_l(p);
    if constexpr (DIRECT) {
        // ---- add (row 3b+i, column 3c+j) and the mirrored entry into the CSR
        //      values, Dirichlet rows and columns left at zero; the elements
        //      of one colour share no row.  Per bx all loads of the nine
        //      entries (and mirrors) before their stores (one round trip for
        //      all 27 measured slower: the scattered read-modify-write of the
        //      CSR values, not its latency, is the cost).
#pragma unroll
        for (int bx = 0; bx < 3; bx++) {
            T vp[9], vq[9];
            int64_t pp[9], pq[9];
            bool ok[9];
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const int cx = t / 3, by = t % 3, b = 9 * bx + 3 * by + bz, c = 9 * cx + 3 * cy + cz;
                ok[t] = sMsk[3 * b + i] == 0 && sMsk[3 * c + j] == 0;
                pp[t] = stencil_pos(M, sRow[3 * b + i], ex + bx, ey + by, ez + bz, ex + cx, ey + cy, ez + cz, j);
                pq[t] = stencil_pos(M, sRow[3 * c + j], ex + cx, ey + cy, ez + cz, ex + bx, ey + by, ez + bz, i);
                vp[t] = vq[t] = (T)0;
                if (ok[t]) {
                    vp[t] = Ke[pp[t]];
                    if (i != j) vq[t] = Ke[pq[t]];
                }
            }
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const T v = K[9 * bx + t];
                if (ok[t]) {
                    Ke[pp[t]] = vp[t] + v;
                    if (i != j) Ke[pq[t]] = vq[t] + v;
                }
            }
        }
        return;
    }
    // ---- K_e: row 3b+i, column 3c+j, and the mirrored block (3c+j, 3b+i)
    T *out = Ke + (int64_t)e * 6561;
#pragma unroll
    for (int bx = 0; bx < 3; bx++)
#pragma unroll
        for (int cx = 0; cx < 3; cx++)
#pragma unroll
            for (int by = 0; by < 3; by++) {
                const int b = 9 * bx + 3 * by + bz, c = 9 * cx + 3 * cy + cz;
                const T v = K[(3 * bx + cx) * 3 + by];
                out[(3 * b + i) * 81 + 3 * c + j] = v;
                if (i != j) out[(3 * c + j) * 81 + 3 * b + i] = v;
            }
}

// element indices of workgroup g: element g, or (DIRECT) element g of the colour S.c
template <bool DIRECT>
__device__ __forceinline__ void sep_index(const MeshK &M, const Scatter &S, int g, int *ed)
{
    if (DIRECT) {
        ed[0] = S.c[0] + 3 * (g / (S.nc[1] * S.nc[2]));
        ed[1] = S.c[1] + 3 * ((g / S.nc[2]) % S.nc[1]);
        ed[2] = S.c[2] + 3 * (g % S.nc[2]);
    } else {
        ed[0] = g / (M.nelem[1] * M.nelem[2]);
        ed[1] = (g / M.nelem[2]) % M.nelem[1];
        ed[2] = g % M.nelem[2];
    }
}

// row starts and Dirichlet flags of the element's 81 rows -> LDS (direct scatter)
__device__ __forceinline__ void sep_rows(const MeshK &M, const Scatter &S, const int *ed, int64_t *sRow, int32_t *sMsk)
{
    const int tid = threadIdx.x;
    if (tid < 81) {
        const int b = tid / 3, i = tid - 3 * b;
        const int64_t cp = ((int64_t)M.nb[1] * M.nb[2]) * (ed[0] + b / 9) + (int64_t)M.nb[2] * (ed[1] + (b / 3) % 3) + (ed[2] + b % 3);
        sRow[tid] = S.rowptr[3 * cp + i];
        sMsk[tid] = S.mask[3 * cp + i];
    }
}

// Shape of the separable tangents' pipeline (E1 buffers, D prefetch, loads of an
// interval all before its first product) and the waves per SIMD it is compiled for.
// Measured at 128x32x32 (kernel time; the same order at 64x16x16):
//   static FP64     two buffers 9.2 ms, one 9.7 (160 KB of LDS leave one workgroup per CU
//                   either way); without the prefetch 9.4
//   static FP32     one buffer and two workgroups per CU (79 KB) 5.3 ms, two buffers and
//                   one workgroup 7.6; with the prefetch 5.8; compiled for one 5.3
//   transient FP64  one buffer is what fits (149 KB), 13.5 ms; with the prefetch 16.7
//   transient FP32  one buffer and two workgroups per CU (76 KB) 10.9 ms, two buffers and one
//                   workgroup 11.5, compiled for one workgroup 12.1; with the prefetch 10.2 (open)
// The order of the loads makes no difference above 1% anywhere; it is the one that
// the registers allow.
template <typename T, int NH> struct SepPipe;
template <> struct SepPipe<double, 1> { typedef PipeShape<2, true, true> S; static constexpr int OCC = 2; };
template <> struct SepPipe<float, 1> { typedef PipeShape<1, false, false> S; static constexpr int OCC = 4; };
template <> struct SepPipe<double, 3> { typedef PipeShape<1, false, true> S; static constexpr int OCC = 2; };
template <> struct SepPipe<float, 3> { typedef PipeShape<1, false, false> S; static constexpr int OCC = 4; };
template <typename T, int NH> using SepShape = typename SepPipe<T, NH>::S;

// Static tangent of a separable patch: a workgroup per element -- tables and
// displacements, jets and strain-measure states of the 64 points (one pass of
// all waves each), then the pipeline of igap_sep_pipeline.h.
// Bound in FP64 by latency with one workgroup per CU: 16.6k vector instructions an
// element take 41% of the issue slots of the 40.6k cycles its workgroup lives, and a wave
// waits 44% of them, at the pipeline's barriers and the set-up's; in FP32, two
// workgroups per CU, by vector issue, 71% of the slots.  The stages on waves of their own, D, z
// and y/x side by side, replace a loop over pencils in which every wave ran all
// stages with a barrier after each and the matrix cores idle, the z stage as four
// lanes' partial sums: at 128x32x32 12.9 -> 9.1 ms in FP64 and 8.1 -> 5.3 ms in
// FP32, at 16x4x4 (FP64) 42 -> 28 us.  FP64 holds two E1 buffers and one
// workgroup per CU (160 KB of LDS); twelve waves at 168 registers (two sets of y
// waves) took 9.65 ms, six waves of one pencil and two workgroups per CU 12.5.
// FP32 fits two workgroups of 79 KB with one E1 buffer.
template <typename T, bool DIRECT>
__global__ __launch_bounds__((SepShape<T, 1>::THREADS), (SepPipe<T, 1>::OCC)) void k_tangent_sep(
    MeshK M, PhysK P, const double *__restrict__ Uh, T *__restrict__ Ke, Scatter S, const T *__restrict__ tabx,
    const T *__restrict__ taby, const T *__restrict__ tabz)
{
    typedef SepShape<T, 1> Sh;
    __shared__ double sPd[3][4][3][3];          // 1-D tables of physical derivatives [d][q_d][order][i]
    __shared__ double sW[3][4];                 // 1-D point weights
    __shared__ double sU[27 * 3];
    __shared__ __attribute__((aligned(16))) double sSt[64 * SST_W];          // strain-measure states (StaticIn)
    __shared__ T sX[36];                        // x table in the contraction's precision
    __shared__ int64_t sRow[DIRECT ? 81 : 1];
    __shared__ int32_t sMsk[DIRECT ? 81 : 1];
    __shared__ __attribute__((aligned(16))) T sD[Sh::D_SIZE];
    __shared__ __attribute__((aligned(16))) T sE[Sh::E_SIZE];   // first the field passes' buffers (1188 doubles)
    static_assert(Sh::E_SIZE * sizeof(T) >= 3 * (108 + 288) * sizeof(double), "field buffers in sE");

    const int tid = threadIdx.x, e = blockIdx.x;
    int ed[3];
    sep_index<DIRECT>(M, S, e, ed);
    if (DIRECT) sep_rows(M, S, ed, sRow, sMsk);
    if (tid >= 256 && tid < 256 + 36) sX[tid - 256] = tabx[ed[0] * TAB_STRIDE + tid - 256];
    sep_element(M, Uh, ed, sU, sPd, sW);
    __syncthreads();
    // ---- displacement jets and strain-measure states
    {
        double J[10];
        sep_fields(M, ed, sU, sPd, reinterpret_cast<double *>(sE), J);
        sep_states(P, J, sW, sSt);
    }
    const StaticIn in{sSt, P.e345, P.le};
    auto out = [&](int p, int bc, int cy, const T *K) {
        sep_write<T, DIRECT>(M, Ke, e, ed[0], ed[1], ed[2], p, bc, cy, K, sRow, sMsk);
    };
    sep_pipeline<T, Sh>(sX, taby + ed[1] * TAB_STRIDE, tabz + ed[2] * TAB_STRIDE, sD, sE, in, out);
}

// Static tangent of a patch with equal weights and any geometry (k_tangent_gen):
// the basis is a tensor product in the parametric directions, so the pipeline of
// k_tangent_sep contracts the parametric tables, and GeneralIn pulls the
// pointwise tangent back to parametric slots.  Set-up: the jets of the three
// coordinates and the three displacements by sum factorisation (one wave per
// field in the last pass), then per point the map's inverse gradient,
// connection and metric (one wave) and the physical displacement jets (three),
// then the strain-measure state.
// Bound by the D wave: 1005 vector instructions an interval (849 FP64; FP32 1076 and
// 930) in one stream, for which the other seven waves wait (62% of a wave's life,
// 32% of the issue slots used), in both precisions.  64x16x16, FP64: 3.47 ms for
// k_tangent_elem, whose matrix-core product of 27 x 27 per point and jet slot alone
// is 55k cycles an element and CU, 2.05 ms here.  A rational basis (unequal
// weights) needs the value slot too and stays with k_tangent_elem.
// Shape as below (128x32x32, kernel): FP64 fits one E1 buffer (148 KB of LDS); FP32 two,
// 15.5 ms, one 16.1 (two workgroups do not fit either way).  Loads all before the
// first product: 16.1 and 15.5 ms, without 16.3 and 15.5.
template <typename T> struct GenPipe;
template <> struct GenPipe<double> { typedef PipeShape<1, false, true> S; };
template <> struct GenPipe<float> { typedef PipeShape<2, false, true> S; };

// the states of GeneralIn at the 64 points (eight waves; lane q of wave f < 6 holds field f's parametric jet at point q in J); ends with a block barrier
__device__ __forceinline__ void gen_states(const MeshK &M, const PhysK &P, const int *ed, double *J, const double (*sW)[4], double *sSt)
{
    constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
    constexpr int PI[6] = {0, 0, 0, 1, 1, 2}, PK[6] = {0, 1, 2, 1, 2, 2};
    const int tid = threadIdx.x, q = tid & 63, part = tid >> 6;
    double *sp = sSt + q * GST_W;
    // the coordinates' jets wait in the places of S, N and G
    if (part < 3) {
#pragma unroll
        for (int a = 0; a < 9; a++) sp[GST_S + 9 * part + a] = J[1 + a];
    }
    __syncthreads();
    if (part >= 3 && part < 7) {
        double G[9], Gi[9], X2[18];
#pragma unroll
        for (int d = 0; d < 3; d++) {
#pragma unroll
            for (int i = 0; i < 3; i++) G[3 * d + i] = sp[GST_S + 9 * d + i];
#pragma unroll
            for (int s = 0; s < 6; s++) X2[6 * d + s] = sp[GST_S + 9 * d + 3 + s];
        }
        const double det = inv3(G, Gi);
        if (part < 6) {
            const int k = part - 3;
            phys_jet(J, Gi, X2);
            sep_macro(M, ed, q, k, J);
#pragma unroll
            for (int i = 0; i < 3; i++) sp[10 * k + i] = J[1 + i] + (k == i ? 1.0 : 0.0);
#pragma unroll
            for (int t = 0; t < 6; t++) sp[10 * k + 4 + t] = J[4 + t];
        } else {
#pragma unroll
            for (int i = 0; i < 9; i++) sp[GST_GI + i] = Gi[i];
            sp[GST_WGT] = sep_weight(q, sW) * det;
#pragma unroll
            for (int n = 0; n < 3; n++)
#pragma unroll
                for (int s = 0; s < 6; s++)
                    sp[GST_GA + 6 * n + s] = Gi[3 * n] * X2[s] + Gi[3 * n + 1] * X2[6 + s] + Gi[3 * n + 2] * X2[12 + s];
#pragma unroll
            for (int s = 0; s < 6; s++)
                sp[GST_M + s] = Gi[3 * PI[s]] * Gi[3 * PK[s]] + Gi[3 * PI[s] + 1] * Gi[3 * PK[s] + 1] + Gi[3 * PI[s] + 2] * Gi[3 * PK[s] + 2];
        }
    }
    __syncthreads();
    if (part < 4) {
        double F[9];
#pragma unroll
        for (int i = 0; i < 9; i++) F[i] = sp[10 * (i / 3) + i % 3];
        const double w = sp[GST_WGT];
        if (part < 3) {
            // row L = part of G_LK = 2 le^2 (E_LL,K - their mean over L), its second index pulled back
            const int L = part;
            const double g = w * 2 * P.le * P.le;
            double GL[3], Gi[9], gh[3];
#pragma unroll
            for (int K = 0; K < 3; K++) {
                double EK[3];
#pragma unroll
                for (int I = 0; I < 3; I++)
                    EK[I] = F[I] * sp[4 + SY[I][K]] + F[3 + I] * sp[14 + SY[I][K]] + F[6 + I] * sp[24 + SY[I][K]];
                const double tr = (EK[0] + EK[1] + EK[2]) / 3.0;
                GL[K] = g * ((L == 0 ? EK[0] : L == 1 ? EK[1] : EK[2]) - tr);
            }
#pragma unroll
            for (int i = 0; i < 9; i++) Gi[i] = sp[GST_GI + i];
            double gl[3];   // Gi_rL
#pragma unroll
            for (int r = 0; r < 3; r++) {
                gh[r] = GL[0] * Gi[3 * r] + GL[1] * Gi[3 * r + 1] + GL[2] * Gi[3 * r + 2];
                gl[r] = L == 0 ? Gi[3 * r] : L == 1 ? Gi[3 * r + 1] : Gi[3 * r + 2];
            }
#pragma unroll
            for (int s = 0; s < 6; s++) {
                double x = gl[PI[s]] * gh[PK[s]];
                if (PI[s] != PK[s]) x += gl[PK[s]] * gh[PI[s]];
                sp[GST_G + 6 * L + s] = x;
            }
        } else {
            double S[9], N[9];
            phys_strain(F, P, S, N);
#pragma unroll
            for (int I = 0; I < 3; I++)
#pragma unroll
                for (int K = I; K < 3; K++) {
                    sp[GST_S + SY[I][K]] = w * S[3 * I + K];
                    sp[GST_N + SY[I][K]] = w * N[3 * I + K];
                }
        }
    }
    __syncthreads();
}

template <typename T, bool DIRECT>
__global__ __launch_bounds__((GenPipe<T>::S::THREADS), 2) void k_tangent_gen(
    MeshK M, PhysK P, const double *__restrict__ Uh, T *__restrict__ Ke, Scatter S, const T *__restrict__ tabx,
    const T *__restrict__ taby, const T *__restrict__ tabz)
{
    typedef typename GenPipe<T>::S Sh;
    __shared__ double sPd[3][4][3][3];          // 1-D parametric tables [d][q_d][order][i]
    __shared__ double sW[3][4];                 // 1-D point weights
    __shared__ double sC[27][6];                // control points, then displacements
    __shared__ __attribute__((aligned(16))) double sSt[64 * GST_W];
    __shared__ T sX[36];
    __shared__ int64_t sRow[DIRECT ? 81 : 1];
    __shared__ int32_t sMsk[DIRECT ? 81 : 1];
    __shared__ __attribute__((aligned(16))) T sD[Sh::D_SIZE];
    __shared__ __attribute__((aligned(16))) T sE[Sh::E_SIZE];   // first the field passes' buffers (2376 doubles)
    static_assert(Sh::THREADS == 512, "gen_states takes eight waves");
    static_assert(Sh::E_SIZE * sizeof(T) >= 6 * (108 + 288) * sizeof(double), "field buffers in sE");

    const int tid = threadIdx.x, e = blockIdx.x;
    int ed[3];
    sep_index<DIRECT>(M, S, e, ed);
    if (DIRECT) sep_rows(M, S, ed, sRow, sMsk);
    if (tid >= 256 && tid < 256 + 36) sX[tid - 256] = tabx[ed[0] * TAB_STRIDE + tid - 256];
    if (tid >= 320 && tid < 320 + 27) {
        const int b = tid - 320, ax = ed[0] + b / 9, ay = ed[1] + (b / 3) % 3, az = ed[2] + b % 3;
        const int64_t id = ((int64_t)M.na[1] * M.na[2]) * ax + (int64_t)M.na[2] * ay + az;
        // (relative to the element's middle point: only derivatives are used, and
        // their rounding errors then scale with the element's size)
        const int64_t mid = ((int64_t)M.na[1] * M.na[2]) * (ed[0] + 1) + (int64_t)M.na[2] * (ed[1] + 1) + ed[2] + 1;
#pragma unroll
        for (int d = 0; d < 3; d++) sC[b][d] = M.X[3 * id + d] - M.X[3 * mid + d];
    }
    sep_element<1, 6>(M, Uh, ed, &sC[0][3], sPd, sW);
    __syncthreads();
    {
        double J[10];
        six_fields(sC, sPd, reinterpret_cast<double *>(sE));
        if (tid < 384) six_jet(reinterpret_cast<double *>(sE), sPd, tid >> 6, tid & 63, J);
        gen_states(M, P, ed, J, sW, sSt);
    }
    const GeneralIn in{sSt, P.e345, P.le};
    auto out = [&](int p, int bc, int cy, const T *K) {
        sep_write<T, DIRECT>(M, Ke, e, ed[0], ed[1], ed[2], p, bc, cy, K, sRow, sMsk);
    };
    sep_pipeline<T, Sh>(sX, taby + ed[1] * TAB_STRIDE, tabz + ed[2] * TAB_STRIDE, sD, sE, in, out);
}

// Transient tangent on a separable patch (k_tangent_sep_t, gradelasttime):
// the rule-weighted pointwise rows of k_tangent_elem<..., 3> (c_row_mom: the
// eight rule-node states us_j = Um + s_j Ud collapsed into moments) in
// the pipeline of k_tangent_sep, plus the inertia term.  The inertia block
// D[(k,0),(k,0)] = w_q (cii / (2 dt) + rho / dt^2) pairs only basis values,
// and w_q and the basis value are products over the directions, so its part
// of K^kk is mc Mx[bx][cx] My[by][cy] Mz[bz][cz] with the 1-D matrices
// M_d[b][c] = sum_q gw_q dX_d g_d(q) rho_b(q) rho_c(q).  Stage A: the jets of
// Um and Ud (two field passes), then the moment states of all 64 points,
// compact and in the contraction's precision (one lane per rule node, sums
// over 8-lane groups), so that the FP32 kernel keeps two workgroups per CU
// (76 KB of LDS; FP64, 149 KB: one).  Bound by latency: a wave waits 46% of its life in
// FP64 (44% of the issue slots used) and 64% in FP32 (58% used; 62 registers spilled),
// for the D wave (534 vector instructions an interval, 363 FP64; FP32 688 and 490) and
// in stage A (all six fields in one pass, a lane per rule node and point, sums by
// lane moves; as two passes, two rounds of half the waves and LDS permutations it took
// 13.5 ms at 128x32x32 in FP32, 10.9 now; FP64 at 24^3 1.78 -> 1.48 ms).  Two
// pencils per interval and one D wave: one pencil and two D waves took 18.8 ms,
// their registers limiting both to two workgroups.
template <typename T, bool DIRECT>
__global__ __launch_bounds__((SepShape<T, 3>::THREADS), (SepPipe<T, 3>::OCC)) void k_tangent_sep_t(
    MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof, T *__restrict__ Ke, Scatter S, const T *__restrict__ tabx,
    const T *__restrict__ taby, const T *__restrict__ tabz)
{
    typedef SepShape<T, 3> Sh;
    __shared__ double sPd[3][4][3][3];
    __shared__ double sW[3][4];
    __shared__ double sC[27][6];                // nodal Um, Ud
    __shared__ double sWgt[64];
    __shared__ double sMass[3][3][3];          // 1-D mass matrices M_d[b][c]
    __shared__ __attribute__((aligned(16))) T sMom[64 * MS_W];   // compact moment states (first the field passes' buffers)
    __shared__ T sX[36];
    __shared__ int64_t sRow[DIRECT ? 81 : 1];
    __shared__ int32_t sMsk[DIRECT ? 81 : 1];
    __shared__ __attribute__((aligned(16))) T sD[Sh::D_SIZE];
    __shared__ __attribute__((aligned(16))) T sE[Sh::E_SIZE];
    static_assert(64 * MS_W * sizeof(T) >= 6 * (108 + 288) * sizeof(double) && Sh::D_SIZE >= 64 * 54, "stage A's buffers");
    static_assert(Sh::THREADS == 512, "a lane per rule node and point");
    T *sJet = sD;                               // [q][h][k][a - 1], stage A only

    const int tid = threadIdx.x, e = blockIdx.x;
    int ed[3];
    sep_index<DIRECT>(M, S, e, ed);
    if (DIRECT) sep_rows(M, S, ed, sRow, sMsk);

    if (tid >= 256 && tid < 256 + 36) sX[tid - 256] = tabx[ed[0] * TAB_STRIDE + tid - 256];
    sep_element<3, 6>(M, Uh, ed, &sC[0][0], sPd, sW, ndof, &sC[0][3]);
    __syncthreads();
    // ---- stage A: jets of Um and Ud, point weights, 1-D mass matrices
    {
        double *work = reinterpret_cast<double *>(sMom);
        six_fields(sC, sPd, work);
        const int q = tid & 63, f = tid >> 6;   // field f < 3: Um, f < 6: Ud
        if (f < 6) {
            double J[10];
            six_jet(work, sPd, f, q, J);
            if (f < 3) sep_macro(M, ed, q, f, J);
#pragma unroll
            for (int a = 1; a < 10; a++) sJet[q * 54 + 9 * f + a - 1] = (T)J[a];
        } else if (f == 6) {
            sWgt[q] = sep_weight(q, sW);
        } else if (q < 27) {
            const int d = q / 9, b = (q / 3) % 3, c = q % 3;
            double m = 0.0;
#pragma unroll
            for (int qq = 0; qq < 4; qq++) m += sW[d][qq] * sPd[d][qq][0][b] * sPd[d][qq][0][c];
            sMass[d][b][c] = m;
        }
    }
    __syncthreads();
    // ---- moment states: lane 8g + j takes rule node j of point g; node sums
    //      over the 8-lane group one entry at a time; F^ and H^ from the jets,
    //      3-4 entries per lane
    {
        Mom mu = {0.0, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            mu.m0 += P.ct[j];
            mu.m1 += P.ct[j] * P.s[j];
            mu.m2 += P.ct[j] * P.s[j] * P.s[j];
        }
        mu.factor();
        const double c12 = 1.0 / (mu.a11 * mu.a22), c22 = 1.0 / mu.d2;
        const int j = tid & 7;
        const int q = tid >> 3;
        const T *jq = sJet + q * 54;
        T *ms = sMom + q * MS_W;
        {
            double us[30];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                us[10 * k] = 0.0;
#pragma unroll
                for (int a = 1; a < 10; a++) us[10 * k + a] = (double)jq[9 * k + a - 1] + P.s[j] * (double)jq[27 + 9 * k + a - 1];
            }
            State st;
            phys_state(us, P, st);
            const double w0 = P.ct[j], w1 = w0 * P.s[j], w2 = w1 * P.s[j];
            constexpr int PR[6] = {0, 1, 2, 4, 5, 8};   // index pairs I <= J in slot order
#pragma unroll
            for (int t = 0; t < 6; t++) {
                double sv = w0 * st.S[PR[t]], n0 = w0 * st.N[PR[t]], n1 = w1 * st.N[PR[t]], n2 = w2 * st.N[PR[t]];
                sv = sum8(sv);
                n0 = sum8(n0);
                n1 = sum8(n1);
                n2 = sum8(n2);
                if (j == 0) {
                    ms[MS_S + t] = (T)sv;
                    ms[MS_N11 + t] = (T)(n0 / mu.m0);
                    ms[MS_N12 + t] = (T)((n1 - mu.lf * n0) * c12);
                    ms[MS_N22 + t] = (T)(((mu.lf * n0 - n1) * mu.lf + (n2 - mu.lf * n1)) * c22);
                }
            }
#pragma unroll
            for (int i = 0; i < 9; i++) {
                const double gv = sum8(w0 * st.G[i]);
                if (j == 0) ms[MS_G + i] = (T)gv;
            }
        }
        // F^ (r < 9: F_kL, k = r / 3, L = r % 3) and H^ (r >= 9: H_k,IK in
        // slot 4 + t of component k = (r - 9) / 6): X^_1 = a11 (X0 + lf Xd),
        // X^_2 = a22 Xd
        for (int r = j; r < 27; r += 8) {
            int src;
            double x0;
            if (r < 9) {
                src = 9 * (r / 3) + (r % 3);
                x0 = (double)jq[src] + ((r / 3) == (r % 3) ? 1.0 : 0.0);
            } else {
                src = 9 * ((r - 9) / 6) + 3 + (r - 9) % 6;
                x0 = (double)jq[src];
            }
            const double xd = (double)jq[27 + src];
            const double x1 = mu.a11 * (x0 + mu.lf * xd), x2 = mu.a22 * xd;
            if (r < 9) {
                ms[18 * (r / 3) + r % 3] = (T)x1;
                ms[18 * (r / 3) + 3 + r % 3] = (T)x2;
            } else {
                ms[18 * ((r - 9) / 6) + 6 + (r - 9) % 6] = (T)x1;
                ms[18 * ((r - 9) / 6) + 12 + (r - 9) % 6] = (T)x2;
            }
        }
    }
    __syncthreads();

    const MomentIn<T> in{sMom, sWgt, P.e345, P.le};
    auto out = [&](int p, int bc, int cy, T *K) {
        // inertia on the diagonal blocks
        const int bz = bc / 3, cz = bc % 3;
        if (blk_k(p) == blk_l(p)) {
            const double mc = P.cii / (2. * P.dt) + P.rho / (P.dt * P.dt);
#pragma unroll
            for (int bx = 0; bx < 3; bx++)
#pragma unroll
                for (int cx = 0; cx < 3; cx++)
#pragma unroll
                    for (int by = 0; by < 3; by++)
                        K[(3 * bx + cx) * 3 + by] += (T)(mc * sMass[0][bx][cx] * sMass[1][by][cy] * sMass[2][bz][cz]);
        }
        sep_write<T, DIRECT>(M, Ke, e, ed[0], ed[1], ed[2], p, bc, cy, K, sRow, sMsk);
    };
    sep_pipeline<T, Sh>(sX, taby + ed[1] * TAB_STRIDE, tabz + ed[2] * TAB_STRIDE, sD, sE, in, out);
}

// ============================================================================
// Residual on a separable patch (k_residual_sep, static physics; volume loop
// of Residual_iga, src/assmcore_iga.c:118-259): the displacement jets of
// sep_fields, the pointwise residual jets r_q (phys/gradelast.c) times the
// point weight, and the projection
//   R_e[b][k] = sum_q sum_a r_q[k][a] R_q[a][b]
// with R_q the tensor product of the physical tables, as the transposed sum
// factorisation x -> y -> z; no quotient or chain rule to undo.
// ============================================================================
// A wave per element: every pass fits 64 lanes component by component (36, 48 and 64
// of them for z, y, x; 48, 36 and 27 back), the jets of a lane's point stay in
// its registers, and nothing waits at a block barrier.  10 KB of LDS an element,
// so at 156 registers (128 spill 38) 12 elements are in flight per CU, whose LDS
// instructions (313 a wave) fill the CU's LDS pipe: that is the bound, a wave waits on
// it 43% of its life.  A whole residual call at 64x16x16, with its gather and back to
// back, 123 -> 67.6 us (this kernel alone 79 us in a kernel trace, where the write-back of each
// dispatch counts); at 16x4x4 9.2 -> 7.1 us, against a workgroup of four waves per element
// with six in flight per CU and the pointwise stage on one of the waves.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Field passes of one nodal component c[STR * b] by a wave: lane q gets its
// parametric or physical jet (the tables decide) at point q.  sA 108, sB 288 doubles.
template <int STR>
__device__ __forceinline__ void wave_field(const double (*sT)[TAB_STRIDE], const double *c, double *sA, double *sB, int lane, double *J)
{
    const int qz = lane & 3, qy = (lane >> 2) & 3, qx = lane >> 4;
    // z: sA[bx*3+by][qz][dz]
    if (lane < 36) {
        const double *cb = c + 3 * STR * (lane >> 2);
#pragma unroll
        for (int dz = 0; dz < 3; dz++) {
            const double *tz = &sT[2][9 * qz + 3 * dz];
            sA[3 * lane + dz] = cb[0] * tz[0] + cb[STR] * tz[1] + cb[2 * STR] * tz[2];
        }
    }
    wave_sync();
    // y: sB[bx][qy][qz][s6], s6 = (dy, dz) in the order (0,0) (1,0) (0,1) (2,0) (1,1) (0,2); bx = qx here
    if (lane < 48) {
        const double *a = sA + 36 * qx + 3 * qz;   // a[12 by + dz]
#pragma unroll
        for (int s6 = 0; s6 < 6; s6++) {
            const int dy = (s6 == 1 || s6 == 4) ? 1 : (s6 == 3 ? 2 : 0);
            const int dz = (s6 == 2 || s6 == 4) ? 1 : (s6 == 5 ? 2 : 0);
            const double *ty = &sT[1][9 * qy + 3 * dy];
            sB[6 * lane + s6] = a[dz] * ty[0] + a[12 + dz] * ty[1] + a[24 + dz] * ty[2];
        }
    }
    wave_sync();
    sf_jet(sB + (lane & 15) * 6, &sT[0][9 * qx], J);
}

// Transposed passes by a wave: lane q's weighted residual jet r[10] of one
// component -> R_e of that component at local point b = lane (0 for lane >= 27).  sR 640 doubles.
__device__ __forceinline__ double wave_project(const double (*sT)[TAB_STRIDE], const double *r, double w, double *sR, double *sA, double *sB,
                                               int lane)
{
    const int qz = lane & 3, qx = lane >> 4;
#pragma unroll
    for (int a = 0; a < 10; a++) sR[64 * a + lane] = w * r[a];
    wave_sync();
    // x^T: C1[bx][qy][qz][s6] = sum_qx sum_{a: S6(a) = s6} r[a] Px[qx][DX(a)][bx]
    if (lane < 48) {
        double c[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const double *rq = sR + 16 * x + (lane & 15), *tx = &sT[0][9 * x + qx];   // bx = qx; tx[3 dx]
            c[0] += rq[0] * tx[0] + rq[64] * tx[3] + rq[4 * 64] * tx[6];
            c[1] += rq[2 * 64] * tx[0] + rq[5 * 64] * tx[3];
            c[2] += rq[3 * 64] * tx[0] + rq[6 * 64] * tx[3];
            c[3] += rq[7 * 64] * tx[0];
            c[4] += rq[8 * 64] * tx[0];
            c[5] += rq[9 * 64] * tx[0];
        }
#pragma unroll
        for (int s6 = 0; s6 < 6; s6++) sB[6 * lane + s6] = c[s6];
    }
    wave_sync();
    // y^T: C2[bx][by][qz][dz] = sum_qy sum_{s6: dz(s6) = dz} C1[..][s6] Py[qy][dy(s6)][by]
    if (lane < 36) {
        const int by = (lane >> 2) % 3, bx = lane / 12;
        double c[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const double *c1 = sB + ((bx * 4 + y) * 4 + qz) * 6, *ty = &sT[1][9 * y + by];   // ty[3 dy]
            c[0] += c1[0] * ty[0] + c1[1] * ty[3] + c1[3] * ty[6];
            c[1] += c1[2] * ty[0] + c1[4] * ty[3];
            c[2] += c1[5] * ty[0];
        }
#pragma unroll
        for (int dz = 0; dz < 3; dz++) sA[3 * lane + dz] = c[dz];
    }
    wave_sync();
    // z^T: R_e = sum_qz sum_dz C2[bx][by][qz][dz] Pz[qz][dz][bz]
    double acc = 0.0;
    if (lane < 27) {
        const double *c2 = sA + (lane / 3) * 12;
#pragma unroll
        for (int z = 0; z < 4; z++)
#pragma unroll
            for (int dz = 0; dz < 3; dz++) acc += c2[3 * z + dz] * sT[2][9 * z + 3 * dz + lane % 3];
    }
    return acc;
}

// the element's 1-D tables [q][order][function] with their point weights, by a wave
__device__ __forceinline__ void wave_tables(const MeshK &M, const int *ed, double (*sT)[TAB_STRIDE], int lane)
{
#pragma unroll
    for (int d = 0; d < 3; d++)
        if (lane < TAB_STRIDE) sT[d][lane] = M.tab[d][(int64_t)ed[d] * TAB_STRIDE + lane];
}
// owned control point of local point b
__device__ __forceinline__ int64_t wave_point(const MeshK &M, const int *ed, int b)
{
    return ((int64_t)M.nb[1] * M.nb[2]) * own1(ed[0] + b / 9, M.nb[0], M.periodic[0])
         + (int64_t)M.nb[2] * own1(ed[1] + (b / 3) % 3, M.nb[1], M.periodic[1]) + own1(ed[2] + b % 3, M.nb[2], M.periodic[2]);
}

__global__ __launch_bounds__(64, 3) void k_residual_sep(MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof,
                                                        double *__restrict__ Re, int nel)
{
    __shared__ double sT[3][TAB_STRIDE], sU[27 * 3], sA[108], sB[288], sR[640];
    const int lane = threadIdx.x, e = blockIdx.x;
    const int nz = M.nelem[2], ny = M.nelem[1];
    const int ed[3] = {e / (ny * nz), (e / nz) % ny, e % nz};
    wave_tables(M, ed, sT, lane);
    if (lane < 27) {
        const int64_t oc = wave_point(M, ed, lane);
#pragma unroll
        for (int k = 0; k < 3; k++) sU[3 * lane + k] = Uh[3 * oc + k];
    }
    wave_sync();
    double u[30], r[30], out[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        wave_field<3>(sT, sU + k, sA, sB, lane, u + 10 * k);
        sep_macro(M, ed, lane, k, u + 10 * k);
    }
    phys_residual_static(P, u, r);
    const double w = sT[0][36 + (lane >> 4)] * sT[1][36 + ((lane >> 2) & 3)] * sT[2][36 + (lane & 3)];
#pragma unroll
    for (int k = 0; k < 3; k++) out[k] = wave_project(sT, r + 10 * k, w, sR, sA, sB, lane);
    if (lane < 27) {
#pragma unroll
        for (int k = 0; k < 3; k++) Re[(int64_t)e * 81 + 3 * lane + k] = out[k];
    }
}

// Transient residual on a separable patch (k_residual_sep_t, gradelasttime), a
// wave per element like the static one: the jets of Um and Ud of a lane's point,
// the rule's eight nodes Um + s_j Ud one after another, weighted by cr_j, all in
// its registers, then the projection.  The value slot's inertia r[10 k] = cii (u - u^2) / (2 dt)
// + rho (u + u^2 - 2 u^1) / dt^2 is linear in the nodal values, so its part of
// R_e is the element mass matrix Mx x My x Mz applied to the nodal
// combination (k_tangent_sep_t's 1-D mass matrices).
// At 128x32x32 2.70 -> 1.37 ms, against a workgroup of four waves per element with a lane
// per node and point, the node sums as lane moves and seven block barriers.  Ud's jets
// wait in LDS: 20 KB an element, eight elements in flight per CU, as many as the registers allow.
__global__ __launch_bounds__(64, 2) void k_residual_sep_t(MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof,
                                                          double *__restrict__ Re, int nel)
{
    __shared__ double sT[3][TAB_STRIDE], sC[27 * 6], sV[27 * 3], sMass[3][3][3], sA[108], sB[288];
    __shared__ double sJ[27 * 64];   // the points' jets of Ud [slot][q], then wave_project's buffer
    const int lane = threadIdx.x, e = blockIdx.x;
    const int nz = M.nelem[2], ny = M.nelem[1];
    const int ed[3] = {e / (ny * nz), (e / nz) % ny, e % nz};
    wave_tables(M, ed, sT, lane);
    if (lane < 27) {
        const int64_t oc = wave_point(M, ed, lane);
        const double cv1 = P.cii / (2. * P.dt), cv2 = P.rho / (P.dt * P.dt);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double u0 = Uh[3 * oc + k], u1 = Uh[ndof + 3 * oc + k], u2 = Uh[2 * ndof + 3 * oc + k];
            sC[6 * lane + k] = 0.5 * (u1 + u2);
            sC[6 * lane + 3 + k] = 0.5 * (u0 - u2);
            sV[3 * lane + k] = cv1 * (u0 - u2) + cv2 * (u0 + u2 - 2 * u1);
        }
    }
    wave_sync();
    if (lane < 27) {
        const int d = lane / 9, b = (lane / 3) % 3, c = lane % 3;
        double m = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) m += sT[d][36 + q] * sT[d][9 * q + b] * sT[d][9 * q + c];
        sMass[d][b][c] = m;
    }
    double r[30], out[3];
    {
        double J1[30];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            double J2[10];
            wave_field<6>(sT, sC + 3 + k, sA, sB, lane, J2);
#pragma unroll
            for (int a = 1; a < 10; a++) sJ[64 * (9 * k + a - 1) + lane] = J2[a];
            wave_field<6>(sT, sC + k, sA, sB, lane, J1 + 10 * k);
            sep_macro(M, ed, lane, k, J1 + 10 * k);
        }
#pragma unroll
        for (int a = 0; a < 30; a++) r[a] = 0.0;
#pragma unroll 1
        for (int j = 0; j < 8; j++) {
            double us[30];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                us[10 * k] = 0.0;
#pragma unroll
                for (int a = 1; a < 10; a++) us[10 * k + a] = J1[10 * k + a] + P.s[j] * sJ[64 * (9 * k + a - 1) + lane];
            }
            State st;
            phys_state(us, P, st);
            phys_residual_acc(st, P.cr[j], r);
        }
    }
    wave_sync();
    const double w = sT[0][36 + (lane >> 4)] * sT[1][36 + ((lane >> 2) & 3)] * sT[2][36 + (lane & 3)];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r[10 * k] = 0.0;   // value slot: the inertia, added below
        out[k] = wave_project(sT, r + 10 * k, w, sJ, sA, sB, lane);
    }
    if (lane < 27) {
        const int bx = lane / 9, by = (lane / 3) % 3, bz = lane % 3;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            double in = 0.0;
#pragma unroll
            for (int cx = 0; cx < 3; cx++)
#pragma unroll
                for (int cy = 0; cy < 3; cy++) {
                    const double mxy = sMass[0][bx][cx] * sMass[1][by][cy];
#pragma unroll
                    for (int cz = 0; cz < 3; cz++) in += mxy * sMass[2][bz][cz] * sV[3 * (9 * cx + 3 * cy + cz) + k];
                }
            Re[(int64_t)e * 81 + 3 * lane + k] = out[k] + in;
        }
    }
}

// Residual of any geometry (k_residual_gen), a wave per element: NH = 1 static, 3
// transient; RAT: unequal weights.  The basis is a tensor product of the
// parametric tables (k_sep_tables; a common factor of the 1-D functions cancels in the
// rational basis), so the coordinates' and displacements' parametric jets come
// from wave_field, with RAT those of w, w X and w U followed by the quotient rule;
// the chain rule gives the physical jets, and the weighted residual jet goes back
// through the transposes of both rules (phys_jet_adj, nurbs_param_adj) into
// wave_project:
//   R_e[b][k] = w_b sum_q (Q_q^T Phi_q^T w_q r_q[k]) . N_b(q).
// Bound by the traffic of its spilled registers (70 static, 134 rational, 118 and 141
// transient, at 256 registers): at 256x64x64 33 GB in 8.0 ms, 4.2 TB/s, for 0.7 GB of
// element vectors, and a wave waits 50 to 67% of its life.
// 64x16x16 distorted beam 282 -> 148 us, 45x23x17 rational 303 -> 248 us, whole
// residual calls at 23x9x14: static 77 -> 39 us (rational 56), transient 155 ->
// 84 us (89), against a workgroup of four waves per element and eight block barriers.
template <int NH, bool RAT>
__global__ __launch_bounds__(64, 2) void k_residual_gen(MeshK M, PhysK P, const double *__restrict__ Uh, int64_t ndof,
                                                        double *__restrict__ Re, int nel)
{
    // nodal fields X (3), U (3) or Um, Ud and the inertia combination (9), w
    constexpr int STR = NH == 1 ? 7 : 13;
    __shared__ double sT[3][TAB_STRIDE], sC[27 * STR], sA[108], sB[288];
    __shared__ double sJ[NH == 1 ? 640 : 27 * 64];   // the points' jets of Ud [slot][q], then wave_project's buffer
    const int lane = threadIdx.x, e = blockIdx.x;
    const int nz = M.nelem[2], ny = M.nelem[1];
    const int ed[3] = {e / (ny * nz), (e / nz) % ny, e % nz};
    wave_tables(M, ed, sT, lane);
    if (lane < 27) {
        const int64_t id = ((int64_t)M.na[1] * M.na[2]) * (ed[0] + lane / 9) + (int64_t)M.na[2] * (ed[1] + (lane / 3) % 3) + ed[2] + lane % 3;
        const int64_t oc = wave_point(M, ed, lane);
        // coordinates relative to the element's middle point: the jets' derivatives
        // are the same, and their rounding errors scale with the element's size
        const int64_t mid = ((int64_t)M.na[1] * M.na[2]) * (ed[0] + 1) + (int64_t)M.na[2] * (ed[1] + 1) + ed[2] + 1;
        const double wb = RAT ? M.w[id] : 1.0;
        double *c = sC + STR * lane;
        c[STR - 1] = wb;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            c[k] = wb * (M.X[3 * id + k] - M.X[3 * mid + k]);
            const double u0 = Uh[3 * oc + k];
            if (NH == 1) {
                c[3 + k] = wb * u0;
            } else {
                const double u1 = Uh[ndof + 3 * oc + k], u2 = Uh[2 * ndof + 3 * oc + k];
                c[3 + k] = wb * (0.5 * (u1 + u2));
                c[(NH == 1 ? 0 : 6) + k] = wb * (0.5 * (u0 - u2));
                c[(NH == 1 ? 0 : 9) + k] = wb * (P.cii * (u0 - u2) / (2. * P.dt) + P.rho * (u0 + u2 - 2 * u1) / (P.dt * P.dt));
            }
        }
    }
    wave_sync();
    double W[10], Gi[9], X2[18], r[30], out[3];
    if (RAT) wave_field<STR>(sT, sC + STR - 1, sA, sB, lane, W);
    auto field = [&](int f, double *J) {
        wave_field<STR>(sT, sC + f, sA, sB, lane, J);
        if (RAT) {
            double N[10];
#pragma unroll
            for (int a = 0; a < 10; a++) N[a] = J[a];
            nurbs_param(N, 1.0, W, J);
        }
    };
    double w = sT[0][36 + (lane >> 4)] * sT[1][36 + ((lane >> 2) & 3)] * sT[2][36 + (lane & 3)];
    {
        double G[9];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double J[10];
            field(d, J);
#pragma unroll
            for (int i = 0; i < 3; i++) G[3 * d + i] = J[1 + i];
#pragma unroll
            for (int t = 0; t < 6; t++) X2[6 * d + t] = J[4 + t];
        }
        w *= inv3(G, Gi);
    }
    {
        double u[30], inert[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (NH != 1) {
                double J[10];
                field(9 + k, J);
                inert[k] = J[0];
                field(6 + k, J);
                phys_jet(J, Gi, X2);
#pragma unroll
                for (int a = 1; a < 10; a++) sJ[64 * (9 * k + a - 1) + lane] = J[a];
            }
            field(3 + k, u + 10 * k);
            phys_jet(u + 10 * k, Gi, X2);
            sep_macro(M, ed, lane, k, u + 10 * k);
        }
        if (NH == 1) {
            phys_residual_static(P, u, r);
        } else {
#pragma unroll
            for (int a = 0; a < 30; a++) r[a] = 0.0;
#pragma unroll 1
            for (int j = 0; j < 8; j++) {
                double us[30];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    us[10 * k] = 0.0;
#pragma unroll
                    for (int a = 1; a < 10; a++) us[10 * k + a] = u[10 * k + a] + P.s[j] * sJ[64 * (9 * k + a - 1) + lane];
                }
                State st;
                phys_state(us, P, st);
                phys_residual_acc(st, P.cr[j], r);
            }
#pragma unroll
            for (int k = 0; k < 3; k++) r[10 * k] = inert[k];
        }
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < 3; k++) {
        double *o = r + 10 * k;
#pragma unroll
        for (int a = 0; a < 10; a++) o[a] *= w;
        phys_jet_adj(o, Gi, X2);
        if (RAT) nurbs_param_adj(o, W);
        out[k] = wave_project(sT, o, 1.0, sJ, sA, sB, lane);
    }
    if (lane < 27) {
#pragma unroll
        for (int k = 0; k < 3; k++) Re[(int64_t)e * 81 + 3 * lane + k] = RAT ? sC[STR * lane + STR - 1] * out[k] : out[k];
    }
}

// the unit diagonal MatZeroRowsColumns(diag = 1) leaves on the Dirichlet rows
// of a non-periodic patch (their other entries stayed zero)
template <typename TV>
__global__ __launch_bounds__(256) void k_dirichlet_diag(MeshK M, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ mask,
                                                        TV *__restrict__ vals, int64_t ncp)
{
    const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= ncp) return;
    const int nb1 = M.nb[1], nb2 = M.nb[2];
    const int az = (int)(a % nb2), ay = (int)((a / nb2) % nb1), ax = (int)(a / ((int64_t)nb1 * nb2));
#pragma unroll
    for (int i = 0; i < 3; i++)
        if (mask[3 * a + i]) vals[csr_pos(M, rowptr, ax, ay, az, i, ax, ay, az, i)] = (TV)1.0;
}

// sorted owned control points within +-2 of a (clipped, or wrapped when periodic)
__device__ __forceinline__ int stencil1(int a, int n, int periodic, int *S)
{
    int cnt = 0;
    if (!periodic) {
        int lo = a - 2 < 0 ? 0 : a - 2, hi = a + 2 > n - 1 ? n - 1 : a + 2;
        for (int b = lo; b <= hi; b++) S[cnt++] = b;
        return cnt;
    }
    int tmp[5];
    for (int t = 0; t < 5; t++) { int v = a + t - 2; v = (v % n + n) % n; tmp[t] = v; }
    for (int i = 1; i < 5; i++)
        for (int j = i; j > 0 && tmp[j] < tmp[j - 1]; j--) { int x = tmp[j]; tmp[j] = tmp[j - 1]; tmp[j - 1] = x; }
    for (int t = 0; t < 5; t++)
        if (cnt == 0 || tmp[t] != S[cnt - 1]) S[cnt++] = tmp[t];
    return cnt;
}

// acc += v in LDS without a round trip; a wave's additions happen in program order
__device__ __forceinline__ void lds_add(double *p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the same set in closed form: point k of it and the place of point b in it
// (wrapped, the points from 0 on come first; a periodic direction has at least five)
struct Stencil {
    int lo, f, n5, cnt;
    __device__ __forceinline__ Stencil(int a, int n, int periodic)
    {
        const bool wrap = periodic && (a < 2 || a + 2 > n - 1);
        const int l = a - 2 > 0 ? a - 2 : 0, h = a + 2 < n - 1 ? a + 2 : n - 1;
        cnt = periodic ? 5 : h - l + 1;
        lo = l;
        f = wrap ? (a + 3 >= n ? a + 3 - n : a + 3) : 0;
        n5 = wrap ? n - 5 : l;
    }
    __device__ __forceinline__ int at(int k) const { return k < f ? k : n5 + k; }
    __device__ __forceinline__ int slot(int b) const { return b < f ? b : b - n5; }
};

// Sum of the element matrices into the CSR rows of control point a, one wave per
// row: the row's entries are summed in LDS, element by element in ascending
// order, by one wave in program order, so nothing waits at a barrier and the sum
// of every entry has a fixed order.  A row has 81 columns per element: 64 are one
// load of the wave, the other 17 of the (up to) three elements along z another, 36 loads
// in flight.  The Dirichlet rows and columns of MatZeroRowsColumns (unit diagonal)
// go in with the write-out.  Ucopy (may be null): where the iterate U is kept.
// Bound by the element matrices' bytes: 256x64x64 FP64 14.4 -> 13.2 ms (65 GB, 4.9
// TB/s), 160x40x40 FP32 3.2 -> 2.0 ms, 16x4x4 (its latency) 17.5 -> 11.4 us, against
// four waves over the three rows with a barrier per element (FP64) and a thread per
// pair of points (FP32).
template <typename TK, typename TV>
__global__ __launch_bounds__(192) void k_tangent_gather_rows(MeshK M, const TK *__restrict__ Ke, const int64_t *__restrict__ rowptr,
                                                             const int32_t *__restrict__ mask, TV *__restrict__ vals, const double *U,
                                                             double *Ucopy)
{
    __shared__ double sAcc[3][376];
    // control-point and dof indices fit in 32 bits (the CSR columns are int32)
    const int a = (int)blockIdx.x, i = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    double *acc = sAcc[i];
    const int row = 3 * a + i;
    if (Ucopy && lane == 0) Ucopy[row] = U[row];
    const int nb1 = M.nb[1], nb2 = M.nb[2];
    const int axy = a / nb2, az = a - axy * nb2, ax = axy / nb1, ay = axy - ax * nb1;
    const Stencil Sx(ax, M.nb[0], M.periodic[0]), Sy(ay, M.nb[1], M.periodic[1]), Sz(az, M.nb[2], M.periodic[2]);
    const ElemRow X(ax, M.nelem[0], M.periodic[0]), Y(ay, M.nelem[1], M.periodic[1]), Z(az, M.nelem[2], M.periodic[2]);
    const int nsz = Sz.cnt, nsyz = Sy.cnt * nsz, n = 3 * Sx.cnt * nsyz;
    // columns c of an element row: c = lane, and 64 + u of element z = h along z
    const int h = lane / 17, u = lane - 17 * h, c2 = 64 + u, z2 = h < 3 ? h : 0;
    TK v[27], w[9];
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3; y++) {
            const int64_t exy = ((int64_t)X.e[x] * M.nelem[1] + Y.e[y]) * M.nelem[2];
            const int lxy = 27 * X.l[x] + 9 * Y.l[y];
#pragma unroll
            for (int z = 0; z < 3; z++) {
                const bool ok = X.ok[x] && Y.ok[y] && Z.ok[z];
                v[9 * x + 3 * y + z] = Ke[ok ? (exy + Z.e[z]) * 6561 + (lxy + 3 * Z.l[z] + i) * 81 + lane : 0];
            }
            const int ez = z2 == 0 ? Z.e[0] : z2 == 1 ? Z.e[1] : Z.e[2], lz = z2 == 0 ? Z.l[0] : z2 == 1 ? Z.l[1] : Z.l[2];
            const bool okz = z2 == 0 ? Z.ok[0] : z2 == 1 ? Z.ok[1] : Z.ok[2];
            w[3 * x + y] = Ke[X.ok[x] && Y.ok[y] && okz ? (exy + ez) * 6561 + (lxy + 3 * lz + i) * 81 + c2 : 0];
        }
    // the write-out's Dirichlet flags and row start
    bool dead[6];
    int col[6];
    const bool drow = mask[row] != 0;
    const int64_t start = rowptr[row];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int r = lane + 64 * k, t = r / 3, j = r - 3 * t, sx = t / nsyz, q = t - sx * nsyz, sy = q / nsz, sz = q - sy * nsz;
        col[k] = r < n ? 3 * ((Sx.at(sx) * nb1 + Sy.at(sy)) * nb2 + Sz.at(sz)) + j : 0;
        dead[k] = drow || mask[col[k]] != 0;
        if (r < n) acc[r] = 0.0;
    }
    // places of the two columns' points: 3 (slot along x) ns_y ns_z + 3 (slot along y) ns_z + 3 (slot along z) + component
    int px[3], py[3], pz[3], qx[3], qy[3], qz;
    {
        const int lb = lane / 3, j = lane - 3 * lb, lb2 = c2 / 3, j2 = c2 - 3 * lb2;
#pragma unroll
        for (int e = 0; e < 3; e++) {
            px[e] = 3 * nsyz * Sx.slot(own1(X.e[e] + lb / 9, M.nb[0], M.periodic[0]));
            py[e] = 3 * nsz * Sy.slot(own1(Y.e[e] + (lb / 3) % 3, M.nb[1], M.periodic[1]));
            pz[e] = 3 * Sz.slot(own1(Z.e[e] + lb % 3, M.nb[2], M.periodic[2])) + j;
            qx[e] = 3 * nsyz * Sx.slot(own1(X.e[e] + lb2 / 9, M.nb[0], M.periodic[0]));
            qy[e] = 3 * nsz * Sy.slot(own1(Y.e[e] + (lb2 / 3) % 3, M.nb[1], M.periodic[1]));
        }
        const int ez = z2 == 0 ? Z.e[0] : z2 == 1 ? Z.e[1] : Z.e[2];
        qz = 3 * Sz.slot(own1(ez + lb2 % 3, M.nb[2], M.periodic[2])) + j2;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3; y++)
#pragma unroll
            for (int z = 0; z < 3; z++)
                if (X.ok[x] && Y.ok[y] && Z.ok[z]) {
                    lds_add(acc + px[x] + py[y] + pz[z], (double)v[9 * x + 3 * y + z]);
                    if (h == z) lds_add(acc + qx[x] + qy[y] + qz, (double)w[3 * x + y]);
                }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int r = lane + 64 * k;
        if (r < n) vals[start + r] = (TV)(dead[k] ? (row == col[k] ? 1.0 : 0.0) : acc[r]);
    }
}

__global__ __launch_bounds__(128) void k_csr_cols(MeshK M, const int64_t *__restrict__ rowptr, int32_t *__restrict__ col)
{
    const int64_t a = blockIdx.x;
    int nb1 = M.nb[1], nb2 = M.nb[2];
    int az = (int)(a % nb2), ay = (int)((a / nb2) % nb1), ax = (int)(a / ((int64_t)nb1 * nb2));
    int Sx[5], Sy[5], Sz[5];
    int nsx = stencil1(ax, M.nb[0], M.periodic[0], Sx);
    int nsy = stencil1(ay, M.nb[1], M.periodic[1], Sy);
    int nsz = stencil1(az, M.nb[2], M.periodic[2], Sz);
    int t = threadIdx.x;
    if (t >= nsx * nsy * nsz) return;
    int sx = t / (nsy * nsz), sy = (t / nsz) % nsy, sz = t % nsz;
    int64_t bcp = ((int64_t)M.nb[1] * M.nb[2]) * Sx[sx] + (int64_t)M.nb[2] * Sy[sy] + Sz[sz];
    for (int i = 0; i < 3; i++) {
        int64_t pos = rowptr[3 * a + i] + 3 * t;
        for (int j = 0; j < 3; j++) col[pos + j] = (int32_t)(3 * bcp + j);
    }
}

template <typename T>
__global__ void k_fill(T *p, T v, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += st) p[i] = v;
}

__global__ void k_copy(double *dst, const double *src, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += st) dst[i] = src[i];
}

__global__ void k_selftest_mfma(double *o64, float *o32)
{
    int l = threadIdx.x;
    int i = l & 15, k = l >> 4;
    // A[i][k] = 1 + i + 0.25 k ; B[k][j] = 2 - 0.5 j + k
    double a = 1.0 + i + 0.25 * k;
    double b = 2.0 - 0.5 * i + k;   // lane holds B[k = l>>4][j = l&15]
    double4_t d = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, (double4_t){0, 0, 0, 0}, 0, 0, 0);
    float4_t f = __builtin_amdgcn_mfma_f32_16x16x4f32((float)a, (float)b, (float4_t){0, 0, 0, 0}, 0, 0, 0);
    // raw result registers: out[(r*64 + lane)]
    for (int r = 0; r < 4; r++) {
        o64[r * 64 + l] = d[r];
        o32[r * 64 + l] = f[r];
    }
}

// ============================================================================
// Pointwise physics at given jets: the device counterpart of the Phys
// callbacks residual / tangent / density (include/physimpl.h:6-9; gradelast,
// phys/gradelast.c; gradelasttime, phys/gradelasttime.c), through the same
// device functions the assembly kernels use (phys_state, phys_residual_acc,
// c_row, c_row_mom, phys_density_*).  Jet layout of one point:
// u[30 h + 10 k + a] with h = 0 the current level, 1 the previous and 2 the
// one before (the reference's u, u1 = u + 30, u0 = u + 60).  Thread t
// evaluates row (k, a) = t % 30 of point t / 30: r[30 p + row],
// C[900 p + 30 row + 10 l + b] and, on row 0, the densities hh[nd p + i].
// ============================================================================
// the moment state of the transient tangent (c_row_mom) for the jets
// Um = (u1 + u0)/2 and Ud = (u - u0)/2, summed over the rule nodes in order
__device__ void moment_state_seq(const double *Um, const double *Ud, const PhysK &P, const Mom &mu, double *ms)
{
    double S[9], G[9], n0[9], n1[9], n2[9];
    for (int i = 0; i < 9; i++) S[i] = G[i] = n0[i] = n1[i] = n2[i] = 0.0;
    for (int j = 0; j < P.nnode; j++) {
        double us[30];
        for (int i = 0; i < 30; i++) us[i] = Um[i] + P.s[j] * Ud[i];
        State st;
        phys_state(us, P, st);
        const double w0 = P.ct[j], w1 = w0 * P.s[j], w2 = w1 * P.s[j];
        for (int i = 0; i < 9; i++) {
            S[i] += w0 * st.S[i];
            G[i] += w0 * st.G[i];
            n0[i] += w0 * st.N[i];
            n1[i] += w1 * st.N[i];
            n2[i] += w2 * st.N[i];
        }
    }
    const double c12 = 1.0 / (mu.a11 * mu.a22), c22 = 1.0 / mu.d2;
    for (int i = 0; i < 9; i++) {
        ms[MS + i] = S[i];
        ms[MG + i] = G[i];
        ms[MN11 + i] = n0[i] / mu.m0;
        ms[MN12 + i] = (n1[i] - mu.lf * n0[i]) * c12;
        ms[MN22 + i] = ((mu.lf * n0[i] - n1[i]) * mu.lf + (n2[i] - mu.lf * n1[i])) * c22;
    }
    for (int i = 0; i < 36; i++) {
        const bool isF = i < 9;
        const int r = isF ? i : i - 9;
        const int slot = isF ? 10 * (r / 3) + 1 + (r % 3) : 10 * (r / 9) + sidx((r % 9) / 3, r % 3);
        double x0 = Um[slot];
        const double xd = Ud[slot];
        if (isF && (r / 3) == (r % 3)) x0 += 1.0;
        const double x1 = mu.a11 * (x0 + mu.lf * xd), x2 = mu.a22 * xd;
        if (isF) { ms[MF1 + r] = x1; ms[MF2 + r] = x2; }
        else { ms[MH1 + r] = x1; ms[MH2 + r] = x2; }
    }
}

template <int NH>
__global__ __launch_bounds__(128) void k_phys_eval(PhysK P, int64_t npts, const double *__restrict__ u, double *__restrict__ r,
                                                  double *__restrict__ C, double *__restrict__ hh)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= npts * 30) return;
    const int64_t p = t / 30;
    const int row = (int)(t - 30 * p), k = row / 10, a = row % 10;
    const double *J = u + p * 30 * NH;
    if (r) {
        double rr[30];
        if (NH == 1) {
            phys_residual_static(P, J, rr);
        } else {
            for (int i = 0; i < 30; i++) rr[i] = 0.0;
            for (int g = 0; g < P.nnode; g++) {
                double us[30];
                for (int i = 0; i < 30; i++) us[i] = 0.5 * (J[30 + i] + J[60 + i]) + P.s[g] * (0.5 * (J[i] - J[60 + i]));
                State st;
                phys_state(us, P, st);
                phys_residual_acc(st, P.cr[g], rr);
            }
            for (int kk = 0; kk < 3; kk++)
                rr[10 * kk] = (P.cii * (J[10 * kk] - J[60 + 10 * kk])) / (2. * P.dt)
                            + (P.rho * (J[10 * kk] + J[60 + 10 * kk] - 2 * J[30 + 10 * kk])) / (P.dt * P.dt);
        }
        r[p * 30 + row] = rr[row];
    }
    if (C) {
        double out[30];
        for (int i = 0; i < 30; i++) out[i] = 0.0;
        if (NH == 1) {
            State st;
            phys_state(J, P, st);
            double sp[STW];
            for (int i = 0; i < 9; i++) sp[ST_F + i] = st.F[i];
            for (int i = 0; i < 27; i++) sp[ST_H + i] = st.H[i];
            for (int i = 0; i < 9; i++) { sp[ST_S + i] = st.S[i]; sp[ST_G + i] = st.G[i]; sp[ST_N + i] = st.N[i]; }
            for (int l = 0; l < 3; l++) c_row<0>(sp, P, k, a, l, 1.0, out + 10 * l);
        } else {
            Mom mu = {0.0, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0};
            for (int j = 0; j < P.nnode; j++) {
                mu.m0 += P.ct[j];
                mu.m1 += P.ct[j] * P.s[j];
                mu.m2 += P.ct[j] * P.s[j] * P.s[j];
            }
            mu.factor();
            double Um[30], Ud[30], ms[MW];
            for (int i = 0; i < 30; i++) {
                Um[i] = 0.5 * (J[30 + i] + J[60 + i]);
                Ud[i] = 0.5 * (J[i] - J[60 + i]);
            }
            moment_state_seq(Um, Ud, P, mu, ms);
            for (int l = 0; l < 3; l++) c_row_mom<0>(ms, P, k, a, l, out + 10 * l);
            if (a == 0) out[10 * k] += P.cii / (2. * P.dt) + P.rho / (P.dt * P.dt);
        }
        for (int i = 0; i < 30; i++) C[p * 900 + 30 * row + i] = out[i];
    }
    if (hh && row == 0) {
        if (NH == 1) {
            double h[ND_STATIC];
            phys_density_static(J, P, h);
            for (int i = 0; i < ND_STATIC; i++) hh[p * ND_STATIC + i] = h[i];
        } else {
            double h[ND_TRANSIENT];
            phys_density_transient(J, P, h);
            for (int i = 0; i < ND_TRANSIENT; i++) hh[p * ND_TRANSIENT + i] = h[i];
        }
    }
}

// ============================================================================
// launchers (host, C++ linkage; called by the C ABI in igap_capi.cpp)
// ============================================================================
}  // namespace igap

#include "igap_launch.h"

namespace igap {

hipError_t launch_density(const MeshK &M, const PhysK &P, const double *Uh, int64_t ndof, double *Hd, double *H, int nel,
                          hipStream_t s)
{
    dim3 grid(nel), block(256);
    if (P.torder == 0) hipLaunchKernelGGL(k_density_elem<1>, grid, block, 0, s, M, P, Uh, ndof, Hd, nel);
    else hipLaunchKernelGGL(k_density_elem<3>, grid, block, 0, s, M, P, Uh, ndof, Hd, nel);
    const int nd = P.torder == 0 ? ND_STATIC : ND_TRANSIENT;
    hipLaunchKernelGGL(k_density_reduce, dim3(nd), dim3(256), 0, s, nel, nd, Hd, H);
    return hipGetLastError();
}

hipError_t launch_residual_elem(const MeshK &M, const PhysK &P, const double *Uh, int64_t ndof, double *Re, int nel, hipStream_t s)
{
    dim3 grid(nel);
    if (P.torder == 0 && M.separable) hipLaunchKernelGGL(k_residual_sep, grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    else if (P.torder == 2 && M.separable) hipLaunchKernelGGL(k_residual_sep_t, grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    else if (P.torder == 0 && M.equalw) hipLaunchKernelGGL((k_residual_gen<1, false>), grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    else if (P.torder == 0) hipLaunchKernelGGL((k_residual_gen<1, true>), grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    else if (M.equalw) hipLaunchKernelGGL((k_residual_gen<3, false>), grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    else hipLaunchKernelGGL((k_residual_gen<3, true>), grid, dim3(64), 0, s, M, P, Uh, ndof, Re, nel);
    return hipGetLastError();
}

hipError_t launch_residual_gather(const MeshK &M, const double *Re, const double *U, double *Ucopy, const double *Fneu,
                                  const int32_t *mask, const double *g, double *R, int64_t ncp, hipStream_t s)
{
    dim3 grid((unsigned)((3 * ncp + 255) / 256)), block(256);
    hipLaunchKernelGGL(k_residual_gather, grid, block, 0, s, M, Re, U, Ucopy, Fneu, mask, g, R, ncp);
    return hipGetLastError();
}

hipError_t launch_tangent_elem(const MeshK &M, const PhysK &P, const double *Uh, int64_t ndof, void *Ke, int prec, int nel,
                               hipStream_t s)
{
    dim3 grid(nel), block(256);
    const Scatter S{};
    if (P.torder == 0 && M.separable) {
        if (prec == 0) hipLaunchKernelGGL((k_tangent_sep<double, false>), grid, dim3(SepShape<double, 1>::THREADS), 0, s, M, P, Uh, (double *)Ke, S, M.tab[0], M.tab[1], M.tab[2]);
        else hipLaunchKernelGGL((k_tangent_sep<float, false>), grid, dim3(SepShape<float, 1>::THREADS), 0, s, M, P, Uh, (float *)Ke, S, M.tabf[0], M.tabf[1], M.tabf[2]);
        return hipGetLastError();
    }
    if (P.torder == 2 && M.separable) {
        if (prec == 0) hipLaunchKernelGGL((k_tangent_sep_t<double, false>), grid, dim3(SepShape<double, 3>::THREADS), 0, s, M, P, Uh, ndof, (double *)Ke, S, M.tab[0], M.tab[1], M.tab[2]);
        else hipLaunchKernelGGL((k_tangent_sep_t<float, false>), grid, dim3(SepShape<float, 3>::THREADS), 0, s, M, P, Uh, ndof, (float *)Ke, S, M.tabf[0], M.tabf[1], M.tabf[2]);
        return hipGetLastError();
    }
    if (P.torder == 0 && M.equalw) {
        if (prec == 0) hipLaunchKernelGGL((k_tangent_gen<double, false>), grid, dim3(512), 0, s, M, P, Uh, (double *)Ke, S, M.tab[0], M.tab[1], M.tab[2]);
        else hipLaunchKernelGGL((k_tangent_gen<float, false>), grid, dim3(512), 0, s, M, P, Uh, (float *)Ke, S, M.tabf[0], M.tabf[1], M.tabf[2]);
        return hipGetLastError();
    }
    if (prec == 0) {
        if (P.torder == 0) hipLaunchKernelGGL((k_tangent_elem<double, 1, false>), grid, block, 0, s, M, P, Uh, ndof, (double *)Ke, nel, S);
        else hipLaunchKernelGGL((k_tangent_elem<double, 3, false>), grid, block, 0, s, M, P, Uh, ndof, (double *)Ke, nel, S);
    } else {
        if (P.torder == 0) hipLaunchKernelGGL((k_tangent_elem<float, 1, false>), grid, block, 0, s, M, P, Uh, ndof, (float *)Ke, nel, S);
        else hipLaunchKernelGGL((k_tangent_elem<float, 3, false>), grid, block, 0, s, M, P, Uh, ndof, (float *)Ke, nel, S);
    }
    return hipGetLastError();
}

// Tangent straight into the CSR values of a non-periodic patch: zero the
// values, one element launch per colour (colours in a fixed order, so every
// entry sums its contributions in the same order on every call), then the
// Dirichlet diagonal.
hipError_t launch_tangent_direct(const MeshK &M, const PhysK &P, const double *Uh, int64_t ndof, const int64_t *rowptr,
                                 const int32_t *mask, void *vals, int prec, int64_t nnz, int64_t ncp, hipStream_t s)
{
    for (int d = 0; d < 3; d++)
        if (M.periodic[d]) return hipErrorInvalidValue;
    const int64_t fb = std::min<int64_t>((nnz + 255) / 256, 65536);
    if (prec == 0) hipLaunchKernelGGL(k_fill<double>, dim3((unsigned)fb), dim3(256), 0, s, (double *)vals, 0.0, nnz);
    else hipLaunchKernelGGL(k_fill<float>, dim3((unsigned)fb), dim3(256), 0, s, (float *)vals, 0.0f, nnz);
    for (int cx = 0; cx < 3; cx++)
        for (int cy = 0; cy < 3; cy++)
            for (int cz = 0; cz < 3; cz++) {
                Scatter S;
                S.rowptr = rowptr;
                S.mask = mask;
                S.c[0] = cx; S.c[1] = cy; S.c[2] = cz;
                for (int d = 0; d < 3; d++) S.nc[d] = (M.nelem[d] - S.c[d] + 2) / 3;
                const int64_t n = (int64_t)S.nc[0] * S.nc[1] * S.nc[2];
                if (n <= 0) continue;
                dim3 grid((unsigned)n), block(256);
                if (P.torder == 0 && M.separable) {
                    if (prec == 0) hipLaunchKernelGGL((k_tangent_sep<double, true>), grid, dim3(SepShape<double, 1>::THREADS), 0, s, M, P, Uh, (double *)vals, S, M.tab[0], M.tab[1], M.tab[2]);
                    else hipLaunchKernelGGL((k_tangent_sep<float, true>), grid, dim3(SepShape<float, 1>::THREADS), 0, s, M, P, Uh, (float *)vals, S, M.tabf[0], M.tabf[1], M.tabf[2]);
                } else if (P.torder == 2 && M.separable) {
                    if (prec == 0) hipLaunchKernelGGL((k_tangent_sep_t<double, true>), grid, dim3(SepShape<double, 3>::THREADS), 0, s, M, P, Uh, ndof, (double *)vals, S, M.tab[0], M.tab[1], M.tab[2]);
                    else hipLaunchKernelGGL((k_tangent_sep_t<float, true>), grid, dim3(SepShape<float, 3>::THREADS), 0, s, M, P, Uh, ndof, (float *)vals, S, M.tabf[0], M.tabf[1], M.tabf[2]);
                } else if (P.torder == 0 && M.equalw) {
                    if (prec == 0) hipLaunchKernelGGL((k_tangent_gen<double, true>), grid, dim3(512), 0, s, M, P, Uh, (double *)vals, S, M.tab[0], M.tab[1], M.tab[2]);
                    else hipLaunchKernelGGL((k_tangent_gen<float, true>), grid, dim3(512), 0, s, M, P, Uh, (float *)vals, S, M.tabf[0], M.tabf[1], M.tabf[2]);
                } else if (prec == 0) {
                    if (P.torder == 0) hipLaunchKernelGGL((k_tangent_elem<double, 1, true>), grid, block, 0, s, M, P, Uh, ndof, (double *)vals, (int)n, S);
                    else hipLaunchKernelGGL((k_tangent_elem<double, 3, true>), grid, block, 0, s, M, P, Uh, ndof, (double *)vals, (int)n, S);
                } else {
                    if (P.torder == 0) hipLaunchKernelGGL((k_tangent_elem<float, 1, true>), grid, block, 0, s, M, P, Uh, ndof, (float *)vals, (int)n, S);
                    else hipLaunchKernelGGL((k_tangent_elem<float, 3, true>), grid, block, 0, s, M, P, Uh, ndof, (float *)vals, (int)n, S);
                }
            }
    const dim3 g((unsigned)((ncp + 255) / 256)), b(256);
    if (prec == 0) hipLaunchKernelGGL(k_dirichlet_diag<double>, g, b, 0, s, M, rowptr, mask, (double *)vals, ncp);
    else hipLaunchKernelGGL(k_dirichlet_diag<float>, g, b, 0, s, M, rowptr, mask, (float *)vals, ncp);
    return hipGetLastError();
}

hipError_t launch_tangent_gather(const MeshK &M, const void *Ke, int prec, const int64_t *rowptr, const int32_t *mask, void *vals,
                                 int64_t ncp, const double *U, double *Ucopy, hipStream_t s)
{
    dim3 grid((unsigned)ncp), block(192);
    if (prec == 0)
        hipLaunchKernelGGL((k_tangent_gather_rows<double, double>), grid, block, 0, s, M, (const double *)Ke, rowptr, mask, (double *)vals, U, Ucopy);
    else
        hipLaunchKernelGGL((k_tangent_gather_rows<float, float>), grid, block, 0, s, M, (const float *)Ke, rowptr, mask, (float *)vals, U, Ucopy);
    return hipGetLastError();
}

hipError_t launch_csr_cols(const MeshK &M, const int64_t *rowptr, int32_t *col, int64_t ncp, hipStream_t s)
{
    dim3 grid((unsigned)ncp), block(128);
    hipLaunchKernelGGL(k_csr_cols, grid, block, 0, s, M, rowptr, col);
    return hipGetLastError();
}

hipError_t launch_sep_tables(const MeshK &M, double *tab, float *tabf, hipStream_t s)
{
    const int m = std::max(M.nelem[0], std::max(M.nelem[1], M.nelem[2]));
    hipLaunchKernelGGL(k_sep_tables, dim3((unsigned)m, 3), dim3(64), 0, s, M, tab, tabf);
    return hipGetLastError();
}

hipError_t launch_fill_f64(double *p, double v, int64_t n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_fill<double>, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

hipError_t launch_copy_f64(double *dst, const double *src, int64_t n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s, dst, src, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- scratch
// The element vectors of igap_gpu_residual_noalloc live in this file-scope
// device array: the code object carries it, so every GPU the library runs on
// holds its own copy (256 MiB) until the process ends, and using it needs no
// allocation.  Host code must not pass the array's name to a kernel (that is
// a host-side stand-in): scratch_setup looks up each device's address once,
// with that device current, and the kernels take that address.
constexpr int64_t SCRATCH_DOUBLES = (int64_t)32 << 20;   // 81 per element: 414,252 elements
static __device__ __align__(256) double scratch[SCRATCH_DOUBLES];
constexpr int SCRATCH_MAX_DEVICES = 64;
static double *g_scratch_dev[SCRATCH_MAX_DEVICES] = {};
static std::mutex g_scratch_mu;

hipError_t scratch_setup(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (device < 0 || device >= SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
    if (g_scratch_dev[device]) return hipSuccess;
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device) return hipErrorInvalidDevice;   // the caller makes the device current
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_dev[device] = static_cast<double *>(ptr);
    return hipSuccess;
}

double *scratch_device_ptr(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return (device >= 0 && device < SCRATCH_MAX_DEVICES) ? g_scratch_dev[device] : nullptr;
}

int64_t scratch_capacity_doubles() { return SCRATCH_DOUBLES; }

hipError_t launch_phys_eval(const PhysK &P, int64_t npts, const double *u, double *r, double *C, double *hh, hipStream_t s)
{
    if (npts <= 0) return hipSuccess;
    const int64_t nt = 30 * npts;
    dim3 grid((unsigned)((nt + 127) / 128)), block(128);
    if (P.torder == 0) hipLaunchKernelGGL(k_phys_eval<1>, grid, block, 0, s, P, npts, u, r, C, hh);
    else hipLaunchKernelGGL(k_phys_eval<3>, grid, block, 0, s, P, npts, u, r, C, hh);
    return hipGetLastError();
}

hipError_t launch_selftest_mfma(double *o64, float *o32, hipStream_t s)
{
    hipLaunchKernelGGL(k_selftest_mfma, dim3(1), dim3(64), 0, s, o64, o32);
    return hipGetLastError();
}

}  // namespace igap
