// igap_sep_pipeline.h -- the contraction of the element tangents on tensor-product
// tables, as a pipeline of specialised waves (included by igap_kernels.hip).
//
// The element tangent is K^kl[b][c] = sum_q sum_{a,a'} R_q[a][b] D_q[(k,a),(l,a')] R_q[a'][c]
// (Tangent_iga, src/assmcore_iga.c:723-749) with R_q[a][b] = Px Py Pz a product of
// 1-D tables.  With s = (dx, dy) the x-y part of a jet slot and for each of the
// six blocks p = (k, l), k <= l, it factors into
//   D   the 9x9 block of the pointwise tangent             one lane per (point, block)
//   z   E1[(s,bz),(s',cz)] = sum_qz sum Pz[bz] D Pz[cz]    per (qx, qy) pencil of four points
//   y   E2[(dx,by,bz),(dx',cy,cz)] += sum Py Py E1         per pencil
//   x   K += sum Px Px E2                                  after a qx's fourth qy
// Each stage has waves of its own, and the chunks of NP pencils move through
// them one interval apart: D of chunk c + 1 (two buffers in LDS) beside z of
// chunk c and y/x of chunk c - 1.  With two E1 buffers (NE = 2) an interval
// ends with one barrier; with one buffer the z waves keep their results in
// registers until y has read the previous chunk, store them after the barrier,
// and a second barrier follows.
#pragma once

namespace igap {

// x-y part s of the jet slots, s = (dx, dy) in the order (0,0) (1,0) (0,1) (2,0) (1,1) (0,2)
constexpr int PIPE_SX[6] = {0, 1, 0, 2, 1, 0}, PIPE_SY[6] = {0, 0, 1, 0, 1, 2};
// LDS layout.  A D block: nine rows (slots 1..9) of ten columns (AT of d_store): the
// two slots of the x-y parts s' = 0, 1, 2 (orders in z ascending), the single ones
// of s' = 3 and 4, that of s' = 5 and a zero, so that a z lane reads a row's entries
// as one aligned pair.  E1 as [pencil][block][bz][cz][s][s'],
// the 36 values of a y lane contiguous.
constexpr int PIPE_DR = 10, PIPE_DB = 90, PIPE_EC = 36, PIPE_EB = 326;

// The waves of the pipeline: three y waves (wave cy, lanes (block, bz, cz)), one
// for D and four z waves, in this order.  Waves four apart share a SIMD, so that a z
// wave (267 vector instructions per interval in k_tangent_sep<double>) stands beside
// each y wave (the contraction's 180 FMAs and products, every other time 162 more,
// and their addresses) and beside the D wave (317; transient 534, any geometry 1005).
template <int NE_, bool PF_, bool DEEP_>
struct PipeShape {
    static constexpr int NP = 2, NE = NE_;
    static constexpr bool PF = PF_;       // D reads its states an interval ahead
    static constexpr bool DEEP = DEEP_;   // every load of an interval before its first product
    static constexpr int NZW = 2 * NP, WAVES = 3 + 1 + NZW, THREADS = 64 * WAVES, NCH = 16 / NP;
    static constexpr int D_SIZE = 2 * NP * 24 * PIPE_DB, E_SIZE = NE * NP * 6 * PIPE_EB;   // entries
    // pencil (qx, qy) = 4 qx + qy of place pen in chunk ch
    static __device__ __forceinline__ int pencil(int ch, int pen) { return ch * NP + pen; }
};

__device__ __forceinline__ void pipe_barrier() { __syncthreads(); }

// block p = (k, l), k <= l
__device__ __forceinline__ int blk_k(int p) { return p < 3 ? 0 : (p < 5 ? 1 : 2); }
__device__ __forceinline__ int blk_l(int p) { return p < 3 ? p : (p < 5 ? p - 2 : 2); }

// a value that is the same for the wave, kept in scalar registers: the
// barriers of the pipeline would otherwise have a scalar load repeated in
// every interval, and a wait on one also drains the LDS reads in flight
__device__ __forceinline__ double wave_const(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)u), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float wave_const(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// y/x role, wave cy, lanes < 54; sX holds the x tables.  At the end
// out(p, bc, cy, K) gets the lane's K[(3 bx + cx) * 3 + by] of block p, bc =
// 3 bz + cz.
template <typename T, class S, class Out>
__device__ __forceinline__ void pipe_y(const T *sX, const T *__restrict__ ty, const T *sE, int cy, int lane, Out out)
{
    typedef T pair_t __attribute__((ext_vector_type(2)));
    T E2[27], K[27];   // E2[dx][by][dx']
#pragma unroll
    for (int i = 0; i < 27; i++) { E2[i] = (T)0; K[i] = (T)0; }
    const int p = lane / 9, bc = lane % 9;
    const T *Eb = sE + p * PIPE_EB + bc * PIPE_EC;
    for (int g = 0; g < S::NCH + 2; g++) {
        if (g >= 2 && lane < 54) {
            const int ch = g - 2;
#pragma unroll
            for (int pen = 0; pen < S::NP; pen++) {
                const int qy = S::pencil(ch, pen) & 3;
                const pair_t *E = reinterpret_cast<const pair_t *>(Eb + ((S::NE == 2 ? (g & 1) * S::NP : 0) + pen) * (6 * PIPE_EB));
                T pb[9], pcy[3];   // Py[qy][dy][by], Py[qy][dy'][cy]
#pragma unroll
                for (int i = 0; i < 9; i++) pb[i] = ty[9 * qy + i];
#pragma unroll
                for (int d = 0; d < 3; d++) pcy[d] = ty[9 * qy + 3 * d + cy];
                pair_t v[6][3];
#pragma unroll
                for (int i = 0; i < 18; i++) v[i / 3][i % 3] = E[i];
                if (S::DEEP) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < 6; s++) {
                    // dx' = 0: s' 0, 2, 5 (dy' 0, 1, 2); 1: s' 1, 4 (dy' 0, 1); 2: s' 3
                    T t[3];
                    t[0] = pcy[0] * v[s][0][0] + pcy[1] * v[s][1][0] + pcy[2] * v[s][2][1];
                    t[1] = pcy[0] * v[s][0][1] + pcy[1] * v[s][2][0];
                    t[2] = pcy[0] * v[s][1][1];
#pragma unroll
                    for (int by = 0; by < 3; by++)
#pragma unroll
                        for (int d = 0; d < 3; d++) E2[(3 * PIPE_SX[s] + by) * 3 + d] += pb[3 * PIPE_SY[s] + by] * t[d];
                }
                if (qy == 3) {
                    const T *px = sX + 9 * (S::pencil(ch, pen) >> 2);   // px[3 dx + b]
#pragma unroll
                    for (int cx = 0; cx < 3; cx++)
#pragma unroll
                        for (int by = 0; by < 3; by++) {
                            T g[3];
#pragma unroll
                            for (int dx = 0; dx < 3; dx++)
                                g[dx] = px[cx] * E2[(3 * dx + by) * 3] + px[3 + cx] * E2[(3 * dx + by) * 3 + 1]
                                      + px[6 + cx] * E2[(3 * dx + by) * 3 + 2];
#pragma unroll
                            for (int bx = 0; bx < 3; bx++) {
                                T &k = K[(3 * bx + cx) * 3 + by];   // three FMAs
                                k += px[bx] * g[0];
                                k += px[3 + bx] * g[1];
                                k += px[6 + bx] * g[2];
                            }
                        }
#pragma unroll
                    for (int i = 0; i < 27; i++) E2[i] = (T)0;
                    if (ch == S::NCH - 1 && pen == S::NP - 1) out(p, bc, cy, K);
                }
            }
        }
        pipe_barrier();
        if (S::NE == 1) pipe_barrier();
    }
}

// z role, z wave zw, lanes < 54: column part s' and row third t of block p in
// one pencil of the chunk.  Row thirds: the slots with x-y parts s = t (two,
// orders dz and dz + 1 in z) and s = 3 + t (one, order 0); columns likewise
// (s' < 3: two slots, s' >= 3: one, the second weight zero).  tz: the z tables.
template <typename T, class S>
__device__ __forceinline__ void pipe_z(const T *__restrict__ tz, const T *sD, T *sE, int zw, int lane)
{
    typedef T pair_t __attribute__((ext_vector_type(2)));
    // slots 1..9 minus 1 of the x-y parts: 0: {2, 8}, 1: {0, 5}, 2: {1, 7}, 3: 3, 4: 4, 5: 6
    const int zi = zw * 54 + (lane < 54 ? lane : 0), st = zi % 18, t = st / 6, sc = st - 6 * t, p = (zi / 18) % 6, pen = zi / 108;
    const int r1 = (t == 0) ? 2 : t - 1, r2 = (t == 0) ? 8 : (t == 1 ? 5 : 7), r3 = (t == 0) ? 3 : (t == 1 ? 4 : 6);
    const int cc = sc < 3 ? 2 * sc : (sc == 5 ? 8 : 6);            // the lane's pair of columns
    const int lo = (t == 0) ? 1 : 0, ro = (sc == 0) ? 1 : 0;       // first order in z
    const bool u1 = sc != 4, u2 = sc < 3 || sc == 4;               // which of the pair the lane takes
    const int o1 = PIPE_DR * r1 + cc, o2 = PIPE_DR * r2 + cc, o3 = PIPE_DR * r3 + cc;
    T w1[4][3], w2[4][3], l1[4][3], l2[4][3], l3[4][3];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int z = 0; z < 3; z++) {
            w1[q][z] = u1 ? tz[9 * q + 3 * ro + z] : (T)0;
            w2[q][z] = u2 ? tz[9 * q + (sc < 3 ? 3 * ro + 3 : 0) + z] : (T)0;
            l1[q][z] = tz[9 * q + 3 * lo + z];
            l2[q][z] = tz[9 * q + 3 * lo + 3 + z];
            l3[q][z] = wave_const(tz[9 * q + z]);
        }
    const T *Dl = sD + (pen * 24 + p) * PIPE_DB;
    T *El = sE + (pen * 6 + p) * PIPE_EB + 6 * t + sc;
    T ea[9], eb[9];   // [bz][cz]
    for (int g = 0; g < S::NCH + 2; g++) {
        const bool on = g >= 1 && g <= S::NCH && lane < 54;
        if (on) {
            const T *Dc = Dl + ((g - 1) & 1) * (S::NP * 24 * PIPE_DB);
#pragma unroll
            for (int i = 0; i < 9; i++) { ea[i] = (T)0; eb[i] = (T)0; }
            pair_t dv[4][3];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const T *d = Dc + q * (6 * PIPE_DB);
                dv[q][0] = *reinterpret_cast<const pair_t *>(d + o1);
                dv[q][1] = *reinterpret_cast<const pair_t *>(d + o2);
                dv[q][2] = *reinterpret_cast<const pair_t *>(d + o3);
            }
            if (S::DEEP) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const T d11 = dv[q][0][0], d12 = dv[q][0][1], d21 = dv[q][1][0], d22 = dv[q][1][1], d31 = dv[q][2][0], d32 = dv[q][2][1];
#pragma unroll
                for (int cz = 0; cz < 3; cz++) {
                    const T f1 = d11 * w1[q][cz] + d12 * w2[q][cz];
                    const T f2 = d21 * w1[q][cz] + d22 * w2[q][cz];
                    const T f3 = d31 * w1[q][cz] + d32 * w2[q][cz];
#pragma unroll
                    for (int bz = 0; bz < 3; bz++) {
                        ea[3 * bz + cz] += l1[q][bz] * f1;
                        ea[3 * bz + cz] += l2[q][bz] * f2;
                        eb[3 * bz + cz] += l3[q][bz] * f3;
                    }
                }
            }
        }
        if (S::NE == 1) pipe_barrier();   // y has read the previous chunk's E1
        if (on) {
            T *o = El + (S::NE == 2 ? ((g - 1) & 1) * (S::NP * 6 * PIPE_EB) : 0);
#pragma unroll
            for (int i = 0; i < 9; i++) {
                o[PIPE_EC * i] = ea[i];
                o[PIPE_EC * i + 18] = eb[i];
            }
        }
        pipe_barrier();
    }
}

// D role: lane (pencil, qz, block) of the chunk.  A chunk's state is read
// (In::load) before the barrier that ends the interval before (PF, where the
// registers allow it), and turned into the block's rows after it.
template <typename T, class S, class In>
__device__ __forceinline__ void pipe_d(T *sD, int lane, In in)
{
    const int p = lane % 6, k = blk_k(p), l = blk_l(p), qz = (lane / 6) & 3, pen = lane / 24;
    T *Dl = sD + (pen * 24 + qz * 6 + p) * PIPE_DB;
    const bool on = lane < 24 * S::NP;
    if (S::PF && on) in.load(S::pencil(0, pen) * 4 + qz, k, l);
    for (int g = 0; g < S::NCH + 2; g++) {
        if (g < S::NCH && on) {
            if (!S::PF) in.load(S::pencil(g, pen) * 4 + qz, k, l);
            __builtin_amdgcn_sched_barrier(0);
            in.template rows<T>(k, l, Dl + (g & 1) * (S::NP * 24 * PIPE_DB));
            if (S::PF && g + 1 < S::NCH) in.load(S::pencil(g + 1, pen) * 4 + qz, k, l);
        }
        pipe_barrier();
        if (S::NE == 1) pipe_barrier();
    }
}

// The whole contraction, in the intervals 0 .. NCH + 1: chunk g in D, g - 1 in z,
// g - 2 in y.
template <typename T, class S, class In, class Out>
__device__ __forceinline__ void sep_pipeline(const T *sX, const T *__restrict__ ty, const T *__restrict__ tz, T *sD, T *sE, In in, Out out)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (wave < 3) pipe_y<T, S>(sX, ty, sE, wave, lane, out);
    else if (wave < 4) pipe_d<T, S>(sD, lane, in);
    else pipe_z<T, S>(tz, sD, sE, wave - 4, lane);
}

// a row of a D block -> LDS: v[a - 1] = D[(k, row), (l, a)], a = 1..9
template <typename T>
__device__ __forceinline__ void d_store(T *row, const double *v)
{
    typedef T pair_t __attribute__((ext_vector_type(2)));
    constexpr int AT[10] = {2, 8, 0, 5, 1, 7, 3, 4, 6, -1};   // slot (minus 1) of each column
    pair_t *o = reinterpret_cast<pair_t *>(row);
#pragma unroll
    for (int c = 0; c < 5; c++) {
        pair_t x;
        x[0] = (T)v[AT[2 * c]];
        x[1] = AT[2 * c + 1] < 0 ? (T)0 : (T)v[AT[2 * c + 1] < 0 ? 0 : AT[2 * c + 1]];
        o[c] = x;
    }
}

// The second-second block of slots from B[I][J] = c(I, J) F_kI F_lJ (c the
// strain-gradient coefficients): row s of the six; pairs without a common index
// have no entry.
__device__ __forceinline__ void d_second(const double (*B)[3], int s, double *v)
{
    constexpr int PI[6] = {0, 0, 0, 1, 1, 2}, PK[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int r = 0; r < 6; r++) {
        const int I = PI[s], K = PK[s], J = PI[r], K2 = PK[r];
        double x = 0.0;
        if (K == K2) x += B[I][J];
        if (J != K2 && K == J) x += B[I][K2];
        if (I != K && I == K2) x += B[K][J];
        if (I != K && J != K2 && I == J) x += B[K][K2];
        v[r] = x;
    }
}

// D block (k, l) of the stored energy at one point from the strain-measure
// state, slots 1..9 both ways: the entries of c_row at compile-time indices,
// sharing the products F_k F_l.  State layout (read in 16-byte pairs; the stride
// of 52 puts the eight points of a chunk on different banks): per component k at
// 10 k F (3), a gap, H (6, symmetric pairs); times the point weight S at 30, N at
// 36 (6 each), G at 42 (9); the weight at 51.
constexpr int SST_S = 30, SST_N = 36, SST_G = 42, SST_WGT = 51, SST_W = 52;
struct StaticIn {
    const double *sSt;
    double e345, le;
    double a[10], b[10], S[6], N[6], G[10];
    __device__ __forceinline__ void load(int q, int k, int l)
    {
        typedef double pair_t __attribute__((ext_vector_type(2)));
        const double *st = sSt + q * SST_W;
        auto get = [&](double *dst, int at, int n) {
#pragma unroll
            for (int i = 0; i < n / 2; i++) {
                const pair_t x = *reinterpret_cast<const pair_t *>(st + at + 2 * i);
                dst[2 * i] = x[0];
                dst[2 * i + 1] = x[1];
            }
        };
        get(a, 10 * k, 10);
        get(b, 10 * l, 10);
        get(N, SST_N, 6);
        get(S, SST_S, 6);
        get(G, SST_G, 10);
    }
    template <typename T>
    __device__ __forceinline__ void rows(int k, int l, T *dst) const
    {
        constexpr int PI[6] = {0, 0, 0, 1, 1, 2}, PK[6] = {0, 1, 2, 1, 2, 2};
        constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
        const double dd = (k == l) ? 1.0 : 0.0, w = G[9], eh = w * 0.5 * e345, g = w * 2.0 * le * le;
        const double g1 = g * (2.0 / 3.0), g0 = g * (-1.0 / 3.0);
        const double *Fk = a, *Fl = b, *Hk = a + 4, *Hl = b + 4;
        double A[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) A[i][j] = Fk[i] * Fl[j];
        // first-gradient rows
        double l1[3], l0[3];   // 2 le^2 (2/3, -1/3) F_l
#pragma unroll
        for (int i = 0; i < 3; i++) { l1[i] = g1 * Fl[i]; l0[i] = g0 * Fl[i]; }
#pragma unroll
        for (int L = 0; L < 3; L++) {
            double v[9];
#pragma unroll
            for (int M = 0; M < 3; M++) {
                const double hh = Hk[SY[L][0]] * Hl[SY[M][0]] + Hk[SY[L][1]] * Hl[SY[M][1]] + Hk[SY[L][2]] * Hl[SY[M][2]];
                double x = N[SY[L][M]] * A[L][M] + dd * S[SY[L][M]];
                x += eh * (L == M ? A[(L + 1) % 3][(L + 1) % 3] + A[(L + 2) % 3][(L + 2) % 3] : A[M][L]);
                x += (L == M ? g1 : g0) * hh;
                v[M] = x;
            }
#pragma unroll
            for (int s = 0; s < 6; s++) {
                const int I = PI[s], K = PK[s];
                double x = Hk[SY[L][K]] * (L == I ? l1[I] : l0[I]);
                if (I != K) x += Hk[SY[L][I]] * (L == K ? l1[K] : l0[K]);
                if (L == I) x += dd * G[3 * I + K];
                else if (L == K) x += dd * G[3 * K + I];
                v[3 + s] = x;
            }
            d_store<T>(dst + PIPE_DR * L, v);
        }
        // second-gradient rows
        double k1[3], k0[3], B[3][3];   // 2 le^2 (2/3, -1/3) F_k
#pragma unroll
        for (int i = 0; i < 3; i++) { k1[i] = g1 * Fk[i]; k0[i] = g0 * Fk[i]; }
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) B[i][j] = (i == j ? g1 : g0) * A[i][j];
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int I = PI[s], K = PK[s];
            double v[9];
#pragma unroll
            for (int L = 0; L < 3; L++) {
                double u = Hl[SY[L][K]] * (L == I ? k1[I] : k0[I]);
                if (I != K) u += Hl[SY[L][I]] * (L == K ? k1[K] : k0[K]);
                if (L == I) u += dd * G[3 * I + K];
                else if (L == K) u += dd * G[3 * K + I];
                v[L] = u;
            }
            d_second(B, s, v + 3);
            d_store<T>(dst + PIPE_DR * (3 + s), v);
        }
    }
};

// D block (k, l) of the stored energy in parametric slots, for a geometry that
// is no product: the pointwise tangent of the physical jet, pulled back to the
// parametric jets of the tensor-product basis (rows and columns through
//   u_,L = sum_i Gi_iL u_i,   u_,IK = sum_ij Gi_iI Gi_jK (u_ij - sum_n Ga^n_ij u_n),
// Gi the inverse of the map's gradient, Ga its connection).  Nothing is pulled
// back entry by entry: with E_IK = sum_L F_LI H_LIK the gradient part of the block is a product
// in each index, so that with
//   a^k_rI = F_kI Gi_rI,  a'^k_Mr = g sum_I c_MI a^k_rI (c = 1 - 1/3 on, -1/3 off the diagonal),
//   h^k_Ls = sum_K H_kLK Gi_sK,  m_rs = sum_K Gi_rK Gi_sK,  B_rn = sum_L a'^k_Lr a^l_nL
// the second-second entry of ((r, s), (n, m)) is B_rn m_sm, symmetrised, the
// physical-first one of (M, (r, s)) is a'_Mr h_Ms, symmetrised, and only the
// connection is left to apply: 850 FP64 instructions per block against 1300 for pulling back the
// physical block.  State layout (16-byte pairs; the stride of 94 puts the eight
// points of a chunk on different banks): per component k at 10 k F (3), a gap, H
// (6); times the point weight S at 30, N at 36 (6 each) and at 42 + 6 L
// G_L(rs) = sum_K G_LK Gi_rL Gi_sK, symmetrised; Gi at 60 (3 r + I), the weight
// at 69, Ga at 70 + 6 n, m at 88.
constexpr int GST_S = 30, GST_N = 36, GST_G = 42, GST_GI = 60, GST_WGT = 69, GST_GA = 70, GST_M = 88, GST_W = 94;
struct GeneralIn {
    const double *sSt;
    double e345, le;
    const double *st;
    int ok, ol;
    __device__ __forceinline__ void load(int q, int k, int l)
    {
        st = sSt + q * GST_W;
        ok = 10 * k;
        ol = 10 * l;
    }
    __device__ __forceinline__ void get(double *dst, int at, int n) const
    {
        typedef double pair_t __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int i = 0; i < n / 2; i++) {
            const pair_t x = *reinterpret_cast<const pair_t *>(st + at + 2 * i);
            dst[2 * i] = x[0];
            dst[2 * i + 1] = x[1];
        }
    }
    // a[r][I] = F_I Gi_rI and ac[M][r] = g sum_I c_MI a[r][I]
    static __device__ __forceinline__ void pull(const double *F, const double *Gi, double g, double (*a)[3], double (*ac)[3])
    {
#pragma unroll
        for (int r = 0; r < 3; r++) {
#pragma unroll
            for (int I = 0; I < 3; I++) a[r][I] = F[I] * Gi[3 * r + I];
            const double t = (a[r][0] + a[r][1] + a[r][2]) * (1.0 / 3.0);
#pragma unroll
            for (int I = 0; I < 3; I++) ac[I][r] = g * (a[r][I] - t);
        }
    }
    // h[L][s] = sum_K H_LK Gi_sK
    static __device__ __forceinline__ void lower(const double *H, const double *Gi, double (*h)[3])
    {
        constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
#pragma unroll
        for (int L = 0; L < 3; L++)
#pragma unroll
            for (int s = 0; s < 3; s++) h[L][s] = H[SY[L][0]] * Gi[3 * s] + H[SY[L][1]] * Gi[3 * s + 1] + H[SY[L][2]] * Gi[3 * s + 2];
    }
    template <typename T>
    __device__ __forceinline__ void rows(int k, int l, T *dst) const
    {
        constexpr int PI[6] = {0, 0, 0, 1, 1, 2}, PK[6] = {0, 1, 2, 1, 2, 2};
        constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
        double Gi[10], Ga[18], Fk[4], Fl[4], Hk[6], Hl[6];
        get(Gi, GST_GI, 10);
        get(Ga, GST_GA, 18);
        const double dd = (k == l) ? 1.0 : 0.0, w = Gi[9], eh = w * 0.5 * e345, g = w * 2.0 * le * le;
        double W[3][3], V[3][6];
#pragma unroll
        for (int i = 0; i < 3; i++) {
#pragma unroll
            for (int n = 0; n < 3; n++) W[i][n] = 0.0;
#pragma unroll
            for (int c = 0; c < 6; c++) V[i][c] = 0.0;
        }
        {
            // second rows (r, s); their part of the first rows through the connection
            // (the states are read again below rather than kept: 256 registers hold
            // Ga, W, V and what a row takes)
            double B[3][3], hl[3][3], a[3][3], al[3][3], akc[3][3], mt[6];
            get(Fk, ok, 4);
            get(Fl, ol, 4);
            get(Hl, ol + 4, 6);
            get(mt, GST_M, 6);
            pull(Fl, Gi, g, al, a);
            pull(Fk, Gi, g, a, akc);
            lower(Hl, Gi, hl);
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int n = 0; n < 3; n++) B[r][n] = akc[0][r] * al[n][0] + akc[1][r] * al[n][1] + akc[2][r] * al[n][2];
#pragma unroll
            for (int t = 0; t < 6; t++) {
                const int r = PI[t], s = PK[t];
                double f[3], v[9];
#pragma unroll
                for (int M = 0; M < 3; M++) {
                    f[M] = akc[M][r] * hl[M][s] + dd * st[GST_G + 6 * M + t];
                    if (r != s) f[M] += akc[M][s] * hl[M][r];
                }
#pragma unroll
                for (int c = 0; c < 6; c++) {
                    const int n = PI[c], m = PK[c];
                    double x = B[r][n] * mt[SY[s][m]];
                    if (n != m) x += B[r][m] * mt[SY[s][n]];
                    if (r != s) x += B[s][n] * mt[SY[r][m]];
                    if (r != s && n != m) x += B[s][m] * mt[SY[r][n]];
                    v[3 + c] = x;
                }
#pragma unroll
                for (int n = 0; n < 3; n++) {
                    double x = f[0] * Gi[3 * n] + f[1] * Gi[3 * n + 1] + f[2] * Gi[3 * n + 2];
#pragma unroll
                    for (int c = 0; c < 6; c++) x -= v[3 + c] * Ga[6 * n + c];
                    v[n] = x;
                }
                d_store<T>(dst + PIPE_DR * (3 + t), v);
#pragma unroll
                for (int i = 0; i < 3; i++) {
#pragma unroll
                    for (int n = 0; n < 3; n++) W[i][n] -= Ga[6 * i + t] * v[n];
#pragma unroll
                    for (int c = 0; c < 6; c++) V[i][c] -= Ga[6 * i + t] * v[3 + c];
                }
            }
        }
        // first rows
        double hk[3][3], al[3][3], alc[3][3], S[6], N[6];
        get(Fk, ok, 4);
        get(Fl, ol, 4);
        get(Hk, ok + 4, 6);
        get(Hl, ol + 4, 6);
        pull(Fl, Gi, g, al, alc);
        lower(Hk, Gi, hk);
        get(S, GST_S, 6);
        get(N, GST_N, 6);
#pragma unroll
        for (int L = 0; L < 3; L++) {
            double f[3], x[6];
#pragma unroll
            for (int M = 0; M < 3; M++) {
                const double hh = Hk[SY[L][0]] * Hl[SY[M][0]] + Hk[SY[L][1]] * Hl[SY[M][1]] + Hk[SY[L][2]] * Hl[SY[M][2]];
                double y = N[SY[L][M]] * (Fk[L] * Fl[M]) + dd * S[SY[L][M]];
                y += eh * (L == M ? Fk[(L + 1) % 3] * Fl[(L + 1) % 3] + Fk[(L + 2) % 3] * Fl[(L + 2) % 3] : Fk[M] * Fl[L]);
                y += g * (L == M ? 2.0 / 3.0 : -1.0 / 3.0) * hh;
                f[M] = y;
            }
#pragma unroll
            for (int c = 0; c < 6; c++) {
                const int n = PI[c], m = PK[c];
                x[c] = alc[L][n] * hk[L][m] + dd * st[GST_G + 6 * L + c];
                if (n != m) x[c] += alc[L][m] * hk[L][n];
            }
            double y[3];
#pragma unroll
            for (int n = 0; n < 3; n++) {
                y[n] = f[0] * Gi[3 * n] + f[1] * Gi[3 * n + 1] + f[2] * Gi[3 * n + 2];
#pragma unroll
                for (int c = 0; c < 6; c++) y[n] -= x[c] * Ga[6 * n + c];
            }
#pragma unroll
            for (int i = 0; i < 3; i++) {
#pragma unroll
                for (int n = 0; n < 3; n++) W[i][n] += Gi[3 * i + L] * y[n];
#pragma unroll
                for (int c = 0; c < 6; c++) V[i][c] += Gi[3 * i + L] * x[c];
            }
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double v[9];
#pragma unroll
            for (int n = 0; n < 3; n++) v[n] = W[i][n];
#pragma unroll
            for (int c = 0; c < 6; c++) v[3 + c] = V[i][c];
            d_store<T>(dst + PIPE_DR * i, v);
        }
    }
};

// The block of StaticIn from the moment state of the transient rule: every product of two
// state factors is the sum over the two transformed components, every N-weighted
// one the form X^T N^ Y.  State layout: per component k at 18 k F^ (3 + 3) and H^
// (6 + 6), then Sb and the three N^ blocks (6 each, symmetric pairs) and Gb (9);
// the point weights apart, in FP64.
constexpr int MS_S = 54, MS_N11 = 60, MS_N12 = 66, MS_N22 = 72, MS_G = 78, MS_W = 88;
template <typename TS>
struct MomentIn {
    const TS *sMom;
    const double *sWgt;
    double e345, le;
    const TS *a, *b, *S, *G;   // read entry by entry: in registers they are 70
    double wgt;
    __device__ __forceinline__ void load(int q, int k, int l)
    {
        a = sMom + q * MS_W + 18 * k;
        b = sMom + q * MS_W + 18 * l;
        S = sMom + q * MS_W + MS_S;
        G = sMom + q * MS_W + MS_G;
        wgt = sWgt[q];
    }
    template <typename T>
    __device__ __forceinline__ void rows(int k, int l, T *dst) const
    {
        constexpr int PI[6] = {0, 0, 0, 1, 1, 2}, PK[6] = {0, 1, 2, 1, 2, 2};
        constexpr int SY[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
        const double w = wgt, dd = (k == l) ? w : 0.0, g = 2.0 * le * le * w;
        const double g1 = g * (2.0 / 3.0), g0 = g * (-1.0 / 3.0);
        auto Fk = [&](int c, int i) { return (double)a[3 * c + i]; };
        auto Fl = [&](int c, int i) { return (double)b[3 * c + i]; };
        auto Hk = [&](int c, int i) { return (double)a[6 + 6 * c + i]; };
        auto Hl = [&](int c, int i) { return (double)b[6 + 6 * c + i]; };
        double A[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) A[i][j] = Fk(0, i) * Fl(0, j) + Fk(1, i) * Fl(1, j);
        const double eh = 0.5 * e345 * w;
#pragma unroll
        for (int L = 0; L < 3; L++) {
            double v[9];
#pragma unroll
            for (int M = 0; M < 3; M++) {
                double hh = 0.0;
#pragma unroll
                for (int c = 0; c < 3; c++) hh += Hk(0, SY[L][c]) * Hl(0, SY[M][c]) + Hk(1, SY[L][c]) * Hl(1, SY[M][c]);
                double x = (double)S[6 + SY[L][M]] * (Fk(0, L) * Fl(0, M)) + (double)S[12 + SY[L][M]] * (Fk(0, L) * Fl(1, M) + Fk(1, L) * Fl(0, M))
                         + (double)S[18 + SY[L][M]] * (Fk(1, L) * Fl(1, M));
                x = w * x + dd * (double)S[SY[L][M]];
                x += eh * (L == M ? A[(L + 1) % 3][(L + 1) % 3] + A[(L + 2) % 3][(L + 2) % 3] : A[M][L]);
                x += (L == M ? g1 : g0) * hh;
                v[M] = x;
            }
#pragma unroll
            for (int s = 0; s < 6; s++) {
                const int I = PI[s], K = PK[s];
                double x = (L == I ? g1 : g0) * (Hk(0, SY[L][K]) * Fl(0, I) + Hk(1, SY[L][K]) * Fl(1, I));
                if (I != K) x += (L == K ? g1 : g0) * (Hk(0, SY[L][I]) * Fl(0, K) + Hk(1, SY[L][I]) * Fl(1, K));
                if (L == I) x += dd * (double)G[3 * I + K];
                else if (L == K) x += dd * (double)G[3 * K + I];
                v[3 + s] = x;
            }
            d_store<T>(dst + PIPE_DR * L, v);
        }
        double B[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) B[i][j] = (i == j ? g1 : g0) * A[i][j];
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int I = PI[s], K = PK[s];
            double v[9];
#pragma unroll
            for (int L = 0; L < 3; L++) {
                double u = (L == I ? g1 : g0) * (Hl(0, SY[L][K]) * Fk(0, I) + Hl(1, SY[L][K]) * Fk(1, I));
                if (I != K) u += (L == K ? g1 : g0) * (Hl(0, SY[L][I]) * Fk(0, K) + Hl(1, SY[L][I]) * Fk(1, K));
                if (L == I) u += dd * (double)G[3 * I + K];
                else if (L == K) u += dd * (double)G[3 * K + I];
                v[L] = u;
            }
            d_second(B, s, v + 3);
            d_store<T>(dst + PIPE_DR * (3 + s), v);
        }
    }
};

}  // namespace igap
