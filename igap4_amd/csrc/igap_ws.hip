// igap_ws.hip -- learned warm start for the Newton load/time steps: a small
// 3-D convolutional network on the control-point grid, trained and evaluated
// with BF16 matrix-core products and FP32 accumulation (gfx950).
//
// Network: NL = 4 layers of 3x3x3 convolutions (zero padding, per-layer
// dilation), 16 channels between layers, ReLU after layers 0..2, linear last
// layer.  Input channels (<= 16) and output channels (<= 16) are zero-padded
// to 16 so that one 16x16x16 BF16 product covers one tap.
//
// Data layout (all device, channels-last):
//   activations  a[v][16]   BF16 bits, v = (x*ny + y)*nz + z  (the control-
//                point numbering of the assembly, z fastest)
//   weights      W[t][co][ci] BF16 (forward B operand), WT[t][ci][co] (input-
//                gradient B operand), t = 9*(dx+1) + 3*(dy+1) + (dz+1)
//   master copy  FP32 params, per layer W[27][16][16] then b[16]; Adam moments
//
// Convolution as an implicit GEMM on V_MFMA_F32_16X16X16_BF16: M = 16 voxels,
// N = 16 output channels, K = 16 input channels of one tap, 27 taps
// accumulated in one FP32 tile.  Lane l supplies A[l&15][4(l>>4)+j] and
// B[4(l>>4)+j][l&15] (j = 0..3); result register r of lane l holds
// D[4(l>>4)+r][l&15] (pinned by igap_ws_selftest_mfma_bf16).
//
// The net is a chain of small kernels (a layer of the 66x18x18 grid is 50 ns of
// matrix-core time), so what bounds a training pair is the number of launches and the
// load latency inside each: nine dependent launches (pack, four layers, four
// backward steps that do the input and the weight gradient side by side) and
// one reduction (one per layer where the partials of all would be large,
// PART_ALL_BYTES), every load of a tile issued before its first product.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "igap_ws_impl.h"

namespace igap {
namespace ws {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f)
{
    // round to nearest even (inputs are finite)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ float4_t mma(short4_t a, short4_t b, float4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

typedef int int4_t __attribute__((ext_vector_type(4)));

enum { FWD_RELU = 0, FWD_LAST = 1, BWD_MASK = 2, FWD_LOSS = 3 };

// One tap's offset along each axis (the dilation, clamped to the grid's size
// there: a tap that far off is outside either way, and the products of the
// offsets then stay within 32 bits).
// myz, mz: reciprocals 2^64 / d of ny nz and nz, rounded up (0 for d = 1): the
// upper half of v m is v / d for every v d < 2^64.  (The 32-bit divisions of a
// run-time divisor were much of a weight-gradient wave's instructions: k_back 18.1 -> 16.7 us.)
struct Shape {
    int nx, ny, nz, dx, dy, dz;
    uint64_t myz, mz;
    __device__ __forceinline__ void point(int v, int &x, int &y, int &z) const
    {
        const int r = mz ? (int)__umul64hi((uint64_t)(uint32_t)v, mz) : v;
        x = myz ? (int)__umul64hi((uint64_t)(uint32_t)v, myz) : v;
        y = r - x * ny;
        z = v - r * nz;
    }
};

// Where the tiles of a lane's voxel lie: the voxel's first channel of the
// lane, and which neighbours along each axis are inside the grid (sgn +1: the
// taps read v + off, -1: v - off).
struct Taps {
    int base;
    bool in[3][3];   // [axis][tap]
    __device__ __forceinline__ Taps(const Shape &g, int v, int V, int kg, int sgn)
    {
        const bool vin = v < V;
        if (!vin) v = V - 1;
        base = v * 16 + 4 * kg;
        int x, y, z;
        g.point(v, x, y, z);
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int s = sgn * (t - 1), xx = x + s * g.dx, yy = y + s * g.dy, zz = z + s * g.dz;
            in[0][t] = vin && xx >= 0 && xx < g.nx;
            in[1][t] = yy >= 0 && yy < g.ny;
            in[2][t] = zz >= 0 && zz < g.nz;
        }
    }
    __device__ __forceinline__ bool ok(int t) const { return in[0][t / 9] && in[1][(t / 3) % 3] && in[2][t % 3]; }
    // the lane's four channels of tap t, from an address inside the array whatever the tap
    __device__ __forceinline__ short4_t load(const Shape &g, const uint16_t *__restrict__ a, int t, int sgn) const
    {
        const int off = sgn * ((t / 9 - 1) * g.dx * (g.ny * g.nz) + ((t / 3) % 3 - 1) * g.dy * g.nz + (t % 3 - 1) * g.dz) * 16;
        return *reinterpret_cast<const short4_t *>(a + (base + (ok(t) ? off : 0)));
    }
};

// One wave per tile of 16 consecutive voxels, all 16 output channels.
//   FWD_RELU  aout = bf16(relu(sum + bias))
//   FWD_LAST  yout[v][c] = sum + bias  (c < cout, FP32)
//   FWD_LOSS  e = sum + bias - target[v][c]: aout = bf16(2 e / (V cout)) (0 for
//             c >= cout), lpart[tile] = sum of e^2
//   BWD_MASK  aout = bf16(sum * (mask > 0))   (input gradient through ReLU)
// sgn = +1 gathers in[v + off_t] (forward), -1 gathers in[v - off_t]
// (gradient with respect to the layer input).
// The 54 loads of a tile (27 activation tiles, 27 weight tiles, all in L2) are
// in flight together; issued tap by tap the kernel waited for each pair:
// 13.5 us a layer at 66x18x18, now 6.2 us.
template <int MODE>
__device__ __forceinline__ void conv_tile(const Shape &g, int tile, int lane, int sgn, const uint16_t *__restrict__ ain,
                                          const uint16_t *__restrict__ Wk, const float *__restrict__ bias,
                                          const uint16_t *__restrict__ mask, const float *__restrict__ tg,
                                          uint16_t *__restrict__ aout, float *__restrict__ yout, float *__restrict__ lpart, int cout)
{
    const int V = g.nx * g.ny * g.nz, v0 = tile * 16;
    if (v0 >= V) return;
    const int i = lane & 15, kg = lane >> 4;
    const Taps tp(g, v0 + i, V, kg, sgn);
    short4_t a[27], b[27];
#pragma unroll
    for (int t = 0; t < 27; t++) {
        a[t] = tp.load(g, ain, t, sgn);
        b[t] = *reinterpret_cast<const short4_t *>(Wk + (t * 16 + i) * 16 + 4 * kg);
    }
    const float bi = MODE == BWD_MASK ? 0.f : bias[i];
    float tv[4];
    uint16_t mv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int vo = v0 + 4 * kg + r;
        tv[r] = (MODE == FWD_LOSS && vo < V && i < cout) ? tg[(size_t)vo * cout + i] : 0.f;
        mv[r] = (MODE == BWD_MASK && vo < V) ? mask[(size_t)vo * 16 + i] : (uint16_t)0;
    }
    __builtin_amdgcn_sched_barrier(0);
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 27; t++) acc = mma(tp.ok(t) ? a[t] : (short4_t){0, 0, 0, 0}, b[t], acc);
    float e2 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int vo = v0 + 4 * kg + r;
        if (vo >= V) continue;
        float val = acc[r];
        if (MODE == FWD_RELU) {
            val += bi;
            aout[(size_t)vo * 16 + i] = f2bf(val > 0.f ? val : 0.f);
        } else if (MODE == FWD_LAST) {
            if (i < cout) yout[(size_t)vo * cout + i] = val + bi;
        } else if (MODE == FWD_LOSS) {
            const float e = i < cout ? (val + bi) - tv[r] : 0.f;
            e2 += e * e;
            aout[(size_t)vo * 16 + i] = f2bf(i < cout ? 2.f * e / ((float)V * (float)cout) : 0.f);
        } else {
            aout[(size_t)vo * 16 + i] = f2bf(bf2f(mv[r]) > 0.f ? val : 0.f);
        }
    }
    if (MODE == FWD_LOSS) {
        for (int o = 32; o > 0; o >>= 1) e2 += __shfl_xor(e2, o, 64);
        if (lane == 0) lpart[tile] = e2;
    }
}

template <int MODE>
__global__ __launch_bounds__(256) void k_conv(Shape g, const uint16_t *__restrict__ ain, const uint16_t *__restrict__ Wk,
                                              const float *__restrict__ bias, const float *__restrict__ tg,
                                              uint16_t *__restrict__ aout, float *__restrict__ yout, float *__restrict__ lpart, int cout)
{
    conv_tile<MODE>(g, blockIdx.x * 4 + (threadIdx.x >> 6), threadIdx.x & 63, 1, ain, Wk, bias, nullptr, tg, aout, yout, lpart, cout);
}

// A 16x16 tile of 16-bit values across the lanes of a wave: X[l&15][4(l>>4)+j]
// in, X[4(l>>4)+j][l&15] out.  The lane's eight bytes are row l&15 of a 16x32
// byte matrix; two exact integer products select the low and the high bytes of
// every column (sel: k == 2n and k == 2n + 1), and the result registers hold them
// transposed.  No LDS, any bit pattern.
struct Transposer {
    long lo, hi;
    __device__ __forceinline__ explicit Transposer(int lane)
    {
        const int k = 2 * (lane & 15) - 8 * (lane >> 4);   // place of column n's low byte in the lane's B[8 kg + j][n]
        lo = (k >= 0 && k < 8) ? (long)(1ull << (8 * k)) : 0;
        hi = (k >= 0 && k < 8) ? (long)(1ull << (8 * k + 8)) : 0;
    }
    __device__ __forceinline__ short4_t operator()(short4_t x) const
    {
        const int4_t zero = {0, 0, 0, 0};
        const long b = __builtin_bit_cast(long, x);
        const int4_t l = __builtin_amdgcn_mfma_i32_16x16x32_i8(b, lo, zero, 0, 0, 0);
        const int4_t h = __builtin_amdgcn_mfma_i32_16x16x32_i8(b, hi, zero, 0, 0, 0);
        uint32_t p[4];   // low byte, high byte, 0, 0
#pragma unroll
        for (int r = 0; r < 4; r++) p[r] = __builtin_amdgcn_perm((uint32_t)h[r], (uint32_t)l[r], 0x0c0c0400u);
        const uint64_t w = (uint64_t)(p[0] | (p[1] << 16)) | ((uint64_t)(p[2] | (p[3] << 16)) << 32);
        return __builtin_bit_cast(short4_t, w);
    }
};

// Backward step of one layer.  Blocks 0 .. ncb - 1 (CONV): the input gradient,
// as k_conv.  The others: the gradients of the weights and the bias, one wave per
// chunk of CHUNK voxels and tap (t = 27: the bias),
//   part[t][c][ci][co] = sum_{v in chunk c} a[v + off_t][ci] dz[v][co]
//   bpart[c][co]       = sum_{v in chunk c} dz[v][co]
// with M = ci, N = co, K = 16 voxels of a product, the chunk's tiles in order.
// Tiles are read as the convolution reads them (eight bytes a lane, eight tiles
// in flight) and transposed in registers.  The gradient of layer l - 1 needs
// only the input gradient, so both run in one launch.
// At 66x18x18 gathering two bytes a lane and tile at a time took 42 us a
// layer for the weights and a loop over single voxels 36 us for the bias;
// now 14.1 us with the input gradient (13 us before) beside, 11.6 us without.
template <bool CONV>
__global__ __launch_bounds__(256) void k_back(Shape g, int ncb, const uint16_t *__restrict__ ain, const uint16_t *__restrict__ dz,
                                              const uint16_t *__restrict__ WTk, uint16_t *__restrict__ dzprev, int nchunk,
                                              float *__restrict__ part, float *__restrict__ bpart)
{
    __shared__ uint4 sdz[CHUNK * 32 / 16];   // one wave's: the bias sums of a chunk
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (CONV && (int)blockIdx.x < ncb) {
        // the mask of the ReLU that made this layer's input is that input
        conv_tile<BWD_MASK>(g, blockIdx.x * 4 + wv, lane, -1, dz, WTk, nullptr, ain, nullptr, dzprev, nullptr, nullptr, 16);
        return;
    }
    static_assert(CHUNK % 128 == 0, "eight tiles a round");
    const int V = g.nx * g.ny * g.nz;
    const int bb = blockIdx.x - ncb, c = bb / 7, t = __builtin_amdgcn_readfirstlane(4 * (bb - 7 * c) + wv);
    const int i = lane & 15, kg = lane >> 4;
    const int vbeg = c * CHUNK, vend = vbeg + CHUNK < V ? vbeg + CHUNK : V;
    if (t == 27) {
        // the whole chunk in flight at once; the sum itself is a chain of CHUNK additions per channel
        constexpr int NL16 = CHUNK * 32 / (64 * 16);
        uint4 d[NL16];
#pragma unroll
        for (int j = 0; j < NL16; j++) {
            const int at = (j * 64 + lane) / 2, v = vbeg + at < V ? vbeg + at : V - 1;   // half a voxel a lane
            d[j] = *reinterpret_cast<const uint4 *>(dz + (size_t)v * 16 + 8 * (lane & 1));
        }
#pragma unroll
        for (int j = 0; j < NL16; j++) sdz[j * 64 + lane] = d[j];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint16_t *q = reinterpret_cast<const uint16_t *>(sdz) + i;
        const int n = vend - vbeg;
        float s = 0.f;
        int v = 0;
        for (; v + 32 <= n; v += 32) {
            uint16_t e[32];
#pragma unroll
            for (int j = 0; j < 32; j++) e[j] = q[16 * (v + j)];
#pragma unroll
            for (int j = 0; j < 32; j++) s += bf2f(e[j]);
        }
        for (; v < n; v++) s += bf2f(q[16 * v]);
        if (kg == 0) bpart[c * 16 + i] = s;
        return;
    }
    const Transposer tr(lane);
    const int tx = t / 9 - 1, ty = (t / 3) % 3 - 1, tz = t % 3 - 1;
    const int sx = tx * g.dx, sy = ty * g.dy, sz = tz * g.dz, off = (sx * (g.ny * g.nz) + sy * g.nz + sz) * 16;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int vb = vbeg; vb < vend; vb += 128) {
        short4_t a[8], d[8];
        bool ok[8], in[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            int v = vb + 16 * j + i;
            in[j] = v < vend;
            if (!in[j]) v = V - 1;
            int x, y, z;
            g.point(v, x, y, z);
            x += sx;
            y += sy;
            z += sz;
            ok[j] = in[j] && x >= 0 && x < g.nx && y >= 0 && y < g.ny && z >= 0 && z < g.nz;
            const int base = v * 16 + 4 * kg;
            a[j] = *reinterpret_cast<const short4_t *>(ain + (base + (ok[j] ? off : 0)));
            d[j] = *reinterpret_cast<const short4_t *>(dz + base);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const short4_t zero = {0, 0, 0, 0};
            if (vb + 16 * j < vend) acc = mma(tr(ok[j] ? a[j] : zero), tr(in[j] ? d[j] : zero), acc);
        }
    }
    // lane (co = i): ci = 4 kg + r, stored [ci][co]
    float *o = part + (((size_t)t * nchunk + c) * 16 + 4 * kg) * 16 + i;
#pragma unroll
    for (int r = 0; r < 4; r++) o[16 * r] = acc[r];
}

// the sum of squared errors from the tiles' partials, by a block; dred: 256 doubles
__device__ __forceinline__ void loss_sum(int ntile, const float *__restrict__ lpart, double *dred, double *__restrict__ hloss)
{
    const int tid = threadIdx.x;
    double s = 0.0;
#pragma unroll 16
    for (int i = tid; i < ntile; i += 256) s += lpart[i];
    dred[tid] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) dred[tid] += dred[tid + o];
        __syncthreads();
    }
    if (tid == 0) *hloss = dred[0];
}
// place in a layer's parameters: tid = ci*16 + co of tap t, co of the bias (t = 27)
__device__ __forceinline__ size_t param_at(int l, int t, int tid)
{
    return (size_t)l * LAYER_P + (t < 27 ? t * 256 + (tid & 15) * 16 + (tid >> 4) : LAYER_W + tid);
}

// The sums over chunks (in order), every layer in one launch (grid.y = layer):
// blocks 0..26 one tap of the weights, grad W[t][co][ci] = sum_c part[t][c][ci][co];
// block 27 the bias, and for layer 0 block 28 the sum of the loss partials (in
// FP64).  The gradients go to the device copy and, where the caller takes them
// (hG), straight to pinned host memory.
__global__ __launch_bounds__(256) void k_grad_reduce(int nchunk, const float *__restrict__ part, const float *__restrict__ bpart,
                                                     int ntile, const float *__restrict__ lpart, float *__restrict__ G,
                                                     float *__restrict__ hG, double *__restrict__ hloss)
{
    __shared__ double dred[256];
    const int l = blockIdx.y, t = blockIdx.x, tid = threadIdx.x;
    if (t == 28) {
        if (l == 0) loss_sum(ntile, lpart, dred, hloss);
        return;
    }
    const int n = t < 27 ? 256 : 16;
    if (tid >= n) return;
    const float *p = t < 27 ? part + (((size_t)l * 27 + t) * nchunk) * 256 + tid : bpart + (size_t)l * nchunk * 16 + tid;
    float s = 0.f;
#pragma unroll 16
    for (int c = 0; c < nchunk; c++) s += p[(size_t)c * n];
    const size_t o = param_at(l, t, tid);
    G[o] = s;
    if (hG) hG[o] = s;
}

// Column sums of n rows in order, for thread tid < COLS: 256 rows a round, 64 of
// each wave in flight while the round before is added from LDS (st: 256 COLS floats)
template <int COLS>
__device__ __forceinline__ float staged_sum(const float *__restrict__ p, int stride, int n, float *st)
{
    constexpr int RPL = 64 / COLS;   // rows of one load of a wave
    const int tid = threadIdx.x, lane = tid & 63, col = lane % COLS, r0 = (tid & ~63) + lane / COLS;
    float e[COLS], s = 0.f;
    auto load = [&](int c0) {
#pragma unroll
        for (int j = 0; j < COLS; j++) {
            const int row = c0 + r0 + RPL * j;
            e[j] = p[(size_t)(row < n ? row : n - 1) * stride + col];
        }
    };
    load(0);
    for (int c0 = 0; c0 < n; c0 += 256) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < COLS; j++) st[(r0 + RPL * j) * COLS + col] = e[j];
        __syncthreads();
        if (c0 + 256 < n) load(c0 + 256);
        if (tid < COLS) {
            const int m = n - c0 < 256 ? n - c0 : 256;
#pragma unroll 16
            for (int r = 0; r < m; r++) s += st[r * COLS + tid];
        }
    }
    return s;
}

// The same sums for one layer (part holds that layer's alone): four blocks per
// tap, of 64 columns each, then the bias and, for layer 0, the loss.  Bound by the
// load latency of few waves: as 28 blocks of 64 loads a thread a training step at
// 128x256x256 (upload included) took 28.8 to 28.9 ms, 27.1 to 27.8 here, 27.2 to
// 28.3 with the partials of all layers.
__global__ __launch_bounds__(256) void k_grad_reduce_layer(int l, int nchunk, const float *__restrict__ part,
                                                           const float *__restrict__ bpart, int ntile, const float *__restrict__ lpart,
                                                           float *__restrict__ G, float *__restrict__ hG, double *__restrict__ hloss)
{
    __shared__ __attribute__((aligned(8))) float st[256 * 64];
    const int b = blockIdx.x, tid = threadIdx.x;
    float s;
    size_t o;
    if (b < 4 * 27) {
        const int t = b / 4, c0 = 64 * (b % 4);
        s = staged_sum<64>(part + (size_t)t * nchunk * 256 + c0, 256, nchunk, st);
        if (tid >= 64) return;
        o = param_at(l, t, c0 + tid);
    } else if (b == 4 * 27) {
        s = staged_sum<16>(bpart + (size_t)l * nchunk * 16, 16, nchunk, st);
        if (tid >= 16) return;
        o = param_at(l, 27, tid);
    } else {
        if (l == 0) loss_sum(ntile, lpart, reinterpret_cast<double *>(st), hloss);
        return;
    }
    G[o] = s;
    if (hG) hG[o] = s;
}

// FP32 input [V][cin] -> BF16 [V][16], zero padded
__global__ void k_pack_input(int V, int cin, const float *__restrict__ x, uint16_t *__restrict__ a)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= V * 16) return;
    const int v = id >> 4, c = id & 15;
    a[id] = c < cin ? f2bf(x[(size_t)v * cin + c]) : (uint16_t)0;
}

// BF16 copies of the master weights: W[l][t][co][ci] and WT[l][t][ci][co]
__global__ void k_pack_weights(int nl, const float *__restrict__ P, uint16_t *__restrict__ Wb, uint16_t *__restrict__ WTb)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;   // l*6912 + t*256 + co*16 + ci
    if (id >= nl * LAYER_W) return;
    const int l = id / LAYER_W, r = id - l * LAYER_W, t = r >> 8, co = (r >> 4) & 15, ci = r & 15;
    const uint16_t b = f2bf(P[(size_t)l * LAYER_P + r]);
    Wb[id] = b;
    WTb[(size_t)l * LAYER_W + t * 256 + ci * 16 + co] = b;
}

// Adam (bias-corrected), FP32 master parameters
__global__ void k_adam(int64_t n, float lr, float b1, float b2, float eps, float c1, float c2, float *__restrict__ P,
                       const float *__restrict__ G, float *__restrict__ M, float *__restrict__ S)
{
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const float g = G[id];
    const float m = b1 * M[id] + (1.f - b1) * g;
    const float s = b2 * S[id] + (1.f - b2) * g * g;
    M[id] = m;
    S[id] = s;
    P[id] -= lr * (m / c1) / (sqrtf(s / c2) + eps);
}

__global__ void k_selftest_bf16(float *out)
{
    const int l = threadIdx.x, i = l & 15, kg = l >> 4;
    short4_t a, b;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = 4 * kg + j;
        a[j] = (short)f2bf(1.f + (float)i + 0.25f * (float)k);   // A[i][k]
        b[j] = (short)f2bf(2.f - 0.5f * (float)i + (float)k);    // B[k][n = i]
    }
    const float4_t d = mma(a, b, (float4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; r++) out[r * 64 + l] = d[r];
}

// ---------------------------------------------------------------- launchers
static Shape shape(const Net &n, int layer)
{
    const int d = n.dil[layer];
    auto recip = [](uint64_t q) { return q > 1 ? ~0ull / q + 1 : 0ull; };   // ceil(2^64 / q)
    return {n.nx, n.ny, n.nz, d < n.nx ? d : n.nx, d < n.ny ? d : n.ny, d < n.nz ? d : n.nz, recip((uint64_t)n.ny * n.nz), recip(n.nz)};
}

hipError_t conv_forward(const Net &n, int layer, const uint16_t *ain, uint16_t *aout, float *yout, hipStream_t s)
{
    const int V = n.nx * n.ny * n.nz;
    const dim3 g((unsigned)((V + 63) / 64)), b(256);
    const uint16_t *W = n.Wb + (size_t)layer * LAYER_W;
    const float *bias = n.P + (size_t)layer * LAYER_P + LAYER_W;
    if (layer < NL - 1)
        hipLaunchKernelGGL(k_conv<FWD_RELU>, g, b, 0, s, shape(n, layer), ain, W, bias, nullptr, aout, nullptr, nullptr, 16);
    else
        hipLaunchKernelGGL(k_conv<FWD_LAST>, g, b, 0, s, shape(n, layer), ain, W, bias, nullptr, nullptr, yout, nullptr, n.cout);
    return hipGetLastError();
}

hipError_t conv_loss(const Net &n, const uint16_t *ain, const float *tg, uint16_t *dz, hipStream_t s)
{
    const int V = n.nx * n.ny * n.nz, l = NL - 1;
    hipLaunchKernelGGL(k_conv<FWD_LOSS>, dim3((unsigned)((V + 63) / 64)), dim3(256), 0, s, shape(n, l), ain,
                       n.Wb + (size_t)l * LAYER_W, n.P + (size_t)l * LAYER_P + LAYER_W, tg, dz, nullptr, n.lpart, n.cout);
    return hipGetLastError();
}

hipError_t layer_back(const Net &n, int layer, const uint16_t *ain, const uint16_t *dz, uint16_t *dzprev, hipStream_t s)
{
    const int V = n.nx * n.ny * n.nz, ncb = dzprev ? (V + 63) / 64 : 0, nb = ncb + 7 * n.nchunk;
    float *part = n.part + (n.part_layers == NL ? (size_t)layer * 27 * n.nchunk * 256 : 0), *bpart = n.bpart + (size_t)layer * n.nchunk * 16;
    if (dzprev)
        hipLaunchKernelGGL(k_back<true>, dim3((unsigned)nb), dim3(256), 0, s, shape(n, layer), ncb, ain, dz,
                           n.WTb + (size_t)layer * LAYER_W, dzprev, n.nchunk, part, bpart);
    else
        hipLaunchKernelGGL(k_back<false>, dim3((unsigned)nb), dim3(256), 0, s, shape(n, layer), 0, ain, dz, nullptr, nullptr,
                           n.nchunk, part, bpart);
    return hipGetLastError();
}

hipError_t grad_reduce(const Net &n, int layer, float *hG, double *hloss, hipStream_t s)
{
    const int V = n.nx * n.ny * n.nz, ntile = (V + 15) / 16;
    if (n.part_layers == NL)
        hipLaunchKernelGGL(k_grad_reduce, dim3(29, NL), dim3(256), 0, s, n.nchunk, n.part, n.bpart, ntile, n.lpart, n.G, hG, hloss);
    else
        hipLaunchKernelGGL(k_grad_reduce_layer, dim3(4 * 27 + 2), dim3(256), 0, s, layer, n.nchunk, n.part, n.bpart, ntile, n.lpart, n.G, hG,
                           hloss);
    return hipGetLastError();
}

hipError_t pack_input(const Net &n, const float *x, uint16_t *a, hipStream_t s)
{
    const int V = n.nx * n.ny * n.nz;
    hipLaunchKernelGGL(k_pack_input, dim3((unsigned)((V * 16 + 255) / 256)), dim3(256), 0, s, V, n.cin, x, a);
    return hipGetLastError();
}

hipError_t pack_weights(const Net &n, hipStream_t s)
{
    hipLaunchKernelGGL(k_pack_weights, dim3((unsigned)((NL * LAYER_W + 255) / 256)), dim3(256), 0, s, NL, n.P, n.Wb, n.WTb);
    return hipGetLastError();
}

hipError_t adam(const Net &n, float lr, float c1, float c2, hipStream_t s)
{
    const int64_t np = (int64_t)NL * LAYER_P;
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, s, np, lr, ADAM_B1, ADAM_B2, ADAM_EPS, c1, c2, n.P,
                       n.G, n.M, n.S);
    return hipGetLastError();
}

hipError_t selftest_bf16(float *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_selftest_bf16, dim3(1), dim3(64), 0, s, out);
    return hipGetLastError();
}

}  // namespace ws
}  // namespace igap
