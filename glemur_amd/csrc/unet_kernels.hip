// Device kernels of the warm-start U-Net.  Convolutions are implicit GEMMs
// on the gfx950 bf16 matrix instruction v_mfma_f32_16x16x32_bf16 (16 x 16
// outputs, K = 32 per instruction, FP32 accumulation): rows are output
// points, columns output channels, K the (tap, input channel) pairs.  A lane
// supplies row (lane & 15) of A and column (lane & 15) of B over
// k = 8 (lane >> 4) .. +7, and receives column (lane & 15), rows
// 4 (lane >> 4) .. +3 of the result.
#include "unet_kernels.hpp"

#include <algorithm>
#include <cmath>

namespace gmu {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf2f(bf16_t h) { return __uint_as_float((uint32_t)h << 16); }

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// two floats -> two bfloat16 in a word, round to nearest even (NaN stays NaN)
__device__ inline uint32_t f2bf2(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

__device__ inline u32x4 ld16(const bf16_t *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ inline void st16(bf16_t *p, u32x4 v) { *reinterpret_cast<u32x4 *>(p) = v; }
__device__ inline bf16x8 as_bf(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ inline float lo16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ inline float hi16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ inline void unpack8(u32x4 v, float *f)
{
    for (int e = 0; e < 4; ++e) {
        f[2 * e] = lo16(v[e]);
        f[2 * e + 1] = hi16(v[e]);
    }
}
__device__ inline u32x4 pack8(const float *f)
{
    u32x4 v;
    for (int e = 0; e < 4; ++e) v[e] = f2bf2(f[2 * e], f[2 * e + 1]);
    return v;
}

__device__ inline void decomp(long long p, int nx, int ny, int &x, int &y, int &z)
{
    x = (int)(p % nx);
    long long q = p / nx;
    y = (int)(q % ny);
    z = (int)(q / ny);
}

// Logical index of workgroup b of n: the eight XCDs (workgroups go to them in
// turn) get contiguous runs, whose halos share lines in their L2
__device__ inline int xcd_run(int b, int n)
{
    const int q = n / 8, r = n % 8, x = b % 8;
    return x * q + min(x, r) + b / 8;
}

// ------------------------------------------------------------------ conv
// Workgroup: a box of 8 x 4 x BZ output points (BZ = MTW WM / 2) and
// 16 NTW WN output channels; WM waves along the points, WN along the
// channels, each with MTW x NTW tiles of 16 points x 16 channels in FP32
// accumulators.  The box's input with a one-point halo, all CIN channels,
// is staged in LDS once and serves the 27 taps by constant row offsets
// (rows outside the grid hold zeros, so no test runs per tap).  A row is 16
// bytes longer than its channels, an odd number of 16-byte words, and a y of
// rows is rounded up to half a turn of the banks past a whole number of
// them: the sixteen points of a tile, eight x of two y, lie on different
// banks.  A thread's staged words differ only in z (and y in a few steps), so
// the grid tests cost next to nothing.  The weights come in the order the lanes take them
// (k_pack), 1 KB a tile and step, straight from memory (L1, L2) into a ring
// of registers kRing steps ahead, the points from LDS one step ahead; the
// scheduling barriers hold the loads where they are written.  The weights are
// the first operand and the points the second, so a lane ends up with four
// consecutive channels of one point and stores them in 8 bytes.
// K runs as (tap, channel) in steps of 32 whatever the layer, one
// accumulator per output: every output is the same sum in the same order
// for any box.
// What bounds it: LDS and L1 reads against the matrix pipe, about even at 32
// output channels (MTW LDS and NTW L1 reads of 1 KB for MTW NTW matrix
// instructions a step); at the coarsest level the few hundred workgroups.
// 65 x 65 x 193, all layers and input gradients of a sample: 5.0 ms with
// operands loaded straight from memory per tap and a grid test per tap and
// lane; 1.6 ms from LDS boxes, but with the weight loads moved down to their
// use by the compiler, a wait for memory every step; 1.2 ms with them held
// (96 -> 32 channels 289 -> 223 us, 192 -> 64 189 -> 108, 128 -> 128 65 -> 36,
// 64 -> 64 41 -> 28, 32 -> 32 77 -> 64).
constexpr int CBX = 8, CBY = 4;                   // box, z planes by the variant
constexpr int CPX = CBX + 2, CPY = CBY + 2;       // halo points per y, y per z
// LDS layout, in 16-byte words: a point, a y and a z of the halo
constexpr int conv_pw(int cin) { return cin == 8 ? 1 : cin / 8 + 1; }
constexpr int conv_yw(int cin) { return (CPX * conv_pw(cin) + 7) / 16 * 16 + 8; }
constexpr int conv_zw(int cin) { return CPY * conv_yw(cin); }

// What becomes of a sum: bias and ReLU (a layer), the bias alone in FP32 (the
// head), nothing or the ReLU's derivative of `mask` (input gradients)
enum ConvEnd { kRelu, kHead, kPlain, kMask };

template <int CIN, int NTW, int WN, int MTW, int WM, int END>
__global__ __launch_bounds__(64 * WN * WM) __attribute__((amdgpu_waves_per_eu(CIN == 192 ? 1 : CIN == 128 ? 2 : 3))) void k_conv(ConvArgs a)
{
    static_assert(MTW % 2 == 0, "two tiles of 16 points make one z plane of the box");
    constexpr int NT = 64 * WN * WM, BZ = MTW * WM / 2, KS = (27 * CIN + 31) / 32, CW = CIN / 8;
    constexpr int PW = conv_pw(CIN), YW = conv_yw(CIN), ZW = conv_zw(CIN), ZERO = ZW * (BZ + 2);
    static_assert(YW >= CPX * PW && YW % 16 == 8);
    extern __shared__ u32x4 Xs[];   // [BZ + 2][CPY][CPX][PW], then two words of zeros
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, r16 = lane & 15;
    const int wn = wave % WN, wm = wave / WN;
    const int nbx = (a.nx + CBX - 1) / CBX, nby = (a.ny + CBY - 1) / CBY;
    const int box = xcd_run(blockIdx.x, gridDim.x);
    const int x0 = box % nbx * CBX, y0 = box / nbx % nby * CBY, z0 = box / (nbx * nby) * BZ;
    const u32x4 zero = {0u, 0u, 0u, 0u};

    // this wave's weights: tile nt of step s at ((s * tiles + nt) * 64 + lane) * 8
    const int nt0 = (blockIdx.y * WN + wn) * NTW;
    const long long wstep = (long long)(a.coutp / 16) * 512;
    const int wlane = (nt0 * 64 + lane) * 8;
    // steps ahead: nine (a z plane of taps) where a step is two tiles, three
    // where it is more or the masks take the registers (nine spilled there:
    // 32 -> 32 channels 87 us against 64); all of the few steps of 8 and 16
    // channels
    constexpr int kRing = CIN < 32 ? KS : NTW <= 2 && !(END == kMask && MTW == 4) ? 9 : 3;
    // staging: LN lanes take one y of the halo, 16 bytes each, YR of them at a time
    constexpr int LN = CPX * CW, Y1 = NT / LN, YR = Y1 >= CPY ? Y1 / CPY * CPY : Y1 >= 3 ? 3 : Y1;
    constexpr int NS = (CPY * (BZ + 2) + YR - 1) / YR;
    static_assert(YR > 0 && (CPY % YR == 0 || YR % CPY == 0), "a thread's y repeats");
    // (every lane loads, from the array's start where its point lies outside: a
    // branch per load would wait for each)
    u32x4 v[NS];
    const int sy = tid / LN, sx = tid % LN / CW, sc = tid % CW, gx = x0 - 1 + sx;
    const bool sok = sy < YR && gx >= 0 && gx < a.nx;
    auto inside = [&](int yz) {
        const int y = y0 - 1 + yz % CPY, z = z0 - 1 + yz / CPY;
        return sok && yz < CPY * (BZ + 2) && y >= 0 && y < a.ny && z >= 0 && z < a.nz;
    };
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int yz = s * YR + sy, y = y0 - 1 + yz % CPY, z = z0 - 1 + yz / CPY;
        const long long p = gx + (long long)a.nx * (y + (long long)a.ny * z);
        v[s] = ld16(a.in + (inside(yz) ? p * a.ldi + 8 * sc : 0));
    }
    // the lane's output points
    const int ox = x0 + (r16 & 7), co = 16 * nt0 + 4 * g;
    long long op[MTW];
    bool ook[MTW];
#pragma unroll
    for (int m = 0; m < MTW; ++m) {
        const int y = y0 + (r16 >> 3) + 2 * (m & 1), z = z0 + wm * (MTW / 2) + (m >> 1);
        ook[m] = ox < a.nx && y < a.ny && z < a.nz;
        op[m] = ook[m] ? ox + (long long)a.nx * (y + (long long)a.ny * z) : 0;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int yz = s * YR + sy;
        if (sy < YR && yz < CPY * (BZ + 2)) Xs[yz * YW + sx * PW + sc] = inside(yz) ? v[s] : zero;
    }
    bf16x8 W[kRing][NTW];
#pragma unroll
    for (int s = 0; s < kRing; ++s)
#pragma unroll
        for (int n = 0; n < NTW; ++n) W[s][n] = as_bf(ld16(a.w + s * wstep + wlane + 512 * n));
    // the ReLU masks of the lane's outputs, ready when the sums are
    u32x2 mask[END == kMask ? MTW : 1][NTW];
    if constexpr (END == kMask)
#pragma unroll
        for (int m = 0; m < MTW; ++m)
#pragma unroll
            for (int n = 0; n < NTW; ++n)
                mask[m][n] = *reinterpret_cast<const u32x2 *>(a.mask + op[m] * a.ldm + co + 16 * n);
    if (CIN < 32 && tid < 2) Xs[ZERO + tid] = zero;
    __syncthreads();

    f32x4 acc[MTW][NTW];
#pragma unroll
    for (int m = 0; m < MTW; ++m)
#pragma unroll
        for (int n = 0; n < NTW; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // word of the lane's point in the wave's first tile; tile m lies two y (m & 1) and m >> 1 z on
    const int lrow = PW * (r16 & 7) + YW * (r16 >> 3) + ZW * (wm * (MTW / 2));
    auto mrow = [](int m) { return 2 * YW * (m & 1) + ZW * (m >> 1); };
    if constexpr (CIN < 32) {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int t = CIN == 8 ? 4 * s + g : 2 * s + (g >> 1), c = CIN == 8 ? 0 : g & 1;
            const int trow = PW * (t % 3) + YW * (t / 3 % 3) + ZW * (t / 9) + c;
#pragma unroll
            for (int m = 0; m < MTW; ++m) {
                const bf16x8 X = as_bf(Xs[t < 27 ? lrow + mrow(m) + trow : ZERO + c]);
#pragma unroll
                for (int n = 0; n < NTW; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[s][n], X, acc[m][n], 0, 0, 0);
            }
        }
    } else {
        // A step's points are read from LDS one step ahead and its weights
        // loaded kRing steps ahead; the scheduling barriers keep them there
        // (left to itself the compiler moves a load down to its use, and
        // every step waits for memory).
        constexpr int CC = CIN / 32, QN = 9 * CC;
        static_assert(QN % kRing == 0 && KS == 3 * QN);
        const u32x4 *xl = Xs + lrow + g;
        auto at = [](int q) { return PW * (q / CC % 3) + YW * (q / CC / 3) + 4 * (q % CC); };
        bf16x8 X[2][MTW];
#pragma unroll
        for (int m = 0; m < MTW; ++m) X[0][m] = as_bf(xl[mrow(m)]);
        // (the last kRing steps load past the weights, into the array's
        // padding, and the last one reads its points again)
        const bf16_t *wr = a.w + kRing * wstep;
#pragma unroll 1
        for (int tz = 0; tz < 3; ++tz) {
            const u32x4 *xn = tz < 2 ? xl + ZW : xl;
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                // (after an odd number of steps the next points lie in X[1])
                bf16x8(&Xq)[MTW] = X[q & 1], (&Xp)[MTW] = X[(q + 1) & 1];
#pragma unroll
                for (int m = 0; m < MTW; ++m)
                    Xp[m] = as_bf(q + 1 < QN ? xl[at(q + 1) + mrow(m)] : xn[mrow(m)]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < MTW; ++m)
#pragma unroll
                    for (int n = 0; n < NTW; ++n)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[q % kRing][n], Xq[m], acc[m][n], 0, 0, 0);
#pragma unroll
                for (int n = 0; n < NTW; ++n) W[q % kRing][n] = as_bf(ld16(wr + q * wstep + wlane + 512 * n));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (QN & 1)
#pragma unroll
                for (int m = 0; m < MTW; ++m) X[0][m] = X[1][m];
            wr += QN * wstep;
            xl = xn;
        }
    }

    f32x4 bias[NTW];
    if constexpr (END == kRelu || END == kHead)
#pragma unroll
        for (int n = 0; n < NTW; ++n) bias[n] = *reinterpret_cast<const f32x4 *>(a.bias + co + 16 * n);
#pragma unroll
    for (int m = 0; m < MTW; ++m) {
        if (!ook[m]) continue;
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
            f32x4 v = acc[m][n];
            if constexpr (END == kRelu || END == kHead) v += bias[n];
            if constexpr (END == kHead) {
                *reinterpret_cast<f32x4 *>(a.outf + op[m] * a.ldf + co + 16 * n) = v;
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (END == kRelu) v[e] = v[e] > 0.f ? v[e] : 0.f;
                if constexpr (END == kMask)
                    v[e] = (e & 1 ? hi16(mask[m][n][e >> 1]) : lo16(mask[m][n][e >> 1])) > 0.f ? v[e] : 0.f;
            }
            *reinterpret_cast<u32x2 *>(a.out + op[m] * a.ldo + co + 16 * n) = u32x2{f2bf2(v[0], v[1]), f2bf2(v[2], v[3])};
        }
    }
}

// Weights of a layer as k_conv's lanes take them, rounded to bfloat16: tile
// nt of step s holds for lane l row 16 nt + (l & 15), k = 32 s + 8 (l >> 4)
// .. + 7.  wf: rows co, k = t cin + ci.  wb, the input gradient's: rows ci,
// k = t' coutp + co with the flipped tap 26 - t' (zero past 27 coutp).
__global__ void k_pack(const float *w, int coutp, int cin, int kpad, bf16_t *wf, bf16_t *wb, int kpadT)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;   // one lane of one tile
    const int nf = coutp * kpad / 8, nb = wb ? cin * kpadT / 8 : 0;
    if (i >= nf + nb) return;
    const bool fwd = i < nf;
    const int j = fwd ? i : i - nf, tiles = (fwd ? coutp : cin) / 16;
    const int l = j & 63, row = 16 * ((j >> 6) % tiles) + (l & 15), k = 32 * ((j >> 6) / tiles) + 8 * (l >> 4);
    float v[8];
    for (int e = 0; e < 8; ++e) {
        if (fwd) {
            v[e] = w[(long long)row * kpad + k + e];
        } else {
            const int t = (k + e) / coutp, co = (k + e) % coutp;
            v[e] = t < 27 ? w[(long long)co * kpad + (26 - t) * cin + row] : 0.f;
        }
    }
    st16((fwd ? wf : wb) + (long long)j * 8, pack8(v));
}

// ------------------------------------------------------------- weight grad
// Workgroup: one chunk of 2048 consecutive points, one z plane of nine taps
// and one block of 16 MCO output by 16 NCI input channels; each of its three
// waves owns the three taps of one y and keeps their FP32 accumulators over
// the chunk, so both tensors are staged once for nine taps.  K runs over
// points, 32 consecutive ones a step, and the chunks' partials are summed in
// turn (k_wgrad_sum): the order of the sum depends on nothing but the grid.
// Both operands lie in LDS point by point as in memory (16 channels, 32
// bytes a row) and ds_read_b64_tr_b16 hands each lane four consecutive
// points of its channel.  A wave stages the input rows of its y: those of
// the tile's points in order, with one row of zeros from each grid row to
// the next (x = -1 and x = nx share it) and zeros where y or z lies outside,
// so a point's row is its index plus the grid rows begun since the tile's
// first point, the three taps are constant row offsets, and no test runs per
// tap.
// What bounds it: the LDS reads (2 MCO + 6 NCI reads of 512 bytes for 3 MCO
// NCI matrix instructions a step) beside the staging's address arithmetic
// and latency, which the workgroups a CU holds cover.  Weight and bias
// gradients of all eleven layers of a 65 x 65 x 193 sample, sums included:
// 13.2 -> 1.4 ms against one workgroup per (chunk, tap, 64 x 64 block), which
// read both tensors once a tap and transposed them by 2-byte LDS stores
constexpr int WCHUNK = 2048;   // points a workgroup sums
constexpr int WT = 96;         // points of a tile: 64 and 128 are 5 to 15% slower (latency; two waves a SIMD for registers)

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ inline s16x4 ld_points(const bf16_t *p)
{
    typedef __attribute__((address_space(3))) s16x4 *lp;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p));
}
__device__ inline bf16x8 join(s16x4 a, s16x4 b)
{
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Input rows of a tile and y: the points, a row of zeros per grid row begun,
// and one row on either side
__host__ __device__ constexpr int wgrad_rows(int nx) { return WT + (WT - 1) / nx + 3; }

// floor(v / n) of 0 <= v < 2^20, n > 0 with inv = 1 / n: (v + 1/2) / n is at
// least 1/(2n) away from a whole number, the roundings move it by at most
// (v + 1/2) 2^-22 / n
__device__ inline int small_div(int v, float inv) { return (int)(((float)v + 0.5f) * inv); }

// Bias gradient partials of 4096 points, by workgroups of the weight
// gradient's launch: a value per channel and k < ph = 256 / c sums the points
// k, k + ph, ... in turn, and the ph sums are added in turn.  A workgroup
// takes 32 channels and stages 384 points of them in LDS at a time, the next
// ones on their way meanwhile; a thread has two of the 256 sums at most.  Its
// chain of loads (20 us a layer as a launch of 200 workgroups) passes beside
// the matrix work.
constexpr int BG_CHUNK = 4096, BG_PTS = 384, BG_CH = 32;
constexpr int kBiasLds = BG_PTS * BG_CH * 2 + 256 * 4;

__device__ inline void bias_part(const WgradArgs &a, bf16_t *st, int chunk, int c0)
{
    float *red = reinterpret_cast<float *>(st + BG_PTS * BG_CH);
    const int c = a.cout, w = c < BG_CH ? c : BG_CH, ph = 256 / c, cw = w / 8;
    const int ch = threadIdx.x % w, k0 = threadIdx.x / w, k1 = k0 + 192 / w;
    const int P = a.nx * a.ny * a.nz, p0 = chunk * BG_CHUNK, p1 = min(p0 + BG_CHUNK, P);
    constexpr int NL = BG_PTS * BG_CH / 8 / 192;
    u32x4 v[NL];
    auto load = [&](int pb) {
        const int n = min(BG_PTS, p1 - pb) * cw;
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int q = min((int)threadIdx.x + 192 * u, n - 1);
            v[u] = ld16(a.g + (long long)(pb + q / cw) * c + c0 + 8 * (q % cw));
        }
    };
    float s0 = 0.f, s1 = 0.f;
    auto sum = [&](int k, int n, float &s) {
        int i = k;
        for (; i + 15 * ph < n; i += 16 * ph) {
            bf16_t e[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) e[u] = st[(i + u * ph) * w + ch];
#pragma unroll
            for (int u = 0; u < 16; ++u) s += bf2f(e[u]);
        }
        for (; i < n; i += ph) s += bf2f(st[i * w + ch]);
    };
    load(p0);
    for (int pb = p0; pb < p1; pb += BG_PTS) {
        const int n = min(BG_PTS, p1 - pb);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int q = threadIdx.x + 192 * u;
            if (q < n * cw) st16(st + 8 * q, v[u]);
        }
        __syncthreads();
        if (pb + BG_PTS < p1) load(pb + BG_PTS);
        if (k0 < ph) sum(k0, n, s0);
        if (k1 < ph) sum(k1, n, s1);
    }
    if (k0 < ph) red[k0 * w + ch] = s0;
    if (k1 < ph) red[k1 * w + ch] = s1;
    __syncthreads();
    if ((int)threadIdx.x < w) {
        float s = red[ch];
        for (int j = 1; j < ph; ++j) s += red[j * w + ch];
        a.bpart[(long long)chunk * c + c0 + ch] = s;
    }
}

// MINNX: the smallest nx the variant takes, which bounds a tile's rows.  A
// level's nx is 2 or more (a grid of nx = 5 has levels of 5, 3 and 2); rows
// nobody stages would hold whatever LDS held before.
template <int MCO, int NCI, int MINNX>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(3))) void k_wgrad(WgradArgs a)
{
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];   // [3][NCI][rows][16] input, [MCO][WT][16] gradient, [3][rows] int
    const int rows = wgrad_rows(a.nx), xn = rows * 16;
    constexpr int gn = WT * 16;
    const int tid = threadIdx.x, lane = tid & 63, ty = tid >> 6, g = lane >> 4, r16 = lane & 15;
    bf16_t *Xs = lds + ty * NCI * xn, *Gs = lds + 3 * NCI * xn;
    // the first workgroups of the launch sum the bias gradient
    const int nbias = (a.cout + BG_CH - 1) / BG_CH, by = (int)blockIdx.y - nbias;
    if (by < 0) {
        if ((int)blockIdx.x * BG_CHUNK < a.nx * a.ny * a.nz) bias_part(a, lds, blockIdx.x, BG_CH * blockIdx.y);
        return;
    }
    const int tz = by % 3, blk = by / 3;
    const int nciB = (a.cin + 16 * NCI - 1) / (16 * NCI);
    const int co0 = blk / nciB * 16 * MCO, ci0 = blk % nciB * 16 * NCI;
    const int P = a.nx * a.ny * a.nz;
    const int chunk = xcd_run(blockIdx.x, gridDim.x);
    const int pbeg = chunk * WCHUNK, pend = min(pbeg + WCHUNK, P);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const float invx = 1.f / (float)(a.nx + 1), invx0 = 1.f / (float)a.nx, invy = 1.f / (float)a.ny;

    f32x4 acc[3][MCO][NCI];
#pragma unroll
    for (int j = 0; j < 3; ++j)
        for (int m = 0; m < MCO; ++m)
            for (int n = 0; n < NCI; ++n) acc[j][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int lch = 4 * (r16 & 3), lpt = 8 * g + (r16 >> 2);
    const int sc = lane % (2 * NCI), sr = lane / (2 * NCI);   // staging: 8-channel group and first row
    const bool cok = ci0 + 8 * sc < a.cin;
    const bf16_t *src = a.in + ci0 + 8 * sc;
    bf16_t *xst = Xs + (sc >> 1) * xn + 8 * (sc & 1);
    constexpr int RS = 32 / NCI;                              // rows a wave stages at a time
    // a tile's words on their way to LDS: loaded while the tile before is multiplied
    constexpr int NX = (wgrad_rows(MINNX) + RS - 1) / RS, NG = (WT * 2 * MCO + 191) / 192;
    u32x4 xv[NX], gv[NG];
    int *const tab = reinterpret_cast<int *>(lds + (3 * NCI * xn + MCO * gn)) + ty * rows;   // the wave's
    auto load = [&](int pb) {
        // the grid points of the rows (-1: zeros), one row a lane: worked out by
        // every lane for the rows it loads, this arithmetic took longer than the
        // matrix instructions
        const int rb = pb / a.nx, xb = pb - rb * a.nx, yb = rb % a.ny;   // first point: grid row, x and y
        for (int r = lane; r < rows; r += 64) {
            // row r is x = xb - 1 + r, counted on over rows of nx + 1
            const int X = xb + a.nx + r, q = small_div(X, invx), x = X - q * (a.nx + 1);
            const int Y = yb + q - 1 + a.ny, y = Y - small_div(Y, invy) * a.ny + ty - 1;   // q - 1 >= -1
            const int p = x + a.nx * (rb + q - 1 + ty - 1 + (tz - 1) * a.ny);
            tab[r] = x < a.nx && y >= 0 && y < a.ny && p >= 0 && p < P ? p : -1;
        }
        // a lane reads what other lanes of its wave wrote: LDS serves a wave in
        // order, the fence keeps the compiler from moving the reads up
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        int p[NX];
#pragma unroll
        for (int u = 0; u < NX; ++u) p[u] = tab[min(sr + u * RS, rows - 1)];
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            xv[u] = zero;
            if (cok && p[u] >= 0) xv[u] = ld16(src + p[u] * a.ldi);
        }
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const int q = tid + 192 * u, i = q / (2 * MCO), c = q % (2 * MCO), p = pb + i;
            gv[u] = zero;
            if (i < WT && p < pend) gv[u] = ld16(a.g + (long long)p * a.cout + co0 + 8 * c);
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int u = 0; u < NX; ++u)
            if (sr + u * RS < rows) st16(xst + (sr + u * RS) * 16, xv[u]);
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const int q = tid + 192 * u, i = q / (2 * MCO), c = q % (2 * MCO);
            if (i < WT) st16(Gs + (c >> 1) * gn + i * 16 + 8 * (c & 1), gv[u]);
        }
    };
    load(pbeg);
    for (int pb = pbeg; pb < pend; pb += WT) {
        const int xb = pb % a.nx;
        __syncthreads();
        store();
        __syncthreads();
        if (pb + WT < pend) load(pb + WT);
        auto step = [&](int s) {
            const int i = 32 * s + lpt;   // the lane's points i, i + 4
            const bf16_t *x1 = Xs + lch + 16 * (i + small_div(xb + i, invx0));
            const bf16_t *x2 = Xs + lch + 16 * (i + 4 + small_div(xb + i + 4, invx0));
            const bf16_t *gp = Gs + lch + 16 * i;
            bf16x8 A[MCO];
#pragma unroll
            for (int m = 0; m < MCO; ++m) A[m] = join(ld_points(gp + m * gn), ld_points(gp + m * gn + 64));
#pragma unroll
            for (int n = 0; n < NCI; ++n) {
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const bf16x8 B = join(ld_points(x1 + n * xn + 16 * j), ld_points(x2 + n * xn + 16 * j));
#pragma unroll
                    for (int m = 0; m < MCO; ++m)
                        acc[j][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[m], B, acc[j][m][n], 0, 0, 0);
                }
            }
        };
        const int steps = (min(WT, pend - pb) + 31) / 32;
#pragma unroll 1
        for (int s = 0; s < steps; ++s) step(s);
    }
    float *part = a.part + ((long long)blk * gridDim.x + chunk) * (27 * MCO * NCI * 256);
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int m = 0; m < MCO; ++m)
#pragma unroll
            for (int n = 0; n < NCI; ++n)
                *reinterpret_cast<f32x4 *>(part + (((9 * tz + 3 * ty + j) * MCO + m) * NCI + n) * 256 + 4 * lane) = acc[j][m][n];
}

// Sums of partials in turn, added to the layer's weight gradient, and (the
// last workgroups of the grid) to its bias gradient: 64 values a workgroup;
// its 256 threads load 64 partials of each into LDS, and one wave adds them
// in order while the next 64 are on their way
template <int MCO, int NCI>
__global__ __launch_bounds__(256) void k_wgrad_sum(WgradArgs a, int nchunks, int kpad, float *grad, int nbparts,
                                                   float *bgrad)
{
    __shared__ float st[2][64][64];
    constexpr int N = 27 * MCO * NCI * 256;
    const int col = threadIdx.x & 63, q = threadIdx.x >> 6;
    const bool bias = blockIdx.x == N / 64;
    const int i = blockIdx.x * 64 + col, bi = blockIdx.y * 64 + col;
    if (bias && (int)blockIdx.y * 64 >= a.cout) return;
    const int n = bias ? nbparts : nchunks;
    const long long ld = bias ? a.cout : N;
    const bool live = !bias || bi < a.cout;
    const float *p = bias ? a.bpart + bi : a.part + (long long)blockIdx.y * nchunks * N + i;
    float v[16], s = 0.f;
    auto load = [&](int c0) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = c0 + 4 * u + q;
            v[u] = live && c < n ? p[c * ld] : 0.f;
        }
    };
    load(0);
    for (int c0 = 0, b = 0; c0 < n; c0 += 64, b ^= 1) {
#pragma unroll
        for (int u = 0; u < 16; ++u) st[b][4 * u + q][col] = v[u];
        __syncthreads();
        if (c0 + 64 < n) load(c0 + 64);
        if (q == 0) {
            const int m = min(64, n - c0);
#pragma unroll 16
            for (int c = 0; c < m; ++c) s += st[b][c][col];
        }
    }
    if (q || !live) return;
    if (bias) {
        bgrad[bi] += s;
        return;
    }
    const int e = i & 3, lane = i >> 2 & 63, m = (i >> 8) / NCI % MCO, nn = (i >> 8) % NCI, t = (i >> 8) / (NCI * MCO);
    const int nciB = (a.cin + 16 * NCI - 1) / (16 * NCI);
    const int co = ((int)(blockIdx.y / nciB) * MCO + m) * 16 + 4 * (lane >> 4) + e;
    const int ci = ((int)(blockIdx.y % nciB) * NCI + nn) * 16 + (lane & 15);
    if (ci < a.cin) grad[(long long)co * kpad + t * a.cin + ci] += s;
}

// ------------------------------------------------------------ pool / up
__global__ void k_pool(const bf16_t *in, long long ldi, int nx, int ny, int nz, int c, bf16_t *out, long long ldo)
{
    const int cx = (nx + 1) / 2, cy = (ny + 1) / 2, cz = (nz + 1) / 2, ng = c / 8;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)cx * cy * cz * ng) return;
    const long long q = idx / ng;
    const int cg = (int)(idx % ng);
    int X, Y, Z;
    decomp(q, cx, cy, X, Y, Z);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int t = 0; t < 27; ++t) {
        const int x = 2 * X + t % 3 - 1, y = 2 * Y + (t / 3) % 3 - 1, z = 2 * Z + t / 9 - 1;
        if (x < 0 || x >= nx || y < 0 || y >= ny || z < 0 || z >= nz) continue;
        float v[8];
        unpack8(ld16(in + (x + (long long)nx * (y + (long long)ny * z)) * ldi + 8 * cg), v);
        for (int e = 0; e < 8; ++e) s[e] += v[e];
    }
    for (int e = 0; e < 8; ++e) s[e] /= 27.f;
    st16(out + q * ldo + 8 * cg, pack8(s));
}

__global__ void k_pool_bwd(const bf16_t *dP, long long ldp, int nx, int ny, int nz, int c, const bf16_t *skip,
                           long long lds, const bf16_t *mask, long long ldm, bf16_t *out, long long ldo)
{
    const int cx = (nx + 1) / 2, cy = (ny + 1) / 2, ng = c / 8;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)nx * ny * nz * ng) return;
    const long long p = idx / ng;
    const int cg = (int)(idx % ng);
    int x, y, z;
    decomp(p, nx, ny, x, y, z);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    // coarse Q with |2Q - f| <= 1: f/2 (f even) or (f-1)/2, (f+1)/2 (f odd)
    const int x0 = x >> 1, x1 = (x + 1) >> 1, y0 = y >> 1, y1 = (y + 1) >> 1, z0 = z >> 1, z1 = (z + 1) >> 1;
    for (int Z = z0; Z <= z1; ++Z)
        for (int Y = y0; Y <= y1; ++Y)
            for (int X = x0; X <= x1; ++X) {
                float v[8];
                unpack8(ld16(dP + (X + (long long)cx * (Y + (long long)cy * Z)) * ldp + 8 * cg), v);
                for (int e = 0; e < 8; ++e) s[e] += v[e];
            }
    float k[8], m[8];
    unpack8(ld16(skip + p * lds + 8 * cg), k);
    unpack8(ld16(mask + p * ldm + 8 * cg), m);
    for (int e = 0; e < 8; ++e) s[e] = m[e] > 0.f ? s[e] / 27.f + k[e] : 0.f;
    st16(out + p * ldo + 8 * cg, pack8(s));
}

__device__ inline void lin1(int f, int &i0, int &i1, float &w0, float &w1)
{
    if ((f & 1) == 0) { i0 = i1 = f >> 1; w0 = 1.f; w1 = 0.f; }
    else { i0 = (f - 1) >> 1; i1 = i0 + 1; w0 = 0.5f; w1 = 0.5f; }
}

__global__ void k_up(const bf16_t *in, long long ldi, int nx, int ny, int nz, int c, bf16_t *out, long long ldo)
{
    const int fx = 2 * nx - 1, fy = 2 * ny - 1, fz = 2 * nz - 1, ng = c / 8;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)fx * fy * fz * ng) return;
    const long long p = idx / ng;
    const int cg = (int)(idx % ng);
    int x, y, z;
    decomp(p, fx, fy, x, y, z);
    int ix[2], iy[2], iz[2];
    float wx[2], wy[2], wz[2];
    lin1(x, ix[0], ix[1], wx[0], wx[1]);
    lin1(y, iy[0], iy[1], wy[0], wy[1]);
    lin1(z, iz[0], iz[1], wz[0], wz[1]);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
            for (int e = 0; e < 2; ++e) {
                const float w = wx[e] * wy[b] * wz[a];
                if (w == 0.f) continue;
                float v[8];
                unpack8(ld16(in + (ix[e] + (long long)nx * (iy[b] + (long long)ny * iz[a])) * ldi + 8 * cg), v);
                for (int j = 0; j < 8; ++j) s[j] += w * v[j];
            }
    st16(out + p * ldo + 8 * cg, pack8(s));
}

__global__ void k_up_bwd(const bf16_t *dF, long long ldf, int nx, int ny, int nz, int c, const bf16_t *mask,
                         long long ldm, bf16_t *out, long long ldo)
{
    const int fx = 2 * nx - 1, fy = 2 * ny - 1, fz = 2 * nz - 1, ng = c / 8;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)nx * ny * nz * ng) return;
    const long long q = idx / ng;
    const int cg = (int)(idx % ng);
    int X, Y, Z;
    decomp(q, nx, ny, X, Y, Z);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int dz = -1; dz <= 1; ++dz) {
        const int z = 2 * Z + dz;
        if (z < 0 || z >= fz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            const int y = 2 * Y + dy;
            if (y < 0 || y >= fy) continue;
            for (int dx = -1; dx <= 1; ++dx) {
                const int x = 2 * X + dx;
                if (x < 0 || x >= fx) continue;
                const float w = (dx ? 0.5f : 1.f) * (dy ? 0.5f : 1.f) * (dz ? 0.5f : 1.f);
                float v[8];
                unpack8(ld16(dF + (x + (long long)fx * (y + (long long)fy * z)) * ldf + 8 * cg), v);
                for (int j = 0; j < 8; ++j) s[j] += w * v[j];
            }
        }
    }
    float m[8];
    unpack8(ld16(mask + q * ldm + 8 * cg), m);
    for (int j = 0; j < 8; ++j) s[j] = m[j] > 0.f ? s[j] : 0.f;
    st16(out + q * ldo + 8 * cg, pack8(s));
}

// ------------------------------------------------------------ loss, adam
constexpr int LOSS_PTS = 1024;   // points per workgroup (256 threads x 4)

__global__ __launch_bounds__(256) void k_loss(const float *y, const float *target, float inv_scale, long long P,
                                              bf16_t *g, double *part)
{
    __shared__ double red[256];
    double s = 0;
    const float gs = 2.f / (3.f * (float)P);
    for (int j = 0; j < 4; ++j) {
        const long long p = (long long)blockIdx.x * LOSS_PTS + j * 256 + threadIdx.x;
        if (p >= P) break;
        float v[16];
        for (int c = 0; c < 16; ++c) v[c] = 0.f;
        for (int c = 0; c < 3; ++c) {
            const float d = y[p * 16 + c] - target[p * 3 + c] * inv_scale;
            s += (double)d * d;
            v[c] = gs * d;
        }
        st16(g + p * 16, pack8(v));
        st16(g + p * 16 + 8, pack8(v + 8));
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// The partials in turn; 256 threads bring them into LDS (one thread's own
// loads, in turn too, took 50 us at 65 x 65 x 193)
__global__ __launch_bounds__(256) void k_loss_final(const double *part, int n, long long P, double *acc)
{
    __shared__ double st[256];
    double s = 0;
    for (int i0 = 0; i0 < n; i0 += 256) {
        __syncthreads();
        if (i0 + (int)threadIdx.x < n) st[threadIdx.x] = part[i0 + threadIdx.x];
        __syncthreads();
        const int m = min(256, n - i0);
        if (threadIdx.x == 0)
#pragma unroll 16
            for (int i = 0; i < m; ++i) s += st[i];
    }
    if (threadIdx.x == 0) acc[0] += s / (3.0 * (double)P);
}

__global__ void k_adam(float *w, const float *g, float *m, float *v, long long n, float gscale, float lr, float b1,
                       float b2, float eps, float c1, float c2)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] * gscale;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

__global__ void k_d2b(const double *in, long long n, bf16_t *out)
{
    const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 8;   // n: a multiple of 8
    if (i >= n) return;
    float v[8];
    for (int e = 0; e < 8; ++e) v[e] = (float)in[i + e];
    st16(out + i, pack8(v));
}
__global__ void k_d2f(const double *in, long long n, float *out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}
__global__ void k_scale_out(const float *y, long long n, double scale, double *out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // 3 p + c
    if (i < n) out[i] = scale * y[i / 3 * 16 + i % 3];
}
// Where parameter i of the caller's array lies in the device arrays
__device__ inline long long param_at(const ParamMap &m, long long i)
{
    int l = 0;
    while (i >= m.first[l + 1]) ++l;
    const int j = (int)(i - m.first[l]), row = j / m.k[l];
    return j < m.nw[l] ? m.at[l] + (long long)row * m.kpad[l] + (j - row * m.k[l]) : m.bias[l] + (j - m.nw[l]);
}
__global__ void k_params_out(ParamMap m, const float *src, double *out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m.first[kLayers]) out[i] = src[param_at(m, i)];
}
__global__ void k_params_in(ParamMap m, const double *in, float *dst)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m.first[kLayers]) dst[param_at(m, i)] = (float)in[i];
}

// ------------------------------------------------- context <-> network
__global__ void k_features(const double *B64, const float *B32, long long Pf, int fsx, long long fsxy, int stride,
                           int nx, int ny, int nz, bf16_t *feat)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)nx * ny * nz) return;
    int i, j, k;
    decomp(q, nx, ny, i, j, k);
    const long long gi = (stride * i + 1) + (long long)fsx * (stride * j + 1) + fsxy * (stride * k + 1);
    float f[8];
    for (int c = 0; c < 3; ++c) {
        const double b = B64 ? B64[c * Pf + gi] : (double)B32[3 * gi + c];   // FP32 B0: triples
        f[c] = (float)(c == 2 ? b - 1.0 : b);
    }
    f[3] = (float)(2.0 * i / (nx - 1) - 1.0);
    f[4] = (float)(2.0 * j / (ny - 1) - 1.0);
    f[5] = (float)(2.0 * k / (nz - 1) - 1.0);
    f[6] = f[7] = 0.f;
    st16(feat + q * 8, pack8(f));
}

__global__ void k_target(const double *X64, const float *Xh, const float *Xl, long long Pf, int fsx, long long fsxy,
                         int nx, int ny, int nz, double Ox, double Oy, double Oz, double dx, double dy, double dz,
                         float *target)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)nx * ny * nz) return;
    int i, j, k;
    decomp(q, nx, ny, i, j, k);
    const long long gi = (i + 1) + (long long)fsx * (j + 1) + fsxy * (k + 1);
    const double o[3] = {Ox + i * dx, Oy + j * dy, Oz + k * dz};
    for (int c = 0; c < 3; ++c) {
        const double x = X64 ? X64[c * Pf + gi] : (double)Xh[3 * gi + c] + (double)Xl[3 * gi + c];
        target[q * 3 + c] = (float)(x - o[c]);
    }
}

__global__ void k_apply(const float *y, int cnx, int cny, int cnz, int stride, double scale, double *X64, float *Xh,
                        float *Xl, long long Pf, int fsx, long long fsxy, int nx, int ny, int nz)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)nx * ny * nz) return;
    int i, j, k;
    decomp(q, nx, ny, i, j, k);
    int ix[2], iy[2], iz[2];
    float wx[2], wy[2], wz[2];
    if (stride == 2) {
        lin1(i, ix[0], ix[1], wx[0], wx[1]);
        lin1(j, iy[0], iy[1], wy[0], wy[1]);
        lin1(k, iz[0], iz[1], wz[0], wz[1]);
    } else {
        ix[0] = ix[1] = i; iy[0] = iy[1] = j; iz[0] = iz[1] = k;
        wx[0] = wy[0] = wz[0] = 1.f;
        wx[1] = wy[1] = wz[1] = 0.f;
    }
    double d[3] = {0, 0, 0};
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
            for (int e = 0; e < 2; ++e) {
                const double w = (double)wx[e] * wy[b] * wz[a];
                if (w == 0.0) continue;
                const float *s = y + (ix[e] + (long long)cnx * (iy[b] + (long long)cny * iz[a])) * 16;
                for (int c = 0; c < 3; ++c) d[c] += w * s[c];
            }
    const long long gi = (i + 1) + (long long)fsx * (j + 1) + fsxy * (k + 1);
    for (int c = 0; c < 3; ++c) {
        const double dc = scale * d[c];
        if (X64) {
            X64[c * Pf + gi] += dc;
        } else {
            const double x = (double)Xh[3 * gi + c] + (double)Xl[3 * gi + c] + dc;   // F32K: triples
            const float h = (float)x;
            Xh[3 * gi + c] = h;
            Xl[3 * gi + c] = (float)(x - (double)h);
        }
    }
    (void)cnz;
}

__global__ __launch_bounds__(256) void k_min_det(const double *det, int nx, int ny, int nz, int sx, long long sxy,
                                                 double *part)
{
    __shared__ double rmin[256];
    __shared__ int rnan[256];
    const long long N = (long long)nx * ny * nz;
    double mn = 1e300;
    int nan = 0;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < N; q += (long long)gridDim.x * 256) {
        int i, j, k;
        decomp(q, nx, ny, i, j, k);
        const double d = det[(i + 1) + (long long)sx * (j + 1) + sxy * (k + 1)];
        if (d != d) nan = 1;
        else if (d < mn) mn = d;
    }
    rmin[threadIdx.x] = mn;
    rnan[threadIdx.x] = nan;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            rmin[threadIdx.x] = fmin(rmin[threadIdx.x], rmin[threadIdx.x + w]);
            rnan[threadIdx.x] |= rnan[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = rmin[0];
        part[2 * blockIdx.x + 1] = rnan[0];
    }
}

__global__ __launch_bounds__(64) void k_min_det_final(const double *part, int n, double *out)
{
    double mn = 1e300;
    int nan = 0;
    for (int i = threadIdx.x; i < n; i += 64) {
        mn = fmin(mn, part[2 * i]);
        if (part[2 * i + 1] != 0) nan = 1;
    }
    for (int o = 32; o > 0; o >>= 1) mn = fmin(mn, __shfl_xor(mn, o, 64));
    nan = __any(nan);
    if (threadIdx.x != 0) return;
    out[0] = mn;
    out[1] = nan;
}

__global__ __launch_bounds__(256) void k_sumsq(const float *v, long long n, double *part)
{
    __shared__ double red[256];
    double s = 0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        s += (double)v[i] * v[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_sum_final(const double *part, int n, double *out)
{
    if (threadIdx.x != 0) return;
    double s = 0;
    for (int i = 0; i < n; ++i) s += part[i];
    out[0] = s;
}

inline unsigned nblk(long long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace

namespace {
template <int CIN, int NTW, int WN, int MTW, int WM, int END>
void launch_conv_k(hipStream_t s, const ConvArgs &a)
{
    constexpr int BZ = MTW * WM / 2, lds = 16 * (conv_zw(CIN) * (BZ + 2) + 2);
    static const hipError_t attr = hipFuncSetAttribute((const void *)k_conv<CIN, NTW, WN, MTW, WM, END>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)attr;
    const int boxes = ((a.nx + CBX - 1) / CBX) * ((a.ny + CBY - 1) / CBY) * ((a.nz + BZ - 1) / BZ);
    k_conv<CIN, NTW, WN, MTW, WM, END><<<dim3(boxes, a.coutp / (16 * NTW * WN)), 64 * WN * WM, lds, s>>>(a);
}
}  // namespace

// The network's layers and their input gradients: boxes of eight planes
// while the halo fits three workgroups a CU (32 channels, 54 KB of 160), of
// four or two above that; channels split over two waves, or two workgroups,
// where the box has few tiles of points.  Four tiles of points a wave at 192
// channels, one workgroup a CU: 131 -> 108 us at 33 x 33 x 97, 29 -> 24 at 17
// x 17 x 49.  The same at 96 and 128 channels gains 4 to 17% on the largest
// grid of a level and loses 9 to 80% on the smallest.
int launch_conv(hipStream_t s, const ConvArgs &a)
{
    const bool fwd = a.bias != nullptr;
    switch (a.cin * 1000 + a.coutp) {
    case 8032: launch_conv_k<8, 2, 1, 4, 4, kRelu>(s, a); return 0;
    case 16032: launch_conv_k<16, 2, 1, 4, 4, kMask>(s, a); return 0;
    case 32016: launch_conv_k<32, 1, 1, 4, 4, kHead>(s, a); return 0;
    case 32032:
        fwd ? launch_conv_k<32, 2, 1, 4, 4, kRelu>(s, a) : launch_conv_k<32, 2, 1, 4, 4, kMask>(s, a);
        return 0;
    case 32064: launch_conv_k<32, 4, 1, 4, 4, kRelu>(s, a); return 0;
    case 32096: launch_conv_k<32, 3, 2, 4, 2, kPlain>(s, a); return 0;
    case 64032: launch_conv_k<64, 2, 1, 2, 4, kPlain>(s, a); return 0;
    case 64064:
        fwd ? launch_conv_k<64, 2, 2, 4, 2, kRelu>(s, a) : launch_conv_k<64, 2, 2, 4, 2, kMask>(s, a);
        return 0;
    case 64128: launch_conv_k<64, 2, 2, 4, 2, kRelu>(s, a); return 0;
    case 64192: launch_conv_k<64, 3, 2, 4, 2, kPlain>(s, a); return 0;
    case 96032: launch_conv_k<96, 2, 1, 2, 4, kRelu>(s, a); return 0;
    case 128064: launch_conv_k<128, 2, 2, 2, 2, kPlain>(s, a); return 0;
    case 128128:
        fwd ? launch_conv_k<128, 2, 2, 2, 2, kRelu>(s, a) : launch_conv_k<128, 2, 2, 2, 2, kMask>(s, a);
        return 0;
    case 192064: launch_conv_k<192, 2, 2, 4, 2, kRelu>(s, a); return 0;
    }
    return -1;   // no layer of the network
}

namespace {
int wgrad_chunks(long long P) { return (int)((P + WCHUNK - 1) / WCHUNK); }
// channel blocks: 32 x 32, 16 wide where the layer has no more
int wgrad_mco(int cout) { return cout % 32 ? 1 : 2; }
int wgrad_nci(int cin) { return cin <= 16 ? 1 : 2; }
int wgrad_blocks(int cin, int cout)
{
    const int nci = 16 * wgrad_nci(cin);
    return cout / (16 * wgrad_mco(cout)) * ((cin + nci - 1) / nci);
}
template <int MCO, int NCI>
void launch_wgrad_k(hipStream_t s, const WgradArgs &a, int kpad, float *grad, float *bgrad)
{
    const int lds = std::max((3 * NCI * wgrad_rows(a.nx) + MCO * WT) * 32 + 3 * wgrad_rows(a.nx) * 4, kBiasLds);   // at most 40 KB
    const long long P = (long long)a.nx * a.ny * a.nz;
    const int nch = wgrad_chunks(P), blocks = wgrad_blocks(a.cin, a.cout), nb = (int)((P + BG_CHUNK - 1) / BG_CHUNK);
    const int nbias = (a.cout + BG_CH - 1) / BG_CH;
    WgradArgs w = a;
    w.bpart = a.part + (long long)nch * blocks * 27 * MCO * NCI * 256;
    // sized for nx = 2 the staging takes two words a lane more than for nx = 4
    const dim3 grid(nch, 3 * blocks + nbias);
    if (a.nx < 4) k_wgrad<MCO, NCI, 2><<<grid, 192, lds, s>>>(w);
    else k_wgrad<MCO, NCI, 4><<<grid, 192, lds, s>>>(w);
    k_wgrad_sum<MCO, NCI><<<dim3(27 * MCO * NCI * 4 + 1, blocks), 256, 0, s>>>(
        w, nch, kpad, grad, nb, bgrad);
}
}  // namespace

long long wgrad_part_floats(int nx, int ny, int nz, int cin, int cout)
{
    const long long P = (long long)nx * ny * nz;
    return (long long)wgrad_chunks(P) * wgrad_blocks(cin, cout) * 27 * wgrad_mco(cout) * wgrad_nci(cin) * 256 +
           (P + BG_CHUNK - 1) / BG_CHUNK * cout;
}

void launch_wgrad(hipStream_t s, const WgradArgs &a, int kpad, float *grad, float *bgrad)
{
    if (wgrad_mco(a.cout) == 1) {
        if (wgrad_nci(a.cin) == 1) launch_wgrad_k<1, 1>(s, a, kpad, grad, bgrad);
        else launch_wgrad_k<1, 2>(s, a, kpad, grad, bgrad);
    } else {
        if (wgrad_nci(a.cin) == 1) launch_wgrad_k<2, 1>(s, a, kpad, grad, bgrad);
        else launch_wgrad_k<2, 2>(s, a, kpad, grad, bgrad);
    }
}

void launch_pool(hipStream_t s, const bf16_t *in, long long ldi, int nx, int ny, int nz, int c, bf16_t *out,
                 long long ldo)
{
    const long long n = (long long)((nx + 1) / 2) * ((ny + 1) / 2) * ((nz + 1) / 2) * (c / 8);
    k_pool<<<nblk(n), 256, 0, s>>>(in, ldi, nx, ny, nz, c, out, ldo);
}

void launch_pool_bwd(hipStream_t s, const bf16_t *dP, long long ldp, int nx, int ny, int nz, int c,
                     const bf16_t *skip, long long lds, const bf16_t *mask, long long ldm, bf16_t *out, long long ldo)
{
    const long long n = (long long)nx * ny * nz * (c / 8);
    k_pool_bwd<<<nblk(n), 256, 0, s>>>(dP, ldp, nx, ny, nz, c, skip, lds, mask, ldm, out, ldo);
}

void launch_up(hipStream_t s, const bf16_t *in, long long ldi, int nx, int ny, int nz, int c, bf16_t *out,
               long long ldo)
{
    const long long n = (long long)(2 * nx - 1) * (2 * ny - 1) * (2 * nz - 1) * (c / 8);
    k_up<<<nblk(n), 256, 0, s>>>(in, ldi, nx, ny, nz, c, out, ldo);
}

void launch_up_bwd(hipStream_t s, const bf16_t *dF, long long ldf, int nx, int ny, int nz, int c,
                   const bf16_t *mask, long long ldm, bf16_t *out, long long ldo)
{
    const long long n = (long long)nx * ny * nz * (c / 8);
    k_up_bwd<<<nblk(n), 256, 0, s>>>(dF, ldf, nx, ny, nz, c, mask, ldm, out, ldo);
}

int loss_blocks(long long P) { return (int)((P + LOSS_PTS - 1) / LOSS_PTS); }

void launch_loss(hipStream_t s, const float *y, const float *target, float inv_scale, long long P, bf16_t *g,
                 double *part, double *loss_acc)
{
    const int n = loss_blocks(P);
    k_loss<<<n, 256, 0, s>>>(y, target, inv_scale, P, g, part);
    k_loss_final<<<1, 256, 0, s>>>(part, n, P, loss_acc);
}

void launch_adam(hipStream_t s, float *w, const float *g, float *m, float *v, long long n, float gscale, float lr,
                 float b1, float b2, float eps, int step)
{
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)b1, step)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)b2, step)));
    k_adam<<<nblk(n), 256, 0, s>>>(w, g, m, v, n, gscale, lr, b1, b2, eps, c1, c2);
}

void launch_pack(hipStream_t s, const float *w, int coutp, int cin, int kpad, bf16_t *wf, bf16_t *wb, int kpadT)
{
    k_pack<<<nblk(((long long)coutp * kpad + (wb ? (long long)cin * kpadT : 0)) / 8), 256, 0, s>>>(w, coutp, cin, kpad,
                                                                                              wf, wb, kpadT);
}

void launch_f64_to_bf16(hipStream_t s, const double *in, long long n, bf16_t *out)
{
    k_d2b<<<nblk(n / 8), 256, 0, s>>>(in, n, out);
}
void launch_f64_to_f32(hipStream_t s, const double *in, long long n, float *out)
{
    k_d2f<<<nblk(n), 256, 0, s>>>(in, n, out);
}
void launch_scale_out(hipStream_t s, const float *y, long long P, double scale, double *out)
{
    k_scale_out<<<nblk(3 * P), 256, 0, s>>>(y, 3 * P, scale, out);
}
void launch_params_out(hipStream_t s, const ParamMap &m, const float *src, double *out)
{
    k_params_out<<<nblk(m.first[kLayers]), 256, 0, s>>>(m, src, out);
}
void launch_params_in(hipStream_t s, const ParamMap &m, const double *in, float *dst)
{
    k_params_in<<<nblk(m.first[kLayers]), 256, 0, s>>>(m, in, dst);
}

void launch_zero(hipStream_t s, void *p, long long bytes) { (void)hipMemsetAsync(p, 0, (size_t)bytes, s); }

void launch_features(hipStream_t s, const double *B0_64, const float *B0_32, long long Pf, int fsx, long long fsxy,
                     int stride, int nx, int ny, int nz, bf16_t *feat)
{
    k_features<<<nblk((long long)nx * ny * nz), 256, 0, s>>>(B0_64, B0_32, Pf, fsx, fsxy, stride, nx, ny, nz, feat);
}

void launch_target(hipStream_t s, const double *X64, const float *Xh, const float *Xl, long long Pf, int fsx,
                   long long fsxy, int nx, int ny, int nz, double Ox, double Oy, double Oz, double dx, double dy,
                   double dz, float *target)
{
    k_target<<<nblk((long long)nx * ny * nz), 256, 0, s>>>(X64, Xh, Xl, Pf, fsx, fsxy, nx, ny, nz, Ox, Oy, Oz, dx,
                                                           dy, dz, target);
}

void launch_apply(hipStream_t s, const float *y, int cnx, int cny, int cnz, int stride, double scale, double *X64,
                  float *Xh, float *Xl, long long Pf, int fsx, long long fsxy)
{
    const int nx = stride == 2 ? 2 * cnx - 1 : cnx, ny = stride == 2 ? 2 * cny - 1 : cny;
    const int nz = stride == 2 ? 2 * cnz - 1 : cnz;
    k_apply<<<nblk((long long)nx * ny * nz), 256, 0, s>>>(y, cnx, cny, cnz, stride, scale, X64, Xh, Xl, Pf, fsx, fsxy,
                                                          nx, ny, nz);
}

void launch_sumsq(hipStream_t s, const float *v, long long n, double *part, double *out)
{
    const int nb = 512;
    k_sumsq<<<nb, 256, 0, s>>>(v, n, part);
    k_sum_final<<<1, 64, 0, s>>>(part, nb, out);
}

void launch_min_det(hipStream_t s, const double *det, int nx, int ny, int nz, int sx, long long sxy, double *part,
                    double *out)
{
    const int nb = 512;
    k_min_det<<<nb, 256, 0, s>>>(det, nx, ny, nz, sx, sxy, part);
    k_min_det_final<<<1, 64, 0, s>>>(part, nb, out);
}

}  // namespace gmu
