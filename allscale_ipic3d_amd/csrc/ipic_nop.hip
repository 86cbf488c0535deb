// ipic_nop.hip -- learned field step for gfx950: 3x3x3 periodic convolutions as implicit GEMMs
// on BF16 MFMA (v_mfma_f32_16x16x16_bf16) with FP32 accumulation, their data and weight
// gradients, the field head (increments of E and of a potential whose forward curl updates Bc),
// the training loss and Adam.  C ABI in include/ipic_nop.h.
//
// Activations are channel-last on the n^3 index lattice: X[v * C + c], v = (x * ny + y) * nz + z.
//
// Forward convolution (k_conv): one persistent block per CU stages the layer's weights in LDS
// once and walks a contiguous range of bricks of output voxels, two at a time, computing every
// output channel of a brick.  A brick is 4 x R x 16 voxels with R = 1 to 5 rows (the rule stands at
// conv(); the last brick of a column may be shorter).  Its input halo (6 x R+2 x 18 voxels x CIN
// channels) is staged in LDS, its 16-byte pieces permuted (swz).  Up to 4 rows the next brick's halo is
// loaded into registers while the current brick computes; 5 rows leave no registers for it, and it
// is requested after the epilogue.  Each wave owns one x-plane of the brick, i.e. R 16-voxel z-rows, and
// for every tap issues one MFMA per (row, 16-output-channel tile): the A operand is 16 output x 32
// (or 16) input channels of the tap's weights, the B operand the input channels of 16 voxels, both
// from LDS.
// A lane then holds 4 consecutive output channels of a voxel.  The epilogue adds the bias,
// optionally multiplies by silu'(z_saved) and adds a residual, and writes FP32 and/or BF16
// (optionally silu-activated) outputs, 16 bytes a lane.
//
// Bound, 32 to 32 channels at 64^3: the first conv of a block 19.2 us (MFMA 1.45e10 flop: 12.4 us
// at the 1.17 PFLOP/s a large product reaches; 13 us with the MFMAs left out), the second 22.2 us
// (101 MB with the FP32 residual stream: 20.4 us at the 4.9 TB/s of a copy).  They took 30 and 42
// us with a weight read ahead of every MFMA pair, 8-byte padded rows (two reads an operand),
// pair stores and bricks dealt to the XCDs in turn.
//
// Data gradient: the same kernel with the weights mirrored in the taps and transposed in the
// channels.  Weight gradient (k_wgrad): per block and brick, dW[tap][co][ci] += sum over the
// brick's voxels of dY[v][co] X[v + tap][ci] as MFMAs with K = voxels; transposing LDS reads form
// the operands, and a second kernel adds up the blocks' partials.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include <cmath>
#include <cstdint>
#include <string>

#include "ipic_gpu.h"
#include "ipic_nop.h"

namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int BX = 4, BY = 4, BZ = 16;               // output brick of a block
constexpr int BV = BX * BY * BZ;                     // 256 voxels
constexpr int HX = BX + 2, HY = BY + 2, HZ = BZ + 2;  // input halo brick
constexpr int HV = HX * HY * HZ;                     // 648 voxels
constexpr int NL = IPIC_NOP_LAYERS;

__host__ __device__ constexpr int lcin(int l) { return l == 0 ? 16 : 32; }
__host__ __device__ constexpr int lcout(int l) { return l == NL - 1 ? 16 : 32; }
__host__ __device__ constexpr long long lsize(int l) { return 27LL * lcin(l) * lcout(l) + lcout(l); }
__host__ __device__ constexpr long long loff(int l) { return l == 0 ? 0 : loff(l - 1) + lsize(l - 1); }
constexpr long long NPARAM = loff(NL);

thread_local std::string g_err;
thread_local const char* g_err_lit = nullptr;  // message of a failure that allocates nothing

int fail(int code, const std::string& m) {
    g_err_lit = nullptr;
    g_err = m;
    return code;
}

int fail_lit(int code, const char* m) {
    g_err_lit = m;
    return code;
}

// round to nearest even (finite inputs)
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// silu and its derivative with the hardware reciprocal (1 ulp): the results feed BF16 values
// and an FP32 residual stream whose error budget is set by the BF16 rounding of the weights
__device__ __forceinline__ float silu(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

__device__ __forceinline__ float dsilu(float x) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-x));
    return s * (1.0f + x * (1.0f - s));
}

__device__ __forceinline__ int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

struct ConvArgs {
    int n[3];
    const uint16_t* x;    // [V][CIN] BF16
    const uint16_t* w;    // [27][COUT][CIN] BF16
    const float* bias;    // [COUT] (nullable)
    const float* zs;      // [V][COUT]: multiply by silu'(zs) (nullable)
    const float* res;     // [V][COUT]: add after the multiply (nullable; may equal outf)
    float* outf;          // [V][COUT] FP32 (nullable)
    uint16_t* outb;       // [V][COUT] BF16 (nullable)
    int act;              // outb = silu(v) (1) or v (0)
};

// Consecutive work ranges go to one XCD (blocks are dealt round-robin over the 8 XCDs), so that
// neighbouring bricks meet in that XCD's L2: the rank of block b of nb.
__device__ __forceinline__ int xcd_rank(int b, int nb) {
    const int per = nb / 8, rem = nb % 8, xcd = b % 8, slot = b / 8;
    return xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
}

// One MFMA operand of 16 rows: 32 input channels (16x16x32) or 16 (16x16x16) of them.
template <bool K32> struct Frag { typedef v8bf T; };
template <> struct Frag<false> { typedef v4s T; };

__device__ __forceinline__ v4f mma(v8bf a, v8bf b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4f mma(v4s a, v4s b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

template <int CIN, int COUT, int BY>
__global__ __launch_bounds__(512) void k_conv(ConvArgs a, int nbricks) {
    constexpr int HY = BY + 2, HV = HX * HY * HZ;
    constexpr bool WHOLE = 4 % BY == 0;  // n[1] is a multiple of 4; else its last bricks may be shorter
    constexpr bool AHEAD = BY <= 4;      // the next brick's halo in registers while this one computes
    constexpr bool K32 = CIN == 32 && COUT == 32;
    typedef typename Frag<K32>::T F;
    constexpr int RB = CIN * 2;             // LDS bytes per halo voxel and per weight row
    constexpr int PV = CIN / 8;             // 16-byte pieces of one
    constexpr int NS = K32 ? 1 : CIN / 16;  // MFMA slices of the input channels
    constexpr int NT = COUT / 16;
    constexpr int TPR = HZ * PV;            // pieces of a halo row (a z-line of 18 voxels)
    constexpr int RPI = 216 / TPR;          // halo rows that 216 of a half's threads move at once
    constexpr int NJ = HX * HY / RPI;
    static_assert(216 % TPR == 0 && HX * HY % RPI == 0, "halo rows divide among the threads");
    __shared__ __align__(16) unsigned char sw[27 * COUT * RB];  // the layer's weights, all bricks
    __shared__ __align__(16) unsigned char sx[2][HV * RB];      // the two current bricks' halos
    const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2];
    const int nbz = n2 / BZ, nby = (n1 + BY - 1) / BY;
    // the block's two halves (4 waves each) work on bricks 2 p and 2 p + 1 of pair p
    const int half = threadIdx.x >> 8, ht = threadIdx.x & 255;
    const int lane = threadIdx.x & 63, w = (threadIdx.x >> 6) & 3;
    const int m = lane & 15, kq = lane >> 4;
    unsigned char* hx_ = sx[half];

    // 16-byte piece p of row r lies at piece p ^ swz(r), so that one piece of 16 consecutive rows covers
    // every bank once.  Not free of conflicts by the counters: 3.5 conflict cycles an LDS instruction at
    // 64^3, 32 to 32 channels (0.8 with 8-byte padded rows, which need two reads an operand); LDS is
    // active a quarter of the time.
    auto swz = [](int r) { return CIN == 32 ? (r >> 2) & 3 : (r >> 3) & 1; };

    // the next brick's halo travels in registers while the current brick computes: this thread
    // moves piece (fz, fp) of rows RPI j + fq
    const int fq = ht / TPR, fr = ht - fq * TPR, fz = fr / PV, fp = fr - fz * PV;
    const bool mover = ht < 216;
    v4u pre[NJ];
    auto fetch = [&](int bb) {
        const int bz = bb % nbz, by = (bb / nbz) % nby, bx = bb / (nbz * nby);
        if (!mover) return;
        const int gz = wrap1(bz * BZ + fz - 1, n2);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            // (rows that divide the plane evenly leave hx a constant)
            const int row = j * RPI + fq, hx = HY % RPI == 0 ? j * RPI / HY : row / HY, hy = row - hx * HY;
            const int gx = wrap1(bx * BX + hx - 1, n0), gy = wrap1(by * BY + hy - 1, n1);
            pre[j] = *(const v4u*)(a.x + (((long long)gx * n1 + gy) * n2 + gz) * CIN + fp * 8);
        }
    };

    const int npairs = (nbricks + 1) / 2, lb = xcd_rank(blockIdx.x, gridDim.x);
    const int p_lo = (int)((long long)lb * npairs / gridDim.x), p_hi = (int)((long long)(lb + 1) * npairs / gridDim.x);
    if (p_lo < p_hi && 2 * p_lo + half < nbricks) fetch(2 * p_lo + half);
    {
        constexpr int NP = 27 * COUT * PV, NW = (NP + 511) / 512;
        v4u q[NW];
#pragma unroll
        for (int j = 0; j < NW; ++j) {
            const int i = threadIdx.x + j * 512;
            if (i < NP) q[j] = *(const v4u*)(a.w + (long long)i * 8);
        }
#pragma unroll
        for (int j = 0; j < NW; ++j) {
            const int i = threadIdx.x + j * 512, row = i / PV, p = i - row * PV;
            if (i < NP) *(v4u*)(sw + row * RB + ((p ^ swz(row & 15)) * 16)) = q[j];
        }
    }

    // lane offsets of the operands: weights row m, voxel z m + dz; slice s adds 32 bytes before the swizzle
    auto piece = [&](int r, int s) {
        if constexpr (K32) return r * RB + ((kq ^ swz(r)) * 16);
        else return r * RB + (((2 * s + (kq >> 1)) ^ swz(r)) * 16) + (kq & 1) * 8;
    };
    int wo[NS], xo[3][NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        wo[s] = piece(m, s);
#pragma unroll
        for (int dz = 0; dz < 3; ++dz) xo[dz][s] = piece(m + dz, s) + w * HY * HZ * RB;
    }

    // the channels of this lane's results after the exchange below
    const bool hi = NT == 2 && m >= 8;
    const int c0 = (hi ? 16 : 0) + 4 * kq;
    v4f bias = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if (a.bias) bias = *(const v4f*)(a.bias + c0);

    for (int pr = p_lo; pr < p_hi; ++pr) {
        const int bb = 2 * pr + half;
        const bool mine = bb < nbricks;
        __syncthreads();  // the previous bricks' halo reads are done
        if (mine && mover) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                *(v4u*)(hx_ + ((j * RPI + fq) * HZ + fz) * RB + ((fp ^ swz(fz)) * 16)) = pre[j];
        }
        __syncthreads();
        if (AHEAD && pr + 1 < p_hi && bb + 2 < nbricks) fetch(bb + 2);
        if (!mine) continue;
        const int bz = bb % nbz, by = (bb / nbz) % nby, bx = bb / (nbz * nby);
        // this lane's results of row y: NT values of 4 channels, at offset o + y n2 COUT, the
        // second 8 voxels further
        const long long o = ((((long long)bx * BX + w) * n1 + by * BY) * n2 + bz * BZ + (hi ? m - 8 : m)) * COUT + c0;
        const int rows = WHOLE ? BY : min(BY, n1 - by * BY);
        v4f res[BY][NT];
        if (a.res)
#pragma unroll
            for (int y = 0; y < BY; ++y)
                if (y < rows)
#pragma unroll
                for (int t = 0; t < NT; ++t) res[y][t] = *(const v4f*)(a.res + o + ((long long)y * n2 + 8 * t) * COUT);
        // zs ahead as well (5 rows leave no registers for it): read after the last tap, the whole half
        // waited for it (a training step at 64^3: 902 -> 846 us, 48^3 547 -> 515)
        constexpr int ZY = BY <= 4 ? BY : 0;
        v4f zs[ZY > 0 ? ZY : 1][NT];
        if (a.zs)
#pragma unroll
            for (int y = 0; y < ZY; ++y)
                if (y < rows)
#pragma unroll
                    for (int t = 0; t < NT; ++t) zs[y][t] = *(const v4f*)(a.zs + o + ((long long)y * n2 + 8 * t) * COUT);

        v4f acc[BY][NT];
#pragma unroll
        for (int y = 0; y < BY; ++y)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[y][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

        // The taps of a result go in the order dx, dy, dz.  A plane's row is read once for its
        // three dy (rows r of xf at dz; a plane's rows at dz are dead when the next plane's are
        // read), and every tap's operands are read while the tap before it computes: left to
        // itself the compiler reads a tap's weights one MFMA ahead and waits for each of them.
        F xf[HY][3][NS], wf[2][NT][NS];
        auto read_tap = [&](int tap) {
            const int dx = tap / 9, dy = tap / 3 % 3, dz = tap % 3;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int s = 0; s < NS; ++s) wf[tap & 1][t][s] = *(const F*)(sw + wo[s] + (tap * COUT + t * 16) * RB);
#pragma unroll
            for (int r = dy == 0 ? 0 : dy + BY - 1; r < dy + BY; ++r)
#pragma unroll
                for (int s = 0; s < NS; ++s) xf[r][dz][s] = *(const F*)(hx_ + xo[dz][s] + (dx * HY + r) * HZ * RB);
        };
        read_tap(0);
#pragma unroll
        for (int tap = 0; tap < 27; ++tap) {
            const int dy = tap / 3 % 3, dz = tap % 3;
            if (tap < 26) read_tap(tap + 1);
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int y = 0; y < BY; ++y)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[y][t] = mma(wf[tap & 1][t][s], xf[y + dy][dz][s], acc[y][t]);
            __builtin_amdgcn_sched_barrier(0);
        }

        // D[row = output channel (t 16 + 4 kq + j)][col = voxel z m].  With 32 output channels,
        // lanes m and m ^ 8 swap one result (a DPP rotation of the 16 lanes by 8): lanes below 8
        // then hold channels 4 kq .. + 3 of voxels m and m + 8, the others channels 16 + 4 kq .. + 3
        // of voxels m - 8 and m, and one 16-byte store instruction covers 8 whole 32-channel rows
        // (a row's halves from two instructions reach memory as partial lines).
#pragma unroll
        for (int y = 0; y < BY; ++y) {
            if (y >= rows) break;
            v4f v[NT];
            if constexpr (NT == 2) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float give = hi ? acc[y][0][j] : acc[y][1][j];
                    const float got =
                        __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(give), 0x128, 0xF, 0xF, false));
                    v[0][j] = hi ? got : acc[y][0][j];
                    v[1][j] = hi ? acc[y][1][j] : got;
                }
            } else {
                v[0] = acc[y][0];
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const long long at = o + ((long long)y * n2 + 8 * t) * COUT;
                v[t] += bias;
                if (a.zs) {
                    const v4f z = y < ZY ? zs[y < ZY ? y : 0][t] : *(const v4f*)(a.zs + at);
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[t][j] *= dsilu(z[j]);
                }
                if (a.res) v[t] += res[y][t];
                if (a.outf) *(v4f*)(a.outf + at) = v[t];
                if (a.outb) {
                    if (a.act)
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[t][j] = silu(v[t][j]);
                    *(v4bf*)(a.outb + at) = __builtin_convertvector(v[t], v4bf);  // v_cvt_pk_bf16_f32
                }
            }
        }
        if (!AHEAD && pr + 1 < p_hi && bb + 2 < nbricks) fetch(bb + 2);
    }
}

struct WgradArgs {
    int n[3];
    const uint16_t* x;    // [V][CIN] BF16, input of the convolution
    const uint16_t* dy;   // [V][COUT] BF16, gradient of its output
    float* part;          // [blocks][27 * COUT * CIN + COUT]: each block's dW, then its db
};

constexpr int WG_BLOCKS = 256;   // most blocks of the weight gradient (one a CU), and of their partials
constexpr int WG_THREADS = 576;  // 9 waves, one for each (dx, dz)

// Four voxels of one channel (a quarter of an MFMA operand) from channel-last rows in LDS: lane i
// of each 16 gives the address of voxel i / 4, channels 4 (i % 4) .. + 3, and gets channel i of
// the four voxels (ds_read_b64_tr_b16).
__device__ __forceinline__ v4s lds_tr4(const uint16_t* p) {
    typedef __attribute__((address_space(3))) v4s L4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((L4*)p);
}

__device__ __forceinline__ v8bf join8(v4s lo, v4s hi) {
    return __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Weight gradient: dW[tap][co][ci] = sum over voxels of dY[v][co] X[v + tap][ci] on
// v_mfma_f32_16x16x32_bf16, K = 32 voxels (a 16-voxel z-row of two neighbouring x-planes).
// Both operands need the voxels of one channel in a lane; the rows stay channel-last in LDS, as
// they are in memory, and the transposing LDS read forms the operands.  One wave per (dx, dz)
// holds its three dy taps (48 accumulator registers) and slides over y, so that a row of X is read
// once for three taps: 4 KB of LDS reads per 12 MFMAs.  One persistent block per CU walks a
// contiguous range of bricks (its XCD's blocks take neighbouring ranges, whose halos share that
// L2), the next brick's rows travelling in registers.  Block sums go to `part` and k_wgrad_sum
// adds them up, so the gradient does not depend on timing.
//
// Bound: at 64^3, 32 to 32 channels, the MFMAs of a CU's fullest SIMD (three of the nine waves)
// take about 8 us and the LDS reads 5; the first bricks' latency, the staging and the 28 MB of
// partials come on top.  Measured 23.7 us (612 TFLOP/s) and 5.9 us for the sum, against 214 us
// with transposed 2-byte LDS stores, 2-byte operand reads and FP32 atomics; a training step at
// 64^3 went from 3.05 to 1.19 ms.
template <int CIN, int COUT>
__global__ __launch_bounds__(WG_THREADS) void k_wgrad(WgradArgs a, int nbricks) {
    constexpr int NS = CIN / 16, NT = COUT / 16;
    constexpr int XP = HV * CIN / 8, YP = BV * COUT / 8;  // 16-byte pieces of a brick
    constexpr int NX = (XP + WG_THREADS - 1) / WG_THREADS, NY = (YP + WG_THREADS - 1) / WG_THREADS;
    __shared__ __align__(16) uint16_t xs[2][HV * CIN];
    __shared__ __align__(16) uint16_t ys[2][BV * COUT];
    const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2];
    const int nbz = n2 / BZ, nby = n1 / BY;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int dx = w / 3, dz = w % 3;
    const int i16 = lane & 15, kq = lane >> 4;
    const int nb = gridDim.x, lb = xcd_rank(blockIdx.x, nb);
    const int b_lo = (int)((long long)lb * nbricks / nb), b_hi = (int)((long long)(lb + 1) * nbricks / nb);

    v4u px[NX], py[NY];
    auto fetch = [&](int b) {
        const int bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
        const int x0 = bx * BX, y0 = by * BY, z0 = bz * BZ;
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int i = tid + j * WG_THREADS;
            if (i < XP) {
                const int v = i / (CIN / 8), p = i - v * (CIN / 8);
                const int hx = v / (HY * HZ), r = v - hx * (HY * HZ), hy = r / HZ, hz = r - hy * HZ;
                const int gx = wrap1(x0 + hx - 1, n0), gy = wrap1(y0 + hy - 1, n1), gz = wrap1(z0 + hz - 1, n2);
                px[j] = *(const v4u*)(a.x + (((long long)gx * n1 + gy) * n2 + gz) * CIN + p * 8);
            }
        }
#pragma unroll
        for (int j = 0; j < NY; ++j) {
            const int i = tid + j * WG_THREADS;
            if (i < YP) {
                const int v = i / (COUT / 8), p = i - v * (COUT / 8);
                const int lx = v / (BY * BZ), r = v - lx * (BY * BZ), ly = r / BZ, lz = r - ly * BZ;
                py[j] = *(const v4u*)(a.dy + (((long long)(x0 + lx) * n1 + (y0 + ly)) * n2 + (z0 + lz)) * COUT + p * 8);
            }
        }
    };

    v4f acc[3][NS][NT];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[d][s][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    float dbacc[8];  // this thread's pieces of dY always hold the same 8 channels
#pragma unroll
    for (int c = 0; c < 8; ++c) dbacc[c] = 0.0f;
    static_assert(WG_THREADS % (COUT / 8) == 0, "a thread's dY pieces hold the same channels");

    // operand offsets of this lane: K element 8 kq + j is voxel z 8 (kq & 1) + j of plane kq >> 1
    const int vz = 8 * (kq & 1) + (i16 >> 2), cq = 4 * (i16 & 3), vp = kq >> 1;
    const int xoff = (((vp + dx) * HY) * HZ + vz + dz) * CIN + cq;
    const int yoff = (vp * BY * BZ + vz) * COUT + cq;

    int buf = 0;
    if (b_lo < b_hi) fetch(b_lo);
    for (int b = b_lo; b < b_hi; ++b, buf ^= 1) {
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int i = tid + j * WG_THREADS;
            if (i < XP) *(v4u*)(xs[buf] + i * 8) = px[j];
        }
#pragma unroll
        for (int j = 0; j < NY; ++j) {
            const int i = tid + j * WG_THREADS;
            if (i < YP) {
                *(v4u*)(ys[buf] + i * 8) = py[j];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    dbacc[2 * c] += __uint_as_float(py[j][c] << 16);
                    dbacc[2 * c + 1] += __uint_as_float(py[j][c] & 0xFFFF0000u);
                }
            }
        }
        // one barrier a brick: the buffer written here was last read before the previous barrier
        __syncthreads();
        if (b + 1 < b_hi) fetch(b + 1);
        const uint16_t* X = xs[buf] + xoff;
        const uint16_t* Y = ys[buf] + yoff;
#pragma unroll
        for (int pp = 0; pp < BX; pp += 2) {
            v8bf xf[HY][NS];
            auto row = [&](int r) {  // halo row r of the wave's (dx, dz)
                const uint16_t* p = X + (pp * HY + r) * HZ * CIN;
#pragma unroll
                for (int s = 0; s < NS; ++s) xf[r][s] = join8(lds_tr4(p + s * 16), lds_tr4(p + 4 * CIN + s * 16));
            };
            row(0);
            row(1);
#pragma unroll
            for (int y = 0; y < BY; ++y) {
                row(y + 2);
                v8bf yf[NT];
                const uint16_t* p = Y + (pp * BY + y) * BZ * COUT;
#pragma unroll
                for (int t = 0; t < NT; ++t) yf[t] = join8(lds_tr4(p + t * 16), lds_tr4(p + 4 * COUT + t * 16));
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            acc[d][s][t] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[y + d][s], yf[t], acc[d][s][t], 0, 0, 0);
            }
        }
    }
    // D[row = input channel (s 16 + 4 kq + j)][col = output channel (t 16 + i16)]
    float* part = a.part + (long long)blockIdx.x * (27 * COUT * CIN + COUT);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int tap = (dx * 3 + d) * 3 + dz;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                *(v4f*)(part + (tap * COUT + t * 16 + i16) * CIN + s * 16 + 4 * kq) = acc[d][s][t];
    }
    // db: lanes with the same channels, then the waves
    __syncthreads();
    float* s_db = (float*)xs[0];  // [wave][COUT]
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        float v = dbacc[c];
#pragma unroll
        for (int d = 32; d >= COUT / 8; d >>= 1) v += __shfl_xor(v, d, 64);
        if (lane < COUT / 8) s_db[w * COUT + lane * 8 + c] = v;
    }
    __syncthreads();
    if (tid < COUT) {
        float v = 0.0f;
        for (int k = 0; k < WG_THREADS / 64; ++k) v += s_db[k * COUT + tid];
        part[27 * COUT * CIN + tid] = v;
    }
}

// grad[i] += sum over the blocks' partials, in block order within each of 8 slices and then over
// the slices: 32 float4 columns x 8 slices per block (28 MB read at 32 to 32 channels).
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* part, int blocks, int n, float* grad) {
    __shared__ float4 s[8][32];
    const int c = threadIdx.x & 31, q = threadIdx.x >> 5;
    const int col = blockIdx.x * 32 + c;
    const bool in = 4 * col < n;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (in)
#pragma unroll 8
        for (int b = q; b < blocks; b += 8) {
            const float4 p = *(const float4*)(part + (long long)b * n + 4 * col);
            v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
        }
    s[q][c] = v;
    __syncthreads();
    if (q == 0 && in) {
        for (int k = 1; k < 8; ++k) {
            const float4 p = s[k][c];
            v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
        }
        // atomic: passes on several streams may add to one gradient
        float* g = grad + 4 * col;
        atomicAdd(g, v.x);
        atomicAdd(g + 1, v.y);
        atomicAdd(g + 2, v.z);
        atomicAdd(g + 3, v.w);
    }
}

// BF16 weight copies: forward layout (as the parameters) and the data-gradient layout
// wb[26 - tap][ci][co] = W[tap][co][ci] of each layer.
__global__ void k_prepare(const float* p, uint16_t* wf, uint16_t* wb) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NPARAM) return;
    int l = 0;
    while (l + 1 < NL && i >= loff(l + 1)) ++l;
    const long long r = i - loff(l);
    const int ci_n = lcin(l), co_n = lcout(l);
    const uint16_t v = f2bf(p[i]);
    wf[i] = v;
    if (wb) {
        if (r < 27LL * ci_n * co_n) {
            const int tap = (int)(r / (ci_n * co_n)), q = (int)(r % (ci_n * co_n));
            const int co = q / ci_n, ci = q % ci_n;
            wb[loff(l) + ((26 - tap) * ci_n + ci) * co_n + co] = v;
        } else {
            wb[i] = 0;
        }
    }
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NPARAM) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

__global__ void k_pack(int n0, int n1, int n2, const float4* E, const float4* B, const float4* J, float iE,
                       float iB, float iJ, uint16_t* u) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)n0 * n1 * n2) return;
    const float4 e = E[i], b = B[i], j = J[i];
    uint4 lo, hi;
    lo.x = f2bf(e.x * iE) | ((uint32_t)f2bf(e.y * iE) << 16);
    lo.y = f2bf(e.z * iE) | ((uint32_t)f2bf(b.x * iB) << 16);
    lo.z = f2bf(b.y * iB) | ((uint32_t)f2bf(b.z * iB) << 16);
    lo.w = f2bf(j.x * iJ) | ((uint32_t)f2bf(j.y * iJ) << 16);
    hi.x = f2bf(j.z * iJ);
    hi.y = hi.z = hi.w = 0u;
    uint4* d = (uint4*)(u + i * 16);
    d[0] = lo;
    d[1] = hi;
}

struct HeadArgs {
    int n[3];
    const float* out;     // [V][16]
    float soE, soP;
    float iw[3];
    float4* E;            // apply: dE (in place)
    float4* B;            // apply: dBc (in place)
    float4* psi;          // [V] scratch
    const float4* tE;     // loss: targets
    const float4* tB;
    float4* g;            // [V] scratch: dL/d(dB_pred)
    float kE, kB;         // 1 / (varE V), 1 / (varB V)
    double* loss;
    uint16_t* dout;       // [V][16]
};

__device__ __forceinline__ void xyz(const HeadArgs& h, long long i, int& x, int& y, int& z) {
    z = (int)(i % h.n[2]);
    const long long r = i / h.n[2];
    y = (int)(r % h.n[1]);
    x = (int)(r / h.n[1]);
}

__device__ __forceinline__ long long lin(const HeadArgs& h, int x, int y, int z) {
    return ((long long)x * h.n[1] + y) * h.n[2] + z;
}

__device__ __forceinline__ void block_add(double v, double* dst) {
    __shared__ double s[4];
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(dst, s[0] + s[1] + s[2] + s[3]);
}

// mode 0: apply dE, store psi; mode 1: loss on dE, dout[0:3], store psi.  The blocks of mode 1 meet
// on the one loss word, about 16 ns each: 256 of them stride over the voxels (64^3: 20 and 17 us
// with a block per 256 voxels, 12 and 11 us so).
__global__ __launch_bounds__(256) void k_head_a(HeadArgs h, int mode) {
    const long long V = (long long)h.n[0] * h.n[1] * h.n[2];
    double l = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < V; i += (long long)gridDim.x * 256) {
        const float* o = h.out + i * 16;
        const float ex = h.soE * o[0], ey = h.soE * o[1], ez = h.soE * o[2];
        h.psi[i] = make_float4(h.soP * o[3], h.soP * o[4], h.soP * o[5], 0.0f);
        if (mode == 0) {
            float4 e = h.E[i];
            e.x += ex; e.y += ey; e.z += ez;
            h.E[i] = e;
        } else {
            const float4 t = h.tE[i];
            const float rx = ex - t.x, ry = ey - t.y, rz = ez - t.z;
            l += (double)(h.kE * (rx * rx + ry * ry + rz * rz));
            uint16_t* d = h.dout + i * 16;
            d[0] = f2bf(2.0f * h.kE * rx * h.soE);
            d[1] = f2bf(2.0f * h.kE * ry * h.soE);
            d[2] = f2bf(2.0f * h.kE * rz * h.soE);
#pragma unroll
            for (int c = 6; c < 16; ++c) d[c] = 0;
        }
    }
    if (mode == 1) block_add(l, h.loss);
}

// dB_pred = -curl+ psi (the leapfrog B update with psi in place of dt E); mode 0 applies it,
// mode 1 adds its loss and stores g = dL/d(dB_pred)
__global__ __launch_bounds__(256) void k_head_b(HeadArgs h, int mode) {
    const long long V = (long long)h.n[0] * h.n[1] * h.n[2];
    double l = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < V; i += (long long)gridDim.x * 256) {
        int x, y, z;
        xyz(h, i, x, y, z);
        const float4 p = h.psi[i];
        const float4 px = h.psi[lin(h, wrap1(x + 1, h.n[0]), y, z)];
        const float4 py = h.psi[lin(h, x, wrap1(y + 1, h.n[1]), z)];
        const float4 pz = h.psi[lin(h, x, y, wrap1(z + 1, h.n[2]))];
        const float bx = -((py.z - p.z) * h.iw[1] - (pz.y - p.y) * h.iw[2]);
        const float by = -((pz.x - p.x) * h.iw[2] - (px.z - p.z) * h.iw[0]);
        const float bz = -((px.y - p.y) * h.iw[0] - (py.x - p.x) * h.iw[1]);
        if (mode == 0) {
            float4 b = h.B[i];
            b.x += bx; b.y += by; b.z += bz;
            h.B[i] = b;
        } else {
            const float4 t = h.tB[i];
            const float rx = bx - t.x, ry = by - t.y, rz = bz - t.z;
            l += (double)(h.kB * (rx * rx + ry * ry + rz * rz));
            h.g[i] = make_float4(2.0f * h.kB * rx, 2.0f * h.kB * ry, 2.0f * h.kB * rz, 0.0f);
        }
    }
    if (mode == 1) block_add(l, h.loss);
}

// dL/dpsi = -(curl+)^T g = -curl- g (backward differences), scaled into dout[3:6]
__global__ __launch_bounds__(256) void k_head_c(HeadArgs h) {
    const long long V = (long long)h.n[0] * h.n[1] * h.n[2];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= V) return;
    int x, y, z;
    xyz(h, i, x, y, z);
    const float4 g = h.g[i];
    const float4 gx = h.g[lin(h, wrap1(x - 1, h.n[0]), y, z)];
    const float4 gy = h.g[lin(h, x, wrap1(y - 1, h.n[1]), z)];
    const float4 gz = h.g[lin(h, x, y, wrap1(z - 1, h.n[2]))];
    const float cx = (g.z - gy.z) * h.iw[1] - (g.y - gz.y) * h.iw[2];
    const float cy = (g.x - gz.x) * h.iw[2] - (g.z - gx.z) * h.iw[0];
    const float cz = (g.y - gx.y) * h.iw[0] - (g.x - gy.x) * h.iw[1];
    uint16_t* d = h.dout + i * 16;
    d[3] = f2bf(-cx * h.soP);
    d[4] = f2bf(-cy * h.soP);
    d[5] = f2bf(-cz * h.soP);
}

__global__ void k_sub4(float4* d, const float4* a, const float4* b, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 x = a[i], y = b[i];
    d[i] = make_float4(x.x - y.x, x.y - y.y, x.z - y.z, 0.0f);
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------

struct Ws {
    float* x[5];          // residual stream x_0..x_4 (train); x[0] only for inference
    uint16_t* a[5];       // silu(x_b), BF16 (train); a[0] only for inference
    float* h[4];          // conv_b1 outputs (train)
    uint16_t* g[4];       // silu(h_b), BF16 (train); g[0] only for inference
    float* dx[2];         // backward: FP32 gradient of the residual stream (ping-pong)
    uint16_t* dxb;        // its BF16 copy
    uint16_t* dhb;        // BF16 gradient of conv_b1's output
    float* part;          // weight-gradient partials of one layer
};

long long voxels(const int32_t n[3]) { return (long long)n[0] * n[1] * n[2]; }

// blocks of a weight gradient: one a CU, at least a brick each
int wgrad_blocks(const int32_t n[3]) {
    const int bricks = (n[0] / BX) * (n[1] / BY) * (n[2] / BZ);
    return bricks < WG_BLOCKS ? bricks : WG_BLOCKS;
}

Ws carve(void* base, const int32_t n[3], int train, long long* bytes) {
    const long long V = voxels(n);
    const long long F = V * 32 * 4, H = V * 32 * 2;
    unsigned char* p = (unsigned char*)base;
    long long o = 0;
    Ws w{};
    auto takef = [&](float** d) { *d = (float*)(p ? p + o : nullptr); o += (F + 255) & ~255LL; };
    auto takeb = [&](uint16_t** d) { *d = (uint16_t*)(p ? p + o : nullptr); o += (H + 255) & ~255LL; };
    const int nb = train ? 5 : 1, nh = train ? 4 : 1;
    for (int k = 0; k < nb; ++k) takef(&w.x[k]);
    for (int k = 0; k < nb; ++k) takeb(&w.a[k]);
    if (train)
        for (int k = 0; k < 4; ++k) takef(&w.h[k]);
    for (int k = 0; k < nh; ++k) takeb(&w.g[k]);
    if (train) {
        takef(&w.dx[0]);
        takef(&w.dx[1]);
        takeb(&w.dxb);
        takeb(&w.dhb);
        w.part = (float*)(p ? p + o : nullptr);
        o += (long long)wgrad_blocks(n) * (27 * 32 * 32 + 32) * (long long)sizeof(float);
    }
    if (bytes) *bytes = o;
    return w;
}

int check_grid(const int32_t n[3]) {
    if (!n || n[0] <= 0 || n[1] <= 0 || n[2] <= 0 || n[0] % BX || n[1] % BY || n[2] % BZ)
        return fail(IPIC_E_ARG, "grid must be positive with nx % 4 == 0, ny % 4 == 0, nz % 16 == 0");
    if (voxels(n) * 32 >= (1LL << 31)) return fail(IPIC_E_RANGE, "grid too large for the operator");
    return 0;
}

#define NOPCK(expr)                                                                                 \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) return fail(IPIC_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// compute units of the current device (cached per device)
int cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) c = 256;
        cached[dev] = c;
    }
    return cached[dev];
}

template <int CIN, int COUT>
int conv(const int32_t n[3], const uint16_t* x, const uint16_t* w, const float* bias, const float* zs,
         const float* res, float* outf, uint16_t* outb, int act, hipStream_t st) {
    ConvArgs a{{n[0], n[1], n[2]}, x, w, bias, zs, res, outf, outb, act};
    // One persistent block per CU: the weights are staged in LDS once per block, and its two
    // halves work on two bricks at a time.  A round of bricks costs about its rows and two rows' time
    // for the halo and the latency: of bricks of 1 to 5 rows (the last of a column shorter where the
    // rows do not divide n[1]) those with the least of it are taken.  The whole network with 1, 2, 3, 4
    // and 5 rows: 32^3 89, 99, 109, 117, 134 us; 52x56x32 171, 161, 131, 136, 154; 64^3 365, 299,
    // 288, 259, 290; 36x60x64 (540 bricks of 4 rows for 512 halves) 245, 217, 195, 217, 175.
    const int planes = (n[0] / BX) * (n[2] / BZ), halves = 2 * cu_count();
    auto bricks = [&](int rows) { return planes * ((n[1] + rows - 1) / rows); };
    auto cost = [&](int rows) { return (bricks(rows) + halves - 1) / halves * (rows + 2); };
    auto go = [&](auto kernel, int rows) {
        hipLaunchKernelGGL(kernel, dim3(std::min((bricks(rows) + 1) / 2, cu_count())), dim3(512), 0, st, a, bricks(rows));
    };
    int rows = 4;
    for (int r : {5, 3, 2, 1})
        if (cost(r) < cost(rows)) rows = r;
    if (rows == 1) go(k_conv<CIN, COUT, 1>, 1);
    else if (rows == 2) go(k_conv<CIN, COUT, 2>, 2);
    else if (rows == 3) go(k_conv<CIN, COUT, 3>, 3);
    else if (rows == 5) go(k_conv<CIN, COUT, 5>, 5);
    else go(k_conv<CIN, COUT, 4>, 4);
    NOPCK(hipGetLastError());
    return 0;
}

// grad: the layer's weights, then its bias (dW and db are added to it)
template <int CIN, int COUT>
int wgrad(const int32_t n[3], const uint16_t* x, const uint16_t* dy, float* part, float* grad, hipStream_t st) {
    WgradArgs a{{n[0], n[1], n[2]}, x, dy, part};
    const int bricks = (n[0] / BX) * (n[1] / BY) * (n[2] / BZ), blocks = wgrad_blocks(n);
    constexpr int len = 27 * CIN * COUT + COUT;
    hipLaunchKernelGGL((k_wgrad<CIN, COUT>), dim3(blocks), dim3(WG_THREADS), 0, st, a, bricks);
    hipLaunchKernelGGL(k_wgrad_sum, dim3((len / 4 + 31) / 32), dim3(256), 0, st, part, blocks, len, grad);
    NOPCK(hipGetLastError());
    return 0;
}

HeadArgs head_args(const int32_t n[3], const float* out, const ipic_nop_scales* s, const float inv_w[3]) {
    HeadArgs h{};
    h.n[0] = n[0]; h.n[1] = n[1]; h.n[2] = n[2];
    h.out = out;
    h.soE = s->out_E;
    h.soP = s->out_P;
    for (int k = 0; k < 3; ++k) h.iw[k] = inv_w ? inv_w[k] : 1.0f;
    return h;
}

// Scratch of ipic_nop_apply_noalloc: the head's potential psi for grids of at most
// IPIC_NOP_NOALLOC_MAX_VOXELS voxels (32 MiB of float4), one copy per GPU the library runs on,
// held until the process ends.  Host code uses the per-device address from
// hipGetSymbolAddress, never the array's name (a host-side stand-in).
static __device__ __align__(256) float4 scratch[IPIC_NOP_NOALLOC_MAX_VOXELS];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::atomic<float4*> g_scratch_ptr[NOALLOC_MAX_DEVICES];

// The current device's copy of `scratch`, looked up on the first call on that device.
int noalloc_scratch(float4** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail_lit(IPIC_E_HIP, "hipGetDevice failed");
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return fail_lit(IPIC_E_RANGE, "device index above 63");
    float4* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        void* q = nullptr;
        if (hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)) != hipSuccess || !q)
            return fail_lit(IPIC_E_HIP, "hipGetSymbolAddress of the scratch array failed");
        p = (float4*)q;
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return 0;
}

}  // namespace

extern "C" {

const char* ipic_nop_last_error(void) { return g_err_lit ? g_err_lit : g_err.c_str(); }

int64_t ipic_nop_param_count(void) { return NPARAM; }

int ipic_nop_layer(int32_t layer, int64_t* w_offset, int64_t* b_offset, int32_t* cin_p, int32_t* cout_p) {
    if (layer < 0 || layer >= NL) return fail(IPIC_E_ARG, "layer out of range");
    if (w_offset) *w_offset = loff(layer);
    if (b_offset) *b_offset = loff(layer) + 27LL * lcin(layer) * lcout(layer);
    if (cin_p) *cin_p = lcin(layer);
    if (cout_p) *cout_p = lcout(layer);
    return 0;
}

int64_t ipic_nop_workspace_bytes(const int32_t n[3], int32_t train) {
    if (check_grid(n)) return -1;
    long long b = 0;
    carve(nullptr, n, train ? 1 : 0, &b);
    return b;
}

int ipic_nop_prepare(const float* params, uint16_t* wf, uint16_t* wb, void* stream) {
    if (!params || !wf) return fail(IPIC_E_ARG, "null pointer");
    hipLaunchKernelGGL(k_prepare, dim3((unsigned)((NPARAM + 255) / 256)), dim3(256), 0, (hipStream_t)stream, params,
                       wf, wb);
    NOPCK(hipGetLastError());
    return 0;
}

int ipic_nop_pack(const int32_t n[3], const float* dE4, const float* dBc4, const float* J4,
                  const ipic_nop_scales* s, uint16_t* u, void* stream) {
    if (int rc = check_grid(n)) return rc;
    if (!dE4 || !dBc4 || !J4 || !s || !u) return fail(IPIC_E_ARG, "null pointer");
    const long long V = voxels(n);
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n[0], n[1],
                       n[2], (const float4*)dE4, (const float4*)dBc4, (const float4*)J4, 1.0f / s->in_E,
                       1.0f / s->in_B, 1.0f / s->in_J, u);
    NOPCK(hipGetLastError());
    return 0;
}

int ipic_nop_forward(const int32_t n[3], const uint16_t* u, const uint16_t* wf, const float* params, void* ws,
                     int32_t train, float* out, void* stream) {
    if (int rc = check_grid(n)) return rc;
    if (!u || !wf || !params || !ws || !out) return fail(IPIC_E_ARG, "null pointer");
    hipStream_t st = (hipStream_t)stream;
    const Ws w = carve(ws, n, train ? 1 : 0, nullptr);
    auto W = [&](int l) { return wf + loff(l); };
    auto Bi = [&](int l) { return params + loff(l) + 27LL * lcin(l) * lcout(l); };
    if (int rc = conv<16, 32>(n, u, W(0), Bi(0), nullptr, nullptr, w.x[0], w.a[0], 1, st)) return rc;
    for (int b = 0; b < 4; ++b) {
        const int xi = train ? b : 0, xo = train ? b + 1 : 0;
        uint16_t* g = train ? w.g[b] : w.g[0];
        if (int rc = conv<32, 32>(n, w.a[xi], W(1 + 2 * b), Bi(1 + 2 * b), nullptr, nullptr, train ? w.h[b] : nullptr,
                                  g, 1, st))
            return rc;
        if (int rc = conv<32, 32>(n, g, W(2 + 2 * b), Bi(2 + 2 * b), nullptr, w.x[xi], w.x[xo], w.a[xo], 1, st))
            return rc;
    }
    return conv<32, 16>(n, w.a[train ? 4 : 0], W(9), Bi(9), nullptr, nullptr, out, nullptr, 0, st);
}

int ipic_nop_apply(const int32_t n[3], const float* out, const ipic_nop_scales* s, const float inv_w[3],
                   float* dE4, float* dBc4, float* psi4, void* stream) {
    if (int rc = check_grid(n)) return rc;
    if (!out || !s || !dE4 || !dBc4 || !psi4) return fail(IPIC_E_ARG, "null pointer");
    HeadArgs h = head_args(n, out, s, inv_w);
    h.E = (float4*)dE4;
    h.B = (float4*)dBc4;
    h.psi = (float4*)psi4;
    const long long V = voxels(n);
    const dim3 g((unsigned)((V + 255) / 256));
    hipLaunchKernelGGL(k_head_a, g, dim3(256), 0, (hipStream_t)stream, h, 0);
    hipLaunchKernelGGL(k_head_b, g, dim3(256), 0, (hipStream_t)stream, h, 0);
    NOPCK(hipGetLastError());
    return 0;
}

int ipic_nop_apply_noalloc(const int32_t n[3], const float* out, const ipic_nop_scales* s, const float inv_w[3],
                           float* dE4, float* dBc4, void* stream) {
    if (!n || n[0] <= 0 || n[1] <= 0 || n[2] <= 0 || n[0] % BX || n[1] % BY || n[2] % BZ)
        return fail_lit(IPIC_E_ARG, "grid must be positive with nx % 4 == 0, ny % 4 == 0, nz % 16 == 0");
    const long long V = voxels(n);
    if (V > IPIC_NOP_NOALLOC_MAX_VOXELS)
        return fail_lit(IPIC_E_RANGE, "grid above IPIC_NOP_NOALLOC_MAX_VOXELS (2097152 voxels) for the "
                                      "no-allocation apply");
    if (!out || !s || !dE4 || !dBc4) return fail_lit(IPIC_E_ARG, "null pointer");
    float4* psi = nullptr;
    if (int rc = noalloc_scratch(&psi)) return rc;
    HeadArgs h = head_args(n, out, s, inv_w);
    h.E = (float4*)dE4;
    h.B = (float4*)dBc4;
    h.psi = psi;  // every entry below V is written by k_head_a before k_head_b reads it
    const dim3 g((unsigned)((V + 255) / 256));
    hipLaunchKernelGGL(k_head_a, g, dim3(256), 0, (hipStream_t)stream, h, 0);
    hipLaunchKernelGGL(k_head_b, g, dim3(256), 0, (hipStream_t)stream, h, 0);
    if (hipGetLastError() != hipSuccess) return fail_lit(IPIC_E_HIP, "kernel launch failed");
    return 0;
}

int ipic_nop_loss(const int32_t n[3], const float* out, const ipic_nop_scales* s, const float inv_w[3],
                  const float* tE4, const float* tB4, float varE, float varB, double* loss, uint16_t* dout,
                  float* g4, float* psi4, void* stream) {
    if (int rc = check_grid(n)) return rc;
    if (!out || !s || !tE4 || !tB4 || !loss || !dout || !g4 || !psi4) return fail(IPIC_E_ARG, "null pointer");
    if (!(varE > 0.0f) || !(varB > 0.0f)) return fail(IPIC_E_ARG, "variances must be positive");
    HeadArgs h = head_args(n, out, s, inv_w);
    const long long V = voxels(n);
    h.psi = (float4*)psi4;
    h.tE = (const float4*)tE4;
    h.tB = (const float4*)tB4;
    h.g = (float4*)g4;
    h.kE = (float)(1.0 / ((double)varE * (double)V));
    h.kB = (float)(1.0 / ((double)varB * (double)V));
    h.loss = loss;
    h.dout = dout;
    const dim3 g((unsigned)((V + 255) / 256));
    const dim3 few((unsigned)std::min<long long>((V + 255) / 256, 256));
    hipLaunchKernelGGL(k_head_a, few, dim3(256), 0, (hipStream_t)stream, h, 1);
    hipLaunchKernelGGL(k_head_b, few, dim3(256), 0, (hipStream_t)stream, h, 1);
    hipLaunchKernelGGL(k_head_c, g, dim3(256), 0, (hipStream_t)stream, h);
    NOPCK(hipGetLastError());
    return 0;
}

int ipic_nop_backward(const int32_t n[3], const uint16_t* u, const uint16_t* wb, const float* params, void* ws,
                      const uint16_t* dout, float* grad, void* stream) {
    if (int rc = check_grid(n)) return rc;
    if (!u || !wb || !params || !ws || !dout || !grad) return fail(IPIC_E_ARG, "null pointer");
    hipStream_t st = (hipStream_t)stream;
    const Ws w = carve(ws, n, 1, nullptr);
    auto Wb = [&](int l) { return wb + loff(l); };
    auto G = [&](int l) { return grad + loff(l); };
    // projection: out = conv9(a4)
    if (int rc = wgrad<32, 16>(n, w.a[4], dout, w.part, G(9), st)) return rc;
    if (int rc = conv<16, 32>(n, dout, Wb(9), nullptr, w.x[4], nullptr, w.dx[0], w.dxb, 0, st)) return rc;
    int cur = 0;
    for (int b = 3; b >= 0; --b) {
        // x_{b+1} = x_b + conv_b2(g_b), g_b = silu(h_b), h_b = conv_b1(a_b), a_b = silu(x_b)
        if (int rc = wgrad<32, 32>(n, w.g[b], w.dxb, w.part, G(2 + 2 * b), st)) return rc;
        if (int rc = conv<32, 32>(n, w.dxb, Wb(2 + 2 * b), nullptr, w.h[b], nullptr, nullptr, w.dhb, 0, st)) return rc;
        if (int rc = wgrad<32, 32>(n, w.a[b], w.dhb, w.part, G(1 + 2 * b), st)) return rc;
        if (int rc = conv<32, 32>(n, w.dhb, Wb(1 + 2 * b), nullptr, w.x[b], w.dx[cur], w.dx[1 - cur], w.dxb, 0, st))
            return rc;
        cur = 1 - cur;
    }
    return wgrad<16, 32>(n, u, w.dxb, w.part, G(0), st);
}

int ipic_nop_adam(float* params, const float* grad, float* m, float* v, int64_t step, float lr, float beta1,
                  float beta2, float eps, uint16_t* wf, uint16_t* wb, void* stream) {
    if (!params || !grad || !m || !v) return fail(IPIC_E_ARG, "null pointer");
    if (step < 1) return fail(IPIC_E_ARG, "Adam step counts from 1");
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)beta1, (double)step)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)beta2, (double)step)));
    const dim3 g((unsigned)((NPARAM + 255) / 256));
    hipLaunchKernelGGL(k_adam, g, dim3(256), 0, (hipStream_t)stream, params, grad, m, v, lr, beta1, beta2, eps, c1,
                       c2);
    NOPCK(hipGetLastError());
    if (wf) return ipic_nop_prepare(params, wf, wb, stream);
    return 0;
}

int ipic_dev_alloc(int64_t bytes, void** out) {
    if (!out || bytes < 0) return fail(IPIC_E_ARG, "bad allocation request");
    *out = nullptr;
    NOPCK(hipMalloc(out, bytes > 0 ? (size_t)bytes : 256));
    return 0;
}

int ipic_dev_free(void* p) {
    if (p) NOPCK(hipFree(p));
    return 0;
}

int ipic_dev_copy(void* dst, const void* src, int64_t bytes) {
    if (bytes < 0 || (bytes > 0 && (!dst || !src))) return fail(IPIC_E_ARG, "bad copy");
    if (bytes) NOPCK(hipMemcpy(dst, src, (size_t)bytes, hipMemcpyDefault));
    return 0;
}

int ipic_dev_zero(void* p, int64_t bytes, void* stream) {
    if (bytes < 0 || (bytes > 0 && !p)) return fail(IPIC_E_ARG, "bad fill");
    if (bytes) NOPCK(hipMemsetAsync(p, 0, (size_t)bytes, (hipStream_t)stream));
    return 0;
}

int ipic_dev_sync(void* stream) {
    NOPCK(hipStreamSynchronize((hipStream_t)stream));
    return 0;
}

int ipic_dev_sub4(float* dst, const float* a, const float* b, int64_t count, void* stream) {
    if (count < 0 || (count > 0 && (!dst || !a || !b))) return fail(IPIC_E_ARG, "bad difference");
    if (count == 0) return 0;
    hipLaunchKernelGGL(k_sub4, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (float4*)dst, (const float4*)a, (const float4*)b, (long long)count);
    NOPCK(hipGetLastError());
    return 0;
}

}  // extern "C"
