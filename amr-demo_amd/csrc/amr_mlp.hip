// amr_mlp.hip -- learned refinement tagger on gfx950: patch features, and
// the forward / backward passes of a 384 -> 64 -> 64 -> 3 ReLU perceptron on
// the MFMA units (gfx950's v_mfma_f32_16x16x32_bf16: BF16 operands, FP32
// accumulate, K = 32 per instruction; the one K = 16 product, by the padded
// logit gradients, uses v_mfma_f32_16x16x16_bf16),
// with a deterministic two-pass gradient reduction and Adam.
//
// The reference has no learned tagger (it refines on density thresholds,
// src/solver/src/tagging_methods_module.F90:14-71); features, labels and the
// network are defined in include/amr_tagger.h.
//
// Work decomposition of a gradient.  A minibatch is a few thousand samples of a
// small network: 2 MFLOP a workgroup if one held 64 samples and all of its
// weight gradients, on a fraction of the CUs.  Three kernels instead, each
// spread over the chip:
//   backprop_kernel  16 samples a workgroup, wave w the 16-wide tile w of every
//                    layer: forward, loss, and the gradients down to the
//                    pre-activations, written out transposed (hidden unit major);
//   wgrad_kernel     the weight gradients, reductions over samples, by output
//                    tile: a partial sum per `chunks` chunks of 64 samples, its
//                    dW1 split over 12 waves, its other parts one workgroup;
//   reduce_kernel    sums the partials in a fixed order (bitwise reproducible)
//                    and applies Adam.
// Every sum has the operands and the order it has when one workgroup walks its
// chunks with the weight gradients in registers, which is how it was before: 42.3
// + 9.5 us a minibatch of 4096 (32 workgroups of 256 CUs), now 9.1 + 9.2 + 3.5.
//
// MFMA operand layouts (lane l, r = l % 16, g = l / 16):
//   16x16x32: A[i][k]: lane holds A[r][8g + t], B[k][j]: lane holds
//             B[8g + t][r], t = 0..7 (eight consecutive k per lane)
//   16x16x16: the same with 4g + t, t = 0..3
//   D[i][j] (both): lane holds D[4g + t][r], t = 0..3

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "amr_hip.h"
#include "amr_internal.h"
#include "amr_tagger.h"

namespace {

constexpr int NIN = AMR_MLP_NIN, NH = AMR_MLP_NH, NOUT = AMR_MLP_NOUT;
constexpr int OW1 = 0, OB1 = NH * NIN, OW2 = OB1 + NH, OB2 = OW2 + NH * NH, OW3 = OB2 + NH,
              OB3 = OW3 + NOUT * NH, NP = OB3 + NOUT;
static_assert(NP == AMR_MLP_NPARAM, "parameter layout");
constexpr int NPP = (NP + 1 + 63) / 64 * 64;     // partial row: gradient + loss, padded
constexpr int SX = NIN + 8;                      // LDS row strides (elements)
constexpr int SH = NH + 8;
constexpr int ROWS = 64;                         // samples per chunk
constexpr int BLK = 256;

typedef short s4v __attribute__((ext_vector_type(4)));
typedef short s8v __attribute__((ext_vector_type(8)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

// round to nearest even (no NaN here); the device has an instruction for it, equal
// for every other bit pattern.  The empty statement keeps the FP32 value a value of
// its own: the compiler would round a double once, straight to BF16.
__host__ __device__ inline uint16_t f2bf(float x)
{
#ifdef __HIP_DEVICE_COMPILE__
    asm("" : "+v"(x));
    return __builtin_bit_cast(uint16_t, (__bf16)x);
#else
    uint32_t u;
    memcpy(&u, &x, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
#endif
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ f4v mfma(s4v a, s4v b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma32(s8v a, s8v b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, a), __builtin_bit_cast(b8v, b), c, 0,
                                                   0, 0);
}

__device__ __forceinline__ unsigned long long d2bits(double v) { return (unsigned long long)__double_as_longlong(v); }

// ---------------------------------------------------------------------------
// features: one wave per 8x8 patch, four patches per workgroup.  Memory is the
// floor (32 bytes read and 12 written per cell).  The four maxima share one
// reduction, are inverted once, a lane each, and a quotient by one is a product
// refined to the correctly rounded value.  5.0M cells: 83.5 us with LDS atomics and
// six IEEE quotients per cell, 51.7 with a DPP reduction per maximum (350 vector
// instructions a patch, which bounded it), 40.9 now (220; 5.4 TB/s).
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const long long b = __double_as_longlong(v);
    int lo = (int)b, hi = (int)(b >> 32);
    lo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_value(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// The maxima of four values' magnitudes over the wave, ignoring NaN: row k of 16
// lanes ends with that of u[0], u[2], u[1], u[3].  Two values exchange the wave's
// halves, then the two results their odd and even rows, so that what is left to
// reduce is one value.
__device__ __forceinline__ double four_abs_max(const double u[4])
{
    auto joint = [](double a, double b, auto swap) {
        const long long p = __double_as_longlong(a), q = __double_as_longlong(b);
        const auto lo = swap((int)p, (int)q), hi = swap((int)(p >> 32), (int)(q >> 32));
        return fmax(fabs(__longlong_as_double(((long long)hi[0] << 32) | (unsigned)lo[0])),
                    fabs(__longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1])));
    };
    auto halves = [](int x, int y) { return __builtin_amdgcn_permlane32_swap(x, y, false, false); };
    auto rows = [](int x, int y) { return __builtin_amdgcn_permlane16_swap(x, y, false, false); };
    double v = joint(joint(u[0], u[1], halves), joint(u[2], u[3], halves), rows);
    v = fmax(v, dpp_move<0xB1>(v));                  // quad_perm 1,0,3,2
    v = fmax(v, dpp_move<0x4E>(v));                  // quad_perm 2,3,0,1
    v = fmax(v, dpp_move<0x141>(v));                 // row_half_mirror
    return fmax(v, dpp_move<0x140>(v));              // row_mirror
}

// RN(a / s) for s in [2^-400, 2^400] and |a| <= 2^400, given r = RN(1 / s): the
// product is within two ulp, the first correction makes it faithful, the second
// correctly rounded (Markstein's theorem).  Where a remainder falls below the
// normal range, so does the quotient's FP32 value: zero either way.  The sign
// of a zero is the caller's.
__device__ __forceinline__ double div_by(double a, double s, double r)
{
    double q = a * r;
    q = fma(fma(-q, s, a), r, q);
    return fma(fma(-q, s, a), r, q);
}
// BF16 of the quotient of `a` and a positive number, its sign from `a` (the
// corrections lose that of a zero)
__device__ __forceinline__ uint16_t quotient_bf16(double q, double a)
{
    const uint32_t sign = (uint32_t)(d2bits(a) >> 32) & 0x80000000u;
    return f2bf(__uint_as_float(__float_as_uint((float)q) | sign));
}

__global__ __launch_bounds__(256) void features_kernel(const double *__restrict__ U,
                                                       const int *__restrict__ nbr, int nquad,
                                                       uint16_t *__restrict__ X)
{
    // densities of the patch, then of its four sides' ghosts
    __shared__ double rho[4][64 + 32];
    const int w = threadIdx.x >> 6, c = threadIdx.x & 63, ci = c & 7, cj = c >> 3;
    const int quad = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + w);
    if (quad >= nquad) return;                       // no barrier follows: each wave has its own densities
    typedef const int __attribute__((address_space(4))) cint4;
    const cint4 *nb = (const cint4 *)nbr + (size_t)quad * 8;
    const double *Q = U + (size_t)quad * 256;
    double u[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) u[f] = Q[f * 64 + c];
    // ghost k of side s: the neighbour's edge cell, the mean of two finer ones',
    // the own cell on a wall
    const int k = c & 7, s = (c >> 3) & 3;
    const bool x = s < 2, hi = s & 1;
    const int lo = x ? k * 8 : k, top = lo + (x ? 7 : 56);
    const int a0 = hi ? nb[2] : nb[0], a1 = hi ? nb[6] : nb[4], b0 = hi ? nb[3] : nb[1], b1 = hi ? nb[7] : nb[5];
    const int na = x ? a0 : a1, nbb = x ? b0 : b1;
    double g = na < 0 ? Q[hi ? top : lo] : U[(size_t)na * 256 + (hi ? lo : top)];
    if (na >= 0 && nbb >= 0) g = 0.5 * (g + U[(size_t)nbb * 256 + (hi ? lo : top)]);
    rho[w][c] = u[0];
    if (c < 32) rho[w][64 + c] = g;
    const double m = four_abs_max(u);
    asm volatile("" ::: "memory");                   // the wave's LDS operations execute in order
    const double re = rho[w][ci < 7 ? c + 1 : 64 + 8 + cj], rw = rho[w][ci > 0 ? c - 1 : 64 + cj];
    const double rn = rho[w][cj < 7 ? c + 8 : 64 + 24 + ci], rs = rho[w][cj > 0 ? c - 8 : 64 + 16 + ci];
    const double num[6] = {u[0], u[1], u[2], u[3], re - rw, rn - rs};
    uint16_t *o = X + (size_t)quad * NIN + c;
    constexpr int at[4] = {0, 32, 16, 48};           // a lane with the maximum of field f
    double sm[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) sm[f] = lane_value(m, at[f]);
    // every maximum zero or in div_by's range, no infinity or NaN among the numerators
    const bool nan = u[0] != u[0] || u[1] != u[1] || u[2] != u[2] || u[3] != u[3];
    if (__all(!nan && fabs(num[4]) <= 0x1p400 && fabs(num[5]) <= 0x1p400 &&
              (m == 0.0 || (m >= 0x1p-400 && m <= 0x1p400)))) {
        // the four reciprocals from one quotient
        const double inv = 1.0 / m;
        double ri[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) ri[f] = lane_value(inv, at[f]);
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const double d = f < 4 ? sm[f] : sm[0], r = f < 4 ? ri[f] : ri[0];
            o[f * 64] = d == 0.0 ? (uint16_t)0 : quotient_bf16(div_by(num[f], d, r), num[f]);
        }
    } else {
        // a maximum is NaN where some lane's value is
#pragma unroll
        for (int f = 0; f < 4; ++f)
            if (__any(u[f] != u[f])) sm[f] = NAN;
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const double d = f < 4 ? sm[f] : sm[0];
            o[f * 64] = f2bf((float)(d > 0.0 ? num[f] / d : 0.0));
        }
    }
}

// 16x16 patches: the tagger reads each patch coarsened to 8x8, every coarse
// cell the mean of its 2x2 block, ((a + b) + c) + d times 0.25 with a..d in
// z-order (the summation of solver_coarsen_operator_2d.F90:49-50 applied
// within a patch).  The neighbours are coarsened alike and keep their ids, so
// features_kernel then runs unchanged on the coarsened state.
__global__ __launch_bounds__(256) void pool16_kernel(const double *__restrict__ U, double *__restrict__ P,
                                                     int nquad)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;     // one coarse cell
    if (t >= (long long)nquad * 64) return;
    const long long q = t >> 6;
    const int c = (int)(t & 63), I = c & 7, J = c >> 3;
    const double *s = U + q * 1024 + (2 * J) * 16 + 2 * I;
    double *d = P + q * 256 + c;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const double *sf = s + f * 256;
        d[f * 64] = 0.25 * (((sf[0] + sf[1]) + sf[16]) + sf[17]);
    }
}

// ---------------------------------------------------------------------------
// shared pieces of the network kernels
// ---------------------------------------------------------------------------
struct Weights {
    const uint16_t *W1, *W2, *W3;   // BF16 copies: [64][384], [64][64], [16][64] (rows 3..15 zero)
    const uint16_t *W2t;            // W2 transposed
    const float *P;                 // FP32 master (biases read from here)
};

template <int THREADS, class Lds>
__device__ void stage_weights(Lds &s, const Weights &wt)
{
    const int tid = threadIdx.x;
    for (int i = tid; i < NH * NIN / 8; i += THREADS) {
        const int row = i / (NIN / 8), c8 = i % (NIN / 8);
        *(uint4 *)&s.W1[row * SX + c8 * 8] = ((const uint4 *)wt.W1)[i];
    }
    for (int i = tid; i < NH * NH / 8; i += THREADS) {
        const int row = i / (NH / 8), c8 = i % (NH / 8);
        *(uint4 *)&s.W2[row * SH + c8 * 8] = ((const uint4 *)wt.W2)[i];
    }
    for (int i = tid; i < 16 * NH / 8; i += THREADS) {
        const int row = i / (NH / 8), c8 = i % (NH / 8);
        *(uint4 *)&s.W3[row * SH + c8 * 8] = ((const uint4 *)wt.W3)[i];
    }
    if (tid < NH) {
        s.b[tid] = wt.P[OB1 + tid];
        s.b[NH + tid] = wt.P[OB2 + tid];
    }
    if (tid < 4) s.b[2 * NH + tid] = tid < NOUT ? wt.P[OB3 + tid] : 0.0f;
}

// Inference: logits (optional) and argmax class (optional) of `count` rows.
// A wave takes 16 rows at a time; their features go from memory straight to
// the matrix operands (a lane's eight consecutive ones are 16 bytes), the next
// 16 rows' while these are evaluated.  Only the weights and a wave's 16 rows of
// activations are in LDS (79 KB with eight waves, two workgroups a CU), and nothing
// but the staging of the weights takes a barrier.  The features' bytes are the
// floor; 77k rows: 44.1 us with each chunk staged in LDS between barriers, 18.8
// with four waves a workgroup (2.4 tiles a wave, so the last third of them on
// their own), 16.6 with eight (3.6 TB/s).
constexpr int IWAVES = 8;
struct __attribute__((aligned(16))) InferLds {
    uint16_t W1[NH * SX];
    uint16_t W2[NH * SH];
    uint16_t W3[16 * SH];
    uint16_t H[IWAVES][16 * SH]; // a wave's first, then second hidden layer
    float b[2 * NH + 4];
};

__global__ __launch_bounds__(64 * IWAVES, 4) void infer_kernel(Weights wt, const uint16_t *__restrict__ X, int count,
                                                    float refine_bias, float *__restrict__ logits,
                                                    int *__restrict__ cls)
{
    __shared__ InferLds s;
    stage_weights<64 * IWAVES>(s, wt);
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    uint16_t *const H = s.H[w];
    constexpr int KK = NIN / 32;
    const int tiles = (count + 15) / 16, step = gridDim.x * IWAVES;
    s8v xn[KK];
    auto load = [&](int tile) {
        // rows past the last read it; nothing of theirs is stored
        const uint16_t *row = X + (size_t)min(tile * 16 + r, count - 1) * NIN + 8 * g;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) xn[kk] = *(const s8v *)(row + 32 * kk);
    };
    int tile = blockIdx.x * IWAVES + w;
    if (tile < tiles) load(tile);
    for (; tile < tiles; tile += step) {
        f4v acc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const s8v a = xn[kk];
#pragma unroll
            for (int c = 0; c < 4; ++c)
                acc[c] = mfma32(a, *(const s8v *)&s.W1[(16 * c + r) * SX + 32 * kk + 8 * g], acc[c]);
        }
        if (tile + step < tiles) load(tile + step);
        auto put = [&](int layer) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    H[(4 * g + t) * SH + 16 * c + r] = f2bf(fmaxf(acc[c][t] + s.b[layer * NH + 16 * c + r], 0.0f));
            asm volatile("" ::: "memory");           // the wave's LDS operations execute in order
        };
        put(0);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NH / 32; ++kk) {
            const s8v a = *(const s8v *)&H[r * SH + 32 * kk + 8 * g];
#pragma unroll
            for (int c = 0; c < 4; ++c)
                acc[c] = mfma32(a, *(const s8v *)&s.W2[(16 * c + r) * SH + 32 * kk + 8 * g], acc[c]);
        }
        asm volatile("" ::: "memory");
        put(1);
        f4v z = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NH / 32; ++kk)
            z = mfma32(*(const s8v *)&H[r * SH + 32 * kk + 8 * g], *(const s8v *)&s.W3[r * SH + 32 * kk + 8 * g], z);
        asm volatile("" ::: "memory");
        // lane (class r, rows 4g..4g+3) holds the logits: row r's three, from
        // the lanes of its group, end in lanes r of group 0
        const float bz = s.b[2 * NH + (r < NOUT ? r : 0)];
#pragma unroll
        for (int t = 0; t < 4; ++t) z[t] += bz;
        float zr[NOUT];
#pragma unroll
        for (int c = 0; c < NOUT; ++c) {
            const int src = (r >> 2) * 16 + c;
            const float v0 = __shfl(z[0], src, 64), v1 = __shfl(z[1], src, 64);
            const float v2 = __shfl(z[2], src, 64), v3 = __shfl(z[3], src, 64);
            zr[c] = (r & 2) ? ((r & 1) ? v3 : v2) : ((r & 1) ? v1 : v0);
        }
        const int row = tile * 16 + r;
        if (g == 0 && row < count) {
            const float z0 = zr[0], z1 = zr[1], z2 = zr[2] + refine_bias;
            if (logits) {
                logits[(size_t)row * 3] = z0;
                logits[(size_t)row * 3 + 1] = z1;
                logits[(size_t)row * 3 + 2] = zr[2];
            }
            if (cls) cls[row] = (z0 >= z1 && z0 >= z2) ? 0 : (z1 >= z2 ? 1 : 2);
        }
    }
}

struct GradArgs {
    const uint16_t *X;
    const int *y;
    const int *perm;       // nullptr: rows first.. in order
    long long first;
    int count;             // rows of this launch
    int chunks;            // chunks per partial sum
    int ld;                // rows of the buffers below: count up to whole partial sums
    float cw[3];           // class weights
    float scale;           // 1 / sum of row weights
    // activations and pre-activation gradients, [64][ld] (dZ: [3][ld])
    uint16_t *H1, *H2, *dA1, *dA2, *dZ;
    float *loss;           // [ld]
    float *partial;        // [partial sums][NPP]
};

// Forward pass, loss and pre-activation gradients of 16 samples.  Latency bounds
// it: every CU has one workgroup or two, its operands come straight from memory
// or L2 (all loads of a layer in flight together), and the three exchanges
// between the waves go through LDS.
__global__ __launch_bounds__(BLK) void backprop_kernel(Weights wt, GradArgs ga)
{
    __shared__ __attribute__((aligned(16))) uint16_t h1s[16 * SH], h2s[16 * SH], a2s[16 * SH];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16, loc = row0 + r;      // the lane's sample
    const bool valid = loc < ga.count;                     // rows past the last: features and weight zero
    const long long gi = ga.first + (valid ? loc : 0);
    const long long src = ga.perm ? (long long)ga.perm[gi] : gi;
    constexpr int KK = NIN / 32;
    s8v xa[KK], wb[KK];
    const uint16_t *const xrow = ga.X + (size_t)src * NIN + 8 * g;
    const uint16_t *const wrow = wt.W1 + (16 * w + r) * NIN + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        wb[kk] = *(const s8v *)(wrow + 32 * kk);
        xa[kk] = valid ? *(const s8v *)(xrow + 32 * kk) : s8v{0, 0, 0, 0, 0, 0, 0, 0};
    }
    const int yy = valid ? ga.y[src] : 0;
    const int hid = 16 * w + r;                            // the lane's unit of either hidden layer
    s8v w2b[2], w3b[2], w2t[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
        w2b[kk] = *(const s8v *)(wt.W2 + hid * NH + 32 * kk + 8 * g);
        w2t[kk] = *(const s8v *)(wt.W2t + hid * NH + 32 * kk + 8 * g);
        w3b[kk] = *(const s8v *)(wt.W3 + r * NH + 32 * kk + 8 * g);
    }
    s4v w3t = s4v{0, 0, 0, 0};                             // W3[class 4g + t][unit]
    if (g == 0)
#pragma unroll
        for (int t = 0; t < NOUT; ++t) w3t[t] = (short)wt.W3[t * NH + hid];
    const float b1 = wt.P[OB1 + hid], b2 = wt.P[OB2 + hid], b3 = wt.P[OB3 + (r < NOUT ? r : 0)];

    // a layer's values of the lane's unit, samples 4g..4g+3: to the other waves
    // by sample, to the weight gradients by unit
    auto put = [&](const uint16_t v[4], uint16_t *lds, uint16_t *out) {
        ushort4 q;
        q.x = v[0]; q.y = v[1]; q.z = v[2]; q.w = v[3];
        *(ushort4 *)(out + (size_t)hid * ga.ld + row0 + 4 * g) = q;
        if (lds)
#pragma unroll
            for (int t = 0; t < 4; ++t) lds[(4 * g + t) * SH + hid] = v[t];
    };
    f4v acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) acc = mfma32(xa[kk], wb[kk], acc);
    uint16_t h1[4], h2[4], da[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) h1[t] = f2bf(fmaxf(acc[t] + b1, 0.0f));
    put(h1, h1s, ga.H1);
    __syncthreads();
    acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) acc = mfma32(*(const s8v *)&h1s[r * SH + 32 * kk + 8 * g], w2b[kk], acc);
#pragma unroll
    for (int t = 0; t < 4; ++t) h2[t] = f2bf(fmaxf(acc[t] + b2, 0.0f));
    put(h2, h2s, ga.H2);
    __syncthreads();
    // logits (every wave all of them): lane holds class r of samples 4g..4g+3,
    // gathered to the sample's lanes
    f4v zc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) zc = mfma32(*(const s8v *)&h2s[r * SH + 32 * kk + 8 * g], w3b[kk], zc);
#pragma unroll
    for (int t = 0; t < 4; ++t) zc[t] += b3;
    float z[NOUT];
#pragma unroll
    for (int c = 0; c < NOUT; ++c) {
        const int from = (r >> 2) * 16 + c;
        const float v0 = __shfl(zc[0], from, 64), v1 = __shfl(zc[1], from, 64);
        const float v2 = __shfl(zc[2], from, 64), v3 = __shfl(zc[3], from, 64);
        z[c] = (r & 2) ? ((r & 1) ? v3 : v2) : ((r & 1) ? v1 : v0);
    }
    // softmax cross-entropy of sample r
    const float m = fmaxf(z[0], fmaxf(z[1], z[2]));
    const float e0 = expf(z[0] - m), e1 = expf(z[1] - m), e2 = expf(z[2] - m);
    const float S = e0 + e1 + e2;
    const float wv = valid ? ga.cw[yy] : 0.0f, gs = wv * ga.scale;
    const float pr[3] = {e0 / S, e1 / S, e2 / S};
    uint16_t dz[NOUT];
#pragma unroll
    for (int c = 0; c < NOUT; ++c) dz[c] = f2bf(gs * (pr[c] - (c == yy ? 1.0f : 0.0f)));
    if (w == 0 && g == 0) {
        const float zy = yy == 0 ? z[0] : yy == 1 ? z[1] : z[2];
        ga.loss[loc] = wv > 0.0f ? gs * (logf(S) - (zy - m)) : 0.0f;
#pragma unroll
        for (int c = 0; c < NOUT; ++c) ga.dZ[(size_t)c * ga.ld + loc] = dz[c];
    }
    // dA2 = (dZ W3) * [H2 > 0]: classes 4g..4g+3 of sample r, all but 0..2 zero
    s4v az = s4v{0, 0, 0, 0};
    if (g == 0)
#pragma unroll
        for (int c = 0; c < NOUT; ++c) az[c] = (short)dz[c];
    acc = mfma(az, w3t, f4v{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int t = 0; t < 4; ++t) da[t] = f2bf(bf2f(h2[t]) > 0.0f ? acc[t] : 0.0f);
    put(da, a2s, ga.dA2);
    __syncthreads();
    // dA1 = (dA2 W2) * [H1 > 0]
    acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) acc = mfma32(*(const s8v *)&a2s[r * SH + 32 * kk + 8 * g], w2t[kk], acc);
#pragma unroll
    for (int t = 0; t < 4; ++t) da[t] = f2bf(bf2f(h1[t]) > 0.0f ? acc[t] : 0.0f);
    put(da, nullptr, ga.dA1);
}

// Weight gradients of one partial sum (blockIdx.x), reductions over samples.
// blockIdx.y 0..2: dW1 += dA1^T X for 128 features, wave w hidden tile w.  A lane
// loads eight consecutive features (16 bytes) of its eight samples and pairs
// samples by byte permutes, so feature tile j is features 8r + j: no transpose
// through LDS.  blockIdx.y 3: dW2, dW3, biases and loss.
constexpr int WG_FEATURES = 128;
__global__ __launch_bounds__(BLK) void wgrad_kernel(GradArgs ga)
{
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * ga.chunks * ROWS, rows = ga.chunks * ROWS;
    float *const part = ga.partial + (size_t)blockIdx.x * NPP;
    if (blockIdx.y < NIN / WG_FEATURES) {
        const int f0 = WG_FEATURES * blockIdx.y + 8 * r;
        f4v acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = f4v{0.f, 0.f, 0.f, 0.f};
        // a chunk's loads in flight together, the ids of its rows a chunk ahead
        long long src[2][8];
        auto ids = [&](int c0) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const long long gi = ga.first + min(c0 + 32 * k + 8 * g + t, ga.count - 1);
                    src[k][t] = ga.perm ? (long long)ga.perm[gi] : gi;
                }
        };
        ids(row0);
        for (int c0 = row0; c0 < row0 + rows; c0 += ROWS) {
            s8v a[2];
            uint4 x[2][8];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                a[k] = *(const s8v *)(ga.dA1 + (size_t)(16 * w + r) * ga.ld + c0 + 32 * k + 8 * g);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    x[k][t] = *(const uint4 *)(ga.X + (size_t)src[k][t] * NIN + f0);
                    if (c0 + 32 * k + 8 * g + t >= ga.count) x[k][t] = make_uint4(0u, 0u, 0u, 0u);
                }
            }
            ids(min(c0 + ROWS, row0 + rows - ROWS));
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    union { unsigned u[4]; s8v v; } b;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const unsigned lo = (&x[k][2 * q].x)[j >> 1], hi = (&x[k][2 * q + 1].x)[j >> 1];
                        // halves j & 1 of two samples, the first one low
                        b.u[q] = __builtin_amdgcn_perm(hi, lo, (j & 1) ? 0x07060302u : 0x05040100u);
                    }
                    acc[j] = mfma32(a[k], b.v, acc[j]);
                }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float *o = part + OW1 + (16 * w + 4 * g + t) * NIN + f0;
            *(float4 *)o = make_float4(acc[0][t], acc[1][t], acc[2][t], acc[3][t]);
            *(float4 *)(o + 4) = make_float4(acc[4][t], acc[5][t], acc[6][t], acc[7][t]);
        }
        return;
    }
    f4v g2[4], g3 = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) g2[c] = f4v{0.f, 0.f, 0.f, 0.f};
    for (int s0 = row0; s0 < row0 + rows; s0 += 32) {
        auto units = [&](const uint16_t *T, int u) { return *(const s8v *)(T + (size_t)u * ga.ld + s0 + 8 * g); };
        const s8v a = units(ga.dA2, 16 * w + r);
#pragma unroll
        for (int c = 0; c < 4; ++c) g2[c] = mfma32(a, units(ga.H1, 16 * c + r), g2[c]);
        const s8v z = r < NOUT ? units(ga.dZ, r) : s8v{0, 0, 0, 0, 0, 0, 0, 0};
        g3 = mfma32(z, units(ga.H2, 16 * w + r), g3);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int t = 0; t < 4; ++t) part[OW2 + (16 * w + 4 * g + t) * NH + 16 * c + r] = g2[c][t];
    if (g == 0)
#pragma unroll
        for (int t = 0; t < NOUT; ++t) part[OW3 + t * NH + 16 * w + r] = g3[t];
    // bias gradients and loss: each chunk's samples in order, then the chunks
    if (tid >= 2 * NH + NOUT + 1) return;
    const uint16_t *const T = tid < NH ? ga.dA1 + (size_t)tid * ga.ld
                              : tid < 2 * NH ? ga.dA2 + (size_t)(tid - NH) * ga.ld
                                             : ga.dZ + (size_t)min(tid - 2 * NH, NOUT - 1) * ga.ld;
    float sum = 0.0f;
    for (int k = 0; k < ga.chunks; ++k) {
        const int c0 = row0 + k * ROWS;
        float acc = 0.0f;
        if (tid < 2 * NH + NOUT) {
            uint4 v[ROWS / 8];
#pragma unroll
            for (int q = 0; q < ROWS / 8; ++q) v[q] = *(const uint4 *)(T + c0 + 8 * q);
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const unsigned d = (&v[q / 8].x)[(q % 8) / 2];
                acc += bf2f((uint16_t)((q & 1) ? d >> 16 : d & 0xffffu));
            }
        } else {
            float v[ROWS];
#pragma unroll
            for (int q = 0; q < ROWS; ++q) v[q] = ga.loss[c0 + q];
#pragma unroll
            for (int q = 0; q < ROWS; ++q) acc += v[q];
        }
        sum += acc;
    }
    part[tid < NH ? OB1 + tid : tid < 2 * NH ? OB2 + tid - NH : tid < 2 * NH + NOUT ? OB3 + tid - 2 * NH : NP] = sum;
}

struct AdamArgs {
    int on;
    float lr, beta1, beta2, eps, bc1, bc2;   // bc = 1 / (1 - beta^t)
};

// Sum of the partials in their order; optional Adam update and BF16 copies.  The
// loads of AHEAD partials are in flight together (the sum stays sequential): with
// one after the other their latency was most of the kernel's time.
__device__ __forceinline__ void put_bf16(int p, float x, uint16_t *W1b, uint16_t *W2b, uint16_t *W2t, uint16_t *W3b)
{
    const uint16_t v = f2bf(x);
    if (p < OB1) {
        W1b[p] = v;
    } else if (p >= OW2 && p < OB2) {
        const int q = p - OW2;
        W2b[q] = v;
        W2t[(q % NH) * NH + q / NH] = v;
    } else if (p >= OW3 && p < OB3) {
        W3b[p - OW3] = v;
    }
}

__global__ __launch_bounds__(64) void reduce_kernel(const float *__restrict__ partial, int nparts,
                                                    float *__restrict__ grad, float *__restrict__ loss, float *P,
                                                    float *M, float *V, uint16_t *W1b, uint16_t *W2b, uint16_t *W2t,
                                                    uint16_t *W3b, AdamArgs ad)
{
#pragma clang fp contract(off)
    constexpr int AHEAD = 32;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > NP) return;
    const bool param = ad.on && p < NP;
    const float m0 = param ? M[p] : 0.0f, v0 = param ? V[p] : 0.0f, x0 = param ? P[p] : 0.0f;
    float gsum = 0.0f;
    int b = 0;
    for (; b + AHEAD <= nparts; b += AHEAD) {
        float v[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) v[k] = partial[(size_t)(b + k) * NPP + p];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) gsum += v[k];
    }
#pragma unroll 8
    for (; b < nparts; ++b) gsum += partial[(size_t)b * NPP + p];
    if (p == NP) {
        if (loss) *loss = gsum;
        return;
    }
    if (grad) grad[p] = gsum;
    if (!ad.on) return;
    // the multiply-adds are written out: an update's bits do not depend on what
    // the compiler finds to fuse
    const float m = fmaf(1.0f - ad.beta1, gsum, ad.beta1 * m0);
    const float v = fmaf(gsum, (1.0f - ad.beta2) * gsum, ad.beta2 * v0);
    M[p] = m;
    V[p] = v;
    const float x = x0 - ad.lr * (m * ad.bc1) / (sqrtf(v * ad.bc2) + ad.eps);
    P[p] = x;
    put_bf16(p, x, W1b, W2b, W2t, W3b);
}

__global__ void bf16_copy_kernel(const float *P, uint16_t *W1b, uint16_t *W2b, uint16_t *W2t, uint16_t *W3b)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NP) put_bf16(p, P[p], W1b, W2b, W2t, W3b);
}

#define MCHK(x)                                                                               \
    do {                                                                                      \
        hipError_t e_ = (x);                                                                  \
        if (e_ != hipSuccess) {                                                               \
            amr_set_error("%s:%d %s: %s", __FILE__, __LINE__, #x, hipGetErrorString(e_));     \
            return AMRGPU_ERR_HIP;                                                            \
        }                                                                                     \
    } while (0)

uint64_t splitmix64(uint64_t &s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
double uniform01(uint64_t &s) { return (double)(splitmix64(s) >> 11) * (1.0 / 9007199254740992.0); }

template <class T>
int grow(T **p, size_t *cap, size_t need, bool keep, size_t used)
{
    if (need <= *cap) return AMRGPU_OK;
    size_t nc = std::max(need, *cap + *cap / 2);
    T *q = nullptr;
    MCHK(hipMalloc((void **)&q, sizeof(T) * nc));
    if (keep && *p && used) MCHK(hipMemcpy(q, *p, sizeof(T) * used, hipMemcpyDeviceToDevice));
    if (*p) (void)hipFree(*p);
    *p = q;
    *cap = nc;
    return AMRGPU_OK;
}

}  // namespace

struct amr_mlp {
    hipStream_t stream = nullptr;
    float *P = nullptr, *M = nullptr, *V = nullptr, *grad = nullptr, *loss = nullptr;
    uint16_t *W1b = nullptr, *W2b = nullptr, *W2t = nullptr, *W3b = nullptr;
    float *partial = nullptr;
    size_t cap_partial = 0;
    uint16_t *act = nullptr;    // GradArgs' activations and gradients
    float *row_loss = nullptr;
    size_t cap_act = 0, cap_row_loss = 0;
    uint16_t *X = nullptr;      // scratch rows (host uploads, context features)
    size_t cap_X = 0;
    int *y = nullptr, *perm = nullptr, *cls = nullptr;
    size_t cap_y = 0, cap_perm = 0, cap_cls = 0;
    float *logits = nullptr;
    size_t cap_logits = 0;
    long long step = 0;
    float refine_bias = 0.0f;
    int cu_count = 256;         // compute units of the device
};

struct amr_tagset {
    uint16_t *X = nullptr;
    int *y = nullptr;
    size_t cap = 0, capy = 0;
    int n = 0;
    std::vector<int> h_y;
    std::vector<double> h_ind;
};

namespace {

Weights weights_of(const amr_mlp *m) { return Weights{m->W1b, m->W2b, m->W3b, m->W2t, m->P}; }

int launch_infer(amr_mlp *m, const uint16_t *dX, int count, float *dlogits, int *dcls, hipStream_t st)
{
    if (count <= 0) return AMRGPU_OK;
    const int grid = std::min((count + 16 * IWAVES - 1) / (16 * IWAVES), 2 * m->cu_count);     // two workgroups a CU
    hipLaunchKernelGGL(infer_kernel, dim3(grid), dim3(64 * IWAVES), 0, st, weights_of(m), dX, count, m->refine_bias,
                       dlogits, dcls);
    MCHK(hipGetLastError());
    return AMRGPU_OK;
}

// One gradient evaluation over `count` rows; partial sums reduced into
// m->grad / m->loss, with an Adam step when ad.on.
int launch_grad(amr_mlp *m, const uint16_t *dX, const int *dy, const int *dperm, long long first, int count,
                const float cw[3], float scale, int chunks, const AdamArgs &ad, float *dloss)
{
    int nblk = (count + ROWS * chunks - 1) / (ROWS * chunks);
    const size_t ld = (size_t)nblk * chunks * ROWS;
    int rc = grow(&m->partial, &m->cap_partial, (size_t)nblk * NPP, false, 0);
    if (!rc) rc = grow(&m->act, &m->cap_act, ld * (4 * NH + NOUT), false, 0);
    if (!rc) rc = grow(&m->row_loss, &m->cap_row_loss, ld, false, 0);
    if (rc) return rc;
    GradArgs ga;
    ga.X = dX; ga.y = dy; ga.perm = dperm; ga.first = first; ga.count = count; ga.chunks = chunks;
    ga.ld = (int)ld;
    ga.cw[0] = cw[0]; ga.cw[1] = cw[1]; ga.cw[2] = cw[2];
    ga.scale = scale;
    ga.H1 = m->act; ga.H2 = ga.H1 + ld * NH; ga.dA1 = ga.H2 + ld * NH; ga.dA2 = ga.dA1 + ld * NH;
    ga.dZ = ga.dA2 + ld * NH;
    ga.loss = m->row_loss;
    ga.partial = m->partial;
    hipLaunchKernelGGL(backprop_kernel, dim3((unsigned)(ld / 16)), dim3(BLK), 0, m->stream, weights_of(m), ga);
    MCHK(hipGetLastError());
    hipLaunchKernelGGL(wgrad_kernel, dim3(nblk, NIN / WG_FEATURES + 1), dim3(BLK), 0, m->stream, ga);
    MCHK(hipGetLastError());
    hipLaunchKernelGGL(reduce_kernel, dim3((NP + 1 + 63) / 64), dim3(64), 0, m->stream, m->partial, nblk,
                       m->grad, dloss, m->P, m->M, m->V, m->W1b, m->W2b, m->W2t, m->W3b, ad);
    MCHK(hipGetLastError());
    return AMRGPU_OK;
}

void default_weights(const std::vector<int> &y, int n, float cw[3])
{
    long long cnt[3] = {0, 0, 0};
    for (int i = 0; i < n; ++i) cnt[y[i]]++;
    for (int c = 0; c < 3; ++c) {
        double v = cnt[c] ? (double)n / (3.0 * (double)cnt[c]) : 1.0;
        cw[c] = (float)std::min(20.0, std::max(0.2, v));
    }
}

}  // namespace

extern "C" {

amr_mlp_t *amr_mlp_create(unsigned long long seed)
{
    amr_mlp *m = new amr_mlp();
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && ncu > 0)
        m->cu_count = ncu;
    std::vector<float> P(NP, 0.0f);
    uint64_t s = seed * 0x2545F4914F6CDD1Dull + 1;
    const double a1 = std::sqrt(6.0 / NIN), a2 = std::sqrt(6.0 / NH);
    for (int i = 0; i < NH * NIN; ++i) P[OW1 + i] = (float)((2.0 * uniform01(s) - 1.0) * a1);
    for (int i = 0; i < NH * NH; ++i) P[OW2 + i] = (float)((2.0 * uniform01(s) - 1.0) * a2);
    for (int i = 0; i < NOUT * NH; ++i) P[OW3 + i] = (float)((2.0 * uniform01(s) - 1.0) * a2);
    bool ok = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->P, sizeof(float) * NP) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->M, sizeof(float) * NP) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->V, sizeof(float) * NP) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->grad, sizeof(float) * NP) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->loss, sizeof(float) * 4) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->W1b, sizeof(uint16_t) * NH * NIN) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->W2b, sizeof(uint16_t) * NH * NH) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->W2t, sizeof(uint16_t) * NH * NH) == hipSuccess;
    ok = ok && hipMalloc((void **)&m->W3b, sizeof(uint16_t) * 16 * NH) == hipSuccess;
    ok = ok && hipMemset(m->W3b, 0, sizeof(uint16_t) * 16 * NH) == hipSuccess;
    if (!ok) {
        amr_set_error("amr_mlp_create: device allocation failed");
        amr_mlp_destroy(m);
        return nullptr;
    }
    if (amr_mlp_set_params(m, P.data())) {
        amr_mlp_destroy(m);
        return nullptr;
    }
    return m;
}

void amr_mlp_destroy(amr_mlp_t *m)
{
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    void *bufs[] = {m->P, m->M, m->V, m->grad, m->loss, m->W1b, m->W2b, m->W2t, m->W3b, m->partial, m->act, m->row_loss,
                    m->X, m->y, m->perm, m->cls, m->logits};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int amr_mlp_get_params(amr_mlp_t *m, float *params)
{
    if (!m || !params) { amr_set_error("amr_mlp_get_params: null argument"); return AMRGPU_ERR_ARG; }
    MCHK(hipStreamSynchronize(m->stream));
    MCHK(hipMemcpy(params, m->P, sizeof(float) * NP, hipMemcpyDeviceToHost));
    return AMRGPU_OK;
}

int amr_mlp_set_params(amr_mlp_t *m, const float *params)
{
    if (!m || !params) { amr_set_error("amr_mlp_set_params: null argument"); return AMRGPU_ERR_ARG; }
    MCHK(hipStreamSynchronize(m->stream));
    MCHK(hipMemcpy(m->P, params, sizeof(float) * NP, hipMemcpyHostToDevice));
    MCHK(hipMemset(m->M, 0, sizeof(float) * NP));
    MCHK(hipMemset(m->V, 0, sizeof(float) * NP));
    hipLaunchKernelGGL(bf16_copy_kernel, dim3((NP + 255) / 256), dim3(256), 0, m->stream, m->P, m->W1b, m->W2b,
                       m->W2t, m->W3b);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(m->stream));
    m->step = 0;
    return AMRGPU_OK;
}

int amr_mlp_set_refine_bias(amr_mlp_t *m, float bias)
{
    if (!m || !std::isfinite(bias)) { amr_set_error("amr_mlp_set_refine_bias: bad argument"); return AMRGPU_ERR_ARG; }
    m->refine_bias = bias;
    return AMRGPU_OK;
}

int amr_mlp_forward(amr_mlp_t *m, const uint16_t *X, int n, float *logits)
{
    if (!m || n < 0 || (n && (!X || !logits))) { amr_set_error("amr_mlp_forward: bad argument"); return AMRGPU_ERR_ARG; }
    if (!n) return AMRGPU_OK;
    int rc = grow(&m->X, &m->cap_X, (size_t)n * NIN, false, 0);
    if (!rc) rc = grow(&m->logits, &m->cap_logits, (size_t)n * 3, false, 0);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(m->X, X, sizeof(uint16_t) * n * NIN, hipMemcpyHostToDevice, m->stream));
    rc = launch_infer(m, m->X, n, m->logits, nullptr, m->stream);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(logits, m->logits, sizeof(float) * n * 3, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return AMRGPU_OK;
}

int amr_mlp_grad(amr_mlp_t *m, const uint16_t *X, const int *y, int n, const float cw[3], float *grad,
                 float *loss)
{
    if (!m || !X || !y || n <= 0 || !cw || !grad) { amr_set_error("amr_mlp_grad: bad argument"); return AMRGPU_ERR_ARG; }
    double sw = 0.0;
    for (int i = 0; i < n; ++i) {
        if (y[i] < 0 || y[i] > 2) { amr_set_error("amr_mlp_grad: label %d of row %d", y[i], i); return AMRGPU_ERR_ARG; }
        sw += cw[y[i]];
    }
    if (!(sw > 0.0)) { amr_set_error("amr_mlp_grad: zero total weight"); return AMRGPU_ERR_ARG; }
    int rc = grow(&m->X, &m->cap_X, (size_t)n * NIN, false, 0);
    if (!rc) rc = grow(&m->y, &m->cap_y, (size_t)n, false, 0);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(m->X, X, sizeof(uint16_t) * n * NIN, hipMemcpyHostToDevice, m->stream));
    MCHK(hipMemcpyAsync(m->y, y, sizeof(int) * n, hipMemcpyHostToDevice, m->stream));
    AdamArgs ad;
    memset(&ad, 0, sizeof(ad));
    rc = launch_grad(m, m->X, m->y, nullptr, 0, n, cw, (float)(1.0 / sw), 1, ad, m->loss);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(grad, m->grad, sizeof(float) * NP, hipMemcpyDeviceToHost, m->stream));
    float l = 0.0f;
    MCHK(hipMemcpyAsync(&l, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    if (loss) *loss = l;
    return AMRGPU_OK;
}

amr_tagset_t *amr_tagset_create(void) { return new amr_tagset(); }

void amr_tagset_destroy(amr_tagset_t *s)
{
    if (!s) return;
    if (s->X) (void)hipFree(s->X);
    if (s->y) (void)hipFree(s->y);
    delete s;
}

int amr_tagset_size(const amr_tagset_t *s) { return s ? s->n : 0; }

int amr_tagset_append(amr_tagset_t *s, const uint16_t *X, const int *y, const double *ind_now, int n)
{
    if (!s || n < 0 || (n && (!X || !y))) { amr_set_error("amr_tagset_append: bad argument"); return AMRGPU_ERR_ARG; }
    for (int i = 0; i < n; ++i)
        if (y[i] < 0 || y[i] > 2) { amr_set_error("amr_tagset_append: label %d of row %d", y[i], i); return AMRGPU_ERR_ARG; }
    size_t need = (size_t)s->n + n;
    int rc = grow(&s->X, &s->cap, need * NIN, true, (size_t)s->n * NIN);
    if (!rc) rc = grow(&s->y, &s->capy, need, true, (size_t)s->n);
    if (rc) return rc;
    MCHK(hipMemcpy(s->X + (size_t)s->n * NIN, X, sizeof(uint16_t) * n * NIN, hipMemcpyHostToDevice));
    MCHK(hipMemcpy(s->y + s->n, y, sizeof(int) * n, hipMemcpyHostToDevice));
    s->h_y.insert(s->h_y.end(), y, y + n);
    for (int i = 0; i < n; ++i) s->h_ind.push_back(ind_now ? ind_now[i] : 0.0);
    s->n += n;
    return AMRGPU_OK;
}

int amr_tagset_get(const amr_tagset_t *s, int first, int n, uint16_t *X, int *y, double *ind_now)
{
    if (!s || first < 0 || n < 0 || first + n > s->n) { amr_set_error("amr_tagset_get: rows out of range"); return AMRGPU_ERR_ARG; }
    if (!n) return AMRGPU_OK;
    if (X) MCHK(hipMemcpy(X, s->X + (size_t)first * NIN, sizeof(uint16_t) * n * NIN, hipMemcpyDeviceToHost));
    if (y) memcpy(y, s->h_y.data() + first, sizeof(int) * n);
    if (ind_now) memcpy(ind_now, s->h_ind.data() + first, sizeof(double) * n);
    return AMRGPU_OK;
}

int amr_tagset_append_from(amr_tagset_t *dst, const amr_tagset_t *src, int first, int n)
{
    if (!dst || !src || dst == src || first < 0 || n < 0 || first + n > src->n) {
        amr_set_error("amr_tagset_append_from: rows out of range");
        return AMRGPU_ERR_ARG;
    }
    size_t need = (size_t)dst->n + n;
    int rc = grow(&dst->X, &dst->cap, need * NIN, true, (size_t)dst->n * NIN);
    if (!rc) rc = grow(&dst->y, &dst->capy, need, true, (size_t)dst->n);
    if (rc) return rc;
    if (n) {
        MCHK(hipMemcpy(dst->X + (size_t)dst->n * NIN, src->X + (size_t)first * NIN, sizeof(uint16_t) * n * NIN,
                       hipMemcpyDeviceToDevice));
        MCHK(hipMemcpy(dst->y + dst->n, src->y + first, sizeof(int) * n, hipMemcpyDeviceToDevice));
    }
    dst->h_y.insert(dst->h_y.end(), src->h_y.begin() + first, src->h_y.begin() + first + n);
    dst->h_ind.insert(dst->h_ind.end(), src->h_ind.begin() + first, src->h_ind.begin() + first + n);
    dst->n += n;
    return AMRGPU_OK;
}

int amrgpu_tagger_features(amrgpu_ctx *c, uint16_t *d_X)
{
    const double *U;
    const int *nbr;
    int nquad, n;
    void *st;
    int rc = amrgpu_device_state(c, &U, &nbr, &nquad, &n, &st);
    if (rc) return rc;
    if (n != 8 && n != 16) {
        amr_set_error("tagger features need 8x8 or 16x16 patches (got %d)", n);
        return AMRGPU_ERR_ARG;
    }
    if (!d_X) { amr_set_error("amrgpu_tagger_features: null output"); return AMRGPU_ERR_ARG; }
    if (n == 16) {
        // the features of the patches coarsened to 8x8, in the context's
        // staging buffer (a quarter of one state vector)
        double *P;
        size_t cap;
        rc = amrgpu_staging(c, &P, &cap);
        if (rc) return rc;
        if (cap < (size_t)nquad * 256) { amr_set_error("amrgpu_tagger_features: staging too small"); return AMRGPU_ERR_ARG; }
        hipLaunchKernelGGL(pool16_kernel, dim3((unsigned)(((long long)nquad * 64 + 255) / 256)), dim3(256), 0,
                           (hipStream_t)st, U, P, nquad);
        MCHK(hipGetLastError());
        U = P;
    }
    hipLaunchKernelGGL(features_kernel, dim3((nquad + 3) / 4), dim3(256), 0, (hipStream_t)st, U, nbr, nquad, d_X);
    MCHK(hipGetLastError());
    return AMRGPU_OK;
}

int amrgpu_tagger_features_host(amrgpu_ctx *c, uint16_t *X)
{
    int nquad = amrgpu_num_quads(c);
    void *st;
    int rc = amrgpu_device_state(c, nullptr, nullptr, nullptr, nullptr, &st);
    if (rc) return rc;
    if (!X) { amr_set_error("amrgpu_tagger_features_host: null output"); return AMRGPU_ERR_ARG; }
    uint16_t *d = nullptr;
    MCHK(hipMalloc((void **)&d, sizeof(uint16_t) * (size_t)nquad * NIN));
    rc = amrgpu_tagger_features(c, d);
    if (!rc) rc = amrgpu_fetch(c, X, d, sizeof(uint16_t) * (size_t)nquad * NIN);
    (void)hipFree(d);
    return rc;
}

int amr_mlp_train(amr_mlp_t *m, const amr_tagset_t *s, int epochs, int batch, float lr, const float *cw_in,
                  unsigned long long seed, float *loss)
{
    if (!m || !s || epochs < 0 || batch <= 0 || batch % ROWS || s->n < batch || !(lr > 0.0f)) {
        amr_set_error("amr_mlp_train: bad argument (batch %d, rows %d)", batch, s ? s->n : 0);
        return AMRGPU_ERR_ARG;
    }
    const int N = s->n, nb = N / batch;
    float cw[3];
    if (cw_in) memcpy(cw, cw_in, sizeof(cw));
    else default_weights(s->h_y, N, cw);
    const int chunks = std::max(1, batch / (ROWS * 32));
    int rc = grow(&m->perm, &m->cap_perm, (size_t)N, false, 0);
    if (!rc) rc = grow(&m->logits, &m->cap_logits, (size_t)nb, false, 0);   // per-minibatch losses
    if (rc) return rc;
    std::vector<int> perm(N);
    std::vector<float> lb(nb);
    for (int i = 0; i < N; ++i) perm[i] = i;
    AdamArgs ad;
    ad.on = 1;
    ad.lr = lr;
    ad.beta1 = 0.9f;
    ad.beta2 = 0.999f;
    ad.eps = 1e-8f;
    for (int e = 0; e < epochs; ++e) {
        uint64_t st = seed * 0x9E3779B97F4A7C15ull + (uint64_t)e + 1;
        for (int i = N - 1; i > 0; --i) {
            int j = (int)(splitmix64(st) % (uint64_t)(i + 1));
            std::swap(perm[i], perm[j]);
        }
        MCHK(hipMemcpyAsync(m->perm, perm.data(), sizeof(int) * N, hipMemcpyHostToDevice, m->stream));
        for (int b = 0; b < nb; ++b) {
            double sw = 0.0;
            for (int i = 0; i < batch; ++i) sw += cw[s->h_y[perm[(size_t)b * batch + i]]];
            m->step++;
            ad.bc1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)m->step)));
            ad.bc2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)m->step)));
            rc = launch_grad(m, s->X, s->y, m->perm, (long long)b * batch, batch, cw, (float)(1.0 / sw), chunks,
                             ad, m->logits + b);
            if (rc) return rc;
        }
        MCHK(hipMemcpyAsync(lb.data(), m->logits, sizeof(float) * nb, hipMemcpyDeviceToHost, m->stream));
        MCHK(hipStreamSynchronize(m->stream));
        if (loss) {
            double a = 0.0;
            for (int b = 0; b < nb; ++b) a += lb[b];
            loss[e] = (float)(a / nb);
        }
    }
    return AMRGPU_OK;
}

int amr_mlp_predict_set(amr_mlp_t *m, const amr_tagset_t *s, int *cls)
{
    if (!m || !s || (s->n && !cls)) { amr_set_error("amr_mlp_predict_set: bad argument"); return AMRGPU_ERR_ARG; }
    if (!s->n) return AMRGPU_OK;
    int rc = grow(&m->cls, &m->cap_cls, (size_t)s->n, false, 0);
    if (!rc) rc = launch_infer(m, s->X, s->n, nullptr, m->cls, m->stream);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(cls, m->cls, sizeof(int) * s->n, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return AMRGPU_OK;
}

int amr_mlp_predict_ctx(amr_mlp_t *m, amrgpu_ctx *c, int *cls)
{
    if (!m || !c || !cls) { amr_set_error("amr_mlp_predict_ctx: bad argument"); return AMRGPU_ERR_ARG; }
    void *st;
    int nquad;
    int rc = amrgpu_device_state(c, nullptr, nullptr, &nquad, nullptr, &st);
    if (!rc) rc = grow(&m->X, &m->cap_X, (size_t)nquad * NIN, false, 0);
    if (!rc) rc = grow(&m->cls, &m->cap_cls, (size_t)nquad, false, 0);
    if (!rc) rc = amrgpu_tagger_features(c, m->X);
    if (!rc) rc = launch_infer(m, m->X, nquad, nullptr, m->cls, (hipStream_t)st);
    if (rc) return rc;
    return amrgpu_fetch(c, cls, m->cls, sizeof(int) * (size_t)nquad);
}

}  // extern "C"
