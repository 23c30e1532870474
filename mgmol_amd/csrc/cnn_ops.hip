// cnn_ops.hip -- the learned orbital preconditioner: a 4-layer 3D CNN
// (1 -> 16 -> 16 -> 16 -> 1 channels, 3^3 taps, zero padding on each box,
// bias, ReLU after layers 0-2, scalar skip y = s x + conv3(h3)) with BF16
// weights and activations and FP32 accumulation on MFMA, its backward pass,
// Adam training, and inference on a box set.  It has no counterpart in the
// reference; it maps an orbital residual to a preconditioned correction in
// place of the V-cycle (Preconditioning::mg, src/Preconditioning.cc:155-216),
// which stays the fallback.
//
// Layouts.  Samples are cubes of edge e, sample s at s*e^3 (the packed box
// layout of a box set whose boxes all have edge e).  Activations are BF16
// [voxel][16] (channel fastest).  Master parameters are FP32, packed
//   w0[27][16][1] b0[16] w1[27][16][16] b1[16] w2[27][16][16] b2[16]
//   w3[27][1][16] b3[1] s
// with tap = (dx*3 + dy)*3 + dz for the offset (dx-1, dy-1, dz-1).
//
// Convolution as MFMA (v_mfma_f32_16x16x16_bf16): one wave computes a tile
// of 16 z-consecutive voxels x 16 output channels, D[cout][voxel] =
// sum_tap W_tap[cout][cin] X[cin][voxel + off(tap)]: A = weights (held in
// registers for all taps), B = input rows (8-byte loads, 16 voxels x 32 B
// contiguous per tap).  Lane l holds A[l%16][4(l/16)+i], B[4(l/16)+i][l%16]
// and D[4(l/16)+i][l%16].
#include "common.hpp"

#include <cmath>
#include <cstring>
#include <vector>

namespace mgx
{
namespace
{

constexpr int kCh      = 16;
constexpr int kTaps    = 27;
constexpr int kWaves   = 4;  // per block
constexpr int kDwBlocks = 512;  // most blocks of a 16 -> 16 weight gradient: two per CU
constexpr int kDwPad    = 256;  // bytes after the activations that its last rows read past their end

// parameter offsets (floats)
constexpr int kW0 = 0, kB0 = kW0 + 27 * 16, kW1 = kB0 + 16, kB1 = kW1 + 27 * 256, kW2 = kB1 + 16,
              kB2 = kW2 + 27 * 256, kW3 = kB2 + 16, kB3 = kW3 + 27 * 16, kS = kB3 + 1, kNP = kS + 1;

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x32_bf16: lane l holds A[l%16][8(l/16)..8(l/16)+7],
// B[8(l/16)..8(l/16)+7][l%16], D[4(l/16)+i][l%16]
__device__ __forceinline__ f4 mfma32(s8 a, s8 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0,
        0);
}

__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

__device__ inline int tap_dx(int t) { return t / 9 - 1; }
__device__ inline int tap_dy(int t) { return (t / 3) % 3 - 1; }
__device__ inline int tap_dz(int t) { return t % 3 - 1; }

struct TileIx
{
    int s, x, y, z0;
};

__device__ inline TileIx decode(int64_t t, int e, int nzt)
{
    TileIx r;
    const int64_t per = (int64_t)e * e * nzt;
    r.s               = (int)(t / per);
    int64_t q         = t - (int64_t)r.s * per;
    r.x               = (int)(q / ((int64_t)e * nzt));
    q -= (int64_t)r.x * e * nzt;
    r.y  = (int)(q / nzt);
    r.z0 = (int)(q - (int64_t)r.y * nzt) * 16;
    return r;
}

enum
{
    CONV_FWD_RELU = 0,  // + bias, ReLU, BF16 out
    CONV_FWD_LIN  = 1,  // + bias, FP32 out (last layer)
    CONV_BWD_MASK = 2   // no bias, times (hmask > 0), BF16 out
};

// One conv layer over nt tiles.  CIN = 1: input FP32 scalar per voxel,
// weights [16 cout][32 taps] BF16 (taps >= 27 zero).  CIN = 16: input BF16
// [voxel][16], weights [27][16 cout][16 cin] BF16.  COUT = 16: output
// [voxel][16]; COUT = 1: FP32 scalar (row 0 of D; weights rows 1..15 zero).
template <int CIN, int COUT, int MODE>
__global__ void __launch_bounds__(64 * kWaves) k_conv(const void* __restrict__ in, const uint16_t* __restrict__ wt,
    const float* __restrict__ bias, void* __restrict__ out, const uint16_t* __restrict__ hmask, int e, int nzt,
    int64_t nt)
{
    const int64_t t = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (t >= nt) return;  // whole wave
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const TileIx T = decode(t, e, nzt);
    const int64_t sbase = (int64_t)T.s * e * e * e;
    f4 acc = { 0.f, 0.f, 0.f, 0.f };
    if (CIN == 16)
    {
        // all 27 input loads in flight before the MFMA chain
        const uint16_t* X = (const uint16_t*)in;
        s4 b[kTaps];
#pragma unroll
        for (int tap = 0; tap < kTaps; tap++)
        {
            const int xi = T.x + tap_dx(tap), yi = T.y + tap_dy(tap), zi = T.z0 + n + tap_dz(tap);
            b[tap] = (s4){ 0, 0, 0, 0 };
            if (xi >= 0 && xi < e && yi >= 0 && yi < e && zi >= 0 && zi < e)
                b[tap] = *(const s4*)(X + (sbase + ((int64_t)xi * e + yi) * e + zi) * 16 + 4 * g);
        }
#pragma unroll
        for (int tap = 0; tap < kTaps; tap++)
        {
            const s4 a = *(const s4*)(wt + ((size_t)tap * 16 + n) * 16 + 4 * g);
            acc        = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[tap], acc, 0, 0, 0);
        }
    }
    else
    {
        const float* X = (const float*)in;
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const s4 a = *(const s4*)(wt + (size_t)n * 32 + 16 * h + 4 * g);
            s4 b;
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const int tap = 16 * h + 4 * g + i;
                float v       = 0.f;
                if (tap < kTaps)
                {
                    const int xi = T.x + tap_dx(tap), yi = T.y + tap_dy(tap), zi = T.z0 + n + tap_dz(tap);
                    if (xi >= 0 && xi < e && yi >= 0 && yi < e && zi >= 0 && zi < e)
                        v = X[sbase + ((int64_t)xi * e + yi) * e + zi];
                }
                b[i] = (short)f2bf(v);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
        }
    }
    const int z = T.z0 + n;
    if (z >= e) return;
    const int64_t vox = sbase + ((int64_t)T.x * e + T.y) * e + z;
    if (COUT == 1)
    {
        if (g == 0) ((float*)out)[vox] = acc[0] + (MODE == CONV_BWD_MASK ? 0.f : bias[0]);
        return;
    }
    s4 o;
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        float v = acc[i];
        if (MODE == CONV_FWD_RELU) v = fmaxf(v + bias[4 * g + i], 0.f);
        if (MODE == CONV_FWD_LIN) v += bias[4 * g + i];
        if (MODE == CONV_BWD_MASK && hmask[vox * 16 + 4 * g + i] == 0) v = 0.f;
        o[i] = (short)f2bf(v);
    }
    *(s4*)((uint16_t*)out + vox * 16 + 4 * g) = o;
}

// A 16 -> 16 layer with the input staged in LDS: a block (4 waves) owns
// rows y0..y0+3 and z0..z0+31 of one sample and marches along x, keeping the
// planes x-1, x, x+1 of its (6 x 34)-voxel window in a ring of 3 LDS slots
// (one new plane loaded per step, 16-byte coalesced loads, zeros outside the
// box).  Wave w computes row y0+w, two 16-voxel z-tiles, 27 MFMAs each, with
// all 27 taps' weights in registers and the B operands read from LDS.
constexpr int kLY = 4, kLZ = 32, kLW = kLZ + 2, kLH = kLY + 2;
constexpr int kPlane = kLH * kLW * 16;  // BF16 values per staged plane

template <int MODE>
__global__ void __launch_bounds__(256) k_conv16_lds(const uint16_t* __restrict__ in, const uint16_t* __restrict__ wt,
    const float* __restrict__ bias, uint16_t* __restrict__ out, const uint16_t* __restrict__ hmask, int e, int nyb,
    int nzb)
{
    __shared__ __align__(16) uint16_t lds[3 * kPlane];
    const int b = blockIdx.x;
    const int s = b / (nyb * nzb), yb = (b / nzb) % nyb, zb = b % nzb;
    const int y0 = yb * kLY, z0 = zb * kLZ;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int64_t e3 = (int64_t)e * e * e;
    const uint16_t* X = in + (int64_t)s * e3 * 16;
    // K = 32 per MFMA: tap pair tp, lane group g: tap 2tp + (g >> 1), channels
    // 8(g & 1)..8(g & 1)+7 (the 28th tap is zero)
    constexpr int kPairs = (kTaps + 1) / 2;
    const int tsel = g >> 1, cs = 8 * (g & 1);
    s8 wa[kPairs];
#pragma unroll
    for (int tp = 0; tp < kPairs; tp++)
    {
        const int tap = 2 * tp + tsel;
        wa[tp]        = tap < kTaps ? *(const s8*)(wt + ((size_t)tap * 16 + n) * 16 + cs) : (s8){ 0, 0, 0, 0, 0, 0, 0, 0 };
    }
    // stage plane xp into slot, as 16-byte chunks (2 per voxel)
    auto stage = [&](int xp, int slot) {
        uint4* dst = (uint4*)(lds + slot * kPlane);
        for (int q = threadIdx.x; q < kLH * kLW * 2; q += blockDim.x)
        {
            const int vox = q >> 1, half = q & 1;
            const int yy = vox / kLW, zz = vox - (vox / kLW) * kLW;
            const int y = y0 - 1 + yy, z = z0 - 1 + zz;
            uint4 v = { 0u, 0u, 0u, 0u };
            if (xp >= 0 && xp < e && y >= 0 && y < e && z >= 0 && z < e)
                v = *(const uint4*)(X + (((int64_t)xp * e + y) * e + z) * 16 + 8 * half);
            dst[q] = v;
        }
    };
    stage(-1, 2);  // zeros
    stage(0, 0);
    const int y = y0 + wid;
    for (int x = 0; x < e; x++)
    {
        stage(x + 1, (x + 1) % 3);
        __syncthreads();
        f4 acc0 = { 0.f, 0.f, 0.f, 0.f }, acc1 = acc0;
#pragma unroll
        for (int tp = 0; tp < kPairs; tp++)
        {
            // the padding tap (27) reads tap 26's operands against zero weights
            const int tap  = min(2 * tp + tsel, kTaps - 1);
            const int slot = (x + 3 + tap_dx(tap)) % 3;
            const int yy   = wid + 1 + tap_dy(tap);
            const uint16_t* row = lds + slot * kPlane + (yy * kLW) * 16;
            const int zz = n + 1 + tap_dz(tap);
            const s8 b0 = *(const s8*)(row + zz * 16 + cs);
            const s8 b1 = *(const s8*)(row + (zz + 16) * 16 + cs);
            acc0 = mfma32(wa[tp], b0, acc0);
            acc1 = mfma32(wa[tp], b1, acc1);
        }
        if (y < e)
        {
#pragma unroll
            for (int t = 0; t < 2; t++)
            {
                const int z = z0 + 16 * t + n;
                if (z >= e) continue;
                const int64_t vox = (int64_t)s * e3 + ((int64_t)x * e + y) * e + z;
                const f4 a = t == 0 ? acc0 : acc1;
                s4 o;
#pragma unroll
                for (int i = 0; i < 4; i++)
                {
                    float v = a[i];
                    if (MODE == CONV_FWD_RELU) v = fmaxf(v + bias[4 * g + i], 0.f);
                    if (MODE == CONV_BWD_MASK && hmask[vox * 16 + 4 * g + i] == 0) v = 0.f;
                    o[i] = (short)f2bf(v);
                }
                *(s4*)(out + vox * 16 + 4 * g) = o;
            }
        }
        __syncthreads();
    }
}

// The first layer (1 -> 16 channels) with the scalar input staged in LDS
// as for k_conv16_lds: a ring of 3 planes of (6 x 34) values; one 16x16x32
// MFMA per 16-voxel tile covers all 27 taps (K = tap, lane group g holds taps
// 8g..8g+7, the last 5 zero).  Bias and ReLU; BF16 out.
template <typename TIN>
__global__ void __launch_bounds__(256) k_conv1_lds(const TIN* __restrict__ in, const double* __restrict__ rms,
    const uint16_t* __restrict__ wt, const float* __restrict__ bias, uint16_t* __restrict__ out, int e, int nyb,
    int nzb)
{
    constexpr int kP1 = kLH * kLW;
    __shared__ float lds[3 * kP1];
    const int b = blockIdx.x;
    const int s = b / (nyb * nzb), yb = (b / nzb) % nyb, zb = b % nzb;
    const int y0 = yb * kLY, z0 = zb * kLZ;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int64_t e3 = (int64_t)e * e * e;
    const TIN* X = in + (int64_t)s * e3;
    // inputs R / rms (the box's normalised residual) when rms is given
    const double rs = rms ? rms[s] : 1.;
    // A: W0[cout = n][taps 8g..8g+7] from the [16][32] layout
    const s8 wa = *(const s8*)(wt + (size_t)n * 32 + 8 * g);
    float bv4[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        bv4[i] = bias[4 * g + i];
    auto stage = [&](int xp, int slot) {
        float* dst = lds + slot * kP1;
        for (int q = threadIdx.x; q < kP1; q += blockDim.x)
        {
            const int yy = q / kLW, zz = q - (q / kLW) * kLW;
            const int y = y0 - 1 + yy, z = z0 - 1 + zz;
            float v = 0.f;
            if (xp >= 0 && xp < e && y >= 0 && y < e && z >= 0 && z < e)
            {
                const TIN r = X[((int64_t)xp * e + y) * e + z];
                v           = rms ? (float)((double)r / rs) : (float)r;
            }
            dst[q] = v;
        }
    };
    stage(-1, 2);
    stage(0, 0);
    const int y = y0 + wid;
    for (int x = 0; x < e; x++)
    {
        stage(x + 1, (x + 1) % 3);
        __syncthreads();
        s8 b0, b1;
#pragma unroll
        for (int i = 0; i < 8; i++)
        {
            const int tap = 8 * g + i;
            float v0 = 0.f, v1 = 0.f;
            if (tap < kTaps)
            {
                const float* row = lds + ((x + 3 + tap_dx(tap)) % 3) * kP1 + (wid + 1 + tap_dy(tap)) * kLW;
                const int zz     = n + 1 + tap_dz(tap);
                v0               = row[zz];
                v1               = row[zz + 16];
            }
            b0[i] = (short)f2bf(v0);
            b1[i] = (short)f2bf(v1);
        }
        const f4 z4 = { 0.f, 0.f, 0.f, 0.f };
        const f4 acc0 = mfma32(wa, b0, z4), acc1 = mfma32(wa, b1, z4);
        if (y < e)
        {
#pragma unroll
            for (int t = 0; t < 2; t++)
            {
                const int z = z0 + 16 * t + n;
                if (z >= e) continue;
                const int64_t vox = (int64_t)s * e3 + ((int64_t)x * e + y) * e + z;
                const f4 a = t == 0 ? acc0 : acc1;
                s4 o;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    o[i] = (short)f2bf(fmaxf(a[i] + bv4[i], 0.f));
                *(s4*)(out + vox * 16 + 4 * g) = o;
            }
        }
        __syncthreads();
    }
}

// The last layer (16 -> 1 channel) with the input staged in LDS: a block
// owns rows y0..y0+7, z0..z0+31 of one sample (one voxel per thread) and
// marches along x with a ring of 3 planes of (10 x 34) voxels; the 27 x 16
// weights are LDS broadcasts of BF16 channel pairs, applied with the BF16
// dot2 instruction (FP32 accumulation):
//   z = b + sum_tap sum_ci W[tap][ci] h[v + off(tap)][ci]   (tap-major)
// With R non-null it also finishes the network on the box: y = s x + z with
// x = (float)(R / rms), written as (T)(y * rms) to out; otherwise z to zout.
constexpr int kOY = 8, kOH = kOY + 2;
template <typename T>
__global__ void __launch_bounds__(256) k_conv_out_lds(const uint16_t* __restrict__ h, const uint16_t* __restrict__ wt,
    const float* __restrict__ prm, float* __restrict__ zout, const double* __restrict__ R,
    const double* __restrict__ rms, T* __restrict__ out, int e, int nyb, int nzb)
{
    constexpr int kPO = kOH * kLW * 16;
    __shared__ __align__(16) uint16_t lds[3 * kPO];
    __shared__ uint32_t w[kTaps * 8];  // channel pairs (2k, 2k+1) of W[tap], BF16
    for (int q = threadIdx.x; q < kTaps * 8; q += blockDim.x)
    {
        const int tap = q / 8, k = q % 8;  // row 0 of the padded [27][16][16] layout
        w[q] = (uint32_t)wt[tap * 256 + 2 * k] | ((uint32_t)wt[tap * 256 + 2 * k + 1] << 16);
    }
    const int b = blockIdx.x;
    const int s = b / (nyb * nzb), yb = (b / nzb) % nyb, zb = b % nzb;
    const int y0 = yb * kOY, z0 = zb * kLZ;
    const int64_t e3 = (int64_t)e * e * e;
    const uint16_t* X = h + (int64_t)s * e3 * 16;
    auto stage = [&](int xp, int slot) {
        uint4* dst = (uint4*)(lds + slot * kPO);
        for (int q = threadIdx.x; q < kOH * kLW * 2; q += blockDim.x)
        {
            const int vox = q >> 1, half = q & 1;
            const int yy = vox / kLW, zz = vox - (vox / kLW) * kLW;
            const int y = y0 - 1 + yy, z = z0 - 1 + zz;
            uint4 v = { 0u, 0u, 0u, 0u };
            if (xp >= 0 && xp < e && y >= 0 && y < e && z >= 0 && z < e)
                v = *(const uint4*)(X + (((int64_t)xp * e + y) * e + z) * 16 + 8 * half);
            dst[q] = v;
        }
    };
    stage(-1, 2);
    stage(0, 0);
    const int ry = threadIdx.x >> 5, rz = threadIdx.x & 31;
    const int y = y0 + ry, z = z0 + rz;
    const float bias = prm[kB3], sk = prm[kS];
    const double rs  = rms ? rms[s] : 1.;
    for (int x = 0; x < e; x++)
    {
        stage(x + 1, (x + 1) % 3);
        __syncthreads();
        float acc = bias;
        for (int tap = 0; tap < kTaps; tap++)
        {
            const uint16_t* src = lds + ((x + 3 + tap_dx(tap)) % 3) * kPO
                                  + ((ry + 1 + tap_dy(tap)) * kLW + (rz + 1 + tap_dz(tap))) * 16;
            const uint4 a = ((const uint4*)src)[0], bq = ((const uint4*)src)[1];
            const uint32_t u[8] = { a.x, a.y, a.z, a.w, bq.x, bq.y, bq.z, bq.w };
            const uint32_t* wr  = w + tap * 8;
#pragma unroll
            for (int k = 0; k < 8; k++)
                acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, u[k]), __builtin_bit_cast(bf2, wr[k]),
                    acc, false);
        }
        if (y < e && z < e)
        {
            const int64_t vox = (int64_t)s * e3 + ((int64_t)x * e + y) * e + z;
            if (R)
            {
                const float xv = (float)(R[vox] / rs);
                const float yv = sk * xv + acc;
                out[vox]       = (T)((double)yv * rs);
            }
            else
                zout[vox] = acc;
        }
        __syncthreads();
    }
}

// The last layer (16 -> 1 channel) on the vector units: one output voxel per
// thread, the 27 x 16 weights and the bias in LDS (FP32 values of the BF16
// weights), two 16-byte loads per tap.  z = b + sum_tap sum_ci W[tap][ci] h[v + off(tap)][ci]
// in FP32, as the MFMA path accumulates it.
__global__ void __launch_bounds__(256) k_conv_out(const uint16_t* __restrict__ h, const uint16_t* __restrict__ wt,
    const float* __restrict__ bias, float* __restrict__ out, int e, int64_t nvox)
{
    __shared__ float w[kTaps * 16];
    for (int q = threadIdx.x; q < kTaps * 16; q += blockDim.x)
        w[q] = bf2f(wt[(q / 16) * 256 + (q % 16)]);  // row 0 of the padded [27][16][16] layout
    __syncthreads();
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    const int64_t e3 = (int64_t)e * e * e;
    const int64_t s  = v / e3;
    int r            = (int)(v - s * e3);
    const int x = r / (e * e), y = (r / e) % e, z = r % e;
    float acc = bias[0];
    for (int tap = 0; tap < kTaps; tap++)
    {
        const int xi = x + tap_dx(tap), yi = y + tap_dy(tap), zi = z + tap_dz(tap);
        if (xi < 0 || xi >= e || yi < 0 || yi >= e || zi < 0 || zi >= e) continue;
        const uint4* p = (const uint4*)(h + (s * e3 + ((int64_t)xi * e + yi) * e + zi) * 16);
        const uint4 a = p[0], b = p[1];
        const uint32_t u[8] = { a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w };
        const float* wr = w + tap * 16;
#pragma unroll
        for (int k = 0; k < 8; k++)
        {
            acc += wr[2 * k] * bf2f((uint16_t)(u[k] & 0xFFFFu));
            acc += wr[2 * k + 1] * bf2f((uint16_t)(u[k] >> 16));
        }
    }
    out[v] = acc;
}

// The two halves of a dword pair (a in the low half)
__device__ __forceinline__ uint32_t pack2(uint32_t a, uint32_t b) { return a | (b << 16); }

// Sums a block's four waves' accumulators (in wave order) through LDS and
// writes them to P: NA fragments D[4g+i][n] at ix(frag, 4g+i, n) of `tot`
// floats, then the 16 row sums of the last fragment (MFMA against ones).
template <int NA, class IX>
__device__ __forceinline__ void dw_block_sum(const f4 (&acc)[NA + 1], float* red, int tot, IX ix, float* __restrict__ P)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    for (int w = 0; w < kWaves; w++)
    {
        if (wid == w)
        {
#pragma unroll
            for (int k = 0; k < NA; k++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                {
                    const int q = ix(k, 4 * g + i, n);
                    if (q >= 0) red[q] = w == 0 ? acc[k][i] : red[q] + acc[k][i];
                }
            if (n == 0)
#pragma unroll
                for (int i = 0; i < 4; i++)
                {
                    const int q = tot + 4 * g + i;
                    red[q]      = w == 0 ? acc[NA][i] : red[q] + acc[NA][i];
                }
        }
        __syncthreads();
    }
    for (int q = threadIdx.x; q < tot + 16; q += blockDim.x)
        P[q] = red[q];
}

// Weight / bias gradient of a 16 -> 16 layer, per block of four waves:
//   dW[tap][cout][cin] = sum_v dZ[v][cout] H[v + off(tap)][cin],  db = sum_v dZ
// as 16x16x32 MFMAs over voxels: A = dZ^T, B = H.  Each group of 16 lanes
// (lane n = channel) owns a column (sample, x, 8 z-voxels) and marches along
// y, so K = 32 is four columns and any box edge fills the lanes.  At row y it
// holds H[x][y] shifted by dz = -1, 0, 1 (three fragments made from ten 2-byte
// loads) and the nine dZ rows (x - dx, y - dy) (three new ones per step, the
// others slide): 27 MFMAs per 34 loads, where one fragment per tap takes
// four loads each; the next step's loads are in flight during the MFMAs.
// Bound by those loads, not by the matrix cores.  64 boxes of 32^3: 41 us
// (0.71 PFLOP/s); one fragment per tap and voxel row took 1744 us.
// A wave takes the tasks (four columns, one chunk of yl rows) t, t + waves, ...
template <bool TAIL>
__global__ void __launch_bounds__(256, 2) k_dw16(const uint16_t* __restrict__ dz, const uint16_t* __restrict__ h,
    int e, int nzs, int ncol, int yl, int nyc, int ntask, float* __restrict__ part)
{
    __shared__ float red[kTaps * 256 + 16];
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    f4 acc[kTaps + 1];
#pragma unroll
    for (int k = 0; k <= kTaps; k++)
        acc[k] = (f4){ 0.f, 0.f, 0.f, 0.f };
    const s8 ones = { 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80 };
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    const int64_t rs = (int64_t)e * 16, ps = rs * e;  // row and plane strides
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int t = blockIdx.x * kWaves + wid; t < ntask; t += gridDim.x * kWaves)
    {
        const int cg = t / nyc, y0 = (t - cg * nyc) * yl, y1 = min(e, y0 + yl);
        const int c  = 4 * cg + g;
        const bool on = c < ncol;
        const int cc  = on ? c : 4 * cg;
        const int zs = cc % nzs, sx = cc / nzs, x = sx % e, z0 = zs * 8;
        // wave-uniform plane base (one plane before the first column's) and
        // this lane's 32-bit offsets from it: its own column's plane, channel n
        // and the ten z-neighbours (the values outside the row are masked)
        const int sx0          = __builtin_amdgcn_readfirstlane(4 * cg / nzs);
        const int64_t ubase    = ((int64_t)sx0 - 1) * ps;
        const uint32_t psb     = 2u * (uint32_t)ps;
        const uint32_t lane0   = (uint32_t)(sx - sx0 + 1) * psb + 2u * (uint32_t)(z0 * 16 + n);
        const uint32_t zlo     = z0 > 0 ? 32u : 0u;  // bytes back to z0 - 1
        // value j (z0 + j - 1) of the row at the wave-uniform address p; a
        // row's last segment reads on past its end (kDwPad at the end of a buffer)
        auto at = [&](const char* p, uint32_t o, int j) -> uint32_t {
            if (j == 0) return *(const uint16_t*)(p + (o - zlo));
            return *(const uint16_t*)(p + 32 * (j - 1) + o);
        };
        const uint32_t mlo = z0 > 0 ? 0xFFFFu : 0u;
        // position j of the segment is outside the box from j = e - z0 on
        const int jend = e - z0;
        uint32_t tm[4] = { ~0u, ~0u, ~0u, ~0u };
        if (TAIL)
        {
#pragma unroll
            for (int k = 0; k < 4; k++)
                tm[k] = (2 * k < jend ? 0xFFFFu : 0u) | (2 * k + 1 < jend ? 0xFFFF0000u : 0u);
        }
        const bool xlo = on && x > 0, xhi = on && x < e - 1;
        // dx = -1, 0, 1: plane x - dx
        const uint32_t dzo[3] = { lane0 + (xhi ? psb : 0u), lane0, lane0 - (xlo ? psb : 0u) };
        const bool dzv[3]    = { xhi, on, xlo };
        uint32_t rh[10], rz[3][8];
        auto load_h = [&](int y) {
            const char* p = (const char*)(h + (ubase + (int64_t)y * rs));
#pragma unroll
            for (int j = 0; j < 10; j++)
                rh[j] = at(p, lane0, j);
        };
        auto load_z = [&](int y) {
            const char* p = (const char*)(dz + (ubase + (int64_t)min(max(y, 0), e - 1) * rs));
#pragma unroll
            for (int d = 0; d < 3; d++)
#pragma unroll
                for (int j = 0; j < 8; j++)
                    rz[d][j] = at(p, dzo[d], j + 1);
        };
        s8 a[3][3];  // [dx + 1][row y - 1, y, y + 1]
        auto pack_z = [&](int y, int row) {
            const bool yv = y >= 0 && y < e;
#pragma unroll
            for (int d = 0; d < 3; d++)
            {
                const uint32_t m = yv && dzv[d] ? ~0u : 0u;
                u4v w;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    w[k] = pack2(rz[d][2 * k], rz[d][2 * k + 1]) & (TAIL ? m & tm[k] : m);
                a[d][row] = __builtin_bit_cast(s8, w);
            }
        };
        load_z(y0 - 1);
        pack_z(y0 - 1, 0);
        load_z(y0);
        pack_z(y0, 1);
        load_h(y0);
        load_z(y0 + 1);
        for (int y = y0; y < y1; y++)
        {
            rh[0] &= mlo;
            if (TAIL)
            {
#pragma unroll
                for (int j = 1; j <= 8; j++)
                    rh[j + 1] = j >= jend ? 0u : rh[j + 1];
            }
            else
                rh[9] = jend == 8 ? 0u : rh[9];
            u4v wm, w0, wp;
#pragma unroll
            for (int k = 0; k < 4; k++)
            {
                wm[k] = pack2(rh[2 * k], rh[2 * k + 1]);
                w0[k] = pack2(rh[2 * k + 1], rh[2 * k + 2]);
                wp[k] = pack2(rh[2 * k + 2], rh[2 * k + 3]);
            }
            const s8 b[3] = { __builtin_bit_cast(s8, wm), __builtin_bit_cast(s8, w0), __builtin_bit_cast(s8, wp) };
            pack_z(y + 1, 2);
            if (y + 1 < y1)
            {
                load_h(y + 1);
                load_z(y + 2);
            }
#pragma unroll
            for (int dx = 0; dx < 3; dx++)
#pragma unroll
                for (int dy = 0; dy < 3; dy++)  // dZ row y - (dy - 1)
#pragma unroll
                    for (int d = 0; d < 3; d++)
                    {
                        const int tap = (dx * 3 + dy) * 3 + d;
                        acc[tap]      = mfma32(a[dx][2 - dy], b[d], acc[tap]);
                    }
            acc[kTaps] = mfma32(a[1][1], ones, acc[kTaps]);
#pragma unroll
            for (int d = 0; d < 3; d++)
            {
                a[d][0] = a[d][1];
                a[d][1] = a[d][2];
            }
        }
    }
    dw_block_sum<kTaps>(acc, red, kTaps * 256, [](int tap, int co, int ci) { return (tap * 16 + co) * 16 + ci; },
        part + (size_t)blockIdx.x * (kTaps * 256 + 16));
}

// Weight gradient of a layer with one scalar side (layer 0: channels dZ0,
// scalars x; layer 3, FLIP: channels h3, scalars dZ3):
//   dW[tap][c] = sum_v C[v][c] S[v + off(tap)]   (FLIP: S[v - off(tap)])
// and the sums of C over v (layer 0's bias), as 16x16x32 MFMAs over voxels,
// A = C^T, B = S shifted (column = tap, two fragments): 2 MFMAs per 32 voxels
// where a fragment per tap would use one row or column of 27.  A block marches
// along x over kSY rows and 32 z-voxels of one sample with the scalars' three
// planes in an LDS ring as BF16; bound by the 2-byte loads of C.
// 64 boxes of 32^3: 31 us (layer 0), 28 us (layer 3), where layer 3 with its
// one output row per tap took 1600 us and layer 0 254 us.
constexpr int kSY = 8, kSW = kLZ + 4, kSP = (kSY + 2) * kSW;
template <bool FLIP>
__global__ void __launch_bounds__(256) k_dw1(const uint16_t* __restrict__ ch, const float* __restrict__ sc, int e,
    int nyb, int nzb, int nxc, int xl, float* __restrict__ part)
{
    __shared__ uint16_t lds[3 * kSP];
    __shared__ float red[kTaps * 16 + 16];
    int b        = blockIdx.x;
    const int xc = b % nxc;
    b /= nxc;
    const int zb = b % nzb, yb = (b / nzb) % nyb, s = b / (nzb * nyb);
    const int x0 = xc * xl, x1 = min(e, x0 + xl), y0 = yb * kSY, z0 = zb * kLZ;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int64_t e3 = (int64_t)e * e * e;
    const float* S    = sc + (int64_t)s * e3;
    const uint16_t* C = ch + (int64_t)s * e3 * 16;
    auto stage = [&](int xp) {
        uint16_t* dst = lds + ((xp + 3) % 3) * kSP;
        for (int q = threadIdx.x; q < (kSY + 2) * kLW; q += blockDim.x)
        {
            const int yy = q / kLW, zz = q - (q / kLW) * kLW;
            const int y = y0 - 1 + yy, z = z0 - 1 + zz;
            float v = 0.f;
            if (xp >= 0 && xp < e && y >= 0 && y < e && z >= 0 && z < e) v = S[((int64_t)xp * e + y) * e + z];
            dst[yy * kSW + zz] = f2bf(v);
        }
    };
    // this lane's taps n and 16 + n (the last five columns repeat tap 26 and are dropped)
    int td[2], to[2];
#pragma unroll
    for (int f = 0; f < 2; f++)
    {
        const int tap = min(16 * f + n, kTaps - 1), tt = FLIP ? kTaps - 1 - tap : tap;
        td[f]         = tap_dx(tt);
        to[f]         = (1 + tap_dy(tt)) * kSW + 1 + tap_dz(tt) + 8 * g;
    }
    f4 acc[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
        acc[k] = (f4){ 0.f, 0.f, 0.f, 0.f };
    const s8 ones = { 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80, 0x3F80 };
    stage(x0 - 1);
    stage(x0);
    for (int x = x0; x < x1; x++)
    {
        stage(x + 1);
        // two rows per wave: y0 + wid, y0 + wid + 4; group g: z0 + 8g .. + 7
        s8 a[2];
#pragma unroll
        for (int r = 0; r < 2; r++)
        {
            const int y = y0 + wid + 4 * r;
#pragma unroll
            for (int i = 0; i < 8; i++)
            {
                const int z = z0 + 8 * g + i;
                a[r][i]     = y < e && z < e ? (short)C[(((int64_t)x * e + y) * e + z) * 16 + n] : (short)0;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 2; r++)
        {
#pragma unroll
            for (int f = 0; f < 2; f++)
            {
                const uint16_t* row = lds + ((x + 3 + td[f]) % 3) * kSP + (wid + 4 * r) * kSW + to[f];
                s8 bv;
#pragma unroll
                for (int i = 0; i < 8; i++)
                    bv[i] = (short)row[i];
                acc[f] = mfma32(a[r], bv, acc[f]);
            }
            acc[2] = mfma32(a[r], ones, acc[2]);
        }
        __syncthreads();
    }
    dw_block_sum<2>(acc, red, kTaps * 16, [](int f, int c, int k) { return 16 * f + k < kTaps ? (16 * f + k) * 16 + c : -1; },
        part + (size_t)blockIdx.x * (kTaps * 16 + 16));
}

// The layers' gradients from their blocks' partials, summed in a fixed order
// in FP64: a block takes 32 neighbouring values of one layer, eight groups of
// threads every eighth partial each.  11 us for the four layers of a
// batch of 64 boxes of 32^3, bound by latency (one thread per value, a chain of
// 1024 loads: 380 us for each layer).
struct DwLayer
{
    const float* part;
    float *gw, *gb;
    int np, nw, nb, stride;  // partials; weights, biases to sum; floats per partial
};
struct DwLayers
{
    DwLayer l[4];
    int first[5];  // first block of each layer
};
__global__ void __launch_bounds__(256) k_dw_reduce(DwLayers L)
{
    __shared__ double red[8][32];
    int k = 0;
    while (k < 3 && (int)blockIdx.x >= L.first[k + 1])
        k++;
    const DwLayer l = L.l[k];
    const int col = threadIdx.x & 31, row = threadIdx.x >> 5;
    const int q = ((int)blockIdx.x - L.first[k]) * 32 + col;
    double s = 0.;
    if (q < l.nw + l.nb)
    {
        // 16 loads in flight, added in order
        const float* p = l.part + q;
        int w          = row;
        for (; w + 120 < l.np; w += 128)
        {
            float v[16];
#pragma unroll
            for (int k2 = 0; k2 < 16; k2++)
                v[k2] = p[(size_t)(w + 8 * k2) * l.stride];
#pragma unroll
            for (int k2 = 0; k2 < 16; k2++)
                s += v[k2];
        }
        for (; w < l.np; w += 8)
            s += p[(size_t)w * l.stride];
    }
    red[row][col] = s;
    __syncthreads();
    if (row == 0 && q < l.nw + l.nb)
    {
        for (int r = 1; r < 8; r++)
            s += red[r][col];
        (q < l.nw ? l.gw[q] : l.gb[q - l.nw]) = (float)s;
    }
}

// loss pieces: y = s x + z; d = y - t; dy = 2 d / N; per block sums of d^2,
// dy*x (for ds) and dy (layer 3's bias), written to part[3*block]
__global__ void __launch_bounds__(256) k_loss(const float* x, const float* z, const float* t, const float* prm,
    int64_t n, float* y, float* dy, double* part)
{
    __shared__ double red[3][4];
    const float s   = prm[kS];
    const double sc = 2.0 / (double)n;
    double a = 0., b = 0., c = 0.;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    {
        const float yv = s * x[i] + z[i];
        if (y) y[i] = yv;
        if (t)
        {
            const double d = (double)yv - (double)t[i];
            const float g  = (float)(sc * d);
            dy[i]          = g;
            a += d * d;
            b += (double)g * (double)x[i];
            c += (double)g;
        }
    }
    for (int o = 32; o > 0; o >>= 1)
    {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
        c += __shfl_xor(c, o, 64);
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
    {
        red[0][wid] = a;
        red[1][wid] = b;
        red[2][wid] = c;
    }
    __syncthreads();
    if (threadIdx.x < 3)
    {
        const double* r                   = red[threadIdx.x];
        part[3 * blockIdx.x + threadIdx.x] = r[0] + r[1] + r[2] + r[3];
    }
}

// the loss blocks' sums: ds and layer 3's bias gradient to the gradient, the
// sum of d^2 to loss
__global__ void __launch_bounds__(192) k_loss_sum(const double* part, int np, float* grad, double* loss)
{
    // wave q sums column q, lane l every 64th block
    const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double s = 0.;
    for (int k = lane; k < np; k += 64)
        s += part[3 * k + q];
    for (int o = 32; o > 0; o >>= 1)
        s += __shfl_xor(s, o, 64);
    if (lane == 0)
    {
        if (q == 0)
            *loss = s;
        else
            grad[q == 1 ? kS : kB3] = (float)s;
    }
}

// BF16 weights for the forward and backward (flipped, transposed) passes
// from the FP32 master parameters
__global__ void k_derive(const float* p, uint16_t* f0, uint16_t* f1, uint16_t* f2, uint16_t* f3, uint16_t* r3,
    uint16_t* r2, uint16_t* r1)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    // forward layer 0: [cout][32 taps]
    if (q < 16 * 32)
    {
        const int co = q / 32, tap = q % 32;
        f0[q]        = tap < kTaps ? f2bf(p[kW0 + tap * 16 + co]) : 0;
    }
    if (q < kTaps * 256)
    {
        const int tap = q / 256, co = (q / 16) % 16, ci = q % 16;
        const int ft  = kTaps - 1 - tap;
        f1[q]         = f2bf(p[kW1 + q]);
        f2[q]         = f2bf(p[kW2 + q]);
        // layer 3 forward: row 0 only
        f3[q] = co == 0 ? f2bf(p[kW3 + tap * 16 + ci]) : 0;
        // backward of layers 2, 1: W'[tap][co' = ci][ci' = co] = W[26 - tap][co][ci]
        r2[q] = f2bf(p[kW2 + (ft * 16 + ci) * 16 + co]);
        r1[q] = f2bf(p[kW1 + (ft * 16 + ci) * 16 + co]);
    }
    // backward of layer 3 (scalar input dZ3 -> 16 channels): [co' = cin][32 taps]
    if (q < 16 * 32)
    {
        const int co = q / 32, tap = q % 32;
        r3[q]        = tap < kTaps ? f2bf(p[kW3 + (kTaps - 1 - tap) * 16 + co]) : 0;
    }
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
    float c1, float c2)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const float gq = g[q];
    const float mq = b1 * m[q] + (1.f - b1) * gq;
    const float vq = b2 * v[q] + (1.f - b2) * gq * gq;
    m[q]           = mq;
    v[q]           = vq;
    p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// per box: rms_j = sqrt(mean R_j^2) (0 -> 1); x = R/rms (FP32); t = KR/rms
__global__ void __launch_bounds__(256) k_box_rms(const double* R, int64_t m, double* rms)
{
    __shared__ double red[4];
    const int j = blockIdx.x;
    double a    = 0.;
    for (int64_t i = threadIdx.x; i < m; i += blockDim.x)
    {
        const double v = R[(int64_t)j * m + i];
        a += v * v;
    }
    for (int o = 32; o > 0; o >>= 1)
        a += __shfl_xor(a, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        const double r = sqrt((red[0] + red[1] + red[2] + red[3]) / (double)m);
        rms[j]         = r > 0. ? r : 1.;
    }
}

__global__ void k_box_scale_to_f32(const double* R, const double* rms, int64_t m, int64_t n, float* x)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = (float)(R[i] / rms[i / m]);
}

template <typename T>
__global__ void k_box_scale_from_f32(const float* y, const double* rms, int64_t m, int64_t n, T* out)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = (T)((double)y[i] * rms[i / m]);
}

}  // namespace
}  // namespace mgx

struct mgx_cnn
{
    mgx_ctx* ctx  = nullptr;
    int edge      = 0;
    int max_batch = 0;
    int step      = 0;  // Adam steps taken
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    uint16_t* wbf = nullptr;  // f0 f1 f2 f3 r3 r2 r1
    uint16_t *f0, *f1, *f2, *f3, *r3, *r2, *r1;
    // activations for max_batch samples
    uint16_t *h1 = nullptr, *h2 = nullptr, *h3 = nullptr, *dza = nullptr, *dzb = nullptr;
    float *z = nullptr, *y = nullptr, *dy = nullptr, *xf = nullptr;
    float *part0 = nullptr, *part1 = nullptr, *part2 = nullptr, *part3 = nullptr;  // weight-gradient partials per layer
    double *lpart = nullptr, *rms = nullptr;
    double* host  = nullptr;  // pinned
    bool dirty    = true;     // BF16 weights need refreshing
};

namespace mgx
{
namespace
{

constexpr int kLossBlocks = 1024;

// planes per x-chunk of a scalar layer's weight gradient: the columns alone
// when they give four blocks per CU, else chunks of at least four planes
int dw1_xl(int e, int64_t cols)
{
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>(1024 / cols, (e + 3) / 4));
    return (int)((e + want - 1) / want);
}

// most blocks of dw1 over batches of 1..max_batch samples
int64_t dw1_blocks(int e, int max_batch)
{
    const int64_t per = (int64_t)((e + kSY - 1) / kSY) * ((e + kLZ - 1) / kLZ);
    return std::max<int64_t>(1024 + per, per * max_batch);
}

int64_t ntiles(int e, int nb) { return (int64_t)nb * e * e * ((e + 15) / 16); }

int derive(mgx_cnn* c)
{
    if (!c->dirty) return MGX_OK;
    hipLaunchKernelGGL(k_derive, dim3((kTaps * 256 + 255) / 256), dim3(256), 0, c->ctx->stream, (const float*)c->p,
        c->f0, c->f1, c->f2, c->f3, c->r3, c->r2, c->r1);
    MGX_CHECK_LAUNCH(c->ctx);
    c->dirty = false;
    return MGX_OK;
}

// forward of nb samples from FP32 x; z (pre-skip last layer) into c->z
// the network over nb samples: from FP32 x (training, z of the last layer to
// c->z), or from FP64 box residuals R with per-box rms (inference: the
// rescaled output rms * (s x + z) written to out in the type of T)
template <typename T>
int forward_any(mgx_cnn* c, const float* x, const double* R, const double* rms, int nb, T* out)
{
    mgx_ctx* ctx = c->ctx;
    int rc;
    if ((rc = derive(c))) return rc;
    const int e   = c->edge;
    const int nyb = (e + kLY - 1) / kLY, nzb = (e + kLZ - 1) / kLZ;
    const dim3 lgrid((unsigned)(nb * nyb * nzb));
    if (R)
        hipLaunchKernelGGL(k_conv1_lds<double>, lgrid, dim3(256), 0, ctx->stream, R, rms, (const uint16_t*)c->f0,
            (const float*)c->p + kB0, c->h1, e, nyb, nzb);
    else
        hipLaunchKernelGGL(k_conv1_lds<float>, lgrid, dim3(256), 0, ctx->stream, x, (const double*)nullptr,
            (const uint16_t*)c->f0, (const float*)c->p + kB0, c->h1, e, nyb, nzb);
    hipLaunchKernelGGL((k_conv16_lds<CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->h1,
        (const uint16_t*)c->f1, (const float*)c->p + kB1, c->h2, (const uint16_t*)nullptr, e, nyb, nzb);
    hipLaunchKernelGGL((k_conv16_lds<CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->h2,
        (const uint16_t*)c->f2, (const float*)c->p + kB2, c->h3, (const uint16_t*)nullptr, e, nyb, nzb);
    const int noy = (e + kOY - 1) / kOY;
    hipLaunchKernelGGL(k_conv_out_lds<T>, dim3((unsigned)(nb * noy * nzb)), dim3(256), 0, ctx->stream,
        (const uint16_t*)c->h3, (const uint16_t*)c->f3, (const float*)c->p, c->z, R, rms, out, e, noy, nzb);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

int forward(mgx_cnn* c, const float* x, int nb)
{
    return forward_any<float>(c, x, nullptr, nullptr, nb, nullptr);
}

// The launch of a weight gradient: 16 -> 16 layers in at most kDwBlocks blocks
// (two resident per CU), with chunks of rows only where the columns alone
// leave waves idle; scalar layers one block per (8 rows, 32 z, x-chunk).
int dw16(mgx_cnn* c, const uint16_t* dz, const uint16_t* h, int nb, float* part, DwLayer& l)
{
    mgx_ctx* ctx  = c->ctx;
    const int e   = c->edge, nzs = (e + 7) / 8, ncol = nb * e * nzs, ncg = (ncol + 3) / 4;
    const int want = std::max(1, std::min(kDwBlocks * kWaves / ncg, (e + 3) / 4));
    const int yl = (e + want - 1) / want, nyc = (e + yl - 1) / yl;
    const int ntask = ncg * nyc, blocks = std::min(kDwBlocks, (ntask + kWaves - 1) / kWaves);
    if (e % 8)
        hipLaunchKernelGGL(k_dw16<true>, dim3(blocks), dim3(256), 0, ctx->stream, dz, h, e, nzs, ncol, yl, nyc, ntask, part);
    else
        hipLaunchKernelGGL(k_dw16<false>, dim3(blocks), dim3(256), 0, ctx->stream, dz, h, e, nzs, ncol, yl, nyc, ntask, part);
    MGX_CHECK_LAUNCH(ctx);
    l.part = part, l.np = blocks, l.nw = kTaps * 256, l.nb = 16, l.stride = kTaps * 256 + 16;
    return MGX_OK;
}

template <bool FLIP>
int dw1(mgx_cnn* c, const uint16_t* ch, const float* sc, int nb, float* part, DwLayer& l)
{
    mgx_ctx* ctx  = c->ctx;
    const int e   = c->edge, nyb = (e + kSY - 1) / kSY, nzb = (e + kLZ - 1) / kLZ, cols = nb * nyb * nzb;
    const int xl  = dw1_xl(e, cols), nxc = (e + xl - 1) / xl;
    hipLaunchKernelGGL(k_dw1<FLIP>, dim3(cols * nxc), dim3(256), 0, ctx->stream, ch, sc, e, nyb, nzb, nxc, xl, part);
    MGX_CHECK_LAUNCH(ctx);
    l.part = part, l.np = cols * nxc, l.nw = kTaps * 16, l.nb = FLIP ? 0 : 16, l.stride = kTaps * 16 + 16;
    return MGX_OK;
}

// loss and gradient into c->g; loss (mean squared error) to *loss
int grad(mgx_cnn* c, const float* x, const float* t, int nb, double* loss)
{
    mgx_ctx* ctx = c->ctx;
    int rc;
    if ((rc = forward(c, x, nb))) return rc;
    const int e = c->edge, nzt = (e + 15) / 16;
    const int64_t n  = (int64_t)nb * e * e * e;
    const int64_t nt = ntiles(e, nb);
    hipLaunchKernelGGL(k_loss, dim3(kLossBlocks), dim3(256), 0, ctx->stream, x, (const float*)c->z, t,
        (const float*)c->p, n, (float*)nullptr, c->dy, c->lpart);
    hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(192), 0, ctx->stream, (const double*)c->lpart, kLossBlocks, c->g,
        c->lpart + 3 * kLossBlocks);
    MGX_CHECK_LAUNCH(ctx);
    DwLayers L;
    // layer 3: dZ3 = dy (scalar; its bias came with the loss)
    if ((rc = dw1<true>(c, c->h3, c->dy, nb, c->part3, L.l[3]))) return rc;
    L.l[3].gw = c->g + kW3, L.l[3].gb = nullptr;
    const dim3 grid((unsigned)((nt + kWaves - 1) / kWaves)), blk(64 * kWaves);
    hipLaunchKernelGGL((k_conv<1, 16, CONV_BWD_MASK>), grid, blk, 0, ctx->stream, (const void*)c->dy, c->r3,
        (const float*)nullptr, (void*)c->dza, (const uint16_t*)c->h3, e, nzt, nt);
    MGX_CHECK_LAUNCH(ctx);
    // layer 2: dZ2 = dza
    if ((rc = dw16(c, c->dza, c->h2, nb, c->part2, L.l[2]))) return rc;
    L.l[2].gw = c->g + kW2, L.l[2].gb = c->g + kB2;
    const int nyb = (e + kLY - 1) / kLY, nzb = (e + kLZ - 1) / kLZ;
    const dim3 lgrid((unsigned)(nb * nyb * nzb));
    hipLaunchKernelGGL((k_conv16_lds<CONV_BWD_MASK>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->dza,
        (const uint16_t*)c->r2, (const float*)nullptr, c->dzb, (const uint16_t*)c->h2, e, nyb, nzb);
    MGX_CHECK_LAUNCH(ctx);
    // layer 1: dZ1 = dzb
    if ((rc = dw16(c, c->dzb, c->h1, nb, c->part1, L.l[1]))) return rc;
    L.l[1].gw = c->g + kW1, L.l[1].gb = c->g + kB1;
    hipLaunchKernelGGL((k_conv16_lds<CONV_BWD_MASK>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->dzb,
        (const uint16_t*)c->r1, (const float*)nullptr, c->dza, (const uint16_t*)c->h1, e, nyb, nzb);
    MGX_CHECK_LAUNCH(ctx);
    // layer 0: dZ0 = dza, input x
    if ((rc = dw1<false>(c, c->dza, x, nb, c->part0, L.l[0]))) return rc;
    L.l[0].gw = c->g + kW0, L.l[0].gb = c->g + kB0;
    L.first[0] = 0;
    for (int k = 0; k < 4; k++)
        L.first[k + 1] = L.first[k] + (L.l[k].nw + L.l[k].nb + 31) / 32;
    hipLaunchKernelGGL(k_dw_reduce, dim3(L.first[4]), dim3(256), 0, ctx->stream, L);
    MGX_CHECK_LAUNCH(ctx);
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(c->host, c->lpart + 3 * kLossBlocks, sizeof(double), hipMemcpyDeviceToHost,
                           ctx->stream));
    MGX_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    *loss = c->host[0] / (double)n;
    return MGX_OK;
}

bool batch_ok(const mgx_cnn* c, int nb) { return nb >= 1 && nb <= c->max_batch; }

}  // namespace

int cnn_apply_boxes(mgx_cnn* c, int nbox, int edge, const double* R, void* out, int out_dtype);

}  // namespace mgx

using namespace mgx;

extern "C" {

int mgx_cnn_nparams(void) { return kNP; }

int mgx_cnn_create(mgx_ctx* ctx, int edge, int max_batch, mgx_cnn** out)
{
    MGX_REQUIRE(ctx, out && edge >= 1 && edge <= 128 && max_batch >= 1, "bad CNN geometry");
    mgx_cnn* c   = new mgx_cnn();
    c->ctx       = ctx;
    c->edge      = edge;
    c->max_batch = max_batch;
    const size_t nv = (size_t)max_batch * edge * edge * edge;
    const size_t nd16 = (size_t)kDwBlocks * (kTaps * 256 + 16), nd1 = (size_t)dw1_blocks(edge, max_batch) * (kTaps * 16 + 16);
    bool ok         = true;
    auto al         = [&](void** p, size_t bytes) { ok = ok && hipMalloc(p, std::max<size_t>(bytes, 256)) == hipSuccess; };
    al((void**)&c->p, kNP * sizeof(float));
    al((void**)&c->g, kNP * sizeof(float));
    al((void**)&c->m, kNP * sizeof(float));
    al((void**)&c->v, kNP * sizeof(float));
    al((void**)&c->wbf, (2 * 512 + 5 * kTaps * 256) * sizeof(uint16_t));
    al((void**)&c->h1, nv * 16 * sizeof(uint16_t) + kDwPad);
    al((void**)&c->h2, nv * 16 * sizeof(uint16_t) + kDwPad);
    al((void**)&c->h3, nv * 16 * sizeof(uint16_t) + kDwPad);
    al((void**)&c->dza, nv * 16 * sizeof(uint16_t) + kDwPad);
    al((void**)&c->dzb, nv * 16 * sizeof(uint16_t) + kDwPad);
    al((void**)&c->z, nv * sizeof(float));
    al((void**)&c->y, nv * sizeof(float));
    al((void**)&c->dy, nv * sizeof(float));
    al((void**)&c->xf, nv * sizeof(float));
    al((void**)&c->part0, nd1 * sizeof(float));
    al((void**)&c->part1, nd16 * sizeof(float));
    al((void**)&c->part2, nd16 * sizeof(float));
    al((void**)&c->part3, nd1 * sizeof(float));
    al((void**)&c->lpart, (3 * kLossBlocks + 1) * sizeof(double));
    al((void**)&c->rms, (size_t)max_batch * sizeof(double));
    ok = ok && hipHostMalloc((void**)&c->host, sizeof(double), hipHostMallocDefault) == hipSuccess;
    if (!ok)
    {
        mgx_cnn_destroy(c);
        return set_err(ctx, MGX_ENOMEM, "CNN allocation failed");
    }
    c->f0 = c->wbf;
    c->r3 = c->f0 + 512;
    c->f1 = c->r3 + 512;
    c->f2 = c->f1 + kTaps * 256;
    c->f3 = c->f2 + kTaps * 256;
    c->r2 = c->f3 + kTaps * 256;
    c->r1 = c->r2 + kTaps * 256;
    hipMemsetAsync(c->p, 0, kNP * sizeof(float), ctx->stream);
    hipMemsetAsync(c->m, 0, kNP * sizeof(float), ctx->stream);
    hipMemsetAsync(c->v, 0, kNP * sizeof(float), ctx->stream);
    if (hipStreamSynchronize(ctx->stream) != hipSuccess)
    {
        mgx_cnn_destroy(c);
        return set_err(ctx, MGX_EHIP, "CNN init failed");
    }
    *out = c;
    return MGX_OK;
}

int mgx_cnn_destroy(mgx_cnn* c)
{
    if (!c) return MGX_OK;
    void* bufs[] = { c->p, c->g, c->m, c->v, c->wbf, c->h1, c->h2, c->h3, c->dza, c->dzb, c->z, c->y, c->dy, c->xf,
        c->part0, c->part1, c->part2, c->part3, c->lpart, c->rms };
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    if (c->host) (void)hipHostFree(c->host);
    delete c;
    return MGX_OK;
}

int mgx_cnn_set_params(mgx_cnn* c, const float* host)
{
    if (!c || !host) return MGX_EINVAL;
    MGX_CHECK_HIP(c->ctx, hipMemcpy(c->p, host, kNP * sizeof(float), hipMemcpyHostToDevice));
    MGX_CHECK_HIP(c->ctx, hipMemsetAsync(c->m, 0, kNP * sizeof(float), c->ctx->stream));
    MGX_CHECK_HIP(c->ctx, hipMemsetAsync(c->v, 0, kNP * sizeof(float), c->ctx->stream));
    MGX_CHECK_HIP(c->ctx, hipStreamSynchronize(c->ctx->stream));
    c->step  = 0;
    c->dirty = true;
    return MGX_OK;
}

int mgx_cnn_get_params(mgx_cnn* c, float* host)
{
    if (!c || !host) return MGX_EINVAL;
    MGX_CHECK_HIP(c->ctx, hipMemcpy(host, c->p, kNP * sizeof(float), hipMemcpyDeviceToHost));
    return MGX_OK;
}

int mgx_cnn_forward(mgx_cnn* c, const float* x, int nb, float* y)
{
    if (!c || !x || !y) return MGX_EINVAL;
    MGX_REQUIRE(c->ctx, batch_ok(c, nb), "batch larger than the CNN was created for");
    int rc = forward(c, x, nb);
    if (rc) return rc;
    const int64_t n = (int64_t)nb * c->edge * c->edge * c->edge;
    hipLaunchKernelGGL(k_loss, dim3(kLossBlocks), dim3(256), 0, c->ctx->stream, x, (const float*)c->z,
        (const float*)nullptr, (const float*)c->p, n, y, (float*)nullptr, c->lpart);
    MGX_CHECK_LAUNCH(c->ctx);
    return sync(c->ctx);
}

int mgx_cnn_grad(mgx_cnn* c, const float* x, const float* t, int nb, double* loss, float* grad_host)
{
    if (!c || !x || !t || !loss) return MGX_EINVAL;
    MGX_REQUIRE(c->ctx, batch_ok(c, nb), "batch larger than the CNN was created for");
    int rc = grad(c, x, t, nb, loss);
    if (rc) return rc;
    if (grad_host) MGX_CHECK_HIP(c->ctx, hipMemcpy(grad_host, c->g, kNP * sizeof(float), hipMemcpyDeviceToHost));
    return MGX_OK;
}

int mgx_cnn_train_step(mgx_cnn* c, const float* x, const float* t, int nb, float lr, double* loss)
{
    if (!c || !x || !t || !loss) return MGX_EINVAL;
    MGX_REQUIRE(c->ctx, batch_ok(c, nb), "batch larger than the CNN was created for");
    MGX_REQUIRE(c->ctx, lr > 0.f, "learning rate must be positive");
    int rc = grad(c, x, t, nb, loss);
    if (rc) return rc;
    c->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)c->step), c2 = 1.f - powf(b2, (float)c->step);
    hipLaunchKernelGGL(k_adam, dim3((kNP + 255) / 256), dim3(256), 0, c->ctx->stream, c->p, (const float*)c->g, c->m,
        c->v, kNP, lr, b1, b2, 1e-8f, c1, c2);
    MGX_CHECK_LAUNCH(c->ctx);
    c->dirty = true;
    return MGX_OK;
}

// out_j = rms_j * net(R_j / rms_j) for nbox boxes of edge e packed one after
// another (FP64 in and out, device); processed in batches of max_batch
int mgx_cnn_apply(mgx_cnn* c, int nbox, const double* R, double* out)
{
    if (!c || !R || !out || nbox < 1) return MGX_EINVAL;
    int rc = cnn_apply_boxes(c, nbox, c->edge, R, out, MGX_F64);
    return rc ? rc : sync(c->ctx);
}

// training pairs: x = R_j / rms_j, t = KR_j / rms_j (FP32, device)
int mgx_cnn_make_pairs(mgx_cnn* c, int nbox, const double* R, const double* KR, float* x, float* t)
{
    if (!c || !R || !KR || !x || !t || nbox < 1) return MGX_EINVAL;
    mgx_ctx* ctx = c->ctx;
    const int64_t m = (int64_t)c->edge * c->edge * c->edge;
    double* rms     = nullptr;
    MGX_CHECK_HIP(ctx, hipMalloc((void**)&rms, (size_t)nbox * sizeof(double)));
    hipLaunchKernelGGL(k_box_rms, dim3(nbox), dim3(256), 0, ctx->stream, R, m, rms);
    hipLaunchKernelGGL(k_box_scale_to_f32, dim3(4096), dim3(256), 0, ctx->stream, R, (const double*)rms, m,
        m * nbox, x);
    hipLaunchKernelGGL(k_box_scale_to_f32, dim3(4096), dim3(256), 0, ctx->stream, KR, (const double*)rms, m,
        m * nbox, t);
    hipError_t e1 = hipGetLastError();
    hipError_t e2 = hipStreamSynchronize(ctx->stream);
    (void)hipFree(rms);
    if (e1 != hipSuccess || e2 != hipSuccess) return set_err(ctx, MGX_EHIP, "make_pairs failed");
    return MGX_OK;
}

}  // extern "C"

namespace mgx
{
// out (type out_dtype) = rms_j * net(R_j / rms_j) per box
int cnn_apply_boxes(mgx_cnn* c, int nbox, int edge, const double* R, void* out, int out_dtype)
{
    mgx_ctx* ctx = c->ctx;
    MGX_REQUIRE(ctx, edge == c->edge, "box edge differs from the CNN's");
    const int64_t m = (int64_t)edge * edge * edge;
    int rc;
    for (int b0 = 0; b0 < nbox; b0 += c->max_batch)
    {
        const int nb     = std::min(c->max_batch, nbox - b0);
        const double* Rb = R + (int64_t)b0 * m;
        hipLaunchKernelGGL(k_box_rms, dim3(nb), dim3(256), 0, ctx->stream, Rb, m, c->rms);
        MGX_CHECK_LAUNCH(ctx);
        rc = out_dtype == MGX_F32
                 ? forward_any<float>(c, nullptr, Rb, c->rms, nb, (float*)out + (int64_t)b0 * m)
                 : forward_any<double>(c, nullptr, Rb, c->rms, nb, (double*)out + (int64_t)b0 * m);
        if (rc) return rc;
    }
    return MGX_OK;
}
}  // namespace mgx
