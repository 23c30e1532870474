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
// Convolution as MFMA (v_mfma_f32_16x16x32_bf16): a tile is 16 z-consecutive
// voxels x 16 output channels, D[cout][voxel] = sum_tap W_tap[cout][cin]
// X[cin][voxel + off(tap)], with the weights of all taps in registers and the
// input rows in LDS, two taps of 16 channels per MFMA.
#include "common.hpp"

#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace mgx
{
namespace
{

constexpr int kTaps    = 27;
constexpr int kWaves   = 4;  // per block
constexpr int kDwBlocks = 512;  // most blocks of a 16 -> 16 weight gradient: two per CU
constexpr int kDwPad    = 256;  // bytes after the activations that its last rows read past their end

// parameter offsets (floats)
constexpr int kW0 = 0, kB0 = kW0 + 27 * 16, kW1 = kB0 + 16, kB1 = kW1 + 27 * 256, kW2 = kB1 + 16,
              kB2 = kW2 + 27 * 256, kW3 = kB2 + 16, kB3 = kW3 + 27 * 16, kS = kB3 + 1, kNP = kS + 1;

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

__device__ inline int tap_dx(int t) { return t / 9 - 1; }
__device__ inline int tap_dy(int t) { return (t / 3) % 3 - 1; }
__device__ inline int tap_dz(int t) { return t % 3 - 1; }

enum
{
    CONV_FWD_RELU = 0,  // + bias, ReLU
    CONV_BWD_MASK = 1   // no bias, times (hmask > 0)
};

// value pairs to BF16 (nearest even; v_cvt_pk_bf16_f32), the first in the low half
__device__ __forceinline__ uint32_t cvt2(float a, float b)
{
    bf2 v;
    v[0] = (__bf16)a;
    v[1] = (__bf16)b;
    return __builtin_bit_cast(uint32_t, v);
}

// A 16-channel layer's input window of ROWS x 34 voxels (one plane of x) in
// LDS, the two 8-channel halves apart, so that 16 lanes reading neighbouring
// voxels touch 256 contiguous bytes.  Every thread keeps its chunks' places:
// load() puts the next plane in registers, store() moves it to LDS.
constexpr int kLZ = 32, kLW = kLZ + 2;
template <int ROWS>
struct Window
{
    static constexpr int kHalf = ROWS * kLW * 8;  // BF16 values per half
    static constexpr int kSize = 2 * kHalf;
    static constexpr int kN    = (ROWS * kLW * 2 + 255) / 256;
    const uint16_t* X;
    int64_t plane;
    int e, off[kN], dst[kN];
    uint4 v[kN];
    __device__ __forceinline__ Window(const uint16_t* x, int e_, int y0, int z0) : X(x), e(e_)
    {
        plane = (int64_t)e * e * 16;
#pragma unroll
        for (int k = 0; k < kN; k++)
        {
            const int q = threadIdx.x + 256 * k, half = q & 1, vox = q >> 1, yy = vox / kLW;
            const int y = y0 - 1 + yy, z = z0 - 1 + vox - yy * kLW;
            const bool in = q < ROWS * kLW * 2;
            off[k] = in && y >= 0 && y < e && z >= 0 && z < e ? (y * e + z) * 16 + 8 * half : -1;
            dst[k] = in ? half * kHalf + vox * 8 : -1;
        }
    }
    __device__ __forceinline__ void load(int xp)
    {
#pragma unroll
        for (int k = 0; k < kN; k++)
        {
            v[k] = (uint4){ 0u, 0u, 0u, 0u };
            if (off[k] >= 0 && xp < e) v[k] = *(const uint4*)(X + xp * plane + off[k]);
        }
    }
    __device__ __forceinline__ void store(uint16_t* lds) const
    {
#pragma unroll
        for (int k = 0; k < kN; k++)
            if (dst[k] >= 0) *(uint4*)(lds + dst[k]) = v[k];
    }
};

// A 16 -> 16 layer.  A block (4 waves) owns rows y0..y0+3, z0..z0+31 of one
// sample and marches along x; wave w computes row y0+w, two 16-voxel z-tiles,
// as D[cout][voxel] += W_tap[cout][cin] X[cin][voxel + off(tap)] with
// 16x16x32 MFMAs (K = two taps of 16 channels).  Each plane of the input is
// in LDS once (two buffers, one barrier per plane, the next plane's loads in
// flight) and enters the three planes of output it reaches (dx = 1, 0, -1),
// whose sums stay in registers: five operand reads per 15 MFMAs, where a
// three-plane ring with one output plane reads 14 per 14.  Taps in pairs:
// (dz = -1, 0) of a row, then dz = 1 of rows y-1, y and of row y+1 (against
// zero weights in its second half).
// Bound by the planes' load latency between the matrix and the memory limits.
// 256 boxes of 32^3 (537 MB, 116 GFLOP): 157 us (3.4 TB/s, 0.74 PFLOP/s); the
// three-plane ring took 240 us.
constexpr int kLY = 4, kLH = kLY + 2;
template <int MODE>
__global__ void __launch_bounds__(256, 4) k_conv16(const uint16_t* __restrict__ in, const uint16_t* __restrict__ wt,
    const float* __restrict__ bias, uint16_t* __restrict__ out, const uint16_t* __restrict__ hmask, int e, int nyb,
    int nzb, int nxc, int xl)
{
    typedef Window<kLH> W;
    __shared__ __align__(16) uint16_t lds[2][W::kSize];
    int b        = blockIdx.x;
    const int xc = b % nxc;
    b /= nxc;
    const int s = b / (nyb * nzb), y0 = (b / nzb) % nyb * kLY, z0 = b % nzb * kLZ;
    const int x0 = xc * xl, x1 = min(e, x0 + xl);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int tsel = g >> 1, cs = 8 * (g & 1);
    const int64_t e3 = (int64_t)e * e * e;
    s8 wa[3][5];  // [dx + 1][pair]
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
#pragma unroll
        for (int k = 0; k < 5; k++)
        {
            const int tap = k < 3 ? (dx * 3 + k) * 3 + tsel : (dx * 3 + (k == 3 ? tsel : 2)) * 3 + 2;
            wa[dx][k]     = *(const s8*)(wt + ((size_t)tap * 16 + n) * 16 + cs);
            if (k == 4 && tsel) wa[dx][k] = (s8){ 0, 0, 0, 0, 0, 0, 0, 0 };
        }
    f4 bv = { 0.f, 0.f, 0.f, 0.f };
    if (MODE == CONV_FWD_RELU) bv = *(const f4*)(bias + 4 * g);
    // the pairs' places in the window: rows wid, wid+1, wid+2 (= y-1, y, y+1)
    const int hb = (g & 1) * W::kHalf, p0 = hb + (wid * kLW + n + tsel) * 8;
    const int q0 = hb + ((wid + tsel) * kLW + n + 2) * 8, q1 = hb + ((wid + 2) * kLW + n + 2) * 8;
    const int y = y0 + wid;
    W w(in + (int64_t)s * e3 * 16, e, y0, z0);
    // this lane's outputs: voxels z0 + n (+ 16) of its row, channels 4g..4g+3
    const int64_t vox0 = ((int64_t)s * e3 + (int64_t)y * e + z0 + n) * 16 + 4 * g, e2 = (int64_t)e * e * 16;
    const bool ok[2]   = { y < e && z0 + n < e, y < e && z0 + 16 + n < e };
    uint2 mp[2], mc[2];  // the masks of planes xp - 1, xp: loaded a plane ahead of their use
    auto emit = [&](int x, const f4 (&a)[2], const uint2 (&mask)[2]) {
#pragma unroll
        for (int t = 0; t < 2; t++)
        {
            if (!ok[t]) continue;
            float v[4];
            if (MODE == CONV_BWD_MASK)
            {
                const uint2 m = mask[t];
                v[0] = m.x & 0xFFFFu ? a[t][0] : 0.f;
                v[1] = m.x >> 16 ? a[t][1] : 0.f;
                v[2] = m.y & 0xFFFFu ? a[t][2] : 0.f;
                v[3] = m.y >> 16 ? a[t][3] : 0.f;
            }
            else
#pragma unroll
                for (int i = 0; i < 4; i++)
                    v[i] = fmaxf(a[t][i] + bv[i], 0.f);
            *(uint2*)(out + vox0 + x * e2 + 256 * t) = (uint2){ cvt2(v[0], v[1]), cvt2(v[2], v[3]) };
        }
    };
    const f4 zero = { 0.f, 0.f, 0.f, 0.f };
    const bool two = z0 + 16 < e;  // the second z-tile holds voxels
    f4 c0[2] = { zero, zero }, c1[2] = { zero, zero }, c2[2] = { zero, zero };  // sums of planes xp + 1, xp, xp - 1
    const int xa = max(x0 - 1, 0), xb = min(x1, e - 1);
    w.load(xa);
    for (int xp = xa; xp <= xb; xp++)
    {
        uint16_t* buf = lds[xp & 1];
        w.store(buf);
        __syncthreads();
        if (MODE == CONV_BWD_MASK)
#pragma unroll
            for (int t = 0; t < 2; t++)
            {
                mp[t] = mc[t];
                if (ok[t]) mc[t] = *(const uint2*)(hmask + vox0 + xp * e2 + 256 * t);
            }
        if (xp < xb) w.load(xp + 1);
#pragma unroll
        for (int t = 0; t < 2; t++)
        {
            c2[t] = c1[t];
            c1[t] = c0[t];
            c0[t] = zero;
            if (t && !two) continue;
#pragma unroll
            for (int k = 0; k < 5; k++)
            {
                const int at = k < 3 ? p0 + k * kLW * 8 : k == 3 ? q0 : q1;
                const s8 bq  = *(const s8*)(buf + at + 16 * t * 8);
                c2[t]        = mfma32(wa[2][k], bq, c2[t]);
                c1[t]        = mfma32(wa[1][k], bq, c1[t]);
                c0[t]        = mfma32(wa[0][k], bq, c0[t]);
            }
        }
        if (xp > x0) emit(xp - 1, c2, mp);
    }
    if (x1 == e) emit(e - 1, c1, mc);
}

// A layer from one scalar per voxel to 16 channels: layer 0 (bias, ReLU), and
// the backward pass of the last layer (times h > 0).  The scalars' planes are
// BF16 in a ring of four (one barrier per plane); one 16x16x32 MFMA per
// 16-voxel tile covers all 27 taps (lane group g holds taps 8g..8g+7, the
// last five zero).  Inputs times 1 / rms (the box's normalised residual) when
// rms is given.  Bound by the 32 bytes written per voxel: 256 boxes of 32^3
// from FP64 (335 MB): 77 us (4.4 TB/s), 121 us with FP64 divisions, FP32
// planes and two barriers per plane.
template <typename TIN, int MODE>
__global__ void __launch_bounds__(256) k_conv1(const TIN* __restrict__ in, const double* __restrict__ rms,
    const uint16_t* __restrict__ wt, const float* __restrict__ bias, uint16_t* __restrict__ out,
    const uint16_t* __restrict__ hmask, int e, int nyb, int nzb, int nxc, int xl)
{
    constexpr int kP1 = kLH * kLW;
    __shared__ uint16_t lds[4 * kP1];
    int b        = blockIdx.x;
    const int xc = b % nxc;
    b /= nxc;
    const int s = b / (nyb * nzb), y0 = (b / nzb) % nyb * kLY, z0 = b % nzb * kLZ;
    const int x0 = xc * xl, x1 = min(e, x0 + xl);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int64_t e2 = (int64_t)e * e, e3 = e2 * e;
    const TIN* X = in + (int64_t)s * e3;
    const double inv = rms ? 1. / rms[s] : 1.;
    // A: W[cout = n][taps 8g..8g+7] from the [16][32] layout
    const s8 wa = *(const s8*)(wt + (size_t)n * 32 + 8 * g);
    f4 bv = { 0.f, 0.f, 0.f, 0.f };
    if (MODE == CONV_FWD_RELU) bv = *(const f4*)(bias + 4 * g);
    // this thread's value of a plane's window
    const int q = threadIdx.x, yy = q / kLW, ys = y0 - 1 + yy, zs = z0 - 1 + q - yy * kLW;
    const bool in_w = q < kP1, in_box = in_w && ys >= 0 && ys < e && zs >= 0 && zs < e;
    const int64_t at = (int64_t)ys * e + zs;
    TIN r = 0;
    auto load = [&](int xp) { r = in_box && xp >= 0 && xp < e ? X[xp * e2 + at] : (TIN)0; };
    auto store = [&](int xp) {
        if (in_w) lds[(xp & 3) * kP1 + q] = (uint16_t)cvt2(rms ? (float)((double)r * inv) : (float)r, 0.f);
    };
    // taps 8g..8g+7: plane and place in the window; the padding taps read the centre
    int td[8], to[8];
#pragma unroll
    for (int i = 0; i < 8; i++)
    {
        const int tap = 8 * g + i < kTaps ? 8 * g + i : 13;
        td[i]         = tap_dx(tap);
        to[i]         = (wid + 1 + tap_dy(tap)) * kLW + n + 1 + tap_dz(tap);
    }
    load(x0 - 1);
    store(x0 - 1);
    load(x0);
    store(x0);
    load(x0 + 1);
    // this lane's outputs: voxels z0 + n (+ 16) of its row, channels 4g..4g+3
    const int y        = y0 + wid;
    const int64_t vox0 = ((int64_t)s * e3 + (int64_t)y * e + z0 + n) * 16 + 4 * g;
    const bool ok[2]   = { y < e && z0 + n < e, y < e && z0 + 16 + n < e };
    for (int x = x0; x < x1; x++)
    {
        store(x + 1);
        const int64_t vox = vox0 + (int64_t)x * e2 * 16;
        uint2 mask[2];
        if (MODE == CONV_BWD_MASK)
#pragma unroll
            for (int t = 0; t < 2; t++)
                if (ok[t]) mask[t] = *(const uint2*)(hmask + vox + 256 * t);
        __syncthreads();
        if (x + 1 < x1) load(x + 2);
        uint32_t u0[8], u1[8];
#pragma unroll
        for (int i = 0; i < 8; i++)
        {
            const uint16_t* p = lds + ((x + td[i]) & 3) * kP1 + to[i];
            u0[i]             = p[0];
            u1[i]             = p[16];
        }
        uint4 v0, v1;
        v0.x = u0[0] | u0[1] << 16, v0.y = u0[2] | u0[3] << 16, v0.z = u0[4] | u0[5] << 16, v0.w = u0[6] | u0[7] << 16;
        v1.x = u1[0] | u1[1] << 16, v1.y = u1[2] | u1[3] << 16, v1.z = u1[4] | u1[5] << 16, v1.w = u1[6] | u1[7] << 16;
        const f4 z4 = { 0.f, 0.f, 0.f, 0.f };
        const f4 acc[2] = { mfma32(wa, __builtin_bit_cast(s8, v0), z4), mfma32(wa, __builtin_bit_cast(s8, v1), z4) };
#pragma unroll
        for (int t = 0; t < 2; t++)
        {
            if (!ok[t]) continue;
            float v[4];
            if (MODE == CONV_BWD_MASK)
            {
                const uint2 m = mask[t];
                v[0] = m.x & 0xFFFFu ? acc[t][0] : 0.f;
                v[1] = m.x >> 16 ? acc[t][1] : 0.f;
                v[2] = m.y & 0xFFFFu ? acc[t][2] : 0.f;
                v[3] = m.y >> 16 ? acc[t][3] : 0.f;
            }
            else
#pragma unroll
                for (int i = 0; i < 4; i++)
                    v[i] = fmaxf(acc[t][i] + bv[i], 0.f);
            *(uint2*)(out + vox + 256 * t) = (uint2){ cvt2(v[0], v[1]), cvt2(v[2], v[3]) };
        }
    }
}

// The last layer (16 -> 1 channel).  A block owns rows y0..y0+7, z0..z0+31 and
// marches along x like k_conv16, two rows per wave.  The rows of the MFMA are
// the nine (dy, dx) of the taps, row 4(dy+1) + dx+1 (the others zero), and dz
// and the channels its K: two MFMAs and two operand reads per 16 voxels of
// input.  Lane group dy+1 then holds, in element dx+1, its share of the output
// plane xp - dx: elements move up by one per plane (the accumulator of the
// next), element 2 is complete, and the three groups' values of the rows y-1,
// y, y+1 are added across the wave.
// With R non-null it also finishes the network on the box: y = s x + z with
// x = (float)(R / rms), written as (T)(y * rms) to out; otherwise z to zout.
// Bound by HBM (32 bytes read per voxel).  256 boxes of 32^3 (403 MB): 90 us
// (4.5 TB/s); 264 us with 27 taps of vector dot products from LDS.
constexpr int kOY = 8, kOH = kOY + 2;
template <typename T>
__global__ void __launch_bounds__(256, 4) k_conv_out(const uint16_t* __restrict__ h, const uint16_t* __restrict__ wt,
    const float* __restrict__ prm, float* __restrict__ zout, const double* __restrict__ R,
    const double* __restrict__ rms, T* __restrict__ out, int e, int nyb, int nzb, int nxc, int xl)
{
    typedef Window<kOH> W;
    __shared__ __align__(16) uint16_t lds[2][W::kSize];
    int b        = blockIdx.x;
    const int xc = b % nxc;
    b /= nxc;
    const int s = b / (nyb * nzb), y0 = (b / nzb) % nyb * kOY, z0 = b % nzb * kLZ;
    const int x0 = xc * xl, x1 = min(e, x0 + xl);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int tsel = g >> 1, cs = 8 * (g & 1);
    const int64_t e3 = (int64_t)e * e * e;
    // A: row n = 4(dy+1) + dx+1; K = (dz = -1, 0) x 16, then dz = 1 (and zeros)
    s8 wa[2];
#pragma unroll
    for (int k = 0; k < 2; k++)
    {
        const int dy = n >> 2, dx = n & 3;
        const bool on = dy < 3 && dx < 3 && !(k && tsel);
        const int tap = on ? (dx * 3 + dy) * 3 + (k ? 2 : tsel) : 0;
        wa[k]         = *(const s8*)(wt + (size_t)tap * 256 + cs);
        if (!on) wa[k] = (s8){ 0, 0, 0, 0, 0, 0, 0, 0 };
    }
    // the wave's rows: outputs y0+2wid, +1; inputs window rows 2wid .. 2wid+3
    const int hb = (g & 1) * W::kHalf;
    const int p0 = hb + (2 * wid * kLW + n + tsel) * 8, q0 = hb + (2 * wid * kLW + n + 2) * 8;
    W w(h + (int64_t)s * e3 * 16, e, y0, z0);
    const float bias = prm[kB3], sk = prm[kS];
    const double rs = rms ? rms[s] : 1., inv = 1. / rs;
    const bool two = z0 + 16 < e;
    // lane (n, g) writes row g >> 1, z-tile g & 1 of the wave's four tiles
    const int yo = y0 + 2 * wid + (g >> 1), zo = z0 + 16 * (g & 1) + n;
    const bool store_ok = yo < e && zo < e;
    const int64_t vox0 = (int64_t)s * e3 + (int64_t)yo * e + zo, e2 = (int64_t)e * e;
    // writes plane x from element EL of the row tiles; rv: R there
    auto emit = [&](auto EL, int x, const f4 (&c)[4][2], double rv) {
        constexpr int el = decltype(EL)::value;
        float mine       = 0.f;
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int t = 0; t < 2; t++)
            {
                const float a0 = c[r][t][el], a1 = c[r + 1][t][el], a2 = c[r + 2][t][el];
                float v = g == 0 ? a0 : a1;
                v       = g == 2 ? a2 : v;
                v       = g == 3 ? 0.f : v;
                v += __shfl_xor(v, 16, 64);
                v += __shfl_xor(v, 32, 64);
                mine = g == 2 * r + t ? v : mine;
            }
        if (!store_ok) return;
        const float z = bias + mine;
        if (R)
            out[vox0 + x * e2] = (T)((double)(sk * (float)(rv * inv) + z) * rs);
        else
            zout[vox0 + x * e2] = z;
    };
    const f4 zero = { 0.f, 0.f, 0.f, 0.f };
    f4 c[4][2];
#pragma unroll
    for (int r = 0; r < 4; r++)
        c[r][0] = c[r][1] = zero;
    const int xa = max(x0 - 1, 0), xb = min(x1, e - 1);
    double rp = 0., rc = 0.;  // R on planes xp - 1, xp: loaded a plane ahead of its use
    w.load(xa);
    for (int xp = xa; xp <= xb; xp++)
    {
        uint16_t* buf = lds[xp & 1];
        w.store(buf);
        __syncthreads();
        rp = rc;
        if (R && store_ok) rc = R[vox0 + xp * e2];
        if (xp < xb) w.load(xp + 1);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < 2; t++)
            {
                if (t && !two) continue;
                const s8 b0 = *(const s8*)(buf + p0 + (r * kLW + 16 * t) * 8);
                const s8 b1 = *(const s8*)(buf + q0 + (r * kLW + 16 * t) * 8);
                const f4 o  = c[r][t];
                f4 d        = { 0.f, o[0], o[1], 0.f };
                d           = mfma32(wa[0], b0, d);
                c[r][t]     = mfma32(wa[1], b1, d);
            }
        if (xp > x0) emit(std::integral_constant<int, 2>(), xp - 1, c, rp);
    }
    if (x1 == e) emit(std::integral_constant<int, 1>(), e - 1, c, rc);
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

// per box: rms_j = sqrt(mean R_j^2) (0 -> 1); x = R/rms (FP32); t = KR/rms.
// One block of 16 waves per box with four loads in flight per thread: 256
// boxes of 32^3 17 us (4 waves, one load at a time: 55 us)
__global__ void __launch_bounds__(1024) k_box_rms(const double* R, int64_t m, double* rms)
{
    __shared__ double red[16];
    const double* r = R + (int64_t)blockIdx.x * m;
    double a[4]     = { 0., 0., 0., 0. };
    int64_t i       = threadIdx.x;
    for (; i + 3 * 1024 < m; i += 4 * 1024)
    {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k] = r[i + 1024 * k];
#pragma unroll
        for (int k = 0; k < 4; k++)
            a[k] += v[k] * v[k];
    }
    for (; i < m; i += 1024)
        a[0] += r[i] * r[i];
    double t = (a[0] + a[1]) + (a[2] + a[3]);
    for (int o = 32; o > 0; o >>= 1)
        t += __shfl_xor(t, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        t = 0.;
        for (int k = 0; k < 16; k++)
            t += red[k];
        t                = sqrt(t / (double)m);
        rms[blockIdx.x] = t > 0. ? t : 1.;
    }
}

__global__ void k_box_scale_to_f32(const double* R, const double* rms, int64_t m, int64_t n, float* x)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = (float)(R[i] / rms[i / m]);
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
    float *z = nullptr, *dy = nullptr;
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

// planes per x-chunk of a marching kernel with `cols` columns of blocks: the
// whole edge when they alone give four blocks per CU (what the registers of
// k_conv16 let reside), else chunks of at least four planes (each reads a plane
// more on either side).  64 boxes of 32^3, k_conv16: 37 us in two chunks, 47 us
// in one
int march_xl(int e, int64_t cols)
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
    const int nyb = (e + kLY - 1) / kLY, nzb = (e + kLZ - 1) / kLZ, cols = nb * nyb * nzb;
    const int xl = march_xl(e, cols), nxc = (e + xl - 1) / xl;
    const dim3 lgrid((unsigned)(cols * nxc));
    const uint16_t* nomask = nullptr;
    if (R)
        hipLaunchKernelGGL((k_conv1<double, CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, R, rms,
            (const uint16_t*)c->f0, (const float*)c->p + kB0, c->h1, nomask, e, nyb, nzb, nxc, xl);
    else
        hipLaunchKernelGGL((k_conv1<float, CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, x, (const double*)nullptr,
            (const uint16_t*)c->f0, (const float*)c->p + kB0, c->h1, nomask, e, nyb, nzb, nxc, xl);
    hipLaunchKernelGGL((k_conv16<CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->h1,
        (const uint16_t*)c->f1, (const float*)c->p + kB1, c->h2, nomask, e, nyb, nzb, nxc, xl);
    hipLaunchKernelGGL((k_conv16<CONV_FWD_RELU>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->h2,
        (const uint16_t*)c->f2, (const float*)c->p + kB2, c->h3, nomask, e, nyb, nzb, nxc, xl);
    const int noy = (e + kOY - 1) / kOY, ocols = nb * noy * nzb, oxl = march_xl(e, ocols), onx = (e + oxl - 1) / oxl;
    hipLaunchKernelGGL(k_conv_out<T>, dim3((unsigned)(ocols * onx)), dim3(256), 0, ctx->stream,
        (const uint16_t*)c->h3, (const uint16_t*)c->f3, (const float*)c->p, c->z, R, rms, out, e, noy, nzb, onx, oxl);
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
    const int xl  = march_xl(e, cols), nxc = (e + xl - 1) / xl;
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
    const int e     = c->edge;
    const int64_t n = (int64_t)nb * e * e * e;
    hipLaunchKernelGGL(k_loss, dim3(kLossBlocks), dim3(256), 0, ctx->stream, x, (const float*)c->z, t,
        (const float*)c->p, n, (float*)nullptr, c->dy, c->lpart);
    hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(192), 0, ctx->stream, (const double*)c->lpart, kLossBlocks, c->g,
        c->lpart + 3 * kLossBlocks);
    MGX_CHECK_LAUNCH(ctx);
    DwLayers L;
    // layer 3: dZ3 = dy (scalar; its bias came with the loss)
    if ((rc = dw1<true>(c, c->h3, c->dy, nb, c->part3, L.l[3]))) return rc;
    L.l[3].gw = c->g + kW3, L.l[3].gb = nullptr;
    const int nyb = (e + kLY - 1) / kLY, nzb = (e + kLZ - 1) / kLZ, cols = nb * nyb * nzb;
    const int xl = march_xl(e, cols), nxc = (e + xl - 1) / xl;
    const dim3 lgrid((unsigned)(cols * nxc));
    const float* nobias = nullptr;
    hipLaunchKernelGGL((k_conv1<float, CONV_BWD_MASK>), lgrid, dim3(256), 0, ctx->stream, (const float*)c->dy,
        (const double*)nullptr, (const uint16_t*)c->r3, nobias, c->dza, (const uint16_t*)c->h3, e, nyb, nzb, nxc, xl);
    MGX_CHECK_LAUNCH(ctx);
    // layer 2: dZ2 = dza
    if ((rc = dw16(c, c->dza, c->h2, nb, c->part2, L.l[2]))) return rc;
    L.l[2].gw = c->g + kW2, L.l[2].gb = c->g + kB2;
    hipLaunchKernelGGL((k_conv16<CONV_BWD_MASK>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->dza,
        (const uint16_t*)c->r2, nobias, c->dzb, (const uint16_t*)c->h2, e, nyb, nzb, nxc, xl);
    MGX_CHECK_LAUNCH(ctx);
    // layer 1: dZ1 = dzb
    if ((rc = dw16(c, c->dzb, c->h1, nb, c->part1, L.l[1]))) return rc;
    L.l[1].gw = c->g + kW1, L.l[1].gb = c->g + kB1;
    hipLaunchKernelGGL((k_conv16<CONV_BWD_MASK>), lgrid, dim3(256), 0, ctx->stream, (const uint16_t*)c->dzb,
        (const uint16_t*)c->r1, nobias, c->dza, (const uint16_t*)c->h1, e, nyb, nzb, nxc, xl);
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
    al((void**)&c->dy, nv * sizeof(float));
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
    void* bufs[] = { c->p, c->g, c->m, c->v, c->wbf, c->h1, c->h2, c->h3, c->dza, c->dzb, c->z, c->dy, c->part0,
        c->part1, c->part2, c->part3, c->lpart, c->rms };
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
    MGX_CHECK_HIP(c->ctx, hipMemcpyAsync(host, c->p, kNP * sizeof(float), hipMemcpyDeviceToHost, c->ctx->stream));
    return sync(c->ctx);
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
    return sync(c->ctx);
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
    hipLaunchKernelGGL(k_box_rms, dim3(nbox), dim3(1024), 0, ctx->stream, R, m, rms);
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
        hipLaunchKernelGGL(k_box_rms, dim3(nb), dim3(1024), 0, ctx->stream, Rb, m, c->rms);
        MGX_CHECK_LAUNCH(ctx);
        rc = out_dtype == MGX_F32
                 ? forward_any<float>(c, nullptr, Rb, c->rms, nb, (float*)out + (int64_t)b0 * m)
                 : forward_any<double>(c, nullptr, Rb, c->rms, nb, (double*)out + (int64_t)b0 * m);
        if (rc) return rc;
    }
    return MGX_OK;
}
}  // namespace mgx
