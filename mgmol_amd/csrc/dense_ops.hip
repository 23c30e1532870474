// dense_ops.hip -- tall-skinny contractions on MFMA and the FP64 dense layer.
//
// ss(i,j) = vel * sum_k A(k,i) B(k,j) over one slab of rows (the reference's
// per-subdomain LocalMatrices, src/LocGridOrbitals.cc:1504-1604).  Each wave
// owns the tiles of one pair of column panels and every so many 16-row chunks:
//   PREC_F64  : v_mfma_f64_16x16x4_f64, FP64 accumulation;
//   PREC_SPLIT: x = hi + lo (hi = fl32(x), lo = fl32(x - hi)),
//               v_mfma_f32_16x16x4_f32 on hi*hi and hi*lo + lo*hi, FP32
//               accumulation over 16 rows, FP64 sums of those.
// Chunk partials are reduced in a fixed order (deterministic) and scaled.
#include "common.hpp"

#include <rocsolver/rocsolver.h>

#include <mutex>
#include <type_traits>

namespace mgx
{
namespace
{

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;  // waves per block, each on its own row sub-chunk

// MFMA 16x16x4 operand layout (CDNA3/CDNA4): lane l supplies A[m=l%16][k=l/16]
// and B[k=l/16][n=l%16].  Accumulator v of lane l holds D[4*(l/16)+v][l%16]
// for v_mfma_f32_16x16x4_f32 and D[l/16+4*v][l%16] for v_mfma_f64_16x16x4_f64
// (both checked on gfx950 by tests/test_gpu_dense.py).
// Panels of TW 16-column tiles: a wave holds the TW x TW output tiles of one
// panel pair for its share of the rows (all of an output up to 64 columns, so
// each operand is read once) and reads its columns straight from memory: lane
// (c, r) takes rows 4r..4r+3 of a 16-row chunk of column c (32 bytes; a column's
// 16 rows are 128 contiguous bytes), which the MFMAs take as their four steps
// (a product does not care which row is which k, as long as A and B agree).
// The next chunk's loads are in flight during the MFMAs.  The four waves of a
// block take neighbouring chunks and add their tiles through LDS in order.
//   PREC_F64  : TW^2 (a Gram's diagonal pair: the lower tiles) MFMAs per step;
//   PREC_SPLIT: hi * hi and hi * lo + lo * hi in FP32 over the 16 rows, added
//               in FP64.
// Bound by the FP64 matrix rate and HBM together.  64 columns of 884736 rows:
// Gram 107 us (4.2 TB/s), product 170 us (5.3 TB/s, 43 TFLOP/s); 16x16 tiles of
// scattered 8-byte loads took 852 us each.
template <int PREC, int TW, bool DIAG, bool VEC>
__device__ __forceinline__ void tsgemm_panels(const double* A, const double* B, int64_t ld, int64_t k_begin,
    int64_t lnp, int n, int i0, int j0, int chunk, int nchunk, double* red, double* out)
{
    typedef double dd2 __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, c = lane & 15, r = lane >> 4;
    const double *pa[TW], *pb[TW];
#pragma unroll
    for (int q = 0; q < TW; q++)
    {
        // columns past n repeat the last one; their results are not written
        pa[q] = A + (int64_t)min(i0 + 16 * q + c, n - 1) * ld + k_begin + 4 * r;
        pb[q] = B + (int64_t)min(j0 + 16 * q + c, n - 1) * ld + k_begin + 4 * r;
    }
    struct Frag
    {
        double v[TW][4];
    };
    auto load = [&](Frag& f, const double* const (&p)[TW], int64_t k) {
#pragma unroll
        for (int q = 0; q < TW; q++)
        {
            if (VEC)
            {
                const dd2 x = *(const dd2*)(p[q] + k), y = *(const dd2*)(p[q] + k + 2);
                f.v[q][0] = x[0], f.v[q][1] = x[1], f.v[q][2] = y[0], f.v[q][3] = y[1];
            }
            else
#pragma unroll
                for (int s = 0; s < 4; s++)
                    f.v[q][s] = p[q][k + s];
        }
    };
    d4 acc[TW][TW];
#pragma unroll
    for (int x = 0; x < TW; x++)
#pragma unroll
        for (int y = 0; y < TW; y++)
            acc[x][y] = (d4){ 0., 0., 0., 0. };
    auto mul = [&](const Frag& a, const Frag& b) {
        if (PREC == MGX_PREC_F64)
        {
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int x = 0; x < TW; x++)
#pragma unroll
                    for (int y = 0; y < TW; y++)
                        if (!DIAG || y <= x)
                            acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[x][s], b.v[y][s], acc[x][y], 0, 0, 0);
            return;
        }
        float ah[TW][4], al[TW][4], bh[TW][4], bl[TW][4];
#pragma unroll
        for (int q = 0; q < TW; q++)
#pragma unroll
            for (int s = 0; s < 4; s++)
            {
                ah[q][s] = (float)a.v[q][s];
                al[q][s] = (float)(a.v[q][s] - (double)ah[q][s]);
                bh[q][s] = DIAG ? ah[q][s] : (float)b.v[q][s];
                bl[q][s] = DIAG ? al[q][s] : (float)(b.v[q][s] - (double)bh[q][s]);
            }
#pragma unroll
        for (int x = 0; x < TW; x++)
#pragma unroll
            for (int y = 0; y < TW; y++)
            {
                if (DIAG && y > x) continue;
                f4 hh = { 0.f, 0.f, 0.f, 0.f }, hx = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
                for (int s = 0; s < 4; s++)
                {
                    hh = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[x][s], bh[y][s], hh, 0, 0, 0);
                    hx = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[x][s], bl[y][s], hx, 0, 0, 0);
                    hx = __builtin_amdgcn_mfma_f32_16x16x4f32(al[x][s], bh[y][s], hx, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[x][y][v] += (double)hh[v] + (double)hx[v];
            }
    };
    // full 16-row chunks first, first + step, ...
    const int64_t nfull = lnp / 16, first = (int64_t)chunk * kWaves + wid, step = (int64_t)nchunk * kWaves;
    Frag a0, b0, a1, b1;
    if (first < nfull)
    {
        load(a0, pa, 16 * first);
        if (!DIAG) load(b0, pb, 16 * first);
        for (int64_t ch = first;;)
        {
            // the last chunk is loaded again where there is no next one
            int64_t nx = ch + step, at = nx < nfull ? nx : ch;
            load(a1, pa, 16 * at);
            if (!DIAG) load(b1, pb, 16 * at);
            mul(a0, DIAG ? a0 : b0);
            if (nx >= nfull) break;
            ch = nx;
            nx = ch + step, at = nx < nfull ? nx : ch;
            load(a0, pa, 16 * at);
            if (!DIAG) load(b0, pb, 16 * at);
            mul(a1, DIAG ? a1 : b1);
            if (nx >= nfull) break;
            ch = nx;
        }
    }
    // the remaining lnp % 16 rows, by the wave whose turn it is
    if (nfull * 16 < lnp && nfull % step == first)
    {
#pragma unroll
        for (int q = 0; q < TW; q++)
#pragma unroll
            for (int s = 0; s < 4; s++)
            {
                const bool in = nfull * 16 + 4 * r + s < lnp;
                a0.v[q][s]    = in ? pa[q][nfull * 16 + s] : 0.;
                if (!DIAG) b0.v[q][s] = in ? pb[q][nfull * 16 + s] : 0.;
            }
        mul(a0, DIAG ? a0 : b0);
    }
    // the waves' tiles, added in wave order
    for (int w = 0; w < kWaves; w++)
    {
        if (wid == w)
        {
#pragma unroll
            for (int x = 0; x < TW; x++)
#pragma unroll
                for (int y = 0; y < TW; y++)
                {
                    if (DIAG && y > x) continue;
#pragma unroll
                    for (int v = 0; v < 4; v++)
                    {
                        double* p      = red + ((x * TW + y) * 4 + v) * 64 + lane;
                        const double t = w == 0 ? acc[x][y][v] : *p + acc[x][y][v];
                        if (w < kWaves - 1)
                            *p = t;
                        else
                        {
                            const int row = i0 + 16 * x + (PREC == MGX_PREC_F64 ? r + 4 * v : 4 * r + v);
                            const int col = j0 + 16 * y + c;
                            if (row < n && col < n) out[(int64_t)col * n + row] = t;
                        }
                    }
                }
        }
        if (w < kWaves - 1) __syncthreads();
    }
}

template <int PREC, int TW, bool VEC>
__global__ void __launch_bounds__(64 * kWaves, TW >= 3 ? 1 : 2) k_tsgemm(const double* A, const double* B, int64_t ld,
    int64_t lnp, int n, int npan, int nchunk, int lower_only, double* part)
{
    __shared__ double red[TW * TW * 256];
    const int chunk = blockIdx.x % nchunk, pair = blockIdx.x / nchunk, slab = blockIdx.z;
    int ti, tj;
    if (lower_only)
    {
        // pairs on and below the diagonal, row by row
        ti = 0;
        while ((ti + 1) * (ti + 2) / 2 <= pair)
            ti++;
        tj = pair - ti * (ti + 1) / 2;
    }
    else
    {
        ti = pair / npan;
        tj = pair - ti * npan;
    }
    const int64_t k0 = (int64_t)slab * lnp;
    double* out      = part + ((int64_t)slab * nchunk + chunk) * n * n;
    if (lower_only && ti == tj)
        tsgemm_panels<PREC, TW, true, VEC>(A, A, ld, k0, lnp, n, ti * 16 * TW, tj * 16 * TW, chunk, nchunk, red, out);
    else
        tsgemm_panels<PREC, TW, false, VEC>(A, B, ld, k0, lnp, n, ti * 16 * TW, tj * 16 * TW, chunk, nchunk, red, out);
}

// ss[slab](i,j) = vel * sum_chunks part; lower_only fills the upper triangle
// from the lower one (SquareLocalMatrices::fillUpperWithLower).  A block takes
// 32 neighbouring entries, eight groups of threads every eighth partial each,
// 16 loads in flight; the groups are added in order.  64 x 64 entries of 256
// partials: 8 us; one thread per entry took 101 us (a chain of loads).
__global__ void __launch_bounds__(256) k_chunk_reduce(const double* part, int n, int nchunk, int subdivx, double vel,
    int lower_only, double* ss)
{
    __shared__ double red[8][32];
    const int64_t nn = (int64_t)n * n, nt = (nn + 31) / 32;
    const int col32 = threadIdx.x & 31, grp = threadIdx.x >> 5;
    for (int64_t t = blockIdx.x; t < nt * subdivx; t += gridDim.x)
    {
        const int64_t slab = t / nt, e = (t - slab * nt) * 32 + col32;
        double s = 0.;
        if (e < nn)
        {
            const int col = (int)(e / n), row = (int)(e - (int64_t)col * n);
            // (col,row) element in col-major above the diagonal
            const double* p = part + slab * nchunk * nn + (lower_only && col > row ? (int64_t)row * n + col : e);
            int c           = grp;
            for (; c + 120 < nchunk; c += 128)
            {
                double v[16];
#pragma unroll
                for (int k = 0; k < 16; k++)
                    v[k] = p[(c + 8 * k) * nn];
#pragma unroll
                for (int k = 0; k < 16; k++)
                    s += v[k];
            }
            for (; c < nchunk; c += 8)
                s += p[c * nn];
        }
        red[grp][col32] = s;
        __syncthreads();
        if (grp == 0 && e < nn)
        {
            for (int g = 1; g < 8; g++)
                s += red[g][col32];
            ss[slab * nn + e] = s * vel;
        }
        __syncthreads();
    }
}

__global__ void k_l2g(const double* ss, const int* gids, int subdivx, int m, int numst, double tol, double* glob)
{
    // LocalMatrices2DistMatrix::convert, src/LocalMatrices2DistMatrix.cc:21-78;
    // one thread per (icolor, jcolor), slabs in order, consecutive same-pair
    // entries summed before the push.
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)m * m;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int ic = (int)(t / m), jc = (int)(t - (t / m) * m);
        int pst_old = -1;
        double val  = 0.;
        int st1o = -1, st2o = -1;
        for (int s = 0; s < subdivx; s++)
        {
            const int st1 = gids[s * m + ic];
            if (st1 == -1) continue;
            const int st2 = gids[s * m + jc];
            if (st2 == -1) continue;
            const int pst = st2 * numst + st1;
            const double v = ss[((int64_t)s * m + jc) * m + ic];
            if (fabs(v) > tol)
            {
                if (pst == pst_old)
                    val += v;
                else
                {
                    if (pst_old >= 0) atomicAdd(&glob[(int64_t)st2o * numst + st1o], val);
                    val     = v;
                    st1o    = st1;
                    st2o    = st2;
                    pst_old = pst;
                }
            }
        }
        if (pst_old >= 0) atomicAdd(&glob[(int64_t)st2o * numst + st1o], val);
    }
}

__global__ void k_tri(double* L, int n, int zero_upper)
{
    // zero_upper: L(i,j) = 0 for j > i ; else symmetrise from the lower triangle
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (t / n) * n);
        if (col <= row) continue;
        L[t] = zero_upper ? 0. : L[(int64_t)row * n + col];
    }
}

// A symmetric positive definite block (order m <= 128, its lower triangle
// read), pivot by pivot in registers.  With the pivot d = a_kk and its row and
// column w, a_ij becomes a_ij - w_i w_j / d:
//   FACTOR false  for every i, j (symmetric sweeps): a_ik turns into w_i / d
//                 and d into -1 / d; m sweeps leave minus the inverse, and P
//                 receives the inverse;
//   FACTOR true   for i > k only, which leaves row k of M, the inverse of the
//                 unit triangle of A = U D U^T, in the places j < k; P
//                 receives D^-1/2 M = L^-1, A = L L^T the Cholesky
//                 factorisation (zeros above the diagonal).
// 528 threads each hold a 4 x 4 tile on or below the diagonal; the pivot's w
// goes through LDS (two buffers, one barrier per pivot).  Bound by the pivots'
// chain, about 0.5 us each: 62 us at m = 128, where the library's blocked
// Cholesky and inverse take about 0.5 ms in 50 launches.  *info (a double
// beside the step's scalars): 1 + the first pivot that is not positive, else 0;
// first: no block came before.
constexpr int kSpdB = 128;
template <bool FACTOR>
__global__ void __launch_bounds__(576) k_spd_block(const double* A, int64_t ld, int m, double* P, int ldp, double* info,
    int k0, int first)
{
    __shared__ double v[2][kSpdB];
    __shared__ double piv[FACTOR ? kSpdB : 1];
    // tile (tr, tc), tc <= tr, of thread t = tr (tr + 1) / 2 + tc
    const int t = threadIdx.x;
    int tr      = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
    while ((tr + 1) * (tr + 2) / 2 <= t)
        tr++;
    while (tr * (tr + 1) / 2 > t)
        tr--;
    const int tc   = t - tr * (tr + 1) / 2;
    const bool act = t < kSpdB / 4 * (kSpdB / 4 + 1) / 2 && 4 * tr < m;
    double a[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
        {
            // a diagonal tile is held in full
            const int r = max(4 * tr + i, 4 * tc + j), c = min(4 * tr + i, 4 * tc + j);
            a[i][j]     = act && r < m ? A[(int64_t)c * ld + r] : (r == c ? 1. : 0.);
        }
    double bad = 0.;
    for (int k4 = 0; 4 * k4 < m; k4++)
    {
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
        {
            const int k = 4 * k4 + kk;  // padding pivots (k >= m) are ones
            double* w   = v[k & 1];
            if (act)
            {
                if (tc == k4)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        w[4 * tr + i] = FACTOR && tr == k4 && i < kk ? a[kk][i] : a[i][kk];
                else if (tr == k4)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        w[4 * tc + j] = a[kk][j];
            }
            __syncthreads();
            const double d = w[k];
            if (!(d > 0.) && bad == 0. && k < m) bad = (double)(k0 + k + 1);
            if (FACTOR && t == 0) piv[k] = d;
            // 1 / d: the hardware's estimate and two Newton steps, a third of
            // the division's chain
            double inv = __builtin_amdgcn_rcp(d);
            inv        = __builtin_fma(inv, __builtin_fma(-d, inv, 1.), inv);
            inv        = __builtin_fma(inv, __builtin_fma(-d, inv, 1.), inv);
            if (!act || (FACTOR && tr < k4)) continue;
            double wr[4], wc[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                wr[i] = w[4 * tr + i] * inv;
                wc[i] = w[4 * tc + i];
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (!FACTOR || tr > k4 || i > kk) a[i][j] = __builtin_fma(-wr[i], wc[j], a[i][j]);
            // the pivot's row and column, in the tiles that hold them
            if (FACTOR)
            {
                if (tc == k4)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (tr > k4 || i > kk) a[i][kk] = -wr[i];
                continue;
            }
            if (tc == k4)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    a[i][kk] = wr[i];
            if (tr == k4)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    a[kk][j] = wc[j] * inv;
            if (tr == k4 && tc == k4) a[kk][kk] = -inv;
        }
    }
    if (FACTOR) __syncthreads();
    if (act)
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const int r    = 4 * tr + i;
            const double s = FACTOR ? 1. / sqrt(piv[r]) : -1.;
#pragma unroll
            for (int j = 0; j < 4; j++)
            {
                const int c = 4 * tc + j;
                if (r >= m || c > r) continue;
                P[(int64_t)c * ldp + r] = FACTOR && r == c ? s : s * a[i][j];
                if (!FACTOR || r != c) P[(int64_t)r * ldp + c] = FACTOR ? 0. : s * a[i][j];
            }
        }
    if (t == 0 && (first || (*info == 0. && bad != 0.))) *info = bad;
}

// the block column [k0, k0 + m) of X to Q (n x m), its own rows the identity
__global__ void k_spd_panel(const double* X, int n, int k0, int m, double* Q)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * m; t += (int64_t)gridDim.x * blockDim.x)
    {
        const int j = (int)(t / n), row = (int)(t - (int64_t)j * n);
        Q[t]        = row >= k0 && row < k0 + m ? (row - k0 == j ? 1. : 0.) : X[(int64_t)k0 * n + t];
    }
}

// and back: block column and row from B = Q L^-T L^-1, the block from minus its
// own rows there
__global__ void k_spd_panel_back(double* X, int n, int k0, int m, const double* B)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * m; t += (int64_t)gridDim.x * blockDim.x)
    {
        const int j = (int)(t / n), row = (int)(t - (int64_t)j * n);
        const bool in = row >= k0 && row < k0 + m;
        X[(int64_t)(k0 + j) * n + row] = in ? -B[t] : B[t];
        if (!in) X[(int64_t)row * n + k0 + j] = B[t];
    }
}

// X <- -X, exactly symmetric (the lower triangle counts)
__global__ void k_spd_neg(double* X, int n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n; t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (int64_t)col * n);
        if (row < col) continue;
        const double v              = -X[t];
        X[t]                        = v;
        X[(int64_t)row * n + col] = v;
    }
}

// single block: out = sum_{i,k} H(i,k) * Sinv(k,i)
__global__ void __launch_bounds__(1024) k_trace_prod(const double* H, const double* Sinv, int n, double* out)
{
    __shared__ double red[1024];
    double s = 0.;
    for (int64_t t = threadIdx.x; t < (int64_t)n * n; t += blockDim.x)
    {
        const int k = (int)(t / n), i = (int)(t - (t / n) * n);  // H(i,k) at t
        s += H[t] * Sinv[(int64_t)i * n + k];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// single block: out = sum_i A(i,i)
__global__ void __launch_bounds__(256) k_diag_sum(const double* A, int n, double* out)
{
    __shared__ double red[256];
    double s = 0.;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        s += A[(int64_t)i * n + i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// per-block max |delta_ij - T(i,j)|, then a second pass over the blocks
__global__ void __launch_bounds__(256) k_id_err(const double* T, int n, double* blockmax)
{
    __shared__ double red[256];
    double m = 0.;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (t / n) * n);
        const double v = fabs(T[t] - (row == col ? 1. : 0.));
        m = v > m ? v : m;
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) blockmax[blockIdx.x] = red[0];
}

// k_id_err that also writes E = I - T and X in FP32 (the operands of the
// FP32 correction product of a Newton-Schulz step)
__global__ void __launch_bounds__(256) k_id_err_f32(const double* T, const double* X, int n, double* blockmax,
    float* E32, float* X32)
{
    __shared__ double red[256];
    double m = 0.;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (t / n) * n);
        const double e = (row == col ? 1. : 0.) - T[t];
        const double v = fabs(e);
        m              = v > m ? v : m;
        E32[t]         = (float)e;
        X32[t]         = (float)X[t];
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) blockmax[blockIdx.x] = red[0];
}

// round to the nearest BF16 (ties to even) through FP32
__device__ __forceinline__ uint16_t bf16_rn(double v)
{
    const float f    = (float)v;
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ double bf16_val(uint16_t h) { return (double)__uint_as_float((uint32_t)h << 16); }

// k_id_err with E = I - T and X as BF16 hi/lo pairs (hi = bf16(v),
// lo = bf16(v - hi)), laid out as the operands of one product with K = 3n:
// A = [Eh Eh El] (n x 3n) and B = [Xh; Xl; Xh] (3n x n), both column-major,
// so that A B = Eh Xh + Eh Xl + El Xh
__global__ void __launch_bounds__(256) k_id_err_bf16(const double* T, const double* X, int n, double* blockmax,
    uint16_t* A, uint16_t* B)
{
    __shared__ double red[256];
    double m = 0.;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (t / n) * n);
        const double e = (row == col ? 1. : 0.) - T[t];
        const double v = fabs(e);
        m              = v > m ? v : m;
        const int64_t nn  = (int64_t)n * n;
        const uint16_t eh = bf16_rn(e);
        A[t]              = eh;
        A[nn + t]         = eh;
        A[2 * nn + t]     = bf16_rn(e - bf16_val(eh));
        const double x    = X[t];
        const uint16_t xh = bf16_rn(x);
        const int64_t bj  = (int64_t)col * 3 * n + row;
        B[bj]             = xh;
        B[bj + n]         = bf16_rn(x - bf16_val(xh));
        B[bj + 2 * n]     = xh;
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) blockmax[blockIdx.x] = red[0];
}

// out = x + (double)y
__global__ void k_add_f32(const double* x, const float* y, double* out, int64_t n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        out[t] = x[t] + (double)y[t];
}

__global__ void __launch_bounds__(256) k_max_reduce(const double* v, int n, double* out)
{
    __shared__ double red[256];
    double m = 0.;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        m = fmax(m, v[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// X = (X + X^T)/2
// X = (X + X^T)/2 by 32 x 32 tile pairs through LDS (coalesced on both
// sides); each pair of entries gets 0.5 (x_pq + x_qp), as k_symmetrize
__global__ void __launch_bounds__(256) k_symmetrize_tiles(double* X, int n)
{
    __shared__ double a[32][33], b[32][33];
    const int ti = blockIdx.y, tj = blockIdx.x;
    if (tj < ti) return;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int k = ty; k < 32; k += 8)
    {
        // a[k][tx] = X(ti*32 + tx, tj*32 + k), b[k][tx] = X(tj*32 + tx, ti*32 + k)
        const int r = ti * 32 + tx, c = tj * 32 + k, r2 = tj * 32 + tx, c2 = ti * 32 + k;
        a[k][tx] = (r < n && c < n) ? X[r + (int64_t)c * n] : 0.;
        b[k][tx] = (r2 < n && c2 < n) ? X[r2 + (int64_t)c2 * n] : 0.;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8)
    {
        const int r = ti * 32 + tx, c = tj * 32 + k, r2 = tj * 32 + tx, c2 = ti * 32 + k;
        if (r < n && c < n) X[r + (int64_t)c * n] = 0.5 * (a[k][tx] + b[tx][k]);
        if (r2 < n && c2 < n) X[r2 + (int64_t)c2 * n] = 0.5 * (b[k][tx] + a[tx][k]);
    }
}

__global__ void k_symmetrize(double* X, int n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (t / n) * n);
        if (col >= row) continue;
        const int64_t u = (int64_t)row * n + col;
        const double a = 0.5 * (X[t] + X[u]);
        X[t] = a;
        X[u] = a;
    }
}

__global__ void k_sub(double* res, const double* hpsi, int64_t ld, int64_t numpt, int n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < numpt * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int64_t f = t / numpt, p = t - f * numpt;
        res[f * ld + p] += -1. * hpsi[f * ld + p];
    }
}

__global__ void __launch_bounds__(256) k_col_sumsq(const double* r, int64_t ld, int64_t numpt, double vel, double* d)
{
    __shared__ double red[256];
    const int f = blockIdx.x;
    double s    = 0.;
    for (int64_t p = threadIdx.x; p < numpt; p += blockDim.x)
        s += r[f * ld + p] * r[f * ld + p];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) d[f] = red[0] * vel;
}

__global__ void __launch_bounds__(256) k_diag_dot(const double* d, const double* Sinv, int n, double* out)
{
    __shared__ double red[256];
    double s = 0.;
    for (int j = threadIdx.x; j < n; j += blockDim.x)
        s += d[j] * Sinv[(int64_t)j * n + j];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = 0.5 * sqrt(red[0]);
}

// Y = X A, A pair-sparse symmetric, by column tiles: block (t, chunk) holds
// kSpTile output columns of tile t for 256 consecutive rows c, walks the
// union of the tile's rows k once (X[c, k] = X[k, c] read down column k,
// coalesced over c) and applies the tile's coefficients from LDS.
// One block per (column tile, 256-row chunk), mapped XCD-aware so that one
// XCD takes all the tiles of a row chunk: the union columns of the tiles it
// runs together then share that XCD's L2 (a row chunk of all of X is n x 2 KB)
__global__ void __launch_bounds__(256) k_spmm_tiles(const double* __restrict__ X, int n,
    const double* __restrict__ val, const int* tptr, const int* tcol, const int* tk, const int* te,
    double* __restrict__ Y, int ntile, int64_t nreal)
{
    constexpr int U = 64;
    __shared__ double cf[U][kSpTile];
    __shared__ int kk[U];
    const int64_t L = xcd_block(blockIdx.x, gridDim.x);
    if (L >= nreal) return;
    const int t = (int)(L % ntile);
    const int c = (int)(L / ntile) * 256 + threadIdx.x;
    double acc[kSpTile];
    for (int q = 0; q < kSpTile; q++)
        acc[q] = 0.;
    const int u0 = tptr[t], u1 = tptr[t + 1];
    for (int ub = u0; ub < u1; ub += U)
    {
        const int m = min(U, u1 - ub);
        for (int z = threadIdx.x; z < U * kSpTile; z += 256)
        {
            const int u = z / kSpTile, q = z - (z / kSpTile) * kSpTile;
            double v    = 0.;
            if (u < m)
            {
                const int e = te[(int64_t)(ub + u) * kSpTile + q];
                if (e >= 0) v = val[e];
            }
            cf[u][q] = v;
        }
        if (threadIdx.x < U) kk[threadIdx.x] = threadIdx.x < m ? tk[ub + threadIdx.x] : 0;
        __syncthreads();
        if (c < n)
            for (int u = 0; u < m; u++)
            {
                const double x = X[c + (int64_t)kk[u] * n];
                for (int q = 0; q < kSpTile; q++)
                    acc[q] += cf[u][q] * x;
            }
        __syncthreads();
    }
    if (c < n)
        for (int q = 0; q < kSpTile; q++)
        {
            const int r = tcol[t * kSpTile + q];
            if (r >= 0) Y[c + (int64_t)r * n] = acc[q];
        }
}

// out = 0.5 (a + a^T)  (MatrixType::transpose(0.5, work, 0.5) after symm)
__global__ void k_sym_half(const double* a, int n, double* out)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (int64_t)col * n);
        out[t] = 0.5 * a[t] + 0.5 * a[(int64_t)row * n + col];
    }
}

}  // namespace

int spmm_pairs(mgx_ctx* ctx, int n, const double* X, const double* val, const PairTiles& pt, double* Y)
{
    if (pt.ntile <= 0) return set_err(ctx, MGX_EINVAL, "no column tiles");
    // X read and Y written once: 16 n^2 bytes
    const int tk = prof_begin(ctx, MGX_PROF_SPMM, 16. * (double)n * n);
    const int64_t nreal = (int64_t)pt.ntile * ((n + 255) / 256);
    hipLaunchKernelGGL(k_spmm_tiles, dim3((unsigned)((nreal + 7) / 8 * 8)), dim3(256), 0, ctx->stream, X, n, val,
        pt.ptr, pt.col, pt.k, pt.e, Y, pt.ntile, nreal);
    prof_end(ctx, tk);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

// Wide products (n >= kWideN): the tiles of k_tsgemm would re-read each
// column strip n/16 times from scattered 8-byte loads.  FP64: the library's
// dgemm (the reference's own DGEMM), split over K into batches (an n x n
// output alone is too few tiles for the chip when K is hundreds of
// thousands of rows) whose partial products are summed in FP64:
// strided-batched dgemm over chunks of kF64Chunk rows or more (at most
// kF64MaxParts partials) plus one dgemm for the remainder.  Split:
// k_tsgemm_split_wide (below).  A Gram (A == B) is mirrored from its lower
// triangle, so it is exactly symmetric.
constexpr int kWideN       = 256;
constexpr int kF64Chunk    = 16384;
constexpr int kF64MaxParts = 64;

// C = sum_c parts[c] (FP64, np partials of n x n); sym: both triangles from
// the lower
__global__ void k_sum_parts(const double* parts, int np, int n, int sym, double* C)
{
    const int64_t nn = (int64_t)n * n;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nn; t += (int64_t)gridDim.x * blockDim.x)
    {
        const int col = (int)(t / n), row = (int)(t - (int64_t)col * n);
        if (sym && row < col) continue;
        double v = 0.;
        for (int c = 0; c < np; c++)
            v += parts[c * nn + t];
        C[t] = v;
        if (sym) C[(int64_t)row * n + col] = v;
    }
}

// The hi/lo split of a wide product on FP32 MFMA.  One block computes a
// kWT x kWT output tile (rows from A's columns i0.., columns from B's j0..)
// over one range of rows (a K-split).  Per chunk of kWK rows the block loads
// both column panels once, coalesced (a wave reads two columns' 512
// contiguous bytes per instruction), splits each value into hi = fl32(x),
// lo = fl32(x - hi) in registers and stores them to LDS column by column
// (stride kWL floats: the stores and the MFMA operand reads are free of bank
// conflicts).  Each wave owns a 32 x 32 quadrant (2 x 2 tiles of
// v_mfma_f32_16x16x4_f32): hi*hi and hi*lo + lo*hi accumulate in FP32 over
// the chunk's kWK rows, then the chunk sums are added in FP64.  Partial
// products of the K-splits go to part (FP64, n x n each, column-major).
constexpr int kWT = 64;  // output tile edge
constexpr int kWK = 64;  // rows per LDS panel
constexpr int kWR = 4;   // rows per FP32 sum of hi*hi (then added in FP64)
constexpr int kWL = 68;  // LDS column stride in floats (64 rows + 4)

__global__ void __launch_bounds__(256, 2) k_tsgemm_split_wide(const double* A, const double* B, int64_t ld,
    int64_t lnp, int n, int ntile, int64_t rows_per_split, int lower_only, double* part)
{
    typedef double dd2 __attribute__((ext_vector_type(2)));
    typedef float ff2 __attribute__((ext_vector_type(2)));
    // lower_only: the grid enumerates the tiles on and below the diagonal
    // only (so the round-robin of blocks over the XCDs stays balanced)
    const int tile = blockIdx.x;
    int ti, tj;
    if (lower_only)
    {
        ti = (int)((sqrtf(8.f * (float)tile + 1.f) - 1.f) * 0.5f);
        while ((ti + 1) * (ti + 2) / 2 <= tile)
            ti++;
        while (ti * (ti + 1) / 2 > tile)
            ti--;
        tj = tile - ti * (ti + 1) / 2;
    }
    else
    {
        ti = tile / ntile;
        tj = tile - ti * ntile;
    }
    const int split  = blockIdx.y;
    const int64_t k0 = (int64_t)split * rows_per_split;
    const int64_t k1 = min(k0 + rows_per_split, lnp);
    // a diagonal tile of a Gram reads one panel for both operands
    const bool one = A == B && ti == tj;
    __shared__ float Ah[kWT * kWL], Al[kWT * kWL], Bh[kWT * kWL], Bl[kWT * kWL];
    const float* Bhr = one ? Ah : Bh;
    const float* Blr = one ? Al : Bl;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wi = w & 1, wj = w >> 1;
    const int c = lane & 15, r = lane >> 4;
    const int i0 = ti * kWT, j0 = tj * kWT;
    // loader: rows 2 rr, 2 rr + 1 of column q * 8 + (t >> 5) for q = 0..7
    const int rr = 2 * (t & 31), cq = t >> 5;
    double acc[2][2][4] = {};
    for (int64_t kc = k0; kc < k1; kc += kWK)
    {
        const int64_t row = kc + rr;
#pragma unroll
        for (int q = 0; q < 8; q++)
        {
            const int col = q * 8 + cq;
            // two rows at once where they are 16-byte aligned (even ld),
            // else one by one
            auto ld2 = [&](const double* p) -> dd2 {
                dd2 v = { 0., 0. };
                if (row + 1 < k1 && (reinterpret_cast<uintptr_t>(p) & 15) == 0)
                    v = *reinterpret_cast<const dd2*>(p);
                else
                {
                    if (row < k1) v[0] = p[0];
                    if (row + 1 < k1) v[1] = p[1];
                }
                return v;
            };
            dd2 a = { 0., 0. }, b = { 0., 0. };
            if (i0 + col < n) a = ld2(A + (int64_t)(i0 + col) * ld + row);
            if (!one && j0 + col < n) b = ld2(B + (int64_t)(j0 + col) * ld + row);
            ff2 h, l;
            h[0] = (float)a[0];
            h[1] = (float)a[1];
            l[0] = (float)(a[0] - (double)h[0]);
            l[1] = (float)(a[1] - (double)h[1]);
            *reinterpret_cast<ff2*>(Ah + col * kWL + rr) = h;
            *reinterpret_cast<ff2*>(Al + col * kWL + rr) = l;
            if (!one)
            {
                h[0] = (float)b[0];
                h[1] = (float)b[1];
                l[0] = (float)(b[0] - (double)h[0]);
                l[1] = (float)(b[1] - (double)h[1]);
                *reinterpret_cast<ff2*>(Bh + col * kWL + rr) = h;
                *reinterpret_cast<ff2*>(Bl + col * kWL + rr) = l;
            }
        }
        __syncthreads();
        // hi*hi: FP32 sums over kWR rows (kWR / 4 MFMA steps), then into
        // FP64; the cross terms (2^-24 of it) in FP32 over the panel's rows
        f4 hx[2][2];
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int y = 0; y < 2; y++)
                hx[x][y] = f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll 2
        for (int s0 = 0; s0 < kWK / 4; s0 += kWR / 4)
        {
            f4 hh[2][2];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
                    hh[x][y] = f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int s = s0; s < s0 + kWR / 4; s++)
            {
                const int kk = 4 * s + r;
                float ah[2], al[2], bh[2], bl[2];
#pragma unroll
                for (int x = 0; x < 2; x++)
                {
                    const int ia = (wi * 32 + x * 16 + c) * kWL + kk;
                    const int jb = (wj * 32 + x * 16 + c) * kWL + kk;
                    ah[x]        = Ah[ia];
                    al[x]        = Al[ia];
                    bh[x]        = Bhr[jb];
                    bl[x]        = Blr[jb];
                }
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int y = 0; y < 2; y++)
                    {
                        hh[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[x], bh[y], hh[x][y], 0, 0, 0);
                        hx[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[x], bl[y], hx[x][y], 0, 0, 0);
                        hx[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(al[x], bh[y], hx[x][y], 0, 0, 0);
                    }
            }
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        acc[x][y][v] += (double)hh[x][y][v];
        }
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int y = 0; y < 2; y++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[x][y][v] += (double)hx[x][y][v];
        __syncthreads();
    }
    // accumulator v of lane l: D[4 (l / 16) + v][l % 16] (FP32 MFMA layout)
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int v = 0; v < 4; v++)
            {
                const int row = i0 + wi * 32 + x * 16 + 4 * r + v;
                const int col = j0 + wj * 32 + y * 16 + c;
                if (row < n && col < n) part[((int64_t)split * n + col) * n + row] = acc[x][y][v];
            }
}

int tsgemm_wide(mgx_ctx* ctx, int prec, const double* A, const double* B, int64_t ld, int64_t lnp, int n,
    int subdivx, double vel, double* ss)
{
    const int64_t nn = (int64_t)n * n;
    const bool same  = A == B;
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    for (int sl = 0; sl < subdivx; sl++)
    {
        const double* As = A + (int64_t)sl * lnp;
        const double* Bs = B + (int64_t)sl * lnp;
        double* C        = ss + sl * nn;
        if (prec == MGX_PREC_F64)
        {
            const double zero  = 0.;
            const int64_t kc   = std::max<int64_t>(kF64Chunk, (lnp + kF64MaxParts - 1) / kF64MaxParts);
            const int64_t nful = lnp / kc, rem = lnp - nful * kc;
            const int np       = (int)(nful + (rem > 0));
            double* parts      = (double*)workspace(ctx, 7, (size_t)np * nn * sizeof(double));
            if (!parts) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
            rocblas_status st = rocblas_status_success;
            // full products also for a Gram: rocBLAS dsyrk measured 10x slower here
            if (nful > 0)
                st = rocblas_dgemm_strided_batched(ctx->blas, rocblas_operation_transpose, rocblas_operation_none,
                    n, n, (rocblas_int)kc, &vel, As, (rocblas_int)ld, kc, Bs, (rocblas_int)ld, kc, &zero, parts, n,
                    nn, (rocblas_int)nful);
            if (st == rocblas_status_success && rem > 0)
                st = rocblas_dgemm(ctx->blas, rocblas_operation_transpose, rocblas_operation_none, n, n,
                    (rocblas_int)rem, &vel, As + nful * kc, (rocblas_int)ld, Bs + nful * kc, (rocblas_int)ld,
                    &zero, parts + nful * nn, n);
            if (st != rocblas_status_success) return set_err(ctx, MGX_EHIP, "rocBLAS FP64 product failed");
            hipLaunchKernelGGL(k_sum_parts, dim3(nblocks(nn)), dim3(kBlock), 0, ctx->stream, (const double*)parts, np,
                n, same ? 1 : 0, C);
            MGX_CHECK_LAUNCH(ctx);
            continue;
        }
        // split: K divided among enough blocks to fill the chip (at least
        // 32 chunks each), rows per split a multiple of the chunk
        const int ntile     = (n + kWT - 1) / kWT;
        const int active    = same ? ntile * (ntile + 1) / 2 : ntile * ntile;
        const int64_t nchk  = (lnp + kWK - 1) / kWK;
        const int64_t want  = std::max<int64_t>(1, (2048 + active - 1) / active);
        const int nsplit    = (int)std::max<int64_t>(1, std::min<int64_t>(want, nchk / 32));
        const int64_t rps   = ((nchk + nsplit - 1) / nsplit) * kWK;
        double* parts       = (double*)workspace(ctx, 7, (size_t)nsplit * nn * sizeof(double));
        if (!parts) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
        dim3 grid(active, nsplit), blk(256);
        hipLaunchKernelGGL(k_tsgemm_split_wide, grid, blk, 0, ctx->stream, As, Bs, ld, lnp, n, ntile, rps,
            same ? 1 : 0, parts);
        MGX_CHECK_LAUNCH(ctx);
        hipLaunchKernelGGL(k_chunk_reduce, dim3(nblocks((nn + 31) / 32, 1)), dim3(256), 0, ctx->stream,
            (const double*)parts, n, nsplit, 1, vel, same ? 1 : 0, C);
        MGX_CHECK_LAUNCH(ctx);
    }
    return MGX_OK;
}

// part_ext: a caller-given buffer of part_cap bytes for the chunk partials
// (the number of chunks is lowered to fit it), else the context's workspace
int tsgemm(mgx_ctx* ctx, int prec, const double* A, const double* B, int64_t ld, int64_t lnp, int n, int subdivx,
    double vel, int lower_only, double* ss, double* part_ext = nullptr, size_t part_cap = 0)
{
    MGX_REQUIRE(ctx, A && B && ss && n > 0 && subdivx > 0 && lnp > 0, "bad product arguments");
    MGX_REQUIRE(ctx, (int64_t)subdivx * lnp <= ld, "slabs exceed the leading dimension");
    MGX_REQUIRE(ctx, prec == MGX_PREC_F64 || prec == MGX_PREC_SPLIT, "bad precision mode");
    if (n >= kWideN) return tsgemm_wide(ctx, prec, A, B, ld, lnp, n, subdivx, vel, ss);
    // the fewest panels of at most four tiles, all of one width.  With few rows
    // a wide pair is a chain of up to 16 tiles' MFMAs per 16 rows beside an idle
    // chip: single tiles where wide pairs would give under 176 (split: 224)
    // blocks of 256 rows.  Product of 100 columns of 1000 rows, split: 49 us in
    // wide pairs, 19 in single tiles; near the line, Gram of 200 columns of 6000
    // rows, split (230 blocks): 53 and 40; product of 48 columns of 50000 rows,
    // FP64 (195 blocks): 32 and 37.
    const int ntile = (n + 15) / 16;
    int npan = (ntile + 3) / 4, tw = (ntile + npan - 1) / npan;
    auto npairs = [&]() { return lower_only ? npan * (npan + 1) / 2 : npan * npan; };
    const int64_t wide = npairs() * subdivx * std::max<int64_t>(1, lnp / 256);
    if (wide < (prec == MGX_PREC_F64 ? 176 : 224)) npan = ntile, tw = 1;
    const int pairs = npairs();
    // blocks of four waves: as many per CU as the tiles' registers let reside
    // (1, 2, 3, 6 for widths 4..1), each wave at least four chunks of 16 rows
    static const int percu[4] = { 6, 3, 2, 1 };
    const int64_t want = (256 * percu[tw - 1] + (int64_t)pairs * subdivx - 1) / ((int64_t)pairs * subdivx);
    int nchunk         = (int)std::max<int64_t>(1, std::min<int64_t>(want, lnp / 256));
    const size_t per_chunk = (size_t)subdivx * n * n * sizeof(double);
    double* part           = part_ext;
    if (part_ext)
    {
        MGX_REQUIRE(ctx, per_chunk <= part_cap, "subdivx * n * n * 8 bytes exceed the scratch buffer");
        nchunk = (int)std::min<size_t>((size_t)nchunk, part_cap / per_chunk);
    }
    else
    {
        part = (double*)workspace(ctx, 7, per_chunk * nchunk);
        if (!part) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    }
    // 16-byte loads where every column of every slab is aligned for them
    const bool vec = ((((uintptr_t)A | (uintptr_t)B) & 15) | (ld & 1) | (subdivx > 1 ? lnp & 1 : 0)) == 0;
    const dim3 grid((unsigned)(pairs * nchunk), 1, subdivx), blk(64 * kWaves);
    auto launch = [&](auto P, auto W) {
        constexpr int PREC = decltype(P)::value, TW = decltype(W)::value;
        if (vec)
            hipLaunchKernelGGL((k_tsgemm<PREC, TW, true>), grid, blk, 0, ctx->stream, A, B, ld, lnp, n, npan, nchunk,
                lower_only, part);
        else
            hipLaunchKernelGGL((k_tsgemm<PREC, TW, false>), grid, blk, 0, ctx->stream, A, B, ld, lnp, n, npan, nchunk,
                lower_only, part);
    };
    auto widths = [&](auto P) {
        switch (tw)
        {
            case 1: launch(P, std::integral_constant<int, 1>()); break;
            case 2: launch(P, std::integral_constant<int, 2>()); break;
            case 3: launch(P, std::integral_constant<int, 3>()); break;
            default: launch(P, std::integral_constant<int, 4>());
        }
    };
    if (prec == MGX_PREC_F64)
        widths(std::integral_constant<int, MGX_PREC_F64>());
    else
        widths(std::integral_constant<int, MGX_PREC_SPLIT>());
    MGX_CHECK_LAUNCH(ctx);
    const int64_t nt = ((int64_t)n * n + 31) / 32 * subdivx;
    hipLaunchKernelGGL(k_chunk_reduce, dim3(nblocks(nt, 1)), dim3(256), 0, ctx->stream, (const double*)part, n,
        nchunk, subdivx, vel, lower_only, ss);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

int chol_inv(mgx_ctx* ctx, int n, const double* S, double* L, double* Sinv)
{
    MGX_REQUIRE(ctx, n > 0 && S && L && Sinv, "bad chol_inv arguments");
    int* info = (int*)workspace(ctx, 6, 64);
    if (!info) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    const size_t bytes = (size_t)n * n * sizeof(double);
    if (L != S) MGX_CHECK_HIP(ctx, hipMemcpyAsync(L, S, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    if (rocsolver_dpotrf(ctx->blas, rocblas_fill_lower, n, L, n, info) != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocsolver_dpotrf failed");
    int hinfo = 0;
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(&hinfo, info, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    MGX_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (hinfo != 0)
        return set_err(ctx, MGX_ENOTSPD, "ERROR in GramMatrix<MatrixType>::updateLS(): potrf info != 0");
    hipLaunchKernelGGL(k_tri, dim3(nblocks((int64_t)n * n)), dim3(kBlock), 0, ctx->stream, L, n, 1);
    MGX_CHECK_LAUNCH(ctx);
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(Sinv, L, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    if (rocsolver_dpotri(ctx->blas, rocblas_fill_lower, n, Sinv, n, info) != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocsolver_dpotri failed");
    hipLaunchKernelGGL(k_tri, dim3(nblocks((int64_t)n * n)), dim3(kBlock), 0, ctx->stream, Sinv, n, 0);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

// X = S^-1 for a symmetric positive definite S (lower triangle read; X apart
// from S), without its Cholesky factor: one launch of symmetric sweeps up to
// order 128, else in place by blocks of 128.  With A the block as the blocks
// before it left it, A = L L^T and Q the block's column of X (identity in its
// own rows): W = Q L^-T, X - W W^T, and the column itself becomes W L^-1.  The
// part not yet reached is so reduced as by a Cholesky factorisation; with the
// block's inverse instead (X - Q A^-1 Q^T) it took errors of the order of
// cond(A) and |I - S X| was 25 times (cond 1e6) to 4e4 times (1e13) the
// library's at n = 400.  Six launches a block.
// info (device) receives 1 + the index of the first pivot that is not
// positive, else 0.  n = 2048: 2.05 ms against the library's 7.3 ms;
// 512: 0.42 ms against 1.6 ms.
int spd_inv_launch(mgx_ctx* ctx, int n, const double* S, double* X, double* info)
{
    if (n <= kSpdB)
    {
        hipLaunchKernelGGL(k_spd_block<false>, dim3(1), dim3(576), 0, ctx->stream, S, (int64_t)n, n, X, n, info, 0, 1);
        MGX_CHECK_LAUNCH(ctx);
        return MGX_OK;
    }
    double* Q = (double*)workspace(ctx, 7, (2 * (size_t)n * kSpdB + (size_t)kSpdB * kSpdB) * sizeof(double));
    if (!Q) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    double *W = Q + (size_t)n * kSpdB, *Li = W + (size_t)n * kSpdB;
    const double one = 1., zero = 0., mone = -1.;
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(X, S, (size_t)n * n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    hipLaunchKernelGGL(k_tri, dim3(nblocks((int64_t)n * n)), dim3(kBlock), 0, ctx->stream, X, n, 0);
    for (int k0 = 0; k0 < n; k0 += kSpdB)
    {
        const int m = std::min(kSpdB, n - k0);
        hipLaunchKernelGGL(k_spd_block<true>, dim3(1), dim3(576), 0, ctx->stream, (const double*)X + (size_t)k0 * n + k0,
            (int64_t)n, m, Li, m, info, k0, k0 == 0);
        hipLaunchKernelGGL(k_spd_panel, dim3(nblocks((int64_t)n * m)), dim3(kBlock), 0, ctx->stream, (const double*)X, n,
            k0, m, Q);
        MGX_CHECK_LAUNCH(ctx);
        // W = Q L^-T, X -= W W^T (the block's own row and column too, which
        // are written next), Q = W L^-1
        if (rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_transpose, n, m, m, &one, Q, n, Li, m,
                &zero, W, n)
                != rocblas_status_success
            || rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_transpose, n, n, m, &mone, W, n, W, n,
                   &one, X, n)
                   != rocblas_status_success
            || rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, m, m, &one, W, n, Li, m, &zero,
                   Q, n)
                   != rocblas_status_success)
            return set_err(ctx, MGX_EHIP, "rocblas_dgemm failed");
        hipLaunchKernelGGL(k_spd_panel_back, dim3(nblocks((int64_t)n * m)), dim3(kBlock), 0, ctx->stream, X, n, k0, m,
            (const double*)Q);
    }
    hipLaunchKernelGGL(k_spd_neg, dim3(nblocks((int64_t)n * n)), dim3(kBlock), 0, ctx->stream, X, n);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

int spd_check(mgx_ctx* ctx, double info)
{
    if (info == 0.) return MGX_OK;
    return set_err(ctx, MGX_ENOTSPD, "matrix not positive definite (pivot " + std::to_string((int)info) + ")");
}

// spd_inv_launch with its check (waits for the stream)
int spd_inv(mgx_ctx* ctx, int n, const double* S, double* X)
{
    double* info = (double*)workspace(ctx, 6, 64);
    if (!info) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    if (int rc = spd_inv_launch(ctx, n, S, X, info)) return rc;
    double h = 0.;
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(&h, info, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MGX_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return spd_check(ctx, h);
}

int diag_sum(mgx_ctx* ctx, int n, const double* A, double* dev_out)
{
    hipLaunchKernelGGL(k_diag_sum, dim3(1), dim3(256), 0, ctx->stream, A, n, dev_out);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

// Refresh X ~ S^-1 by Newton-Schulz steps from the previous inverse (S changes
// little between orbital steps, so the iteration starts well inside its
// quadratic basin), S pair-sparse (values Sv per pair, column tiles pt):
// T = X S on the sparse product, X <- 2X - T X as one dense GEMM (written to
// the other half of the work buffer, operands swapped, no copies).  Stops
// before a step once delta = max|I - X S| < tol.  With FP64 products it also
// stops after a step once delta^2 (the error that step leaves) < tol; with
// lowp the correction E X, E = I - X S, is one FP32 product, whose rounding
// (~1e-7 |E| |X|) can exceed delta^2, so only measured deltas end the loop.
// Falls back to spd_inv when delta does not start below 0.25 (a large change)
// or fails to contract; *steps = steps taken (-1: spd_inv ran).  work: 2 n^2.
int inverse_update_pairs(mgx_ctx* ctx, int n, const double* S, const double* Sv, const PairTiles& pt, double* X,
    double* work, int* steps, double tol, bool lowp)
{
    const double mone = -1., two = 2.;
    const size_t nn = (size_t)n * n;
    double* T   = work;
    double* cur = X;
    double* nxt = work + nn;
    double* bm  = (double*)workspace(ctx, 4, 1024 * sizeof(double));
    if (!bm) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    float *E32 = nullptr, *X32 = nullptr, *Y32 = nullptr;
    if (lowp)
    {
        E32 = (float*)workspace(ctx, 7, 3 * nn * sizeof(float));
        if (!E32) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
        X32 = E32 + nn;
        Y32 = X32 + nn;
    }
    const double gflop = 2. * (double)n * n * n;
    double prev = 1e300;
    *steps      = 0;
    int rc;
    for (int it = 0; it < 10; it++)
    {
        if ((rc = spmm_pairs(ctx, n, cur, Sv, pt, T))) return rc;
        const int nb = 512;
        if (lowp)
            hipLaunchKernelGGL(k_id_err_f32, dim3(nb), dim3(256), 0, ctx->stream, (const double*)T,
                (const double*)cur, n, bm, E32, X32);
        else
            hipLaunchKernelGGL(k_id_err, dim3(nb), dim3(256), 0, ctx->stream, (const double*)T, n, bm);
        hipLaunchKernelGGL(k_max_reduce, dim3(1), dim3(256), 0, ctx->stream, (const double*)bm, nb, bm + nb);
        MGX_CHECK_LAUNCH(ctx);
        double delta = 0.;
        MGX_CHECK_HIP(ctx, hipMemcpyAsync(&delta, bm + nb, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        MGX_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (!(delta < 0.25) || delta > 0.5 * prev)
        {
            *steps = -1;
            return spd_inv(ctx, n, S, X);
        }
        if (delta < tol) break;
        if (lowp)
        {
            // nxt = cur + E cur
            const float onef = 1.f, zerof = 0.f;
            if (rocblas_sgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, n, &onef, E32, n, X32,
                    n, &zerof, Y32, n)
                != rocblas_status_success)
                return set_err(ctx, MGX_EHIP, "rocblas_sgemm failed");
            hipLaunchKernelGGL(k_add_f32, dim3(nblocks((int64_t)nn)), dim3(kBlock), 0, ctx->stream,
                (const double*)cur, (const float*)Y32, nxt, (int64_t)nn);
            MGX_CHECK_LAUNCH(ctx);
        }
        else
        {
            // nxt = 2 cur - T cur
            const int tk = prof_begin(ctx, MGX_PROF_NSGEMM, gflop);
            if (rocblas_gemm_ex(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, n, &mone, T,
                    rocblas_datatype_f64_r, n, cur, rocblas_datatype_f64_r, n, &two, cur, rocblas_datatype_f64_r, n,
                    nxt, rocblas_datatype_f64_r, n, rocblas_datatype_f64_r, rocblas_gemm_algo_standard, 0, 0)
                != rocblas_status_success)
                return set_err(ctx, MGX_EHIP, "rocblas_gemm_ex failed");
            prof_end(ctx, tk);
        }
        std::swap(cur, nxt);
        (*steps)++;
        prev = delta;
        if (!lowp && delta * delta < tol) break;  // the error after this step is ~delta^2
    }
    if (cur != X) MGX_CHECK_HIP(ctx, hipMemcpyAsync(X, cur, nn * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    hipLaunchKernelGGL(k_symmetrize, dim3(nblocks((int64_t)nn)), dim3(kBlock), 0, ctx->stream, X, n);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

// inverse_update_pairs without host waits: nsteps Newton-Schulz steps from
// X, each recording delta_k = max|I - X_k S| (before step k) in deltas[k]
// on the device.  With bf16 the correction E X of a step is one BF16 product
// with K = 3n of hi/lo parts (Eh Xh + Eh Xl + El Xh, FP32 sums; relative
// error ~1e-5 of |E| |X|), so delta^2 does not bound the error a step leaves:
// the delta of the final X is measured too, into deltas[nsteps].  The caller
// reads the deltas later with its other scalars and checks them
// (ns_spec_check).
// the start of a refresh: X <- 2 X - P (on) and P <- the X it was given: the
// linear extrapolation of the last two inverses, S changing little from one
// step to the next (the steps then start an order closer)
__global__ void k_extrap(double* X, double* P, int64_t n, int on)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    {
        const double t = X[i];
        if (on) X[i] = 2. * t - P[i];
        P[i] = t;
    }
}

// xprev (may be null): the inverse of the step before, n x n; with extrap the
// steps start from 2 X - xprev, and xprev receives the X they were given
int inverse_update_spec(mgx_ctx* ctx, int n, const double* Sv, const PairTiles& pt, double* X, double* work,
    int nsteps, bool bf16, double* deltas, double* xprev, bool extrap)
{
    if (xprev)
    {
        hipLaunchKernelGGL(k_extrap, dim3(nblocks((int64_t)n * n)), dim3(kBlock), 0, ctx->stream, X, xprev,
            (int64_t)n * n, extrap ? 1 : 0);
        MGX_CHECK_LAUNCH(ctx);
    }
    const double mone = -1., two = 2.;
    const size_t nn = (size_t)n * n;
    double* T   = work;
    double* cur = X;
    double* nxt = work + nn;
    double* bm  = (double*)workspace(ctx, 4, 1024 * sizeof(double));
    if (!bm) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    float* Y32     = nullptr;
    uint16_t* H16  = nullptr;
    if (bf16)
    {
        Y32 = (float*)workspace(ctx, 7, nn * sizeof(float) + 6 * nn * sizeof(uint16_t));
        if (!Y32) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
        H16 = reinterpret_cast<uint16_t*>(Y32 + nn);
    }
    const double flop = 2. * (double)n * n * n;
    int rc;
    const int nb = 512;
    for (int it = 0; it < nsteps; it++)
    {
        if ((rc = spmm_pairs(ctx, n, cur, Sv, pt, T))) return rc;
        if (bf16)
            hipLaunchKernelGGL(k_id_err_bf16, dim3(nb), dim3(256), 0, ctx->stream, (const double*)T,
                (const double*)cur, n, bm, H16, H16 + 3 * nn);
        else
            hipLaunchKernelGGL(k_id_err, dim3(nb), dim3(256), 0, ctx->stream, (const double*)T, n, bm);
        hipLaunchKernelGGL(k_max_reduce, dim3(1), dim3(256), 0, ctx->stream, (const double*)bm, nb, deltas + it);
        MGX_CHECK_LAUNCH(ctx);
        if (bf16)
        {
            const float onef = 1.f, zerof = 0.f;
            const int tk = prof_begin(ctx, MGX_PROF_NSGEMM16, 3. * flop);
            if (rocblas_gemm_ex(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, 3 * n, &onef, H16,
                    rocblas_datatype_bf16_r, n, H16 + 3 * nn, rocblas_datatype_bf16_r, 3 * n, &zerof, Y32,
                    rocblas_datatype_f32_r, n, Y32, rocblas_datatype_f32_r, n, rocblas_datatype_f32_r,
                    rocblas_gemm_algo_standard, 0, 0)
                != rocblas_status_success)
                return set_err(ctx, MGX_EHIP, "rocblas_gemm_ex (bf16) failed");
            prof_end(ctx, tk);
            hipLaunchKernelGGL(k_add_f32, dim3(nblocks((int64_t)nn)), dim3(kBlock), 0, ctx->stream,
                (const double*)cur, (const float*)Y32, nxt, (int64_t)nn);
            MGX_CHECK_LAUNCH(ctx);
        }
        else
        {
            const int tk = prof_begin(ctx, MGX_PROF_NSGEMM, flop);
            if (rocblas_gemm_ex(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, n, &mone, T,
                    rocblas_datatype_f64_r, n, cur, rocblas_datatype_f64_r, n, &two, cur, rocblas_datatype_f64_r, n,
                    nxt, rocblas_datatype_f64_r, n, rocblas_datatype_f64_r, rocblas_gemm_algo_standard, 0, 0)
                != rocblas_status_success)
                return set_err(ctx, MGX_EHIP, "rocblas_gemm_ex failed");
            prof_end(ctx, tk);
        }
        std::swap(cur, nxt);
    }
    if (cur != X) MGX_CHECK_HIP(ctx, hipMemcpyAsync(X, cur, nn * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    hipLaunchKernelGGL(k_symmetrize_tiles, dim3((n + 31) / 32, (n + 31) / 32), dim3(256), 0, ctx->stream, X, n);
    MGX_CHECK_LAUNCH(ctx);
    if (bf16)
    {
        // the error the last BF16 step left, on the symmetrised X
        if ((rc = spmm_pairs(ctx, n, X, Sv, pt, T))) return rc;
        hipLaunchKernelGGL(k_id_err, dim3(nb), dim3(256), 0, ctx->stream, (const double*)T, n, bm);
        hipLaunchKernelGGL(k_max_reduce, dim3(1), dim3(256), 0, ctx->stream, (const double*)bm, nb, deltas + nsteps);
        MGX_CHECK_LAUNCH(ctx);
    }
    return MGX_OK;
}

// The checks inverse_update_pairs makes step by step, on the deltas of
// inverse_update_spec: 0 = the steps were enough (*needed = the steps the
// checked loop would have taken), 1 = they converge but more are needed,
// -1 = they do not converge (spd_inv).  With final (the BF16 steps)
// deltas[nsteps] holds the measured error of the final X, and only a
// measured delta below tol accepts.
int ns_spec_check(const double* deltas, int nsteps, double tol, bool final, int* needed)
{
    double prev = 1e300;
    for (int k = 0; k < nsteps; k++)
    {
        const double d = deltas[k];
        if (!(d < 0.25) || d > 0.5 * prev) return -1;
        if (d < tol)
        {
            *needed = k;
            return 0;
        }
        if (!final && d * d < tol)
        {
            *needed = k + 1;
            return 0;
        }
        prev = d;
    }
    if (final)
    {
        const double d = deltas[nsteps];
        if (!(d < 0.25) || d > 0.5 * prev) return -1;
        if (d < tol)
        {
            *needed = nsteps;
            return 0;
        }
    }
    *needed = nsteps;
    return 1;
}

int theta(mgx_ctx* ctx, int n, const double* Sinv, const double* H, double* th)
{
    const double one = 1., zero = 0.;
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    if (rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, n, &one, Sinv, n, H, n, &zero,
            th, n)
        != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocblas_dgemm failed");
    return MGX_OK;
}

int trace_prod(mgx_ctx* ctx, int n, const double* H, const double* Sinv, double* dev_out)
{
    hipLaunchKernelGGL(k_trace_prod, dim3(1), dim3(1024), 0, ctx->stream, H, Sinv, n, dev_out);
    MGX_CHECK_LAUNCH(ctx);
    return MGX_OK;
}

int ritz(mgx_ctx* ctx, int n, const double* H, const double* S, double* eig, double* Z)
{
    const size_t bytes = (size_t)n * n * sizeof(double);
    double* w          = (double*)workspace(ctx, 5, 2 * bytes + (size_t)n * sizeof(double) + 256);
    if (!w) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    double* A  = w;
    double* B  = w + (size_t)n * n;
    double* E  = B + (size_t)n * n;
    int* info  = (int*)workspace(ctx, 6, 64);
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(A, H, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(B, S, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    if (rocsolver_dsygvd(ctx->blas, rocblas_eform_ax, Z ? rocblas_evect_original : rocblas_evect_none,
            rocblas_fill_lower, n, A, n, B, n, eig, E, info)
        != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocsolver_dsygvd failed");
    int hinfo = 0;
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(&hinfo, info, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    MGX_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (hinfo != 0) return set_err(ctx, hinfo > n ? MGX_ENOTSPD : MGX_ENUMERIC, "sygvd did not converge / S not SPD");
    if (Z) MGX_CHECK_HIP(ctx, hipMemcpyAsync(Z, A, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    return MGX_OK;
}

}  // namespace mgx

// Scratch of mgx_local_gram_noalloc: the chunk partials of k_tsgemm, at most
// kNoAllocBytes.  The array is the device memory itself (one copy per GPU,
// held until the process ends); host code uses only the device address that
// scratch_init() takes from hipGetSymbolAddress, never the array's name.
constexpr size_t kNoAllocBytes = size_t(16) << 20;
static __device__ __align__(256) double scratch[kNoAllocBytes / sizeof(double)];

namespace mgx
{
namespace
{
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// once per device, with that device current (context creation): the device
// address of this GPU's copy of `scratch`
int scratch_init(mgx_ctx* ctx, int device)
{
    if (device < 0 || device >= kMaxDevices) return set_err(ctx, MGX_EINVAL, "device index out of range for scratch");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return MGX_OK;
    void* p        = nullptr;
    hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
        return set_err(ctx, MGX_EHIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(err));
    g_scratch_ptr[device] = p;
    return MGX_OK;
}

}  // namespace mgx

using namespace mgx;

extern "C" {

int mgx_local_gram(mgx_ctx* ctx, int prec, const double* psi, int64_t ld, int64_t lnp, int n, int subdivx,
    double vel, double* ss)
{
    int rc = tsgemm(ctx, prec, psi, psi, ld, lnp, n, subdivx, vel, 1, ss);
    return rc ? rc : sync(ctx);
}

int mgx_local_gram_noalloc(mgx_ctx* ctx, int prec, const double* psi, int64_t ld, int64_t lnp, int n, int subdivx,
    double vel, double* ss)
{
    if (!ctx) return MGX_EINVAL;
    MGX_REQUIRE(ctx, n > 0 && n < kWideN, "mgx_local_gram_noalloc takes n < 256 (wider products use rocBLAS)");
    void* p = ctx->device >= 0 && ctx->device < kMaxDevices ? g_scratch_ptr[ctx->device] : nullptr;
    MGX_REQUIRE(ctx, p, "scratch address of this device not set up (mgx_ctx_create)");
    // every partial the reduction reads is written by the same call: nothing
    // to clear; calls that overlap on one GPU share the array and race
    int rc = tsgemm(ctx, prec, psi, psi, ld, lnp, n, subdivx, vel, 1, ss, (double*)p, kNoAllocBytes);
    return rc ? rc : sync(ctx);
}

int mgx_local_product(mgx_ctx* ctx, int prec, const double* a, const double* b, int64_t ld, int64_t lnp, int n,
    int subdivx, double vel, double* ss)
{
    int rc = tsgemm(ctx, prec, a, b, ld, lnp, n, subdivx, vel, 0, ss);
    return rc ? rc : sync(ctx);
}

int mgx_local_to_global(mgx_ctx* ctx, const double* ss, const int* gids, int subdivx, int m, int numst, double tol,
    double* glob)
{
    MGX_REQUIRE(ctx, ss && gids && glob && subdivx > 0 && m > 0 && numst > 0, "bad local_to_global arguments");
    hipLaunchKernelGGL(k_l2g, dim3(nblocks((int64_t)m * m)), dim3(kBlock), 0, ctx->stream, ss, gids, subdivx, m,
        numst, tol, glob);
    MGX_CHECK_LAUNCH(ctx);
    return sync(ctx);
}

int mgx_chol_inv(mgx_ctx* ctx, int n, const double* S, double* L, double* Sinv)
{
    int rc = chol_inv(ctx, n, S, L, Sinv);
    return rc ? rc : sync(ctx);
}

int mgx_theta(mgx_ctx* ctx, int n, const double* Sinv, const double* H, double* th)
{
    MGX_REQUIRE(ctx, n > 0 && Sinv && H && th, "bad theta arguments");
    int rc = theta(ctx, n, Sinv, H, th);
    return rc ? rc : sync(ctx);
}

int mgx_eigsum(mgx_ctx* ctx, int n, const double* H, const double* Sinv, double* trace)
{
    MGX_REQUIRE(ctx, n > 0 && H && Sinv && trace, "bad eigsum arguments");
    double* d = (double*)workspace(ctx, 4, 256);
    if (!d) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    int rc = trace_prod(ctx, n, H, Sinv, d);
    if (rc) return rc;
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(trace, d, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

int mgx_ritz(mgx_ctx* ctx, int n, const double* H, const double* S, double* eig, double* Z)
{
    MGX_REQUIRE(ctx, n > 0 && H && S && eig, "bad ritz arguments");
    int rc = ritz(ctx, n, H, S, eig, Z);
    return rc ? rc : sync(ctx);
}

int mgx_mehr_projected(mgx_ctx* ctx, int n, const double* S, const double* Sinv, const double* B, const double* H,
    double* invB, double* theta, double* HB, double* eigsum)
{
    MGX_REQUIRE(ctx, n > 0 && S && Sinv && B && H && invB && theta && HB, "bad projected-matrix arguments");
    const size_t nn = (size_t)n * n;
    double* w       = (double*)workspace(ctx, 5, 2 * nn * sizeof(double) + 64);
    if (!w) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    // invB (ProjectedMatricesMehrstellen::computeInvB: potrf + potri)
    if (invB == B)
        MGX_CHECK_HIP(ctx, hipMemcpyAsync(w, B, nn * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    int rc = spd_inv(ctx, n, invB == B ? w : B, invB);
    if (rc) return rc;
    // theta = invB H (updateTheta)
    if ((rc = mgx::theta(ctx, n, invB, H, theta))) return rc;
    // HB = 0.5 (S theta + (S theta)^T) (updateHB)
    const double one = 1., zero = 0.;
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    if (rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, n, n, n, &one, S, n, theta, n, &zero,
            w, n)
        != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocblas_dgemm failed");
    hipLaunchKernelGGL(k_sym_half, dim3(nblocks((int64_t)nn)), dim3(kBlock), 0, ctx->stream, (const double*)w, n, HB);
    MGX_CHECK_LAUNCH(ctx);
    // eigsum = tr(HB Sinv) (getEigSum)
    if (eigsum)
    {
        double* dv = w + nn;
        if ((rc = trace_prod(ctx, n, HB, Sinv, dv))) return rc;
        MGX_CHECK_HIP(ctx, hipMemcpyAsync(eigsum, dv, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    }
    return sync(ctx);
}

int mgx_residual(mgx_ctx* ctx, const double* psi, const double* hpsi, const double* th, int64_t ld, int64_t numpt,
    int n, double* res)
{
    MGX_REQUIRE(ctx, psi && hpsi && th && res && n > 0 && numpt > 0 && ld >= numpt, "bad residual arguments");
    const double one = 1., zero = 0.;
    rocblas_set_pointer_mode(ctx->blas, rocblas_pointer_mode_host);
    if (rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, (rocblas_int)numpt, n, n, &one, psi,
            (rocblas_int)ld, th, n, &zero, res, (rocblas_int)ld)
        != rocblas_status_success)
        return set_err(ctx, MGX_EHIP, "rocblas_dgemm failed");
    hipLaunchKernelGGL(k_sub, dim3(nblocks(numpt * n)), dim3(kBlock), 0, ctx->stream, res, hpsi, ld, numpt, n);
    MGX_CHECK_LAUNCH(ctx);
    return sync(ctx);
}

int mgx_residual_norm(mgx_ctx* ctx, const double* res, int64_t ld, int64_t numpt, int n, double vel,
    const double* Sinv, double* norm)
{
    MGX_REQUIRE(ctx, res && Sinv && norm && n > 0, "bad residual_norm arguments");
    double* d = (double*)workspace(ctx, 4, (n + 8) * sizeof(double));
    if (!d) return set_err(ctx, MGX_ENOMEM, "workspace allocation failed");
    hipLaunchKernelGGL(k_col_sumsq, dim3(n), dim3(256), 0, ctx->stream, res, ld, numpt, vel, d);
    hipLaunchKernelGGL(k_diag_dot, dim3(1), dim3(256), 0, ctx->stream, (const double*)d, Sinv, n, d + n);
    MGX_CHECK_LAUNCH(ctx);
    MGX_CHECK_HIP(ctx, hipMemcpyAsync(norm, d + n, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    return sync(ctx);
}

}  // extern "C"
