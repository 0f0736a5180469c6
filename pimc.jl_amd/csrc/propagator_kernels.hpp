// Integral terms of the pair-product propagator on the device
// (prop_rel_interpolate_terms, src/propagator.jl:36-70):
//
//   terms(r1, r2) = -term1 - term2 + term3
//                 = sum_q [ -a_q J0(k_q r1) J0(k_q r2)
//                           - b_q (J0(k_q r1) Y0(k_q r2) + J0(k_q r2) Y0(k_q r1))
//                           + a_q Y0(k_q r1) Y0(k_q r2) ]
//
// over the nodes k_q of a fixed Gauss-Legendre rule on [0, K] (in place of
// quadgk), with a_q = w_q k_q e^{-tau k_q^2} / (2 pi) tk^2 / (1 + tk^2) and
// b_q = ... tk / (1 + tk^2), tk = 1 / ((2/pi)(eulergamma + log(k/2)) - 4/g0).
// The node list and a_q, b_q are built on the host (pimc_prop_int_terms).
//
// Step 1 (k_prop_bessel) tabulates J0 and Y0 at every (grid radius, node);
// step 2 (k_prop_terms, k_prop_fold) is the contraction over the nodes, a
// product of an (n x 2nk) and a (2nk x n) matrix with the 2 x 2 node weights
// [[-a, -b], [-b, a]] folded into one operand.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

namespace pimc {

// J[q * n + i] = J0(k_q r_i), Y[q * n + i] = Y0(k_q r_i), r_i = r0 + i h.
__global__ void k_prop_bessel(const double *__restrict__ k, int nk, double r0, double h, int n, double *__restrict__ J,
                              double *__restrict__ Y)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * nk) return;
    const int q = (int)(t / n), i = (int)(t - (long long)q * n);
    const double r = r0 + i * h;
    J[t] = j0(k[q] * r);
    Y[t] = y0(k[q] * r);
}

constexpr int kPropTile = 64, kPropChunk = 16, kPropThreads = 256;
constexpr int kPropRow = kPropTile + 16; // LDS row of a staged operand: the rows of a half wave start 128 B apart
                                         // modulo the 256 B of the banks
typedef double double4_t __attribute__((ext_vector_type(4)));

// Tiles (ti <= tl) of the upper triangle of the symmetric product, row by row.
__host__ __device__ inline int prop_tiles(int n)
{
    const int nt = (n + kPropTile - 1) / kPropTile;
    return nt * (nt + 1) / 2;
}

// Ranges the nodes are split into: enough workgroups for two on every CU (the
// 55 tiles of n = 600 alone would leave four fifths of the chip idle), each
// range at least 8 chunks long.
inline int prop_splits(int n, int nk, int cus)
{
    const int chunks = (nk + kPropChunk - 1) / kPropChunk;
    return std::max(1, std::min((2 * cus + prop_tiles(n) - 1) / prop_tiles(n), chunks / 8));
}

// part[(split * tiles + tile) * 64 * 64 + ...]: the split's share of one 64 x 64
// tile of terms(r_i, r_l).  The contraction runs on the FP64 matrix unit: each of
// the four waves owns 32 x 32 outputs as 2 x 2 tiles of v_mfma_f64_16x16x4 and
// takes both operands from LDS, where a chunk of 16 nodes (32 rows: u, v of the
// tile's rows against J, Y of its columns) is staged while the next chunk's loads
// are in flight.  Grid (tiles, splits).  What bounds it is the matrix unit's FP64
// rate; only the upper triangle is computed.  n = 600, whole call: 1.68 ms with the
// product on the vector unit (one workgroup per tile of the square, all nodes each),
// 0.43 ms so.
__global__ void __launch_bounds__(kPropThreads)
    k_prop_terms(const double *__restrict__ J, const double *__restrict__ Y, const double *__restrict__ ca,
                 const double *__restrict__ cb, int nk, int n, double *__restrict__ part)
{
    __shared__ double sA[2 * kPropChunk][kPropRow], sB[2 * kPropChunk][kPropRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nt = (n + kPropTile - 1) / kPropTile;
    int ti = 0, rest = blockIdx.x;
    while (rest >= nt - ti) rest -= nt - ti, ++ti;
    const int i0 = ti * kPropTile, l0 = (ti + rest) * kPropTile;
    const int chunks = (nk + kPropChunk - 1) / kPropChunk;
    const int c0 = (int)((long long)chunks * blockIdx.y / gridDim.y);
    const int c1 = (int)((long long)chunks * (blockIdx.y + 1) / gridDim.y);

    // a wave stages nodes wave, wave + 4, ... of row `lane` of both operands
    double Ji[4], Yi[4], Jl[4], Yl[4], a[4], b[4];
    const int gi = i0 + lane, gl = l0 + lane;
    auto load = [&](int c) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int q = c * kPropChunk + wave + 4 * x;
            const bool in = q < nk, oi = in && gi < n, ol = in && gl < n;
            a[x] = in ? ca[q] : 0.0;
            b[x] = in ? cb[q] : 0.0;
            Ji[x] = oi ? J[(size_t)q * n + gi] : 0.0;
            Yi[x] = oi ? Y[(size_t)q * n + gi] : 0.0;
            Jl[x] = ol ? J[(size_t)q * n + gl] : 0.0;
            Yl[x] = ol ? Y[(size_t)q * n + gl] : 0.0;
        }
    };
    double4_t acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = double4_t{0.0, 0.0, 0.0, 0.0};
    const int wi = (wave & 1) * 32, wl = (wave >> 1) * 32; // the wave's corner of the tile
    const int fr = lane & 15, fk = lane >> 4;              // operand layout: row (column) lane % 16, depth lane / 16

    if (c0 < c1) load(c0);
    for (int c = c0; c < c1; ++c) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int q = wave + 4 * x;
            sA[2 * q][lane] = -a[x] * Ji[x] - b[x] * Yi[x];
            sA[2 * q + 1][lane] = -b[x] * Ji[x] + a[x] * Yi[x];
            sB[2 * q][lane] = Jl[x];
            sB[2 * q + 1][lane] = Yl[x];
        }
        __syncthreads();
        if (c + 1 < c1) load(c + 1);
#pragma unroll
        for (int k = 0; k < 2 * kPropChunk; k += 4) {
            double fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                fa[x] = sA[k + fk][wi + 16 * x + fr];
                fb[x] = sB[k + fk][wl + 16 * x + fr];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[x], fb[y], acc[x][y], 0, 0, 0);
        }
        __syncthreads();
    }
    double *out = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kPropTile * kPropTile;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) // result layout: row 4 r + lane / 16, column lane % 16
                out[(wi + 16 * x + 4 * r + fk) * kPropTile + wl + 16 * y + fr] = acc[x][y][r];
}

// out[i * n + l] = out[l * n + i] = the splits' shares of terms(r_i, r_l), in
// split order; grid (tiles, 16 rows each), one thread per element.
__global__ void __launch_bounds__(kPropThreads)
    k_prop_fold(const double *__restrict__ part, int splits, int n, double *__restrict__ out)
{
    const int nt = (n + kPropTile - 1) / kPropTile;
    int ti = 0, rest = blockIdx.x;
    while (rest >= nt - ti) rest -= nt - ti, ++ti;
    const int i0 = ti * kPropTile, l0 = (ti + rest) * kPropTile;
    const size_t tile = kPropTile * kPropTile, step = (size_t)gridDim.x * tile;
    const int e0 = blockIdx.y * kPropTile * 4;
    for (int e = e0 + (int)threadIdx.x; e < e0 + kPropTile * 4; e += kPropThreads) {
        const double *p = part + (size_t)blockIdx.x * tile + e;
        double s = 0.0;
        for (int k = 0; k < splits; ++k) s += p[k * step];
        const int gi = i0 + e / kPropTile, gl = l0 + e % kPropTile;
        if (gi < n && gl < n && gl >= gi) {
            out[(size_t)gi * n + gl] = s;
            out[(size_t)gl * n + gi] = s;
        }
    }
}

} // namespace pimc
