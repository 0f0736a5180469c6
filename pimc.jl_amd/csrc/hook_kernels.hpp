// Single-move and single-estimate kernels behind the C ABI: one reference
// move (ReshapeLinear, SingleCenterOfMass), one interaction_action! value, one
// Energy or Density evaluation, and the adjoint of the potential action.
// They reuse the device physics of the sweep kernels on one chain's HBM
// paths, so checking them against the oracle checks that arithmetic.
#pragma once
#include "sweep_kernels.hpp"

namespace pimc {

struct HookArgs {
    const ChainDev *chains;
    void *pos;
    int *cell_cnt;
    unsigned short *cell_mem;
    int *bins;
    int *status;
    int chain, n, j0, m, op;  // op: 0 propose, 1 propose + Metropolis + commit
    int want_rows;            // moves: the proposed rows are wanted
    int n_chains;             // chains of the context (status words)
    const double *in;         // normals ((m-1) x dim) or displacement (dim)
    double u;
    double *out;              // r' then the four weights, the accept flag and the first chain whose
                              // status is set (-1: none)
    double *work;             // scratch of moves whose rows and link terms exceed kHookLds
    double *part;             // energy, adjoint: partial sums [block][kHookSums]
    int use_cells;
    const int *next;          // the chain's permutation (next[p] follows p across slice M - 1)
};

// Workgroup of the hook kernels, and the lanes that share one neighbour sum.
// A hook call is one link or one ring: what bounds it is the chain of dependent
// loads (cell counts, members, beads) of each sum, so the links run side by side
// and, in FP64, eight lanes split each sum's candidates (the order of the sum
// then only moves its last bits).  FP32 sums keep the candidate order, one lane each.
constexpr int kHookThreads = 512;
constexpr size_t kHookLds = 64 * 1024; // moves whose scratch fits keep it in LDS
constexpr int kHookSums = 5;           // partial sums per block of the energy and adjoint kernels
template <typename T> constexpr int hook_lanes() { return sizeof(T) == 8 ? 8 : 1; }

// Scratch of one move: rows x dim beads, then the four terms of each link.
__host__ __device__ inline size_t hook_scratch(int rows, int links, int dim, int tsize)
{
    return align16((size_t)rows * dim * tsize) + (size_t)4 * links * sizeof(double);
}

template <typename T, int DIM> __device__ inline Cells hook_cells(const HookArgs &a, const ChainDev &ch)
{
    return Cells{a.cell_cnt + ch.cell_off, a.cell_mem + ch.mem_off, a.bins + ch.bin_off, ch.M,
                 ch.ncell, ch.cap, ch.nbins, ch.swaps > 0 ? a.next : nullptr};
}

// The pair sum of link j with particle n's beads there at pj, pj1, over the
// lanes of an aligned group of hook_lanes<T>() (lane g of it): every lane gets it.
template <typename T, int DIM, bool CELLS, typename PathT>
__device__ inline T hook_link(const PathT &path, const Cells &C, const ChainDev &ch, const Prm<T> &P, int n,
                              int j, const T *pj, const T *pj1, int g)
{
    if (ch.pair == kPairNone) return T(0);
    constexpr int G = hook_lanes<T>();
    const T x = link_part<T, DIM, CELLS>(path, C, ch.N, ch.nbins, P, n, j, pj, pj1, g, G);
    return G > 1 ? group_sum_dpp(x, G) : x;
}

// The end of a single move: the link terms of every link t of the move's nl
// links from slice j0 (old beads in the path, new beads row(t), row(t + 1)),
// their sums in link order, the Metropolis test, and the commit of the first
// nput rows.  Terms of a link by a group of lanes per (link, old or new); the
// four sums by one thread each.  out: four weights, accept flag, status.
template <typename T, int DIM, bool CELLS, typename PathT, typename Row>
__device__ inline void hook_finish(const HookArgs &a, const ChainDev &ch, const Prm<T> &P, const PathT &path,
                                   const Cells &C, int j0, int nl, int nput, double *terms, double *w, Row row)
{
    __shared__ double s_w[4];
    __shared__ int s_bad, s_acc;
    const int M = ch.M, n = a.n, tid = threadIdx.x, nt = blockDim.x;
    constexpr int G = hook_lanes<T>();
    const int g = tid & (G - 1);
    for (int it = tid / G; it < 2 * nl; it += nt / G) {
        const int t = it >> 1, upd = it & 1;
        const int j = (j0 + t) % M, jn = (j + 1) % M;
        T x0[DIM], x1[DIM];
        if (upd) {
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                x0[e] = row(t)[e];
                x1[e] = row(t + 1)[e];
            }
        } else {
            path.get(n, j, x0);
            path.get(n, jn, x1);
        }
        const T wu = hook_link<T, DIM, CELLS>(path, C, ch, P, n, j, x0, x1, g);
        if (g == 0) {
            terms[upd * nl + t] = (double)((T(-0.5) * P.tau) * (potV<T, DIM>(x0, P) + potV<T, DIM>(x1, P)));
            terms[(2 + upd) * nl + t] = (double)wu;
        }
    }
    if (tid == 0) s_bad = 0x7fffffff;
    __syncthreads();
    if (tid < 4) {
        double s = 0.0;
        const double *x = terms + tid * nl;
#pragma unroll 8
        for (int t = 0; t < nl; ++t) s += x[t];
        s_w[tid] = s;
    }
    __syncthreads();
    if (tid == 0) {
        int acc = 0;
        if (a.op == 1) {
            T lw = (T)(s_w[1] - s_w[0]);
            if (ch.pair != kPairNone && ch.pair_in_accept) lw += (T)(s_w[3] - s_w[2]);
            acc = metropolis(ex(lw), (T)a.u) ? 1 : 0;
        }
        s_acc = acc;
        for (int k = 0; k < 4; ++k) w[k] = s_w[k];
        w[4] = (double)acc;
    }
    __syncthreads();
    if (s_acc) {
        // distinct slices: one thread per slice files its bead
        for (int t = tid; t < nput; t += nt) {
            const int j = (j0 + t) % M;
            path.put(n, j, row(t));
            if (CELLS && !cells_move<T, DIM>(C, P, n, j, row(t))) atomicOr(a.status + a.chain, 1);
        }
    }
    __syncthreads();
    for (int i = tid; i < a.n_chains; i += nt)
        if (a.status[i]) atomicMin(&s_bad, i);
    __syncthreads();
    if (tid == 0) w[5] = s_bad == 0x7fffffff ? -1.0 : (double)s_bad;
}

// ReshapeLinear on particle n, start slice j0, m links (src/updates/
// reshape.jl:31-91): the bridge of levy! with the injected normals, then the
// link sums w_initial / w_updated of the potential and pair actions.  One
// workgroup: the normals (host memory) are fetched together, one thread runs the
// recursion, the links follow side by side (hook_finish).  What bounds it is the
// latency of the launch and of the dependent loads: N = 256, M = 128, Gaussian
// pair, cell lists, FP64, a move of either kind with its share of an energy and a
// density every ten moves took 2.2 ms with one thread per move and takes 67 us.
template <typename T, int DIM, bool CELLS, bool SM>
__global__ void __launch_bounds__(kHookThreads) k_hook_reshape(HookArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const ChainDev ch = a.chains[a.chain];
    const Prm<T> P = Prm<T>::make(ch);
    const int M = ch.M, m = a.m, n = a.n, j0 = a.j0, nrows = m + 1, tid = threadIdx.x, nt = blockDim.x;
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const Cells C = hook_cells<T, DIM>(a, ch);
    unsigned char *const scratch = a.work ? reinterpret_cast<unsigned char *>(a.work) : smem;
    T *rp = reinterpret_cast<T *>(scratch); // (m+1) x DIM, row-major per bead
    double *terms = reinterpret_cast<double *>(scratch + align16((size_t)nrows * DIM * sizeof(T)));
    for (int i = tid; i < (m - 1) * DIM; i += nt) terms[i] = a.in[i]; // room of 4 m terms
    __syncthreads();
    if (tid == 0) {
        const int jm = (j0 + m) % M;
        T e0[DIM], em[DIM];
        path.get(n, j0, e0);
        path.get(n, jm, em);
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            em[e] = shift_end(e0[e], em[e], P);
            rp[0 * DIM + e] = teleport(e0[e], P);
            rp[m * DIM + e] = teleport(em[e], P);
        }
        T cur[DIM];
#pragma unroll
        for (int e = 0; e < DIM; ++e) cur[e] = e0[e];
        for (int i = 1; i < m; ++i) {
            const T alpha = bridge_alpha<T>(m, i);
            const T sd = bridge_sd(alpha, P);
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                cur[e] = bridge_step(cur[e], em[e], alpha, (T)terms[(i - 1) * DIM + e], sd);
                rp[i * DIM + e] = teleport(cur[e], P);
            }
        }
    }
    __syncthreads();
    if (a.want_rows)
        for (int i = tid; i < nrows * DIM; i += nt) a.out[(i % DIM) * nrows + i / DIM] = (double)rp[i];
    // rows 0..m-1 are written back, the start bead as teleported (src/updates/reshape.jl:82-86)
    hook_finish<T, DIM, CELLS>(a, ch, P, path, C, j0, m, m, terms, a.out + nrows * DIM,
                               [&](int t) { return rp + t * DIM; });
}

// SingleCenterOfMass with displacement in[0..dim) (src/updates/com.jl:136-224).
template <typename T, int DIM, bool CELLS, bool SM>
__global__ void __launch_bounds__(kHookThreads) k_hook_com(HookArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const ChainDev ch = a.chains[a.chain];
    const Prm<T> P = Prm<T>::make(ch);
    const int M = ch.M, n = a.n, tid = threadIdx.x, nt = blockDim.x;
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const Cells C = hook_cells<T, DIM>(a, ch);
    unsigned char *const scratch = a.work ? reinterpret_cast<unsigned char *>(a.work) : smem;
    T *rp = reinterpret_cast<T *>(scratch); // M x DIM row-major
    double *terms = reinterpret_cast<double *>(scratch + align16((size_t)M * DIM * sizeof(T)));
    T d[DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) d[e] = (T)a.in[e];
    for (int j = tid; j < M; j += nt)
#pragma unroll
        for (int e = 0; e < DIM; ++e) rp[j * DIM + e] = teleport(path.at(n, e, j) + d[e], P);
    __syncthreads();
    if (a.want_rows)
        for (int i = tid; i < M * DIM; i += nt) a.out[(i % DIM) * M + i / DIM] = (double)rp[i];
    hook_finish<T, DIM, CELLS>(a, ch, P, path, C, 0, M, M, terms, a.out + M * DIM,
                               [&](int t) { return rp + (t == M ? 0 : t) * DIM; });
}

// Rows (particle, coordinate) k0 .. k0 + nk - 1 of a chain's paths as the caller
// has them, M beads each, into host memory: grid (slice tiles, row tiles),
// 256 threads.  The turn of slice-major paths goes through LDS here; on the host it
// was bound by the strided side of the turn (N = 2000, M = 64, FP32, the whole call: 511 us from the
// pinned copy, 116 us from a pageable one, 80 us so; FP64 448, 284 and 116 us).
constexpr int kRowTileK = 32, kRowTileM = 64;
template <typename T>
__global__ void __launch_bounds__(256) k_read_rows(const T *pos, int rows, int M, int sm, int k0, int nk, T *out)
{
    __shared__ T tile[kRowTileK][kRowTileM + 1];
    const int t = threadIdx.x, kb = blockIdx.y * kRowTileK, jb = blockIdx.x * kRowTileM;
    if (sm) {
        const int k = kb + t % kRowTileK;
        for (int q = t / kRowTileK; q < kRowTileM; q += 256 / kRowTileK)
            if (k < nk && jb + q < M) tile[t % kRowTileK][q] = pos[(size_t)(jb + q) * rows + k0 + k];
        __syncthreads();
    }
    const int j = jb + t % kRowTileM;
    for (int q = t / kRowTileM; q < kRowTileK; q += 256 / kRowTileM)
        if (kb + q < nk && j < M)
            out[(size_t)(kb + q) * M + j] = (sm ? tile[q][t % kRowTileM] : pos[(size_t)(k0 + kb + q) * M + j]);
}

// interaction_action! value for particle n at slice j (src/updates/helper.jl:306-324)
template <typename T, int DIM, bool CELLS, bool SM> __global__ void k_hook_interaction(HookArgs a)
{
    constexpr int G = hook_lanes<T>();
    if (threadIdx.x >= G || blockIdx.x != 0) return;
    const ChainDev ch = a.chains[a.chain];
    const Prm<T> P = Prm<T>::make(ch);
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const Cells C = hook_cells<T, DIM>(a, ch);
    T r0[DIM], r1[DIM];
    path.get(a.n, a.j0, r0);
    path.get(a.n, (a.j0 + 1) % ch.M, r1);
    const T x = hook_link<T, DIM, CELLS>(path, C, ch, P, a.n, a.j0, r0, r1, (int)threadIdx.x);
    if (threadIdx.x == 0) a.out[0] = (double)x;
}

// Bead b of a chain as (particle i, slice j): consecutive threads take
// consecutive addresses (the particles of a slice in the slice-major layout,
// the slices of a ring otherwise).
template <bool SM> __device__ __forceinline__ void hook_bead(int b, int N, int M, int &i, int &j)
{
    if (SM) {
        j = b / N;
        i = b - j * N;
    } else {
        i = b / M;
        j = b - i * M;
    }
}

// The sum of each partial over the blocks, in every thread's v[] (one workgroup).
template <int NV> __device__ inline void hook_fold(const double *part, int nblk, double (&v)[NV], double *buf)
{
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double x = 0.0;
        for (int b = threadIdx.x; b < nblk; b += blockDim.x) x += part[(size_t)b * kHookSums + k];
        v[k] = block_sum(x, buf);
    }
}

// Energy (src/measurement.jl:92-122) plus the pair energy.  Beads (with a pair
// action in groups of 8 lanes that split the neighbours) spread over the grid,
// FP64 partial sums per block, folded by k_hook_energy_fold.  It is bound by the
// latency of the neighbour loads: N = 64, M = 256 FP64 all-pairs, an energy and an
// adjoint call with their copies took 5.9 ms with one workgroup for the energy and
// one thread per bead for the gradient, 93 us so.
template <typename T, int DIM, bool CELLS, bool SM> __global__ void __launch_bounds__(256) k_hook_energy(HookArgs a)
{
    __shared__ double buf[16];
    const ChainDev ch = a.chains[a.chain];
    const Prm<T> P = Prm<T>::make(ch);
    const int N = ch.N, M = ch.M;
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const Cells C = hook_cells<T, DIM>(a, ch);
    const double inv_s2 = (ch.pair == kPairGaussian) ? 1.0 / (ch.sigma * ch.sigma) : 0.0;
    const int G = ch.pair == kPairGaussian ? 8 : 1, lg = threadIdx.x & (G - 1);
    const int ngroups = (int)(gridDim.x * blockDim.x) / G;
    double link = 0.0, pot = 0.0, vkin = 0.0, su = 0.0, rgp = 0.0;
    for (int b = (int)(blockIdx.x * blockDim.x + threadIdx.x) / G; b < N * M; b += ngroups) {
        int i, j;
        hook_bead<SM>(b, N, M, i, j);
        if (ch.pair == kPairGaussian) { // no pair energy for the tabulated propagator
            double x, y;
            pair_energy_bead<T, DIM, CELLS>(path, C, N, ch.nbins, P, inv_s2, i, j, x, y, lg, G);
            su += x;
            rgp += y;
        }
        if (lg != 0) continue;
        const int jn = (j + 1 == M) ? 0 : j + 1;
        T r0[DIM], r1[DIM];
        path.get(i, j, r0);
        path.get(jn == 0 ? a.next[i] : i, jn, r1); // inext of src/measurement.jl:98
        T dd = T(0);
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            const T dx = mindist(r0[e], r1[e], P);
            dd += dx * dx;
        }
        link += (double)dd;
        pot += (double)(potV<T, DIM>(r0, P) + potV<T, DIM>(r1, P));
        vkin += (double)rgradV<T, DIM>(r0, P);
    }
    double v[kHookSums] = {link, pot, vkin, su, rgp};
#pragma unroll
    for (int k = 0; k < kHookSums; ++k) v[k] = block_sum(v[k], buf);
    if (threadIdx.x == 0)
        for (int k = 0; k < kHookSums; ++k) a.part[(size_t)blockIdx.x * kHookSums + k] = v[k];
}

static __global__ void __launch_bounds__(256) k_hook_energy_fold(HookArgs a, int nblk)
{
    __shared__ double buf[16];
    double v[kHookSums];
    hook_fold(a.part, nblk, v, buf);
    if (threadIdx.x == 0) {
        const ChainDev &ch = a.chains[a.chain];
        const double tau = ch.tau, link = v[0], pot = v[1], vkin = v[2], su = v[3], rgp = v[4];
        const int M = ch.M;
        a.out[0] = ((double)(ch.dim * ch.N) / (2.0 * tau) - (1.0 / (((4.0 * ch.lambda) * (tau * tau)) * M)) * link) +
                   (1.0 / (2.0 * M)) * pot;
        a.out[1] = (1.0 / (2.0 * M)) * vkin + (1.0 / (2.0 * M)) * pot;
        a.out[2] = ch.g * su / ch.beta;
        a.out[3] = ch.g * (su / ch.beta + rgp / (2.0 * ch.beta));
    }
}

// Density (src/measurement.jl:45-55): counts into a uint64 histogram.
template <typename T, int DIM, bool SM> __global__ void k_hook_density(HookArgs a, int nbins, unsigned long long *hist)
{
    const ChainDev ch = a.chains[a.chain];
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const double bw = (2.0 * ch.L) / nbins;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < ch.N * ch.M; b += gridDim.x * blockDim.x) {
        const int i = b / ch.M, j = b - i * ch.M;
        long long idx = 0, stride = 1;
        bool ok = true;
        for (int e = 0; e < DIM; ++e) {
            const long long ib = (long long)floor(((double)path.at(i, e, j) + ch.L) / bw);
            ok = ok && ib > 0 && ib < nbins + 1;
            idx += (ib - 1) * stride;
            stride *= nbins;
        }
        if (ok) atomicAdd(&hist[idx], 1ull);
    }
}

// Adjoint of S_pot = tau sum_beads V + S_U with
// S_U = sum_links sum_{pairs within h at slice j} tau/2 (v(r_j) + v(r_j+1)).
// dS/dr of bead (n, j) collects tau grad V and the pair terms of links j
// (neighbour set at slice j) and j-1 (set at slice j-1); distances are
// recomputed, nothing is stored.  hook_lanes<T>() lanes per bead split its
// neighbours (FP32: one lane, in order), beads spread over the grid; partial
// sums per block give S_pot, dS/domega and dS/dg (k_hook_adjoint_fold).
template <typename T, int DIM, bool CELLS, bool SM> __global__ void __launch_bounds__(256) k_hook_adjoint(HookArgs a)
{
    __shared__ double buf[16];
    const ChainDev ch = a.chains[a.chain];
    const Prm<T> P = Prm<T>::make(ch);
    const int N = ch.N, M = ch.M;
    const Path<T, DIM, SM> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    const Cells C = hook_cells<T, DIM>(a, ch);
    const T inv_s2 = (ch.pair != kPairNone) ? T(1.0 / (ch.sigma * ch.sigma)) : T(0);
    const T ht = T(0.5) * P.tau;
    constexpr int GL = hook_lanes<T>();
    const int G = ch.pair != kPairNone ? GL : 1, lg = threadIdx.x & (G - 1);
    const int ngroups = (int)(gridDim.x * blockDim.x) / G;
    double S = 0.0, Sw = 0.0, SU = 0.0;
    for (int b = (int)(blockIdx.x * blockDim.x + threadIdx.x) / G; b < N * M; b += ngroups) {
        int n, j;
        hook_bead<SM>(b, N, M, n, j);
        const int jp = (j == 0) ? M - 1 : j - 1;
        T r[DIM], g[DIM];
        path.get(n, j, r);
#pragma unroll
        for (int e = 0; e < DIM; ++e) g[e] = T(0);
        if (lg == 0) {
            gradV<T, DIM>(r, P, g);
#pragma unroll
            for (int e = 0; e < DIM; ++e) g[e] *= P.tau;
            S += (double)(P.tau * potV<T, DIM>(r, P));
            if (ch.pot == kPotHarmonic) Sw += (double)(P.tau * dVdomega<T, DIM>(r, ch.omega));
        }
        if (ch.pair != kPairNone) {
            // link j: the neighbour set at slice j around bead (n, j); link j-1: the set at slice j-1
            for (int side = 0; side < 2; ++side) {
                const int js = side == 0 ? j : jp;
                T rs[DIM];
                path.get(n, js, rs);
                auto visit = [&](int k, int mult) {
                    T rk[DIM];
                    path.get(k, js, rk);
                    T d0 = mindist(rk[0], rs[0], P);
                    T r2 = d0 * d0;
                    if (DIM > 1) {
                        T d1 = mindist(rk[1], rs[1], P);
                        r2 += d1 * d1;
                    }
                    if (r2 > P.h2) return;
                    // gradient at slice j of v(|r_n^j - r_k^j|), signed minimum image
                    T rkj[DIM], x[DIM];
                    path.get(k, j, rkj);
                    T x2 = T(0);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) {
                        T dx = r[e] - rkj[e];
                        dx -= P.twoL * fl(dx * P.inv2L + T(0.5));
                        x[e] = dx;
                        x2 += dx * dx;
                    }
                    const T v = P.g * ex(-x2 * P.inv2s2);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) g[e] += T(mult) * ht * (-(x[e] * inv_s2) * v);
                    if (side == 0) {
                        // S_U: each unordered pair of link j counted once (half from each end)
                        const int jn = (j + 1 == M) ? 0 : j + 1;
                        T rkn[DIM], rnn[DIM];
                        path.get(k, jn, rkn);
                        path.get(n, jn, rnn);
                        T e0 = mindist(rkn[0], rnn[0], P);
                        T s2 = e0 * e0;
                        if (DIM > 1) {
                            T e1 = mindist(rkn[1], rnn[1], P);
                            s2 += e1 * e1;
                        }
                        // per unit coupling: S_U = g * SU, dS/dg = SU
                        SU += 0.5 * (double)(T(mult) * ht * (ex(-r2 * P.inv2s2) + ex(-s2 * P.inv2s2)));
                    }
                };
                constexpr int NS = (DIM == 1) ? 3 : 9;
                if (CELLS) {
                    const int c0 = cell_of<T, DIM>(rs, P, C.nbins);
                    int at = lg; // this lane's next candidate, counted through the stencil's lists
                    for (int s = 0; s < NS; ++s) {
                        const int cc = stencil_cell(c0, s, C.nbins, DIM);
                        const int cnt = C.count(js, cc);
                        const unsigned short *mem = C.members(js, cc);
                        for (; at < cnt; at += G)
                            if (mem[at] != n) visit(mem[at], 1);
                        at -= cnt;
                    }
                } else {
                    const int c0 = (ch.nbins < 3) ? cell_of<T, DIM>(rs, P, ch.nbins) : 0;
                    for (int k = lg; k < N; k += G) {
                        if (k == n) continue;
                        int mult = 1;
                        if (ch.nbins < 3) {
                            T rk[DIM];
                            path.get(k, js, rk);
                            const int ck = cell_of<T, DIM>(rk, P, ch.nbins);
                            mult = 0;
                            for (int s = 0; s < NS; ++s) mult += (stencil_cell(c0, s, ch.nbins, DIM) == ck);
                            if (!mult) continue;
                        }
                        visit(k, mult);
                    }
                }
            }
            if (G > 1) {
#pragma unroll
                for (int e = 0; e < DIM; ++e) g[e] = group_sum_dpp(g[e], G);
            }
        }
        if (lg == 0)
            for (int e = 0; e < DIM; ++e) a.out[((size_t)n * DIM + e) * M + j] = (double)g[e];
    }
    double v[3] = {S, Sw, SU};
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = block_sum(v[k], buf);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) a.part[(size_t)blockIdx.x * kHookSums + k] = v[k];
}

// out[0..3): S_pot, dS/d omega, dS/d g.
static __global__ void __launch_bounds__(256) k_hook_adjoint_fold(HookArgs a, int nblk)
{
    __shared__ double buf[16];
    double v[3];
    hook_fold(a.part, nblk, v, buf);
    if (threadIdx.x == 0) {
        a.out[0] = v[0] + a.chains[a.chain].g * v[2]; // S_pot
        a.out[1] = v[1];                              // dS/d omega
        a.out[2] = v[2];                              // dS/d g
    }
}

// init_world (src/system.jl:36-78) with a = 0: each particle's first bead
// uniform in [-L, L)^dim, the last bead equal to it, and levy! over the M - 1
// links in between (the bridge arithmetic of levy_segment, teleport of every
// row).  One thread per particle, FP64 arithmetic, stored in the chain's
// layout; Philox purposes kInitStart and kInitLevy, sweep word 0.
template <typename T, int DIM>
__global__ void k_init_paths(const ChainDev *chains, const int *part_chain, const int *part_idx, int q0, int nq,
                             void *pos, uint64_t seed)
{
    const int gq = q0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gq >= q0 + nq) return;
    const int c = part_chain[gq], p = part_idx[gq];
    const ChainDev ch = chains[c];
    const Prm<double> P = Prm<double>::make(ch);
    const int M = ch.M, N = ch.N;
    T *base = reinterpret_cast<T *>(pos) + ch.pos_off;
    auto put = [&](int j, int d, double v) {
        T x = (T)v;
        if (x >= (T)ch.L) x = nextafter((T)ch.L, (T)(-ch.L)); // keep [-L, L) after rounding to T
        if (ch.sm) base[((size_t)j * N + p) * DIM + d] = x;
        else base[((size_t)p * DIM + d) * M + j] = x;
    };
    U4 x = draw(seed, (uint32_t)p, 0u, (uint32_t)c, kInitStart);
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
    double r0[DIM], cur[DIM], em[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        r0[d] = 2.0 * ch.L * (u01d(w[d]) - 0.5);
        cur[d] = r0[d];
        em[d] = shift_end(r0[d], r0[d], P); // the ends coincide: no shift
    }
    const int K = M - 1; // links of the bridge
    for (int i = 1; i < K; ++i) {
        if (i & 1) x = draw(seed, (uint32_t)(p * M + i), 0u, (uint32_t)c, kInitLevy);
        double n[2];
        if (i & 1) box_muller(x.x, x.y, n[0], n[1]);
        else box_muller(x.z, x.w, n[0], n[1]);
        const double alpha = bridge_alpha<double>(K, i);
        const double sd = bridge_sd(alpha, P);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            cur[d] = bridge_step(cur[d], em[d], alpha, n[d], sd);
            put(i, d, teleport(cur[d], P));
        }
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        put(0, d, teleport(r0[d], P));
        put(M - 1, d, teleport(em[d], P));
    }
}

// init_world (src/system.jl:36-78) with hard spheres of radius a = hs_a > 0:
// one workgroup per listed chain, particles in order.  Try t of particle p is
// k_init_paths's path with sweep word t (thread 0 runs the bridge into LDS in
// FP64); the workgroup then tests every slice against the earlier particles'
// beads (FP64 copies in hs64, N x M x DIM per chain at its position offset):
// a bead closer than a (norm of the per-component |minimum-image| offsets)
// rejects the try.  At most 10 000 tries per particle, else status bit 4 and
// the chain's remaining particles keep their old paths.
template <typename T, int DIM>
__global__ void __launch_bounds__(256) k_init_paths_hs(const ChainDev *chains, const int *ids, int n, void *pos,
                                                       double *hs64, uint64_t seed, int *status)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if ((int)blockIdx.x >= n) return;
    const int c = ids[blockIdx.x], tid = threadIdx.x, nt = blockDim.x;
    const ChainDev ch = chains[c];
    const Prm<double> P = Prm<double>::make(ch);
    const int M = ch.M, N = ch.N;
    const double a = ch.hs_a;
    double *cand = reinterpret_cast<double *>(smem); // [M][DIM]
    int *flag = reinterpret_cast<int *>(cand + (size_t)M * DIM);
    double *done = hs64 + ch.pos_off;                // [p][j][d] of the placed particles
    T *base = reinterpret_cast<T *>(pos) + ch.pos_off;
    for (int p = 0; p < N; ++p) {
        uint32_t t = 0;
        for (;; ++t) {
            if (t >= 10000u) {
                if (tid == 0) atomicOr(status + c, 4);
                return; // uniform: every thread reads the same flags
            }
            if (tid == 0) {
                U4 x = draw(seed, (uint32_t)p, t, (uint32_t)c, kInitStart);
                const uint32_t w[4] = {x.x, x.y, x.z, x.w};
                double r0[DIM], cur[DIM], em[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    r0[d] = 2.0 * ch.L * (u01d(w[d]) - 0.5);
                    cur[d] = r0[d];
                    em[d] = shift_end(r0[d], r0[d], P);
                }
                const int K = M - 1;
                for (int i = 1; i < K; ++i) {
                    if (i & 1) x = draw(seed, (uint32_t)(p * M + i), t, (uint32_t)c, kInitLevy);
                    double nn[2];
                    if (i & 1) box_muller(x.x, x.y, nn[0], nn[1]);
                    else box_muller(x.z, x.w, nn[0], nn[1]);
                    const double alpha = bridge_alpha<double>(K, i);
                    const double sd = bridge_sd(alpha, P);
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        cur[d] = bridge_step(cur[d], em[d], alpha, nn[d], sd);
                        cand[i * DIM + d] = teleport(cur[d], P);
                    }
                }
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    cand[d] = teleport(r0[d], P);
                    cand[(M - 1) * DIM + d] = teleport(em[d], P);
                }
                *flag = 0;
            }
            __syncthreads();
            for (int it = tid; it < p * M; it += nt) {
                const int i = it / M, j = it - i * M;
                double d2 = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    const double dd = mindist(done[((size_t)i * M + j) * DIM + d], cand[j * DIM + d], P);
                    d2 += dd * dd;
                }
                if (sqrt(d2) < a) *flag = 1;
            }
            __syncthreads();
            const bool clash = *flag != 0;
            __syncthreads();
            if (!clash) break;
        }
        for (int it = tid; it < M * DIM; it += nt) {
            const int j = it / DIM, d = it - j * DIM;
            const double v = cand[it];
            done[((size_t)p * M + j) * DIM + d] = v;
            T x = (T)v;
            if (x >= (T)ch.L) x = nextafter((T)ch.L, (T)(-ch.L)); // keep [-L, L) after rounding to T
            if (ch.sm) base[((size_t)j * N + p) * DIM + d] = x;
            else base[((size_t)p * DIM + d) * M + j] = x;
        }
        __syncthreads();
    }
}

// The batched kernel's FP32 fast paths on one particle of a tile chain whose
// staging length ell = MAXL divides M (every segment and centre-of-mass chunk
// is one skew block of the LDS rows): the particle's ring is staged into LDS
// in the tile kernel's row layout, and one wave runs the same device code as
// k_sweep_tiles with the caller's draws.  Staging (m = MAXL links from j0):
// levy_full_propose with the injected normals; centre of mass: com_chunk_full
// per chunk, summed by the lane-group butterfly when the chunks form an
// aligned lane group (nseg a power of two <= 64), else in chunk order.  The
// outputs follow k_hook_reshape / k_hook_com, with the log-weight change in
// w[1] (w[0] = 0: the fast paths form the difference directly).
template <int DIM, int MAXL, int POT> __global__ void __launch_bounds__(64) k_hook_tile_fast(HookArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const ChainDev ch = a.chains[a.chain];
    const Prm<float> P = Prm<float>::make(ch);
    const int M = ch.M, n = a.n, lane = threadIdx.x;
    int sh = 0;
    while ((2 << sh) <= MAXL) ++sh;
    const LdsRow R{tile_row_len(M, sh), sh};
    float *sp = reinterpret_cast<float *>(smem);
    float *s_red = sp + DIM * R.Mp; // nseg chunk sums, then nseg wrap flags
    float *s_wr = s_red + M / MAXL;
    __shared__ float s_tot;
    float *gp = reinterpret_cast<float *>(a.pos) + ch.pos_off + (size_t)n * DIM * M;
    for (int i = lane; i < DIM * M; i += 64) {
        const int d = i / M, j = i - d * M;
        sp[R.at(d, j)] = gp[i];
    }
    __shared__ double s_in[(MAXL - 1) * DIM];
    if (a.m > 0)
        for (int i = lane; i < (MAXL - 1) * DIM; i += 64) s_in[i] = a.in[i];
    int bad = 0x7fffffff; // first chain whose status is set
    for (int i = lane; i < a.n_chains; i += 64)
        if (a.status[i]) bad = min(bad, i);
    for (int off = 32; off >= 1; off >>= 1) bad = min(bad, __shfl_xor(bad, off, 64));
    const double status = bad == 0x7fffffff ? -1.0 : (double)bad;
    __syncthreads();
    double *w = nullptr;
    if (a.m > 0) { // staging segment
        const int j0 = a.j0, nrows = MAXL + 1;
        w = a.out + nrows * DIM;
        if (lane == 0) {
            float nb[MAXL - 1][DIM];
            GivenNormals<DIM> ns{s_in};
            const float lw = levy_full_propose<DIM, MAXL, POT>(sp, R, M, j0, P, ns, nb);
            const int jm = (j0 + MAXL) % M;
            if (a.want_rows)
                for (int e = 0; e < DIM; ++e) {
                    a.out[e * nrows] = (double)sp[R.at(e, j0)];
                    a.out[e * nrows + MAXL] = (double)sp[R.at(e, jm)];
                    for (int i = 1; i < MAXL; ++i) a.out[e * nrows + i] = (double)nb[i - 1][e];
                }
            w[0] = 0.0;
            w[1] = (double)lw;
            w[2] = w[3] = 0.0;
            const bool acc = a.op == 1 && metropolis(ex(lw), (float)a.u);
            w[4] = acc ? 1.0 : 0.0;
            w[5] = status;
            if (acc) {
                for (int i = 1; i < MAXL; ++i) {
                    const int j = (j0 + i) % M;
                    for (int e = 0; e < DIM; ++e) gp[e * M + j] = nb[i - 1][e];
                }
            }
        }
        return;
    }
    // centre of mass: chunk k = lane (every lane takes part in the butterfly)
    const int nseg = M / MAXL;
    float d[DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) d[e] = (float)a.in[e];
    w = a.out + M * DIM;
    const bool grouped = nseg <= 64 && (nseg & (nseg - 1)) == 0;
    for (int k0 = 0; k0 < nseg; k0 += 64) {
        const int k = k0 + lane;
        bool wr = false;
        float v = 0.0f;
        if (k < nseg) {
            v = com_chunk_full<DIM, MAXL, POT>(sp + k * (MAXL + 1), R, d, P, wr);
            s_red[k] = v;
            s_wr[k] = wr ? 1.0f : 0.0f;
        }
        if (grouped) {
            const float tot = group_sum_dpp(v, nseg);
            if (lane == 0) s_red[0] = tot;
        }
    }
    __syncthreads();
    if (lane == 0) {
        float tot = s_red[0];
        if (!grouped) {
            tot = 0.0f;
            for (int k = 0; k < nseg; ++k) tot += s_red[k];
        }
        s_tot = tot;
    }
    __syncthreads();
    const float lw = -P.tau * s_tot;
    const bool acc = a.op == 1 && metropolis(ex(lw), (float)a.u);
    for (int i = lane; i < DIM * M; i += 64) { // the moved beads
        const int e = i / M, j = i - e * M;
        const float x0 = sp[R.at(e, j)], x = s_wr[j / MAXL] != 0.0f ? teleport(x0 + d[e], P) : x0 + d[e];
        if (a.want_rows) a.out[i] = (double)x;
        if (acc) gp[i] = x;
    }
    if (lane == 0) {
        w[0] = 0.0;
        w[1] = (double)lw;
        w[2] = w[3] = 0.0;
        w[4] = acc ? 1.0 : 0.0;
        w[5] = status;
    }
}

} // namespace pimc
