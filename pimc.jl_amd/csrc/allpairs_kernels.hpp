// Sweep kernel of small chains with a Gaussian pair action: every particle
// interacts with every other one (no cell lists) and the path fits in LDS.
//
// The schedule is k_sweep_whole's, one particle after another.  What bounds a
// particle's step is its pair sum over all links and all other particles, which
// is vector arithmetic: a periodic distance and an exponential per bead pair.  A
// link's term needs the pair potential at both of its slices, and the next link
// needs the second one again; here a lane owns a slice, evaluates each bead pair
// of it once, and takes the next slice's value from the neighbouring lane (a
// wavefront shift), so one exponential per bead pair is left of two.  A wave takes
// 64 consecutive slices against every G-th particle; the path is particle-major
// in LDS, so its lanes read consecutive addresses.  The order of every sum is
// k_sweep_whole's.
//
// A particle's bridge needs only its own end beads, which no staging move
// writes, so it is built while the previous particle is decided: two barriers a
// particle instead of five.
//
// 512 chains of N = 64, M = 256, FP32, 16 measuring sweeps: 67.5 ms on
// k_sweep_whole, 46.5 ms here, 36.6 ms with the estimators of k_meas_allpairs.
#pragma once
#include "sweep_kernels.hpp"
#include "window_kernels.hpp"

namespace pimc {

constexpr int kAllPairsThreads = 1024, kAllPairsMaxM = 512;

// One particle's row in LDS: M beads, padded by one so that lanes which walk the
// particles of a slice hit distinct banks.
__host__ __device__ inline size_t allpairs_row(int M, int dim) { return (size_t)(M + 1) * dim; }

struct AllPairsLds {
    size_t path, nb[2], nrm, dvb, du, wsum, end;
};
__host__ __device__ inline AllPairsLds allpairs_lds(int N, int M, int dim, int tsize, int G)
{
    AllPairsLds L;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o = align16(o + bytes);
        return at;
    };
    L.path = take((size_t)N * allpairs_row(M, dim) * tsize);
    L.nb[0] = take((size_t)M * dim * tsize);
    L.nb[1] = take((size_t)M * dim * tsize);
    L.nrm = take((size_t)M * dim * tsize);
    L.dvb = take((size_t)M * tsize);
    L.du = take((size_t)G * M * tsize);
    L.wsum = take(32 * sizeof(double));
    L.end = o;
    return L;
}

// Particles a link's pair sum is split over: as many as the workgroup has waves
// for (k_sweep_whole's lanes per link).
inline int allpairs_groups(int maxM)
{
    int G = 1;
    while (G < 16 && 2 * G * maxM <= kAllPairsThreads) G <<= 1;
    return std::max(2, G);
}

template <typename T, int DIM> struct RowPath {
    T *base;
    int M, N, ld;
    __device__ __forceinline__ T *at(int n, int j) const { return base + (size_t)n * ld + (size_t)j * DIM; }
    __device__ __forceinline__ void get(int n, int j, T *r) const
    {
        const T *x = at(n, j);
#pragma unroll
        for (int e = 0; e < DIM; ++e) r[e] = x[e];
    }
    __device__ __forceinline__ void put(int n, int j, const T *r) const
    {
        T *x = at(n, j);
#pragma unroll
        for (int e = 0; e < DIM; ++e) x[e] = r[e];
    }
};

// The next lane's value; lane 63 gets `last`.
__device__ __forceinline__ float next_lane(float v, float last)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(last), __float_as_int(v), 0x130, 0xF, 0xF, false));
}
__device__ __forceinline__ double next_lane(double v, double last)
{
    const long long b = __double_as_longlong(v), o = __double_as_longlong(last);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, 0x130, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), 0x130, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Lane l's value in every lane (l uniform).
__device__ __forceinline__ float lane_value(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// acc - (in ? half_tau (g e0 + ge1) : 0): a link's pair_lnU added to a sum, from
// the exponential at its first slice and g times the one at its second.
template <typename T> __device__ __forceinline__ T sub_link(T acc, bool in, T half_tau, T g, T e0, T ge1)
{
#pragma clang fp contract(off)
    const T l = half_tau * fma_(g, e0, ge1);
    return in ? acc - l : acc;
}

// This lane's link (slice j, clamped to the ring for the lanes past it) of the
// pair sums of particle p with its beads at nw (new) and od (old): sum of the
// link's pair_lnU over the particles g, g + G, ... other than p, new minus old.
// The wave holds slices 64 jb .. 64 jb + last; nB, oB are the beads of the slice
// after its last one.
// FULL: last is 63.
template <typename T, int DIM, bool FULL>
__device__ __forceinline__ T link_delta_lanes(const RowPath<T, DIM> &path, const Prm<T> &P, int p, int j, int jB, int last,
                                            const T *nw, const T *od, const T *nB, const T *oB, int g, int G)
{
    const int lane = threadIdx.x & 63, N = path.N;
    const T ht = T(0.5) * P.tau;
    T an = T(0), ao = T(0);
    for (int k0 = g; k0 < N; k0 += 64 * G) {
        const int cnt = min(64, (N - k0 + G - 1) / G);
        // the slice after the wave's last: lane i takes particle k0 + i G
        T bn = T(0), bo = T(0);
        if (lane < cnt) {
            T r[DIM];
            path.get(k0 + lane * G, jB, r);
            bn = vpair_r2(dist2_min<T, DIM>(r, nB, P), P);
            bo = vpair_r2(dist2_min<T, DIM>(r, oB, P), P);
        }
        for (int i = 0; i < cnt; ++i) {
            const int k = k0 + i * G;
            if (k == p) continue; // uniform
            T r[DIM];
            path.get(k, j, r);
            const T dn = dist2_min<T, DIM>(r, nw, P), dd = dist2_min<T, DIM>(r, od, P);
            const T en = ex(-dn * P.inv2s2), eo = ex(-dd * P.inv2s2);
            const T gn = lane_value(bn, i), go = lane_value(bo, i);
            T n1 = next_lane(P.g * en, gn), o1 = next_lane(P.g * eo, go);
            if (!FULL) {
                n1 = lane == last ? gn : n1;
                o1 = lane == last ? go : o1;
            }
            an = sub_link(an, dn <= P.h2, ht, P.g, en, n1);
            ao = sub_link(ao, dd <= P.h2, ht, P.g, eo, o1);
        }
    }
    return sub_(an, ao);
}
template <typename T, int DIM>
__device__ __forceinline__ T link_delta_row(const RowPath<T, DIM> &path, const Prm<T> &P, int p, int j, int jB, int last,
                                            const T *nw, const T *od, const T *nB, const T *oB, int g, int G)
{
    return last == 63 ? link_delta_lanes<T, DIM, true>(path, P, p, j, jB, last, nw, od, nB, oB, g, G)
                      : link_delta_lanes<T, DIM, false>(path, P, p, j, jB, last, nw, od, nB, oB, g, G);
}

template <typename T, int DIM> __global__ void __launch_bounds__(kAllPairsThreads) k_sweep_allpairs(SweepArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double s_buf[16], s_q[kNQ];
    const int c = a.whole[blockIdx.x];
    const ChainDev ch = a.chains[c];
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, nwv = nt >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int N = ch.N, M = ch.M, ell = ch.ell, nseg = ch.nseg, G = a.link_group;
    const AllPairsLds L = allpairs_lds(N, M, DIM, (int)sizeof(T), G);
    T *const gpath = reinterpret_cast<T *>(a.pos) + ch.pos_off;
    const RowPath<T, DIM> path{reinterpret_cast<T *>(smem + L.path), M, N, (int)allpairs_row(M, DIM)};
    T *const s_nb0 = reinterpret_cast<T *>(smem + L.nb[0]), *const s_nb1 = reinterpret_cast<T *>(smem + L.nb[1]);
    T *const s_nrm = reinterpret_cast<T *>(smem + L.nrm);
    T *const s_dvb = reinterpret_cast<T *>(smem + L.dvb), *const s_du = reinterpret_cast<T *>(smem + L.du);
    double *const s_wsum = reinterpret_cast<double *>(smem + L.wsum);
    for (int i = tid; i < N * M; i += nt) {
        const int j = i / N, n = i - j * N;
        path.put(n, j, gpath + (size_t)i * DIM);
    }
    if (tid < kNQ) s_q[tid] = 0.0;
    const Cells none{nullptr, nullptr, nullptr, M, 0, 0, ch.nbins};
    const uint32_t sweep0 = a.rs->sweep + (uint32_t)a.sweep_off;
    int lacc = 0, cacc = 0, ctry = 0;
    int meas_in = (int)((uint32_t)a.measure_every - 1u - sweep0 % (uint32_t)a.measure_every);
    const int hp = ell >> 1; // Philox blocks per segment: interior bead pairs (i, i + 1), i odd
    // this wave's links: slices 64 jb .. 64 jb + last against the particles g, g + G, ...
    const int jblocks = (M + 63) / 64;
    const int g = wave % G, jb = wave / G;
    const bool links = jb < jblocks;
    const int j = min(64 * jb + lane, M - 1), last = min(63, M - 1 - 64 * jb), jB = (64 * jb + last + 1) % M;
    const bool own = links && 64 * jb + lane < M;
    __syncthreads();

    for (int s = 0; s < a.nsweeps; ++s) {
        const uint32_t sw = sweep0 + (uint32_t)s;
        const bool meas_now = a.measure && !a.split && meas_in == 0;
        meas_in = (meas_in == 0) ? a.measure_every - 1 : meas_in - 1;
        if (pass_on(ch.every_st, sw)) {
            const U4 xo = draw(a.seed, 0u, sw, (uint32_t)c, kOffset); // one offset per chain and sweep
            const int off = (int)(((uint64_t)xo.x * (uint64_t)ell) >> 32);
            // the segment of slice jj and the slice's place in it
            auto place = [&](int jj, int &k, int &t, int &m) {
                int rel = jj - off;
                if (rel < 0) rel += M;
                k = rel / ell;
                t = rel - k * ell;
                m = min(ell, M - k * ell);
            };
            auto normals = [&](int p) {
                for (int w = tid; w < nseg * hp; w += nt) {
                    const int k = w / hp, i = 2 * (w - k * hp) + 1;
                    const int m = min(ell, M - k * ell);
                    if (i < m) {
                        int b = off + k * ell + i;
                        if (b >= M) b -= M;
                        const U4 xr = draw(a.seed, (uint32_t)(p * M + b), sw, (uint32_t)c, kLevy);
                        T n0, n1;
                        box_muller(xr.x, xr.y, n0, n1);
                        s_nrm[b * DIM] = n0;
                        if (DIM > 1) s_nrm[b * DIM + DIM - 1] = n1;
                        if (i + 1 < m) {
                            const int b1 = (b + 1 == M) ? 0 : b + 1;
                            box_muller(xr.z, xr.w, n0, n1);
                            s_nrm[b1 * DIM] = n0;
                            if (DIM > 1) s_nrm[b1 * DIM + DIM - 1] = n1;
                        }
                    }
                }
            };
            auto bridges = [&](int p) { // by the last threads: the first ones decide meanwhile
                T *buf = (p & 1) ? s_nb1 : s_nb0;
                for (int k = nt - 1 - tid; k < nseg; k += nt) {
                    const int m = min(ell, M - k * ell);
                    if (m < 2) continue;
                    int start = off + k * ell;
                    if (start >= M) start -= M;
                    int jm = start + m;
                    if (jm >= M) jm -= M;
                    T cur[DIM], em[DIM];
                    path.get(p, start, cur);
                    path.get(p, jm, em);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) em[e] = shift_end(cur[e], em[e], P);
                    for (int i = 1; i < m; ++i) {
                        int b = start + i;
                        if (b >= M) b -= M;
                        const T alpha = bridge_alpha<T>(m, i);
                        const T sd = bridge_sd(alpha, P);
#pragma unroll
                        for (int e = 0; e < DIM; ++e) {
                            cur[e] = bridge_step(cur[e], em[e], alpha, s_nrm[b * DIM + e], sd);
                            buf[b * DIM + e] = teleport(cur[e], P);
                        }
                    }
                }
            };
            normals(0);
            __syncthreads();
            bridges(0);
            __syncthreads();
            int kj, tj, mj, kB, tB, mB;
            place(j, kj, tj, mj);
            place(jB, kB, tB, mB);
            for (int p = 0; p < N; ++p) {
                const T *buf = (p & 1) ? s_nb1 : s_nb0;
                if (links) {
                    T od[DIM], nw[DIM], oB[DIM], nB[DIM];
                    path.get(p, j, od);
                    path.get(p, jB, oB);
                    const bool in = tj >= 1 && mj >= 2, inB = tB >= 1 && mB >= 2; // interior: moved
#pragma unroll
                    for (int e = 0; e < DIM; ++e) {
                        nw[e] = in ? buf[j * DIM + e] : od[e];
                        nB[e] = inB ? buf[jB * DIM + e] : oB[e];
                    }
                    const T du = link_delta_row<T, DIM>(path, P, p, j, jB, last, nw, od, nB, oB, g, G);
                    if (own) {
                        s_du[(size_t)g * M + j] = du;
                        if (g == 0) s_dvb[j] = in ? potV<T, DIM>(nw, P) - potV<T, DIM>(od, P) : T(0);
                    }
                }
                if (p + 1 < N) normals(p + 1);
                __syncthreads();
                // decisions: every slice's thread takes its segment's sums, Delta V over the interior beads,
                // then the links, in order; and moves its bead
                for (int jj = tid; jj < M; jj += nt) {
                    int k, t, m;
                    place(jj, k, t, m);
                    if (m < 2 || t < 1) continue;
                    int start = off + k * ell;
                    if (start >= M) start -= M;
                    T dv = T(0);
                    for (int i = 1; i < m; ++i) {
                        int b = start + i;
                        if (b >= M) b -= M;
                        dv = add_(dv, s_dvb[b]);
                    }
                    T lw = -P.tau * dv;
                    for (int i = 0; i < m; ++i) {
                        int b = start + i;
                        if (b >= M) b -= M;
                        const T *x = s_du + b;
                        // the groups' shares by halves, as a lane butterfly adds them
                        T sum;
                        auto four = [&](int q) { return add_(add_(x[(size_t)q * M], x[(size_t)(q + 1) * M]),
                                                             add_(x[(size_t)(q + 2) * M], x[(size_t)(q + 3) * M])); };
                        if (G == 2) sum = add_(x[0], x[M]);
                        else if (G == 4) sum = four(0);
                        else if (G == 8) sum = add_(four(0), four(4));
                        else sum = add_(add_(four(0), four(4)), add_(four(8), four(12)));
                        lw = add_(lw, sum);
                    }
                    const U4 xa = draw(a.seed, (uint32_t)(p * M + start), sw, (uint32_t)c, kLevyAccept);
                    if (metropolis(ex(lw), Uniform<T>::get(xa.x))) {
                        path.put(p, jj, buf + jj * DIM);
                        lacc += t == 1 ? 1 : 0;
                    }
                }
                if (p + 1 < N) bridges(p + 1);
                __syncthreads();
            }
        }
        if (pass_on(ch.every_com, sw)) {
            for (int p = 0; p < N; ++p) {
                ctry += (tid == 0) ? 1 : 0;
                const U4 y = draw(a.seed, (uint32_t)p, sw, (uint32_t)c, kCom);
                const T step2 = (T)a.com_step[c] * T(2);
                T d[DIM];
                d[0] = step2 * (Uniform<T>::get(y.x) - T(0.5));
                if (DIM > 1) d[DIM - 1] = step2 * (Uniform<T>::get(y.y) - T(0.5));
                double x = 0.0;
                if (links) {
                    T od[DIM], nw[DIM], oB[DIM], nB[DIM];
                    path.get(p, j, od);
                    path.get(p, jB, oB);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) {
                        nw[e] = teleport(od[e] + d[e], P);
                        nB[e] = teleport(oB[e] + d[e], P);
                    }
                    T part = T(0);
                    if (g == 0) part += -P.tau * (potV<T, DIM>(nw, P) - potV<T, DIM>(od, P));
                    part = add_(part, link_delta_row<T, DIM>(path, P, p, j, jB, last, nw, od, nB, oB, g, G));
                    x = own ? (double)part : 0.0;
                }
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
                double *ws = s_wsum + (p & 1) * 16;
                if (lane == 0) ws[wave] = x;
                __syncthreads();
                double lw = 0.0;
                for (int w = 0; w < nwv; ++w) lw += ws[w];
                if (metropolis(ex((T)lw), Uniform<T>::get(y.z))) { // uniform
                    cacc += (tid == 0) ? 1 : 0;
                    for (int jj = tid; jj < M; jj += nt) {
                        T r[DIM];
                        path.get(p, jj, r);
#pragma unroll
                        for (int e = 0; e < DIM; ++e) r[e] = teleport(r[e] + d[e], P);
                        path.put(p, jj, r);
                    }
                }
                __syncthreads();
            }
        }
        if (meas_now) {
            const ChainMeas r = measure_chain<T, DIM, false>(path, none, ch, P, s_buf, a.radial, a.radial_bins, a.radial_winv,
                                                             a.cart, a.cart_bins, c, 8);
            if (tid == 0) fold_meas(r, ch, s_q);
        }
    }
    __syncthreads();
    for (int i = tid; i < N * M; i += nt) {
        const int jj = i / N, n = i - jj * N;
        T r[DIM];
        path.get(n, jj, r);
#pragma unroll
        for (int e = 0; e < DIM; ++e) gpath[(size_t)i * DIM + e] = r[e];
    }
    const double la = block_sum((double)lacc, s_buf);
    if (tid == 0) {
        double *out = a.chain_meas + (size_t)c * (kNQ + kCnt);
        const bool add = a.split && a.sweep_off > 0; // later one-sweep launches of a split step add their counts
        if (!add)
            for (int k = 0; k < kNQ; ++k) out[k] = s_q[k]; // zero when split: k_meas_fold adds
        const double n[5] = {la, (double)cacc, (double)ctry, 0.0, 0.0};
        for (int k = 0; k < 5; ++k) out[kNQ + k] = (add ? out[kNQ + k] : 0.0) + n[k];
    }
}

// Estimators of these chains in measuring runs that take them outside the sweep
// kernel: grid (windows of kMeasSlices slices, chains of a.ids), 256 threads.  The
// window's beads in LDS, one pair of particles per thread over the window's links
// (each unordered pair once, with the weight of both ends); the single-bead terms
// as measure_beads takes them.  part[(y * nblk + window) * 6]: the window's sums,
// folded in window order by k_meas_fold.  It is bound by the FP64 sums of the pair
// terms; walking a pair along the window takes one exponential per pair and slice,
// where k_meas_beads takes two per bead, neighbour and link and each pair from both
// its ends: 16 measuring sweeps of 512 chains of N = 64, M = 256, FP32, went from
// 46.5 to 36.6 ms.
constexpr int kMeasSlices = 16;
template <typename T, int DIM> __global__ void __launch_bounds__(256) k_meas_allpairs(MeasArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double s_sum[6 * 16];
    if (!split_measured(a)) return;
    const int y = blockIdx.y, c = a.ids[y], tid = threadIdx.x, nt = blockDim.x;
    ChainDev ch = a.chains[c];
    const int N = ch.N, M = ch.M, s0 = blockIdx.x * kMeasSlices;
    double *out = a.part + ((size_t)y * a.nblk + blockIdx.x) * 6;
    if (s0 >= M) {
        if (tid < 6) out[tid] = 0.0;
        return;
    }
    const int m = min(kMeasSlices, M - s0);
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    T *const gpath = reinterpret_cast<T *>(const_cast<void *>(a.pos)) + ch.pos_off;
    T *const ob = reinterpret_cast<T *>(smem); // [slice][particle][d]
    for (int i = tid; i < (m + 1) * N * DIM; i += nt) {
        const int t = i / (N * DIM), j = s0 + t < M ? s0 + t : 0;
        ob[i] = gpath[(size_t)j * N * DIM + (i - t * N * DIM)];
    }
    __syncthreads();
    const double inv_s2 = 1.0 / (ch.sigma * ch.sigma), wq = 2.0 * (0.5 * (0.5 * (double)P.tau));
    ch.pair = kPairNone; // the single-bead terms
    const Path<T, DIM, true> path{gpath, M, N};
    const Cells none{nullptr, nullptr, nullptr, M, 0, 0, ch.nbins};
    ChainMeas r = measure_beads<T, DIM, false>(path, none, ch, P, a.radial, a.radial_bins, a.radial_winv, a.cart,
                                               a.cart_bins, c, 1, nullptr, s0 * N, (s0 + m) * N);
    // pairs q < p: thread i takes pairs i, i + nt, ... of the triangle, row by row
    const int pairs = N * (N - 1) / 2;
    int p = 1, q = tid;
    for (int i = tid; i < pairs; i += nt, q += nt) {
        while (q >= p) q -= p, ++p;
        const T *rp = ob + (size_t)p * DIM, *rq = ob + (size_t)q * DIM;
        pair_energy_window<T, DIM>([&](int t, T *x, T *z) {
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                x[e] = rp[(size_t)t * N * DIM + e];
                z[e] = rq[(size_t)t * N * DIM + e];
            }
        }, m, P, 3, wq, inv_s2, r.su, r.rgp);
    }
    double v[6] = {r.link, r.V, r.rg, r.su, r.rgp, r.r2w};
    block_sums(v, s_sum);
    if (tid == 0)
        for (int k = 0; k < 6; ++k) out[k] = v[k];
}

} // namespace pimc
