// Sweep kernel of chains without a pair action that are run whole per
// workgroup: chains with swap moves (permutation cycles) and chains that record
// the products of the reweighting derivatives.
//
// Without a pair action a staging or centre-of-mass try reads and writes only
// its own beads, so the tries of all particles of a pass are independent and the
// result is that of the particle-by-particle schedule (k_sweep_whole): the
// staging windows of the particles, which follow the cycles, share one offset
// and tile the beads.  The path stays in LDS for the launch; a pass runs as a few
// phases over all N M beads with a barrier between them, instead of several
// barriers per particle.  Swap tries depend on each other and stay in order;
// their random numbers do not depend on the path and are drawn together before
// them, and the sums over the partners are taken by every thread from terms that
// were computed in parallel, which saves the round trips through one thread.
//
// One workgroup per chain, so what bounds it is the length of this chain of
// phases and not a unit of the chip.  256 chains of N = 10, M = 64 with 10 swap
// tries, FP32, 100 measuring sweeps with their results read: 22.1 ms on
// k_sweep_whole, 12.2 ms here (40 us a sweep in the kernel).
#pragma once
#include "sweep_kernels.hpp"

namespace pimc {

constexpr int kIdealThreads = 512;
constexpr int kSwapBatch = 16; // swap tries whose draws are made together

// LDS of k_sweep_ideal: path, new beads and normals (later Delta V per bead), the
// segments' flags (room for the shortest staging length, 2), next[], the swap
// tries' terms, bridges and draws.
struct IdealLds {
    size_t path, nb, nrm, flag, next, E, B, f, g, h, r, bridge, sn, dv, sx, end;
};
__host__ __device__ inline IdealLds ideal_lds(int N, int M, int dim, int tsize, int swaps, int swap_m)
{
    IdealLds L;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o = align16(o + bytes);
        return at;
    };
    const size_t beads = (size_t)N * M * dim * tsize;
    L.path = take(beads);
    L.nb = take(beads);
    L.nrm = take(beads);
    L.flag = take((size_t)N * ((M + 1) / 2) * 4);
    const size_t n = swaps > 0 ? N : 0, m = swaps > 0 ? swap_m + 1 : 0, b = swaps < kSwapBatch ? swaps : kSwapBatch;
    L.next = take(n * 4);
    L.E = take(n * dim * tsize);
    L.B = take(n * dim * tsize);
    L.f = take(n * tsize);
    L.g = take(n * tsize);
    L.h = take(n * tsize);
    L.r = take(n * tsize);
    L.bridge = take(2 * m * dim * tsize);
    L.sn = take(b * 2 * m * dim * tsize);
    L.dv = take(2 * m * tsize);
    L.sx = take(b * 16);
    L.end = o;
    return L;
}
__host__ __device__ inline IdealLds ideal_lds(const ChainDev &h, int tsize)
{
    return ideal_lds(h.N, h.M, h.dim, tsize, h.swaps, h.swap_m);
}

template <typename T, int DIM> __global__ void __launch_bounds__(kIdealThreads) k_sweep_ideal(SweepArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double s_sum[6 * 16], s_q[kNQ]; // s_q: estimator sums of the launch
    const int c = a.whole[blockIdx.x];
    const ChainDev ch = a.chains[c];
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = nt >> 6;
    const int N = ch.N, M = ch.M, ell = ch.ell, nseg = ch.nseg;
    const IdealLds L = ideal_lds(ch, (int)sizeof(T));
    T *const lpath = reinterpret_cast<T *>(smem + L.path);
    T *const s_new = reinterpret_cast<T *>(smem + L.nb); // [p][slice][d]
    T *const s_nrm = reinterpret_cast<T *>(smem + L.nrm);
    T *const s_dvb = s_nrm; // once the bridges are built
    int *const s_flag = reinterpret_cast<int *>(smem + L.flag);
    int *const s_next = reinterpret_cast<int *>(smem + L.next);
    T *const gpath = reinterpret_cast<T *>(a.pos) + ch.pos_off;
    int *const gnext = a.next + ch.part_base;
    const bool perm = ch.swaps > 0;
    for (int i = tid; i < N * M * DIM; i += nt) lpath[i] = gpath[i];
    for (int i = tid; i < (perm ? N : 0); i += nt) s_next[i] = gnext[i];
    const Path<T, DIM, true> path{lpath, M, N};
    const Cells none{nullptr, nullptr, nullptr, M, 0, 0, ch.nbins};
    const uint32_t sweep0 = a.rs->sweep + (uint32_t)a.sweep_off;
    // the particle holding bead u of the window that starts on particle p (see k_sweep_whole)
    auto owner = [&](int p, int u) { return (perm && u >= M) ? s_next[p] : p; };
    if (tid < kNQ) s_q[tid] = 0.0;
    int lacc = 0, cacc = 0, ctry = 0, sacc = 0, stry = 0;
    const int hp = ell >> 1; // Philox blocks per segment: interior bead pairs (i, i + 1), i odd
    int meas_in = (int)((uint32_t)a.measure_every - 1u - sweep0 % (uint32_t)a.measure_every);
    __syncthreads();

    for (int s = 0; s < a.nsweeps; ++s) {
        const uint32_t sw = sweep0 + (uint32_t)s;
        const bool meas_now = a.measure && !a.split && meas_in == 0;
        meas_in = (meas_in == 0) ? a.measure_every - 1 : meas_in - 1;
        if (pass_on(ch.every_st, sw)) {
            const U4 xo = draw(a.seed, 0u, sw, (uint32_t)c, kOffset); // one offset per chain and sweep
            const int off = (int)(((uint64_t)xo.x * (uint64_t)ell) >> 32);
            // normals of the interior beads, one bead pair per thread
            const int per = nseg * hp;
            for (int w = tid; w < N * per; w += nt) {
                const int p = w / per, v = w - p * per, k = v / hp, i = 2 * (v - k * hp) + 1;
                const int m = min(ell, M - k * ell);
                if (i < m) {
                    int b = off + k * ell + i;
                    if (b >= M) b -= M;
                    const U4 xr = draw(a.seed, (uint32_t)(p * M + b), sw, (uint32_t)c, kLevy);
                    T n0, n1;
                    box_muller(xr.x, xr.y, n0, n1);
                    T *x = s_nrm + ((size_t)p * M + b) * DIM;
                    x[0] = n0;
                    if (DIM > 1) x[DIM - 1] = n1;
                    if (i + 1 < m) {
                        const int b1 = (b + 1 == M) ? 0 : b + 1;
                        box_muller(xr.z, xr.w, n0, n1);
                        T *y = s_nrm + ((size_t)p * M + b1) * DIM;
                        y[0] = n0;
                        if (DIM > 1) y[DIM - 1] = n1;
                    }
                }
            }
            __syncthreads();
            // bridges, one segment per thread
            for (int it = tid; it < N * nseg; it += nt) {
                const int p = it / nseg, k = it - p * nseg;
                const int m = min(ell, M - k * ell);
                if (m < 2) continue;
                const int us = off + k * ell; // window position of the start bead (< 2M)
                const int start = us >= M ? us - M : us;
                int jm = start + m;
                if (jm >= M) jm -= M;
                T cur[DIM], em[DIM];
                path.get(owner(p, us), start, cur);
                path.get(owner(p, us + m), jm, em);
#pragma unroll
                for (int e = 0; e < DIM; ++e) em[e] = shift_end(cur[e], em[e], P);
                for (int i = 1; i < m; ++i) {
                    int b = start + i;
                    if (b >= M) b -= M;
                    const size_t at = ((size_t)p * M + b) * DIM;
                    const T alpha = bridge_alpha<T>(m, i);
                    const T sd = bridge_sd(alpha, P);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) {
                        cur[e] = bridge_step(cur[e], em[e], alpha, s_nrm[at + e], sd);
                        s_new[at + e] = teleport(cur[e], P);
                    }
                }
            }
            __syncthreads();
            // Delta V per interior bead
            for (int it = tid; it < N * M; it += nt) {
                const int p = it / M, j = it - p * M;
                int rel = j - off;
                if (rel < 0) rel += M;
                const int k = rel / ell, t = rel - k * ell;
                if (t < 1 || min(ell, M - k * ell) < 2) continue;
                T n0[DIM], o0[DIM];
#pragma unroll
                for (int e = 0; e < DIM; ++e) n0[e] = s_new[(size_t)it * DIM + e];
                path.get(owner(p, j >= off ? j : j + M), j, o0);
                s_dvb[it] = potV<T, DIM>(n0, P) - potV<T, DIM>(o0, P);
            }
            __syncthreads();
            // decisions, summing over the interior beads in order
            for (int it = tid; it < N * nseg; it += nt) {
                const int p = it / nseg, k = it - p * nseg;
                const int m = min(ell, M - k * ell);
                int acc = 0;
                if (m >= 2) {
                    int start = off + k * ell;
                    if (start >= M) start -= M;
                    T dv = T(0);
                    for (int i = 1; i < m; ++i) {
                        int b = start + i;
                        if (b >= M) b -= M;
                        dv += s_dvb[p * M + b];
                    }
                    const T lw = -P.tau * dv;
                    const U4 xa = draw(a.seed, (uint32_t)(p * M + start), sw, (uint32_t)c, kLevyAccept);
                    acc = metropolis(ex(lw), Uniform<T>::get(xa.x)) ? 1 : 0;
                }
                s_flag[it] = acc;
                lacc += acc;
            }
            __syncthreads();
            // commit interior beads of accepted segments
            for (int it = tid; it < N * M; it += nt) {
                const int p = it / M, j = it - p * M;
                int rel = j - off;
                if (rel < 0) rel += M;
                const int k = rel / ell, t = rel - k * ell;
                if (t < 1 || min(ell, M - k * ell) < 2 || !s_flag[p * nseg + k]) continue;
                T rn[DIM];
#pragma unroll
                for (int e = 0; e < DIM; ++e) rn[e] = s_new[(size_t)it * DIM + e];
                path.put(owner(p, j >= off ? j : j + M), j, rn);
            }
            __syncthreads();
        }
        // centre of mass: one wave per particle, 1-cycles only
        if (pass_on(ch.every_com, sw)) {
            for (int p = wave; p < N; p += nw) {
                if (perm && s_next[p] != p) continue;
                ctry += (lane == 0) ? 1 : 0;
                const U4 y = draw(a.seed, (uint32_t)p, sw, (uint32_t)c, kCom);
                const T step2 = (T)a.com_step[c] * T(2);
                T d[DIM];
                d[0] = step2 * (Uniform<T>::get(y.x) - T(0.5));
                if (DIM > 1) d[DIM - 1] = step2 * (Uniform<T>::get(y.y) - T(0.5));
                double x = 0.0;
                // (slices 512 apart are added in T, as k_sweep_whole's lanes take them)
                for (int l = lane; l < min(M, 512); l += 64) {
                    T part = T(0);
                    for (int j = l; j < M; j += 512) {
                        T o0[DIM], n0[DIM];
                        path.get(p, j, o0);
#pragma unroll
                        for (int e = 0; e < DIM; ++e) n0[e] = teleport(o0[e] + d[e], P);
                        part += -P.tau * (potV<T, DIM>(n0, P) - potV<T, DIM>(o0, P));
                    }
                    x += (double)part;
                }
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
                if (!metropolis(ex((T)x), Uniform<T>::get(y.z))) continue;
                cacc += (lane == 0) ? 1 : 0;
                for (int j = lane; j < M; j += 64) {
                    T r[DIM];
                    path.get(p, j, r);
#pragma unroll
                    for (int e = 0; e < DIM; ++e) r[e] = teleport(r[e] + d[e], P);
                    path.put(p, j, r);
                }
            }
            __syncthreads();
        }
        // swap tries (see k_sweep_whole for the move): the draws of a batch together, then try by try
        const int tries = (perm && pass_on(ch.every_sw, sw)) ? ch.swaps : 0, m = ch.swap_m;
        T *const s_E = reinterpret_cast<T *>(smem + L.E), *const s_B = reinterpret_cast<T *>(smem + L.B);
        T *const s_f = reinterpret_cast<T *>(smem + L.f), *const s_g = reinterpret_cast<T *>(smem + L.g);
        T *const s_h = reinterpret_cast<T *>(smem + L.h), *const s_r = reinterpret_cast<T *>(smem + L.r);
        T *const s_br = reinterpret_cast<T *>(smem + L.bridge); // [w][i][d], beads 1..m-1 of path w
        T *const s_sn = reinterpret_cast<T *>(smem + L.sn);     // [try][w][i][d]
        T *const s_dw = reinterpret_cast<T *>(smem + L.dv);     // [w][i]
        U4 *const s_sx = reinterpret_cast<U4 *>(smem + L.sx);
        for (int a0 = 0; a0 < tries; a0 += kSwapBatch) {
            const int nb = min(kSwapBatch, tries - a0), hs = m >> 1;
            for (int w = tid; w < nb; w += nt) s_sx[w] = draw(a.seed, (uint32_t)(a0 + w), sw, (uint32_t)c, kSwap);
            for (int w = tid; w < nb * 2 * hs; w += nt) {
                const int tw = w / hs, i = 2 * (w - tw * hs) + 1; // tw = 2 try + path
                if (i >= m) continue;
                const U4 xr = draw(a.seed, (uint32_t)((2 * a0 + tw) * M + i), sw, (uint32_t)c, kSwapLevy);
                T *x = s_sn + ((size_t)tw * (m + 1) + i) * DIM, n0, n1;
                box_muller(xr.x, xr.y, n0, n1);
                x[0] = n0;
                if (DIM > 1) x[DIM - 1] = n1;
                if (i + 1 < m) {
                    box_muller(xr.z, xr.w, n0, n1);
                    x[DIM] = n0;
                    if (DIM > 1) x[2 * DIM - 1] = n1;
                }
            }
            for (int t = 0; t < nb; ++t) {
                __syncthreads(); // the draws, and the previous try's commit
                const U4 xs = s_sx[t];
                const int j0 = (int)(((uint64_t)xs.x * (uint64_t)M) >> 32);
                const int n1 = (int)(((uint64_t)xs.y * (uint64_t)N) >> 32);
                const int jm = j0 + m, sm = jm >= M ? jm - M : jm;
                stry += (tid == 0) ? 1 : 0;
                if (N < 2) continue;
                // ends E_i and starts B_i of every partner, and the weights against n1
                T A[DIM], C[DIM];
                path.get(n1, j0, A);
                path.get(jm < M ? n1 : s_next[n1], sm, C);
                for (int i = tid; i < N; i += nt) {
                    T e[DIM], b[DIM];
                    path.get(jm < M ? i : s_next[i], sm, e);
                    path.get(i, j0, b);
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        s_E[i * DIM + d] = e[d];
                        s_B[i * DIM + d] = b[d];
                    }
                    s_f[i] = rho0<T, DIM>(A, e, P, m);
                    s_r[i] = rho0<T, DIM>(b, C, P, m);
                }
                __syncthreads();
                // the partner: every thread takes the same sums in particle order
                T W1 = T(0);
                for (int i = 0; i < N; ++i) W1 += s_f[i] * s_r[i];
                const T target = Uniform<T>::get(xs.z) * W1;
                T cum = T(0);
                int n2 = N - 1;
                for (int i = 0; i < N; ++i) {
                    cum += s_f[i] * s_r[i];
                    if (cum > target) {
                        n2 = i;
                        break;
                    }
                }
                if (n2 == n1) continue; // uniform
                // the two bridges: n1 from r_n1(j0) to E_n2, n2 from r_n2(j0) to E_n1 (wave 0);
                // the weights against n2 (the other waves)
                if (tid < 2) {
                    const int w = tid;
                    T *bw = s_br + (size_t)w * (m + 1) * DIM;
                    const T *st0 = s_B + (w == 0 ? n1 : n2) * DIM, *en = s_E + (w == 0 ? n2 : n1) * DIM;
                    const T *sn = s_sn + (size_t)(2 * t + w) * (m + 1) * DIM;
                    T cur[DIM], em[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        cur[d] = st0[d];
                        em[d] = shift_end(cur[d], en[d], P);
                    }
                    for (int i = 1; i < m; ++i) {
                        const T alpha = bridge_alpha<T>(m, i);
                        const T sd = bridge_sd(alpha, P);
#pragma unroll
                        for (int d = 0; d < DIM; ++d) {
                            cur[d] = bridge_step(cur[d], em[d], alpha, sn[i * DIM + d], sd);
                            bw[i * DIM + d] = teleport(cur[d], P);
                        }
                    }
                } else if (wave > 0 && ch.swap_rule == 0) {
                    for (int i = tid - 64; i < N; i += nt - 64) {
                        s_g[i] = rho0<T, DIM>(s_B + n2 * DIM, s_E + i * DIM, P, m);
                        s_h[i] = rho0<T, DIM>(s_B + i * DIM, s_E + n2 * DIM, P, m);
                    }
                }
                __syncthreads();
                // Delta V of the interior beads of both paths (old beads along the old cycles)
                for (int it = tid; it < 2 * m; it += nt) {
                    const int w = it >= m ? 1 : 0, i = it - w * m;
                    if (i < 1) continue;
                    const int u = j0 + i;
                    T nb_[DIM], ob[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) nb_[d] = s_br[((size_t)w * (m + 1) + i) * DIM + d];
                    path.get(owner(w == 0 ? n1 : n2, u), u >= M ? u - M : u, ob);
                    s_dw[w * (m + 1) + i] = potV<T, DIM>(nb_, P) - potV<T, DIM>(ob, P);
                }
                __syncthreads();
                // the decision: again every thread the same sums
                T dv = T(0);
                for (int w = 0; w < 2; ++w)
                    for (int i = 1; i < m; ++i) dv += s_dw[w * (m + 1) + i];
                T ratio = ex(-P.tau * dv);
                if (ch.swap_rule == 0) {
                    // reverse over forward partner-choice probability, either particle drawn first:
                    // after the swap n1 ends at E_n2 and n2 at E_n1
                    T V1 = T(0), W2 = T(0), W1p = T(0), W2p = T(0);
                    for (int i = 0; i < N; ++i) {
                        const int ip = i == n1 ? n2 : (i == n2 ? n1 : i);
                        V1 += s_f[i] * s_r[i];
                        W2 += s_g[i] * s_h[i];
                        W1p += s_f[ip] * s_h[i];
                        W2p += s_g[ip] * s_r[i];
                    }
                    ratio *= (T(1) / W1p + T(1) / W2p) / (T(1) / V1 + T(1) / W2);
                }
                if (!metropolis(ratio, Uniform<T>::get(xs.w))) continue; // uniform
                const int q1 = s_next[n1], q2 = s_next[n2];
                for (int i = 1 + tid; i < m; i += nt) {
                    const int u = j0 + i, j = u >= M ? u - M : u;
                    const int qa = u < M ? n1 : q2, qb = u < M ? n2 : q1; // along the new cycles
                    path.put(qa, j, s_br + i * DIM);
                    path.put(qb, j, s_br + ((size_t)(m + 1) + i) * DIM);
                }
                if (jm < M) {
                    for (int j = jm + tid; j < M; j += nt) {
                        T r1[DIM], r2[DIM];
                        path.get(n1, j, r1);
                        path.get(n2, j, r2);
                        path.put(n1, j, r2);
                        path.put(n2, j, r1);
                    }
                }
                __syncthreads();
                if (tid == 0) {
                    s_next[n1] = q2;
                    s_next[n2] = q1;
                    sacc += 1;
                }
            }
            __syncthreads();
        }
        if (meas_now) {
            const ChainMeas r = measure_beads<T, DIM, false>(path, none, ch, P, a.radial, a.radial_bins, a.radial_winv, a.cart,
                                                             a.cart_bins, c, 1, perm ? s_next : nullptr, 0, -1);
            double v[6] = {r.link, r.V, r.rg, r.su, r.rgp, r.r2w};
            block_sums(v, s_sum);
            if (tid == 0) fold_meas(ChainMeas{v[0], v[1], v[2], v[3], v[4], v[5]}, ch, s_q);
        }
    }
    __syncthreads();
    for (int i = tid; i < N * M * DIM; i += nt) gpath[i] = lpath[i];
    for (int i = tid; i < (perm ? N : 0); i += nt) gnext[i] = s_next[i];
    double n[5] = {(double)lacc, (double)cacc, (double)ctry, (double)sacc, (double)stry};
    block_sums(n, s_sum);
    if (tid == 0) {
        double *out = a.chain_meas + (size_t)c * (kNQ + kCnt);
        const bool add = a.split && a.sweep_off > 0; // later one-sweep launches of a split step add their counts
        if (!add)
            for (int k = 0; k < kNQ; ++k) out[k] = s_q[k]; // zero when split: k_meas_fold adds
        for (int k = 0; k < 5; ++k) out[kNQ + k] = (add ? out[kNQ + k] : 0.0) + n[k];
    }
}

} // namespace pimc
