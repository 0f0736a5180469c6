// Sweep kernels of chains with a Gaussian pair action (the interacting
// workloads): staging moves by slice windows, centre-of-mass moves by
// speculation and dependency rounds.
//
// Staging (k_stage_win).  All particles of a chain share one staging offset
// per sweep, so their segments occupy the same slice windows [s, s + ell].
// A move of particle p in window w reads and writes only beads at the
// window's slices; the end slices s and s + ell are written by no staging
// move.  Moves in different windows therefore touch disjoint beads and
// commute: the result is the particle-by-particle schedule whatever order the
// windows run in.  One workgroup owns one window.
//
// Within a window every proposal depends only on the particle's own fixed end
// beads and its own draws, so all of them are formed first.  The log-weight
// change of particle p's try against the configuration the schedule presents
// to it is
//   Delta V_p + sum_q A(p, q) + sum_{q < p accepted} C(p, q),
// with, per link, T(x, y) the pair term of p's beads x (o: old, n: new) with
// q's beads y:  A = T(n, o) - T(o, o)  and  C = T(n, n) - T(o, n) - A.
// Both are computed for every pair whose window bounds (centre and radius of
// the old and new beads) come within the cut-off; other pairs have no term
// within the cut-off, so A = C = 0 exactly.  The decisions then need only the
// acceptances of each try's earlier partners: a chunk of 64 tries is decided
// in rounds, each round taking every try whose earlier partners in the chunk
// are decided.  Every sum runs in a fixed order (partners by index), so the
// result does not depend on thread timing.
//
// Centre of mass.  The sums A and C over the whole ring are taken window by
// window before any decision, for every pair of particles that can meet:
// k_com_bounds bounds each particle's beads per window and per ring,
// k_com_pairs lists the pairs p > q whose ring bounds (old or shifted) come
// within the cut-off, k_com_spec evaluates, per window, the listed pairs whose
// window bounds do, each pair once for A(p, q), A(q, p) and C(p, q), and
// k_com_dec (one workgroup per chain) only adds the windows' values and decides
// in rounds as above; k_com_apply moves the accepted rings.
//
// The cell lists are not used by these kernels; k_cells_win rebuilds them
// (members by particle index) where the estimators or other callers need them.
#pragma once
#include "sweep_kernels.hpp"

namespace pimc {

constexpr int kChunk = 64; // tries decided per block of rounds (one wave)

// Slices per centre-of-mass window: at most 32 windows per ring.
__host__ __device__ inline int com_win_len(int M) { return M <= 256 ? 8 : (M + 31) / 32; }
__host__ __device__ inline int com_nwin(int M) { return (M + com_win_len(M) - 1) / com_win_len(M); }

// Signed minimum-image offset x1 - x2.
template <typename T> __device__ __forceinline__ T signed_mindist(T x1, T x2, const Prm<T> &p)
{
    T d = x1 - x2;
    if (d > p.L) d -= p.twoL;
    else if (d < -p.L) d += p.twoL;
    return d;
}

// Multiplicity of particle k (bead rk) among the stencil candidates of a
// query at q: 1 within the cut-off for nbins >= 3; when nbins < 3 the number
// of stencil slots of q's cell that hold rk's cell (find_nns repeats cells
// then).  Symmetric in q and rk.
template <typename T, int DIM>
__device__ __forceinline__ T stencil_mult(const T *q, const T *rk, const Prm<T> &P, int nbins)
{
    if (nbins >= 3) return T(1);
    constexpr int NS = (DIM == 1) ? 3 : 9;
    const int c0 = cell_of<T, DIM>(q, P, nbins), ck = cell_of<T, DIM>(rk, P, nbins);
    int mm = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) mm += (stencil_cell(c0, s, nbins, DIM) == ck);
    return T(mm);
}

// Exclusive prefix of one value per lane over a wave; returns the lane's
// prefix and sets the wave total.
__device__ __forceinline__ int wave_prefix(int v, int lane, int &total)
{
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    total = __shfl(x, 63, 64);
    return x - v;
}

// --- window bounds (FP32; the overlap test's margin covers the rounding) ---

__device__ __forceinline__ float mi_f(float d, float twoL, float inv2L) { return d - twoL * rintf(d * inv2L); }

// Whether beads within ar of (ax, ay) and beads within br of (bx, by) can
// come within the cut-off h of each other (periodic box of side twoL).
template <int DIM>
__device__ __forceinline__ bool bnd_near(float ax, float ay, float ar, float bx, float by, float br, float h,
                                         float twoL, float inv2L)
{
    const float dx = mi_f(ax - bx, twoL, inv2L);
    float d2 = dx * dx;
    if (DIM > 1) {
        const float dy = mi_f(ay - by, twoL, inv2L);
        d2 += dy * dy;
    }
    const float reach = (ar + br + h) * 1.00001f + 1e-5f * twoL;
    return d2 <= reach * reach;
}

// The four pairings of two bounds shifted by their centre-of-mass shifts
// (x: particle a old/new, y: particle b old/new).
template <int DIM>
__device__ __forceinline__ bool bnd_near4(float4 A, const float *da, float4 B, const float *db, float h, float twoL,
                                          float inv2L)
{
    const float ax1 = A.x + da[0], ay1 = DIM > 1 ? A.y + da[1] : 0.f;
    const float bx1 = B.x + db[0], by1 = DIM > 1 ? B.y + db[1] : 0.f;
    return bnd_near<DIM>(A.x, A.y, A.z, B.x, B.y, B.z, h, twoL, inv2L) ||
           bnd_near<DIM>(ax1, ay1, A.z, B.x, B.y, B.z, h, twoL, inv2L) ||
           bnd_near<DIM>(A.x, A.y, A.z, bx1, by1, B.z, h, twoL, inv2L) ||
           bnd_near<DIM>(ax1, ay1, A.z, bx1, by1, B.z, h, twoL, inv2L);
}

// --- pair terms of one window ---

// Sums and products of the pair terms keep their own roundings, whatever code
// surrounds them.
template <typename T> __device__ __forceinline__ T add_(T x, T y)
{
#pragma clang fp contract(off)
    return x + y;
}
template <typename T> __device__ __forceinline__ T sub_(T x, T y)
{
#pragma clang fp contract(off)
    return x - y;
}
template <bool MULT, typename T> __device__ __forceinline__ T link_term(T mult, T ctau, T e0, T e1)
{
#pragma clang fp contract(off)
    const T s = ctau * (e0 + e1);
    return MULT ? mult * s : s;
}
__device__ __forceinline__ bool is_neg_zero(float x) { return __float_as_uint(x) == 0x80000000u; }
__device__ __forceinline__ bool is_neg_zero(double x) { return __double_as_longlong(x) == (long long)0x8000000000000000ull; }

// dist2 with the minimum taken by one instruction instead of a compare and a select.
template <typename T> __device__ __forceinline__ T mindist_min(T x1, T x2, const Prm<T> &p)
{
    const T dx = fabs(x1 - x2);
    return min_(p.twoL - dx, dx);
}
template <typename T, int DIM> __device__ __forceinline__ T dist2_min(const T *x, const T *y, const Prm<T> &P)
{
    const T d0 = mindist_min(x[0], y[0], P);
    if (DIM == 1) return d0 * d0;
    const T d1 = mindist_min(x[DIM - 1], y[DIM - 1], P);
    return fma_(d0, d0, d1 * d1);
}

// --- ordered pair lists of a chunk of particles ---

// LDS layout of the chunk machinery: candidate masks (kChunk x nq words),
// counts, offsets, then the slots (partner index and owner).
struct ChunkLds {
    size_t mask, cnt, off, misc, pq, po, end;
};
__host__ __device__ inline ChunkLds chunk_lds(size_t o, int N, int cap)
{
    ChunkLds L;
    const int nq = (N + 63) / 64;
    L.mask = o;
    o = align16(o + (size_t)kChunk * nq * 8);
    L.cnt = o;
    o = align16(o + kChunk * 4);
    L.off = o;
    o = align16(o + kChunk * 4);
    L.misc = o;
    o = align16(o + 16);
    L.pq = o;
    o = align16(o + (size_t)cap * 2);
    L.po = o;
    L.end = align16(o + (size_t)cap);
    return L;
}

struct ChunkPtr {
    unsigned long long *mask;
    int *cnt, *off, *misc;
    unsigned short *pq;
    unsigned char *po;
    __device__ __forceinline__ ChunkPtr(unsigned char *s, const ChunkLds &L)
        : mask(reinterpret_cast<unsigned long long *>(s + L.mask)), cnt(reinterpret_cast<int *>(s + L.cnt)),
          off(reinterpret_cast<int *>(s + L.off)), misc(reinterpret_cast<int *>(s + L.misc)),
          pq(reinterpret_cast<unsigned short *>(s + L.pq)), po(s + L.po)
    {
    }
};

// --- grid of window centres ---

// A uniform periodic grid over the particles' bound centres, rebuilt per
// window: cells of side >= 2 rmax + h (rmax the largest bound radius), so two
// bounds within reach sit in neighbouring cells and a particle's candidates
// are the members of its 3^DIM stencil.  ng cells per dimension, at most
// kGridMax; no grid (ng = 0) when the stencil would cover more than a quarter
// (2D: ng < 6) or three eighths (1D: ng < 8) of the box, where the full scan
// is cheaper.
constexpr int kGridMax = 16;

struct GridLds {
    size_t start, mem, pcell, misc, end;
};
__host__ __device__ inline GridLds grid_lds(size_t o, int N, int dim)
{
    GridLds L;
    const int nc = dim == 1 ? kGridMax : kGridMax * kGridMax;
    L.start = o;
    o = align16(o + (size_t)(nc + 1) * 4);
    L.mem = o;
    o = align16(o + (size_t)N * 2);
    L.pcell = o;
    o = align16(o + (size_t)N * 2);
    L.misc = o;
    o = align16(o + 16);
    L.end = o;
    return L;
}

struct WinGrid {
    int *start;            // after the build: cell c's members are mem[c ? start[c - 1] : 0 .. start[c])
    unsigned short *mem;   // particles by cell
    unsigned short *pcell; // each particle's cell
    int *misc;             // [0] largest radius (float bits)
    int ng;
    __device__ __forceinline__ WinGrid(unsigned char *s, const GridLds &L)
        : start(reinterpret_cast<int *>(s + L.start)), mem(reinterpret_cast<unsigned short *>(s + L.mem)),
          pcell(reinterpret_cast<unsigned short *>(s + L.pcell)), misc(reinterpret_cast<int *>(s + L.misc)), ng(0)
    {
    }
};

// Build the grid from centre(p, x, y, r) (all threads of the workgroup); sets G.ng.
template <int DIM, typename Centre>
__device__ inline void grid_build(WinGrid &G, int N, float h, float twoL, float inv2L, Centre centre)
{
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) G.misc[0] = 0;
    __syncthreads();
    for (int p = tid; p < N; p += nt) {
        float x, y, r;
        centre(p, x, y, r);
        atomicMax(G.misc, __float_as_int(fmaxf(r, 0.f)));
    }
    __syncthreads();
    const float rmax = __int_as_float(G.misc[0]);
    const float side = (2.f * rmax + h) * 1.0001f + 2e-5f * twoL;
    int ng = min((int)floorf(twoL / side), kGridMax);
    G.ng = ng >= (DIM == 1 ? 8 : 6) ? ng : 0;
    if (G.ng == 0) return; // uniform: every thread read the same rmax
    const int ncell = DIM == 1 ? ng : ng * ng;
    for (int c = tid; c <= ncell; c += nt) G.start[c] = 0;
    __syncthreads();
    const float scale = (float)ng * inv2L;
    auto axis = [&](float v) {
        const float w = v - twoL * floorf(v * inv2L + 0.5f); // into [-L, L]
        return min(max((int)((w + 0.5f * twoL) * scale), 0), ng - 1);
    };
    for (int p = tid; p < N; p += nt) {
        float x, y, r;
        centre(p, x, y, r);
        const int c = DIM == 1 ? axis(x) : axis(x) + ng * axis(y);
        G.pcell[p] = (unsigned short)c;
        atomicAdd(G.start + c + 1, 1);
    }
    __syncthreads();
    if (wave == 0) { // inclusive prefix: start[c] = members of the cells before c
        int base = 0;
        for (int c0 = 0; c0 <= ncell; c0 += 64) {
            const int c = c0 + lane;
            const int v = c <= ncell ? G.start[c] : 0;
            int tot;
            const int pre = wave_prefix(v, lane, tot);
            if (c <= ncell) G.start[c] = base + pre + v;
            base += tot;
        }
    }
    __syncthreads();
    for (int p = tid; p < N; p += nt) {
        const int at = atomicAdd(G.start + G.pcell[p], 1); // start[c] ends at cell c's end
        G.mem[at] = (unsigned short)p;
    }
    __syncthreads();
}

// The members of particle p's stencil, flattened over the lanes of a wave.
template <int DIM, typename Visit> __device__ __forceinline__ void grid_visit(const WinGrid &G, int p, int lane, Visit visit)
{
    const int ng = G.ng;
    constexpr int NS = DIM == 1 ? 3 : 9;
    const int pc = G.pcell[p];
    const int ix = DIM == 1 ? pc : pc % ng, iy = DIM == 1 ? 0 : pc / ng;
    int b[NS], pre[NS + 1];
    pre[0] = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        int cx = ix + k % 3 - 1, cy = iy + (DIM == 1 ? 0 : k / 3 - 1);
        cx += cx < 0 ? ng : (cx >= ng ? -ng : 0);
        cy += cy < 0 ? ng : (cy >= ng ? -ng : 0);
        const int cc = cx + ng * cy;
        b[k] = cc ? G.start[cc - 1] : 0;
        pre[k + 1] = pre[k] + G.start[cc] - b[k];
    }
    for (int i = lane; i < pre[NS]; i += 64) {
        int at = b[0] + i;
#pragma unroll
        for (int k = 1; k < NS; ++k) at = i >= pre[k] ? b[k] + (i - pre[k]) : at;
        visit((int)G.mem[at]);
    }
}

// Slots of the chunk's particles pa, pa + 1, ... (at most kc <= kChunk): for
// each the partners q with cand(p, q), by index.  Fills as many particles as
// the pool holds (at least one: cap >= N).  Returns the number of particles filled (0: a caller's
// loop over the particles has to end); X.misc[1] is the slot count.  All threads of the workgroup.
template <int DIM = 2, typename Cand>
__device__ inline int chunk_slots(ChunkPtr &X, int pa, int N, int cap, int kc, Cand cand,
                                  const WinGrid *G = nullptr)
{
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nwv = nt >> 6;
    const int nq = (N + 63) / 64, nc = min(kc, N - pa);
    if (G && G->ng > 0) {
        // candidates from the grid stencil (one wave per particle, the stencil's members
        // flattened over the lanes), set as bits of the particle's mask
        for (int i = tid; i < nc * nq; i += nt) X.mask[i] = 0ull;
        __syncthreads();
        for (int l = wave; l < nc; l += nwv) {
            const int p = pa + l;
            grid_visit<DIM>(*G, p, lane, [&](int q) {
                if (cand(p, q)) atomicOr(X.mask + l * nq + (q >> 6), 1ull << (q & 63));
            });
        }
        __syncthreads();
        for (int l = tid; l < nc; l += nt) {
            int cnt = 0;
            for (int k = 0; k < nq; ++k) cnt += __popcll(X.mask[l * nq + k]);
            X.cnt[l] = cnt;
        }
    } else {
        for (int l = wave; l < nc; l += nwv) {
            const int p = pa + l;
            int cnt = 0;
            for (int q0 = 0; q0 < N; q0 += 64) {
                const int q = q0 + lane;
                const bool ok = q < N && cand(p, q);
                const unsigned long long bal = __ballot(ok);
                if (lane == 0) X.mask[l * nq + (q0 >> 6)] = bal;
                cnt += __popcll(bal);
            }
            if (lane == 0) X.cnt[l] = cnt;
        }
    }
    __syncthreads();
    if (wave == 0) {
        const int v = lane < nc ? X.cnt[lane] : 0;
        int tot;
        const int pre = wave_prefix(v, lane, tot);
        const bool fits = lane < nc && pre + v <= cap;
        const int nf = __popcll(__ballot(fits));
        const int used = __shfl(pre + v, max(nf - 1, 0), 64);
        X.off[lane] = pre;
        if (lane == 0) {
            X.misc[0] = nf;
            X.misc[1] = nf > 0 ? used : 0;
        }
    }
    __syncthreads();
    const int nf = X.misc[0];
    for (int it = tid; it < nf * nq; it += nt) {
        const int l = it / nq, wd = it - l * nq;
        const unsigned long long *mk = X.mask + (size_t)l * nq;
        int s = X.off[l];
        for (int k = 0; k < wd; ++k) s += __popcll(mk[k]);
        unsigned long long b = mk[wd];
        while (b) {
            const int bit = __ffsll((long long)b) - 1;
            b &= b - 1;
            X.pq[s] = (unsigned short)(wd * 64 + bit);
            X.po[s] = (unsigned char)l;
            ++s;
        }
    }
    __syncthreads();
    return nf;
}

// Decisions of the chunk's tries pa .. pa + nf - 1 in index order (one wave,
// lane l decides try pa + l).  pq(i), pc(i), i in o0 .. o1, are the try's earlier
// partners by index (hit flag in bit 15) and their C values, sp its sum against
// the configuration at the start, u its uniform; acc[q] holds the decisions of
// the tries before the chunk.  A try waits for its earlier partners inside the
// chunk that have a term within the cut-off (the others add exactly zero).  Each
// round decides every try whose such partners are decided; a try's sum takes the
// partners before the chunk in index order, then the partners inside the chunk as
// they are accepted (by round, in index order within a round), a fixed order.
// The earliest undecided try is always ready, so nf rounds decide the chunk; a list that names a
// partner at or after its own try would leave tries undecided (not accepted), and `whole` is false.
// Returns the acceptance mask.
template <typename T, typename Q, typename C>
__device__ inline unsigned long long chunk_decide(Q pq, C pc, int o0, int o1, double sp, T u, int pa, int nf,
                                                  const unsigned char *acc, bool &whole)
{
    const int l = threadIdx.x & 63;
    const bool in = l < nf;
    T tot = T(0);
    unsigned long long dep = 0ull, pm = 0ull; // in-chunk partners with a term within the cut-off, all
    int si = o1;                              // first in-chunk partner's slot
    for (int i = o0; i < o1; ++i) {
        const int qq = pq(i), q = qq & 0x7fff;
        if (q < pa) {
            if (acc[q]) tot += pc(i);
        } else {
            if (si == o1) si = i;
            pm |= 1ull << (q - pa);
            if (qq & 0x8000) dep |= 1ull << (q - pa);
        }
    }
    unsigned long long decided = nf >= 64 ? 0ull : (~0ull << nf), am = 0ull;
    for (int round = 0; round < nf && decided != ~0ull; ++round) {
        const bool ready = in && !((decided >> l) & 1ull) && (dep & ~decided) == 0ull;
        bool ok = false;
        if (ready) {
            const T lw = (T)(sp + (double)tot);
            ok = metropolis(ex(lw), u);
        }
        decided |= __ballot(ready);
        const unsigned long long na = __ballot(ok);
        am |= na;
        if (!((decided >> l) & 1ull)) {
            unsigned long long b = na & pm;
            while (b) {
                const int k = __ffsll((long long)b) - 1;
                b &= b - 1;
                tot += pc(si + __popcll(pm & ((1ull << k) - 1ull)));
            }
        }
    }
    whole = decided == ~0ull;
    return am;
}

// Clear the per-launch outputs of the listed chains (the kernels of a launch
// step add into them).
__global__ void k_clear_chain_meas(double *chain_meas, const int *ids, int n)
{
    const int i = blockIdx.x;
    if (i >= n) return;
    double *o = chain_meas + (size_t)ids[i] * (kNQ + kCnt);
    for (int k = threadIdx.x; k < kNQ + kCnt; k += blockDim.x) o[k] = 0.0;
}

// Index of pair (p, q = 0) among the pairs p > q of a chain.
__host__ __device__ __forceinline__ size_t pair_row(int p) { return (size_t)p * (size_t)(p - 1) / 2; }

// Buffers of the centre-of-mass kernels.  Per particle (window chains only, by
// part_base) wbnd[. * nwin + w] bounds its old beads in window w, rbnd its old
// ring, shift its try's displacement, cnt the listed partners; per pair slot
// (ChainDev::pair_off + pair_row(p) + k, the k-th listed partner of p by index)
// partner; per window and slot (at nval times the chain's pair offset)
// cval: C of the window, with +0 for "no term within the cut-off" (a value of
// zero with one is stored as -0).  The staging kernel keeps the pairs that do not
// fit its LDS in cval, before the centre-of-mass pass of the sweep fills it.
template <typename T> struct ComBuf {
    float4 *wbnd, *rbnd;
    T *shift;
    double *spec; // [particle * nwin + w]: the window's Delta V + sum_q A
    int *cnt;
    unsigned short *partner;
    T *cval;
    int nwin, nval; // windows of a particle; values kept per pair slot
    __device__ __forceinline__ unsigned short *row(const ChainDev &ch, int p) const
    {
        return partner + ch.pair_off + pair_row(p);
    }
    __device__ __forceinline__ T *vals(const ChainDev &ch, int w) const
    {
        return cval + (size_t)ch.pair_off * nval + (size_t)w * pair_row(ch.N);
    }
};

// A(p, q), A(q, p) and C(p, q) of one pair over the links 0 .. m - 1 of a window,
// the pairings of old (o) and new (n) beads each evaluated once for both
// particles.  A link's term is the one a neighbour adds in interaction_action!
// (src/updates/helper.jl:326-346), from the link's first slice, 0 for a bead
// outside the cut-off there (not among find_nns's neighbours).  bead(t, who, ro,
// rn): old and new bead of particle p (who 0) or q (who 1) at window slice t.
// hit: some pairing has a term within the cut-off.  MULT: chains with nbins < 3, whose terms carry a
// stencil multiplicity.  ENDS: the old and new beads coincide at slices 0 and m
// (staging), so one pairing is evaluated there.
template <typename T, int DIM, bool MULT, bool ENDS = false, typename BeadFn>
__device__ __forceinline__ void pair_window_both(BeadFn bead, int m, const Prm<T> &P, int nbins, T &Apq, T &Aqp, T &C,
                                                 bool &hit)
{
    const T ctau = T(-0.5) * P.tau;
    T e0[4], u0[4]; // the previous slice's pair potential and multiplicity: oo, no, on, nn
    bool in0[4];
    Apq = Aqp = C = T(0);
    hit = false;
    for (int t = 0; t <= m; ++t) {
        T po[DIM], pn[DIM], qo[DIM], qn[DIM];
        bead(t, 0, po, pn);
        bead(t, 1, qo, qn);
        const T *x[4] = {po, pn, po, pn}, *y[4] = {qo, qo, qn, qn};
        T e[4], u[4], tl[4];
        bool in[4];
        auto eval = [&](int k) {
            const T d2 = dist2_min<T, DIM>(x[k], y[k], P);
            in[k] = d2 <= P.h2;
            e[k] = vpair_r2(d2, P);
            u[k] = MULT ? stencil_mult<T, DIM>(x[k], y[k], P, nbins) : T(1);
        };
        eval(0);
        if (ENDS && (t == 0 || t == m)) {
#pragma unroll
            for (int k = 1; k < 4; ++k) {
                in[k] = in[0];
                e[k] = e[0];
                u[k] = u[0];
            }
        } else {
#pragma unroll
            for (int k = 1; k < 4; ++k) eval(k);
        }
        if (t > 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) tl[k] = in0[k] ? link_term<MULT>(u0[k], ctau, e0[k], e[k]) : T(0);
            const T a1 = sub_(tl[1], tl[0]);
            Apq = add_(Apq, a1);
            Aqp = add_(Aqp, sub_(tl[2], tl[0]));
            C = add_(C, sub_(sub_(tl[3], tl[2]), a1));
        }
        if (t < m) hit = hit || in[0] || in[1] || in[2] || in[3];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            e0[k] = e[k];
            in0[k] = in[k];
            if (MULT) u0[k] = u[k];
        }
    }
}

// --- staging ---

// Candidate partners (both sides) that one chunk of tries may have together: a
// chunk ends where its tries would exceed it.  A try's sum takes the partners of
// earlier chunks by index and those of its own chunk by round, so the chunk
// boundaries are part of the order of the sums; this rule (what fitted 64 KiB of
// LDS beside the window's beads when the pairs of a chunk were held for both
// sides) keeps them where they were.
inline int stage_budget(int N, int ell, int dim, int tsize)
{
    size_t o = 0;
    auto take = [&](size_t bytes) { o = align16(o + bytes); };
    take((size_t)(ell + 1) * N * dim * tsize);
    take((size_t)(ell > 1 ? ell - 1 : 1) * N * dim * tsize);
    take((size_t)N * 16);
    take((size_t)N * tsize);
    take((size_t)N * tsize);
    take((size_t)N);
    o = grid_lds(o, N, dim).end;
    take((size_t)kChunk * ((N + 63) / 64) * 8);
    for (int bytes : {kChunk * 4, (kChunk + 1) * 4, kChunk * 4, kChunk * 8, 16}) take((size_t)bytes);
    const size_t fixed = o;
    auto bytes = [&](int cap) { // per pair: partner, owner, two values
        o = fixed;
        take((size_t)cap * 2);
        take((size_t)cap);
        take((size_t)cap * tsize);
        take((size_t)cap * tsize);
        return o;
    };
    int cap = std::min(8192, kChunk * std::max(1, N - 1));
    while (cap > N && bytes(cap) > 64 * 1024) cap -= 64;
    return std::max(cap, N);
}

// LDS of k_stage_win: old beads of the window's ell + 1 slices, new interior
// beads, bounds, sums, candidate counts, grid; masks of a block of R rows
// (partners q < p in words of 64, and each particle's rows), the block's pool of
// cap pairs (the two A values), then the window's pairs by row: partner
// with the hit flag in bit 15 and C, the first `keep` of them here and the rest
// in memory.  What one workgroup needs with the smallest blocks (R = 64, cap = N,
// keep = 0) sets the largest chain, so arrays that are not in use together share
// their place: the A values follow the row masks, the decisions the column masks,
// a row's end in the pair list is the fourth word of its particle's bound, and a
// pair's row waits in the place of its C.  2D FP32, ell = 8: N <= 922 (868 with a
// place each, 914 on the pair slots per chunk).
struct StageLds {
    size_t ob, nb, bnd, sp, ncand, cmask, coff, misc, pa, pq, pc, end;
    GridLds gr;
};
__host__ __device__ inline StageLds stage_lds(int N, int ell, int dim, int tsize, int R, int cap, int keep)
{
    StageLds L;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o = align16(o + bytes);
        return at;
    };
    L.ob = take((size_t)(ell + 1) * N * dim * tsize);
    L.nb = take((size_t)(ell > 1 ? ell - 1 : 1) * N * dim * tsize);
    L.bnd = take((size_t)N * 16);
    L.sp = take((size_t)N * 8);
    L.ncand = take((size_t)N * 2);
    L.gr = grid_lds(o, N, dim);
    o = L.gr.end;
    L.cmask = take((size_t)N * (R / 64) * 8); // after the last block: the decisions
    L.coff = take((size_t)N * 2);
    L.misc = take(16);
    const size_t rows = (size_t)R * ((N + 63) / 64) * 8, vals = 2 * (size_t)cap * tsize;
    L.pa = take(rows > vals ? rows : vals); // the row masks, then the A(p, q) and the A(q, p)
    L.pq = take((size_t)keep * 2);
    L.pc = take((size_t)keep * tsize);
    L.end = o;
    return L;
}

// The pairs of one staging window by row: the first `keep` in LDS, the others in
// the window's part of the pair buffer (T values of all windows, then partners).
template <typename T> struct StagePairs {
    T *lc, *gc;
    unsigned short *lq, *gq;
    int keep;
    __device__ __forceinline__ void put(int i, int q, T c) const
    {
        if (i < keep) {
            lq[i] = (unsigned short)q;
            lc[i] = c;
        } else {
            gq[i] = (unsigned short)q;
            gc[i] = c;
        }
    }
    // before it is evaluated, pair i's row in the place of its C
    __device__ __forceinline__ void put_row(int i, int q, int l) const
    {
        T c;
        if constexpr (sizeof(T) == 4) c = __int_as_float(l);
        else c = __longlong_as_double(l);
        put(i, q, c);
    }
    __device__ __forceinline__ int row(int i) const
    {
        if constexpr (sizeof(T) == 4) return __float_as_int(c(i));
        else return (int)__double_as_longlong(c(i));
    }
    __device__ __forceinline__ int q(int i) const { return i < keep ? lq[i] : gq[i]; }
    __device__ __forceinline__ T c(int i) const { return i < keep ? lc[i] : gc[i]; }
};

// One staging window of one chain per workgroup: grid (windows, chains of the
// list a.whole), one sweep (a.rs->sweep + a.sweep_off).  The rows (particles) are
// taken in blocks of at most R whose pairs q < p in reach fit the pool; each pair
// is evaluated once, for A(p, q), A(q, p) and C(p, q), one pair per thread.  When
// every pair is done the tries are decided chunk by chunk.  Pair terms are VALU
// work (four pairings a slice); two workgroups share a CU, so one's decisions,
// a serial chain, run beside the other's pairs.  Against pair slots per chunk of 64
// tries, each pair from both sides (six pairings): 16 measuring sweeps of 256 chains
// of N = 256, M = 128, FP32, 45.2 -> 40.0 ms; 64 chains of N = 400, M = 512 stayed at 67 ms
// while their blocks took a CU alone and take 61 ms since two fit (StageLds).
template <typename T, int DIM>
__global__ void __launch_bounds__(1024) k_stage_win(SweepArgs a, ComBuf<T> B, int R, int cap, int keep, int budget)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = a.whole[blockIdx.y];
    const ChainDev ch = a.chains[c];
    const int w = blockIdx.x, tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nwv = nt >> 6;
    const int M = ch.M, N = ch.N, ell = ch.ell;
    if (w >= ch.nseg) return;
    const int m = min(ell, M - w * ell); // links of this window
    if (m < 2) return;                   // no interior bead
    const uint32_t sw = a.rs->sweep + (uint32_t)a.sweep_off;
    if (!pass_on(ch.every_st, sw)) return; // no staging pass in this sweep (move weights)
    if (cap < N) { // the host sizes the pool for every particle's partners
        if (tid == 0) atomicOr(a.status + c, 2);
        return;
    }
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const U4 xo = draw(a.seed, 0u, sw, (uint32_t)c, kOffset); // the chain's offset of this sweep
    const int off = (int)(((uint64_t)xo.x * (uint64_t)ell) >> 32);
    int s0 = off + w * ell;
    if (s0 >= M) s0 -= M;
    auto slice = [&](int t) { const int j = s0 + t; return j >= M ? j - M : j; };

    const StageLds L = stage_lds(N, ell, DIM, (int)sizeof(T), R, cap, keep);
    T *ob = reinterpret_cast<T *>(smem + L.ob); // [t][k][d], t = 0..m
    T *nb = reinterpret_cast<T *>(smem + L.nb); // [t - 1][k][d], t = 1..m-1
    float4 *bnd = reinterpret_cast<float4 *>(smem + L.bnd);
    double *const sp = reinterpret_cast<double *>(smem + L.sp);
    unsigned char *const acc = smem + L.cmask;
    unsigned short *const ncand = reinterpret_cast<unsigned short *>(smem + L.ncand);
    // row p's pairs are row_start(p) .. row_end(p) of the list
    int *const bnd_w = reinterpret_cast<int *>(smem + L.bnd) + 3;
    auto row_end = [&](int p) -> int & { return bnd_w[4 * p]; };
    auto row_start = [&](int p) { return p > 0 ? bnd_w[4 * p - 4] : 0; };
    unsigned long long *const rmask = reinterpret_cast<unsigned long long *>(smem + L.pa);
    unsigned long long *const cmask = reinterpret_cast<unsigned long long *>(smem + L.cmask);
    unsigned short *const coff = reinterpret_cast<unsigned short *>(smem + L.coff);
    int *const misc = reinterpret_cast<int *>(smem + L.misc);
    T *const pa_ = reinterpret_cast<T *>(smem + L.pa), *const pb_ = pa_ + cap;
    const size_t tri = pair_row(N);
    T *const gval = B.vals(ch, 0);
    const StagePairs<T> S{reinterpret_cast<T *>(smem + L.pc), gval + (size_t)w * tri,
                          reinterpret_cast<unsigned short *>(smem + L.pq),
                          reinterpret_cast<unsigned short *>(gval + (size_t)ch.nseg * tri) + (size_t)w * tri, keep};

    T *const gpath = reinterpret_cast<T *>(a.pos) + ch.pos_off;
    for (int t = 0; t <= m; ++t) {
        const T *src = gpath + (size_t)slice(t) * N * DIM;
        T *dst = ob + (size_t)t * N * DIM;
        for (int i = tid; i < N * DIM; i += nt) dst[i] = src[i];
    }
    __syncthreads();

    // proposals: the closed form of levy!'s recursion (src/updates/helper.jl:118-139): bead i
    // of a segment of m links from c0 to e is c0 + (i/m)(e - c0) + (m - i) S_i with
    // S_i = sum_{k <= i} sd_k xi_k / (m - k), sd_k = sqrt(2 lambda tau alpha_k),
    // alpha_k = (m - k)/(m - k + 1); Delta V of the interior beads; the window bound
    for (int p = tid; p < N; p += nt) {
        T c0[DIM], em[DIM], S[DIM], g1[2] = {T(0), T(0)};
        float ref[DIM];
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            c0[e] = ob[(size_t)p * DIM + e];
            em[e] = shift_end(c0[e], ob[((size_t)m * N + p) * DIM + e], P);
            S[e] = T(0);
            ref[e] = (float)c0[e];
        }
        T dv = T(0);
        for (int i = 1; i < m; ++i) {
            T xi[2];
            if (i & 1) {
                const U4 xr = draw(a.seed, (uint32_t)(p * M + slice(i)), sw, (uint32_t)c, kLevy);
                box_muller(xr.x, xr.y, xi[0], xi[1]);
                box_muller(xr.z, xr.w, g1[0], g1[1]);
            } else {
                xi[0] = g1[0];
                xi[1] = g1[1];
            }
            const T wi = bridge_sd(bridge_alpha<T>(m, i), P) / T(m - i);
            const T fi = T(i) / T(m);
            T rn[DIM], ro[DIM];
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                S[e] += wi * xi[e];
                rn[e] = teleport((c0[e] + fi * (em[e] - c0[e])) + T(m - i) * S[e], P);
                nb[((size_t)(i - 1) * N + p) * DIM + e] = rn[e];
                ro[e] = ob[((size_t)i * N + p) * DIM + e];
            }
            dv += -P.tau * (potV<T, DIM>(rn, P) - potV<T, DIM>(ro, P));
        }
        // bound of the old beads 0..m and the new interior beads, as offsets from bead 0
        auto offset = [&](int k, float *o) {
            const T *r = k <= m ? ob + ((size_t)k * N + p) * DIM : nb + ((size_t)(k - m - 1) * N + p) * DIM;
#pragma unroll
            for (int e = 0; e < DIM; ++e) o[e] = (float)signed_mindist(r[e], c0[e], P);
        };
        const int npts = 2 * m; // m + 1 old, m - 1 new
        float mean[DIM] = {};
        for (int k = 0; k < npts; ++k) {
            float o[DIM];
            offset(k, o);
#pragma unroll
            for (int e = 0; e < DIM; ++e) mean[e] += o[e];
        }
#pragma unroll
        for (int e = 0; e < DIM; ++e) mean[e] /= (float)npts;
        float r2 = 0.f;
        for (int k = 0; k < npts; ++k) {
            float o[DIM], d2 = 0.f;
            offset(k, o);
#pragma unroll
            for (int e = 0; e < DIM; ++e) d2 += (o[e] - mean[e]) * (o[e] - mean[e]);
            r2 = fmaxf(r2, d2);
        }
        bnd[p] = make_float4(ref[0] + mean[0], DIM > 1 ? ref[DIM - 1] + mean[DIM - 1] : 0.f, sqrtf(r2), 0.f);
        sp[p] = (double)dv;
        ncand[p] = 0;
    }
    __syncthreads();

    const float h = (float)ch.h, twoL = (float)(2.0 * ch.L), inv2L = 1.0f / twoL;
    auto bead = [&](int p, int q) {
        return [=](int t, int who, T *ro, T *rn) {
            const int k = who ? q : p;
            const T *so = ob + ((size_t)t * N + k) * DIM;
            const T *sn = (t > 0 && t < m) ? nb + ((size_t)(t - 1) * N + k) * DIM : so;
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                ro[e] = so[e];
                rn[e] = sn[e];
            }
        };
    };
    WinGrid G(smem, L.gr);
    grid_build<DIM>(G, N, h, twoL, inv2L, [&](int p, float &x, float &y, float &r) {
        const float4 b = bnd[p];
        x = b.x;
        y = b.y;
        r = b.z;
    });
    auto near = [&](int p, int q) {
        const float4 A = bnd[p], Bq = bnd[q];
        return bnd_near<DIM>(A.x, A.y, A.z, Bq.x, Bq.y, Bq.z, h, twoL, inv2L);
    };
    const int nq = (N + 63) / 64, nc = R / 64; // words of a row mask, of a column mask
    for (int pa = 0; pa < N;) {
        const int nr = min(R, N - pa), base = row_start(pa);
        for (int i = tid; i < N * nc; i += nt) cmask[i] = 0ull;
        // partners q < p in reach of each row
        if (G.ng > 0) {
            for (int i = tid; i < nr * nq; i += nt) rmask[i] = 0ull;
            __syncthreads();
            for (int l = wave; l < nr; l += nwv) {
                const int p = pa + l;
                grid_visit<DIM>(G, p, lane, [&](int q) {
                    if (q < p && near(p, q)) atomicOr(rmask + (size_t)l * nq + (q >> 6), 1ull << (q & 63));
                });
            }
            __syncthreads();
            for (int l = tid; l < nr; l += nt) {
                int cnt = 0;
                for (int k = 0; k < nq; ++k) cnt += __popcll(rmask[(size_t)l * nq + k]);
                row_end(pa + l) = cnt;
            }
        } else {
            for (int l = wave; l < nr; l += nwv) {
                const int p = pa + l;
                int cnt = 0;
                for (int q0 = 0; q0 < p; q0 += 64) {
                    const int q = q0 + lane;
                    const unsigned long long bal = __ballot(q < p && near(p, q));
                    if (lane == 0) rmask[(size_t)l * nq + (q0 >> 6)] = bal;
                    cnt += __popcll(bal);
                }
                if (lane == 0) row_end(p) = cnt;
            }
        }
        __syncthreads();
        if (wave == 0) { // prefix; the rows whose pairs fit the pool
            int sum = 0, nf = 0;
            for (int l0 = 0; l0 < nr; l0 += 64) {
                const int l = l0 + lane, v = l < nr ? row_end(pa + l) : 0;
                int tot;
                const int pre = wave_prefix(v, lane, tot);
                const bool fits = l < nr && sum + pre + v <= cap;
                if (fits) {
                    row_end(pa + l) = base + sum + pre + v;
                    ncand[pa + l] = (unsigned short)(ncand[pa + l] + v);
                }
                nf += __popcll(__ballot(fits));
                sum += tot;
            }
            if (lane == 0) misc[0] = nf;
        }
        __syncthreads();
        const int nf = misc[0];
        if (nf < 1) { // uniform; not reached while a row's pairs fit the pool (cap >= N)
            if (tid == 0) atomicOr(a.status + c, 2);
            return;
        }
        const int total = row_end(pa + nf - 1) - base;
        for (int it = tid; it < nf * nq; it += nt) {
            const int l = it / nq, wd = it - l * nq;
            if (wd * 64 >= pa + l) continue;
            const unsigned long long *mk = rmask + (size_t)l * nq;
            int s = row_start(pa + l) - base;
            for (int k = 0; k < wd; ++k) s += __popcll(mk[k]);
            unsigned long long b = mk[wd];
            while (b) {
                const int q = wd * 64 + __ffsll((long long)b) - 1;
                b &= b - 1;
                S.put_row(base + s, q, l);
                atomicOr(cmask + (size_t)q * nc + (l >> 6), 1ull << (l & 63));
                ++s;
            }
        }
        __syncthreads();
        if (wave == 0) { // where each particle's rows start
            int sum = 0;
            for (int q0 = 0; q0 < N; q0 += 64) {
                const int q = q0 + lane;
                int v = 0, tot;
                if (q < N)
                    for (int k = 0; k < nc; ++k) v += __popcll(cmask[(size_t)q * nc + k]);
                const int pre = wave_prefix(v, lane, tot);
                if (q < N) {
                    coff[q] = (unsigned short)(sum + pre);
                    ncand[q] = (unsigned short)(ncand[q] + v);
                }
                sum += tot;
            }
        }
        __syncthreads();
        for (int i = tid; i < total; i += nt) {
            const int l = S.row(base + i), p = pa + l, q = S.q(base + i);
            T Apq, Aqp, C;
            bool hit;
            if (ch.nbins >= 3) pair_window_both<T, DIM, false, true>(bead(p, q), m, P, ch.nbins, Apq, Aqp, C, hit);
            else pair_window_both<T, DIM, true, true>(bead(p, q), m, P, ch.nbins, Apq, Aqp, C, hit);
            int at = coff[q];
            for (int k = 0; k < (l >> 6); ++k) at += __popcll(cmask[(size_t)q * nc + k]);
            at += __popcll(cmask[(size_t)q * nc + (l >> 6)] & ((1ull << (l & 63)) - 1ull));
            pa_[i] = Apq;
            pb_[at] = Aqp;
            S.put(base + i, hit ? q | 0x8000 : q, C);
        }
        __syncthreads();
        for (int x = tid; x < N; x += nt) { // partners by index: the particle's own row, then the rows that name it
            double s = sp[x];
            if (x >= pa && x < pa + nf)
                for (int i = row_start(x) - base; i < row_end(x) - base; ++i) s += (double)pa_[i];
            int n = 0;
            for (int k = 0; k < nc; ++k) n += __popcll(cmask[(size_t)x * nc + k]);
            for (int i = coff[x]; i < coff[x] + n; ++i) s += (double)pb_[i];
            sp[x] = s;
        }
        __syncthreads();
        pa += nf;
    }
    // decisions, chunk by chunk, by one wave
    if (wave == 0) {
        int lacc = 0;
        for (int pa = 0; pa < N;) {
            const int p = pa + lane, v = p < N ? (int)ncand[p] : 0;
            int tot;
            const int pre = wave_prefix(v, lane, tot);
            const int nf = __popcll(__ballot(p < N && pre + v <= budget));
            if (nf < 1) { // not reached while a try's partners fit (budget >= N)
                if (lane == 0) atomicOr(a.status + c, 2);
                for (int k = p; k < N; k += 64) acc[k] = 0;
                break;
            }
            bool whole;
            const bool in = lane < nf;
            const T u = Uniform<T>::get(draw(a.seed, (uint32_t)(p * M + s0), sw, (uint32_t)c, kLevyAccept).x);
            const unsigned long long am = chunk_decide<T>([&](int i) { return S.q(i); }, [&](int i) { return S.c(i); },
                                                          in ? row_start(p) : 0, in ? row_end(p) : 0, in ? sp[p] : 0.0, u,
                                                          pa, nf, acc, whole);
            if (!whole && lane == 0) atomicOr(a.status + c, 2);
            if (in) acc[p] = (unsigned char)((am >> lane) & 1ull);
            __builtin_amdgcn_wave_barrier(); // the next chunk reads the decisions
            lacc += __popcll(am);
            pa += nf;
        }
        if (lane == 0) atomicAdd(a.chain_meas + (size_t)c * (kNQ + kCnt) + kNQ, (double)lacc);
    }
    __syncthreads();
    // accepted proposals to HBM
    for (int i = 1; i < m; ++i) {
        T *dst = gpath + (size_t)slice(i) * N * DIM;
        const T *src = nb + (size_t)(i - 1) * N * DIM;
        for (int k = tid; k < N; k += nt)
            if (acc[k]) {
#pragma unroll
                for (int e = 0; e < DIM; ++e) dst[k * DIM + e] = src[k * DIM + e];
            }
    }
}

// --- centre of mass ---

// The try of particle p in this sweep: shift (words 0..dim-1) and uniform (word 2).
template <typename T, int DIM>
__device__ __forceinline__ void com_try(const SweepArgs &a, int c, uint32_t sw, int p, T *d, T &u)
{
    const U4 y = draw(a.seed, (uint32_t)p, sw, (uint32_t)c, kCom);
    const T s2 = (T)a.com_step[c] * T(2);
    d[0] = s2 * (Uniform<T>::get(y.x) - T(0.5));
    if (DIM > 1) d[1] = s2 * (Uniform<T>::get(y.y) - T(0.5));
    u = Uniform<T>::get(y.z);
}

// Whether the bounds of two particles come within reach in one of the four
// pairings of old and shifted beads.
template <typename T, int DIM>
__device__ __forceinline__ bool com_near(float4 A, const T *da, float4 B, const T *db, float h, float twoL, float inv2L)
{
    float fa[2], fb[2];
    fa[0] = (float)da[0];
    fb[0] = (float)db[0];
    fa[1] = DIM > 1 ? (float)da[DIM - 1] : 0.f;
    fb[1] = DIM > 1 ? (float)db[DIM - 1] : 0.f;
    return bnd_near4<DIM>(A, fa, B, fb, h, twoL, inv2L);
}

constexpr int kBndPart = 64; // particles per workgroup of k_com_bounds

// The tries' shifts and the bounds of the old beads: grid (particle blocks,
// chains), one wave per window of 64 particles (the particles of a slice are
// consecutive in memory), up to 16 waves: a bound is a chain of dependent loads.
// With 4 waves a workgroup 64 chains of N = 400, M = 256 took 121 us, sparse chains
// of N = 97, M = 128 39 us of a sweep of 390.  A window's bound: the middle of the beads'
// extent, and the largest distance from it; a ring's: the same of its windows'
// bounds, unwrapped against window 0's.
template <typename T, int DIM> __global__ void __launch_bounds__(1024) k_com_bounds(SweepArgs a, ComBuf<T> B)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = a.whole[blockIdx.y];
    const ChainDev ch = a.chains[c];
    const int N = ch.N, M = ch.M, lc = com_win_len(M), nw = com_nwin(M);
    const int l = threadIdx.x & 63, p = blockIdx.x * kBndPart + l;
    if ((int)blockIdx.x * kBndPart >= N) return;
    const uint32_t sw = a.rs->sweep + (uint32_t)a.sweep_off;
    if (!pass_on(ch.every_com, sw)) return; // no centre-of-mass pass in this sweep
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    float4 *s_b = reinterpret_cast<float4 *>(smem); // [window][64]
    const T *const gpath = reinterpret_cast<const T *>(a.pos) + ch.pos_off;
    const size_t part = (size_t)ch.part_base + p;
    for (int w = threadIdx.x >> 6; w < nw; w += (int)blockDim.x >> 6) {
        if (p >= N) continue;
        const int s0 = w * lc, m = min(lc, M - s0);
        T r0[DIM];
        float lo[DIM], hi[DIM];
        auto offset = [&](int t, float *o) {
            int j = s0 + t;
            if (j >= M) j -= M;
            const T *r = gpath + ((size_t)j * N + p) * DIM;
#pragma unroll
            for (int e = 0; e < DIM; ++e) o[e] = (float)signed_mindist(r[e], r0[e], P);
        };
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            r0[e] = gpath[((size_t)s0 * N + p) * DIM + e];
            lo[e] = hi[e] = 0.f;
        }
        for (int t = 1; t <= m; ++t) {
            float o[DIM];
            offset(t, o);
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                lo[e] = fminf(lo[e], o[e]);
                hi[e] = fmaxf(hi[e], o[e]);
            }
        }
        float r2 = 0.f;
        for (int t = 0; t <= m; ++t) {
            float o[DIM], d2 = 0.f;
            offset(t, o);
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                const float x = o[e] - 0.5f * (lo[e] + hi[e]);
                d2 += x * x;
            }
            r2 = fmaxf(r2, d2);
        }
        const float4 b = make_float4((float)r0[0] + 0.5f * (lo[0] + hi[0]),
                                     DIM > 1 ? (float)r0[DIM - 1] + 0.5f * (lo[DIM - 1] + hi[DIM - 1]) : 0.f,
                                     sqrtf(r2) * 1.00001f, 0.f);
        s_b[w * 64 + l] = b;
        B.wbnd[part * B.nwin + w] = b;
    }
    __syncthreads();
    if (threadIdx.x >= 64 || p >= N) return;
    const float twoL = (float)(2.0 * ch.L), inv2L = 1.0f / twoL;
    const float4 b0 = s_b[l];
    float lx = 0.f, hx = 0.f, ly = 0.f, hy = 0.f;
    for (int w = 1; w < nw; ++w) {
        const float4 b = s_b[w * 64 + l];
        const float x = mi_f(b.x - b0.x, twoL, inv2L), y = DIM > 1 ? mi_f(b.y - b0.y, twoL, inv2L) : 0.f;
        lx = fminf(lx, x), hx = fmaxf(hx, x);
        ly = fminf(ly, y), hy = fmaxf(hy, y);
    }
    const float cx = 0.5f * (lx + hx), cy = 0.5f * (ly + hy);
    float r = 0.f;
    for (int w = 0; w < nw; ++w) {
        const float4 b = s_b[w * 64 + l];
        const float x = mi_f(b.x - b0.x, twoL, inv2L) - cx, y = (DIM > 1 ? mi_f(b.y - b0.y, twoL, inv2L) : 0.f) - cy;
        r = fmaxf(r, sqrtf(x * x + y * y) + b.z);
    }
    B.rbnd[part] = make_float4(b0.x + cx, b0.y + cy, r * 1.00001f, 0.f);
    T d[DIM], u;
    com_try<T, DIM>(a, c, sw, p, d, u);
#pragma unroll
    for (int e = 0; e < DIM; ++e) B.shift[part * 2 + e] = d[e];
}

// The listed partners q < p of each particle, by index: grid (blocks of 64
// particles, chains), one wave per particle and 64 partners at a time, 16 waves.
template <typename T, int DIM> __global__ void __launch_bounds__(1024) k_com_pairs(SweepArgs a, ComBuf<T> B)
{
    const int c = a.whole[blockIdx.y];
    const ChainDev ch = a.chains[c];
    const int N = ch.N, lane = threadIdx.x & 63;
    if (!pass_on(ch.every_com, a.rs->sweep + (uint32_t)a.sweep_off)) return;
    const float h = (float)ch.h, twoL = (float)(2.0 * ch.L), inv2L = 1.0f / twoL;
    const float4 *rb = B.rbnd + ch.part_base;
    const T *sd = B.shift + (size_t)ch.part_base * 2;
    const int p1 = min(N, ((int)blockIdx.x + 1) * 64);
    for (int p = (int)blockIdx.x * 64 + (threadIdx.x >> 6); p < p1; p += (int)blockDim.x >> 6) {
        unsigned short *row = B.row(ch, p);
        const float4 A = rb[p];
        const T da[2] = {sd[p * 2], DIM > 1 ? sd[p * 2 + 1] : T(0)};
        int n = 0;
        for (int q0 = 0; q0 < p; q0 += 64) {
            const int q = q0 + lane;
            const bool ok = q < p && com_near<T, DIM>(A, da, rb[q], sd + q * 2, h, twoL, inv2L);
            const unsigned long long bal = __ballot(ok);
            if (ok) row[n + __popcll(bal & ((1ull << lane) - 1ull))] = (unsigned short)q;
            n += __popcll(bal);
        }
        if (lane == 0) B.cnt[ch.part_base + p] = n;
    }
}

// LDS of k_com_spec for blocks of R particles (rows) and a pool of cap pairs:
// beads of the window's slices, shifts, sums, masks of the rows' partners in
// reach (words of 64 list entries) and of each particle's rows (words of 64
// rows), then the pool: row, list index, partner and the two A values.
struct ComSpecLds {
    size_t ob, sd, sp, roff, cmask, coff, misc, prow, pk, pq, pa, pb, end;
};
__host__ __device__ inline ComSpecLds com_spec_lds(int N, int lc, int dim, int tsize, int R, int cap)
{
    ComSpecLds L;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o = align16(o + bytes);
        return at;
    };
    const int nq = (N + 63) / 64;
    L.ob = take((size_t)(lc + 1) * N * dim * tsize);
    L.sd = take((size_t)N * dim * tsize);
    L.sp = take((size_t)N * 8);
    L.roff = take((size_t)(R + 1) * 4);
    L.cmask = take((size_t)N * (R / 64) * 8);
    L.coff = take((size_t)N * 2);
    L.misc = take(16);
    L.prow = take((size_t)cap * 2);
    L.pk = take((size_t)cap * 2);
    L.pq = take((size_t)cap * 2);
    const size_t rows = (size_t)R * nq * 8, vals = (size_t)cap * tsize;
    L.pa = take(rows > vals ? rows : vals); // the row masks, then the A(p, q)
    L.pb = take(vals);
    L.end = o;
    return L;
}

// Phase 1 of the centre-of-mass moves: one workgroup per (window, chain),
// windows of com_win_len(M) slices from slice 0, every try against the
// configuration at the start of the phase.  Blocks of at most R particles whose
// pairs in reach fit the pool; per block the pairs are found from the list by
// window bounds, evaluated one per thread, and each particle's sum takes its
// partners by index (the block's own rows first, then the rows that name it).
// The pair terms are VALU work, four pairings of two beads a slice; a pool of the
// whole window's pairs keeps the threads evenly loaded.  All C here instead of those
// of accepted partners in k_com_dec: more pairs, but on every CU (see k_com_dec).
template <typename T, int DIM>
__global__ void __launch_bounds__(1024) k_com_spec(SweepArgs a, ComBuf<T> B, int R, int cap)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = a.whole[blockIdx.y];
    const ChainDev ch = a.chains[c];
    const int w = blockIdx.x, tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nwv = nt >> 6;
    const int M = ch.M, N = ch.N, lc = com_win_len(M);
    if (w * lc >= M) return;
    const int m = min(lc, M - w * lc), s0 = w * lc;
    if (!pass_on(ch.every_com, a.rs->sweep + (uint32_t)a.sweep_off)) return; // no centre-of-mass pass in this sweep
    if (cap < N) { // the host sizes the pool for every particle's partners
        if (tid == 0) atomicOr(a.status + c, 2);
        return;
    }
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const ComSpecLds L = com_spec_lds(N, lc, DIM, (int)sizeof(T), R, cap);
    T *const ob = reinterpret_cast<T *>(smem + L.ob), *const sd = reinterpret_cast<T *>(smem + L.sd);
    double *const sp = reinterpret_cast<double *>(smem + L.sp);
    unsigned long long *const rmask = reinterpret_cast<unsigned long long *>(smem + L.pa);
    unsigned long long *const cmask = reinterpret_cast<unsigned long long *>(smem + L.cmask);
    int *const roff = reinterpret_cast<int *>(smem + L.roff), *const misc = reinterpret_cast<int *>(smem + L.misc);
    unsigned short *const coff = reinterpret_cast<unsigned short *>(smem + L.coff);
    unsigned short *const prow = reinterpret_cast<unsigned short *>(smem + L.prow);
    unsigned short *const pk = reinterpret_cast<unsigned short *>(smem + L.pk);
    unsigned short *const pq = reinterpret_cast<unsigned short *>(smem + L.pq);
    T *const pa_ = reinterpret_cast<T *>(smem + L.pa), *const pb_ = reinterpret_cast<T *>(smem + L.pb);
    const T *const gpath = reinterpret_cast<const T *>(a.pos) + ch.pos_off;
    for (int t = 0; t <= m; ++t) {
        const int j = (s0 + t) % M;
        const T *src = gpath + (size_t)j * N * DIM;
        T *dst = ob + (size_t)t * N * DIM;
        for (int i = tid; i < N * DIM; i += nt) dst[i] = src[i];
    }
    const size_t part = (size_t)ch.part_base;
    for (int p = tid; p < N; p += nt)
#pragma unroll
        for (int e = 0; e < DIM; ++e) sd[p * DIM + e] = B.shift[(part + p) * 2 + e];
    __syncthreads();
    for (int p = tid; p < N; p += nt) {
        T dv = T(0);
        for (int t = 0; t < m; ++t) {
            T ro[DIM], rn[DIM];
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                ro[e] = ob[((size_t)t * N + p) * DIM + e];
                rn[e] = teleport(ro[e] + sd[p * DIM + e], P);
            }
            dv += -P.tau * (potV<T, DIM>(rn, P) - potV<T, DIM>(ro, P));
        }
        sp[p] = (double)dv;
    }
    const float h = (float)ch.h, twoL = (float)(2.0 * ch.L), inv2L = 1.0f / twoL;
    const int nq = (N + 63) / 64, nc = R / 64; // words of a row mask, of a column mask
    T *const cval = B.vals(ch, w);
    for (int pa = 0; pa < N;) {
        const int nr = min(R, N - pa);
        for (int i = tid; i < N * nc; i += nt) cmask[i] = 0ull;
        // partners in reach of each row; the others' C is zero
        for (int l = wave; l < nr; l += nwv) {
            const int p = pa + l, n = B.cnt[part + p];
            const unsigned short *row = B.row(ch, p);
            const float4 bp = B.wbnd[(part + p) * B.nwin + w];
            int cnt = 0;
            for (int k0 = 0; k0 < n; k0 += 64) {
                const int k = k0 + lane;
                bool ok = false;
                if (k < n) {
                    const int q = row[k];
                    ok = com_near<T, DIM>(bp, sd + p * DIM, B.wbnd[(part + q) * B.nwin + w], sd + q * DIM, h, twoL, inv2L);
                    if (!ok) cval[pair_row(p) + k] = T(0);
                }
                const unsigned long long bal = __ballot(ok);
                if (lane == 0) rmask[(size_t)l * nq + (k0 >> 6)] = bal;
                cnt += __popcll(bal);
            }
            if (lane == 0) roff[l + 1] = cnt;
        }
        __syncthreads();
        if (wave == 0) { // prefix; the rows whose pairs fit
            int base = 0, nf = 0;
            for (int l0 = 0; l0 < nr; l0 += 64) {
                const int l = l0 + lane, v = l < nr ? roff[l + 1] : 0;
                int tot;
                const int pre = wave_prefix(v, lane, tot);
                if (l < nr) roff[l + 1] = base + pre + v;
                nf += __popcll(__ballot(l < nr && base + pre + v <= cap));
                base += tot;
            }
            if (lane == 0) {
                roff[0] = 0;
                misc[0] = nf;
            }
        }
        __syncthreads();
        const int nf = misc[0], total = roff[nf];
        if (nf < 1) { // uniform; not reached while a row's pairs fit the pool (cap >= N)
            if (tid == 0) atomicOr(a.status + c, 2);
            return;
        }
        for (int l = wave; l < nf; l += nwv) {
            const int p = pa + l, n = B.cnt[part + p];
            const unsigned short *row = B.row(ch, p);
            int at = roff[l];
            for (int k0 = 0; k0 < n; k0 += 64) {
                const unsigned long long bal = rmask[(size_t)l * nq + (k0 >> 6)];
                if ((bal >> lane) & 1ull) {
                    const int s = at + __popcll(bal & ((1ull << lane) - 1ull)), q = row[k0 + lane];
                    prow[s] = (unsigned short)l;
                    pk[s] = (unsigned short)(k0 + lane);
                    pq[s] = (unsigned short)q;
                    atomicOr(cmask + (size_t)q * nc + (l >> 6), 1ull << (l & 63));
                }
                at += __popcll(bal);
            }
        }
        __syncthreads();
        if (wave == 0) { // where each particle's rows start
            int base = 0;
            for (int q0 = 0; q0 < N; q0 += 64) {
                const int q = q0 + lane;
                int v = 0, tot;
                if (q < N)
                    for (int k = 0; k < nc; ++k) v += __popcll(cmask[(size_t)q * nc + k]);
                const int pre = wave_prefix(v, lane, tot);
                if (q < N) coff[q] = (unsigned short)(base + pre);
                base += tot;
            }
        }
        __syncthreads();
        for (int i = tid; i < total; i += nt) {
            const int l = prow[i], p = pa + l, q = pq[i];
            auto bead = [&](int t, int who, T *ro, T *rn) {
                const int k = who ? q : p;
#pragma unroll
                for (int e = 0; e < DIM; ++e) {
                    ro[e] = ob[((size_t)t * N + k) * DIM + e];
                    rn[e] = teleport(ro[e] + sd[k * DIM + e], P);
                }
            };
            T Apq, Aqp, C;
            bool hit;
            if (ch.nbins >= 3) pair_window_both<T, DIM, false>(bead, m, P, ch.nbins, Apq, Aqp, C, hit);
            else pair_window_both<T, DIM, true>(bead, m, P, ch.nbins, Apq, Aqp, C, hit);
            int at = coff[q];
            for (int k = 0; k < (l >> 6); ++k) at += __popcll(cmask[(size_t)q * nc + k]);
            at += __popcll(cmask[(size_t)q * nc + (l >> 6)] & ((1ull << (l & 63)) - 1ull));
            pa_[i] = Apq;
            pb_[at] = Aqp;
            cval[pair_row(p) + pk[i]] = !hit ? T(0) : (C == T(0) ? T(-0.0) : C);
        }
        __syncthreads();
        for (int x = tid; x < N; x += nt) {
            double s = sp[x];
            if (x >= pa && x < pa + nf)
                for (int i = roff[x - pa]; i < roff[x - pa + 1]; ++i) s += (double)pa_[i];
            int n = 0;
            for (int k = 0; k < nc; ++k) n += __popcll(cmask[(size_t)x * nc + k]);
            for (int i = coff[x]; i < coff[x] + n; ++i) s += (double)pb_[i];
            sp[x] = s;
        }
        __syncthreads();
        pa += nf;
    }
    for (int p = tid; p < N; p += nt) B.spec[(part + p) * B.nwin + w] = sp[p];
}

// LDS of k_com_dec: the tries' sums, uniforms and decisions, then two chunk
// buffers of cap pairs each.
struct ComDecLds {
    size_t spec, su, acc, off, ck[2], end;
};
__host__ __device__ inline size_t com_dec_chunk(int cap, int tsize)
{
    return align16((size_t)cap * tsize) + align16((size_t)cap * 2) + align16((kChunk + 1) * 4) + 16;
}
__host__ __device__ inline ComDecLds com_dec_lds(int N, int tsize, int cap)
{
    ComDecLds L;
    size_t o = 0;
    L.spec = o;
    o = align16(o + (size_t)N * 8);
    L.su = o;
    o = align16(o + (size_t)N * tsize);
    L.acc = o;
    o = align16(o + (size_t)N);
    for (int k = 0; k < 2; ++k) {
        L.ck[k] = o;
        o += com_dec_chunk(cap, tsize);
    }
    L.end = o;
    return L;
}

// Phase 2 of the centre-of-mass moves: one workgroup per chain.  Per chunk of 64
// tries the listed pairs' C values are added over the windows (window order; zero
// outside reach) into LDS, and one wave decides the chunk in rounds while the
// other waves fetch the next chunk's.  What bounds it is the serial chain of
// rounds of that wave.  With 64 chains (N = 400, M = 512, FP32) on 64 of 256 CUs it
// took 1.78 ms a sweep while it evaluated the C terms itself, 0.21 ms now; 16
// measuring sweeps 77.5 -> 65.0 ms, and 49.3 -> 45.2 ms for 256 chains of N = 256,
// M = 128.  cacc[part]: 1 when the particle's try was accepted.
template <typename T, int DIM>
__global__ void __launch_bounds__(1024) k_com_dec(SweepArgs a, ComBuf<T> B, int cap, unsigned char *cacc)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = a.whole[blockIdx.x];
    const ChainDev ch = a.chains[c];
    const int N = ch.N, nw = com_nwin(ch.M), tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6;
    const int nwv = nt >> 6;
    const uint32_t sw = a.rs->sweep + (uint32_t)a.sweep_off;
    if (!pass_on(ch.every_com, sw)) return; // no centre-of-mass pass in this sweep: no tries
    if (cap < N) {
        if (tid == 0) atomicOr(a.status + c, 2);
        return;
    }
    const ComDecLds L = com_dec_lds(N, (int)sizeof(T), cap);
    double *const s_spec = reinterpret_cast<double *>(smem + L.spec);
    T *const su = reinterpret_cast<T *>(smem + L.su);
    unsigned char *const acc = smem + L.acc;
    const size_t part = (size_t)ch.part_base;
    struct Chunk {
        T *c;
        unsigned short *q;
        int *off, *n;
    };
    auto chunk = [&](int k) {
        unsigned char *s = smem + L.ck[k];
        Chunk x;
        x.c = reinterpret_cast<T *>(s);
        s += align16((size_t)cap * sizeof(T));
        x.q = reinterpret_cast<unsigned short *>(s);
        s += align16((size_t)cap * 2);
        x.off = reinterpret_cast<int *>(s);
        x.n = reinterpret_cast<int *>(s + align16((kChunk + 1) * 4));
        return x;
    };
    // the pairs of the chunk that starts at try pa, by waves w0, w0 + 1, ...: as many tries as the
    // buffer holds (each wave takes the same prefix of the counts)
    auto fetch = [&](const Chunk &x, int pa, int w0) {
        if (pa >= N) return;
        const int v = pa + lane < N ? B.cnt[part + pa + lane] : 0;
        int tot;
        const int pre = wave_prefix(v, lane, tot);
        const int nf = __popcll(__ballot(pa + lane < N && pre + v <= cap));
        if (wave == w0) {
            x.off[lane] = pre;
            if (lane == nf - 1) x.off[nf] = pre + v;
            if (lane == 0) *x.n = nf;
        }
        for (int l = wave - w0; l < nf; l += nwv - w0) {
            const int p = pa + l, n = __shfl(v, l, 64), o = __shfl(pre, l, 64);
            const unsigned short *row = B.row(ch, p);
            const T *val = B.vals(ch, 0) + pair_row(p);
            const size_t step = pair_row(N);
            for (int k = lane; k < n; k += 64) {
                T s = T(0);
                bool hit = false;
#pragma unroll 8
                for (int w = 0; w < nw; ++w) {
                    const T y = val[(size_t)w * step + k];
                    hit = hit || y != T(0) || is_neg_zero(y);
                    s = add_(s, y);
                }
                x.c[o + k] = s;
                x.q[o + k] = (unsigned short)(row[k] | (hit ? 0x8000 : 0));
            }
        }
    };
    fetch(chunk(0), 0, 0);
    for (int p = tid; p < N; p += nt) {
        double s = 0.0;
        for (int w = 0; w < nw; ++w) s += B.spec[(part + p) * B.nwin + w];
        s_spec[p] = s;
        T d[DIM], u;
        com_try<T, DIM>(a, c, sw, p, d, u);
        su[p] = u;
        acc[p] = 0;
    }
    __syncthreads();
    int nacc = 0;
    for (int pa = 0, k = 0; pa < N; k ^= 1) {
        const Chunk x = chunk(k);
        const int nf = *x.n;
        if (nf < 1) { // uniform; not reached while a try's partners fit (cap >= N)
            if (tid == 0) atomicOr(a.status + c, 2);
            break;
        }
        if (wave > 0) {
            fetch(chunk(k ^ 1), pa + nf, 1);
        } else {
            bool whole;
            const unsigned long long am = chunk_decide<T>([&](int i) { return (int)x.q[i]; }, [&](int i) { return x.c[i]; },
                                                          lane < nf ? x.off[lane] : 0, lane < nf ? x.off[lane + 1] : 0,
                                                          lane < nf ? s_spec[pa + lane] : 0.0, lane < nf ? su[pa + lane] : T(0),
                                                          pa, nf, acc, whole);
            if (!whole && lane == 0) atomicOr(a.status + c, 2);
            if (lane < nf) acc[pa + lane] = (unsigned char)((am >> lane) & 1ull);
            nacc += __popcll(am);
        }
        __syncthreads();
        pa += nf;
    }
    for (int p = tid; p < N; p += nt) cacc[part + p] = acc[p];
    if (tid == 0) {
        double *out = a.chain_meas + (size_t)c * (kNQ + kCnt);
        out[kNQ + 1] += (double)nacc;
        out[kNQ + 2] += (double)N;
    }
}

// The accepted centre-of-mass tries move their rings: grid (bead blocks,
// chains), one thread per (slice, particle).
template <typename T, int DIM>
__global__ void __launch_bounds__(256) k_com_apply(SweepArgs a, const unsigned char *cacc, const T *cshift)
{
    const int c = a.whole[blockIdx.y];
    const ChainDev ch = a.chains[c];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)ch.M * ch.N) return;
    const int j = (int)(i / ch.N), k = (int)(i - (long long)j * ch.N);
    const size_t q = (size_t)ch.part_base + k;
    // the flags are those of this sweep's k_com_dec only when the pass ran
    if (!pass_on(ch.every_com, a.rs->sweep + (uint32_t)a.sweep_off) || !cacc[q]) return;
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const Path<T, DIM, true> path{reinterpret_cast<T *>(a.pos) + ch.pos_off, ch.M, ch.N};
    T r[DIM];
    path.get(k, j, r);
#pragma unroll
    for (int e = 0; e < DIM; ++e) r[e] = teleport(r[e] + cshift[q * 2 + e], P);
    path.put(k, j, r);
}

// --- estimators ---

struct MeasWinLds {
    size_t ob, bnd;
    GridLds gr;
    ChunkLds ck;
};
__host__ __device__ inline MeasWinLds meas_win_lds(int N, int lc, int dim, int tsize, int cap)
{
    MeasWinLds L;
    size_t o = 0;
    L.ob = o;
    o = align16(o + (size_t)(lc + 1) * N * dim * tsize);
    L.bnd = o;
    o = align16(o + (size_t)N * 16);
    L.gr = grid_lds(o, N, dim);
    L.ck = chunk_lds(L.gr.end, N, cap);
    return L;
}

// Whether the LDS of a workgroup holds the smallest blocks and pools of all four kernels that a
// window chain runs on (N, ell and lc the largest of the chains that share their launches): 160 KiB,
// of which k_meas_win has kMeasWinStatic in arrays of its own.
constexpr size_t kMeasWinStatic = 32 * sizeof(double);
inline bool win_fits(int N, int ell, int lc, int dim, int tsize)
{
    const size_t most = 160 * 1024;
    return stage_lds(N, ell, dim, tsize, 64, N, 0).end <= most && com_spec_lds(N, lc, dim, tsize, 64, N).end <= most &&
           com_dec_lds(N, tsize, N).end <= most && meas_win_lds(N, lc, dim, tsize, N).ck.end + kMeasWinStatic <= most;
}

// Pair energy and pair virial of one pair over the slices 0 .. m - 1 of a window,
// added to su and rg with weight wq per link and stencil multiplicity: the terms of
// pair_energy_bead.  Each bead pair's distance and exponential serve the link
// before it and the link after it (16 measuring sweeps of 256 chains of N = 256,
// M = 128, FP32: 40.0 ms with two exponentials per link, 39.4 ms with one per slice).
// bead(t, x, y): the pair's beads at slice t.
template <typename T, int DIM, typename BeadFn>
__device__ __forceinline__ void pair_energy_window(BeadFn bead, int m, const Prm<T> &P, int nbins, double wq, double inv_s2,
                                                   double &su, double &rg)
{
    T x[DIM], y[DIM];
    bead(0, x, y);
    T r2 = dist2_min<T, DIM>(y, x, P);
    double ea = (double)ex(-r2 * P.inv2s2);
    for (int t = 0; t < m; ++t) {
        const bool in = r2 <= P.h2;
        const double wt = nbins >= 3 ? wq : wq * (double)stencil_mult<T, DIM>(x, y, P, nbins);
        bead(t + 1, x, y);
        const T s2 = dist2_min<T, DIM>(y, x, P);
        const double eb = (double)ex(-s2 * P.inv2s2);
        if (in) {
            su += wt * (ea + eb);
            rg += wt * (-((double)r2 * inv_s2) * ea - ((double)s2 * inv_s2) * eb);
        }
        r2 = s2;
        ea = eb;
    }
}

// Estimators of Gaussian-pair chains after a sweep, by the centre-of-mass
// windows: one 512-thread workgroup per (window, chain of a.ids).  The terms of
// measure_chain for the beads of slices s0 .. s0 + m - 1: kinetic link to the
// next slice, V, r.grad V, dV/d omega, the radial and Cartesian histograms,
// and the pair energy and pair virial of each bead as pair_energy_bead takes
// them (every neighbour within the cut-off at the bead's slice, weight
// tau/4 times its stencil multiplicity), the neighbours found from window
// bounds.  part[(y * nwin + w) * 6]: the window's sums (link, V, r.grad V,
// S_U/g, pair virial, dV/d omega), folded in window order by k_meas_fold.
template <typename T, int DIM> __global__ void __launch_bounds__(512) k_meas_win(MeasArgs a, int nwin, int cap)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double wbuf[kMeasWinStatic / sizeof(double)];
    if (!split_measured(a)) return;
    const int y = blockIdx.y, c = a.ids[y], w = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const ChainDev ch = a.chains[c];
    const int N = ch.N, M = ch.M, lc = com_win_len(M);
    double *out = a.part + ((size_t)y * nwin + w) * 6;
    if (w * lc >= M || cap < N) { // no such window for this chain (the host sizes cap >= N)
        if (tid < 6) out[tid] = 0.0;
        return;
    }
    const int m = min(lc, M - w * lc), s0 = w * lc;
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(a.prm)[c];
    const MeasWinLds L = meas_win_lds(N, lc, DIM, (int)sizeof(T), cap);
    T *ob = reinterpret_cast<T *>(smem + L.ob);
    float4 *bnd = reinterpret_cast<float4 *>(smem + L.bnd);
    ChunkPtr X(smem, L.ck);
    const T *const gpath = reinterpret_cast<const T *>(a.pos) + ch.pos_off;
    for (int t = 0; t <= m; ++t) {
        const int j = (s0 + t) % M;
        const T *src = gpath + (size_t)j * N * DIM;
        T *dst = ob + (size_t)t * N * DIM;
        for (int i = tid; i < N * DIM; i += nt) dst[i] = src[i];
    }
    __syncthreads();
    for (int p = tid; p < N; p += nt) {
        float mean[DIM] = {};
        for (int t = 0; t <= m; ++t) {
#pragma unroll
            for (int e = 0; e < DIM; ++e)
                mean[e] += (float)signed_mindist(ob[((size_t)t * N + p) * DIM + e], ob[(size_t)p * DIM + e], P);
        }
#pragma unroll
        for (int e = 0; e < DIM; ++e) mean[e] /= (float)(m + 1);
        float r2 = 0.f;
        for (int t = 0; t <= m; ++t) {
            float d2 = 0.f;
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                const float o = (float)signed_mindist(ob[((size_t)t * N + p) * DIM + e], ob[(size_t)p * DIM + e], P) - mean[e];
                d2 += o * o;
            }
            r2 = fmaxf(r2, d2);
        }
        bnd[p] = make_float4((float)ob[(size_t)p * DIM] + mean[0],
                             DIM > 1 ? (float)ob[(size_t)p * DIM + DIM - 1] + mean[DIM - 1] : 0.f, sqrtf(r2), 0.f);
    }
    // single-bead terms, one thread per (particle, slice)
    double l = 0.0, v = 0.0, g = 0.0, r2w = 0.0, su = 0.0, rgp = 0.0;
    for (int it = tid; it < N * m; it += nt) {
        const int p = it / m, t = it - p * m;
        T r0[DIM], r1[DIM];
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            r0[e] = ob[((size_t)t * N + p) * DIM + e];
            r1[e] = ob[((size_t)(t + 1) * N + p) * DIM + e];
        }
        T dd = T(0);
#pragma unroll
        for (int e = 0; e < DIM; ++e) {
            const T dx = mindist(r0[e], r1[e], P);
            dd += dx * dx;
        }
        l += (double)dd;
        v += (double)potV<T, DIM>(r0, P);
        g += (double)rgradV<T, DIM>(r0, P);
        if (ch.pot == kPotHarmonic) r2w += (double)dVdomega<T, DIM>(r0, ch.omega);
        if (a.radial_bins > 0) {
            T rr = r0[0] * r0[0];
            if (DIM > 1) rr += r0[1] * r0[1];
            const double qb = (double)sq(rr) * a.radial_winv;
            if (qb < (double)a.radial_bins) atomicAdd(&a.radial[(size_t)c * a.radial_bins + (int)qb], 1ull);
        }
        if (a.cart_bins > 0) {
            const double bw = (2.0 * ch.L) / a.cart_bins;
            long long idx = 0, stride = 1;
            bool ok = true;
#pragma unroll
            for (int e = 0; e < DIM; ++e) {
                const long long ib = (long long)floor(((double)r0[e] + ch.L) / bw);
                ok = ok && ib > 0 && ib < a.cart_bins + 1;
                idx += (ib - 1) * stride;
                stride *= a.cart_bins;
            }
            if (ok) atomicAdd(&a.cart[(size_t)c * stride + idx], 1ull);
        }
    }
    __syncthreads();
    // pair terms: bead (p, t) with each neighbour q within the cut-off at slice t.  The term is
    // symmetric in p and q (distances, stencil multiplicity, the link to the next slice), so each
    // unordered pair is taken once, from its lower index, with the weight of both ends
    const float h = (float)ch.h, twoL = (float)(2.0 * ch.L), inv2L = 1.0f / twoL;
    const double inv_s2 = 1.0 / (ch.sigma * ch.sigma), wq = 2.0 * (0.5 * (0.5 * (double)P.tau));
    WinGrid G(smem, L.gr);
    grid_build<DIM>(G, N, h, twoL, inv2L, [&](int p, float &x, float &y, float &r) {
        const float4 b = bnd[p];
        x = b.x;
        y = b.y;
        r = b.z;
    });
    for (int pa = 0; pa < N;) {
        const int nf = chunk_slots<DIM>(X, pa, N, cap, kChunk, [&](int p, int q) {
            if (q <= p) return false;
            const float4 A = bnd[p], B = bnd[q];
            return bnd_near<DIM>(A.x, A.y, A.z, B.x, B.y, B.z, h, twoL, inv2L);
        }, &G);
        if (nf < 1) break; // uniform; not reached (cap >= N)
        const int total = X.misc[1];
        for (int i = tid; i < total; i += nt) {
            const int p = pa + X.po[i], q = X.pq[i];
            const T *rp = ob + (size_t)p * DIM, *rq = ob + (size_t)q * DIM;
            pair_energy_window<T, DIM>([&](int t, T *x, T *y) {
#pragma unroll
                for (int e = 0; e < DIM; ++e) {
                    x[e] = rp[(size_t)t * N * DIM + e];
                    y[e] = rq[(size_t)t * N * DIM + e];
                }
            }, m, P, ch.nbins, wq, inv_s2, su, rgp);
        }
        __syncthreads();
        pa += nf;
    }
    const double sl = block_sum(l, wbuf), sv = block_sum(v, wbuf), sg = block_sum(g, wbuf);
    const double ssu = block_sum(su, wbuf), srg = block_sum(rgp, wbuf), sw = block_sum(r2w, wbuf);
    if (tid == 0) {
        out[0] = sl;
        out[1] = sv;
        out[2] = sg;
        out[3] = ssu;
        out[4] = srg;
        out[5] = sw;
    }
}

// --- cell lists ---

// Rebuild the cell lists of the listed chains (those with cell lists): one
// wave per slice, grid (slice blocks, chains), LDS of ncell counts per wave.
// Members of each cell by particle index; a cell beyond cap is reported
// through the status word as in the incremental updates.
template <typename T, int DIM>
__global__ void k_cells_win(const ChainDev *chains, const void *prm, const int *ids, int n, const void *pos,
                            int *cell_cnt, unsigned short *cell_mem, int *bins, int *status, int ncell_max)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int c = ids[blockIdx.y];
    const ChainDev ch = chains[c];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const int j = blockIdx.x * nwv + wave;
    if (ch.ncell <= 0 || j >= ch.M) return;
    int *cnt = reinterpret_cast<int *>(smem) + (size_t)wave * ncell_max;
    const Prm<T> P = reinterpret_cast<const Prm<T> *>(prm)[c];
    const Path<T, DIM, true> path{const_cast<T *>(reinterpret_cast<const T *>(pos)) + ch.pos_off, ch.M, ch.N};
    const Cells C{cell_cnt + ch.cell_off, cell_mem + ch.mem_off, bins + ch.bin_off, ch.M, ch.ncell, ch.cap,
                  ch.nbins};
    for (int cc = lane; cc < ch.ncell; cc += 64) cnt[cc] = 0;
    int nbits = 1;
    while ((1 << nbits) < ch.ncell) ++nbits;
    bool over = false;
    for (int k0 = 0; k0 < ch.N; k0 += 64) {
        const int k = k0 + lane;
        const bool act = k < ch.N;
        int key = 0;
        if (act) {
            T r[DIM];
            path.get(k, j, r);
            key = cell_of<T, DIM>(r, P, ch.nbins);
        }
        // lanes with the same cell
        unsigned long long peers = __ballot(act);
        for (int b = 0; b < nbits; ++b) {
            const bool bit = (key >> b) & 1;
            const unsigned long long bal = __ballot(act && bit);
            peers &= bit ? bal : ~bal;
        }
        const int rank = __popcll(peers & ((1ull << lane) - 1ull));
        const int base = act ? cnt[key] : 0;
        const int pos = base + rank;
        if (act && rank == 0) cnt[key] = base + __popcll(peers);
        if (act) {
            if (pos < ch.cap) {
                C.members(j, key)[pos] = (unsigned short)k;
                C.bin[(long long)k * ch.M + j] = key;
            } else {
                C.bin[(long long)k * ch.M + j] = -1;
                over = true;
            }
        }
    }
    for (int cc = lane; cc < ch.ncell; cc += 64) C.count(j, cc) = min(cnt[cc], ch.cap);
    if (__ballot(over) && lane == 0) atomicOr(status + c, 1);
}

} // namespace pimc
