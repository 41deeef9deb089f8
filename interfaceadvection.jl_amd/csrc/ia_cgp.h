// ia_cgp.h -- the single-reduction CG of a coarse level in one launch.
#pragma once
#include "ia_poisson.h"

namespace ia {

// ---------------------------------------------------------------------------
// All iterations of the single-reduction CG (k_cg1_init, k_cg1_step: the same
// recurrence, the same operations per cell) in one launch of at most CGP_MAXWG
// workgroups that are resident together.  Each workgroup owns a box of cells
// whose r, w, s, p, x, iD and L stay in registers; u = r·iD of the box and of
// its one-cell halo is in LDS.  The halo cells' r and s follow the owners'
// recurrence, so an iteration needs from outside only the neighbours' new w
// and everyone's partial sums, once.
//
// Both travel as 64-bit words of 32 data bits and a 32-bit tag that names the
// launch and the iteration, written and read as single relaxed agent-scope
// atomics: a word whose tag fits is the value itself, so no fence and no
// ordering between words is needed.  Two slots alternate.  A workgroup writes
// a slot again two iterations later, after it has read every workgroup's
// partial of the iteration between, which each of them publishes only after
// it has read the slot's words.
//
// Up to CGP_ONE workgroups of the smaller kind run on one XCD if they fit there: of CGP_XCDS times as many only every
// CGP_XCDS'th takes part, and they say where they run with the first sum.  All on one, the words need only reach its L2:
// store to load 0.5 µs instead of 0.8 past the L2s of the eight XCDs (0.47 against 1.27 with 64 workgroups reading
// everyone's).  Each context has an XCD of its own in turn, so that contexts do not wait for one another's places.
//
// Levels of up to 2M cells take every CU's registers and LDS (BIG: 16 cells of a thread, x, p, s and a tile in 155 KB):
// an iteration reads nothing from memory but the faces.
//
// Measured, µs per iteration of 64, one launch per iteration / here: 128^3 22-24 / 9.0 (6 iterations 145 / 83), 64^3
// 6.6-7.5 / 3.1, 60x44x36 5.4 / 2.2, 32^3 4.6 / 1.55, 192x128 4.5 / 1.3, 96x64 4.3 / 1.2.  What is left on the small
// ones is the exchange and as much again for the operator, the
// recurrence and the two sums, a chain of some 2000 cycles in which a wavefront mostly waits for itself: nothing in it
// stands behind a branch, faces are published through a tile, and a workgroup's words of a sum lie together.
//
// A workgroup that waits longer than CGP_WAIT (other work kept some
// workgroups off the device) writes the x it has, raises *fail and ends, so
// the launch always ends; x is then a less exact solution.  The host then
// solves by one launch per iteration for a while (cgp_give_up).
// ---------------------------------------------------------------------------
constexpr int CGP_MAXWG = 256;
constexpr int CGP_XCDS = 8;   // workgroups go to the XCDs in turn, so those of every eighth number share one
constexpr int CGP_XCU = 32;   // compute units of an XCD
constexpr int CGP_ONE = 64;   // up to so many workgroups everyone reads every partial sum
constexpr int CGP_GROUP = 16; // above, the sums of groups of this many, which the group's first workgroup forms
// cycles/64 before the first look for the sums past the L2s: a look takes about 1100 cycles and disturbs the words' way,
// so the first one should find them (64 workgroups, 32^3: 3.0 µs an iteration without, 2.5 with 6, 2.25 with 12, 2.3
// with 18); within one L2 waiting first gains nothing
constexpr int CGP_NAP = 12;
constexpr long CGP_WAIT = 2000000;  // ticks of the 100 MHz counter: 20 ms
constexpr int CGP_REST = 16, CGP_REST_MAX = 4096;  // projections without one-launch solves after one that gave up
constexpr long CGP_LDS = 158 * 1024;  // of the 160 KiB of a CU
struct CgpBox {
    int k[3], b[3];  // boxes per axis, cells per box and axis (the last box may have fewer, at least 2)
    int nwg, amax;   // workgroups, the largest face of a box
    int spread;      // CGP_XCDS: they fit on one XCD, else 1
};
struct CgpArgs {
    Grid g;
    CgpBox box;
    const float *L, *iD, *r;
    float *x;
    const float *xc;  // the coarser level's x, to prolongate! and increment! by first (not BIG), or nullptr
    Grid gc;
    unsigned long long *hw;  // 2 slots of nwg * 2D * amax words: w of the cells at a box's faces
    unsigned long long *pw;  // 2 slots of CGP_PW words: the partial sums, then the groups' sums
    unsigned tag;            // of iteration 0
    int it;
    int spread, xcd;  // of spread workgroups one takes part, those of blockIdx.x % spread == xcd
    const int *halt;
    int *fail;  // in host memory
    int *stat;  // in device memory: whether one gave up; how many ran on one XCD
};
// a slot of partial sums: 4 words for each workgroup of a group in CGP_COPY copies, then 4 words for each workgroup
constexpr int CGP_COPY = 16;
constexpr int CGP_P1 = CGP_COPY * 4 * CGP_ONE;
constexpr int CGP_PW = CGP_P1 + 5 * CGP_MAXWG;  // the fifth: the XCD (a launch's first sum, if it asked for one)
typedef unsigned long long cgp_word;
constexpr int CGP_SC0 = 1, CGP_VOLATILE = (int)0x80000000u;  // of a buffer load's last argument
// near: all workgroups run on one XCD, so a word need only reach its L2.  What makes the difference is the store: of
// workgroup scope (compiled to sc0) it stays there, of agent scope (sc1) it goes past the L2s.  The loads have to pass
// the compute unit's own cache: the volatile bit makes them system scope (sc0 sc1), and with sc0 alone they were never
// shown another unit's words (every solve gave up), nor are atomic loads of workgroup scope.  Such a load still finds the
// word in its XCD's L2; the far ones are of agent scope (sc1).  Should a load ever take an old word, its tag shows it.
__device__ inline void cgp_put(cgp_word *p, unsigned v, unsigned tag, bool near) {
    const cgp_word q = ((cgp_word)tag << 32) | v;
    if (near) __hip_atomic_store(p, q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else __hip_atomic_store(p, q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// word i of p (the same for the wavefront)
__device__ inline cgp_word cgp_get(const cgp_word *p, int i, bool near) {
    if (!near) return __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    typedef unsigned v2 __attribute__((ext_vector_type(2)));
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0x7ffffff8, 0x00027000);
    const v2 q = __builtin_amdgcn_raw_buffer_load_b64(rs, i * (int)sizeof(cgp_word), 0, CGP_SC0 | CGP_VOLATILE);
    return ((cgp_word)q[1] << 32) | q[0];
}
// words i to i + N - 1 (i a multiple of N = 2 or 4)
template <int N> __device__ inline void cgp_getn(const cgp_word *p, int i, cgp_word (&v)[N], bool near) {
    if (near) {
        typedef unsigned v4 __attribute__((ext_vector_type(4)));
        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0x7ffffff8, 0x00027000);
#pragma unroll
        for (int j = 0; j < N; j += 2) {
            const v4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, (i + j) * (int)sizeof(cgp_word), 0,
                                                               CGP_SC0 | CGP_VOLATILE);
            v[j] = ((cgp_word)q[1] << 32) | q[0];
            v[j + 1] = ((cgp_word)q[3] << 32) | q[2];
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = __hip_atomic_load(p + i + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
__device__ inline void cgp_count(int *n) {  // no read to wait for
    (void)__hip_atomic_fetch_add(n, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the XCD this wavefront runs on (HW_REG_XCC_ID)
__device__ inline unsigned cgp_xcd() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)); }
// whether the nwg (<= CGP_ONE) workgroups said that they run on this wavefront's XCD; w: their words of that, written
// with those of the sum just gathered.  Every workgroup comes to the same answer.
__device__ inline bool cgp_near(const cgp_word *w, int nwg, unsigned tag) {
    const int lane = threadIdx.x & 63;
    const long t0 = wall_clock64();
    for (;;) {
        bool here = true, same = true;
        for (int q = lane; q < nwg; q += 64) {
            const cgp_word v = cgp_get(w, q, false);
            here = here && (unsigned)(v >> 32) == tag;
            same = same && (unsigned)v == cgp_xcd();
        }
        if (__all(here)) return __all(same);
        if (wall_clock64() - t0 > CGP_WAIT) return false;
    }
}
// planes past the end of a box of b cells along the columns that columns of C cells reach
__host__ __device__ inline int cgp_spare(int b, int C) { return (b + C - 1) / C * C - b; }
// BIG's tile has a column's cells side by side, read and written four at a time: a column of b cells starts at word 4,
// the halo cells at 3 and 4 + b; an odd number of fours from column to column spreads them over the banks
__host__ __device__ inline int cgp_zstride(int b, int C) { return 4 * (((5 + b + cgp_spare(b, C) + 3) / 4) | 1); }
// words of LDS of a box: the tiles of u and w, or BIG's tile and x, p and s
__host__ __device__ inline int cgp_tile(int D, int NB, int C, const int *b) {
    const int t1 = b[0] + 2, t2 = t1 * (b[1] + 2);
    if (NB * C > 4096) return t2 * cgp_zstride(b[2], C) + 4;
    return D > 2 ? t2 * (b[2] + 2 + cgp_spare(b[2], C)) + 1 : t1 * (b[1] + 2 + cgp_spare(b[1], C)) + 1;
}
__host__ __device__ inline int cgp_words(int D, int NB, int C, const int *b) {
    const int t = cgp_tile(D, NB, C, b);
    return NB * C > 4096 ? t + 3 * NB * C : 2 * t;
}

// the prolonged x at cell P, A times it
template <int D, class A> __device__ inline float cgp_parent(const A &a, const int P[3]) {
    return a.xc[(long)((P[0] + 3) / 2 - 1) + a.gc.st[1] * ((P[1] + 3) / 2 - 1) +
                (D > 2 ? a.gc.st[2] * ((P[2] + 3) / 2 - 1) : 0)];
}
template <int D, class A> __device__ inline float cgp_mult_parent(const A &a, const int P[3], long I) {
    return mgmult_fc<D>(a.g, P, I, a.L, [&](const int *q) { return cgp_parent<D>(a, q); });
}

// The exchange, for both kernels.  (Their halo cells' geometry is written out in each: formed by one inlined function it
// kept its flags in scalar registers that were then spilled in the loops, 0.5% of a step at 64³.)
// m parts (m <= 64) of a sum, N words each, one part a lane of this wavefront; false: not there in time
template <int N>
__device__ __forceinline__ bool cgp_sums(const cgp_word *w, int m, unsigned tag, bool near, int lane, cgp_word (&v)[N]) {
    const long t0 = wall_clock64();
    for (int spin = 0;; ++spin) {
        bool ok = true;
        if (lane < m) {
            cgp_getn(w, N * lane, v, near);
#pragma unroll
            for (int j = 0; j < N; ++j) ok = ok && (unsigned)(v[j] >> 32) == tag;
        }
        if (__all(ok)) break;
        if ((spin & 31) == 31 && wall_clock64() - t0 > CGP_WAIT) return false;
    }
    return true;
}

// the words of the halo cells, from their owners; false: not there in time
template <int HC>
__device__ __forceinline__ bool cgp_words_at(const cgp_word *hw, const bool (&on)[HC], const int (&wo)[HC], unsigned tag,
                                             bool near, cgp_word (&h)[HC]) {
    const long t0 = wall_clock64();
    for (int spin = 0;; ++spin) {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < HC; ++k) h[k] = cgp_get(hw, wo[k], near);
#pragma unroll
        for (int k = 0; k < HC; ++k) ok = ok && (!on[k] || (unsigned)(h[k] >> 32) == tag);
        if (__all(ok)) break;
        if ((spin & 31) == 31 && wall_clock64() - t0 > CGP_WAIT) return false;
    }
    return true;
}
// publishes the values at the box's faces, from their tile
template <int HC>
__device__ __forceinline__ void cgp_faces(cgp_word *hw, const float *tile, const bool (&on)[HC], const int (&ti)[HC],
                                          const int (&wo)[HC], unsigned tag, bool near) {
    float f[HC];
#pragma unroll
    for (int k = 0; k < HC; ++k) f[k] = tile[ti[k]];
    if (near) {
#pragma unroll
        for (int k = 0; k < HC; ++k)
            if (on[k]) cgp_put(hw + wo[k], __float_as_uint(f[k]), tag, true);
    } else {
#pragma unroll
        for (int k = 0; k < HC; ++k)
            if (on[k]) cgp_put(hw + wo[k], __float_as_uint(f[k]), tag, false);
    }
}
// the place of workgroup wg's box: its indices, first cell lo (ghost-inclusive), sides n
template <int D> struct CgpAt {
    int bi[3], lo[3], n[3];
    __device__ __forceinline__ CgpAt(const Grid &g, const CgpBox &box, int wg) {
        bi[0] = wg % box.k[0];
        bi[1] = wg / box.k[0] % box.k[1];
        bi[2] = wg / box.k[0] / box.k[1];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = d < D ? 1 + bi[d] * box.b[d] : 0;
            n[d] = d < D ? min(box.b[d], g.Ng[d] - 1 - lo[d]) : 1;
        }
    }
};

// NB threads; a thread owns a column of C cells along the last axis (so two of a cell's neighbours are mostly its own
// registers); the halo cells are those of wavefronts 1.. (HC each), while wavefront 0 waits for the sums.
template <int D, int NB, int C, int HC>
__global__ void __launch_bounds__(NB) k_cgp(CgpArgs a) {
    HALT_IF(a)
    if ((int)blockIdx.x % a.spread != a.xcd) return;
    const int wg = (int)blockIdx.x / a.spread;
    extern __shared__ __align__(16) float cgp_u[];
    constexpr bool XL = NB * C >= 4096;  // x in LDS: the registers do not hold it
    constexpr bool BIG = NB * C > 4096;  // p and s in LDS too, u and the diagonal formed again, w in u's tile
    constexpr int CR = BIG ? 1 : C;
    __shared__ float xs[XL && !BIG ? NB * C : 1];
    __shared__ double shp[2][NB / 64], sht[2];
    __shared__ int dead, nears;
    const Grid &g = a.g;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const CgpAt<D> B(g, a.box, wg);
    const auto &bi = B.bi, &lo = B.lo, &n = B.n;
    // strides of the u tile, along a column last
    const int zs = BIG ? cgp_zstride(a.box.b[2], C) : 1, t0 = BIG ? zs : 1, t1 = t0 * (a.box.b[0] + 2);
    const int tz = BIG ? 1 : D > 2 ? t1 * (a.box.b[1] + 2) : t1;
    auto at = [&](int x, int y, int z) {
        return t0 * (x + 1) + t1 * (y + 1) + (D > 2 ? tz * (z + 1) : 0) + (BIG ? 3 : 0);
    };
    const long sz = g.st[D - 1];
    // every thread works on all C cells of its column: those past its cnt are all zeros, read the tile's spare planes
    // and write its last word, so no load or store waits behind a branch
    const int dump = cgp_tile(D, NB, C, a.box.b) - (BIG ? 4 : 1);
    float *const xl = BIG ? cgp_u + dump + 4 : xs;  // cell k at k * NB + tid; BIG: four cells together
    float4 *const x4 = (float4 *)xl, *const p4 = x4 + NB * C / 4, *const s4 = p4 + NB * C / 4;
    for (int q = tid; q <= dump; q += NB) cgp_u[q] = 0.f;
    if (tid == 0) dead = 0;
    __syncthreads();
    // own cells: lateral position (x, y), first cell z0 of the column, cnt of them
    const int nl = D > 2 ? n[0] * n[1] : n[0];
    const int col = tid % nl, x0 = col % n[0], y0 = D > 2 ? col / n[0] : 0, z0 = (tid / nl) * C;
    const int cnt = max(0, min(C, n[D - 1] - z0));
    const int ti = D > 2 ? at(x0, y0, cnt > 0 ? z0 : 0) : at(x0, cnt > 0 ? z0 : 0, 0);
    auto tw = [&](int t, int k) { return k < cnt ? t + k * tz : dump; };
    // the column's place in the tile; BIG: anew at each use, or the cells' places would be kept in registers
    auto place = [&]() {
        int t = ti;
        if (BIG) asm volatile("" : "+v"(t));
        return t;
    };
    const long I0 = (long)(lo[0] + x0) + (D > 2 ? g.st[1] * (lo[1] + y0) : 0) + sz * (lo[D - 1] + z0);
    float r[C], s[CR], w[C], p[CR], x[XL ? 1 : C], id[C], u[CR], dg[CR], lx[C], lxp[C], ly[C], lyp[C], lz[C + 1];
#pragma unroll
    for (int k = 0; k <= C; ++k) lz[k] = cnt > 0 && k <= cnt ? a.L[g.ns * (D - 1) + I0 + k * sz] : 0.f;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        float xk = 0.f;
        r[k] = w[k] = id[k] = lx[k] = lxp[k] = ly[k] = lyp[k] = 0.f;
        if (k < cnt) {
            long I = I0 + k * sz;
            r[k] = a.r[I];
            id[k] = a.iD[I];
            xk = a.x[I];
            lx[k] = a.L[I];
            lxp[k] = a.L[I + 1];
            if (D > 2) {
                ly[k] = a.L[g.ns + I];
                lyp[k] = a.L[g.ns + I + g.st[1]];
            }
            if (!BIG && a.xc) {
                const int P[3] = {lo[0] + x0, D > 2 ? lo[1] + y0 : lo[1] + z0 + k, D > 2 ? lo[2] + z0 + k : 0};
                r[k] = r[k] - cgp_mult_parent<D>(a, P, I);
                xk += cgp_parent<D>(a, P);
            }
        }
        if (BIG) xl[4 * (k / 4 * NB + tid) + k % 4] = xk;
        else if (XL) xl[k * NB + tid] = xk;
        else x[XL ? 0 : k] = xk;
    }
    auto diag = [&](int k) {
        float d = 0.f - (lx[k] + lxp[k]);
        if (D > 2) d -= (ly[k] + lyp[k]);
        return d - (lz[k] + lz[k + 1]);
    };
#pragma unroll
    for (int k = 0; k < CR; ++k) dg[k] = BIG ? 0.f : diag(k);
    auto U = [&](int k) { return BIG ? r[k] * id[k] : u[BIG ? 0 : k]; };
    // halo cells of the box's faces (2d + side); none across a wall (u = 0 there, L = 0)
    // the same threads publish the cells on this side of the faces
    bool hon[HC], fon[HC];
    int hti[HC], hwo[HC];  // place in the tile, word of the cell's w in the slot
    int fti[HC], fwo[HC];
    float *const cgp_w = BIG ? cgp_u : cgp_u + dump + 1;  // a tile of w
    float hr[HC], hs[HC], hid[HC], hv[HC];
    {
        const int area[3] = {n[1] * n[2], n[0] * n[2], n[0] * n[1]};
        const int hc = 2 * area[0] + 2 * area[1] + (D > 2 ? 2 * area[2] : 0);
#pragma unroll
        for (int k = 0; k < HC; ++k) {
            int h = tid - 64 + k * (NB - 64);
            hon[k] = fon[k] = false;
            hti[k] = fti[k] = dump;
            hwo[k] = fwo[k] = 0;
            hr[k] = hs[k] = hid[k] = hv[k] = 0.f;
            if (tid >= 64 && h < hc) {
                int d = 0;
                if (h >= 2 * area[0]) {
                    h -= 2 * area[0];
                    d = 1;
                    if (D > 2 && h >= 2 * area[1]) {
                        h -= 2 * area[1];
                        d = 2;
                    }
                }
                const int ar = d == 0 ? area[0] : d == 1 ? area[1] : area[2];
                const int side = h >= ar;
                h -= side * ar;
                // element h of the face: the two other coordinates in x-y-z order
                const int m = d == 0 ? n[1] : n[0], e0 = h % m, e1 = h / m;
                const int qd = side ? (d == 0 ? n[0] : d == 1 ? n[1] : n[2]) : -1;
                const int q[3] = {d == 0 ? qd : e0, d == 1 ? qd : (d == 0 ? e0 : e1), d == 2 ? qd : e1};
                const int tq = at(q[0], q[1], q[2]);
                fon[k] = true;
                fti[k] = tq + (side ? -1 : 1) * (d == 0 ? t0 : d == 1 ? t1 : tz);
                fwo[k] = (wg * 2 * D + 2 * d + side) * a.box.amax + h;
                int P[3] = {lo[0] + q[0], lo[1] + q[1], D > 2 ? lo[2] + q[2] : 0}, c[3] = {bi[0], bi[1], bi[2]};
                bool wall = false;
#pragma unroll
                for (int b = 0; b < D; ++b)
                    if (b == d) {
                        wall = !g.per[b] && (P[b] == 0 || P[b] == g.Ng[b] - 1);
                        P[b] = P[b] == 0 ? g.Ng[b] - 2 : P[b] == g.Ng[b] - 1 ? 1 : P[b];
                        c[b] += side ? 1 : -1;
                        c[b] = c[b] < 0 ? a.box.k[b] - 1 : c[b] == a.box.k[b] ? 0 : c[b];
                    }
                if (!wall) {
                    hon[k] = true;
                    hti[k] = tq;
                    long J = (long)P[0] + g.st[1] * P[1] + (D > 2 ? g.st[2] * P[2] : 0);
                    hr[k] = a.r[J];
                    hid[k] = a.iD[J];
                    if (!BIG && a.xc) hr[k] = hr[k] - cgp_mult_parent<D>(a, P, J);
                    // the neighbour's facing side holds the same cells in the same order
                    hwo[k] = ((c[0] + a.box.k[0] * (c[1] + a.box.k[1] * c[2])) * 2 * D + 2 * d + 1 - side) * a.box.amax + h;
                }
            }
        }
    }
    const long hslot = (long)a.box.nwg * 2 * D * a.box.amax;
    const int nwg = a.box.nwg, ngrp = (nwg + CGP_GROUP - 1) / CGP_GROUP;
    const bool two = nwg > CGP_ONE;
    constexpr bool FAR = NB * C >= 4096;  // too large for one XCD
    bool near = false;  // known once the first sum is
    auto half_of = [](double va, double vb, int j) {  // word j of a pair of sums
        double v = j < 2 ? va : vb;
        return (unsigned)((j & 1) ? __double2hiint(v) : __double2loint(v));
    };
    auto faces = [&](unsigned tag) {  // w of the box's faces, from its tile
        cgp_word *hw = a.hw + (tag & 1 ? hslot : 0);
        cgp_faces(hw, cgp_w, fon, fti, fwo, tag, near);
    };
    auto own = [&](float *tl, const float (&v)[C]) {  // the own cells' values to a tile
        const int t = place();
        if (BIG && cnt == C) {
#pragma unroll
            for (int k = 0; k < C; k += 4)
                *(float4 *)(tl + t + k) = make_float4(v[k], v[k + 1 < C ? k + 1 : k], v[k + 2 < C ? k + 2 : k],
                                                      v[k + 3 < C ? k + 3 : k]);
        } else {
#pragma unroll
            for (int k = 0; k < C; ++k) tl[tw(t, k)] = v[k];
        }
    };
    auto tile = [&]() {  // u of the box and its halo
        float uk[C];
#pragma unroll
        for (int k = 0; k < C; ++k) {
            uk[k] = r[k] * id[k];
            if (!BIG) u[BIG ? 0 : k] = uk[k];
        }
        own(cgp_u, uk);
#pragma unroll
        for (int k = 0; k < HC; ++k) cgp_u[hti[k]] = hr[k] * hid[k];
    };
    auto apply = [&](unsigned tag) {  // w = A u, published at the box's faces; the partials of r·u and u·w
        double gd = 0, dd = 0;
        {
            const int tc = place();
            const float ulo = cgp_u[tc - tz], uhi = cgp_u[tc + cnt * tz];
            constexpr int G = BIG ? 4 : C;  // cells whose neighbours are read together
            float um[G], up[G], vm[D > 2 ? G : 1], vp[D > 2 ? G : 1];
            if (!BIG) {
#pragma unroll
                for (int k = 0; k < C; ++k) {
                    const int t = tc + k * tz;
                    um[k % G] = cgp_u[t - 1];
                    up[k % G] = cgp_u[t + 1];
                    if (D > 2) {
                        vm[D > 2 ? k % G : 0] = cgp_u[t - t1];
                        vp[D > 2 ? k % G : 0] = cgp_u[t + t1];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < C; ++k) {
                if (BIG && k % 4 == 0) {
                    // no loads of later groups: the registers do not hold them
                    __builtin_amdgcn_sched_barrier(0);
                    auto rd = [&](float *v, int t) {
                        const float4 q = *(const float4 *)(cgp_u + t + k);
                        v[0] = q.x;
                        v[BIG ? 1 : 0] = q.y;
                        v[BIG ? 2 : 0] = q.z;
                        v[BIG ? 3 : 0] = q.w;
                    };
                    rd(um, tc - t0);
                    rd(up, tc + t0);
                    rd(vm, tc - t1);
                    rd(vp, tc + t1);
                }
                float sl = 0, su = 0;
                sl += um[k % G] * lx[k];
                su += up[k % G] * lxp[k];
                if (D > 2) {
                    sl += vm[D > 2 ? k % G : 0] * ly[k];
                    su += vp[D > 2 ? k % G : 0] * lyp[k];
                }
                float hi = uhi;
                if (k + 1 < C) {
                    const float un = U(k + 1 < C ? k + 1 : k);
                    hi = k + 1 < cnt ? un : uhi;
                }
                const float uk = U(k);
                sl += (k > 0 ? U(k > 0 ? k - 1 : 0) : ulo) * lz[k];
                su += hi * lz[k + 1];
                w[k] = (uk * (BIG ? diag(k) : dg[BIG ? 0 : k]) + sl) + su;
                // the products are exact
                gd = __builtin_fma((double)r[k], (double)uk, gd);
                dd = __builtin_fma((double)uk, (double)w[k], dd);
            }
            if (BIG) __syncthreads();  // everyone has read u
            own(cgp_w, w);
        }
        wave_sum2(gd, dd);
        if (lane == 0) {
            shp[0][wv] = gd;
            shp[1][wv] = dd;
        }
        __syncthreads();
        if (wv == 0) {
            double va = 0, vb = 0;
#pragma unroll
            for (int q = 0; q < NB / 64; ++q) va += shp[0][q];
#pragma unroll
            for (int q = 0; q < NB / 64; ++q) vb += shp[1][q];
            cgp_word *pw = a.pw + (tag & 1 ? CGP_PW : 0) + CGP_P1;
            if (lane < 4) cgp_put(pw + 4 * wg + lane, half_of(va, vb, lane), tag, near);
            if (a.spread > 1 && tag == a.tag && lane == 4) cgp_put(pw + 4 * CGP_MAXWG + wg, cgp_xcd(), tag, near);
        }
        faces(tag);
    };
    // the sums of m pairs (m <= 64) of four words each by this wavefront; false: not there in time
    auto gather = [&](const cgp_word *w4, int m, unsigned tag, double &va, double &vb) {
        cgp_word v[4];
        if (!cgp_sums(w4, m, tag, near, lane, v)) return false;
        va = lane < m ? __hiloint2double((int)(unsigned)v[1], (int)(unsigned)v[0]) : 0.0;
        vb = lane < m ? __hiloint2double((int)(unsigned)v[3], (int)(unsigned)v[2]) : 0.0;
        wave_sum2(va, vb);
        return true;
    };
    // the halo cells' w
    auto halo = [&](const cgp_word *hw, unsigned tag) {
        cgp_word h[HC];
        if (!cgp_words_at(hw, hon, hwo, tag, near, h)) return false;
#pragma unroll
        for (int k = 0; k < HC; ++k) hv[k] = hon[k] ? __uint_as_float((unsigned)h[k]) : 0.f;
        return true;
    };
    tile();
    __syncthreads();
    apply(a.tag);
#pragma unroll
    for (int k = 0; k < C; ++k) {
        if (BIG) {
            ((float *)p4)[4 * (k / 4 * NB + tid) + k % 4] = U(k);
            ((float *)s4)[4 * (k / 4 * NB + tid) + k % 4] = w[k];
        } else {
            p[BIG ? 0 : k] = U(k);
            s[BIG ? 0 : k] = w[k];
        }
    }
    float rho = 0, al = 0;
    for (int q = 1; q <= a.it; ++q) {
        const double irho = inverse((double)rho), ial = inverse((double)al);
        const unsigned tag = a.tag + q - 1;
        cgp_word *pw = a.pw + (tag & 1 ? CGP_PW : 0), *hw = a.hw + (tag & 1 ? hslot : 0);
        bool ok = true;
        if (wv == 0) {
            double sa = 0, sb = 0;
            if (!near) __builtin_amdgcn_s_sleep(CGP_NAP);
            if (two) {
                if (wg % CGP_GROUP == 0) {
                    ok = gather(pw + CGP_P1 + 4 * wg, min(CGP_GROUP, nwg - wg), tag, sa, sb);
                    if (ok)  // a copy for each of the group's workgroups
                        cgp_put(pw + 4 * ((lane >> 2) * CGP_ONE + wg / CGP_GROUP) + (lane & 3),
                                half_of(sa, sb, lane & 3), tag, near);
                }
                if (ok) ok = gather(pw + (wg % CGP_COPY) * 4 * CGP_ONE, ngrp, tag, sa, sb);
            } else {
                ok = gather(pw + CGP_P1, nwg, tag, sa, sb);
            }
            const bool nr =
                near || (a.spread > 1 && q == 1 && ok && cgp_near(pw + CGP_P1 + 4 * CGP_MAXWG, nwg, tag));
            if (lane == 0) {
                sht[0] = sa;
                sht[1] = sb;
                nears = nr;
            }
        } else {
            ok = halo(hw, tag);
        }
        if (!ok) dead = 1;
        __syncthreads();
        if (dead) {
            if (tid == 0) *a.fail = a.stat[0] = 1;
            break;
        }
        near = !FAR && nears != 0;
        const float gam = (float)sht[0], del = (float)sht[1];
        if (fabs(gam) < 10 * eps_of<float>()) break;
        float beta = 0;
        if (q == 1) {
            al = gam / del;
        } else {
            beta = quotient(gam, irho);
            al = quotient(gam, inverse((double)(del - quotient(beta * gam, ial))));
        }
        rho = gam;
        const bool stop = q == a.it || fabs((double)al) < 1e-2;
        auto cell = [&](int k, float &pk, float &sk, float &xk) {
            if (q > 1) {
                pk = U(k) + beta * pk;
                sk = w[k] + beta * sk;
            }
            xk = xk + al * pk;
            r[k] = r[k] - al * sk;
        };
        if constexpr (BIG) {
#pragma unroll
            for (int k = 0; k < C; k += 4) {
                const int j = k / 4 * NB + tid;
                __builtin_amdgcn_sched_barrier(0);
                float4 pk = p4[j], sk = s4[j], xk = x4[j];
                cell(k, pk.x, sk.x, xk.x);
                cell(k + 1, pk.y, sk.y, xk.y);
                cell(k + 2, pk.z, sk.z, xk.z);
                cell(k + 3, pk.w, sk.w, xk.w);
                p4[j] = pk;
                s4[j] = sk;
                x4[j] = xk;
            }
        } else {
#pragma unroll
            for (int k = 0; k < C; ++k) cell(k, p[k], s[k], XL ? xl[k * NB + tid] : x[XL ? 0 : k]);
        }
        if (stop) break;
#pragma unroll
        for (int k = 0; k < HC; ++k) {
            hs[k] = q > 1 ? hv[k] + beta * hs[k] : hv[k];
            hr[k] = hr[k] - al * hs[k];
        }
        tile();
        __syncthreads();
        apply(tag + 1);
    }
    if (near && wg == 0 && tid == 0) cgp_count(a.stat + 1);
#pragma unroll
    for (int k = 0; k < C; ++k)
        if (k < cnt)
            a.x[I0 + k * sz] = BIG ? xl[4 * (k / 4 * NB + tid) + k % 4] : XL ? xl[k * NB + tid] : x[XL ? 0 : k];
}

// ---------------------------------------------------------------------------
// WaterLily's pcg! on a level in one launch, on the same boxes and words: two
// sums an iteration, so two exchanges, the first with the face values of
// z = A ϵ; the halo cells' r and ϵ follow the owners' recurrence.  With xc it
// begins with the prolongate! and increment! before it (the coarse x's parents
// at the cell and its neighbours, on the halo cells too), and on the finest
// level (r2 set) it ends with what solver! does next: r, z, the next Jacobi!'s
// ϵ and the workgroups' parts of Σr², in host memory.  x and r are written
// only after the last exchange, which every workgroup reaches only when all
// have read their halo, so they are updated in place.
//
// 6 iterations on 256x256 (64 workgroups) and on 128x128 were 18 and 13
// launches of 2.7-3.0 µs, each 4 µs of the host's time, which set the pace; now 15.5 and 11.2 µs.
// ---------------------------------------------------------------------------
struct PcgpArgs {
    Grid g;
    CgpBox box;
    const float *L, *iD;
    float *x, *r, *z, *e;
    const float *xc;  // the coarser level's x, or nullptr
    Grid gc;
    cgp_word *hw, *pw;
    unsigned tag;
    int it;
    double *r2;
    int spread, xcd;  // of spread workgroups one takes part, those of wg % spread == xcd
    const int *halt;
    int *fail;  // in host memory
    int *stat;  // in device memory: whether one gave up; how many ran on one XCD
};
template <int D, int NB, int C, int HC>
__global__ void __launch_bounds__(NB) k_pcgp(PcgpArgs a) {
    HALT_IF(a)
    if ((int)blockIdx.x % a.spread != a.xcd) return;
    const int wg = (int)blockIdx.x / a.spread;
    extern __shared__ __align__(16) float cgp_u[];
    constexpr bool XL = NB * C >= 4096;  // x in LDS, as k_cgp
    __shared__ float xl[XL ? NB * C : 1];
    __shared__ double shp[NB / 64], sht;
    __shared__ int dead, nears;
    const Grid &g = a.g;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const CgpAt<D> B(g, a.box, wg);
    const auto &bi = B.bi, &lo = B.lo, &n = B.n;
    const int t1 = a.box.b[0] + 2, t2 = t1 * (a.box.b[1] + 2);  // strides of the u tile
    const int tz = D > 2 ? t2 : t1;                            // along a column
    const long sz = g.st[D - 1];
    // every thread works on all C cells of its column: those past its cnt are all zeros, read the tile's spare planes
    // and write its last word, so no load or store waits behind a branch
    const int dump = t1 * (a.box.b[1] + 2) * (D > 2 ? a.box.b[2] + 2 : 1) + cgp_spare(a.box.b[D - 1], C) * tz;
    for (int q = tid; q <= dump; q += NB) cgp_u[q] = 0.f;
    if (tid == 0) dead = 0;
    __syncthreads();
    // own cells: lateral position (x, y), first cell z0 of the column, cnt of them
    const int nl = D > 2 ? n[0] * n[1] : n[0];
    const int col = tid % nl, x0 = col % n[0], y0 = D > 2 ? col / n[0] : 0, z0 = (tid / nl) * C;
    const int cnt = max(0, min(C, n[D - 1] - z0));
    const int ti = (x0 + 1) + (D > 2 ? t1 * (y0 + 1) : 0) + tz * (cnt > 0 ? z0 + 1 : 1);
    int tw[C];
#pragma unroll
    for (int k = 0; k < C; ++k) tw[k] = k < cnt ? ti + k * tz : dump;
    const long I0 = (long)(lo[0] + x0) + (D > 2 ? g.st[1] * (lo[1] + y0) : 0) + sz * (lo[D - 1] + z0);
    float r[C], w[C], x[XL ? 1 : C], id[C], u[C], dg[C], lx[C], lxp[C], ly[C], lyp[C], lz[C + 1];
#pragma unroll
    for (int k = 0; k <= C; ++k) lz[k] = cnt > 0 && k <= cnt ? a.L[g.ns * (D - 1) + I0 + k * sz] : 0.f;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        if (XL) xl[k * NB + tid] = 0.f;
        else x[XL ? 0 : k] = 0.f;
        r[k] = w[k] = id[k] = u[k] = dg[k] = lx[k] = lxp[k] = ly[k] = lyp[k] = 0.f;
        if (k < cnt) {
            long I = I0 + k * sz;
            r[k] = a.r[I];
            id[k] = a.iD[I];
            if (XL) xl[k * NB + tid] = a.x[I];
            else x[XL ? 0 : k] = a.x[I];
            lx[k] = a.L[I];
            lxp[k] = a.L[I + 1];
            dg[k] -= (lx[k] + lxp[k]);
            if (D > 2) {
                ly[k] = a.L[g.ns + I];
                lyp[k] = a.L[g.ns + I + g.st[1]];
                dg[k] -= (ly[k] + lyp[k]);
            }
            dg[k] -= (lz[k] + lz[k + 1]);
            if (a.xc) {  // prolongate! and increment!
                const int P[3] = {lo[0] + x0, D > 2 ? lo[1] + y0 : lo[1] + z0 + k, D > 2 ? lo[2] + z0 + k : 0};
                const float ec = cgp_parent<D>(a, P);
                r[k] = r[k] - cgp_mult_parent<D>(a, P, I);
                if (XL) xl[k * NB + tid] += ec;
                else x[XL ? 0 : k] = x[XL ? 0 : k] + ec;
            }
        }
    }
    // halo cells of the box's faces (2d + side); none across a wall (u = 0 there, L = 0)
    // the same threads publish the cells on this side of the faces
    bool hon[HC], fon[HC];
    int hti[HC], hwo[HC];  // place in the tile, word of the cell's w in the slot
    int fti[HC], fwo[HC];
    float *const cgp_w = cgp_u + dump + 1;  // a tile of w
    float hr[HC], hu[HC], hid[HC], hv[HC];
    {
        const int area[3] = {n[1] * n[2], n[0] * n[2], n[0] * n[1]};
        const int hc = 2 * area[0] + 2 * area[1] + (D > 2 ? 2 * area[2] : 0);
#pragma unroll
        for (int k = 0; k < HC; ++k) {
            int h = tid - 64 + k * (NB - 64);
            hon[k] = fon[k] = false;
            hti[k] = fti[k] = dump;
            hwo[k] = fwo[k] = 0;
            hr[k] = hu[k] = hid[k] = hv[k] = 0.f;
            if (tid >= 64 && h < hc) {
                int d = 0;
                if (h >= 2 * area[0]) {
                    h -= 2 * area[0];
                    d = 1;
                    if (D > 2 && h >= 2 * area[1]) {
                        h -= 2 * area[1];
                        d = 2;
                    }
                }
                const int ar = d == 0 ? area[0] : d == 1 ? area[1] : area[2];
                const int side = h >= ar;
                h -= side * ar;
                // element h of the face: the two other coordinates in x-y-z order
                const int m = d == 0 ? n[1] : n[0], e0 = h % m, e1 = h / m;
                const int qd = side ? (d == 0 ? n[0] : d == 1 ? n[1] : n[2]) : -1;
                const int q[3] = {d == 0 ? qd : e0, d == 1 ? qd : (d == 0 ? e0 : e1), d == 2 ? qd : e1};
                const int tq = (q[0] + 1) + t1 * (q[1] + 1) + (D > 2 ? t2 * (q[2] + 1) : 0);
                fon[k] = true;
                fti[k] = tq + (side ? -1 : 1) * (d == 0 ? 1 : d == 1 ? t1 : t2);
                fwo[k] = (wg * 2 * D + 2 * d + side) * a.box.amax + h;
                int P[3] = {lo[0] + q[0], lo[1] + q[1], D > 2 ? lo[2] + q[2] : 0}, c[3] = {bi[0], bi[1], bi[2]};
                bool wall = false;
#pragma unroll
                for (int b = 0; b < D; ++b)
                    if (b == d) {
                        wall = !g.per[b] && (P[b] == 0 || P[b] == g.Ng[b] - 1);
                        P[b] = P[b] == 0 ? g.Ng[b] - 2 : P[b] == g.Ng[b] - 1 ? 1 : P[b];
                        c[b] += side ? 1 : -1;
                        c[b] = c[b] < 0 ? a.box.k[b] - 1 : c[b] == a.box.k[b] ? 0 : c[b];
                    }
                if (!wall) {
                    hon[k] = true;
                    hti[k] = tq;
                    long J = (long)P[0] + g.st[1] * P[1] + (D > 2 ? g.st[2] * P[2] : 0);
                    hr[k] = a.r[J];
                    hid[k] = a.iD[J];
                    if (a.xc) hr[k] = hr[k] - cgp_mult_parent<D>(a, P, J);
                    // the neighbour's facing side holds the same cells in the same order
                    hwo[k] = ((c[0] + a.box.k[0] * (c[1] + a.box.k[1] * c[2])) * 2 * D + 2 * d + 1 - side) * a.box.amax + h;
                }
            }
        }
    }
    const long hslot = (long)a.box.nwg * 2 * D * a.box.amax;
    const int nwg = a.box.nwg, ngrp = (nwg + CGP_GROUP - 1) / CGP_GROUP;
    const bool two = nwg > CGP_ONE;
    constexpr bool FAR = NB * C >= 4096;  // too large for one XCD
    bool near = false;  // known once the first sum is
    auto half_of = [](double v, int j) { return (unsigned)((j & 1) ? __double2hiint(v) : __double2loint(v)); };
    auto faces = [&](unsigned tag) {  // w of the box's faces, from its tile
        cgp_word *hw = a.hw + (tag & 1 ? hslot : 0);
        cgp_faces(hw, cgp_w, fon, fti, fwo, tag, near);
    };
    auto tile = [&]() {  // ϵ of the box and its halo
#pragma unroll
        for (int k = 0; k < C; ++k) cgp_u[tw[k]] = u[k];
#pragma unroll
        for (int k = 0; k < HC; ++k) cgp_u[hti[k]] = hu[k];
    };
    auto publish = [&](unsigned tag, double v) {  // this workgroup's part of a sum
        v = wave_sum1(v);
        if (lane == 0) shp[wv] = v;
        __syncthreads();
        if (wv == 0) {
            double t = 0;
#pragma unroll
            for (int q = 0; q < NB / 64; ++q) t += shp[q];
            cgp_word *pw = a.pw + (tag & 1 ? CGP_PW : 0) + CGP_P1;
            if (lane < 2) cgp_put(pw + 2 * wg + lane, half_of(t, lane), tag, near);
            if (a.spread > 1 && tag == a.tag && lane == 4) cgp_put(pw + 4 * CGP_MAXWG + wg, cgp_xcd(), tag, near);
        }
    };
    // the sum of m parts (m <= 64) of two words each by this wavefront; false: not there in time
    auto gather = [&](const cgp_word *w2, int m, unsigned tag, double &v) {
        cgp_word q[2];
        if (!cgp_sums(w2, m, tag, near, lane, q)) return false;
        v = wave_sum1(lane < m ? __hiloint2double((int)(unsigned)q[1], (int)(unsigned)q[0]) : 0.0);
        return true;
    };
    // the halo cells' z = A ϵ
    auto halo = [&](const cgp_word *hw, unsigned tag) {
        cgp_word h[HC];
        if (!cgp_words_at(hw, hon, hwo, tag, near, h)) return false;
#pragma unroll
        for (int k = 0; k < HC; ++k) hv[k] = hon[k] ? __uint_as_float((unsigned)h[k]) : 0.f;
        return true;
    };
    // the total of a published sum, in FP32 (and the halo with it); false: gave up
    auto total = [&](unsigned tag, const cgp_word *hw, float &out) {
        cgp_word *pw = a.pw + (tag & 1 ? CGP_PW : 0);
        bool ok = true;
        if (wv == 0) {
            double v = 0;
            if (!near) __builtin_amdgcn_s_sleep(CGP_NAP);
            if (two) {
                if (wg % CGP_GROUP == 0) {
                    ok = gather(pw + CGP_P1 + 2 * wg, min(CGP_GROUP, nwg - wg), tag, v);
                    if (ok && lane < 2 * CGP_COPY)  // a copy for each of the group's workgroups
                        cgp_put(pw + 2 * ((lane >> 1) * CGP_ONE + wg / CGP_GROUP) + (lane & 1), half_of(v, lane & 1),
                                tag, near);
                }
                if (ok) ok = gather(pw + (wg % CGP_COPY) * 2 * CGP_ONE, ngrp, tag, v);
            } else {
                ok = gather(pw + CGP_P1, nwg, tag, v);
            }
            const bool nr =
                near || (a.spread > 1 && tag == a.tag && ok && cgp_near(pw + CGP_P1 + 4 * CGP_MAXWG, nwg, tag));
            if (lane == 0) {
                sht = v;
                nears = nr;
            }
        } else if (hw) {
            ok = halo(hw, tag);
        }
        if (!ok) dead = 1;
        __syncthreads();
        out = (float)sht;
        near = !FAR && nears != 0;
        return dead == 0;
    };
    // z = ϵ = r·iD, ρ = r·z
    double v = 0;
#pragma unroll
    for (int k = 0; k < C; ++k) {
        u[k] = r[k] * id[k];
        v = __builtin_fma((double)r[k], (double)u[k], v);  // the products are exact
    }
#pragma unroll
    for (int k = 0; k < HC; ++k) hu[k] = hr[k] * hid[k];
    tile();
    publish(a.tag, v);
    float rho = 0;
    bool ok = total(a.tag, nullptr, rho);
    bool done = !ok || fabs(rho) < 10 * eps_of<float>();
    const bool zset = !done;
    for (int i = 1; i <= a.it && !done; ++i) {
        // z = A ϵ, published at the box's faces; z·ϵ (total's barrier came after the tile's last write)
        const unsigned ta = a.tag + 2 * i - 1, tb = ta + 1;
        const cgp_word *hw = a.hw + (ta & 1 ? hslot : 0);
        v = 0;
        {
            const float ulo = cgp_u[ti - tz], uhi = cgp_u[ti + cnt * tz];
            float um[C], up[C], vm[D > 2 ? C : 1], vp[D > 2 ? C : 1];
#pragma unroll
            for (int k = 0; k < C; ++k) {
                const int t = ti + k * tz;
                um[k] = cgp_u[t - 1];
                up[k] = cgp_u[t + 1];
                if (D > 2) {
                    vm[D > 2 ? k : 0] = cgp_u[t - t1];
                    vp[D > 2 ? k : 0] = cgp_u[t + t1];
                }
            }
#pragma unroll
            for (int k = 0; k < C; ++k) {
                float sl = 0, su = 0;
                sl += um[k] * lx[k];
                su += up[k] * lxp[k];
                if (D > 2) {
                    sl += vm[D > 2 ? k : 0] * ly[k];
                    su += vp[D > 2 ? k : 0] * lyp[k];
                }
                float hi = uhi;
                if (k + 1 < C) {
                    const float un = u[k + 1 < C ? k + 1 : k];
                    hi = k + 1 < cnt ? un : uhi;
                }
                sl += (k > 0 ? u[k > 0 ? k - 1 : 0] : ulo) * lz[k];
                su += hi * lz[k + 1];
                w[k] = (u[k] * dg[k] + sl) + su;
            }
#pragma unroll
            for (int k = 0; k < C; ++k) cgp_w[tw[k]] = w[k];
#pragma unroll
            for (int k = 0; k < C; ++k)
                v = __builtin_fma((double)w[k], (double)u[k], v);
        }
        publish(ta, v);
        faces(ta);
        float ze;
        if (!total(ta, hw, ze)) {
            ok = false;
            break;
        }
        const float alpha = rho / ze;
        v = 0;
#pragma unroll
        for (int k = 0; k < C; ++k) {
            if (XL) xl[k * NB + tid] += alpha * u[k];
            else x[XL ? 0 : k] = x[XL ? 0 : k] + alpha * u[k];
            r[k] = r[k] - alpha * w[k];
            w[k] = r[k] * id[k];
            v = __builtin_fma((double)r[k], (double)w[k], v);
        }
        if (i == a.it || fabs((double)alpha) < 1e-2) break;
        publish(tb, v);
        float rho2;
        if (!total(tb, nullptr, rho2)) {
            ok = false;
            break;
        }
        if (fabs(rho2) < 10 * eps_of<float>()) break;
        const float beta = rho2 / rho;
#pragma unroll
        for (int k = 0; k < C; ++k) u[k] = beta * u[k] + w[k];
#pragma unroll
        for (int k = 0; k < HC; ++k) {
            hr[k] = hr[k] - alpha * hv[k];
            hu[k] = beta * hu[k] + hr[k] * hid[k];
        }
        tile();
        __syncthreads();
        rho = rho2;
    }
    if (!ok && tid == 0) *a.fail = a.stat[0] = 1;
    if (near && wg == 0 && tid == 0) cgp_count(a.stat + 1);
    v = 0;
#pragma unroll
    for (int k = 0; k < C; ++k)
        if (k < cnt) {
            const long I = I0 + k * sz;
            a.x[I] = XL ? xl[k * NB + tid] : x[XL ? 0 : k];
            if (a.r2) {
                a.r[I] = r[k];
                const float zz = r[k] * id[k];
                if (zset) a.z[I] = zz;
                a.e[I] = zz;
                v = __builtin_fma((double)r[k], (double)r[k], v);
            }
        }
    if (a.r2) {
        v = wave_sum1(v);
        __syncthreads();
        if (lane == 0) shp[wv] = v;
        __syncthreads();
        if (tid == 0) {
            double t = 0;
            for (int q = 0; q < NB / 64; ++q) t += shp[q];
            a.r2[wg] = t;
        }
    }
}
// The variants: threads and cells per thread, the fewest first, as more cells per workgroup cost more than more
// workgroups up to CGP_ONE (32^3: 1.9 µs with 2 cells on 256 threads, 2.4 with 4 on 512).  8 cells on 512 threads take
// 3.37 µs at 64^3, 4 on 1024 (at their limit of 128 registers, with spills) 3.77; 16 on 512 hold the largest levels,
// where 8 on 1024 took 14.5 µs with spills.
struct CgpVariant {
    int D, NB, C, HC;
    void (*k)(CgpArgs);
};
inline const CgpVariant *cgp_variants(int &n) {
    static const CgpVariant v[] = {{2, 256, 1, 1, k_cgp<2, 256, 1, 1>}, {2, 256, 2, 1, k_cgp<2, 256, 2, 1>},
                                   {2, 512, 4, 1, k_cgp<2, 512, 4, 1>}, {2, 1024, 4, 1, k_cgp<2, 1024, 4, 1>},
                                   {3, 256, 1, 2, k_cgp<3, 256, 1, 2>}, {3, 256, 2, 3, k_cgp<3, 256, 2, 3>},
                                   {3, 512, 4, 3, k_cgp<3, 512, 4, 3>}, {3, 512, 8, 4, k_cgp<3, 512, 8, 4>},
                                   {3, 512, 16, 6, k_cgp<3, 512, 16, 6>}};
    n = 9;
    return v;
}
// pcg! in one launch: the variant of cgp_variants with the same number
typedef void (*PcgpKernel)(PcgpArgs);
inline PcgpKernel pcgp_kernel(int q) {
    static const PcgpKernel k[] = {k_pcgp<2, 256, 1, 1>, k_pcgp<2, 256, 2, 1>, k_pcgp<2, 512, 4, 1>,
                                   k_pcgp<2, 1024, 4, 1>, k_pcgp<3, 256, 1, 2>, k_pcgp<3, 256, 2, 3>,
                                   k_pcgp<3, 512, 4, 3>, k_pcgp<3, 512, 8, 4>, nullptr};
    return k[q];
}
// boxes of a level of n cells per axis for a variant, at most maxwg of them; false: none fits
inline bool cgp_boxes(const int *n, const CgpVariant &v, int maxwg, CgpBox &o) {
    long best = -1;
    for (int k2 = 1; k2 <= (v.D > 2 ? n[2] : 1) && k2 <= maxwg; ++k2)
        for (int k1 = 1; k1 <= n[1] && k1 * k2 <= maxwg; ++k1)
            for (int k0 = 1; k0 <= n[0] && (long)k0 * k1 * k2 <= maxwg; ++k0) {
                const int k[3] = {k0, k1, k2};
                int b[3] = {1, 1, 1};
                bool ok = true;
                for (int d = 0; d < v.D; ++d) {
                    b[d] = (n[d] + k[d] - 1) / k[d];
                    ok = ok && n[d] - (k[d] - 1) * b[d] >= 2;  // a box's two faces along an axis are different cells
                }
                if (!ok) continue;
                const long lat = (long)b[0] * (v.D > 2 ? b[1] : 1), thr = lat * ((b[v.D - 1] + v.C - 1) / v.C);
                const long f0 = (long)b[1] * b[2], f1 = (long)b[0] * b[2], f2 = v.D > 2 ? (long)b[0] * b[1] : 0;
                const long h = 2 * (f0 + f1 + f2);
                if (cgp_words(v.D, v.NB, v.C, b) * 4L > CGP_LDS) continue;
                if (thr > v.NB || h > (long)(v.NB - 64) * v.HC) continue;
                const long cost = (long)b[0] * b[1] * b[2] + h + (long)k0 * k1 * k2;
                if (best >= 0 && cost >= best) continue;
                best = cost;
                for (int d = 0; d < 3; ++d) {
                    o.k[d] = k[d];
                    o.b[d] = b[d];
                }
                o.nwg = k0 * k1 * k2;
                o.amax = (int)(f0 > f1 ? (f0 > f2 ? f0 : f2) : (f1 > f2 ? f1 : f2));
            }
    return best >= 0;
}

}  // namespace ia
