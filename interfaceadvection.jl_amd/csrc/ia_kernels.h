// ia_kernels.h -- kernels of the two-phase step (templated on the field type).
#pragma once
#include "ia_device.h"

namespace ia {

constexpr int NT = TX * TY;  // threads per block (256 = 4 wave64)

// ---------------------------------------------------------------------------
// block reductions (deterministic: fixed shuffle tree, fixed LDS order)
// ---------------------------------------------------------------------------
// a double moved across lanes by a DPP pattern (both halves; every source
// lane is inside the row, so the bound control never applies)
template <int CTRL> __device__ inline double dpp_d(double v) {
    int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
    int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ inline double lane_d(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// sum over the 64 lanes of a fully active wavefront, the same value in every
// lane: pairwise within each 16-lane row (lane pairs l^1, l^2 by quad
// permutes, then the half-row and row mirrors), each pair added in the same
// two operands by both of its lanes; then the four row sums in row order.
// DPP and readlane instead of LDS permutes keep it off the LDS pipeline.
__device__ inline double wave_sum(double v) {
    v += dpp_d<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_d<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_d<0x141>(v);  // row_half_mirror
    v += dpp_d<0x140>(v);  // row_mirror
    return ((lane_d(v, 0) + lane_d(v, 16)) + lane_d(v, 32)) + lane_d(v, 48);
}
__device__ inline double block_sum(double v) {
    __shared__ double sh[NT / 64];
    v = wave_sum(v);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int q = 0; q < NT / 64; ++q) s += sh[q];
    return s;  // valid in thread 0
}

// argmax/argmin partials of a VOF sweep (findmax/findmin, advection.jl:146-147)
struct FillPart {
    double vmax, vmin;
    long imax, imin;
    int nan, pad;
};
__device__ inline void fill_combine(FillPart &a, const FillPart &b) {
    if (b.vmax > a.vmax || (b.vmax == a.vmax && b.imax < a.imax)) { a.vmax = b.vmax; a.imax = b.imax; }
    if (b.vmin < a.vmin || (b.vmin == a.vmin && b.imin < a.imin)) { a.vmin = b.vmin; a.imin = b.imin; }
    a.nan |= b.nan;
}
// a wavefront's max / min of a double and the smallest index holding it, by
// the DPP pattern of wave_sum (order-independent)
template <int CTRL> __device__ inline long dpp_l(long v) {
    int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v & 0xffffffffL), CTRL, 0xF, 0xF, true);
    int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, 0xF, 0xF, true);
    return (long)(((unsigned long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ inline long lane_l(long v, int l) {
    unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v & 0xffffffffL), l);
    unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), l);
    return (long)(((unsigned long)hi << 32) | lo);
}
__device__ inline double wave_max_d(double v) {
    v = fmax(v, dpp_d<0xB1>(v));
    v = fmax(v, dpp_d<0x4E>(v));
    v = fmax(v, dpp_d<0x141>(v));
    v = fmax(v, dpp_d<0x140>(v));
    return fmax(fmax(fmax(lane_d(v, 0), lane_d(v, 16)), lane_d(v, 32)), lane_d(v, 48));
}
__device__ inline double wave_min_d(double v) {
    v = fmin(v, dpp_d<0xB1>(v));
    v = fmin(v, dpp_d<0x4E>(v));
    v = fmin(v, dpp_d<0x141>(v));
    v = fmin(v, dpp_d<0x140>(v));
    return fmin(fmin(fmin(lane_d(v, 0), lane_d(v, 16)), lane_d(v, 32)), lane_d(v, 48));
}
__device__ inline long wave_min_l(long v) {
    long t;
    t = dpp_l<0xB1>(v); v = t < v ? t : v;
    t = dpp_l<0x4E>(v); v = t < v ? t : v;
    t = dpp_l<0x141>(v); v = t < v ? t : v;
    t = dpp_l<0x140>(v); v = t < v ? t : v;
    long a = lane_l(v, 0), b = lane_l(v, 16), c = lane_l(v, 32), d = lane_l(v, 48);
    a = b < a ? b : a;
    a = c < a ? c : a;
    return d < a ? d : a;
}
// a block's combined FillPart, each wavefront by DPP (order-independent);
// valid in thread 0
__device__ inline FillPart block_fill(FillPart v) {
    __shared__ FillPart sh[NT / 64];
    FillPart p;
    p.vmax = wave_max_d(v.vmax);
    p.vmin = wave_min_d(v.vmin);
    p.imax = wave_min_l(v.vmax == p.vmax ? v.imax : (1L << 60));
    p.imin = wave_min_l(v.vmin == p.vmin ? v.imin : (1L << 60));
    p.nan = __ballot(v.nan != 0) != 0;
    p.pad = 0;
    __syncthreads();  // before sh is written again
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = p;
    __syncthreads();
    FillPart r = sh[0];
    if (threadIdx.x == 0)
        for (int q = 1; q < NT / 64; ++q) fill_combine(r, sh[q]);
    return r;
}
// a block's two maxima, sum, minimum and maximum; valid in thread 0.  The sum
// is block_sum's, wavefront by wavefront.
struct Red5 {
    double a, b, s, mn, mx;
};
__device__ inline Red5 block_red5(Red5 v) {
    __shared__ Red5 sh[NT / 64];
    v.a = wave_max_d(v.a);
    v.b = wave_max_d(v.b);
    v.s = wave_sum(v.s);
    v.mn = wave_min_d(v.mn);
    v.mx = wave_max_d(v.mx);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    Red5 r = sh[0];
    if (threadIdx.x == 0) {
        r.s = 0;
        for (int q = 0; q < NT / 64; ++q) {
            r.a = fmax(r.a, sh[q].a);
            r.b = fmax(r.b, sh[q].b);
            r.s += sh[q].s;
            r.mn = fmin(r.mn, sh[q].mn);
            r.mx = fmax(r.mx, sh[q].mx);
        }
    }
    return r;
}

// device-resident state of a step (flags) and of a solve (pcg scalars)
struct StepState {
    int status, nwarn;
    double maxf, minf;
    long imax, imin;
};
// what a step hands back to the host: written by its last kernel into pinned
// host memory (no copies)
struct StepOut {
    double cfl[5];  // the two CFL maxima, Σf, min f, max f
    StepState st;
    int fail;       // workgroups of a one-launch coarse solve did not run together
    int pad;
    double r2[256]; // the parts of Σr² of a one-launch pcg!
};

// ---------------------------------------------------------------------------
// c̄ = f≥½ (advection.jl:40, flow.jl:172) and ρu = u·ρ(f) (VOFutil.jl:208-211);
// with `st` the step's flags are cleared, with `zero` the vector field there
// (instead of two memsets' launches): all of it, or with `shell` the entries
// outside the interior, where the sweeps along every axis that follow write
// the rest.  Columns of cells: a workgroup's start costs more than a cell
// (200x132x148 FP32: 29.6 µs with one cell per thread, 18.0 with 8).
// ---------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(NT) k_prepare(Grid g, Tiling t, const T *__restrict__ f, const T *__restrict__ usrc,
                                                 T *__restrict__ ru, int8_t *__restrict__ cb, T lr, int do_ru,
                                                 StepState *st, T *__restrict__ zero, int shell) {
    if (st && blockIdx.x == 0 && threadIdx.x == 0) *st = StepState{0, 0, 0.0, 0.0, 0, 0};
    if (zero) {
        const long n = shell ? shell_size(g) : g.ns;
        for (long q = (long)blockIdx.x * NT + threadIdx.x; q < n * g.D; q += (long)gridDim.x * NT) {
            const long d = q / n;
            zero[g.ns * d + (shell ? shell_entry(g, q - n * d) : q - n * d)] = T(0);
        }
    }
    struct V {
        T f, m[3], u[3];
    };
    col_cells(
        g, t,
        [&](long I) {
            V v;
            v.f = f[I];
            if (do_ru)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (d < g.D) {
                        v.m[d] = f[I - g.st[d]];
                        v.u[d] = usrc[g.ns * d + I];
                    }
            return v;
        },
        [&](const int *p, long I, const V &v) {
            int8_t c = v.f < T(0.5) ? 0 : 1;
            write_row<int8_t>(g, cb, p, I, c);
            if (do_ru)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (d < g.D) ru[g.ns * d + I] = v.u[d] * linp((v.f + v.m[d]) / 2, lr);
        });
}

// ---------------------------------------------------------------------------
// one cVOF sweep along d in two passes: the face pass reconstructs each
// donor cell on the fly and computes every swept-volume face flux once; the
// cell pass makes the conservative update with the c̄ dilation term, the fill
// report, cleanWisp! and BCf! (advection.jl:80-137, normalEstimation.jl:10-28)
// ---------------------------------------------------------------------------
// the coordinates of flat index K of the ghost-inclusive grid; 32-bit
// division whenever the grid has fewer than 2^31 entries (64-bit integer
// division costs several times more)
__device__ inline void ghost_coord(const Grid &g, long K, int q[3]) {
    if (g.ns < (1L << 31)) {
        unsigned k = (unsigned)K, n0 = (unsigned)g.Ng[0], n1 = (unsigned)g.Ng[1];
        unsigned r = k / n0;
        q[0] = (int)(k - r * n0);
        q[1] = (int)(r % n1);
        q[2] = (int)(r / n1);
    } else {
        q[0] = (int)(K % g.Ng[0]);
        long r = K / g.Ng[0];
        q[1] = (int)(r % g.Ng[1]);
        q[2] = (int)(r / g.Ng[1]);
    }
}
template <class T> struct SweepArgs {
    Grid g;
    Tiling t, ct;        // of k_vof_face, of k_vof_update
    const T *fin;
    T *fout;
    const T *u1, *u2;    // face velocities, component d
    const int8_t *cb;
    T *ruf;              // mass flux, component d
    const T *fn;         // f^n for the mid-point f (predictor) or null
    T *fmid;
    FillPart *part;
    int d, scheme, mode; // mode 0: MPFMomStep! (ρuf·inv(δt) + BC!); 1: advect! (ρuf as computed)
    T dt, lr, idt, rtol, ctol, ubc_d;
};

// fup, fdn: f at the face's upper and lower cells, loaded with the face
// velocities (the donor is known only once δl's sign is)
template <class T>
__device__ inline T vof_face_flux(const SweepArgs<T> &a, const int q[3], long IF, T dl, T fup, T fdn) {
    const Grid &g = a.g;
    int d = a.d;
    int c[3] = {q[0], q[1], q[2]};
    if (dl > 0) c[d] -= 1;
    long IC = IF - (dl > 0 ? g.st[d] : 0);
    T fc = dl > 0 ? fdn : fup;
    bool ghost = c[d] == 0 || c[d] == g.Ng[d] - 1;
    if (fullorempty(fc) || (ghost && !g.per[d])) return fc * dl;
    long ICr = IC;
    if (ghost) {  // BCVOF! copies n̂, α of the periodic image (VOFutil.jl:44-62)
        int cc[3] = {c[0], c[1], c[2]};
        cc[d] = map_scalar(g, d, c[d]);
        ICr = lin(g, cc);
    }
    T n[3];
    if (g.D == 3 && a.scheme == 0) normal_wh_block3(g, a.fin, ICr, n);
    else normal_scheme(a.scheme, g, a.fin, ICr, n);
    T al = getIntercept(g.D, n, fc);
    T aa = dl > 0 ? al - n[d] * (1 - dl) : al;
    T nc[3];
    for (int ii = 0; ii < g.D; ++ii) nc[ii] = n[ii] * (ii == d ? fabs(dl) : T(1));
    return getVolumeFraction(g.D, nc, aa) * dl;
}

// pass 1 of a sweep: the swept-volume flux of every face along d, once (each
// cell's lower face; the last cell also its upper face), into `face`, and the
// mass flux ρuf of that face (advection.jl:108-137, flow.jl:207)
// the flux through the lower d-face of cell p (flat index I)
template <class T> __device__ inline void vof_face_one(const SweepArgs<T> &a, T *__restrict__ face, const int p[3],
                                                       long I) {
    const Grid &g = a.g;
    int d = a.d;
    T fup = a.fin[I], fdn = a.fin[I - g.st[d]];
    T dl = (a.dt / 2) * (a.u1[I] + a.u2[I]);
    T ff = dl == T(0) ? T(0) : vof_face_flux(a, p, I, dl, fup, fdn);
    face[I] = ff;
    T m = dl == T(0) ? T(0) : T(0) + (dl * a.lr + (1 - a.lr) * ff);
    if (a.mode == 0)
        m = !g.per[d] && (p[d] == 1 || (p[d] == g.Ng[d] - 1 && !(g.exitx && d == 0))) ? a.ubc_d : m * a.idt;
    a.ruf[I] = m;
}
template <class T>
__global__ void __launch_bounds__(NT) k_vof_face(SweepArgs<T> a, T *__restrict__ face) {
    const Grid &g = a.g;
    if (a.d == 0 && (long)blockIdx.x >= a.t.nblk) {
        // the blocks past the tiling: the upper x-face of each x-row
        int p[3];
        if (!top_face_x(g, (long)(blockIdx.x - a.t.nblk) * NT + threadIdx.x, p)) return;
        vof_face_one(a, face, p, lin(g, p));
        return;
    }
    int p[3];
    if (!thread_cell(g, a.t, p)) return;
    int d = a.d;
    long I = lin(g, p);
    vof_face_one(a, face, p, I);
    if (d != 0 && p[d] == g.Ng[d] - 2) {
        int pu[3] = {p[0], p[1], p[2]};
        pu[d] += 1;
        vof_face_one(a, face, pu, I + g.st[d]);
    }
}
// pass 2: the conservative update with the c̄ dilation term (advection.jl:83),
// fill-report partials, cleanWisp! (VOFutil.jl:127-137) and BCf!
template <class T>
__global__ void __launch_bounds__(NT) k_vof_update(SweepArgs<T> a, const T *__restrict__ face) {
    const Grid &g = a.g;
    struct V {
        T f, ff0, ff1, du, fn;
        int8_t c;
    };
    T mx = 0, mn = 0;
    long imx = 1L << 60, imn = 1L << 60;
    int nan = 0;
    col_cells(
        g, a.ct,
        [&](long I) {
            const long J = I + g.st[a.d];
            // the difference of each velocity, then their sum
            return V{a.fin[I], face[I], face[J], (a.u1[J] - a.u1[I]) + (a.u2[J] - a.u2[I]), a.fmid ? a.fn[I] : T(0),
                     a.cb[I]};
        },
        [&](const int *p, long I, const V &v) {
            T fnew = v.f + ((v.ff0 - v.ff1) + (((T)v.c * v.du) * a.dt) / 2);
            if (fnew != fnew) {
                nan = 1;
            } else {  // I grows along the column
                if (imx == 1L << 60 || fnew > mx) {
                    mx = fnew;
                    imx = I;
                }
                if (imn == 1L << 60 || fnew < mn) {
                    mn = fnew;
                    imn = I;
                }
            }
            T fc = fnew < a.ctol ? T(0) : (fnew > 1 - a.ctol ? T(1) : fnew);
            write_row<T>(g, a.fout, p, I, fc);
            if (a.fmid) write_row<T>(g, a.fmid, p, I, (fc + v.fn) / 2);
        });
    FillPart r;
    r.vmax = imx < 1L << 60 ? (double)mx : -1e300;
    r.vmin = imn < 1L << 60 ? (double)mn : 1e300;
    r.imax = imx;
    r.imin = imn;
    r.nan = nan;
    r.pad = 0;
    r = block_fill(r);
    if (threadIdx.x == 0) a.part[blockIdx.x] = r;
}

__device__ inline FillPart fill_identity() {
    FillPart acc;
    acc.vmax = -1e300;
    acc.vmin = 1e300;
    acc.imax = acc.imin = 1L << 60;
    acc.nan = 0;
    acc.pad = 0;
    return acc;
}
// first stage of the fill reduction: FILL_R2 blocks per sweep fold the
// per-block partials of each of gridDim.y sweeps (fill_combine is
// order-independent: ties go to the smallest index)
constexpr int FILL_R2 = 256;
__global__ void __launch_bounds__(NT) k_fill_reduce(const FillPart *part, long nblk, FillPart *out) {
    part += nblk * blockIdx.y;
    FillPart acc = fill_identity();
    for (long b = (long)blockIdx.x * NT + threadIdx.x; b < nblk; b += (long)gridDim.x * NT) fill_combine(acc, part[b]);
    FillPart r = block_fill(acc);
    if (threadIdx.x == 0) out[(long)gridDim.x * blockIdx.y + blockIdx.x] = r;
}
// reportFillError (advection.jl:145-189) on one sweep's partials (thread 0)
template <class T>
__device__ inline void fill_report(const Grid &g, const FillPart &r, const T *u1, const T *u2, double tol,
                                   StepState *st) {
    int s = 0;
    if (r.nan) s = 1;
    else {
        auto divabs = [&](const T *u, long I) {
            T sdiv = 0;
            for (int i = 0; i < g.D; ++i) sdiv += u[g.ns * i + I + g.st[i]] - u[g.ns * i + I];
            return fabs(sdiv);
        };
        if (r.vmax - 1 > tol) {
            T du0 = divabs(u1, r.imax), du = divabs(u2, r.imax);
            s = (du0 + du > T(10) || (du0 + du) != (du0 + du)) ? 2 : 3;
        }
        if (s != 2 && -r.vmin > tol) {
            T du0 = divabs(u1, r.imin), du = divabs(u2, r.imin);
            int s2 = (du0 + du > T(10) || (du0 + du) != (du0 + du)) ? 2 : 3;
            s = s2 == 2 ? 2 : (s ? s : s2);
        }
    }
    if (s == 3) st->nwarn += 1;
    int old = st->status;
    int worst = (old == 1 || s == 1) ? 1 : ((old == 2 || s == 2) ? 2 : (old > s ? old : s));
    if (worst != old && (s == 1 || s == 2 || old == 0)) {
        st->maxf = r.vmax;
        st->minf = r.vmin;
        st->imax = r.imax;
        st->imin = r.imin;
    }
    st->status = worst;
}
// The end of a run of sweeps, in one block: the sweeps' fill reports in their
// order (n partials each; u1, u2 still hold the velocities they were made
// with), then the CFL partials (ncfl > 0: k_cfl's, five values each), then
// everything into pinned host memory (out).  One launch where there were two
// per sweep, one for the CFL and two copies.
template <class T>
__global__ void __launch_bounds__(NT) k_step_finish(Grid g, const FillPart *part, long n, int nsweep, const T *u1,
                                                    const T *u2, double tol, StepState *st, const double *cfl,
                                                    long ncfl, StepOut *out) {
    StepState s = *st;
    for (int w = 0; w < nsweep; ++w) {
        FillPart acc = fill_identity();
        for (long b = threadIdx.x; b < n; b += NT) fill_combine(acc, part[n * w + b]);
        FillPart r = block_fill(acc);
        if (threadIdx.x == 0) fill_report(g, r, u1, u2, tol, &s);
    }
    if (ncfl > 0) {
        Red5 v{0, 0, 0, 1e300, -1e300};
        for (long q = threadIdx.x; q < ncfl; q += NT) {
            const double *o = cfl + 5 * q;
            v.a = o[0] > v.a ? o[0] : v.a;
            v.b = o[1] > v.b ? o[1] : v.b;
            v.s += o[2];
            v.mn = o[3] < v.mn ? o[3] : v.mn;
            v.mx = o[4] > v.mx ? o[4] : v.mx;
        }
        v = block_red5(v);
        if (threadIdx.x == 0 && out) {
            out->cfl[0] = v.a;
            out->cfl[1] = v.b;
            out->cfl[2] = v.s;
            out->cfl[3] = v.mn;
            out->cfl[4] = v.mx;
        }
    }
    if (threadIdx.x == 0) {
        *st = s;
        if (out) out->st = s;
    }
}

// ---------------------------------------------------------------------------
// CMOM momentum sweep along d with the SynDRoM blend (flow.jl:20-57, :212-241)
// ---------------------------------------------------------------------------
template <class T> struct MomArgs {
    Grid g;
    Tiling t;
    const T *ru_in;
    T *ru_out;
    const T *fpre;       // f before this sweep's VOF update (Φ), with ghosts
    const T *ruf;        // mass flux ×inv(δt), component d (BC! applied on read)
    const int8_t *cb;
    const T *u1, *u2;    // velocity component d (dilation)
    const T *uold;       // uOld (vector)
    T *us;               // uStar (vector, every cell incl. ghosts): the reference's n̂ alias
    int d, lim;
    T dt, lr;
    T ubc[3];
};

template <class T> __device__ inline T mom_ustar(const MomArgs<T> &a, int i, const int q[3]) {
    const Grid &g = a.g;
    // exitBC: BC! leaves uStar's exit face at what the reference's scratch r
    // (Flow.f) holds there: ρu2u! does not reach it and the forcing left 0
    // (g_x = 0) or the previous sweep's fill!(r, 0) (flow.jl:197, :215)
    if (exit_face(g, i, q)) return T(0);
    if (vel_dirichlet(g, i, q)) return a.ubc[i];
    long K = lin_vel(g, i, q);
    return a.ru_in[g.ns * i + K] / linp((a.fpre[K] + a.fpre[K - g.st[i]]) / 2, a.lr);
}
template <class T> __device__ inline T mom_drho(const MomArgs<T> &a, int i, const int q[3]) {
    const Grid &g = a.g;
    int qq[3];
    if (!face_map(g, i, q, qq)) return T(1);  // dρ = ones(...) is never written there (cVOF.jl:198)
    long K = lin(g, qq);
    return (a.fpre[K] + a.fpre[K - g.st[i]]) / 2;
}
// uStar at every cell of the ghost-inclusive grid (flow.jl:196-206 with the
// BC! images): computed once per sweep, read by every face that needs it
template <class T>
__global__ void __launch_bounds__(NT) k_ustar(MomArgs<T> a) {
    const Grid &g = a.g;
    long K = (long)blockIdx.x * NT + threadIdx.x;
    if (K >= g.ns) return;
    int q[3];
    ghost_coord(g, K, q);
    for (int i = 0; i < g.D; ++i) a.us[g.ns * i + K] = mom_ustar(a, i, q);
}
// the sweep with the axis d and the dimension as compile-time constants
template <int DIR, class T> __device__ inline T mom_ruf(const MomArgs<T> &a, const int q[3]) {
    const Grid &g = a.g;
    // exitBC: ρuf keeps the computed mass flux of the exit face (flow.jl:207)
    if (DIR == 0 && exit_face(g, 0, q))
        return a.ruf[(long)q[0] + g.st[1] * map_scalar(g, 1, q[1]) + g.st[2] * map_scalar(g, 2, q[2])];
    if (!g.per[DIR] && (q[DIR] == 0 || q[DIR] == 1 || q[DIR] == g.Ng[DIR] - 1)) return a.ubc[DIR];
    return a.ruf[lin_scalar(g, q[0], q[1], q[2])];
}
template <int DIR, class T> __device__ inline T mom_dila(const MomArgs<T> &a, const int q[3]) {
    const Grid &g = a.g;
    long K = lin_scalar(g, q[0], q[1], q[2]);
    long s = g.st[DIR];
    return (linp((T)a.cb[K], a.lr) * ((a.u1[K + s] - a.u1[K]) + (a.u2[K + s] - a.u2[K]))) / 2;
}
template <int DIR, class T>
__device__ inline T mom_phiq(const MomArgs<T> &a, int i, const int q[3], T Psi, T uu, T cc, T dd) {
    int c[3] = {q[0], q[1], q[2]};
    if (Psi > 0) c[DIR] -= 1;
    T vI = cc, vd = limiter(a.lim, uu, cc, dd);
    T va = 2 * vI - vd;
    T mOut = fabs(Psi) * a.dt;
    T mOld = linp(mom_drho(a, i, c), a.lr);
    if (mOut > mOld) return Psi * vI;
    T l2 = fabs(mOut) / mOld, l1 = 1 - l2;
    T vb = l2 * va + l1 * vd;
    return (Psi * (vb + vd)) / 2;
}
template <int DIR, class T> __device__ inline T mom_face(const MomArgs<T> &a, int i, const int qin[3]) {
    const Grid &g = a.g;
    int n = g.Ng[DIR];
    int q[3] = {qin[0], qin[1], qin[2]};
    if (g.per[DIR] && q[DIR] == n - 1) q[DIR] = 1;  // flow.jl:241 reuses the lower-boundary flux
    int qm[3] = {q[0], q[1], q[2]};
    qm[i] -= 1;
    T Psi = (mom_ruf<DIR>(a, q) + mom_ruf<DIR>(a, qm)) / 2;
    const T *__restrict__ us = a.us + g.ns * i;
    long Q = lin(g, q), sd = g.st[DIR];
    auto u = [&](int off) { return us[Q + off * sd]; };
    // the limiter's (upwind, centre, downwind) triple for the sign of Psi,
    // selected first so that a wave whose lanes differ in sign evaluates the
    // face value once
    T uu, cc, dd;
    if (q[DIR] == 1 && !g.per[DIR]) {  // ϕuL
        T c0 = u(0), cm = u(-1);
        bool pos = Psi > 0;
        uu = pos ? 2 * cm - c0 : u(1);
        cc = pos ? cm : c0;
        dd = pos ? c0 : cm;
    } else if (q[DIR] == 1) {  // ϕuP: the far-upwind value is the periodic image of I-2δ
        bool pos = Psi > 0;
        uu = pos ? u(n - 4) : u(1);
        cc = pos ? u(-1) : u(0);
        dd = pos ? u(0) : u(-1);
    } else if (q[DIR] == n - 1) {  // ϕuR
        T c0 = u(0), cm = u(-1);
        bool neg = Psi < 0;
        uu = neg ? 2 * c0 - cm : u(-2);
        cc = neg ? c0 : cm;
        dd = neg ? cm : c0;
    } else {
        bool pos = Psi > 0;
        uu = pos ? u(-2) : u(1);
        cc = pos ? u(-1) : u(0);
        dd = pos ? u(0) : u(-1);
    }
    return mom_phiq<DIR>(a, i, q, Psi, uu, cc, dd);
}
// the momentum sweep along DIR in two passes.  Face pass: the SynDRoM face
// flux of every component at every face along DIR, once (each cell's lower
// face; the last cell also its upper face), into `face` (components last)
template <int D, int DIR, class T>
__global__ void __launch_bounds__(NT) k_mom_face(MomArgs<T> a, T *__restrict__ face) {
    const Grid &g = a.g;
    int p[3];
    if (DIR == 0 && (long)blockIdx.x >= a.t.nblk) {
        // the blocks past the tiling: the upper x-face of each x-row
        if (!top_face_x(g, (long)(blockIdx.x - a.t.nblk) * NT + threadIdx.x, p)) return;
        long It = lin(g, p);
#pragma unroll
        for (int i = 0; i < D; ++i) face[g.ns * i + It] = mom_face<DIR>(a, i, p);
        return;
    }
    if (!thread_cell(g, a.t, p)) return;
    long I = lin(g, p), sd = g.st[DIR];
    bool top = DIR != 0 && p[DIR] == g.Ng[DIR] - 2;
    int pu[3] = {p[0], p[1], p[2]};
    pu[DIR] += 1;
    // every component's face value before any store, so that the loads of
    // the components overlap (a store could alias them)
    T fv[D];
#pragma unroll
    for (int i = 0; i < D; ++i) fv[i] = mom_face<DIR>(a, i, p);
#pragma unroll
    for (int i = 0; i < D; ++i) face[g.ns * i + I] = fv[i];
    if (top) {
#pragma unroll
        for (int i = 0; i < D; ++i) fv[i] = mom_face<DIR>(a, i, pu);
#pragma unroll
        for (int i = 0; i < D; ++i) face[g.ns * i + I + sd] = fv[i];
    }
}
// cell pass: the two-pass difference of the face fluxes, the uOld dilation
// term and ρu += δt·r (flow.jl:216-231)
template <int D, int DIR, class T>
__global__ void __launch_bounds__(NT) k_mom_update(MomArgs<T> a, const T *__restrict__ face) {
    const Grid &g = a.g;
    int p[3];
    if (!thread_cell(g, a.t, p)) return;
    long I = lin(g, p), sd = g.st[DIR];
    T dl0 = mom_dila<DIR>(a, p);
    T rn[D];  // every component before any store (a store could alias the loads)
#pragma unroll
    for (int i = 0; i < D; ++i) {
        T flo = face[g.ns * i + I], fup = face[g.ns * i + I + sd];
        int pm[3] = {p[0], p[1], p[2]};
        pm[i] -= 1;
        T r = (T(0) + flo) - fup;
        r += a.uold[g.ns * i + I] * ((dl0 + mom_dila<DIR>(a, pm)) / 2);
        long o = g.ns * i + I;
        rn[i] = a.ru_in[o] + a.dt * r;
    }
#pragma unroll
    for (int i = 0; i < D; ++i) a.ru_out[g.ns * i + I] = rn[i];
}
// ---------------------------------------------------------------------------
// viscous stress (flow.jl:113-153) fused with the RK update (flow.jl:244-252)
// and the Poisson coefficients (flow.jl:254-259)
// ---------------------------------------------------------------------------
template <class T> struct ViscArgs {
    Grid g;
    Tiling t;
    const T *u;       // velocity the stress is taken from (ghosts valid)
    const T *fv;      // f for the face fractions
    const T *ff;      // the face fractions fFace (every cell incl. ghosts): the reference's n̂ alias
    T lm, mu, lr;
    T ubc[3];
    int has_mu;
};
// face fraction fFace[q, c] as left by f2face!/BCv! into n̂ (VOFutil.jl:229-234)
template <class T> __device__ inline T visc_ff(const ViscArgs<T> &a, int c, const int q[3]) {
    const Grid &g = a.g;
    int qq[3];
    // n̂ there still holds uStar (flow.jl:206): u_BC, or 0 on the exit face under exitBC
    if (!face_map(g, c, q, qq)) return exit_face(g, c, q) ? T(0) : a.ubc[c];
    long K = lin(g, qq);
    return (a.fv[K] + a.fv[K - g.st[c]]) / 2;
}
// f2face! + BCv! into n̂ (VOFutil.jl:229-234): fFace at every cell of the
// ghost-inclusive grid, once per use
template <class T>
__global__ void __launch_bounds__(NT) k_fface(ViscArgs<T> a, T *ff) {
    const Grid &g = a.g;
    long K = (long)blockIdx.x * NT + threadIdx.x;
    if (K >= g.ns) return;
    int q[3];
    ghost_coord(g, K, q);
    for (int c = 0; c < g.D; ++c) ff[g.ns * c + K] = visc_ff(a, c, q);
}
// viscF(i, j, Q) (flow.jl:144, getμ VOFutil.jl:186-191) on loaded values:
// f1..f4 the face fractions ff_i[Q-δj], ff_i[Q], ff_j[Q-δi], ff_j[Q]; then
// u_i[Q], u_i[Q-δj], u_j[Q], u_j[Q-δi]
template <class T>
__device__ inline T viscF_v(const ViscArgs<T> &a, T f1, T f2, T f3, T f4, T ui, T uim, T uj, T ujm) {
    T s = (((f1 + f2) + f3) + f4) / 4;
    T fr = a.lr < T(1) ? tmin(tmin(tmin(f1, f2), f3), f4) : tmax(tmax(tmax(f1, f2), f3), f4);
    T mu = a.mu * tmin(linp(s, a.lm), (s > T(0.5) ? T(1) : a.lm / a.lr) * linp(fr, a.lr));
    return mu * ((ui - uim) + (uj - ujm));
}
// the viscous force of every component of cell p (visc!, flow.jl:119-138):
// F_i = Σ_j -viscF(i,j,p) + viscF(i,j,p+δj), with each value loaded once.
// The D² viscF at p share the face fractions and velocities of p and its
// lower neighbours; viscF(i,j,p+δj) reads p's values again at its lower
// j-side (q wraps to the first interior cell on a periodic axis, flow.jl:153).
template <int D, class T> __device__ inline void visc_force_all(const ViscArgs<T> &a, const int p[3], T F[D]) {
    if (!a.has_mu) {
#pragma unroll
        for (int i = 0; i < D; ++i) F[i] = T(0);
        return;
    }
    const Grid &g = a.g;
    const T *__restrict__ ff = a.ff;
    const T *__restrict__ u = a.u;
    const long ns = g.ns, I = lin(g, p);
    T ffc[D], uc[D], ffm[D][D], um[D][D];  // [c][k]: component c at I - δk
#pragma unroll
    for (int c = 0; c < D; ++c) {
        ffc[c] = ff[ns * c + I];
        uc[c] = u[ns * c + I];
#pragma unroll
        for (int k = 0; k < D; ++k) {
            ffm[c][k] = ff[ns * c + I - g.st[k]];
            um[c][k] = u[ns * c + I - g.st[k]];
        }
    }
#pragma unroll
    for (int i = 0; i < D; ++i) F[i] = 0;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        // q = p + δj, wrapped to the first interior cell on a periodic axis (flow.jl:153)
        bool wrap = g.per[j] && p[j] + 1 == g.Ng[j] - 1;
        long Q = wrap ? I - (long)(g.Ng[j] - 3) * g.st[j] : I + g.st[j];
        T ffq[D], uq[D], ffjm[D], ujm[D];  // at Q: every component; component j at Q - δi
#pragma unroll
        for (int c = 0; c < D; ++c) {
            ffq[c] = ff[ns * c + Q];
            uq[c] = u[ns * c + Q];
        }
        T ffb[D], ub[D];  // every component at Q - δj (p itself unless wrapped)
#pragma unroll
        for (int c = 0; c < D; ++c) {
            ffb[c] = wrap ? ff[ns * c + Q - g.st[j]] : ffc[c];
            ub[c] = wrap ? u[ns * c + Q - g.st[j]] : uc[c];
        }
#pragma unroll
        for (int i = 0; i < D; ++i) {
            ffjm[i] = i == j ? ffb[j] : ff[ns * j + Q - g.st[i]];
            ujm[i] = i == j ? ub[j] : u[ns * j + Q - g.st[i]];
        }
#pragma unroll
        for (int i = 0; i < D; ++i) {
            T lo = viscF_v(a, ffm[i][j], ffc[i], ffm[j][i], ffc[j], uc[i], um[i][j], uc[j], um[j][i]);
            T hi = viscF_v(a, ffb[i], ffq[i], ffjm[i], ffq[j], uq[i], ub[i], uq[j], ujm[i]);
            F[i] += -lo;
            F[i] -= -hi;
        }
    }
}

// ---------------------------------------------------------------------------
// diagnostics (metrics.jl:15-50) integrated over the interior, in FP64:
// Σρke, Σρu_i, Σρgh, Σ enstrophy (ω by backward differences at the cell's
// lower edges, which EnsI averages), Σf.  Seven block partials per block.
// ---------------------------------------------------------------------------
template <int D, class T> __device__ inline double vort_edge(const Grid &g, const T *u, long I, int a) {
    if (D == 2) {
        return (double)((u[g.ns + I] - u[g.ns + I - g.st[0]]) - (u[I] - u[I - g.st[1]]));
    }
    int j = (a + 1) % 3, k = (a + 2) % 3;
    return (double)((u[g.ns * k + I] - u[g.ns * k + I - g.st[j]]) - (u[g.ns * j + I] - u[g.ns * j + I - g.st[k]]));
}
// the metrics.jl integrands of interior cell p added into acc[0..6]
template <int D, class T>
__device__ inline void metrics_cell(const Grid &g, const T *u, const T *f, T lr, const double U[3], const double gv[3],
                                    const double wl[3], const int p[3], double acc[7]) {
    long I = lin(g, p);
    double rho = (double)linp(f[I], lr);
    double ke = 0, pe = 0;
    for (int i = 0; i < D; ++i) {
        const T *ui = u + g.ns * i;
        double a = (double)ui[I] - U[i], b = (double)ui[I + g.st[i]] - U[i];
        ke += (a * a + b * b) * rho;
        acc[1 + i] += 0.5 * (((double)ui[I] + (double)ui[I + g.st[i]]) - 2 * U[i]) * rho;
        pe += gv[i] * ((p[i] - 0.5) - wl[i]);
    }
    acc[0] += 0.25 * ke;
    acc[4] += -rho * pe;
    double en = 0;
    if (D == 2) {
        double a = vort_edge<D>(g, u, I, 0), b = vort_edge<D>(g, u, I + g.st[0], 0),
               c = vort_edge<D>(g, u, I + g.st[1], 0), d = vort_edge<D>(g, u, I + g.st[0] + g.st[1], 0);
        en = ((a * a + b * b) + c * c) + d * d;
    } else {
        for (int i = 0; i < 3; ++i) {
            int ix = (i + 1) % 3, iy = (i + 2) % 3;
            double a = vort_edge<D>(g, u, I, i), b = vort_edge<D>(g, u, I + g.st[ix], i),
                   c = vort_edge<D>(g, u, I + g.st[iy], i), d = vort_edge<D>(g, u, I + g.st[ix] + g.st[iy], i);
            en += ((a * a + b * b) + c * c) + d * d;
        }
    }
    acc[5] += 0.5 * 0.25 * en;
    acc[6] += (double)f[I];
}
template <int D, class T>
__global__ void __launch_bounds__(NT) k_metrics(Grid g, Tiling t, const T *u, const T *f, T lr, double U0, double U1,
                                                double U2, double g0, double g1, double g2, double w0, double w1,
                                                double w2, double *part) {
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    int p[3];
    if (thread_cell(g, t, p)) {
        double U[3] = {U0, U1, U2}, gv[3] = {g0, g1, g2}, wl[3] = {w0, w1, w2};
        metrics_cell<D, T>(g, u, f, lr, U, gv, wl, p, acc);
    }
    for (int q = 0; q < 7; ++q) {
        double s = block_sum(acc[q]);
        if (threadIdx.x == 0) part[(long)blockIdx.x * 7 + q] = s;
    }
}

// ---------------------------------------------------------------------------
// surface tension (surfaceTension.jl:7-124), per momentum direction d
// ---------------------------------------------------------------------------
template <class T> __device__ inline bool contain_if(T v) { return v > T(0) && v < T(1); }  // VOFutil.jl:144
// getPopinetHeightAdaptive(I, f, i, monotonic=true) about cell p (0-based,
// ghost-inclusive) along the signed axis i (1-based): to the air side, then to
// the water side; a walk stops at the array's end (validCI, util.jl:82)
template <class T> __device__ inline T popinet_height(const Grid &g, const T *f, const int p[3], int i) {
    int ax = abs(i) - 1, s = i > 0 ? 1 : -1;
    long st = g.st[ax] * s;
    long I0 = lin(g, p);
    T fnow = f[I0], H = fnow - T(0.5);
    bool fin = fnow < T(1);
    int c = p[ax];
    long In = I0;
    while (!fin || contain_if(fnow)) {
        c += s;
        In += st;
        if (c < 0 || c > g.Ng[ax] - 1) break;
        T v = f[In];
        fnow = v > fnow ? T(0) : v;
        H += fnow;
        if (contain_if(fnow)) fin = true;
    }
    fnow = f[I0];
    fin = fnow > T(0);
    c = p[ax];
    In = I0;
    while (!fin || contain_if(fnow)) {
        c -= s;
        In -= st;
        if (c < 0 || c > g.Ng[ax] - 1) break;
        T v = f[In];
        fnow = v < fnow ? T(1) : v;
        H += fnow - 1;
        if (contain_if(fnow)) fin = true;
    }
    return H;
}
template <class T> __device__ inline T root1p5(T a) { return sqrt((a * a) * a); }  // surfaceTension.jl:89
// getCurvature (surfaceTension.jl:35-80) with getXdir / getXYdir (util.jl:62-63):
// the cell of its k-th height about q along the signed axis i, H[u+1] in 2D,
// H[u+1][v+1] in 3D
template <int D> __device__ inline void height_cell(int i, int k, int q[3]) {
    const int s = i > 0 ? 1 : -1, ai = abs(i);
    const int ix = D == 2 ? (ai == 1 ? -2 * s : s) : s * (ai % 3 + 1);
    const int du = (D == 2 ? k - 1 : k / 3 - 1) * (ix > 0 ? 1 : -1), iy = (ai + 1) % 3;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (a == abs(ix) - 1) q[a] += du;
        if (D == 3 && a == iy) q[a] += k % 3 - 1;
    }
}
template <int D, class T> __device__ inline T curvature(const T (&h)[D == 3 ? 9 : 3]) {
    if constexpr (D == 2) {
        T Hx = (h[2] - h[0]) / 2;
        T Hxx = (h[2] + h[0]) - 2 * h[1];
        return Hxx / root1p5(1 + Hx * Hx);
    } else {
        T H[3][3], flt = T(0.2);
#pragma unroll
        for (int k = 0; k < 9; ++k) H[k / 3][k % 3] = h[k];
        T Hx = (H[2][1] - H[0][1]) / 2, Hy = (H[1][2] - H[1][0]) / 2;
        T Hxx = (((H[2][1] + H[0][1]) - 2 * H[1][1]) + ((H[2][0] + H[0][0]) - 2 * H[1][0]) * flt +
                 ((H[2][2] + H[0][2]) - 2 * H[1][2]) * flt) / (1 + 2 * flt);
        T Hyy = (((H[1][2] + H[1][0]) - 2 * H[1][1]) + ((H[0][2] + H[0][0]) - 2 * H[0][1]) * flt +
                 ((H[2][2] + H[2][0]) - 2 * H[2][1]) * flt) / (1 + 2 * flt);
        T Hxy = (((H[2][2] + H[0][0]) - H[2][0]) - H[0][2]) / 4;
        return ((Hxx * (1 + Hy * Hy) + Hyy * (1 + Hx * Hx)) - ((2 * Hxy) * Hx) * Hy) /
               root1p5((1 + Hx * Hx) + Hy * Hy);
    }
}
// The forcing's buffer of direction d is component d of a vector, so that one
// launch serves all directions: in a launch for one of them most wavefronts
// end at once and the few at the interface leave the chip idle.
// fbuffer[I] = ϕ(d, I, f) = (f[I] + f[I-δd]) / 2 on the interior
template <class T> __global__ void __launch_bounds__(NT) k_st_fbuf(Grid g, Tiling t, const T *f, T *fb) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    for (int d = 0; d < g.D; ++d) fb[g.ns * d + I] = (f[I] + f[I - g.st[d]]) / 2;
}
// BCf!(d, fbuffer) on the ghost planes of axis j (VOFutil.jl:76-89), axis by
// axis as the reference loops; the upper plane of axis d, which BCf!(d, ·)
// does not write, is set to 0
template <class T> __global__ void __launch_bounds__(NT) k_st_bc(Grid g, T *fb, int j) {
    long n = g.ns / g.Ng[j];
    long q = (long)blockIdx.x * NT + threadIdx.x;
    if (q >= n) return;
    const int d = blockIdx.y;
    fb += g.ns * d;
    int c[3];
    long r = q;
    for (int a = 0; a < 3; ++a) {
        if (a == j) continue;
        c[a] = (int)(r % g.Ng[a]);
        r /= g.Ng[a];
    }
    c[j] = 0;
    long lo = lin(g, c), st = g.st[j], N = g.Ng[j];
    long hi = lo + (N - 1) * st;
    if (g.per[j]) {
        fb[lo] = fb[lo + (N - 2) * st];
        fb[hi] = fb[lo + st];
    } else if (j == d) {
        fb[lo] = fb[lo + 2 * st];
        fb[hi] = T(0);
    } else {
        fb[lo] = fb[lo + st];
        fb[hi] = fb[hi - st];
    }
}
// forcing[I,d] (+)= η κ(I, fbuffer, majorDir) (-∂_d f) at interface cells of
// fbuffer, 0 elsewhere (surfaceTension.jl:7-19).  A height is a walk of
// dependent loads and a curvature takes nine of them (three in 2D), but few of
// a wavefront's cells are at the interface: its heights are dealt out to all
// lanes, one each (48³ FP64: 54 µs a direction with each cell walking its own
// nine, 26 all three together).
template <int D, class T>
__global__ void __launch_bounds__(NT) k_surften(Grid g, Tiling t, const T *fbv, const T *f, T eta, T *out, int acc) {
    constexpr int NH = D == 3 ? 9 : 3, PER = 64 / NH;  // heights of a cell, cells at a time
    __shared__ unsigned char who[NT / 64][64];
    int p[3];
    const int d = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool in = thread_cell(g, t, p);
    const long I = in ? lin(g, p) : 0;
    const T *fb = fbv + g.ns * d;
    const bool hit = in && contain_if(fb[I]);
    int i = 1;  // the major direction
    if (hit) {
        T n[3];
        normal_wy(g, fb, I, n);
        int im = argabsmax(g.D, n);
        i = (signbit(n[im]) ? -1 : 1) * (im + 1);
    }
    const unsigned long long m = __ballot(hit);
    const int rank = __popcll(m & ((1ull << lane) - 1)), nhit = __popcll(m);
    if (hit) who[wv][rank] = (unsigned char)lane;
    wave_lds_order();
    T H[NH];
    for (int b = 0; b < nhit; b += PER) {
        const int s = lane / NH, k = lane % NH;
        const bool on = s < PER && b + s < nhit;
        const int src = on ? who[wv][b + s] : lane;
        int q[3] = {__shfl(p[0], src), __shfl(p[1], src), __shfl(p[2], src)};
        const int qi = __shfl(i, src);
        T h = 0;
        if (on) {
            height_cell<D>(qi, k, q);
            h = popinet_height(g, fb, q, qi);
        }
#pragma unroll
        for (int j = 0; j < NH; ++j) {
            const T v = __shfl(h, ((rank - b) * NH + j) & 63);
            if (hit && rank >= b && rank < b + PER) H[j] = v;
        }
    }
    if (!in) return;
    const T st = hit ? eta * curvature<D>(H) * -(f[I] - f[I - g.st[d]]) : T(0);
    long o = g.ns * d + I;
    if (!acc) out[o] = st;
    else if (hit) out[o] = out[o] + st;
}

template <class T> struct UpdArgs {
    ViscArgs<T> v;
    const T *u0;      // Flow.u⁰ (for ρu⁰ = u⁰ρ(f_cur), flow.jl:76/:99)
    const T *fcur;    // cVOF.f
    const T *fupd;    // f of the update and of the coefficients
    const T *ru;      // ρu after advection
    T *uout;
    T *L;             // μ₀
    const T *st;      // surface tension forcing (vector), or nullptr when η == nothing
    T dt, w, g[3];
};
template <int D, class T>
__global__ void __launch_bounds__(NT) k_visc_update(UpdArgs<T> a) {
    const Grid &g = a.v.g;
    int p[3];
    if (!thread_cell(g, a.v.t, p)) return;
    long I = lin(g, p);
    T wT = a.w, ac = T(1) / wT - 1;
    // every component's stress divergence first: its loads then share one
    // another's addresses, as no store intervenes
    T Fv[D];
    visc_force_all<D>(a.v, p, Fv);
    T un[D], rh[D];  // every component before any store (a store could alias the loads)
#pragma unroll
    for (int i = 0; i < D; ++i) {
        long o = g.ns * i + I;
        T F = Fv[i];
        if (a.st) F = F + a.st[o];
        T ru0 = a.u0[o] * linp((a.fcur[I] + a.fcur[I - g.st[i]]) / 2, a.v.lr);
        T run = ((ac * ru0 + a.ru[o]) + F * a.dt) * wT;
        T rho = linp((a.fupd[I] + a.fupd[I - g.st[i]]) / 2, a.v.lr);
        T u1 = run / rho;
        un[i] = u1 + (a.dt * wT) * a.g[i];
        rh[i] = rho;
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
        // exitBC: updateU!'s axpy! (flow.jl:251) is the only update of the exit face
        T xv = i == 0 && g.exitx ? a.v.u[I + g.st[0]] + (a.dt * wT) * a.g[0] : T(0);
        write_row_u<T>(g, a.uout + g.ns * i, p, I, un[i], true, i, a.v.ubc[i], xv);
        write_row_u<T>(g, a.L + g.ns * i, p, I, T(1) / rh[i], false, i, T(0));
    }
}
// viscSurfTenρu! alone (stage entry point): Flow.f = visc
template <int D, class T>
__global__ void __launch_bounds__(NT) k_visc_force(ViscArgs<T> a, T *F) {
    const Grid &g = a.g;
    int p[3];
    if (!thread_cell(g, a.t, p)) return;
    long I = lin(g, p);
    T Fv[D];
    visc_force_all<D>(a, p, Fv);
#pragma unroll
    for (int i = 0; i < D; ++i) F[g.ns * i + I] = Fv[i];
}
// updateL! alone (stage entry point)
template <class T>
__global__ void __launch_bounds__(NT) k_update_L(Grid g, Tiling t, const T *f, T *L, T lr) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    for (int i = 0; i < g.D; ++i)
        write_row_u<T>(g, L + g.ns * i, p, I, T(1) / linp((f[I] + f[I - g.st[i]]) / 2, lr), false, i, T(0));
}

// z = div(u); (flow.jl:345)
template <class T>
__global__ void __launch_bounds__(NT) k_div(Grid g, Tiling t, const T *u, T *z) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    T s = 0;
    for (int i = 0; i < g.D; ++i) s += u[g.ns * i + I + g.st[i]] - u[g.ns * i + I];
    z[I] = s;
}
template <class T>
__global__ void k_scale(T *x, long n, T s) {
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) x[q] = x[q] * s;
}
template <class T>
__global__ void k_fill(T *x, long n, T v) {
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) x[q] = v;
}
template <class T> __device__ inline T xper(const Grid &g, const T *x, int p0, int p1, int p2) {
    return x[(long)map_per(g, 0, p0) + g.st[1] * map_per(g, 1, p1) + g.st[2] * map_per(g, 2, p2)];
}
template <class T>
__global__ void __launch_bounds__(NT) k_set_diag(Grid g, Tiling t, const T *L, T *Dg, T *iD) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    T s = 0;
    for (int d = 0; d < g.D; ++d) s -= (L[g.ns * d + I] + L[g.ns * d + I + g.st[d]]);
    Dg[I] = s;
    iD[I] = (s * s) < 2 * eps_of<T>() ? T(0) : T(1) / s;
}
// the coarse coefficient of the lower face along ii of the cell p (restrictL!:
// half the sum of the fine faces it covers), from the finer level's
template <int D, class T>
__device__ inline T coarse_face(const Grid &gf, const T *__restrict__ Lf, const int p[3], int ii) {
    const T *b = Lf + gf.ns * ii + (2 * p[0] - 1) + gf.st[1] * (2 * p[1] - 1) + (D > 2 ? gf.st[2] * (2 * p[2] - 1) : 0);
    T v[1 << (D - 1)];
#pragma unroll
    for (int k = 0; k < (1 << (D - 1)); ++k) {  // the other axes' offsets, lower axes first
        const int a0 = ii == 0 ? 1 : 0, a1 = D > 2 && ii < 2 ? 2 : 1;
        v[k] = b[(k & 1) * gf.st[a0] + (D > 2 ? (k >> 1) * gf.st[a1] : 0)];
    }
    T s = 0;
#pragma unroll
    for (int k = 0; k < (1 << (D - 1)); ++k) s += v[k];
    return (T)(0.5 * (double)s);
}
// restrictL! and the diagonal of coarse cell p in one go: the upper faces'
// coefficients are formed again here instead of being read back by a second
// launch
template <int D, class T>
__device__ inline void coarse_cell(const Grid &gc, const Grid &gf, const T *__restrict__ Lf, T *__restrict__ Lc,
                                   T *__restrict__ Dg, T *__restrict__ iD, const int p[3]) {
    T lo[D], up[D], s = 0;
#pragma unroll
    for (int ii = 0; ii < D; ++ii) {  // 0 on walls
        lo[ii] = up[ii] = T(0);
        int q[3] = {p[0], p[1], p[2]};
        if (gc.per[ii] || p[ii] > 1) lo[ii] = coarse_face<D>(gf, Lf, q, ii);
        q[ii] = p[ii] < gc.Ng[ii] - 2 ? p[ii] + 1 : 1;
        if (gc.per[ii] || q[ii] > 1) up[ii] = coarse_face<D>(gf, Lf, q, ii);
    }
#pragma unroll
    for (int ii = 0; ii < D; ++ii) s -= (lo[ii] + up[ii]);
#pragma unroll
    for (int ii = 0; ii < D; ++ii) write_images<T>(gc, Lc + gc.ns * ii, p, lo[ii], 1, ii, T(0));
    long I = lin(gc, p);
    Dg[I] = s;
    iD[I] = (s * s) < 2 * eps_of<T>() ? T(0) : T(1) / s;
}
template <class T>
__global__ void __launch_bounds__(NT) k_coarse_level(Grid gc, Tiling t, Grid gf, const T *Lf, T *Lc, T *Dg, T *iD) {
    int p[3];
    if (!thread_cell(gc, t, p)) return;
    if (gc.D == 3) coarse_cell<3>(gc, gf, Lf, Lc, Dg, iD, p);
    else coarse_cell<2>(gc, gf, Lf, Lc, Dg, iD, p);
}
// the same for the levels of at most MGU_NT cells, one after the other in one
// workgroup: a launch of 3-4 µs less per level
constexpr int MGU_LEV = 12, MGU_NT = 1024;
template <class T> struct MguArgs {
    Grid g[MGU_LEV];
    T *L[MGU_LEV], *Dg[MGU_LEV], *iD[MGU_LEV];
    int l0, nlev;  // levels l0 (>= 1) .. nlev-1
};
template <class T> __global__ void __launch_bounds__(MGU_NT) k_coarse_levels(MguArgs<T> a) {
    for (int l = a.l0; l < a.nlev; ++l) {
        const Grid gc = a.g[l], gf = a.g[l - 1];
        const int n0 = gc.Ng[0] - 2, n1 = gc.Ng[1] - 2, n2 = gc.D > 2 ? gc.Ng[2] - 2 : 1;
        for (int c = threadIdx.x; c < n0 * n1 * n2; c += MGU_NT) {
            int r = c / n0;
            int p[3] = {1 + c - r * n0, 1 + r % n1, gc.D > 2 ? 1 + r / n1 : 0};
            if (gc.D == 3) coarse_cell<3>(gc, gf, a.L[l - 1], a.L[l], a.Dg[l], a.iD[l], p);
            else coarse_cell<2>(gc, gf, a.L[l - 1], a.L[l], a.Dg[l], a.iD[l], p);
        }
        __threadfence_block();
        __syncthreads();
    }
}
// myproject!: u -= L ∂x ; BC!(u)  (flow.jl:331-333, :82)
template <class T>
__global__ void __launch_bounds__(NT) k_project(Grid g, Tiling t, T *u, const T *L, const T *x, T ubc0, T ubc1, T ubc2) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    T ub[3] = {ubc0, ubc1, ubc2};
    for (int i = 0; i < g.D; ++i) {
        int q[3] = {p[0], p[1], p[2]};
        q[i] -= 1;
        T dx = x[I] - xper(g, x, q[0], q[1], q[2]);
        T un = u[g.ns * i + I] - L[g.ns * i + I] * dx;
        T xv = i == 0 && g.exitx ? u[I + g.st[0]] : T(0);  // exitBC: the exit face is left alone
        write_row_u<T>(g, u + g.ns * i, p, I, un, true, i, ub[i], xv);
    }
}
// applyVOF! from SDF samples (VOFutil.jl:203-225) + cleanWisp! + BCf!
template <class T>
__global__ void __launch_bounds__(NT) k_apply_vof(Grid g, Tiling t, const T *sdf, T *f, T *al, T *nh, T ctol) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    long q = (long)(p[0] - 1) + (long)(g.Ng[0] - 2) * ((g.D > 1 ? p[1] - 1 : 0) + (long)(g.D > 1 ? g.Ng[1] - 2 : 1) * (g.D > 2 ? p[2] - 1 : 0));
    const T *s = sdf + q * (1 + 2 * g.D);
    T sumN = 0, sumN2 = 0, n[3];
    for (int d = 0; d < g.D; ++d) {
        T dd = s[2 * d + 1] - s[2 * d + 2];
        nh[g.ns * d + I] = dd;
        n[d] = dd;
        sumN += dd;
        sumN2 += dd * dd;
    }
    T a = sumN / 2 - sqrt(sumN2) * s[0];
    al[I] = a;
    T fv = getVolumeFraction(g.D, n, a);
    fv = fv < ctol ? T(0) : (fv > 1 - ctol ? T(1) : fv);
    write_images<T>(g, f, p, fv, 0, 0, T(0));
}
// reconstructInterface! materialised (stage entry point; BCVOF! on periodic sides)
template <class T>
__global__ void __launch_bounds__(NT) k_reconstruct(Grid g, Tiling t, const T *f, T *al, T *nh, int scheme) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    T n[3] = {0, 0, 0}, a = 0;
    if (!fullorempty(f[I])) {
        normal_scheme(scheme, g, f, I, n);
        a = getIntercept(g.D, n, f[I]);
    }
    // periodic images only (non-periodic ghosts of n̂/α are zero)
    int alt[3][2], na[3];
    for (int ax = 0; ax < 3; ++ax) {
        na[ax] = 1;
        alt[ax][0] = p[ax];
        if (ax < g.D && g.per[ax]) {
            if (p[ax] == 1) { alt[ax][1] = g.Ng[ax] - 1; na[ax] = 2; }
            else if (p[ax] == g.Ng[ax] - 2) { alt[ax][1] = 0; na[ax] = 2; }
        }
    }
    for (int i2 = 0; i2 < na[2]; ++i2)
        for (int i1 = 0; i1 < na[1]; ++i1)
            for (int i0 = 0; i0 < na[0]; ++i0) {
                long J = (long)alt[0][i0] + g.st[1] * alt[1][i1] + g.st[2] * alt[2][i2];
                al[J] = a;
                for (int d = 0; d < g.D; ++d) nh[g.ns * d + J] = n[d];
            }
}

// ---------------------------------------------------------------------------
// level-set reinitialisation (redistaning.jl)
// ---------------------------------------------------------------------------
// LevelSet(sim) (redistaning.jl:14-25): ϕ = 2f - 1 on every entry, ghosts
// included, and ϕini = ϕ
template <class T> __global__ void __launch_bounds__(NT) k_ls_init(long ns, const T *f, T *phi, T *ini) {
    long q = (long)blockIdx.x * NT + threadIdx.x;
    if (q >= ns) return;
    T v = 2 * f[q] - 1;
    phi[q] = v;
    ini[q] = v;
}
// redistaning.jl:110 minmod
template <class T> __device__ inline T ls_minmod(T a, T b) { return fabs(a) <= fabs(b) ? a : b; }
// redistaning.jl:122-143 𝛁ϕᵢ²: second-order ENO (minmod-limited) one-sided
// derivatives of ϕ[I-2..I+2], the upwind one for the sign s squared, else 0
template <class T> __device__ inline T ls_grad2(T a, T b, T c, T d, T e, T s) {
    T dp = d - c, dm = c - b;
    T d2p = (e + c) - 2 * d, d2o = (d + b) - 2 * c, d2m = (c + a) - 2 * b;
    T dR = dp - ls_minmod(d2p, d2o) / 2;
    T dL = dm + ls_minmod(d2o, d2m) / 2;
    T wR = dR * s, wL = dL * s;
    if (wR < 0 && (wR + wL) < 0) return dR * dR;
    if (wL > 0 && (wR + wL) > 0) return dL * dL;
    return T(0);
}
// One stage of redistaning! (redistaning.jl:28-31, :67-108, BCf! of
// VOFutil.jl:64-75):  L = ϕini (1 - |∇ϕ|) with |∇ϕ|² summed axis by axis
// (the first and last interior cells of an axis take the mirrored (Neumann)
// or wrapped (periodic) point two cells out), then
// out = α ϕ⁰ + (1-α)(ϕ + dτ L), written with its ghost images.  ϕ and out are
// different buffers; ϕ⁰ is read at I only and may be `out`.
template <int D, class T>
__global__ void __launch_bounds__(NT) k_ls_stage(Grid g, Tiling t, const T *phi, const T *phi0, const T *ini, T *out,
                                                 T dtau, T alpha) {
    int p[3];
    if (!thread_cell(g, t, p)) return;
    long I = lin(g, p);
    T si = ini[I];
    T s = si > 0 ? T(1) : (si < 0 ? T(-1) : si);
    T c = phi[I];
    T acc = 0;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        long st = g.st[i], w = (long)(g.Ng[i] - 4) * st;
        int q = p[i];
        T b = phi[I - st], d = phi[I + st];
        T a = q == 1 ? (g.per[i] ? phi[I + w] : b) : phi[I - 2 * st];
        T e = q == g.Ng[i] - 2 ? (g.per[i] ? phi[I - w] : d) : phi[I + 2 * st];
        acc = acc + ls_grad2(a, b, c, d, e, s);
    }
    T L = si * (T(1) - sqrt(acc));
    T v = alpha * phi0[I] + (T(1) - alpha) * (c + dtau * L);
    write_images<T>(g, out, p, v, 0, 0, T(0));
}

}  // namespace ia
