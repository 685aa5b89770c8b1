// DM fitting on the GPU (gpu_fit_*): the CG solve after tomography,
//
//   (sum_f wt_f HA_f' W HA_f + NW NW' + S + tikdiag I) a = sum_f wt_f HA_f' W HX_f x,
//   W = W0 - W1 W1',
//
// replacing curecon_t::fit with cufit_grid (cuda/recon.cu:277-288,
// cuda/fit.cu:47-230, cuda/recon_base.cu:75-139) and the CPU FitR / FitL
// (maos/recon_utils.c:483-560) with fit.precond=0 (plain CG, lib/pcg.c:28-113
// with Mmul = NULL).
//
// Design.  A fit is small (the 30 m system with two DMs: 8.5k actuators,
// 4k fitting-grid points per direction) and its CG is a chain of dependent
// passes.  Each pass is one launch over the whole GPU, with work items
// (point, direction, system) or (actuator, direction, system), so that a
// thread does one short chain of dependent loads per pass, and a batch of
// systems shares every launch.  An iteration is two launches with the assembled
// operator (local boxes plus low rank, below) and five without it (HA, W, HA' +
// low-rank terms, x/r update, p update).  Scalars (alpha, beta, the W1 and NW
// projections) are fixed-order sums of per-workgroup partials, summed again
// by every workgroup that needs them, so no launch waits on the host and a
// system's bits do not depend on its batch neighbours.  (Running the whole
// solve of a system inside one 1024-thread workgroup, with workgroup
// barriers between the passes, was 20x slower for one system: every thread
// then walks ~35 dependent load chains per pass.)  Every operator is a
// gather:
//   HX_f, HA_f  bilinear interpolation of the layers / DM grids at the
//               fitting-grid points along direction f, from per-axis tap
//               tables (the grids are square and axis-aligned, so a 2-D tap
//               is the product of an x and a y tap, as mkh builds it);
//   W           9-point W0 stencil per point (rows of the reference's sparse
//               W0) minus the W1 piston projection, per direction;
//   HA_f'       per actuator, the fitting-grid columns and rows whose taps
//               land on it (transposed per-axis lists), no atomics;
//   NW, S       low-rank dots (block reductions) and a CSR row gather.
// Arithmetic is FP64 throughout: the fitting matrix carries a Tikhonov term
// of 4e-7/nact relative to its largest eigenvalue, too ill-conditioned for
// FP32 vectors at 1e-4 parity, and the solve is latency-bound, not
// FLOP-bound.  Reductions are fixed-order (a system's bits do not depend on
// its batch neighbours).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "fit_internal.hpp"
#include "maos_tomo.h"

namespace mt {
void set_error(const std::string &msg);
}

namespace {

struct FitErr {
    int code;
    std::string msg;
};
#define FCHK(call)                                                                          \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) throw FitErr{MT_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)}; \
    } while (0)
[[noreturn]] void ffail(int code, const std::string &m) { throw FitErr{code, m}; }

template <typename T>
struct DBuf {
    T *p = nullptr;
    size_t n = 0;
    void alloc(size_t count) {
        free();
        n = count;
        if (count) FCHK(hipMalloc((void **)&p, sizeof(T) * count));
    }
    void upload(const std::vector<T> &h) {
        alloc(h.size());
        if (n) FCHK(hipMemcpy(p, h.data(), sizeof(T) * n, hipMemcpyHostToDevice));
    }
    void free() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    ~DBuf() { free(); }
};

constexpr int FMAXDM = 8, FMAXFIT = 32, FMAXL = 16, FMAXNW = 32;
constexpr double FEPS = 1e-15;  // tap weights not above this are dropped (lib/mkh.c:109, sys/common.h:88)

// One axis tap pair of a forward interpolation: nodes n and n+1 with
// weights w0, w1 (0 where the node is off the grid).
struct Tap2 {
    int n;
    int pad_;
    double w0, w1;
};
// One entry of a transposed axis list: output-grid index and weight.
struct TapT {
    int i;
    int pad_;
    double w;
};

// A tile of FTX x FTY actuators of one DM, the rows of one wave of kf_mv (lane
// = column + FTX * row), with all that the wave needs to know of it (one
// scalar round trip).
constexpr int FTX = 16, FTY = 4;
struct FTile {
    long coef;            // first coefficient
    int d, ia0, ja0;      // DM and first actuator
    int a0, anx;          // the first actuator's index, the DM's row length
    int nx, ny;           // actuators of the tile that exist
    int eo, cls[5];       // the row's entries: window offsets in FMv::eo, bounds of the four sums
    int wn, lst;          // window: nodes, their actuators in FMv::list
    int pitch, own;       // the window's row length, the first actuator's own node
    int pad_;
};
constexpr int FNC = 20;           // coefficients of a row that a wave keeps in registers
constexpr int FSW = 16;           // most systems per workgroup of kf_mv
constexpr int FVT = 512;          // threads of kf_vec
constexpr int FCH = 2 * FVT;      // actuators per workgroup of kf_vec
// What kf_mv and kf_vec read of a plan, by value (kernel arguments arrive
// before the first instruction; a record in memory is a round trip away).
struct FMv {
    const FTile *tile;
    const int *list, *eo;
    const double *coef;       // [tile][entry][64 rows]
    const double *lr, *lrc;
    double *r, *p, *p2, *Ap, *b, *part, *res;
    int *stop;
    long na, pstride;
    int nlr, nch, ntile;
    int o2, o3, o4, o5, o6;
};

// Everything the kernel reads of one plan (device resident, read through
// scalar loads as kernel arguments are).
struct FitDev {
    int nfit, ndm, npsr, nnw;
    int fnx, fny;
    long nfloc, nact, nxtot;
    int anx[FMAXDM], any[FMAXDM];
    long aoff[FMAXDM + 1];
    int xnx[FMAXL], xny[FMAXL];
    long xoff[FMAXL + 1];
    double wt[FMAXFIT];
    // forward taps: HA (f, dm) and HX (f, layer), per fitting-grid column / row
    const Tap2 *hax, *hay;  // [(f*ndm + d)*fnx + px], [(f*ndm + d)*fny + py]
    const Tap2 *hxx, *hxy;  // [(f*npsr + l)*fnx + px], ...
    // transposed HA lists: per (f, d) and actuator column ia (row ja) the
    // entries [tp[b + ia], tp[b + ia + 1]) of te, b = f tpx + tdx[d] (the
    // pointer arrays of the (f, d) pairs in order, anx[d] + 1 entries each)
    int tpx, tpy, tdx[FMAXDM], tdy[FMAXDM];
    const int *txp, *typ;
    const TapT *txe, *tye;
    const double *W0, *W1;  // 9 per point (row form), per point
    const long *slp, *sli;  // S in CSR (slp null: none)
    const double *slx;
    double tikdiag;
    // low-rank columns lr [nlr][nact] with coefficients lrc: NW (coefficient
    // 1) and, with the assembled operator, HA_f' W1 (coefficient -wt_f)
    int nlr;
    const double *lr;
    double lrc[FMAXNW + FMAXFIT];
    // assembled operator (asm_ok), see kf_mv: row (ia, ja) of DM d1 reaches in
    // DM d2 (pair d1 * FMAXDM + d2) the kx x ky actuators from (ia + bx, ja + by)
    // on; its etot[d1] entries over all DMs at epos[ebase[d1]]: column | row <<
    // 12 | DM << 24
    const int *epos;
    int ebase[FMAXDM];
    int asm_ok, ntile, etot[FMAXDM];
    int kx[FMAXDM * FMAXDM], ky[FMAXDM * FMAXDM], bx[FMAXDM * FMAXDM], by[FMAXDM * FMAXDM];
    const struct FTile *tile;
    // launch shape: point chunks of 256 per direction (nc1), actuator chunks
    // of hab actuators x nfit directions (nc3), actuator chunks of 256 (nc4)
    int nc1, nc3, nc4, hab;
    int nch;  // vector chunks whose partials are kept: of FCH actuators (assembled), else nc4
    // per-system partials, pstride doubles each: W1 . opd_f [nfit][nc1] at
    // o1, p . Ap [ntile or nc3] at o2, the low-rank projections [nlr][nch] at
    // o3, r . r in two slots [2][nch] at o4 (iteration parity), b . b [nch]
    // at o5, the projections of p in two slots [2][nlr] at o6 (assembled)
    int o1, o2, o3, o4, o5, o6;
    long pstride;
    // per-system workspace
    double *opd, *opd2;     // [s][nfit][nfloc]
    double *tnw;            // [s][FMAXNW]: NW' p of the current p
    double *r, *p, *Ap, *b; // [s][nact]
    double *part;           // [s][pstride]
    int *stop;              // [s]: 1 once a step size was not finite
    double *res;            // [s]
};

constexpr int FB = 256;  // threads per workgroup of every fit kernel

// Sum of v over the 256 threads of a workgroup in a fixed order (lane tree,
// then the four waves in order); the result is valid in thread 0.  Every
// thread of the workgroup must call it.
__device__ double fit_bred(double v, double *wsum) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0) s = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
    return s;
}

// Sum of the n partials at q in a fixed order (thread-strided sums, then the
// lane tree and the four waves in order), returned to every thread.  Every
// thread of the workgroup must call it; psh is its own LDS (not fit_bred's).
__device__ double psum(const double *q, int n, double *psh) {
    double v = 0;
    for (int i = threadIdx.x; i < n; i += FB) v += q[i];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    __syncthreads();  // the previous call's readers are done with psh
    if ((threadIdx.x & 63) == 0) psh[threadIdx.x >> 6] = v;
    __syncthreads();
    return ((psh[0] + psh[1]) + psh[2]) + psh[3];
}

__device__ __forceinline__ double *fpart(const FitDev &D, int s) { return D.part + (long)s * D.pstride; }

// opd_f = sum over sources (DMs or layers) of the bilinear interpolation at
// the fitting-grid point, and the workgroup's partial of W1 . opd_f.
// Grid (point chunks, directions, systems).  SRC 0: actuator vectors
// (double), 1: layer vectors (float).  Sources are taken GS at a time with
// clamped indexes so that the tap loads of a group issue together.
template <int SRC, int GS>
__global__ __launch_bounds__(FB) void kf_fwd(const FitDev *__restrict__ Dp, const void *__restrict__ srcv,
                                              long sstride, int ws0) {
    const FitDev &D = *Dp;
    __shared__ double wsum[4];
    const int f = blockIdx.y, s = ws0 + blockIdx.z;
    const long nf = D.nfloc;
    const long pt = (long)blockIdx.x * FB + threadIdx.x;
    const bool on = pt < nf;
    const long ptc = on ? pt : nf - 1;
    // 32-bit index arithmetic (a 64-bit division is a long instruction
    // sequence; every grid here is far below 2^31 points)
    const int py = (int)ptc / D.fnx, px = (int)ptc - py * D.fnx;
    const int nsrc = SRC ? D.npsr : D.ndm;
    const Tap2 *tx = SRC ? D.hxx : D.hax, *ty = SRC ? D.hxy : D.hay;
    const int *snx = SRC ? D.xnx : D.anx;
    const long *soff = SRC ? D.xoff : D.aoff;
    double acc = 0;
    for (int d0 = 0; d0 < nsrc; d0 += GS) {
        Tap2 a[GS], b[GS];
#pragma unroll
        for (int j = 0; j < GS; j++) {
            const int d = min(d0 + j, nsrc - 1);
            a[j] = tx[((long)f * nsrc + d) * D.fnx + px];
            b[j] = ty[((long)f * nsrc + d) * D.fny + py];
        }
        double v[GS][4];
#pragma unroll
        for (int j = 0; j < GS; j++) {
            const int d = min(d0 + j, nsrc - 1);
            const long base = soff[d] + (long)blockIdx.z * sstride;
            const int nx = snx[d];
            const long i00 = base + (long)b[j].n * nx + a[j].n;
            // taps of zero weight point at node 0 or -1 of an axis; clamp the
            // address into the source so the load stays in bounds
            const long lo = base, hi = base + (long)snx[d] * (SRC ? D.xny[d] : D.any[d]) - 1;
            const long k[4] = {i00, i00 + 1, i00 + nx, i00 + nx + 1};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long kk = k[q] < lo ? lo : (k[q] > hi ? hi : k[q]);
                v[j][q] = SRC ? (double)((const float *)srcv)[kk] : ((const double *)srcv)[kk];
            }
        }
#pragma unroll
        for (int j = 0; j < GS; j++) {
            if (d0 + j >= nsrc) break;
            const double wx[2] = {a[j].w0, a[j].w1}, wy[2] = {b[j].w0, b[j].w1};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double w = wx[q & 1] * wy[q >> 1];
                if (w > FEPS) acc += w * v[j][q];
            }
        }
    }
    if (on) D.opd[((long)s * D.nfit + f) * nf + pt] = acc;
    const double pw = fit_bred(on ? D.W1[pt] * acc : 0.0, wsum);
    if (threadIdx.x == 0) fpart(D, s)[D.o1 + f * D.nc1 + blockIdx.x] = pw;
}

// opd2_f = wt_f (W0 opd_f - W1 (W1' opd_f)) (applyW, maos/recon_utils.c:155-180).
// With nwdots, the first workgroup of each system also sums the partials of
// NW' p once for the kf_hat that follows (instead of every kf_hat workgroup:
// those sums were a quarter of its time).
__global__ __launch_bounds__(FB) void kf_w(const FitDev *__restrict__ Dp, int ws0, int nwdots) {
    const FitDev &D = *Dp;
    __shared__ double psh[4];
    const int f = blockIdx.y, s = ws0 + blockIdx.z;
    const long nf = D.nfloc;
    const long i = (long)blockIdx.x * FB + threadIdx.x;
    if (nwdots && blockIdx.x == 0 && blockIdx.y == 0)
        for (int k = 0; k < D.nnw; k++) {
            const double v = psum(fpart(D, s) + D.o3 + k * D.nc4, D.nc4, psh);
            if (threadIdx.x == 0) D.tnw[(long)s * FMAXNW + k] = v;
        }
    const double dot = psum(fpart(D, s) + D.o1 + f * D.nc1, D.nc1, psh);
    if (i >= nf) return;
    const int fnx = D.fnx, fny = D.fny;
    const int iy = (int)i / fnx, ix = (int)i - iy * fnx;
    const double *o = D.opd + ((long)s * D.nfit + f) * nf;
    const double *w0 = D.W0 + 9 * i;
    double acc = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const int jx = ix + k % 3 - 1, jy = iy + k / 3 - 1;
        const double c = w0[k];
        if (c != 0.0 && jx >= 0 && jx < fnx && jy >= 0 && jy < fny) acc += c * o[(long)jy * fnx + jx];
    }
    D.opd2[((long)s * D.nfit + f) * nf + i] = D.wt[f] * (acc - D.W1[i] * dot);
}

enum { HAT_R = 0, HAT_L = 1 };
constexpr int HAH = 2;  // actuator groups per kf_hat workgroup (each thread gathers for HAH actuators)

// out[a] = sum_f HA_f' opd2_f at actuator a; HAT_L adds NW (NW' p) + S p +
// tikdiag p and writes the workgroup's partial of p . out.  A workgroup holds
// HAH groups of hab actuators x nfit directions, one thread per (actuator of
// each group, direction) (two actuators per thread halve the workgroups and
// their fixed reduction and barrier cost),
// gathering through the transposed per-axis lists (no atomics); the
// directions of an actuator are summed in index order.  Actuators are the
// fast index of the threads, so a wave's gathers of one direction read
// neighbouring fitting-grid points (with directions fastest, every lane read
// another direction's grid: one cache line per lane and load).  Grid
// (actuator chunks, systems); p and out are per-system vectors of stride nact.
template <int MODE>
__global__ __launch_bounds__(FB) void kf_hat(const FitDev *__restrict__ Dp, const double *__restrict__ p,
                                              double *__restrict__ out, int ws0) {
    const FitDev &D = *Dp;
    __shared__ double red[HAH * FB];
    __shared__ double tnw[FMAXNW];
    __shared__ double wsum[4];
    const int s = ws0 + blockIdx.y;
    const int nfit = D.nfit, t = threadIdx.x, hab = D.hab;
    const int f = t / hab, al = t - f * hab;
    const long na = D.nact, nf = D.nfloc;
    const long a0 = (long)blockIdx.x * HAH * hab;  // first actuator of the workgroup
    if (MODE == HAT_L && t < D.nnw) tnw[t] = D.tnw[(long)s * FMAXNW + t];
    const double *o = D.opd2 + ((long)s * nfit + f) * nf;
    const int fnx = D.fnx;
#pragma unroll
    for (int j = 0; j < HAH; j++) {
        const long a = a0 + j * hab + al;
        double acc = 0;
        if (f < nfit && a < na) {
            int d = 0;
            while (a >= D.aoff[d + 1]) d++;
            const int k = (int)(a - D.aoff[d]);
            const int ja = k / D.anx[d], ia = k - ja * D.anx[d];
            const int bx = f * D.tpx + D.tdx[d] + ia, by = f * D.tpy + D.tdy[d] + ja;
            const int x0 = D.txp[bx], x1 = D.txp[bx + 1];
            const int y0 = D.typ[by], y1 = D.typ[by + 1];
            for (int ey = y0; ey < y1; ey++) {
                const TapT ty = D.tye[ey];
                for (int ex = x0; ex < x1; ex++) {
                    const TapT tx = D.txe[ex];
                    const double w = tx.w * ty.w;
                    if (w > FEPS) acc += w * o[(long)ty.i * fnx + tx.i];
                }
            }
        }
        red[j * FB + t] = acc;
    }
    __syncthreads();
    double pap = 0;
    for (int e = t; e < HAH * hab; e += FB) {
        const int j = e / hab, el = e - j * hab;
        const long a = a0 + e;
        if (a >= na) break;
        double v = 0;
        for (int q = 0; q < nfit; q++) v += red[j * FB + q * hab + el];
        if (MODE == HAT_L) {
            const double *ps = p + (long)blockIdx.y * na;
            for (int q = 0; q < D.nnw; q++) v += D.lr[(long)q * na + a] * tnw[q];
            if (D.slp) {
                double sl = 0;
                for (long e2 = D.slp[a]; e2 < D.slp[a + 1]; e2++) sl += D.slx[e2] * ps[D.sli[e2]];
                v += sl;
            }
            v += D.tikdiag * ps[a];
            pap += ps[a] * v;
        }
        out[(long)blockIdx.y * na + a] = v;
    }
    if (MODE == HAT_L) {
        pap = fit_bred(pap, wsum);
        if (t == 0) fpart(D, s)[D.o2 + blockIdx.x] = pap;
    }
}

// Partials of NW' v (into o3) for a per-system actuator vector v; with
// INIT also zeroes v first when the start is cold, writes the partials of
// b . b (o5) and clears the system's stop flag.  Grid (actuator chunks of
// 256, systems).
template <bool INIT>
__global__ __launch_bounds__(FB) void kf_init(const FitDev *__restrict__ Dp, double *__restrict__ v, int ws0,
                                               int warm) {
    const FitDev &D = *Dp;
    __shared__ double wsum[4];
    const int s = ws0 + blockIdx.y;
    const long na = D.nact;
    const long a = (long)blockIdx.x * FB + threadIdx.x;
    const bool on = a < na;
    double *vs = v + (long)blockIdx.y * na;
    double val = 0;
    if (on) {
        if (INIT && !warm) vs[a] = 0;
        else val = vs[a];
    }
    double *q = fpart(D, s);
    for (int k = 0; k < D.nlr; k++) {
        const double c = on ? D.lr[(long)k * na + a] * val : 0.0;
        const double t = fit_bred(c, wsum);
        if (threadIdx.x == 0) q[D.o3 + k * D.nc4 + blockIdx.x] = t;
        __syncthreads();
    }
    if (INIT) {
        const double bv = on ? D.b[(long)s * na + a] : 0.0;
        const double t = fit_bred(bv * bv, wsum);
        if (threadIdx.x == 0) {
            q[D.o5 + blockIdx.x] = t;
            if (blockIdx.x == 0) D.stop[s] = 0;
        }
    }
}

// CG (re)start at iteration k: r = b - Ap (COLD: r = b, x being zero),
// p = r; partials of r . r into slot k & 1 and of NW' p.
template <bool COLD>
__global__ __launch_bounds__(FB) void kf_restart(const FitDev *__restrict__ Dp, int ws0, int k) {
    const FitDev &D = *Dp;
    __shared__ double wsum[4];
    const int s = ws0 + blockIdx.y;
    const long na = D.nact;
    const long a = (long)blockIdx.x * FB + threadIdx.x;
    const bool on = a < na;
    double v = 0;
    if (on) {
        const long i = (long)s * na + a;
        v = COLD ? D.b[i] : D.b[i] - D.Ap[i];
        D.r[i] = v;
        D.p[i] = v;
    }
    double *q = fpart(D, s);
    const double t = fit_bred(v * v, wsum);
    if (threadIdx.x == 0) q[D.o4 + (k & 1) * D.nc4 + blockIdx.x] = t;
    for (int j = 0; j < D.nlr; j++) {
        __syncthreads();
        const double c = on ? D.lr[(long)j * na + a] * v : 0.0;
        const double u = fit_bred(c, wsum);
        if (threadIdx.x == 0) q[D.o3 + j * D.nc4 + blockIdx.x] = u;
    }
}

// Iteration k, first half: alpha = rr_k / p.Ap; x += alpha p; r -= alpha Ap;
// partials of r . r into slot (k + 1) & 1.  A non-finite alpha stops the
// system (x keeps its value, the residual is NaN).
__global__ __launch_bounds__(FB) void kf_upd(const FitDev *__restrict__ Dp, double *__restrict__ x, int ws0,
                                             int k) {
    const FitDev &D = *Dp;
    __shared__ double wsum[4], psh[4];
    const int s = ws0 + blockIdx.y;
    if (D.stop[s]) return;
    const double *q = fpart(D, s);
    const double rr = psum(q + D.o4 + (k & 1) * D.nc4, D.nc4, psh);
    const double pap = psum(q + D.o2, D.nc3, psh);
    const double ak = rr / pap;
    if (!isfinite(ak)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            D.stop[s] = 1;
            D.res[s] = NAN;
        }
        return;
    }
    const long na = D.nact;
    const long a = (long)blockIdx.x * FB + threadIdx.x;
    double v = 0;
    if (a < na) {
        const long i = (long)s * na + a;
        x[(long)blockIdx.y * na + a] += ak * D.p[i];
        v = D.r[i] - ak * D.Ap[i];
        D.r[i] = v;
    }
    const double t = fit_bred(v * v, wsum);
    if (threadIdx.x == 0) fpart(D, s)[D.o4 + ((k + 1) & 1) * D.nc4 + blockIdx.x] = t;
}

// Iteration k, second half: beta = rr_(k+1) / rr_k; p = beta p + r and the
// partials of NW' p; after the last iteration the residual sqrt(rr / b.b).
__global__ __launch_bounds__(FB) void kf_p(const FitDev *__restrict__ Dp, int ws0, int k, int last) {
    const FitDev &D = *Dp;
    __shared__ double wsum[4], psh[4];
    const int s = ws0 + blockIdx.y;
    if (D.stop[s]) return;
    const double *qs = fpart(D, s);
    const double rr2 = psum(qs + D.o4 + ((k + 1) & 1) * D.nc4, D.nc4, psh);
    if (last) {
        if (blockIdx.x == 0) {
            const double bb = psum(qs + D.o5, D.nc4, psh);
            if (threadIdx.x == 0) D.res[s] = sqrt(rr2 / bb);
        }
        return;
    }
    const double rr = psum(qs + D.o4 + (k & 1) * D.nc4, D.nc4, psh);
    const double bk = rr2 / rr;
    const long na = D.nact;
    const long a = (long)blockIdx.x * FB + threadIdx.x;
    const bool on = a < na;
    double v = 0;
    if (on) {
        const long i = (long)s * na + a;
        v = bk * D.p[i] + D.r[i];
        D.p[i] = v;
    }
    double *q = fpart(D, s);
    for (int j = 0; j < D.nnw; j++) {
        const double c = on ? D.lr[(long)j * na + a] * v : 0.0;
        const double u = fit_bred(c, wsum);
        if (threadIdx.x == 0) q[D.o3 + j * D.nc4 + blockIdx.x] = u;
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Assembled operator.  HA, W0, S and the Tikhonov term act within a few
// actuators, so a row of
//   A = sum_f wt_f HA_f' W0 HA_f + S + tikdiag I
// is a box of kx x ky actuators of each DM around the row's own position (30 m
// system: 5 x 5 on its own DM, 7 x 7 on the other), and the rest of FitL is
// low rank: NW NW' - sum_f wt_f v_f v_f', v_f = HA_f' W1.  The plan holds the
// box coefficients and the columns NW, v_f, built once on the GPU in FP64.
// Applying them is one pass with fewer operations than the matrix-free one
// (about 75 against 106 multiply-adds per actuator) and no fitting-grid arrays
// in between, and the projections v_f . p follow p's own recurrence, so a CG
// iteration is two launches (kf_mv, kf_vec) instead of five: for one system
// of the 30 m fit 12 us of kernels instead of 32 (6 + 6), for 64 systems 43
// instead of 161 (29 + 14).
// ---------------------------------------------------------------------------

// hi + lo += a b in twice the precision (two-sum, and a two-product by fused
// multiply-add).  The set-up kernels sum their terms so: a coefficient is then
// right to its last place and not a unit or two off, an error that every
// iteration would repeat.  Against 80 bits, 10 iterations of 48 fits of the 30 m
// system: 3.0e-15 in matrix-free passes, 3.3e-15 assembled with plain sums,
// 2.8e-15 with these; kf_assemble 425 -> 440 us, once a plan.
__device__ __forceinline__ void dd_fma(double &hi, double &lo, double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b, e = fma(a, b, -p);
    const double t = hi + p, z = t - hi;
    lo += ((hi - (t - z)) + (p - z)) + e;
    hi = t;
}

// Coefficients of the boxes, one thread per (actuator, entry).  Grid (tiles,
// groups of 4 entries), 256 threads: 4 entries x the 64 actuators of the tile.
__global__ __launch_bounds__(FB) void kf_assemble(const FitDev *__restrict__ Dp, double *__restrict__ coef) {
    const FitDev &D = *Dp;
    const FTile &T = D.tile[blockIdx.x];
    const int lane = threadIdx.x & 63, d1 = T.d, nd = D.ndm;
    int e = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (e >= D.etot[d1]) return;
    const int ps = D.epos[D.ebase[d1] + e], d2 = ps >> 24;
    const int pr = d1 * FMAXDM + d2;
    const int ia = T.ia0 + (lane & (FTX - 1)), ja = T.ja0 + lane / FTX;
    const int jx = ia + D.bx[pr] + (ps & 0xfff), jy = ja + D.by[pr] + (ps >> 12 & 0xfff);
    double v = 0, vl = 0;
    if (ia < D.anx[d1] && ja < D.any[d1] && jx >= 0 && jx < D.anx[d2] && jy >= 0 && jy < D.any[d2]) {
        const int fnx = D.fnx, fny = D.fny;
        for (int f = 0; f < D.nfit; f++) {
            const int px = f * D.tpx + D.tdx[d1] + ia, py = f * D.tpy + D.tdy[d1] + ja;
            const Tap2 *hx = D.hax + (long)(f * nd + d2) * fnx, *hy = D.hay + (long)(f * nd + d2) * fny;
            double vf = 0, vfl = 0;
            for (int ey = D.typ[py]; ey < D.typ[py + 1]; ey++)
                for (int ex = D.txp[px]; ex < D.txp[px + 1]; ex++) {
                    const TapT ty = D.tye[ey], tx = D.txe[ex];
                    const double w1 = tx.w * ty.w;
                    if (!(w1 > FEPS)) continue;
                    const double *w0 = D.W0 + 9 * ((long)ty.i * fnx + tx.i);
                    double u = 0, ul = 0;
                    for (int k = 0; k < 9; k++) {
                        const int qx = tx.i + k % 3 - 1, qy = ty.i + k / 3 - 1;
                        if (w0[k] == 0.0 || qx < 0 || qx >= fnx || qy < 0 || qy >= fny) continue;
                        const Tap2 a = hx[qx], b = hy[qy];
                        const double wx = a.n == jx ? a.w0 : a.n + 1 == jx ? a.w1 : 0.0;
                        const double wy = b.n == jy ? b.w0 : b.n + 1 == jy ? b.w1 : 0.0;
                        const double w2 = wx * wy;
                        if (w2 > FEPS) dd_fma(u, ul, w0[k], w2);
                    }
                    dd_fma(vf, vfl, w1, u);
                    vfl += w1 * ul;
                }
            dd_fma(v, vl, D.wt[f], vf);
            vl += D.wt[f] * vfl;
        }
        const long a1 = D.aoff[d1] + (long)ja * D.anx[d1] + ia, a2 = D.aoff[d2] + (long)jy * D.anx[d2] + jx;
        if (D.slp)
            for (long q = D.slp[a1]; q < D.slp[a1 + 1]; q++)
                if (D.sli[q] == a2) dd_fma(v, vl, D.slx[q], 1.0);
        if (a1 == a2) dd_fma(v, vl, D.tikdiag, 1.0);
    }
    coef[T.coef + (long)e * 64 + lane] = v + vl;
}

// v_f = HA_f' W1.  Grid (actuator chunks, directions).
__global__ __launch_bounds__(FB) void kf_lowrank(const FitDev *__restrict__ Dp, double *__restrict__ out) {
    const FitDev &D = *Dp;
    const long a = (long)blockIdx.x * FB + threadIdx.x;
    const int f = blockIdx.y;
    if (a >= D.nact) return;
    int d = 0;
    while (a >= D.aoff[d + 1]) d++;
    const int k = (int)(a - D.aoff[d]);
    const int ja = k / D.anx[d], ia = k - ja * D.anx[d];
    const int px = f * D.tpx + D.tdx[d] + ia, py = f * D.tpy + D.tdy[d] + ja;
    double v = 0, vl = 0;
    for (int ey = D.typ[py]; ey < D.typ[py + 1]; ey++)
        for (int ex = D.txp[px]; ex < D.txp[px + 1]; ex++) {
            const double w = D.txe[ex].w * D.tye[ey].w;
            if (w > FEPS) dd_fma(v, vl, w, D.W1[(long)D.tye[ey].i * D.fnx + D.txe[ex].i]);
        }
    out[(long)f * D.nact + a] = v + vl;
}

// Reduces sixteen values per lane over a wave and scatters the sums: lane l
// ends with value l >> 2, in 17 exchanges instead of 6 per value.
template <int H, int X>
__device__ __forceinline__ void red_half(double *u, int lane) {
    const bool up = (lane & X) != 0;
#pragma unroll
    for (int j = 0; j < H; j++) {
        const double lo = u[j], hi = u[j + H];  // by value: a choice between elements would index memory
        u[j] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, X, 64);
    }
}
__device__ __forceinline__ double wave_red16(double (&u)[16]) {
    const int lane = threadIdx.x & 63;
    red_half<8, 32>(u, lane);
    red_half<4, 16>(u, lane);
    red_half<2, 8>(u, lane);
    red_half<1, 4>(u, lane);
    double v = u[0];
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 1, 64);
    return v;
}

// out = FitL v.  MV_CG (iteration k): v is the new direction p = r + beta
// p_old, formed here for the whole window a workgroup reads (each neighbour
// needs it, so no pass of its own) and stored for the tile's own actuators;
// its low-rank projections are t = t(r) + beta t_old; partials of p . out per
// tile.  MV_PLAIN: v is given, its projections are the partials at o3.
enum { MV_PLAIN = 0, MV_CG = 1 };

// Projections tl[s][j] and beta of S systems from their partials, four lanes
// per sum, in a fixed order (all threads of the workgroup; no barrier).
template <int MODE>
__device__ __forceinline__ void mv_scalars(const FMv &M, int s0, int ns, int k, double (*tl)[FMAXNW + FMAXFIT],
                                           double *bet) {
    const int nlr = M.nlr, nch = M.nch, nj = nlr + (MODE == MV_CG ? 1 : 0), sub = threadIdx.x & 3;
#pragma unroll 2
    for (int w = threadIdx.x >> 2; w < ns * nj; w += FB / 4) {
        const int s = w / nj, j = w - s * nj;
        const double *q = M.part + (long)(s0 + s) * M.pstride;
        const double *a = j == nlr ? q + M.o4 + (k & 1) * nch : q + M.o3 + j * nch;
        const double *a2 = q + M.o4 + ((k + 1) & 1) * nch;
        double u = 0, u2 = 0;
        for (int i = sub; i < nch; i += 12) {  // three loads each in flight
            double b[3], b2[3];
#pragma unroll
            for (int h = 0; h < 3; h++) {
                b[h] = a[min(i + 4 * h, nch - 1)];
                b2[h] = a2[min(i + 4 * h, nch - 1)];
            }
#pragma unroll
            for (int h = 0; h < 3; h++) {
                u += i + 4 * h < nch ? b[h] : 0.0;
                u2 += i + 4 * h < nch ? b2[h] : 0.0;
            }
        }
        u += __shfl_xor(u, 2, 64);
        u2 += __shfl_xor(u2, 2, 64);
        u += __shfl_xor(u, 1, 64);
        u2 += __shfl_xor(u2, 1, 64);
        if (sub == 0) {
            if (j == nlr) bet[s] = u / u2;
            else tl[s][j] = u;
        }
    }
}
// The projections of the new direction (times their coefficients in tl);
// the first workgroup keeps them for the next iteration.
template <int MODE>
__device__ __forceinline__ void mv_project(const FMv &M, int s0, int ns, int k, bool old, bool keep,
                                           double (*tl)[FMAXNW + FMAXFIT], const double *bet) {
    const int nlr = M.nlr;
    for (int w = threadIdx.x; w < ns * 64; w += FB) {
        const int s = w >> 6, j = w & 63;
        if (j >= nlr) continue;
        double u = tl[s][j];
        if (MODE == MV_CG) {
            double *q = M.part + (long)(s0 + s) * M.pstride + M.o6;
            if (old) u += bet[s] * q[((k + 1) & 1) * nlr + j];
            if (keep) q[(k & 1) * nlr + j] = u;
        }
        tl[s][j] = u * M.lrc[j];
    }
}

// A workgroup holds a tile of 64 rows, one per lane, for up to FSW systems in
// turn; its four waves share a row's entries and low-rank columns.  What does
// not depend on the system stays in registers: a wave's quarter of the
// coefficients (FNC of them; wider boxes read the rest again) and of the
// low-rank columns at its rows.  Per system, the window of p (all DMs) goes
// to LDS, loaded a system ahead, and a box is a sum over entries of a
// coefficient times the window node at an offset common to the lanes.
// One system alone (157 workgroups for the 30 m fit) waits for the chain
// arguments -> tile -> window -> boxes, so whatever does not depend on beta is
// loaded ahead of it; many systems are bound by the LDS reads, one per
// multiply-add, and the window loads.  Grid (tiles, padded to a multiple of 8;
// groups of spw systems); each XCD gets a contiguous run of tiles and finds
// their coefficients in its own L2.
template <int MODE>
__global__ __launch_bounds__(FB, 5) void kf_mv(const FMv M, const double *__restrict__ v, double *__restrict__ out,
                                             int ws0, int n, int spw, int k, int first) {
    constexpr int NP = 2;  // window nodes per thread that are loaded ahead
    constexpr int NLR = 4;  // low-rank columns of a wave that stay in registers
    extern __shared__ double win[];  // [2][wn]
    __shared__ double red[2][4][64];
    __shared__ double tl[FSW][FMAXNW + FMAXFIT], bet[FSW];
    const int run = gridDim.x >> 3;
    const int ti = (blockIdx.x & 7) * run + (blockIdx.x >> 3);
    if (ti >= M.ntile) return;
    const int g0 = blockIdx.y * spw, ns = min(spw, n - g0);
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const FTile &T = M.tile[ti];
    const int wn = T.wn, nlr = M.nlr;
    const int *lst = M.list + T.lst;
    const long na = M.na;
    double *pn = (k & 1) ? M.p2 : M.p;
    const double *po = (k & 1) ? M.p : M.p2;
    const double *src = MODE == MV_PLAIN ? v : M.r;
    const bool old = MODE == MV_CG && !first;
    const long sb = (long)((MODE == MV_CG ? ws0 : 0) + g0) * na;
    int wa[NP];
    double wu[NP], wp[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        wa[i] = lst[min(t + i * FB, wn - 1)];
        wu[i] = src[sb + wa[i]];
        wp[i] = old ? po[sb + wa[i]] : 0.0;
    }
    const int c0 = T.cls[wv], nc = T.cls[wv + 1] - c0;
    const double *cf = M.coef + T.coef + (long)c0 * 64 + lane;
    const int *eo = M.eo + T.eo + c0;
    const int eol = eo[min(lane, max(nc - 1, 0))];  // window offsets of the first entries, one per lane
    double c[FNC];
#pragma unroll
    for (int e = 0; e < FNC; e++) {
        const double ce = cf[e * 64];
        c[e] = e < nc ? ce : 0.0;
    }
    const int ix = lane & (FTX - 1), iy = lane / FTX;
    const bool on = ix < T.nx && iy < T.ny;
    const long a = T.a0 + (long)min(iy, T.ny - 1) * T.anx + min(ix, T.nx - 1);
    const double *lrp = M.lr + a;
    double cl[NLR];
#pragma unroll
    for (int j = 0; j < NLR; j++) cl[j] = lrp[(long)min(wv + 4 * j, nlr - 1) * na];
    mv_scalars<MODE>(M, ws0 + g0, ns, k, tl, bet);
    __syncthreads();
    mv_project<MODE>(M, ws0 + g0, ns, k, old, ti == 0, tl, bet);
    const int nd0 = iy * T.pitch + ix, own = T.own + nd0;
    for (int s = 0; s < ns; s++) {
        const long so = sb + (long)s * na;
        double *wb = win + (s & 1) * wn;
        const double be = MODE == MV_CG ? bet[s] : 0.0;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (t + i * FB < wn) wb[t + i * FB] = old ? be * wp[i] + wu[i] : wu[i];
        for (int w = t + NP * FB; w < wn; w += FB) {
            const int b = lst[w];
            const double u = src[so + b];
            wb[w] = old ? be * po[so + b] + u : u;
        }
        if (s + 1 < ns)
#pragma unroll
            for (int i = 0; i < NP; i++) {  // the next system's window
                wu[i] = src[so + na + wa[i]];
                wp[i] = old ? po[so + na + wa[i]] : 0.0;
            }
        __syncthreads();
        const double *wr = wb + nd0;
        double acc = 0;
#pragma unroll
        for (int e = 0; e < FNC; e++) acc += c[e] * wr[__builtin_amdgcn_readlane(eol, e)];
        for (int e = FNC; e < nc; e++) acc += cf[(long)e * 64] * wr[eo[e]];
#pragma unroll
        for (int j = 0; j < NLR; j++)
            if (wv + 4 * j < nlr) acc += cl[j] * tl[s][wv + 4 * j];
        for (int j = wv + 4 * NLR; j < nlr; j += 4) acc += lrp[(long)j * na] * tl[s][j];
        red[s & 1][wv][lane] = acc;
        __syncthreads();
        if (wv != (s & 3)) continue;
        // the waves finish systems in turn
        const double(*q)[64] = red[s & 1];
        const double y = ((q[0][lane] + q[1][lane]) + q[2][lane]) + q[3][lane];
        if (on) out[so + a] = y;
        if (MODE == MV_CG) {
            const double pv = wb[own];
            if (on) pn[so + a] = pv;
            double pap = on ? pv * y : 0.0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) pap += __shfl_down(pap, o, 64);
            if (lane == 0) M.part[(long)(ws0 + g0 + s) * M.pstride + M.o2 + ti] = pap;
        }
    }
}

// Vector passes of the assembled solve, FCH actuators per workgroup (few
// partials, since every kf_mv workgroup sums them again), two per thread:
//   VEC_STEP   iteration k, second half: alpha = rr_k / p.Ap; x += alpha p;
//              r -= alpha Ap; partials of r . r into slot (k + 1) & 1 and of
//              the projections of r.  A non-finite alpha stops the system (x
//              keeps its value, the residual is NaN);
//   VEC_COLD   cold start: x = 0, r = b, stop = 0, partials of b . b, of r . r
//              (slot 0) and of the projections of r;
//   VEC_WARM   warm start: stop = 0, partials of b . b and the projections of x;
//   VEC_PROJ   the projections of x;
//   VEC_RESTART r = b - Ap, partials of r . r into slot k & 1 and of its
//              projections.
// All loads, the low-rank columns among them, are issued before alpha is
// known: one system alone waits for one round trip and two reductions.
// x: per-system vectors of stride nact from the launch's first system.  Grid
// (chunks, systems).
enum { VEC_STEP, VEC_COLD, VEC_WARM, VEC_PROJ, VEC_RESTART };
template <int MODE>
__global__ __launch_bounds__(FVT) void kf_vec(const FMv M, double *__restrict__ x, int ws0, int k) {
    constexpr int NE = FCH / FVT, NW = FVT / 64;
    __shared__ double psh[NW][2];
    __shared__ double sums[16][NW + 1];
    const int s = ws0 + blockIdx.y, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    double *q = M.part + (long)s * M.pstride;
    const long na = M.na;
    const int nlr = M.nlr, nch = M.nch;
    const int stopped = MODE == VEC_STEP ? M.stop[s] : 0;
    long ac[NE];
    bool on[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const long a = (long)blockIdx.x * FCH + i * FVT + t;
        on[i] = a < na;
        ac[i] = on[i] ? a : na - 1;
    }
    const long base = (long)s * na, xb = (long)blockIdx.y * na;
    double w[NE], bv[NE], pv[NE], ap[NE], xv[NE];  // w: the vector that is projected
    double c[16][NE];
#pragma unroll
    for (int i = 0; i < NE; i++) {
        w[i] = bv[i] = pv[i] = ap[i] = xv[i] = 0;
        if (MODE == VEC_STEP) {
            pv[i] = ((k & 1) ? M.p2 : M.p)[base + ac[i]];
            w[i] = M.r[base + ac[i]];
        }
        if (MODE == VEC_STEP || MODE == VEC_RESTART) ap[i] = M.Ap[base + ac[i]];
        if (MODE == VEC_COLD || MODE == VEC_WARM || MODE == VEC_RESTART) bv[i] = M.b[base + ac[i]];
        if (MODE == VEC_STEP || MODE == VEC_WARM || MODE == VEC_PROJ) xv[i] = x[xb + ac[i]];
    }
#pragma unroll
    for (int j = 0; j < 16; j++)
#pragma unroll
        for (int i = 0; i < NE; i++) c[j][i] = M.lr[(long)max(min(j, nlr - 1), 0) * na + ac[i]];
    if (MODE == VEC_STEP) {
        double rr = 0, pap = 0;
        for (int i = t; i < nch; i += FVT) rr += q[M.o4 + (k & 1) * nch + i];
        for (int i = t; i < M.ntile; i += FVT) pap += q[M.o2 + i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            rr += __shfl_down(rr, o, 64);
            pap += __shfl_down(pap, o, 64);
        }
        if (lane == 0) {
            psh[wv][0] = rr;
            psh[wv][1] = pap;
        }
        __syncthreads();
        rr = pap = 0;
#pragma unroll
        for (int i = 0; i < NW; i++) {
            rr += psh[i][0];
            pap += psh[i][1];
        }
        const double ak = rr / pap;
        if (stopped || !isfinite(ak)) {
            if (!stopped && blockIdx.x == 0 && t == 0) {
                M.stop[s] = 1;
                M.res[s] = NAN;
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NE; i++) {
            w[i] = on[i] ? w[i] - ak * ap[i] : 0.0;
            if (on[i]) {
                x[xb + ac[i]] = xv[i] + ak * pv[i];
                M.r[base + ac[i]] = w[i];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < NE; i++) {
            w[i] = MODE == VEC_COLD ? bv[i] : MODE == VEC_RESTART ? bv[i] - ap[i] : xv[i];
            if (!on[i]) w[i] = bv[i] = 0;
            if (MODE == VEC_COLD && on[i]) x[xb + ac[i]] = 0;
            if ((MODE == VEC_COLD || MODE == VEC_RESTART) && on[i]) M.r[base + ac[i]] = w[i];
        }
        if ((MODE == VEC_COLD || MODE == VEC_WARM) && blockIdx.x == 0 && t == 0) M.stop[s] = 0;
    }
    // sums of the nlr projections, of w . w and of b . b, sixteen at a time
    for (int j0 = 0; j0 < nlr + 2; j0 += 16) {
        double u[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            u[j] = 0;
#pragma unroll
            for (int i = 0; i < NE; i++) {
                const double wi = w[i], bi = bv[i];
                double cj = c[j][i];
                if (j0) cj = M.lr[(long)max(min(j0 + j, nlr - 1), 0) * na + ac[i]];
                if (j0 + j == nlr) cj = wi;
                u[j] += j0 + j > nlr ? bi * bi : cj * wi;
            }
        }
        const double v = wave_red16(u);
        if (j0) __syncthreads();  // the previous sixteen are read
        if ((lane & 3) == 0) sums[lane >> 2][wv] = v;
        __syncthreads();
        const int j = j0 + t;
        if (t < 16 && j < nlr + 2) {
            double z = 0;
#pragma unroll
            for (int i = 0; i < NW; i++) z += sums[t][i];
            const int slot = MODE == VEC_STEP ? (k + 1) & 1 : MODE == VEC_RESTART ? k & 1 : 0;
            if (j < nlr) q[M.o3 + j * nch + blockIdx.x] = z;
            else if (j == nlr && (MODE == VEC_STEP || MODE == VEC_COLD || MODE == VEC_RESTART))
                q[M.o4 + slot * nch + blockIdx.x] = z;
            else if (j == nlr + 1 && (MODE == VEC_COLD || MODE == VEC_WARM)) q[M.o5 + blockIdx.x] = z;
        }
    }
}

// Residual sqrt(r.r / b.b) after the last iteration k.  One workgroup per system.
__global__ __launch_bounds__(FB) void kf_res(const FitDev *__restrict__ Dp, int ws0, int k) {
    const FitDev &D = *Dp;
    __shared__ double psh[4];
    const int s = ws0 + blockIdx.x;
    if (D.stop[s]) return;
    const double *q = fpart(D, s);
    const double rr = psum(q + D.o4 + ((k + 1) & 1) * D.nch, D.nch, psh);
    const double bb = psum(q + D.o5, D.nch, psh);
    if (threadIdx.x == 0) D.res[s] = sqrt(rr / bb);
}

// Forward taps of one axis: output coordinates u_k (in source grid units).
std::vector<Tap2> axis_taps(const std::vector<double> &u, long nsrc) {
    std::vector<Tap2> t(u.size());
    for (size_t k = 0; k < u.size(); k++) {
        const double fl = std::floor(u[k]);
        const long n0 = (long)fl;
        const double f = u[k] - fl;
        Tap2 &a = t[k];
        a.n = (int)n0;
        a.pad_ = 0;
        a.w0 = (n0 >= 0 && n0 < nsrc) ? 1 - f : 0;
        a.w1 = (n0 + 1 >= 0 && n0 + 1 < nsrc) ? f : 0;
        // weights of off-grid nodes are zero; keep the node index in range
        // so the (never used) address stays inside the source
        if (a.w0 == 0 && a.w1 == 0) a.n = 0;
        else if (a.n < 0) a.n = -1;
    }
    return t;
}

}  // namespace

struct gpu_fit {
    int device = 0, nbatch = 1, maxit = 10, warm = 0;
    hipStream_t stream = nullptr;
    FitDev H{};
    DBuf<FitDev> dev;
    DBuf<Tap2> hax, hay, hxx, hxy;
    DBuf<int> txp, typ;
    DBuf<TapT> txe, tye;
    DBuf<double> W0, W1, slx;
    DBuf<long> slp, sli;
    DBuf<double> lr, coef;
    FMv M{};  // assembled operator
    int wmax = 0;  // largest window
    DBuf<int> list, eo, epos;
    DBuf<FTile> tile;
    DBuf<double> lrc;
    DBuf<double> opd, opd2, tnw, r, p, p2, Ap, b, part, res, x;
    DBuf<int> stop;
    DBuf<float> xin;
    std::vector<float> hstage;
    // captured solves (the ~500 launches of a 100-iteration solve replay with
    // graph-node gaps instead of launch gaps), keyed by their arguments
    struct Graph {
        const float *xin;
        long xstride;
        double *x;
        int ws0, n, warm, maxit;
        hipGraph_t graph;
        hipGraphExec_t exec;
        hipEvent_t done;  // recorded after each launch
    };
    std::vector<Graph> graphs;  // most recently used last
    hipStream_t cap = nullptr;  // capture stream
};

namespace {

template <typename F>
int fguarded(F &&f) {
    try {
        f();
        return MT_OK;
    } catch (const FitErr &e) {
        mt::set_error(e.msg);
        return e.code;
    } catch (const std::bad_alloc &) {
        mt::set_error("out of host memory");
        return MT_ENOMEM;
    } catch (const std::exception &e) {
        mt::set_error(e.what());
        return MT_EINVAL;
    }
}

// The assembled operator is used up to this mean box (entries of a row over all
// DMs): an entry costs about 0.3 us per iteration of 32 systems of the 30 m
// fit, a direction of the matrix-free passes 11 us, which also cost three more
// launches.  Nine directions on a ring, 20 warm iterations, assembled against
// matrix-free, one system / 32: 15" (about 75 entries) 267 against 663 / 678
// against 1993 us, 30" (150) 291 / 652, 823 / 2023, 60" (350) 655 / 656,
// 2265 / 2088, 90" 1093 / 655, 5515 / 2189.
constexpr int FASM_ENTRIES = 256, FASM_BASE = 64, FASM_PER_DIR = 24;
// ... and to this much memory for the coefficients.
constexpr size_t FASM_BYTES = (size_t)1 << 30;
constexpr int FLDS = 65536;  // LDS of a workgroup without an attribute

// LDS of a kf_mv workgroup besides its windows.
constexpr size_t MV_STATIC = sizeof(double) * (8 * 64 + FSW * (FMAXNW + FMAXFIT + 1));

// Boxes, tiles and windows of the assembled operator (kf_mv); false when the
// boxes are too large for it (directions far apart on a high DM).
bool plan_assembled(gpu_fit *g, const std::vector<Tap2> &hax, const std::vector<Tap2> &hay, const std::vector<int> &txp,
                    const std::vector<int> &typ, const std::vector<TapT> &txe, const std::vector<TapT> &tye,
                    const mt_fit_recon_t *F) {
    FitDev &D = g->H;
    const int nd = D.ndm;
    // a row's nodes in DM d2 relative to its own indices: the nodes its taps
    // reach through W0 along any direction, its slaving entries, itself; one
    // box per pair, the hull over the rows (a row uses less of it where the
    // DMs' spacings differ)
    int lo[2][FMAXDM * FMAXDM], hi[2][FMAXDM * FMAXDM];
    auto add = [&](int ax, int pr, int a, int j) {
        lo[ax][pr] = std::min(lo[ax][pr], j - a);
        hi[ax][pr] = std::max(hi[ax][pr], j - a);
    };
    for (int d1 = 0; d1 < nd; d1++)
        for (int d2 = 0; d2 < nd; d2++)
            for (int ax = 0; ax < 2; ax++) {
                const int pr = d1 * FMAXDM + d2;
                const int n1 = (int)(ax ? F->any[d1] : F->anx[d1]), n2 = (int)(ax ? F->any[d2] : F->anx[d2]);
                const int fn = ax ? D.fny : D.fnx;
                const std::vector<Tap2> &h = ax ? hay : hax;
                const std::vector<int> &tp = ax ? typ : txp;
                const std::vector<TapT> &te = ax ? tye : txe;
                const int stride = ax ? D.tpy : D.tpx, base = ax ? D.tdy[d1] : D.tdx[d1];
                lo[ax][pr] = INT32_MAX;
                hi[ax][pr] = INT32_MIN;
                if (d1 == d2) add(ax, pr, 0, 0);
                for (int a = 0; a < n1; a++)
                    for (int f = 0; f < D.nfit; f++)
                        for (int e = tp[f * stride + base + a]; e < tp[f * stride + base + a + 1]; e++)
                            for (int q = std::max(te[e].i - 1, 0); q <= std::min(te[e].i + 1, fn - 1); q++) {
                                const Tap2 &t = h[(size_t)(f * nd + d2) * fn + q];
                                if (t.w0 != 0 && t.n >= 0 && t.n < n2) add(ax, pr, a, t.n);
                                if (t.w1 != 0 && t.n + 1 >= 0 && t.n + 1 < n2) add(ax, pr, a, t.n + 1);
                            }
            }
    if (F->sl_p) {
        for (int d1 = 0; d1 < nd; d1++)
            for (long a = D.aoff[d1]; a < D.aoff[d1 + 1]; a++)
                for (long e = F->sl_p[a]; e < F->sl_p[a + 1]; e++) {
                    int d2 = 0;
                    while (F->sl_i[e] >= D.aoff[d2 + 1]) d2++;
                    const long k1 = a - D.aoff[d1], k2 = F->sl_i[e] - D.aoff[d2];
                    const int pr = d1 * FMAXDM + d2;
                    add(0, pr, (int)(k1 % F->anx[d1]), (int)(k2 % F->anx[d2]));
                    add(1, pr, (int)(k1 / F->anx[d1]), (int)(k2 / F->anx[d2]));
                }
    }
    double entries = 0;
    for (int d1 = 0; d1 < nd; d1++) {
        D.etot[d1] = 0;
        for (int d2 = 0; d2 < nd; d2++) {
            const int pr = d1 * FMAXDM + d2;
            const bool any = lo[0][pr] <= hi[0][pr] && lo[1][pr] <= hi[1][pr];
            D.bx[pr] = any ? lo[0][pr] : 0;
            D.by[pr] = any ? lo[1][pr] : 0;
            D.kx[pr] = any ? hi[0][pr] - lo[0][pr] + 1 : 0;
            D.ky[pr] = any ? hi[1][pr] - lo[1][pr] + 1 : 0;
            if ((double)D.kx[pr] * D.ky[pr] > 4096) return false;  // positions are kept in 12 bits
            D.etot[d1] += D.kx[pr] * D.ky[pr];
        }
        entries += (double)D.etot[d1] * (D.aoff[d1 + 1] - D.aoff[d1]);
    }
    if (entries > (double)std::min(FASM_ENTRIES, FASM_BASE + FASM_PER_DIR * D.nfit) * D.nact) return false;
    // entries of a row in the order of the sums: DM, box column, box row; the
    // four sums take consecutive quarters
    std::vector<int> epos;
    for (int d1 = 0; d1 < nd; d1++) {
        D.ebase[d1] = (int)epos.size();
        for (int d2 = 0; d2 < nd; d2++)
            for (int x = 0; x < D.kx[d1 * FMAXDM + d2]; x++)
                for (int y = 0; y < D.ky[d1 * FMAXDM + d2]; y++) epos.push_back(x | y << 12 | d2 << 24);
    }
    // window of a tile: the boxes' nodes in every DM, all at one pitch, so that
    // an entry is at one offset from every row
    int pitch[FMAXDM], woff[FMAXDM * FMAXDM], wn[FMAXDM], eob[FMAXDM];
    std::vector<int> eo;
    g->wmax = 0;
    for (int d1 = 0; d1 < nd; d1++) {
        pitch[d1] = wn[d1] = 0;
        for (int d2 = 0; d2 < nd; d2++) pitch[d1] = std::max(pitch[d1], FTX - 1 + D.kx[d1 * FMAXDM + d2]);
        for (int d2 = 0; d2 < nd; d2++) {
            const int pr = d1 * FMAXDM + d2;
            woff[pr] = wn[d1];
            if (D.ky[pr]) wn[d1] += pitch[d1] * (FTY - 1 + D.ky[pr]);
        }
        eob[d1] = (int)eo.size();
        for (int e = 0; e < D.etot[d1]; e++) {
            const int ps = epos[D.ebase[d1] + e];
            eo.push_back(woff[d1 * FMAXDM + (ps >> 24)] + (ps >> 12 & 0xfff) * pitch[d1] + (ps & 0xfff));
        }
        g->wmax = std::max(g->wmax, wn[d1]);
    }
    if (sizeof(double) * 2 * g->wmax + MV_STATIC > FLDS) return false;
    std::vector<FTile> tile;
    std::vector<int> list;
    long coef = 0;
    for (int d1 = 0; d1 < nd; d1++)
        for (int ja = 0; ja < D.any[d1]; ja += FTY)
            for (int ia = 0; ia < D.anx[d1]; ia += FTX) {
                FTile T{};
                T.coef = coef;
                T.d = d1;
                T.ia0 = ia;
                T.ja0 = ja;
                T.anx = D.anx[d1];
                T.a0 = (int)D.aoff[d1] + ja * D.anx[d1] + ia;
                T.nx = std::min(FTX, D.anx[d1] - ia);
                T.ny = std::min(FTY, D.any[d1] - ja);
                T.eo = eob[d1];
                for (int q = 0; q <= 4; q++) T.cls[q] = (int)((long)D.etot[d1] * q / 4);
                T.wn = wn[d1];
                T.lst = (int)list.size();
                T.pitch = pitch[d1];
                T.own = woff[d1 * FMAXDM + d1] - D.by[d1 * FMAXDM + d1] * pitch[d1] - D.bx[d1 * FMAXDM + d1];
                // nodes outside a DM read any actuator (their coefficients are zero)
                list.resize(list.size() + wn[d1], T.a0);
                for (int d2 = 0; d2 < nd; d2++) {
                    const int pr = d1 * FMAXDM + d2;
                    for (int y = 0; D.ky[pr] && y < FTY - 1 + D.ky[pr]; y++)
                        for (int x = 0; x < FTX - 1 + D.kx[pr]; x++) {
                            const int jx = ia + D.bx[pr] + x, jy = ja + D.by[pr] + y;
                            if (jx < 0 || jx >= D.anx[d2] || jy < 0 || jy >= D.any[d2]) continue;
                            list[T.lst + woff[pr] + y * pitch[d1] + x] = (int)D.aoff[d2] + jy * D.anx[d2] + jx;
                        }
                }
                tile.push_back(T);
                coef += (long)D.etot[d1] * FTX * FTY;
            }
    if ((size_t)coef * sizeof(double) > FASM_BYTES || list.size() > (size_t)INT32_MAX) return false;
    D.ntile = (int)tile.size();
    g->tile.upload(tile);
    g->epos.upload(epos);
    g->list.upload(list);
    g->eo.upload(eo);
    g->coef.alloc(coef + FTX * FTY * FNC);  // kf_mv loads FNC entries of any wave
    D.tile = g->tile.p;
    D.epos = g->epos.p;
    return true;
}

void build_fit_plan(gpu_fit *g, const mt_recon_t *R, const mt_fit_recon_t *F) {
    FitDev &D = g->H;
    if (F->ndm <= 0 || F->ndm > FMAXDM) ffail(MT_EINVAL, "gpu_fit_setup: 1 to 8 DMs");
    if (F->nfit <= 0 || F->nfit > FMAXFIT) ffail(MT_EINVAL, "gpu_fit_setup: 1 to 32 fitting directions");
    if (R->npsr <= 0 || R->npsr > FMAXL) ffail(MT_EINVAL, "gpu_fit_setup: 1 to 16 layers");
    if (F->nnw < 0 || F->nnw > FMAXNW) ffail(MT_EINVAL, "gpu_fit_setup: at most 32 low-rank terms");
    D.nfit = F->nfit;
    D.ndm = F->ndm;
    D.npsr = R->npsr;
    D.nnw = F->nnw;
    D.fnx = (int)F->fnx;
    D.fny = (int)F->fny;
    D.nfloc = F->fnx * F->fny;
    D.aoff[0] = 0;
    for (int d = 0; d < D.ndm; d++) {
        D.anx[d] = (int)F->anx[d];
        D.any[d] = (int)F->any[d];
        D.aoff[d + 1] = D.aoff[d] + F->anx[d] * F->any[d];
    }
    D.nact = D.aoff[D.ndm];
    D.xoff[0] = 0;
    for (int l = 0; l < D.npsr; l++) {
        D.xnx[l] = (int)R->xnx[l];
        D.xny[l] = (int)R->xny[l];
        D.xoff[l + 1] = D.xoff[l] + R->xnx[l] * R->xny[l];
    }
    D.nxtot = D.xoff[D.npsr];
    for (int f = 0; f < D.nfit; f++) D.wt[f] = F->wt[f];
    // forward taps, as mkh computes the interpolation point: source-grid
    // coordinate = (x * scale + theta * ht - origin) / dx
    const long fnx = F->fnx, fny = F->fny;
    std::vector<Tap2> hax, hay, hxx, hxy;
    std::vector<int> txb, tyb, txp, typ;
    std::vector<TapT> txe, tye;
    for (int f = 0; f < D.nfit; f++) {
        for (int d = 0; d < D.ndm; d++) {
            const double ht = F->aht[d], sc = 1. - ht / F->hs[f];
            std::vector<double> ux(fnx), uy(fny);
            for (long i = 0; i < fnx; i++) ux[i] = ((F->fox + i * F->fdx) * sc + F->thetax[f] * ht - F->aox[d]) / F->adx[d];
            for (long i = 0; i < fny; i++) uy[i] = ((F->foy + i * F->fdx) * sc + F->thetay[f] * ht - F->aoy[d]) / F->adx[d];
            const std::vector<Tap2> tx = axis_taps(ux, F->anx[d]), ty = axis_taps(uy, F->any[d]);
            hax.insert(hax.end(), tx.begin(), tx.end());
            hay.insert(hay.end(), ty.begin(), ty.end());
            // transposed lists per actuator column / row
            auto transpose = [](const std::vector<Tap2> &t, long nsrc, std::vector<int> &bases, std::vector<int> &ptr,
                                std::vector<TapT> &ent) {
                std::vector<std::vector<TapT>> lists(nsrc);
                for (size_t k = 0; k < t.size(); k++) {
                    if (t[k].w0 != 0) lists[t[k].n].push_back(TapT{(int)k, 0, t[k].w0});
                    if (t[k].w1 != 0) lists[t[k].n + 1].push_back(TapT{(int)k, 0, t[k].w1});
                }
                bases.push_back((int)ptr.size());
                for (long a = 0; a < nsrc; a++) {
                    ptr.push_back((int)ent.size());
                    ent.insert(ent.end(), lists[a].begin(), lists[a].end());
                }
                ptr.push_back((int)ent.size());
            };
            transpose(tx, F->anx[d], txb, txp, txe);
            transpose(ty, F->any[d], tyb, typ, tye);
        }
        for (int l = 0; l < D.npsr; l++) {
            const double ht = R->ht[l], sc = 1. - ht / F->hs[f];
            std::vector<double> ux(fnx), uy(fny);
            for (long i = 0; i < fnx; i++) ux[i] = ((F->fox + i * F->fdx) * sc + F->thetax[f] * ht - R->xox[l]) / R->xdx[l];
            for (long i = 0; i < fny; i++) uy[i] = ((F->foy + i * F->fdx) * sc + F->thetay[f] * ht - R->xoy[l]) / R->xdx[l];
            const std::vector<Tap2> tx = axis_taps(ux, R->xnx[l]), ty = axis_taps(uy, R->xny[l]);
            hxx.insert(hxx.end(), tx.begin(), tx.end());
            hxy.insert(hxy.end(), ty.begin(), ty.end());
        }
    }
    if (txe.size() > (size_t)INT32_MAX || tye.size() > (size_t)INT32_MAX || D.nfloc * D.nfit >= INT32_MAX ||
        D.nact >= INT32_MAX)
        ffail(MT_EINVAL, "fitting tables too large");
    g->hax.upload(hax);
    g->hay.upload(hay);
    g->hxx.upload(hxx);
    g->hxy.upload(hxy);
    // the pointer arrays' bases follow from the grid sizes
    D.tpx = D.tpy = 0;
    for (int d = 0; d < D.ndm; d++) {
        D.tdx[d] = D.tpx;
        D.tdy[d] = D.tpy;
        D.tpx += D.anx[d] + 1;
        D.tpy += D.any[d] + 1;
    }
    for (int f = 0; f < D.nfit; f++)
        for (int d = 0; d < D.ndm; d++)
            if (txb[f * D.ndm + d] != f * D.tpx + D.tdx[d] || tyb[f * D.ndm + d] != f * D.tpy + D.tdy[d])
                ffail(MT_EINVAL, "fitting tables: unexpected layout");
    g->txp.upload(txp);
    g->typ.upload(typ);
    g->txe.upload(txe);
    g->tye.upload(tye);
    g->W0.upload(std::vector<double>(F->W0, F->W0 + 9 * D.nfloc));
    g->W1.upload(std::vector<double>(F->W1, F->W1 + D.nfloc));
    if (F->sl_p) {
        std::vector<long> p(F->sl_p, F->sl_p + D.nact + 1);
        const long nz = p[D.nact];
        g->slp.upload(p);
        g->sli.upload(std::vector<long>(F->sl_i, F->sl_i + nz));
        g->slx.upload(std::vector<double>(F->sl_x, F->sl_x + nz));
    }
    D.hax = g->hax.p;
    D.hay = g->hay.p;
    D.hxx = g->hxx.p;
    D.hxy = g->hxy.p;
    D.txp = g->txp.p;
    D.typ = g->typ.p;
    D.txe = g->txe.p;
    D.tye = g->tye.p;
    D.W0 = g->W0.p;
    D.W1 = g->W1.p;
    D.slp = g->slp.p;
    D.sli = g->sli.p;
    D.slx = g->slx.p;
    D.tikdiag = F->tikdiag;
    D.asm_ok = plan_assembled(g, hax, hay, txp, typ, txe, tye, F) ? 1 : 0;
    D.nlr = D.nnw + (D.asm_ok ? D.nfit : 0);
    for (int k = 0; k < D.nlr; k++) D.lrc[k] = k < D.nnw ? 1.0 : -D.wt[k - D.nnw];
    g->lr.alloc((size_t)D.nlr * D.nact);
    if (D.nnw)
        FCHK(hipMemcpy(g->lr.p, F->NW, sizeof(double) * D.nnw * D.nact, hipMemcpyHostToDevice));
    D.lr = g->lr.p;
    // workspace
    const long ns = g->nbatch;
    g->opd.alloc(ns * D.nfit * D.nfloc);
    g->opd2.alloc(ns * D.nfit * D.nfloc);
    g->r.alloc(ns * D.nact);
    g->p.alloc(ns * D.nact);
    if (D.asm_ok) g->p2.alloc(ns * D.nact);
    g->Ap.alloc(ns * D.nact);
    g->b.alloc(ns * D.nact);
    g->tnw.alloc(ns * FMAXNW);
    D.tnw = g->tnw.p;
    D.nc1 = (int)((D.nfloc + FB - 1) / FB);
    D.hab = FB / D.nfit;
    D.nc3 = (int)((D.nact + (long)HAH * D.hab - 1) / ((long)HAH * D.hab));
    D.nc4 = (int)((D.nact + FB - 1) / FB);
    D.o1 = 0;
    D.o2 = D.o1 + D.nfit * D.nc1;
    D.nch = D.asm_ok ? (int)((D.nact + FCH - 1) / FCH) : D.nc4;
    D.o3 = D.o2 + (D.asm_ok ? D.ntile : D.nc3);
    D.o4 = D.o3 + D.nlr * D.nch;
    D.o5 = D.o4 + 2 * D.nch;
    D.o6 = D.o5 + D.nch;
    D.pstride = D.o6 + (D.asm_ok ? 2 * D.nlr : 0);
    g->part.alloc(ns * D.pstride);
    g->stop.alloc(ns);
    FCHK(hipMemset(g->stop.p, 0, sizeof(int) * ns));
    g->res.alloc(ns);
    g->x.alloc(ns * D.nact);
    g->xin.alloc(ns * D.nxtot);
    FCHK(hipMemset(g->x.p, 0, sizeof(double) * ns * D.nact));
    D.opd = g->opd.p;
    D.opd2 = g->opd2.p;
    D.r = g->r.p;
    D.p = g->p.p;
    D.Ap = g->Ap.p;
    D.b = g->b.p;
    D.part = g->part.p;
    D.stop = g->stop.p;
    D.res = g->res.p;
    g->dev.alloc(1);
    FCHK(hipMemcpy(g->dev.p, &D, sizeof(FitDev), hipMemcpyHostToDevice));
    if (D.asm_ok) {
        FMv &M = g->M;
        g->lrc.upload(std::vector<double>(D.lrc, D.lrc + D.nlr));
        M.tile = g->tile.p;
        M.list = g->list.p;
        M.eo = g->eo.p;
        M.coef = g->coef.p;
        M.lr = D.lr;
        M.lrc = g->lrc.p;
        M.r = D.r;
        M.p = D.p;
        M.p2 = g->p2.p;
        M.Ap = D.Ap;
        M.b = D.b;
        M.part = D.part;
        M.res = D.res;
        M.stop = D.stop;
        M.na = D.nact;
        M.pstride = D.pstride;
        M.nlr = D.nlr;
        M.nch = D.nch;
        M.ntile = D.ntile;
        M.o2 = D.o2;
        M.o3 = D.o3;
        M.o4 = D.o4;
        M.o5 = D.o5;
        M.o6 = D.o6;
        const int emax = *std::max_element(D.etot, D.etot + D.ndm);
        hipLaunchKernelGGL(kf_assemble, dim3(D.ntile, (emax + 3) / 4), dim3(FB), 0, 0, g->dev.p, g->coef.p);
        hipLaunchKernelGGL(kf_lowrank, dim3(D.nc4, D.nfit), dim3(FB), 0, 0, g->dev.p, g->lr.p + (size_t)D.nnw * D.nact);
        FCHK(hipGetLastError());
        FCHK(hipStreamSynchronize(0));
    }
}

// Launch sequences.  ws0: first workspace slot; n: systems; external
// vectors are given for the first system of the launch, stride nact (actuator
// vectors) or xstride (layer vectors).
dim3 grid_pts(const FitDev &D, int n) { return dim3(D.nc1, D.nfit, n); }
dim3 grid_hat(const FitDev &D, int n) { return dim3(D.nc3, n); }
dim3 grid_act(const FitDev &D, int n) { return dim3(D.nc4, n); }
dim3 grid_vec(const FitDev &D, int n) { return dim3(D.nch, n); }  // assembled

// Interpolation from nsrc sources, GS of them per group of loads: 2 for up
// to two sources, 3 for three, else 4 (a partial last group reloads the
// last source).
template <int SRC>
void launch_fwd(const FitDev &D, int nsrc, dim3 grid, hipStream_t st, const FitDev *dev, const void *src, long sstride,
                int ws0) {
    if (nsrc <= 2) hipLaunchKernelGGL((kf_fwd<SRC, 2>), grid, dim3(FB), 0, st, dev, src, sstride, ws0);
    else if (nsrc == 3) hipLaunchKernelGGL((kf_fwd<SRC, 3>), grid, dim3(FB), 0, st, dev, src, sstride, ws0);
    else hipLaunchKernelGGL((kf_fwd<SRC, 4>), grid, dim3(FB), 0, st, dev, src, sstride, ws0);
}

// out = sum_f wt_f HA_f' W HX_f x (FitR)
void enq_rhs(gpu_fit *g, hipStream_t st, const float *xin, long xstride, double *out, int ws0, int n) {
    const FitDev &D = g->H;
    launch_fwd<1>(D, D.npsr, grid_pts(D, n), st, g->dev.p, (const void *)xin, xstride, ws0);
    hipLaunchKernelGGL(kf_w, grid_pts(D, n), dim3(FB), 0, st, g->dev.p, ws0, 0);
    hipLaunchKernelGGL(kf_hat<HAT_R>, grid_hat(D, n), dim3(FB), 0, st, g->dev.p, (const double *)nullptr, out, ws0);
}

// FitL of n systems with the assembled operator.
template <int MODE>
void launch_mv(gpu_fit *g, hipStream_t st, const double *v, double *out, int ws0, int n, int k, int first) {
    const int nt = (g->M.ntile + 7) / 8 * 8;
    // about five workgroups per CU (what its registers hold), each with at
    // least one system and at most FSW
    const int groups = std::max(std::min(n, 1280 / nt), (n + FSW - 1) / FSW);
    const int spw = (n + groups - 1) / groups;
    hipLaunchKernelGGL((kf_mv<MODE>), dim3(nt, (n + spw - 1) / spw), dim3(FB), sizeof(double) * 2 * g->wmax, st, g->M, v,
                       out, ws0, n, spw, k, first);
}

// out = FitL p; the partials of the low-rank projections of p must be in
// place (kf_init, kf_restart or kf_p wrote them).
void enq_L(gpu_fit *g, hipStream_t st, const double *p, double *out, int ws0, int n) {
    const FitDev &D = g->H;
    if (D.asm_ok) {
        launch_mv<MV_PLAIN>(g, st, p, out, ws0, n, 0, 0);
        return;
    }
    launch_fwd<0>(D, D.ndm, grid_pts(D, n), st, g->dev.p, (const void *)p, D.nact, ws0);
    hipLaunchKernelGGL(kf_w, grid_pts(D, n), dim3(FB), 0, st, g->dev.p, ws0, 1);
    hipLaunchKernelGGL(kf_hat<HAT_L>, grid_hat(D, n), dim3(FB), 0, st, g->dev.p, p, out, ws0);
}

// The whole solve of n systems (lib/pcg.c:28-113 with Mmul = NULL: z = r,
// restart every 100 iterations): 2 launches per iteration with the assembled
// operator, else 5.
void enq_solve(gpu_fit *g, hipStream_t st, const float *xin, long xstride, double *x, int ws0, int n, int warm,
               int maxit) {
    const FitDev &D = g->H;
    const long na = D.nact;
    double *b = g->b.p + (long)ws0 * na, *p = g->p.p + (long)ws0 * na, *Ap = g->Ap.p + (long)ws0 * na;
    enq_rhs(g, st, xin, xstride, b, ws0, n);
    if (!D.asm_ok) hipLaunchKernelGGL(kf_init<true>, grid_act(D, n), dim3(FB), 0, st, g->dev.p, x, ws0, warm);
    else if (warm) hipLaunchKernelGGL(kf_vec<VEC_WARM>, grid_vec(D, n), dim3(FVT), 0, st, g->M, x, ws0, 0);
    else hipLaunchKernelGGL(kf_vec<VEC_COLD>, grid_vec(D, n), dim3(FVT), 0, st, g->M, x, ws0, 0);
    for (int k = 0; k < maxit; k++) {
        if (k % 100 == 0) {
            if (D.asm_ok) {
                if (k > 0) hipLaunchKernelGGL(kf_vec<VEC_PROJ>, grid_vec(D, n), dim3(FVT), 0, st, g->M, x, ws0, k);
                if (k > 0 || warm) {
                    enq_L(g, st, x, Ap, ws0, n);
                    hipLaunchKernelGGL(kf_vec<VEC_RESTART>, grid_vec(D, n), dim3(FVT), 0, st, g->M, x, ws0, k);
                }
            } else if (k == 0 && !warm) {
                hipLaunchKernelGGL(kf_restart<true>, grid_act(D, n), dim3(FB), 0, st, g->dev.p, ws0, k);
            } else {
                if (k > 0) hipLaunchKernelGGL(kf_init<false>, grid_act(D, n), dim3(FB), 0, st, g->dev.p, x, ws0, 1);
                enq_L(g, st, x, Ap, ws0, n);
                hipLaunchKernelGGL(kf_restart<false>, grid_act(D, n), dim3(FB), 0, st, g->dev.p, ws0, k);
            }
        }
        if (D.asm_ok) {
            launch_mv<MV_CG>(g, st, nullptr, g->Ap.p, ws0, n, k, (int)(k % 100 == 0));
            hipLaunchKernelGGL(kf_vec<VEC_STEP>, grid_vec(D, n), dim3(FVT), 0, st, g->M, x, ws0, k);
            if (k + 1 == maxit) hipLaunchKernelGGL(kf_res, dim3(n), dim3(FB), 0, st, g->dev.p, ws0, k);
            continue;
        }
        enq_L(g, st, p, Ap, ws0, n);
        hipLaunchKernelGGL(kf_upd, grid_act(D, n), dim3(FB), 0, st, g->dev.p, x, ws0, k);
        hipLaunchKernelGGL(kf_p, grid_act(D, n), dim3(FB), 0, st, g->dev.p, ws0, k, (int)(k + 1 == maxit));
    }
    FCHK(hipGetLastError());
}

constexpr size_t FIT_GRAPHS = 8;  // captured solves kept per plan

// Destroy a captured solve once its last launch (which an asynchronous
// caller may not have waited for) has completed.
void drop_graph(gpu_fit::Graph &e) {
    if (e.done) {
        (void)hipEventSynchronize(e.done);
        (void)hipEventDestroy(e.done);
    }
    if (e.exec) (void)hipGraphExecDestroy(e.exec);
    if (e.graph) (void)hipGraphDestroy(e.graph);
}
void drop_graphs(gpu_fit *g) {
    for (auto &e : g->graphs) drop_graph(e);
    g->graphs.clear();
}

// The solve as a replay of a captured graph on st (captured on first use of
// these arguments); direct launches when st is itself being captured.
void run_solve(gpu_fit *g, hipStream_t st, const float *xin, long xstride, double *x, int ws0, int n, int warm,
               int maxit) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FCHK(hipStreamIsCapturing(st, &cs));
    if (cs != hipStreamCaptureStatusNone) {
        enq_solve(g, st, xin, xstride, x, ws0, n, warm, maxit);
        return;
    }
    size_t k = 0;
    for (; k < g->graphs.size(); k++) {
        const auto &e = g->graphs[k];
        if (e.xin == xin && e.xstride == xstride && e.x == x && e.ws0 == ws0 && e.n == n && e.warm == warm &&
            e.maxit == maxit)
            break;
    }
    if (k == g->graphs.size()) {
        if (!g->cap) FCHK(hipStreamCreateWithFlags(&g->cap, hipStreamNonBlocking));
        gpu_fit::Graph e{xin, xstride, x, ws0, n, warm, maxit, nullptr, nullptr, nullptr};
        FCHK(hipStreamBeginCapture(g->cap, hipStreamCaptureModeThreadLocal));
        try {
            enq_solve(g, g->cap, xin, xstride, x, ws0, n, warm, maxit);
        } catch (...) {
            hipGraph_t dropped = nullptr;
            (void)hipStreamEndCapture(g->cap, &dropped);
            if (dropped) (void)hipGraphDestroy(dropped);
            throw;
        }
        FCHK(hipStreamEndCapture(g->cap, &e.graph));
        hipError_t ie = hipGraphInstantiate(&e.exec, e.graph, nullptr, nullptr, 0);
        if (ie == hipSuccess) ie = hipEventCreateWithFlags(&e.done, hipEventDisableTiming);
        if (ie != hipSuccess) {
            drop_graph(e);
            FCHK(ie);
        }
        if (g->graphs.size() >= FIT_GRAPHS) {
            drop_graph(g->graphs.front());
            g->graphs.erase(g->graphs.begin());
        }
        g->graphs.push_back(e);
        k = g->graphs.size() - 1;
    } else if (k + 1 != g->graphs.size()) {
        std::rotate(g->graphs.begin() + k, g->graphs.begin() + k + 1, g->graphs.end());
        k = g->graphs.size() - 1;
    }
    FCHK(hipGraphLaunch(g->graphs[k].exec, st));
    FCHK(hipEventRecord(g->graphs[k].done, st));
}

void stage_x(gpu_fit *g, int isys, const double *opdr) {
    const long n = g->H.nxtot;
    g->hstage.resize(n);
    for (long i = 0; i < n; i++) {
        if (!std::isfinite(opdr[i])) ffail(MT_ENOTFINITE, "non-finite tomography input");
        g->hstage[i] = (float)opdr[i];
    }
    FCHK(hipMemcpyAsync(g->xin.p + (long)isys * n, g->hstage.data(), sizeof(float) * n, hipMemcpyHostToDevice,
                        g->stream));
}

}  // namespace

extern "C" {

int gpu_fit_setup(const mt_recon_t *recon, const mt_fit_recon_t *fit, int device, int nbatch, gpu_fit_t **out) {
    if (!out) return MT_EINVAL;
    *out = nullptr;
    if (!recon || !fit || nbatch <= 0 || nbatch > 65535 || fit->maxit <= 0 || fit->maxit > 100000) {
        mt::set_error("gpu_fit_setup: invalid arguments");
        return MT_EINVAL;
    }
    std::unique_ptr<gpu_fit> g(new (std::nothrow) gpu_fit());
    if (!g) return MT_ENOMEM;
    int rc = fguarded([&] {
        int ndev = 0;
        FCHK(hipGetDeviceCount(&ndev));
        if (device < 0 || device >= ndev) ffail(MT_EINVAL, "gpu_fit_setup: no such device");
        g->device = device;
        FCHK(hipSetDevice(device));
        g->nbatch = nbatch;
        g->maxit = fit->maxit;
        g->warm = fit->warm ? 1 : 0;
        build_fit_plan(g.get(), recon, fit);
        FCHK(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
        FCHK(hipDeviceSynchronize());
    });
    if (rc == MT_OK) *out = g.release();
    return rc;
}

int gpu_fit_solve(gpu_fit_t *g, int isys, const double *opdr, double *dmfit, double *cgres) {
    if (!g || !opdr || !dmfit || isys < 0 || isys >= g->nbatch) return MT_EINVAL;
    double res = NAN;
    int rc = fguarded([&] {
        FCHK(hipSetDevice(g->device));
        stage_x(g, isys, opdr);
        const long na = g->H.nact;
        run_solve(g, g->stream, g->xin.p + (long)isys * g->H.nxtot, g->H.nxtot, g->x.p + (long)isys * na, isys, 1,
                  g->warm, g->maxit);
        FCHK(hipMemcpyAsync(dmfit, g->x.p + (long)isys * na, sizeof(double) * na, hipMemcpyDeviceToHost, g->stream));
        FCHK(hipMemcpyAsync(&res, g->res.p + isys, sizeof(double), hipMemcpyDeviceToHost, g->stream));
        FCHK(hipStreamSynchronize(g->stream));
    });
    if (cgres) *cgres = res;
    if (rc == MT_OK && !(res <= 1.0)) rc = MT_NOTCONV;
    return rc;
}

int gpu_fit_solve_dev(gpu_fit_t *g, const float *d_opdr, double *d_dmfit, int nsys, void *stream) {
    if (!g || !d_opdr || !d_dmfit || nsys <= 0 || nsys > g->nbatch) return MT_EINVAL;
    return fguarded([&] {
        FCHK(hipSetDevice(g->device));
        hipStream_t st = stream ? (hipStream_t)stream : g->stream;
        run_solve(g, st, d_opdr, g->H.nxtot, d_dmfit, 0, nsys, g->warm, g->maxit);
    });
}

int gpu_fit_R(gpu_fit_t *g, const double *opdr, double *out, double alpha) {
    if (!g || !opdr || !out) return MT_EINVAL;
    return fguarded([&] {
        FCHK(hipSetDevice(g->device));
        stage_x(g, 0, opdr);
        const long na = g->H.nact;
        enq_rhs(g, g->stream, g->xin.p, g->H.nxtot, g->Ap.p, 0, 1);
        FCHK(hipGetLastError());
        std::vector<double> h(na);
        FCHK(hipMemcpyAsync(h.data(), g->Ap.p, sizeof(double) * na, hipMemcpyDeviceToHost, g->stream));
        FCHK(hipStreamSynchronize(g->stream));
        for (long i = 0; i < na; i++) out[i] = alpha * h[i];
    });
}

int gpu_fit_L(gpu_fit_t *g, const double *a, double *out, double alpha, double beta) {
    if (!g || !a || !out) return MT_EINVAL;
    return fguarded([&] {
        FCHK(hipSetDevice(g->device));
        const long na = g->H.nact;
        for (long i = 0; i < na; i++)
            if (!std::isfinite(a[i])) ffail(MT_ENOTFINITE, "non-finite input vector");
        // the input goes to the p slot of system 0, the output to its r slot
        FCHK(hipMemcpyAsync(g->p.p, a, sizeof(double) * na, hipMemcpyHostToDevice, g->stream));
        if (g->H.asm_ok)
            hipLaunchKernelGGL(kf_vec<VEC_PROJ>, grid_vec(g->H, 1), dim3(FVT), 0, g->stream, g->M, g->p.p, 0, 0);
        else
            hipLaunchKernelGGL(kf_init<false>, grid_act(g->H, 1), dim3(FB), 0, g->stream, g->dev.p, g->p.p, 0, 1);
        enq_L(g, g->stream, g->p.p, g->r.p, 0, 1);
        FCHK(hipGetLastError());
        std::vector<double> h(na);
        FCHK(hipMemcpyAsync(h.data(), g->r.p, sizeof(double) * na, hipMemcpyDeviceToHost, g->stream));
        FCHK(hipStreamSynchronize(g->stream));
        for (long i = 0; i < na; i++) out[i] = beta * out[i] + alpha * h[i];
    });
}

int gpu_fit_info(const gpu_fit_t *g, int *assembled, int *entries, int *lowrank) {
    if (!g) return MT_EINVAL;
    const FitDev &D = g->H;
    if (assembled) *assembled = D.asm_ok;
    if (entries) *entries = D.asm_ok ? *std::max_element(D.etot, D.etot + D.ndm) : 0;
    if (lowrank) *lowrank = D.nlr;
    return MT_OK;
}

int gpu_fit_residuals(gpu_fit_t *g, double *cgres, int nsys) {
    if (!g || !cgres || nsys <= 0 || nsys > g->nbatch) return MT_EINVAL;
    return fguarded([&] {
        FCHK(hipSetDevice(g->device));
        FCHK(hipStreamSynchronize(g->stream));
        FCHK(hipMemcpy(cgres, g->res.p, sizeof(double) * nsys, hipMemcpyDeviceToHost));
    });
}

void gpu_fit_free(gpu_fit_t *g) {
    if (!g) return;
    (void)hipSetDevice(g->device);
    if (g->stream) (void)hipStreamSynchronize(g->stream);
    (void)hipDeviceSynchronize();
    drop_graphs(g);
    if (g->cap) (void)hipStreamDestroy(g->cap);
    if (g->stream) (void)hipStreamDestroy(g->stream);
    delete g;
}

}  // extern "C"

int fit_enqueue_cold(gpu_fit_t *g, const float *d_x, long xstride, double *d_dm, int nsys, hipStream_t st) {
    if (!g || !d_x || !d_dm || nsys <= 0) return MT_EINVAL;
    return fguarded([&] {
        const long na = g->H.nact;
        for (int s0 = 0; s0 < nsys; s0 += g->nbatch) {
            const int n = std::min(g->nbatch, nsys - s0);
            run_solve(g, st, d_x + (long)s0 * xstride, xstride, d_dm + (long)s0 * na, 0, n, 0, g->maxit);
        }
    });
}
long fit_nact(const gpu_fit_t *g) { return g->H.nact; }
long fit_nxtot(const gpu_fit_t *g) { return g->H.nxtot; }
int fit_device(const gpu_fit_t *g) { return g->device; }

