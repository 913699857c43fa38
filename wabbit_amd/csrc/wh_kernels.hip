// wh_kernels.hip -- FP64 HIP kernels of the block time step for gfx950.
//
// Every kernel works on the device block pool in the reference's heavy-data
// layout [Nb][neq][nz][ny][nx] (allocate_forest.f90:228) and on the active
// list hvy_active.  Arithmetic follows the reference's term order and is
// compiled with -ffp-contract=off, so each product and sum rounds on its own
// exactly as the CPU code does.
#include "wh_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace wh {

// ---------------------------------------------------------------------------
// FD stencils (rhs_ACM.f90:335-344 and :958-965).  Coefficients are compile-
// time constants; each stencil takes a value accessor f(o) -> field at offset
// o along one direction, so the same code reads global memory, an LDS tile or
// a register queue (constant offsets keep the queue in registers).
// ---------------------------------------------------------------------------
constexpr double A4_m2 = 1.0 / 12.0, A4_m1 = -2.0 / 3.0, A4_p1 = 2.0 / 3.0, A4_p2 = -1.0 / 12.0;
constexpr double B4_m2 = -1.0 / 12.0, B4_m1 = 4.0 / 3.0, B4_0 = -5.0 / 2.0, B4_p1 = 4.0 / 3.0,
                 B4_p2 = -1.0 / 12.0;
constexpr double TW_m3 = -0.02651995, TW_m2 = 0.18941314, TW_m1 = -0.79926643,
                 TW_p1 = 0.79926643, TW_p2 = -0.18941314, TW_p3 = 0.02651995;
constexpr double A6_m3 = -1.0 / 60.0, A6_m2 = 3.0 / 20.0, A6_m1 = -3.0 / 4.0, A6_p1 = 3.0 / 4.0,
                 A6_p2 = -3.0 / 20.0, A6_p3 = 1.0 / 60.0;
constexpr double B6_m3 = 1.0 / 90.0, B6_m2 = -3.0 / 20.0, B6_m1 = 3.0 / 2.0, B6_0 = -49.0 / 18.0,
                 B6_p1 = 3.0 / 2.0, B6_p2 = -3.0 / 20.0, B6_p3 = 1.0 / 90.0;

template <int S> struct Reach;
template <> struct Reach<WH_FD2> { static constexpr int R = 1; };
template <> struct Reach<WH_FD4> { static constexpr int R = 2; };
template <> struct Reach<WH_FD4_TW> { static constexpr int R = 3; };
template <> struct Reach<WH_FD6> { static constexpr int R = 3; };

// first derivative; terms summed from the most negative offset up
template <int S, class F>
__device__ __forceinline__ double d1(const F &f, double inv)
{
    if constexpr (S == WH_FD2) {
        return (f(1) - f(-1)) * inv * 0.5;
    } else if constexpr (S == WH_FD4) {
        return (A4_m2 * f(-2) + A4_m1 * f(-1) + A4_p1 * f(1) + A4_p2 * f(2)) * inv;
    } else if constexpr (S == WH_FD4_TW) {
        return (TW_m3 * f(-3) + TW_m2 * f(-2) + TW_m1 * f(-1) + TW_p1 * f(1) + TW_p2 * f(2) +
                TW_p3 * f(3)) * inv;
    } else {
        return (A6_m3 * f(-3) + A6_m2 * f(-2) + A6_m1 * f(-1) + A6_p1 * f(1) + A6_p2 * f(2) +
                A6_p3 * f(3)) * inv;
    }
}

// first derivative of the product fa*fb (skew-symmetric form); terms (c*fa)*fb
template <int S, class F, class G>
__device__ __forceinline__ double d1p(const F &fa, const G &fb, double inv)
{
    if constexpr (S == WH_FD2) {
        return (fa(1) * fb(1) - fa(-1) * fb(-1)) * inv * 0.5;
    } else if constexpr (S == WH_FD4) {
        return (A4_m2 * fa(-2) * fb(-2) + A4_m1 * fa(-1) * fb(-1) + A4_p1 * fa(1) * fb(1) +
                A4_p2 * fa(2) * fb(2)) * inv;
    } else if constexpr (S == WH_FD4_TW) {
        return (TW_m3 * fa(-3) * fb(-3) + TW_m2 * fa(-2) * fb(-2) + TW_m1 * fa(-1) * fb(-1) +
                TW_p1 * fa(1) * fb(1) + TW_p2 * fa(2) * fb(2) + TW_p3 * fa(3) * fb(3)) * inv;
    } else {
        return (A6_m3 * fa(-3) * fb(-3) + A6_m2 * fa(-2) * fb(-2) + A6_m1 * fa(-1) * fb(-1) +
                A6_p1 * fa(1) * fb(1) + A6_p2 * fa(2) * fb(2) + A6_p3 * fa(3) * fb(3)) * inv;
    }
}

template <int S, class F>
__device__ __forceinline__ double d2(const F &f, double inv2)
{
    if constexpr (S == WH_FD2) {
        return (f(-1) - 2.0 * f(0) + f(1)) * inv2;
    } else if constexpr (S == WH_FD4 || S == WH_FD4_TW) {
        return (B4_m2 * f(-2) + B4_m1 * f(-1) + B4_0 * f(0) + B4_p1 * f(1) + B4_p2 * f(2)) * inv2;
    } else {
        return (B6_m3 * f(-3) + B6_m2 * f(-2) + B6_m1 * f(-1) + B6_0 * f(0) + B6_p1 * f(1) +
                B6_p2 * f(2) + B6_p3 * f(3)) * inv2;
    }
}

// a value that is the same in every lane, moved to scalar registers
__device__ __forceinline__ double wave_uniform(double v)
{
    union { double d; int i[2]; } x{v};
    x.i[0] = __builtin_amdgcn_readfirstlane(x.i[0]);
    x.i[1] = __builtin_amdgcn_readfirstlane(x.i[1]);
    return x.d;
}

// the mask components of a point, if it has any: in memory (components cs
// apart) or in registers
struct MaskMem {
    const double *p;
    ptrdiff_t cs;
    __device__ __forceinline__ bool on() const { return p != nullptr; }
    __device__ __forceinline__ double operator()(int i) const { return p[i * cs]; }
};
struct MaskReg {
    double v[6];
    bool has;
    __device__ __forceinline__ bool on() const { return has; }
    __device__ __forceinline__ double operator()(int i) const { return v[i]; }
};

// ACM right-hand side at one point (RHS_2D_acm / RHS_3D_acm).  A(c, d, o) is
// component c of the state at offset o along direction d from the point;
// mk: the point's mask (MaskMem or MaskReg).
// The components one after the other, so that few derivatives are live at
// once (3D FD4: 90 instead of 144 registers in the flat kernel, 147 instead of
// 201 in the z-marching one; 2D FD4 75 instead of 96).
template <int DIM, int S, bool SKEW, class ACC, class MASK>
__device__ __forceinline__ void acm_point(const ACC &A, const double *inv, const double *inv2, const AcmDev &a,
                                              const MASK &mk, double *r)
{
    double chi = 0.0, spo = 0.0;
    if (a.penal && mk.on()) {
        const int color = (int)mk(4);
        chi = mk(0) * (color == 0 ? 0.0 : a.Cinv);
    }
    if (a.sponge && mk.on()) spo = mk(5) * a.Csp_inv;
    double div = 0.0;
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        const double uc = A(c, 0, 0);
        double du[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) du[d] = d1<S>([&](int o) { return A(c, d, o); }, inv[d]);
        double lap = d2<S>([&](int o) { return A(c, 0, o); }, inv2[0]);
#pragma unroll
        for (int d = 1; d < DIM; ++d)
            lap = lap + d2<S>([&](int o) { return A(c, d, o); }, inv2[d]);
        double t;
        if constexpr (SKEW) {
            double sum = d1p<S>([&](int o) { return A(c, 0, o); },
                                [&](int o) { return A(0, 0, o); }, inv[0]);
#pragma unroll
            for (int d = 1; d < DIM; ++d)
                sum = sum + d1p<S>([&](int o) { return A(c, d, o); },
                                   [&](int o) { return A(d, d, o); }, inv[d]);
#pragma unroll
            for (int d = 0; d < DIM; ++d) sum = sum + A(d, 0, 0) * du[d];
            t = -(0.5 * sum);
        } else {
            t = -(A(0, 0, 0) * du[0]);
#pragma unroll
            for (int d = 1; d < DIM; ++d) t = t - A(d, 0, 0) * du[d];
        }
        t = t - d1<S>([&](int o) { return A(DIM, c, o); }, inv[c]);
        t = t + a.nu * lap;
        if (a.penal && mk.on()) t = t + (-(chi * (uc - mk(1 + c))));
        if (a.sponge && mk.on()) t = t - (uc - a.ums[c]) * spo;
        r[c] = t;
        div = c == 0 ? du[0] : div + du[c];
    }
    const double p = A(DIM, 0, 0);
    r[DIM] = -(a.c02 * div) - a.gamma_p * p;
    if (a.sponge && mk.on()) r[DIM] = r[DIM] - p * spo;
}

// accessor over one strided storage: base = component 0 of the point,
// components cs apart, strides s[d] along direction d
template <int DIM>
struct StridedAcc {
    const double *base;
    ptrdiff_t cs;
    ptrdiff_t s[3];
    __device__ __forceinline__ double operator()(int c, int d, int o) const
    {
        return base[c * cs + o * s[d]];
    }
};

// Workgroups are dispatched to the 8 XCDs (each with its own L2) round-robin:
// workgroup w runs on XCD w % 8.  The swizzle gives XCD x the consecutive
// logical indices [start(x), start(x) + count(x)), so the workgroups of one
// block share an L2 instead of being spread over all eight.  A permutation
// of [0, nw) for any nw.
__device__ __forceinline__ int xcd_swizzle(int w, int nw)
{
    constexpr int NX = 8;
    const int q = nw / NX, r = nw - q * NX, x = w % NX;
    return x * q + min(x, r) + w / NX;
}

// Runge-Kutta epilogue of the fused stage kernel.
//   mode 0 (first stage): u0 = input state; acc = u0 + (dt*b)*k; tout = u0 + (dt*a)*k
//   mode 1 (middle):      acc = acc + (dt*b)*k;  tout = u0 + (dt*a)*k
//   mode 2 (last):        sout = acc + (dt*b)*k
// b == 0 skips the acc term as the reference skips |coef| < 1e-8
// (runge_kutta_generic.f90:99,144).
// The accumulator lives only through one RK step and holds block interiors
// only: point p (x fastest) of component c of block b at b*NC*npts + c*npts
// + p, so its reads and writes cover whole cache lines.  u0, tout and sout
// are in the ghost-including block layout.
struct StageArgs {
    const double *u0;
    double *acc, *tout, *sout;
    const double *scal;
    const double *dtb;  // per active-list position dt (independent forests), or null
    double a, b;
    int mode, use_b, use_a;
    int full_rows;      // tout written in whole rows (stage_ghost_cols)
    // halo gather: the senders of each block's 4 (2D) or 6 faces by active
    // position (-1: own ghost nodes), or null
    const int32_t *gnb;
    // 3D z-marching kernel: the stage input / the next stage input hold block
    // interiors only, laid out as the accumulator
    int in_compact, out_compact;
};

struct NoEpilogue {};

// The arrays of one block of a fused stage: base pointers of block b (the
// same in every lane, so they stay in scalar registers); the epilogue
// addresses points by 32-bit offsets inside the block.
struct StageBlk {
    const double *u0;
    double *acc, *tout, *sout;
};

template <int NC>
__device__ __forceinline__ StageBlk stage_blk(const StageArgs &sa, int b, size_t blk, int npts)
{
    const size_t o = (size_t)b * blk;
    const size_t oc = (size_t)b * NC * npts;
    return StageBlk{sa.u0 ? sa.u0 + o : nullptr, sa.acc + oc, sa.tout ? sa.tout + (sa.out_compact ? oc : o) : nullptr,
                    sa.sout ? sa.sout + o : nullptr};
}

// point p of the interior (offset gi in the block, components cs apart)
template <int NC>
__device__ __forceinline__ void stage_epilogue(const StageArgs &sa, const StageBlk &B, int k, int gi, int cs, int p,
                                               int npts, const double *r, const double *ucen, ptrdiff_t ucs)
{
    const double dt = sa.dtb ? sa.dtb[k] : sa.scal[DS_DT];
    const double ca = dt * sa.a, cb = dt * sa.b;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = gi + c * cs, ia = p + c * npts;
        if (sa.mode == 0) {
            const double u0 = ucen[c * ucs];
            B.acc[ia] = sa.use_b ? u0 + cb * r[c] : u0;
            if (sa.use_a) B.tout[i] = u0 + ca * r[c];
        } else if (sa.mode == 1) {
            const double u0 = B.u0[i];
            if (sa.use_b) B.acc[ia] = B.acc[ia] + cb * r[c];
            if (sa.use_a) B.tout[i] = u0 + ca * r[c];
        } else {
            B.sout[i] = sa.use_b ? B.acc[ia] + cb * r[c] : B.acc[ia];
        }
    }
}

// the fused epilogue with the acc / u0 values of the point already loaded
// (accv, u0v: one value per component); with COMPACT the next stage input may
// be laid out as the accumulator
template <int NC, bool COMPACT = false>
__device__ __forceinline__ void stage_epilogue_pre(const StageArgs &sa, const StageBlk &B, int k, int gi, int cs,
                                                   int p, int npts, const double *r, const double *ucen,
                                                   ptrdiff_t ucs, const double *accv, const double *u0v)
{
    const int ti = COMPACT && sa.out_compact ? p : gi, tcs = COMPACT && sa.out_compact ? npts : cs;
    const double dt = sa.dtb ? sa.dtb[k] : sa.scal[DS_DT];
    const double ca = dt * sa.a, cb = dt * sa.b;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = gi + c * cs, ia = p + c * npts;
        if (sa.mode == 0) {
            const double u0 = ucen[c * ucs];
            B.acc[ia] = sa.use_b ? u0 + cb * r[c] : u0;
            if (sa.use_a) B.tout[ti + c * tcs] = u0 + ca * r[c];
        } else if (sa.mode == 1) {
            if (sa.use_b) B.acc[ia] = accv[c] + cb * r[c];
            if (sa.use_a) B.tout[ti + c * tcs] = u0v[c] + ca * r[c];
        } else {
            B.sout[i] = sa.use_b ? accv[c] + cb * r[c] : accv[c];
        }
    }
}

// Zeros in the ghost columns (x < g and x >= g + bs0) of one interior row of
// the next stage input, written by the threads of the row's first 2g points
// (where sa.full_rows: stages whose arrays exceed the last-level cache):
// with the interior written point by point, every cache line of the row is
// then written whole, so no line is merged with its old contents in memory.
// Before the next stage the ghost fill overwrites every ghost value its
// stencil reads (the stencils run along the axes, within g_rhs of the
// interior); the other ghost values of a stage input are not read.  row: the
// offset of the row's first (x = 0) element in the block.
template <int NC>
__device__ __forceinline__ void stage_ghost_cols(const StageArgs &sa, const StageBlk &B, int row, int cs, int ix,
                                                 int bs0, int g)
{
    if (!sa.full_rows || sa.mode == 2 || !sa.use_a) return;
    for (int x = ix; x < 2 * g; x += bs0) {
        const int i = row + (x < g ? x : bs0 + x);
#pragma unroll
        for (int c = 0; c < NC; ++c) B.tout[i + c * cs] = 0.0;
    }
}

// stage_ghost_cols for the rows [y0, y0 + ty0) of a 2D block, by the whole
// workgroup after its points (no per-point registers live meanwhile)
template <int NC>
__device__ __forceinline__ void stage_ghost_cols_2d(const StageArgs &sa, const StageBlk &B, const Geo &G, int y0,
                                                    int ty0)
{
    if (!sa.full_rows || sa.mode == 2 || !sa.use_a) return;
    const int w = 2 * G.g, cs = (int)G.cs;
    for (int i = threadIdx.x; i < ty0 * w; i += blockDim.x) {
        const int r = i / w, x = i - r * w;
        const int o = (G.g + y0 + r) * G.nx + (x < G.g ? x : G.bs0 + x);
#pragma unroll
        for (int c = 0; c < NC; ++c) B.tout[o + c * cs] = 0.0;
    }
}

// 2D: a slab of ty0 rows of one block per workgroup (a thread per point where
// the slab has no more points than threads), its points and the R layers
// around them staged in LDS -- the edges only: the stencils run along the
// axes.  Everything a thread's first point needs is requested before the tile
// barrier: its own value and one halo position (per component), the mask and
// the accumulator and u0 values of the fused stages.
// Bound by the launch for small grids (4.3 us for 256 blocks of 16^2, before
// 6.2; 4.3 for 64 of 32^2, before 14.9), by memory for large ones: 4096 blocks
// of 24^2 38.6 us = 7.1 TB/s from the cache-resident arrays with FD4 (before
// 74), 52 us with FD6 (102): one slab's loads are few enough to be in flight
// together, and no index is divided per tile element.
// rhs2d_slab is the work of one workgroup on the rows [y0, y0 + ty0) of block
// b (active position k), shared by the one-pool and the multi-pool kernel.
// mk: the mask of block b or null.  faces: the ids of the same-level
// neighbours (-x, +x, -y, +y) whose interior holds the values beyond the
// block's faces, or null (and -1) for the block's own ghost nodes.
template <int S, bool SKEW, bool FUSED>
__device__ __forceinline__ void rhs2d_slab(double *tile, const double *__restrict__ in, double *__restrict__ out,
                                           const double *__restrict__ mk, int b, int k, int y0, int ty0,
                                           const double *__restrict__ x0dx, const int32_t *__restrict__ faces,
                                           const Geo &G, const AcmDev &a, const StageArgs &sa)
{
    constexpr int R = Reach<S>::R;
    const int tx = G.bs0 + 2 * R, tcs = tx * (ty0 + 2 * R), cs = (int)G.cs;
    const int npts = G.bs0 * ty0, nall = G.bs0 * G.bs1, nt = (int)blockDim.x, tid = (int)threadIdx.x;
    const double *u = in + (size_t)b * G.blk;
    const StageBlk SB = FUSED ? stage_blk<3>(sa, b, G.blk, nall) : StageBlk{};
    const double dx0 = x0dx[6 * k + 3], dx1 = x0dx[6 * k + 4];
    // what to add to a place in the ghost nodes beyond face f to read it there
    auto face = [&](int f) -> ptrdiff_t {
        const int nb = faces ? faces[f] : -1;
        const int sh = f < 2 ? G.bs0 : G.bs1 * G.nx;
        return nb < 0 ? 0 : ((ptrdiff_t)nb - b) * (ptrdiff_t)G.blk + (f & 1 ? -sh : sh);
    };
    const ptrdiff_t fxm = face(0), fxp = face(1), fym = face(2), fyp = face(3);
    // halo position h of the slab: its place in the tile and where it is read
    const int nrow = 2 * R * G.bs0, nhalo = nrow + 2 * R * ty0;
    auto halo = [&](int h, int &l) -> const double * {
        int px, py;
        ptrdiff_t o;
        if (h < nrow) {  // rows below and above
            const int r = h / G.bs0;
            px = R + h - r * G.bs0;
            py = r < R ? r : ty0 + r;
            const int y = y0 - R + py;  // a slab of fewer than R rows reaches beyond the face from inside, too
            o = y < 0 ? fym : y >= G.bs1 ? fyp : 0;
        } else {  // columns left and right
            const int e = h - nrow, r = e / (2 * R), c = e - r * (2 * R);
            py = R + r;
            px = c < R ? c : G.bs0 + c;
            o = c < R ? fxm : fxp;
        }
        l = py * tx + px;
        return u + o + (ptrdiff_t)(G.g + y0 - R + py) * G.nx + (G.g - R + px);
    };
    const int iy0 = tid / G.bs0, ix0 = tid - iy0 * G.bs0;
    const int gi0 = (G.g + y0 + iy0) * G.nx + G.g + ix0;
    MaskReg mpre{};
    mpre.has = mk != nullptr;
    double upt[3] = {0, 0, 0}, hv[3] = {0, 0, 0}, apre[3] = {0, 0, 0}, upre[3] = {0, 0, 0};
    int hl = 0;
    if (tid < npts) {
#pragma unroll
        for (int c = 0; c < 3; ++c) upt[c] = u[c * cs + gi0];
    }
    if (tid < nhalo) {
        const double *h = halo(tid, hl);
#pragma unroll
        for (int c = 0; c < 3; ++c) hv[c] = h[c * cs];
    }
    if (tid < npts) {
        if (mk) {
#pragma unroll
            for (int c = 0; c < 6; ++c)
                if (c != 3) mpre.v[c] = mk[c * cs + gi0];  // component 3 (u_s,z) is 3D only
        }
        if (FUSED && sa.mode >= 1) {
            const int p = y0 * G.bs0 + tid;
#pragma unroll
            for (int c = 0; c < 3; ++c) apre[c] = SB.acc[c * nall + p];
            if (sa.mode == 1) {
#pragma unroll
                for (int c = 0; c < 3; ++c) upre[c] = SB.u0[c * cs + gi0];
            }
        }
    }
    const double inv[2] = {1.0 / dx0, 1.0 / dx1};
    const double inv2[2] = {1.0 / (dx0 * dx0), 1.0 / (dx1 * dx1)};
    if (tid < npts) {
        double *t = tile + (iy0 + R) * tx + ix0 + R;
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c * tcs] = upt[c];
    }
    if (tid < nhalo) {
#pragma unroll
        for (int c = 0; c < 3; ++c) tile[c * tcs + hl] = hv[c];
    }
    for (int p = tid + nt; p < npts; p += nt) {  // slabs with more points or halo than threads
        const int iy = p / G.bs0, ix = p - iy * G.bs0;
#pragma unroll
        for (int c = 0; c < 3; ++c)
            tile[c * tcs + (iy + R) * tx + ix + R] = u[c * cs + (G.g + y0 + iy) * G.nx + G.g + ix];
    }
    for (int h = tid + nt; h < nhalo; h += nt) {
        int l;
        const double *src = halo(h, l);
#pragma unroll
        for (int c = 0; c < 3; ++c) tile[c * tcs + l] = src[c * cs];
    }
    __syncthreads();
    auto point = [&](int iy, int ix, const auto &m, auto &&epilogue) {
        const double *uc = tile + (iy + R) * tx + (ix + R);
        const int gi = (G.g + y0 + iy) * G.nx + (G.g + ix);
        double r[3];
        const StridedAcc<2> A{uc, tcs, {1, tx, 0}};
        acm_point<2, S, SKEW>(A, inv, inv2, a, m, r);
        if constexpr (FUSED) {
            epilogue(gi, (y0 + iy) * G.bs0 + ix, r, uc);
        } else {
#pragma unroll
            for (int c = 0; c < 3; ++c) out[(size_t)b * G.blk + gi + c * cs] = r[c];
        }
    };
    if (tid < npts)
        point(iy0, ix0, mpre, [&](int gi, int p, const double *r, const double *uc) {
            stage_epilogue_pre<3>(sa, SB, k, gi, cs, p, nall, r, uc, tcs, apre, upre);
        });
    for (int pnt = tid + nt; pnt < npts; pnt += nt) {
        const int iy = pnt / G.bs0, ix = pnt - iy * G.bs0;
        const int gi0n = (G.g + y0 + iy) * G.nx + (G.g + ix);
        point(iy, ix, MaskMem{mk ? mk + gi0n : nullptr, cs}, [&](int gi, int p, const double *r, const double *uc) {
            stage_epilogue<3>(sa, SB, k, gi, cs, p, nall, r, uc, tcs);
        });
    }
    if constexpr (FUSED) stage_ghost_cols_2d<3>(sa, SB, G, y0, ty0);
}

template <int S, bool SKEW, bool FUSED>
__global__ __launch_bounds__(256) void k_rhs2d(const double *__restrict__ in, double *__restrict__ out,
                                               const double *__restrict__ mask,
                                               const int32_t *__restrict__ act,
                                               const double *__restrict__ x0dx, Geo G, AcmDev a,
                                               StageArgs sa, int ysplit, int ty0)
{
    extern __shared__ double tile[];
    const int wg = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int k = wg / ysplit, y0 = (wg - k * ysplit) * ty0;
    const int b = act[k];
    const double *mk = mask ? mask + (G.mask_per_block ? (size_t)b * G.mblk : 0) : nullptr;
    rhs2d_slab<S, SKEW, FUSED>(tile, in, out, mk, b, k, y0, min(ty0, G.bs1 - y0), x0dx,
                               FUSED && sa.gnb ? sa.gnb + (size_t)k * 4 : nullptr, G, a, sa);
}

// ---------------------------------------------------------------------------
// Several pools in one launch (independent forests of a batch, any block
// size): item k of the launch is a part (2D: one of nslab slabs, 3D: the
// whole) of the block at position (k - ent0) / nslab of the active list of
// the pool whose item range holds k (pools[] in item order), with that
// position's origin/spacing and block group g = goff + grp[..] (dt dtg[g],
// constants gacm[g]), all read from the pool's own device tables; once per
// step k_entries resolves every item into a record (MEnt) that the stage
// kernels read with one load.  The
// stage's input and output arrays are selected per pool from arr[]:
// 0 hvy_block, 1 work slot 0 (the RK accumulator), 2 / 3 work slots 1 / 2.
// The kernels are persistent (grid-stride over the items, their count read
// from device memory), so one captured launch serves any number of blocks.
// ---------------------------------------------------------------------------
// the last pool whose first entry (s < 0), first chunk of sync stage s (0..2) or
// first patch of sync stage s - 3 (3..5) is <= x
__device__ __forceinline__ int pool_of(const MPoolDev *__restrict__ pools, int npools, int64_t x, int s)
{
    int lo = 0, hi = npools - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        const int64_t first = s < 0 ? (int64_t)pools[mid].ent0 : s < 3 ? pools[mid].s0[s] : pools[mid].q0[s - 3];
        if (first <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ StageArgs multi_stage_args(const MPoolDev &P, const MStage &st, const double *dtp)
{
    StageArgs sa{};
    sa.u0 = P.arr[0];
    sa.acc = P.arr[1];
    sa.tout = P.arr[st.out_sel];
    sa.sout = P.arr[st.sout_sel];
    sa.dtb = dtp;  // the entry's dt at index 0
    sa.a = st.a;
    sa.b = st.b;
    sa.mode = st.mode;
    sa.use_a = st.use_a;
    sa.use_b = st.use_b;
    sa.full_rows = st.full_rows;
    return sa;
}

// the item records of a launch: one thread per item
__global__ __launch_bounds__(256) void k_entries(const MPoolDev *__restrict__ pools, int npools,
                                                 const int64_t *__restrict__ tot, MEnt *__restrict__ ents)
{
    const int n = (int)tot[0];
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int p = pool_of(pools, npools, k, -1);
        const MPoolDev &P = pools[p];
        const int j = (k - P.ent0) / P.nslab, y0 = (k - P.ent0 - j * P.nslab) * P.ty0;
        ents[k] = MEnt{p, P.act[j], P.goff + P.grp[j], j, y0, min(P.ty0, P.G.bs1 - y0)};
    }
}

// an item's record with every field wave-uniform, so that the descriptor and
// the group's constants are read through scalar loads
__device__ __forceinline__ MEnt uniform(const MEnt &e)
{
    return MEnt{__builtin_amdgcn_readfirstlane(e.pool), __builtin_amdgcn_readfirstlane(e.b),
                __builtin_amdgcn_readfirstlane(e.g),    __builtin_amdgcn_readfirstlane(e.j),
                __builtin_amdgcn_readfirstlane(e.y0),   __builtin_amdgcn_readfirstlane(e.ty0)};
}

// 2D: items are slabs (slab_rows) of the pools' blocks; the next item's record
// is requested while an item is worked on.
template <int S, bool SKEW>
__global__ __launch_bounds__(256) void k_rhs2d_multi(const MPoolDev *__restrict__ pools,
                                                     const MEnt *__restrict__ ents, const double *__restrict__ dtg,
                                                     const AcmDev *__restrict__ gacm,
                                                     const int64_t *__restrict__ tot, MStage st)
{
    extern __shared__ double tile[];
    const int nent = (int)tot[0];
    int k = blockIdx.x;
    if (k >= nent) return;
    MEnt next = ents[k];
    for (; k < nent; k += gridDim.x) {
        const MEnt e = uniform(next);
        next = ents[min(k + (int)gridDim.x, nent - 1)];
        const MPoolDev &P = pools[e.pool];
        const int b = e.b, g = e.g;
        const Geo &G = P.G;
        const AcmDev &a = gacm[g];
        const StageArgs sa = multi_stage_args(P, st, dtg + g);
        const double *mk = P.mask ? P.mask + (G.mask_per_block ? (size_t)b * G.mblk : 0) : nullptr;
        rhs2d_slab<S, SKEW, true>(tile, P.arr[st.in_sel], nullptr, mk, b, 0, e.y0, e.ty0, P.x0dx + 6 * (size_t)e.j,
                                  nullptr, G, a, sa);
        __syncthreads();  // the tile is reused by the next item
    }
}

// 3D: 256 interior points per workgroup, stencil reads served by L1/L2;
// XCD: workgroup indices swizzled so that a block's workgroups share an L2.
template <int S, bool SKEW, bool FUSED, bool XCD>
__global__ __launch_bounds__(256) void k_rhs3d(const double *__restrict__ in, double *__restrict__ out,
                                               const double *__restrict__ mask,
                                               const int32_t *__restrict__ act,
                                               const double *__restrict__ x0dx, Geo G, AcmDev a,
                                               StageArgs sa)
{
    const int npts = G.bs0 * G.bs1 * G.bs2;
    const int nchunk = (npts + 255) / 256;
    const int wg = XCD ? xcd_swizzle((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
    const int k = wg / nchunk;
    const int pnt = (wg - k * nchunk) * 256 + threadIdx.x;
    if (pnt >= npts) return;
    const int b = act[k];
    const int ix = pnt % G.bs0, iy = (pnt / G.bs0) % G.bs1, iz = pnt / (G.bs0 * G.bs1);
    const double dx0 = x0dx[6 * k + 3], dx1 = x0dx[6 * k + 4], dx2 = x0dx[6 * k + 5];
    const double inv[3] = {1.0 / dx0, 1.0 / dx1, 1.0 / dx2};
    const double inv2[3] = {1.0 / (dx0 * dx0), 1.0 / (dx1 * dx1), 1.0 / (dx2 * dx2)};
    const size_t gi = ((size_t)(G.g + iz) * G.ny + (G.g + iy)) * G.nx + (G.g + ix);
    const double *uc = in + (size_t)b * G.blk + gi;
    const double *mk = mask ? mask + (G.mask_per_block ? (size_t)b * G.mblk : 0) + gi : nullptr;
    double r[4];
    const StridedAcc<3> A{uc, (ptrdiff_t)G.cs, {1, G.nx, (ptrdiff_t)G.nx * G.ny}};
    acm_point<3, S, SKEW>(A, inv, inv2, a, MaskMem{mk, (ptrdiff_t)G.cs}, r);
    const size_t o = (size_t)b * G.blk + gi;
    if constexpr (FUSED) {
        const StageBlk SB = stage_blk<4>(sa, b, G.blk, npts);
        stage_epilogue<4>(sa, SB, k, (int)gi, (int)G.cs, pnt, npts, r, uc, G.cs);
        stage_ghost_cols<4>(sa, SB, (int)gi - (G.g + ix), (int)G.cs, ix, G.bs0, G.g);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) out[o + c * G.cs] = r[c];
    }
}

// 3D, several pools in one launch (same arithmetic per point as k_rhs3d):
// work item t = (entry, chunk of 256 points), nchunk chunks per entry (the
// largest block of the launch; points past a smaller block's end idle);
// persistent over the items, their count nent * nchunk from device memory.
// With XCD the item index is swizzled so that a block's chunks run on one
// XCD (the grid is a multiple of 8, so item t runs on XCD t % 8).
template <int S, bool SKEW, bool XCD>
__global__ __launch_bounds__(256) void k_rhs3d_multi(const MPoolDev *__restrict__ pools,
                                                     const MEnt *__restrict__ ents,
                                                     const double *__restrict__ dtg,
                                                     const AcmDev *__restrict__ gacm,
                                                     const int64_t *__restrict__ tot, MStage st, int nchunk)
{
    const int total = (int)tot[0] * nchunk;
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        const int w = XCD ? xcd_swizzle(t, total) : t;
        const int k = w / nchunk;
        const int pnt = (w - k * nchunk) * 256 + threadIdx.x;
        const MEnt e = uniform(ents[k]);
        const MPoolDev &P = pools[e.pool];
        const Geo &G = P.G;
        const int npts = G.bs0 * G.bs1 * G.bs2;
        if (pnt >= npts) continue;
        const int j = e.j, b = e.b, g = e.g;
        const AcmDev &a = gacm[g];
        const StageArgs sa = multi_stage_args(P, st, dtg + g);
        const double *xd = P.x0dx + 6 * (size_t)j;
        const int ix = pnt % G.bs0, iy = (pnt / G.bs0) % G.bs1, iz = pnt / (G.bs0 * G.bs1);
        const double dx0 = xd[3], dx1 = xd[4], dx2 = xd[5];
        const double inv[3] = {1.0 / dx0, 1.0 / dx1, 1.0 / dx2};
        const double inv2[3] = {1.0 / (dx0 * dx0), 1.0 / (dx1 * dx1), 1.0 / (dx2 * dx2)};
        const size_t gi = ((size_t)(G.g + iz) * G.ny + (G.g + iy)) * G.nx + (G.g + ix);
        const double *uc = P.arr[st.in_sel] + (size_t)b * G.blk + gi;
        const double *mk = P.mask ? P.mask + (G.mask_per_block ? (size_t)b * G.mblk : 0) + gi : nullptr;
        double r[4];
        const StridedAcc<3> A{uc, (ptrdiff_t)G.cs, {1, G.nx, (ptrdiff_t)G.nx * G.ny}};
        acm_point<3, S, SKEW>(A, inv, inv2, a, MaskMem{mk, (ptrdiff_t)G.cs}, r);
        const StageBlk SB = stage_blk<4>(sa, b, G.blk, npts);
        stage_epilogue<4>(sa, SB, 0, (int)gi, (int)G.cs, pnt, npts, r, uc, G.cs);
        stage_ghost_cols<4>(sa, SB, (int)gi - (G.g + ix), (int)G.cs, ix, G.bs0, G.g);
    }
}

// 3D, z-marching: a workgroup owns a slab of ty0 rows of (x, y) columns of
// one block (ysplit workgroups per block, one thread per column) and marches
// through z.  The x/y stencils read an LDS copy of the current z-plane slab
// (interior from the threads' registers, the R-wide x/y ring from global
// memory); the z stencil reads a per-thread register queue of 2R+1 planes.
// Everything the next plane needs -- the queue's new plane, the ring, the
// accumulator and u0 values of the epilogue -- is requested before the
// current plane is computed, so a plane's memory latency runs under the
// previous plane's arithmetic.  Two LDS planes (nbuf 2) leave one barrier per
// plane; one plane (nbuf 1, slabs too wide for two) needs a second one.
// Every input value is read from memory once (plus the slab ring), except
// that with zsplit > 1 the z range of a block is cut into zsplit pieces,
// each with its own workgroups, which read the 2R planes around their cut.
// Halo: with sa.gnb the values beyond a face of the block come from the
// interior of the same-level neighbour there (6 ids per block: -x, +x, -y,
// +y, -z, +z), or from the block's own ghost nodes where the id is -1;
// without it always from the ghost nodes.  The stencils run along the axes,
// so edges and corners are not read.
// Bound by the memory system: over 4096 24^3 blocks (FD4, g 6, the stages of
// RK4) 2.26 ms a launch for 9.2 GB = 4.1 TB/s (before: 4.34 ms, and 3.30 ms by
// the flat kernel); with the stage inputs held without ghost nodes, in rows
// that fill cache lines, 1.92 ms = 4.8 TB/s, where a large copy reaches 4.4.
// Over 512 blocks 0.29 and 0.25 ms (0.56, 0.42).
template <int S, bool SKEW, bool FUSED>
__global__ __launch_bounds__(512) void k_rhs3d_zm(const double *__restrict__ in,
                                                  double *__restrict__ out,
                                                  const double *__restrict__ mask,
                                                  const int32_t *__restrict__ act,
                                                  const double *__restrict__ x0dx, Geo G, AcmDev a,
                                                  StageArgs sa, int ysplit, int zsplit, int nbuf)
{
    constexpr int R = Reach<S>::R;
    constexpr int W = 2 * R + 1;
    extern __shared__ double planes[];
    const int per_block = ysplit * zsplit;
    const int wg = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int k = wg / per_block;
    const int rem = wg - k * per_block;
    const int zpart = rem / ysplit, part = rem - zpart * ysplit;
    const int tz0 = G.bs2 / zsplit, z0 = zpart * tz0, z1 = z0 + tz0;
    const int b = act[k];
    const int ty0 = G.bs1 / ysplit;
    const int y0 = part * ty0;
    const int tid = threadIdx.x;
    const int iyl = tid / G.bs0, ix = tid - iyl * G.bs0, iy = y0 + iyl;
    const int tx = G.bs0 + 2 * R, ty = ty0 + 2 * R, tcs = tx * ty;
    const int zs = G.nx * G.ny, cs = (int)G.cs, npts = G.bs0 * G.bs1 * G.bs2;
    // the input's layout: ghost-including blocks, or interiors only
    const bool ci = FUSED && sa.in_compact;
    const int ig = ci ? 0 : G.g, inx = ci ? G.bs0 : G.nx, izs = ci ? G.bs0 * G.bs1 : zs, ics = ci ? npts : cs;
    const size_t iblk = ci ? (size_t)4 * npts : G.blk;
    const double *u = in + (size_t)b * iblk;
    // where the values beyond each face are read, relative to their place in
    // this block's ghost nodes
    ptrdiff_t fo[6] = {0, 0, 0, 0, 0, 0};
    if (FUSED && sa.gnb) {
        const int32_t *nb = sa.gnb + (size_t)k * 6;
        const ptrdiff_t sh[3] = {G.bs0, (ptrdiff_t)G.bs1 * inx, (ptrdiff_t)G.bs2 * izs};
#pragma unroll
        for (int f = 0; f < 6; ++f)
            if (nb[f] >= 0) fo[f] = ((ptrdiff_t)nb[f] - b) * (ptrdiff_t)iblk + (f & 1 ? -sh[f >> 1] : sh[f >> 1]);
    }
    const int col = (G.g + iy) * G.nx + (G.g + ix), icol = (ig + iy) * inx + (ig + ix);
    const double dx0 = x0dx[6 * k + 3], dx1 = x0dx[6 * k + 4], dx2 = x0dx[6 * k + 5];
    const double inv[3] = {wave_uniform(1.0 / dx0), wave_uniform(1.0 / dx1), wave_uniform(1.0 / dx2)};
    const double inv2[3] = {wave_uniform(1.0 / (dx0 * dx0)), wave_uniform(1.0 / (dx1 * dx1)),
                            wave_uniform(1.0 / (dx2 * dx2))};
    const double *mk = mask ? mask + (G.mask_per_block ? (size_t)b * G.mblk : 0) : nullptr;

    // thread h holds position h of the slab's x/y ring (without corners; the
    // host checks that there are no more positions than threads)
    const bool ringer = tid < 2 * R * (G.bs0 + ty0);
    int r_lds = 0;
    const double *r_src = u;
    if (ringer) {
        int px, py;
        ptrdiff_t o = 0;
        if (tid < 2 * R * G.bs0) {  // rows below and above the slab
            py = iyl < R ? iyl : ty0 + iyl;
            px = R + ix;
            if (iyl < R && part == 0) o = fo[2];
            if (iyl >= R && part == ysplit - 1) o = fo[3];
        } else {  // columns left and right
            const int e = tid - 2 * R * G.bs0, kk = e % (2 * R);
            py = R + e / (2 * R);
            px = kk < R ? kk : G.bs0 + kk;
            o = kk < R ? fo[0] : fo[1];
        }
        r_lds = py * tx + px;
        r_src = u + o + (ptrdiff_t)(ig + y0 - R + py) * inx + (ig - R + px);
    }
    // the slab's own points of plane iz (-R .. Bs2 + R - 1), component c
    auto own = [&](int iz, int c) -> double {
        const double *p = u + (iz < 0 ? fo[4] : iz >= G.bs2 ? fo[5] : (ptrdiff_t)0);
        return p[c * ics + (ig + iz) * izs + icol];
    };
    const StageBlk SB = FUSED ? stage_blk<4>(sa, b, G.blk, npts) : StageBlk{};
    double apre[4] = {0, 0, 0, 0}, upre[4] = {0, 0, 0, 0};
    double q[4][W];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 2 * R; ++j) q[c][j] = own(z0 - R + j, c);
    double nq[4], nr[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) nq[c] = own(z0 + R, c);
    if (ringer)
#pragma unroll
        for (int c = 0; c < 4; ++c) nr[c] = r_src[c * ics + (ig + z0) * izs];

    const int lc = (iyl + R) * tx + (ix + R);
    for (int iz = z0; iz < z1; ++iz) {
        double *plane = planes + (nbuf == 2 && ((iz - z0) & 1) ? 4 * tcs : 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            q[c][2 * R] = nq[c];
            plane[c * tcs + lc] = q[c][R];
        }
        if (ringer)
#pragma unroll
            for (int c = 0; c < 4; ++c) plane[c * tcs + r_lds] = nr[c];
        const int gi = (G.g + iz) * zs + col, pnt = (iz * G.bs1 + iy) * G.bs0 + ix;
        if constexpr (FUSED) {  // the epilogue's operands
            if (sa.mode >= 1) {
#pragma unroll
                for (int c = 0; c < 4; ++c) apre[c] = SB.acc[c * npts + pnt];
            }
            if (sa.mode == 1) {
#pragma unroll
                for (int c = 0; c < 4; ++c) upre[c] = SB.u0[c * cs + gi];
            }
        }
        if (iz + 1 < z1) {  // the next plane's values
#pragma unroll
            for (int c = 0; c < 4; ++c) nq[c] = own(iz + 1 + R, c);
            if (ringer)
#pragma unroll
                for (int c = 0; c < 4; ++c) nr[c] = r_src[c * ics + (ig + iz + 1) * izs];
        }
        __syncthreads();
        // x/y from the LDS plane, z from the register queue
        const auto A = [&](int c, int d, int o) -> double {
            if (d == 2 || o == 0) return q[c][R + (d == 2 ? o : 0)];
            return plane[c * tcs + lc + o * (d == 0 ? 1 : tx)];
        };
        double r[4];
        acm_point<3, S, SKEW>(A, inv, inv2, a, MaskMem{mk ? mk + gi : nullptr, (ptrdiff_t)G.cs}, r);
        if constexpr (FUSED) {
            const double u0c[4] = {q[0][R], q[1][R], q[2][R], q[3][R]};
            stage_epilogue_pre<4, true>(sa, SB, k, gi, cs, pnt, npts, r, u0c, 1, apre, upre);
            if (!sa.out_compact) stage_ghost_cols<4>(sa, SB, gi - (G.g + ix), cs, ix, G.bs0, G.g);
        } else {
            double *o = out + (size_t)b * G.blk + gi;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c * cs] = r[c];
        }
        if (nbuf == 1) __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < 2 * R; ++j) q[c][j] = q[c][j + 1];
    }
}

int reach_of(int scheme)
{
    return scheme == WH_FD2 ? 1 : scheme == WH_FD4 ? 2 : 3;
}

// Is the z-marching kernel usable with this z-split?  It divides Bs2, and
// each piece has at least 2R planes.
bool zm_zvalid(int bs2, int scheme, int zs)
{
    return zs >= 1 && bs2 % zs == 0 && bs2 / zs >= 2 * reach_of(scheme);
}

// Is the z-marching kernel usable with this y-split?  Threads per workgroup
// in [64, 512], the slab ring fits the per-thread ring registers, LDS <= 64 KB.
bool zm_valid(int bs0, int bs1, int scheme, int ys)
{
    if (ys < 1 || bs1 % ys) return false;
    const int R = reach_of(scheme), ty0 = bs1 / ys, nthr = bs0 * ty0;
    if (nthr < 64 || nthr > 512) return false;
    if (2 * R * (bs0 + ty0) > nthr) return false;
    return sizeof(double) * 4 * (bs0 + 2 * R) * (ty0 + 2 * R) <= 64 * 1024;
}

// the 2D stages take blocks whose whole tile would fit a compute unit's LDS (the
// slabs need less of it; what was refused before them still is)
bool tile2d_ok(int bs0, int bs1, int R)
{
    return sizeof(double) * 3 * (bs0 + 2 * R) * (bs1 + 2 * R) <= 160 * 1024;
}

// Rows of a 2D slab: as many as give at most 256 points, a thread each, and
// slabs of about equal size.  Launch times of a fused FD4 stage by the number
// of slabs a block is cut into: 64 blocks of 32^2 (skew-symmetric) 9.6 / 6.1 /
// 4.3 / 4.7 us in 1 / 2 / 4 / 6, 4096 of 24^2 46 / 47 / 39 / 44 us in 1 / 2 /
// 3 / 4, 1024 of 48^2 58 / 45 / 41 / 39 us in 1 / 2 / 4 / 6; 16^2 whole 4.3 us
// for 256 blocks, in 2 slabs 4.6.
int slab_rows(int bs0, int bs1)
{
    const int most = std::max(1, 256 / bs0), ys = (bs1 + most - 1) / most;
    return (bs1 + ys - 1) / ys;
}

// y-split of the 3D stage kernel: the pool's tuned value, or of the valid
// splits (zm_valid: up to 512 threads) the one that gives most lanes of a
// compute unit a column, reckoned as 12 resident wavefronts (3 per SIMD; the
// widest stencils' registers leave 2) that hold whole workgroups only, the widest
// slab among equals; 0 selects the flat kernel.  24x24 with FD4: 3 slabs of
// 192 threads, 4 workgroups of 3 wavefronts, 768 lanes, against 2 slabs of 288,
// 2 workgroups of 5, 576.
static int zm_split(const wh_pool *P, const Geo &G, int scheme)
{
    if (P->k3d_ysplit == 0) return 0;
    if (P->k3d_ysplit > 0 && zm_valid(G.bs0, G.bs1, scheme, P->k3d_ysplit)) return P->k3d_ysplit;
    int best = 0, most = 0;
    for (int ys = 1; ys <= 8; ++ys) {
        if (!zm_valid(G.bs0, G.bs1, scheme, ys)) continue;
        const int nthr = G.bs0 * (G.bs1 / ys), waves = (nthr + 63) / 64, lanes = 12 / waves * nthr;
        if (lanes > most) {
            best = ys;
            most = lanes;
        }
    }
    return best;
}

// z-split: the pool's tuned value where it is valid.  With the automatic
// y-split and no z-split asked for: the FD2 / FD4 stencils without the
// skew-symmetric products take the largest valid one up to 8 -- short
// marches even out the last round of workgroups (24^3 blocks, y-split 3:
// 2335 / 2294 / 2259 us in 1 / 3 / 6 pieces over 4096 blocks, 322 / 300 /
// 291 us over 512; 20x16x18 over 64 blocks 46 / 20 us in 1 / 3).  The others
// pay more for the planes read twice (512 blocks: FD6 318 / 330 us in 1 / 2,
// skew-symmetric FD4 301 / 306 us): the smallest split that gives every
// compute unit 4 workgroups, else the largest (skew-symmetric FD6, 64 blocks:
// 67 / 48 / 44 us in 1 / 2 / 4).
static int zm_zsplit(const wh_pool *P, const Geo &G, const AcmDev &a, int nwg)
{
    if (P->k3d_ysplit >= 0 || P->k3d_zsplit != 1)
        return zm_zvalid(G.bs2, a.scheme, P->k3d_zsplit) ? P->k3d_zsplit : 1;
    const bool fill_only = a.skew || reach_of(a.scheme) > 2;
    int best = 1;
    for (int zs = 1; zs <= 8; ++zs) {
        if (!zm_zvalid(G.bs2, a.scheme, zs)) continue;
        best = zs;
        if (fill_only && (long)nwg * zs >= 4L * P->n_cu) break;
    }
    return best;
}

bool stage_gathers(const wh_pool *P, int scheme) { return P->d.dim == 3 && zm_split(P, make_geo(P), scheme) > 0; }

Geo make_geo(const wh_pool *P)
{
    Geo G;
    G.bs0 = P->d.bs[0];
    G.bs1 = P->d.bs[1];
    G.bs2 = P->d.dim == 3 ? P->d.bs[2] : 1;
    G.g = P->d.g;
    G.nx = P->nx;
    G.ny = P->ny;
    G.blk = P->blk;
    G.cs = P->cs;
    G.mblk = P->mblk;
    G.mask_per_block = P->d.mask_per_block;
    return G;
}

template <bool FUSED>
static int dispatch_rhs(wh_pool *P, const AcmDev &a, const double *in, double *out,
                        const int32_t *act, const double *x0dx, int nact, const StageArgs &sa)
{
    if (nact <= 0) return WH_OK;
    const Geo G = make_geo(P);
    const double *mask = (P->mask && (a.penal || a.sponge)) ? P->mask : nullptr;
    if (P->d.dim == 2) {
        const int R = reach_of(a.scheme);
        const int ty0 = slab_rows(G.bs0, G.bs1), ys = (G.bs1 + ty0 - 1) / ty0;
        const size_t lds = sizeof(double) * 3 * (G.bs0 + 2 * R) * (ty0 + 2 * R);
        WH_CHECK(tile2d_ok(G.bs0, G.bs1, R), WH_E_ARG, "2D block tile exceeds LDS");
        const dim3 grid(nact * ys), blockd(std::min(256, (G.bs0 * ty0 + 63) / 64 * 64));
#define L2D(SC, SK)                                                                                             \
    hipLaunchKernelGGL((k_rhs2d<SC, SK, FUSED>), grid, blockd, lds, P->stream, in, out, mask, act, x0dx, G, a, sa, \
                       ys, ty0)
        switch (a.scheme * 2 + a.skew) {
        case WH_FD2 * 2: L2D(WH_FD2, false); break;
        case WH_FD2 * 2 + 1: L2D(WH_FD2, true); break;
        case WH_FD4 * 2: L2D(WH_FD4, false); break;
        case WH_FD4 * 2 + 1: L2D(WH_FD4, true); break;
        case WH_FD4_TW * 2: L2D(WH_FD4_TW, false); break;
        case WH_FD4_TW * 2 + 1: L2D(WH_FD4_TW, true); break;
        case WH_FD6 * 2: L2D(WH_FD6, false); break;
        case WH_FD6 * 2 + 1: L2D(WH_FD6, true); break;
        default: set_error("unknown scheme"); return WH_E_ARG;
        }
#undef L2D
    } else if (const int ys = zm_split(P, G, a.scheme); ys > 0) {
        const int R = reach_of(a.scheme);
        const int zs = zm_zsplit(P, G, a, nact * ys);
        const size_t plane = sizeof(double) * 4 * (G.bs0 + 2 * R) * (G.bs1 / ys + 2 * R);
        const int nbuf = 2 * plane <= 64 * 1024 ? 2 : 1;
        const size_t lds = nbuf * plane;
        dim3 grid(nact * ys * zs), blockd(G.bs0 * (G.bs1 / ys));
#define L3D(SC, SK)                                                                                      \
    hipLaunchKernelGGL((k_rhs3d_zm<SC, SK, FUSED>), grid, blockd, lds, P->stream, in, out, mask, act, x0dx, G, \
                       a, sa, ys, zs, nbuf)
        switch (a.scheme * 2 + a.skew) {
        case WH_FD2 * 2: L3D(WH_FD2, false); break;
        case WH_FD2 * 2 + 1: L3D(WH_FD2, true); break;
        case WH_FD4 * 2: L3D(WH_FD4, false); break;
        case WH_FD4 * 2 + 1: L3D(WH_FD4, true); break;
        case WH_FD4_TW * 2: L3D(WH_FD4_TW, false); break;
        case WH_FD4_TW * 2 + 1: L3D(WH_FD4_TW, true); break;
        case WH_FD6 * 2: L3D(WH_FD6, false); break;
        case WH_FD6 * 2 + 1: L3D(WH_FD6, true); break;
        default: set_error("unknown scheme"); return WH_E_ARG;
        }
#undef L3D
    } else {
        const int npts = G.bs0 * G.bs1 * G.bs2;
        dim3 grid(nact * ((npts + 255) / 256)), blockd(256);
#define L3D(SC, SK)                                                                                          \
    do {                                                                                                     \
        if (P->k3d_xcd)                                                                                      \
            hipLaunchKernelGGL((k_rhs3d<SC, SK, FUSED, true>), grid, blockd, 0, P->stream, in, out, mask, act, \
                               x0dx, G, a, sa);                                                              \
        else                                                                                                 \
            hipLaunchKernelGGL((k_rhs3d<SC, SK, FUSED, false>), grid, blockd, 0, P->stream, in, out, mask, act, \
                               x0dx, G, a, sa);                                                              \
    } while (0)
        switch (a.scheme * 2 + a.skew) {
        case WH_FD2 * 2: L3D(WH_FD2, false); break;
        case WH_FD2 * 2 + 1: L3D(WH_FD2, true); break;
        case WH_FD4 * 2: L3D(WH_FD4, false); break;
        case WH_FD4 * 2 + 1: L3D(WH_FD4, true); break;
        case WH_FD4_TW * 2: L3D(WH_FD4_TW, false); break;
        case WH_FD4_TW * 2 + 1: L3D(WH_FD4_TW, true); break;
        case WH_FD6 * 2: L3D(WH_FD6, false); break;
        case WH_FD6 * 2 + 1: L3D(WH_FD6, true); break;
        default: set_error("unknown scheme"); return WH_E_ARG;
        }
#undef L3D
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_rhs(wh_pool *P, const AcmDev &a, const double *in, double *out, const int32_t *act,
               const double *x0dx, int nact)
{
    StageArgs sa{};
    return dispatch_rhs<false>(P, a, in, out, act, x0dx, nact, sa);
}

int launch_fused_stage(wh_pool *P, const AcmDev &a, const double *tin, double *tout,
                       const double *u0, double *acc, double *sout, int mode, double acoef,
                       double bcoef, const double *dtb, const int32_t *gnb, bool in_compact, bool out_compact)
{
    StageArgs sa{};
    sa.gnb = gnb;
    sa.in_compact = in_compact;
    sa.out_compact = out_compact;
    sa.dtb = dtb;
    sa.u0 = u0;
    sa.acc = acc;
    sa.tout = tout;
    sa.sout = sout;
    sa.scal = P->scal;
    sa.a = acoef;
    sa.b = bcoef;
    sa.mode = mode;
    sa.use_a = std::abs(acoef) >= 1.0e-8;
    sa.use_b = std::abs(bcoef) >= 1.0e-8;
    sa.full_rows = stage_full_rows(P->nact, sizeof(double) * (double)make_geo(P).blk);
    return dispatch_rhs<true>(P, a, tin, nullptr, P->d_active, P->d_x0dx, P->nact, sa);
}


// Interpolating prediction (module_wavelets.f90:96-284, `prediction`) at one
// point of the refined grid.  f[d] is the point's index in the doubled
// ghost-inclusive index space of the coarse block u (coarse point c sits at
// fine index 2c).  Even indices copy, odd ones interpolate with the centred
// stencil of `order` (2: (1,1)/2, 4: (-1,9,9,-1)/16, 6: (3,-25,150,150,-25,3)/256)
// separably, x innermost, then y, then z, each sum left to right -- the
// reference's separable passes evaluated at one point.
template <int N>
__device__ __forceinline__ double pred_point(const double *__restrict__ u, int nx, int ny,
                                             int dim, const int f[3])
{
    constexpr double c2[2] = {0.5, 0.5};
    constexpr double c4[4] = {-1.0 / 16.0, 9.0 / 16.0, 9.0 / 16.0, -1.0 / 16.0};
    constexpr double c6[6] = {3.0 / 256.0, -25.0 / 256.0, 150.0 / 256.0,
                              150.0 / 256.0, -25.0 / 256.0, 3.0 / 256.0};
    const double *cf = (N == 1) ? c2 : (N == 2) ? c4 : c6;
    const int cx = f[0] >> 1, px = f[0] & 1;
    const int cy = f[1] >> 1, py = f[1] & 1;
    const int cz = dim == 3 ? f[2] >> 1 : 0, pz = dim == 3 ? (f[2] & 1) : 0;
    auto vx = [&](int jy, int kz) -> double {
        const double *row = u + ((size_t)kz * ny + jy) * nx;
        if (!px) return row[cx];
        double s = cf[0] * row[cx - N + 1];
#pragma unroll
        for (int t = 1; t < 2 * N; ++t) s = s + cf[t] * row[cx - N + 1 + t];
        return s;
    };
    auto vy = [&](int kz) -> double {
        if (!py) return vx(cy, kz);
        double s = cf[0] * vx(cy - N + 1, kz);
#pragma unroll
        for (int t = 1; t < 2 * N; ++t) s = s + cf[t] * vx(cy - N + 1 + t, kz);
        return s;
    };
    if (!pz) return vy(cz);
    double s = cf[0] * vy(cz - N + 1);
#pragma unroll
    for (int t = 1; t < 2 * N; ++t) s = s + cf[t] * vy(cz - N + 1 + t);
    return s;
}

__device__ __forceinline__ double pred_any(const double *u, int nx, int ny, int dim, const int f[3],
                                           int order)
{
    if (order == 4) return pred_point<2>(u, nx, ny, dim, f);
    if (order == 2) return pred_point<1>(u, nx, ny, dim, f);
    return pred_point<3>(u, nx, ny, dim, f);
}

// The points [r0, r_end) of one ghost patch (x fastest), taken by the 64
// lanes of a wavefront in steps of 64 (lane l starts at r0 + l): per point
// the copy of a same-level sender, the decimation of a finer one (every
// other point) or the prediction of a coarser one (pred_any), every
// component, into the receiver's ghost nodes.  P is the same in every lane
// (read through the scalar unit); sbase: block P.send of the sender array.
__device__ __forceinline__ void sync_patch(double *__restrict__ arr, const wh_patch &P,
                                           const double *__restrict__ sbase, size_t blk, size_t cs, int nx, int ny,
                                           int neq, int dim, int r0, int r_end = 1 << 30)
{
    const int n0 = P.n[0], n1 = P.n[1], np = min(n0 * n1 * P.n[2], r_end);
    double *dbase = arr + (size_t)P.recv * blk;
    const int op = P.op & 0xff;
    const int st = (op == WH_PATCH_RESTRICT) ? 2 : 1;
    for (int r = r0; r < np; r += 64) {
        const int i = r % n0, j = (r / n0) % n1, kk = r / (n0 * n1);
        double *dst = dbase + ((size_t)(P.recv_lo[2] + kk) * ny + (P.recv_lo[1] + j)) * nx + (P.recv_lo[0] + i);
        if (op == WH_PATCH_PREDICT) {
            const int f[3] = {P.send_lo[0] + i, P.send_lo[1] + j, P.send_lo[2] + kk};
            for (int c = 0; c < neq; ++c) dst[c * cs] = pred_any(sbase + c * cs, nx, ny, dim, f, P.aux);
        } else {
            const double *src = sbase + ((size_t)(P.send_lo[2] + st * kk) * ny + (P.send_lo[1] + st * j)) * nx +
                                (P.send_lo[0] + st * i);
            for (int c = 0; c < neq; ++c) dst[c * cs] = src[c * cs];
        }
    }
}

// 2D ghost fill of the patches [p0, p1): one wavefront per patch (patch
// p0 + w for wavefront w of the launch), its record read once through the
// scalar unit -- no search; a 2D ghost patch has a few dozen points, so the
// wavefront takes them in one or two steps (3D patches are far larger and
// are cut into chunks, k_sync_chunks).  Bits 8-9 of a patch's op select the
// array its sender is read from (0: the synced array itself, 1/2: the
// alternates in S).
__global__ __launch_bounds__(256) void k_sync_patches(double *__restrict__ arr, const wh_patch *__restrict__ pt,
                                                      int p0, int p1, size_t blk, size_t cs, int nx, int ny,
                                                      int neq, SyncSrc S)
{
    const int q = p0 + (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (q >= p1) return;
    const wh_patch P = pt[q];
    const int sel = (P.op >> 8) & 3;
    const double *sbase = sel == 0 ? arr + (size_t)P.send * blk
                                   : S.alt[sel - 1] + (size_t)P.send * S.blk_alt[sel - 1];
    sync_patch(arr, P, sbase, blk, cs, nx, ny, neq, 2, (int)(threadIdx.x & 63u));
}

// 3D ghost fill of the chunks [c0, c1): one wavefront per chunk (chunk c0 + w
// for wavefront w of the launch), chunk and patch records read once through
// the scalar unit, lane l takes points first + l, first + l + 64, ... of the
// chunk.
__global__ __launch_bounds__(256) void k_sync_chunks(double *__restrict__ arr, const wh_patch *__restrict__ pt,
                                                     const SyncChunk *__restrict__ ch, int c0, int c1, size_t blk,
                                                     size_t cs, int nx, int ny, int neq, SyncSrc S)
{
    const int q = c0 + (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (q >= c1) return;
    const SyncChunk c = ch[q];
    const wh_patch P = pt[c.patch];
    const int sel = (P.op >> 8) & 3;
    const double *sbase = sel == 0 ? arr + (size_t)P.send * blk
                                   : S.alt[sel - 1] + (size_t)P.send * S.blk_alt[sel - 1];
    sync_patch(arr, P, sbase, blk, cs, nx, ny, neq, 3, c.first + (int)(threadIdx.x & 63u), c.first + SYNC_CHUNK);
}

int launch_sync_flat(wh_pool *P, double *arr, const wh_patch *d_patches, const SyncChunk *d_chunks, int p0, int p1,
                     int c0, int c1, const SyncSrc &S)
{
    if (P->d.dim == 2) {
        if (p1 > p0)
            hipLaunchKernelGGL(k_sync_patches, dim3((unsigned)((p1 - p0 + 3) / 4)), dim3(256), 0, P->stream, arr,
                               d_patches, p0, p1, P->blk, P->cs, P->nx, P->ny, P->d.neq, S);
    } else if (c1 > c0) {
        hipLaunchKernelGGL(k_sync_chunks, dim3((unsigned)((c1 - c0 + 3) / 4)), dim3(256), 0, P->stream, arr,
                           d_patches, d_chunks, c0, c1, P->blk, P->cs, P->nx, P->ny, P->d.neq, S);
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

// 3D ghost fill over the chunks of several pools (one sync stage s): the
// stage's chunks are the pools' chunk ranges [c0[s], c1[s]) one after the
// other (pool p's from s0[s] on); wavefront w of the launch fills chunk
// w - s0[s] + c0[s] of the pool whose range holds w, as k_sync_chunks.
// Persistent over the chunks, their count tot[stage] read from device
// memory; into array `sel` of the pool.
__global__ __launch_bounds__(256) void k_sync_multi(const MPoolDev *__restrict__ pools, int npools, int sel,
                                                    int stage, const int64_t *__restrict__ tot)
{
    const int s = stage - 1;
    const int64_t nc = tot[stage];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int64_t w = (int64_t)blockIdx.x * 4 + wv; w < nc; w += (int64_t)gridDim.x * 4) {
        const MPoolDev &M = pools[__builtin_amdgcn_readfirstlane(pool_of(pools, npools, w, s))];
        const SyncChunk c = M.ch[M.c0[s] + (int)(w - M.s0[s])];
        const wh_patch P = M.pt[c.patch];
        double *arr = M.arr[sel];
        const Geo &G = M.G;
        sync_patch(arr, P, arr + (size_t)P.send * G.blk, G.blk, G.cs, G.nx, G.ny, M.neq, 3,
                   c.first + (int)(threadIdx.x & 63u), c.first + SYNC_CHUNK);
    }
}

// 2D ghost fill over the patches of several pools (one sync stage s): the
// stage's patches are the pools' patch ranges [p0[s], p1[s]) one after the
// other (pool p's from q0[s] on); wavefront w of the launch fills patch
// w - q0[s] + p0[s] of the pool whose range holds w, as k_sync_patches.
// Persistent over the patches, their count tot[4 + s] read from device
// memory.
__global__ __launch_bounds__(256) void k_sync_multi_patches(const MPoolDev *__restrict__ pools, int npools,
                                                            int sel, int stage, const int64_t *__restrict__ tot)
{
    const int s = stage - 1;
    const int64_t nq = tot[4 + s];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int64_t w = (int64_t)blockIdx.x * 4 + wv; w < nq; w += (int64_t)gridDim.x * 4) {
        const MPoolDev &M = pools[__builtin_amdgcn_readfirstlane(pool_of(pools, npools, w, 3 + s))];
        const wh_patch P = M.pt[M.p0[s] + (int)(w - M.q0[s])];
        double *arr = M.arr[sel];
        const Geo &G = M.G;
        sync_patch(arr, P, arr + (size_t)P.send * G.blk, G.blk, G.cs, G.nx, G.ny, M.neq, 2,
                   (int)(threadIdx.x & 63u));
    }
}

int launch_sync_multi(hipStream_t stream, const MPoolDev *d_pools, int npools, int sel, int stage,
                      const int64_t *d_tot, int grid, int dim)
{
    if (dim == 2)
        hipLaunchKernelGGL(k_sync_multi_patches, dim3(grid), dim3(256), 0, stream, d_pools, npools, sel, stage,
                           d_tot);
    else
        hipLaunchKernelGGL(k_sync_multi, dim3(grid), dim3(256), 0, stream, d_pools, npools, sel, stage, d_tot);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_entries(hipStream_t stream, const MPoolDev *d_pools, int npools, const int64_t *d_tot, MEnt *d_ents,
                   int grid)
{
    hipLaunchKernelGGL(k_entries, dim3(grid), dim3(256), 0, stream, d_pools, npools, d_tot, d_ents);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_stage_multi(hipStream_t stream, int dim, int scheme, int skew, int xcd, const MPoolDev *d_pools,
                       int npools, const MEnt *d_ents, const double *d_dtg, const AcmDev *d_gacm,
                       const int64_t *d_tot, const MStage &ms, size_t lds, int grid, int nchunk)
{
    (void)npools;
    if (dim == 2) {
#define M2D(SC, SK)                                                                                           \
    hipLaunchKernelGGL((k_rhs2d_multi<SC, SK>), dim3(grid), dim3(256), lds, stream, d_pools, d_ents, d_dtg, d_gacm, \
                       d_tot, ms)
        switch (scheme * 2 + skew) {
        case WH_FD2 * 2: M2D(WH_FD2, false); break;
        case WH_FD2 * 2 + 1: M2D(WH_FD2, true); break;
        case WH_FD4 * 2: M2D(WH_FD4, false); break;
        case WH_FD4 * 2 + 1: M2D(WH_FD4, true); break;
        case WH_FD4_TW * 2: M2D(WH_FD4_TW, false); break;
        case WH_FD4_TW * 2 + 1: M2D(WH_FD4_TW, true); break;
        case WH_FD6 * 2: M2D(WH_FD6, false); break;
        case WH_FD6 * 2 + 1: M2D(WH_FD6, true); break;
        default: set_error("unknown scheme"); return WH_E_ARG;
        }
#undef M2D
    } else {
#define M3D(SC, SK)                                                                                           \
    do {                                                                                                      \
        if (xcd)                                                                                              \
            hipLaunchKernelGGL((k_rhs3d_multi<SC, SK, true>), dim3(grid), dim3(256), 0, stream, d_pools, d_ents, \
                               d_dtg, d_gacm, d_tot, ms, nchunk);                                              \
        else                                                                                                  \
            hipLaunchKernelGGL((k_rhs3d_multi<SC, SK, false>), dim3(grid), dim3(256), 0, stream, d_pools, d_ents, \
                               d_dtg, d_gacm, d_tot, ms, nchunk);                                              \
    } while (0)
        switch (scheme * 2 + skew) {
        case WH_FD2 * 2: M3D(WH_FD2, false); break;
        case WH_FD2 * 2 + 1: M3D(WH_FD2, true); break;
        case WH_FD4 * 2: M3D(WH_FD4, false); break;
        case WH_FD4 * 2 + 1: M3D(WH_FD4, true); break;
        case WH_FD4_TW * 2: M3D(WH_FD4_TW, false); break;
        case WH_FD4_TW * 2 + 1: M3D(WH_FD4_TW, true); break;
        case WH_FD6 * 2: M3D(WH_FD6, false); break;
        case WH_FD6 * 2 + 1: M3D(WH_FD6, true); break;
        default: set_error("unknown scheme"); return WH_E_ARG;
        }
#undef M3D
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

// Per-receiver ghost fill (the plain one-launch-per-block path): one
// workgroup walks the patches of one (stage, receiver) row of the table.
__global__ __launch_bounds__(256) void k_sync(double *__restrict__ arr,
                                              const wh_patch *__restrict__ pt,
                                              const int32_t *__restrict__ off, int row0,
                                              int stage, size_t blk, size_t cs, int nx, int ny,
                                              int neq)
{
    const int row = row0 + blockIdx.x;
    const int dim = (cs == (size_t)nx * ny) ? 2 : 3;
    for (int q = off[row]; q < off[row + 1]; ++q) {
        const wh_patch P = pt[q];
        if (stage > 0 && P.stage != stage) continue;
        const int n0 = P.n[0], n1 = P.n[1], n2 = P.n[2];
        const int npt = n0 * n1 * n2;
        const int st = (P.op == WH_PATCH_RESTRICT) ? 2 : 1;
        double *dst = arr + (size_t)P.recv * blk;
        const double *src = arr + (size_t)P.send * blk;
        for (int e = threadIdx.x; e < npt * neq; e += blockDim.x) {
            const int c = e / npt, r = e - c * npt;
            const int i = r % n0, j = (r / n0) % n1, kk = r / (n0 * n1);
            const size_t ri = ((size_t)(P.recv_lo[2] + kk) * ny + (P.recv_lo[1] + j)) * nx +
                              (P.recv_lo[0] + i);
            if (P.op == WH_PATCH_PREDICT) {
                const int f[3] = {P.send_lo[0] + i, P.send_lo[1] + j, P.send_lo[2] + kk};
                dst[c * cs + ri] = pred_any(src + c * cs, nx, ny, dim, f, P.aux);
                continue;
            }
            const size_t si = ((size_t)(P.send_lo[2] + st * kk) * ny + (P.send_lo[1] + st * j)) * nx +
                              (P.send_lo[0] + st * i);
            dst[c * cs + ri] = src[c * cs + si];
        }
    }
}

// refineBlock (refinementExecute.f90:4-116): daughter k of a mother takes
// points g + Bs*off_k + i (i over its ghost-inclusive block) of the mother's
// interpolated grid; one thread per daughter point.
__global__ __launch_bounds__(256) void k_refine(double *__restrict__ arr,
                                                const int32_t *__restrict__ pairs, int npairs,
                                                int bs0, int bs1, int bs2, int g, int nx, int ny,
                                                int nz, size_t blk, size_t cs, int neq, int dim,
                                                int order)
{
    const size_t npt = (size_t)nx * ny * nz;
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= npt * npairs) return;
    const int q = (int)(e / npt);
    const int r = (int)(e - (size_t)q * npt);
    const int i = r % nx, j = (r / nx) % ny, k = r / (nx * ny);
    const int mother = pairs[3 * q], daughter = pairs[3 * q + 1], dg = pairs[3 * q + 2];
    const int off[3] = {(dg >> 1) & 1, dg & 1, (dg >> 2) & 1};
    const int f[3] = {g + bs0 * off[0] + i, g + bs1 * off[1] + j,
                      dim == 3 ? g + bs2 * off[2] + k : 0};
    const double *src = arr + (size_t)mother * blk;
    double *dst = arr + (size_t)daughter * blk + r;
    for (int c = 0; c < neq; ++c) dst[c * cs] = pred_any(src + c * cs, nx, ny, dim, f, order);
}

// 2D refineBlock with the mother's component plane staged in LDS: one
// workgroup per (pair, component), each daughter point pred_point of the
// staged plane -- k_refine's arithmetic, its stencil reads from LDS
// instead of up to (2N)^2 cached global loads per point.  The host's
// stencil-range check keeps every read inside the plane.
template <int N>
__global__ __launch_bounds__(256) void k_refine2d_lds(double *__restrict__ arr, const int32_t *__restrict__ pairs,
                                                      int bs0, int bs1, int g, int nx, int ny, size_t blk, size_t cs,
                                                      int neq)
{
    extern __shared__ double plane[];
    const int q = (int)blockIdx.x / neq, c = (int)blockIdx.x - q * neq;
    const int mother = pairs[3 * q], daughter = pairs[3 * q + 1], dg = pairs[3 * q + 2];
    const int npt = nx * ny;
    const double *src = arr + (size_t)mother * blk + (size_t)c * cs;
    for (int e = threadIdx.x; e < npt; e += blockDim.x) plane[e] = src[e];
    __syncthreads();
    double *dst = arr + (size_t)daughter * blk + (size_t)c * cs;
    const int o0 = g + bs0 * ((dg >> 1) & 1), o1 = g + bs1 * (dg & 1);
    for (int r = threadIdx.x; r < npt; r += blockDim.x) {
        const int j = r / nx, i = r - j * nx;
        const int f[3] = {o0 + i, o1 + j, 0};
        dst[r] = pred_point<N>(plane, nx, ny, 2, f);
    }
}

// 3D refineBlock, one thread per (x, y) column of a daughter component,
// marching in z: the x-then-y interpolated values of the mother's coarse
// planes (pred_point's vy) pass through a register window of 2N planes, and
// each fine z point is either the window's centre plane (even index) or the
// left-to-right z sum over the window (odd index) -- pred_point's arithmetic
// in pred_point's order, each vy computed once per column instead of once
// per output point.  Window planes outside the mother are set to zero; the
// host's stencil-range check guarantees no output reads them.
template <int N>
__global__ __launch_bounds__(256) void k_refine3d(double *__restrict__ arr,
                                                  const int32_t *__restrict__ pairs, int npairs,
                                                  int wpc, int bs0, int bs1, int bs2, int g, int nx,
                                                  int ny, int nz, size_t blk, size_t cs, int neq)
{
    constexpr double c2[2] = {0.5, 0.5};
    constexpr double c4[4] = {-1.0 / 16.0, 9.0 / 16.0, 9.0 / 16.0, -1.0 / 16.0};
    constexpr double c6[6] = {3.0 / 256.0, -25.0 / 256.0, 150.0 / 256.0,
                              150.0 / 256.0, -25.0 / 256.0, 3.0 / 256.0};
    const double *cf = (N == 1) ? c2 : (N == 2) ? c4 : c6;
    // `wpc` workgroups per (pair, component): the pair and component are a
    // scalar division of the (XCD-swizzled: the daughters of a mother, listed
    // together, read it through one L2) workgroup index
    const int ncol = nx * ny;
    const int wg = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int qc = wg / wpc;
    const int q = qc / neq, c = qc - q * neq;
    const int r = (wg - qc * wpc) * (int)blockDim.x + (int)threadIdx.x;
    if (r >= ncol) return;
    const int j = r / nx, i = r - j * nx;
    const int mother = pairs[3 * q], daughter = pairs[3 * q + 1], dg = pairs[3 * q + 2];
    const int f0 = g + bs0 * ((dg >> 1) & 1) + i, f1 = g + bs1 * (dg & 1) + j;
    const int fz0 = g + bs2 * ((dg >> 2) & 1);
    const int cx = f0 >> 1, px = f0 & 1, cy = f1 >> 1, py = f1 & 1;
    const double *u = arr + (size_t)mother * blk + (size_t)c * cs;
    double *dst = arr + (size_t)daughter * blk + (size_t)c * cs + (size_t)j * nx + i;
    auto vx = [&](int jy, int kz) -> double {
        const double *row = u + ((size_t)kz * ny + jy) * nx;
        if (!px) return row[cx];
        double s = cf[0] * row[cx - N + 1];
#pragma unroll
        for (int t = 1; t < 2 * N; ++t) s = s + cf[t] * row[cx - N + 1 + t];
        return s;
    };
    auto vy = [&](int kz) -> double {
        if (kz < 0 || kz >= nz) return 0.0;
        if (!py) return vx(cy, kz);
        double s = cf[0] * vx(cy - N + 1, kz);
#pragma unroll
        for (int t = 1; t < 2 * N; ++t) s = s + cf[t] * vx(cy - N + 1 + t, kz);
        return s;
    };
    int cz = fz0 >> 1;
    double w[2 * N];  // vy(cz - N + 1 .. cz + N)
#pragma unroll
    for (int t = 0; t < 2 * N; ++t) w[t] = vy(cz - N + 1 + t);
    const size_t pstride = (size_t)ncol;
    for (int k = 0; k < nz; ++k) {
        const int f2 = fz0 + k;
        if ((f2 >> 1) != cz) {
            ++cz;
#pragma unroll
            for (int t = 0; t < 2 * N - 1; ++t) w[t] = w[t + 1];
            w[2 * N - 1] = vy(cz + N);
        }
        double v;
        if (f2 & 1) {
            v = cf[0] * w[0];
#pragma unroll
            for (int t = 1; t < 2 * N; ++t) v = v + cf[t] * w[t];
        } else {
            v = w[N - 1];
        }
        dst[(size_t)k * pstride] = v;
    }
}

// 3D refineBlock, one workgroup per (pair, component), marching through the
// mother's coarse planes: per plane kz the coarse rows and columns the
// daughter reaches are staged in LDS (A), the x interpolation of every
// staged row at every fine x goes to LDS (B; pred_point's vx), and each
// thread takes the y interpolation (vy) of its own fine (x, y) points into a
// register window of the last 2N planes.  When the window ends at plane
// cz + N, the fine planes 2cz and 2cz + 1 are complete: the even one is the
// window's centre plane, the odd one the left-to-right z sum over the window
// -- pred_point's arithmetic in its order.  Coarse points outside the mother
// are staged as zero; the host's stencil-range check guarantees no output
// reads them.  PPT: fine (x, y) points per thread.
template <int N, int PPT>
__global__ __launch_bounds__(256) void k_refine3d_lds(double *__restrict__ arr,
                                                      const int32_t *__restrict__ pairs, int bs0, int bs1,
                                                      int bs2, int g, int nx, int ny, int nz, size_t blk,
                                                      size_t cs, int neq)
{
    constexpr double c2[2] = {0.5, 0.5};
    constexpr double c4[4] = {-1.0 / 16.0, 9.0 / 16.0, 9.0 / 16.0, -1.0 / 16.0};
    constexpr double c6[6] = {3.0 / 256.0, -25.0 / 256.0, 150.0 / 256.0,
                              150.0 / 256.0, -25.0 / 256.0, 3.0 / 256.0};
    const double *cf = (N == 1) ? c2 : (N == 2) ? c4 : c6;
    extern __shared__ double lds[];
    const int wg = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int q = wg / neq, c = wg - q * neq;
    const int mother = pairs[3 * q], daughter = pairs[3 * q + 1], dg = pairs[3 * q + 2];
    const int fx0 = g + bs0 * ((dg >> 1) & 1), fy0 = g + bs1 * (dg & 1), fz0 = g + bs2 * ((dg >> 2) & 1);
    // staged coarse window: columns [cxa, cxa + ncol), rows [cya, cya + nrow)
    const int cxa = (fx0 >> 1) - N + 1, ncol = ((fx0 + nx - 1) >> 1) + N - cxa + 1;
    const int cya = (fy0 >> 1) - N + 1, nrow = ((fy0 + ny - 1) >> 1) + N - cya + 1;
    double *A = lds, *B = lds + nrow * ncol;
    const double *u = arr + (size_t)mother * blk + (size_t)c * cs;
    double *dst = arr + (size_t)daughter * blk + (size_t)c * cs;
    const int nxy = nx * ny, tid = threadIdx.x;
    double win[PPT][2 * N];
    const int kz0 = (fz0 >> 1) - N + 1, kz1 = ((fz0 + nz - 1) >> 1) + N;
    for (int kz = kz0; kz <= kz1; ++kz) {
        const bool inz = kz >= 0 && kz < nz;
        __syncthreads();  // the previous plane's B reads are done
        for (int e = tid; e < nrow * ncol; e += 256) {
            const int r = e / ncol, cc = e - r * ncol;
            const int y = cya + r, x = cxa + cc;
            A[e] = (inz && y >= 0 && y < ny && x >= 0 && x < nx) ? u[((size_t)kz * ny + y) * nx + x] : 0.0;
        }
        __syncthreads();
        for (int e = tid; e < nrow * nx; e += 256) {
            const int r = e / nx, i = e - r * nx;
            const int f0 = fx0 + i, cx = (f0 >> 1) - cxa;
            const double *row = A + r * ncol;
            double v;
            if (f0 & 1) {
                v = cf[0] * row[cx - N + 1];
#pragma unroll
                for (int t = 1; t < 2 * N; ++t) v = v + cf[t] * row[cx - N + 1 + t];
            } else {
                v = row[cx];
            }
            B[e] = v;
        }
        __syncthreads();
#pragma unroll
        for (int pp = 0; pp < PPT; ++pp) {
            const int pt = tid + 256 * pp;
            double v = 0.0;
            if (pt < nxy) {
                const int j = pt / nx, i = pt - j * nx;
                const int f1 = fy0 + j, cy = (f1 >> 1) - cya;
                if (f1 & 1) {
                    v = cf[0] * B[(cy - N + 1) * nx + i];
#pragma unroll
                    for (int t = 1; t < 2 * N; ++t) v = v + cf[t] * B[(cy - N + 1 + t) * nx + i];
                } else {
                    v = B[cy * nx + i];
                }
            }
#pragma unroll
            for (int t = 0; t < 2 * N - 1; ++t) win[pp][t] = win[pp][t + 1];
            win[pp][2 * N - 1] = v;
        }
        // fine planes whose window ends here
        const int cz = kz - N;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int f2 = 2 * cz + h, k = f2 - fz0;
            if (k < 0 || k >= nz) continue;
#pragma unroll
            for (int pp = 0; pp < PPT; ++pp) {
                const int pt = tid + 256 * pp;
                if (pt >= nxy) continue;
                double v;
                if (h) {
                    v = cf[0] * win[pp][0];
#pragma unroll
                    for (int t = 1; t < 2 * N; ++t) v = v + cf[t] * win[pp][t];
                } else {
                    v = win[pp][N - 1];
                }
                dst[(size_t)k * nxy + pt] = v;
            }
        }
    }
}

// LDS bytes of k_refine3d_lds for this pool and order, 0 if it does not apply
static size_t refine3d_lds_bytes(const wh_pool *P, int N)
{
    if (P->nx * P->ny > 8 * 256) return 0;
    const int ncol = P->nx / 2 + 2 * N + 2, nrow = P->ny / 2 + 2 * N + 2;  // upper bounds
    const size_t b = sizeof(double) * ((size_t)nrow * ncol + (size_t)nrow * P->nx);
    return b <= 64 * 1024 ? b : 0;
}

int launch_refine(wh_pool *P, double *arr, const int32_t *d_pairs, int npairs, int order)
{
    if (npairs <= 0) return WH_OK;
    if (P->d.dim == 3 && refine3d_lds_bytes(P, order / 2) > 0) {
        const int N = order / 2, ppt = (P->nx * P->ny + 255) / 256;
        const size_t lds = refine3d_lds_bytes(P, N);
        const dim3 grid((unsigned)((size_t)P->d.neq * npairs));
#define LRL(NN, PP)                                                                                    \
    hipLaunchKernelGGL((k_refine3d_lds<NN, PP>), grid, dim3(256), lds, P->stream, arr, d_pairs, P->d.bs[0], \
                       P->d.bs[1], P->d.bs[2], P->d.g, P->nx, P->ny, P->nz, P->blk, P->cs, P->d.neq)
#define LRN(NN)                        \
    do {                               \
        if (ppt <= 2) LRL(NN, 2);      \
        else if (ppt <= 4) LRL(NN, 4); \
        else if (ppt <= 6) LRL(NN, 6); \
        else LRL(NN, 8);               \
    } while (0)
        if (N == 2) LRN(2);
        else if (N == 1) LRN(1);
        else LRN(3);
#undef LRN
#undef LRL
        WH_HIP(hipGetLastError());
        return WH_OK;
    }
    if (P->d.dim == 3) {
        const int wpc = (P->nx * P->ny + 255) / 256;
        const dim3 grid((unsigned)((size_t)wpc * P->d.neq * npairs));
#define LR3(NN)                                                                                    \
    hipLaunchKernelGGL(k_refine3d<NN>, grid, dim3(256), 0, P->stream, arr, d_pairs, npairs, wpc,   \
                       P->d.bs[0], P->d.bs[1], P->d.bs[2], P->d.g, P->nx, P->ny, P->nz, P->blk,    \
                       P->cs, P->d.neq)
        if (order == 4) LR3(2);
        else if (order == 2) LR3(1);
        else LR3(3);
#undef LR3
        WH_HIP(hipGetLastError());
        return WH_OK;
    }
    const size_t plane = sizeof(double) * (size_t)P->nx * P->ny;
    if (P->d.dim == 2 && plane <= 64 * 1024) {
        const dim3 grid((unsigned)((size_t)P->d.neq * npairs));
#define LR2(NN)                                                                                              \
    hipLaunchKernelGGL(k_refine2d_lds<NN>, grid, dim3(256), plane, P->stream, arr, d_pairs, P->d.bs[0], P->d.bs[1], \
                       P->d.g, P->nx, P->ny, P->blk, P->cs, P->d.neq)
        if (order == 4) LR2(2);
        else if (order == 2) LR2(1);
        else LR2(3);
#undef LR2
        WH_HIP(hipGetLastError());
        return WH_OK;
    }
    const size_t npt = (size_t)P->nx * P->ny * P->nz * npairs;
    hipLaunchKernelGGL(k_refine, dim3((unsigned)((npt + 255) / 256)), dim3(256), 0, P->stream, arr,
                       d_pairs, npairs, P->d.bs[0], P->d.bs[1], P->d.dim == 3 ? P->d.bs[2] : 1,
                       P->d.g, P->nx, P->ny, P->nz, P->blk, P->cs, P->d.neq, P->d.dim, order);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_sync(wh_pool *P, int sync_case, double *arr, int one_receiver)
{
    PatchSet &ps = P->ps[sync_case];
    if (ps.n == 0) return WH_OK;
    if (one_receiver >= 0) {
        // one launch per (stage, receiver) row: the reference's per-block loop
        hipLaunchKernelGGL(k_sync, dim3(1), dim3(256), 0, P->stream, arr, ps.d_patches,
                           ps.d_recv_off, one_receiver, 0, P->blk, P->cs, P->nx, P->ny, P->d.neq);
        WH_HIP(hipGetLastError());
        return WH_OK;
    }
    for (int stage = 1; stage <= 3; ++stage) {
        const int p0 = ps.stage_begin[stage], p1 = ps.stage_begin[stage + 1];
        if (p1 <= p0) continue;
        if (int rc = launch_sync_flat(P, arr, ps.d_patches, ps.d_chunks, p0, p1, ps.chunk_begin[stage],
                                      ps.chunk_begin[stage + 1], SyncSrc{}))
            return rc;
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

// ---------------------------------------------------------------------------
// RK combination over block interiors: out = base + sum coef_i * term_i
// ---------------------------------------------------------------------------
struct CombineArgs {
    const double *base;
    const double *terms[8];
    double coefs[8];
    int nterms;
};

__global__ __launch_bounds__(256) void k_combine(double *__restrict__ out, CombineArgs ca,
                                                 const int32_t *__restrict__ act, Geo G, int neq)
{
    const int npts = G.bs0 * G.bs1 * G.bs2;
    const int nchunk = (npts * neq + 255) / 256;
    const int k = blockIdx.x / nchunk;
    const int e = (blockIdx.x - k * nchunk) * 256 + threadIdx.x;
    if (e >= npts * neq) return;
    const int b = act[k];
    const int c = e / npts, pnt = e - c * npts;
    const int ix = pnt % G.bs0, iy = (pnt / G.bs0) % G.bs1, iz = pnt / (G.bs0 * G.bs1);
    const int zoff = (G.bs2 > 1) ? G.g : 0;
    const size_t i = (size_t)b * G.blk + c * G.cs +
                     ((size_t)(zoff + iz) * G.ny + (G.g + iy)) * G.nx + (G.g + ix);
    double v = ca.base[i];
    for (int t = 0; t < ca.nterms; ++t) v = v + ca.coefs[t] * ca.terms[t][i];
    out[i] = v;
}

int launch_combine(wh_pool *P, double *out, const double *base, int nterms,
                   const double *const *terms, const double *coefs, const int32_t *act, int nact)
{
    WH_CHECK(nterms >= 0 && nterms <= 8, WH_E_ARG, "rk_combine: at most 8 terms");
    if (nact <= 0) return WH_OK;
    CombineArgs ca{};
    ca.base = base;
    ca.nterms = nterms;
    for (int t = 0; t < nterms; ++t) {
        ca.terms[t] = terms[t];
        ca.coefs[t] = coefs[t];
    }
    const Geo G = make_geo(P);
    const int npts = G.bs0 * G.bs1 * G.bs2;
    const int nchunk = (npts * P->d.neq + 255) / 256;
    hipLaunchKernelGGL(k_combine, dim3(nact * nchunk), dim3(256), 0, P->stream, out, ca, act, G,
                       P->d.neq);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

// ---------------------------------------------------------------------------
// reductions: per-block dt (GET_DT_BLOCK_ACM) and max |u| (divergence guard)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ double block_max(double v)
{
    __shared__ double red[16];
    v = wave_max(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) red[w] = v;
    __syncthreads();
    if (w == 0) {
        v = (l < (int)(blockDim.x >> 6)) ? red[l] : -1.0;
        v = wave_max(v);
    }
    return v;
}

// dt clamps of calculate_time_step.f90:58-118 on the device, so that a whole
// step can be replayed from a hipGraph without a host round trip, and the
// time advance of the step that takes this dt (its stages read DS_DT only).
__device__ void dt_finalize(double *scal, double dtmin, const TimeDev &tc)
{
    const double time = scal[DS_TIME];
    double dt;
    if (tc.dt_fixed > 0.0) {
        dt = tc.dt_fixed;
    } else {
        dt = dtmin;
        if (tc.dt_max > 0.0) dt = fmin(tc.dt_max, dt);
    }
    if (tc.write_fixed_time) {
        if (fmod(time + dt, tc.write_time) < fmod(time + 1e-12, tc.write_time) &&
            !(fabs(fmod(time, tc.write_time)) < 1e-12) && time + 1e-12 > tc.write_time_first)
            dt = tc.write_time - fmod(time, tc.write_time);
    }
    if (tc.write_backup_n > 0) {
        const double wb = tc.write_backup_time;
        if (fmod(time + dt, wb) < fmod(time + 1e-12, wb) && !(fabs(fmod(time, wb)) < 1e-12))
            dt = wb - fmod(time, wb);
    }
    if (tc.use_stats) {
        const double ts = tc.tsave_stats;
        if (fmod(time + dt, ts) < fmod(time + 1e-12, ts) && !(fabs(fmod(time, ts)) < 1e-12))
            dt = ts - fmod(time, ts);
    }
    if (time + dt > tc.time_max && time <= tc.time_max) dt = tc.time_max - time;
    if (!(time < tc.time_max)) dt = 0.0;  // main.f90:293 loop condition
    scal[DS_DT] = dt;
    if (dt > 0.0) {
        scal[DS_TIME] = time + dt;
        scal[DS_ITER] = scal[DS_ITER] + 1.0;
    }
}

// The minimum over all active blocks of a launch without groups: every
// workgroup adds its minimum to DS_DTACC; the one that counts the last hands
// the result on (DS_DTMIN_BITS; with STEP also dt_finalize) and leaves the
// accumulator and the counter as it found them.  One launch instead of four
// (clear, reduce, clamps, time advance): for small grids each of them cost as
// much as a stage.
template <bool STEP>
__device__ void dt_combine(double *scal, double v, const TimeDev &tc)
{
    unsigned long long *acc = (unsigned long long *)(scal + DS_DTACC), *cnt = (unsigned long long *)(scal + DS_DTCNT);
    if (v < DT_NONE)
        __hip_atomic_fetch_min(acc, (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    if (__hip_atomic_fetch_add(cnt, 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) + 1 != gridDim.x) return;
    // the others' minima were released through the counter: only the last
    // workgroup, which reads them, has to acquire
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const double m = __longlong_as_double(
        (long long)__hip_atomic_exchange(acc, (unsigned long long)__double_as_longlong(DT_NONE), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT));
    __hip_atomic_store(cnt, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    scal[DS_DTMIN_BITS] = m;
    if constexpr (STEP) dt_finalize(scal, m, tc);
}

// GET_DT_BLOCK_ACM of the active blocks.  WAVES 1: a wavefront per block, four
// blocks per workgroup at a time (2D blocks of a few hundred points), 0: the
// workgroup per block; a workgroup goes on to the next ones until all are
// done.  Four points per lane are requested at a time.  The max and min are
// exact whatever the order, so the minimum may be combined in any grouping:
// per group with grp (into dtmin[group]), else over the launch (dt_combine).
template <int WAVES, bool STEP>
__global__ __launch_bounds__(256) void k_dt(const double *__restrict__ in,
                                            const int32_t *__restrict__ act,
                                            const double *__restrict__ x0dx, Geo G, AcmDev a0,
                                            unsigned long long *dtmin, const int32_t *__restrict__ grp,
                                            const AcmDev *__restrict__ gacm, int nact, double *scal, TimeDev tc)
{
    const int lane = WAVES ? (int)(threadIdx.x & 63) : (int)threadIdx.x, step = WAVES ? 64 : (int)blockDim.x;
    const int w = (int)(threadIdx.x >> 6);
    const int nxy = G.bs0 * G.bs1, npts = nxy * G.bs2, zoff = (G.bs2 > 1) ? G.g : 0;
    double all = DT_NONE;  // the minimum of this wavefront's (workgroup's) blocks, in lane 0
    for (int k0 = (int)blockIdx.x * (WAVES ? 4 : 1); k0 < nact; k0 += (int)gridDim.x * (WAVES ? 4 : 1)) {
        const int k = k0 + (WAVES ? w : 0);
        const bool live = k < nact;  // wave-uniform
        double dt = DT_NONE;
        if (live) {
            const double *u = in + (size_t)act[k] * G.blk;
            double m = -1.0;
            for (int p0 = lane; p0 < npts; p0 += 4 * step) {
                double v[4][3];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int p = min(p0 + j * step, npts - 1);  // the last point again past the end
                    const int iz = G.bs2 > 1 ? p / nxy : 0, r = p - iz * nxy, iy = r / G.bs0, ix = r - iy * G.bs0;
                    const size_t i = ((size_t)(zoff + iz) * G.ny + (G.g + iy)) * G.nx + (G.g + ix);
                    v[j][0] = u[i];
                    v[j][1] = u[G.cs + i];
                    v[j][2] = G.bs2 > 1 ? u[2 * G.cs + i] : 0.0;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    double s = v[j][0] * v[j][0] + v[j][1] * v[j][1];
                    if (G.bs2 > 1) s = s + v[j][2] * v[j][2];
                    m = fmax(m, s);
                }
            }
            m = WAVES ? wave_max(m) : block_max(m);
            if (lane == 0) {
                const AcmDev &a = gacm ? gacm[grp[k]] : a0;  // per-group constants of independent forests
                double dxmin = x0dx[6 * k + 3];
                for (int d = 1; d < a.dim; ++d) dxmin = fmin(dxmin, x0dx[6 * k + 3 + d]);
                const double ueig = sqrt(m) + sqrt(a.c_0 * a.c_0 + m);
                dt = (ueig >= 1.0e-6) ? a.CFL * dxmin / ueig : 1.0e-2;
                if (a.nu > 1.0e-13) dt = fmin(dt, a.CFL_nu * (dxmin * dxmin) / a.nu);
                if (a.gamma_p > 0.0) dt = fmin(dt, a.CFL_eta * a.gamma_p);
                if (a.penal) dt = fmin(dt, a.CFL_eta * a.C_eta);
                if (a.sponge) dt = fmin(dt, a.CFL_eta * a.C_sponge);
                if (!WAVES && grp) atomicMin(dtmin + grp[k], (unsigned long long)__double_as_longlong(dt));
                all = fmin(all, dt);
            }
        }
        if (!WAVES) {
            __syncthreads();  // block_max's shared memory is reused
        } else if (grp) {
            // the workgroup's four blocks (consecutive active entries: mostly one
            // group) combined first, one atomic per distinct group
            __shared__ double sdt[4];
            __shared__ int sgr[4];
            __syncthreads();
            if (lane == 0) {
                sdt[w] = dt;
                sgr[w] = live ? grp[k] : -1;
            }
            __syncthreads();
            if (threadIdx.x == 0)
                for (int x = 0; x < 4; ++x) {
                    if (sgr[x] < 0) continue;
                    bool first = true;
                    for (int y = 0; y < x; ++y) first = first && sgr[y] != sgr[x];
                    if (!first) continue;
                    double v = sdt[x];
                    for (int y = x + 1; y < 4; ++y)
                        if (sgr[y] == sgr[x]) v = fmin(v, sdt[y]);
                    atomicMin(dtmin + sgr[x], (unsigned long long)__double_as_longlong(v));
                }
        }
    }
    if (grp) return;
    if (WAVES) {
        __shared__ double part[4];
        if (lane == 0) part[w] = all;
        __syncthreads();
        all = fmin(fmin(part[0], part[1]), fmin(part[2], part[3]));
    }
    if (threadIdx.x == 0) dt_combine<STEP>(scal, all, tc);
}

__global__ __launch_bounds__(256) void k_maxabs(const double *__restrict__ in,
                                                const int32_t *__restrict__ act, Geo G, int neq,
                                                unsigned long long *mx)
{
    const int k = blockIdx.x, b = act[k];
    const int npts = G.bs0 * G.bs1 * G.bs2;
    const int zoff = (G.bs2 > 1) ? G.g : 0;
    const double *u = in + (size_t)b * G.blk;
    double m = 0.0;
    for (int e = threadIdx.x; e < npts * neq; e += blockDim.x) {
        const int c = e / npts, p = e - c * npts;
        const int ix = p % G.bs0, iy = (p / G.bs0) % G.bs1, iz = p / (G.bs0 * G.bs1);
        const size_t i = c * G.cs + ((size_t)(zoff + iz) * G.ny + (G.g + iy)) * G.nx + (G.g + ix);
        m = fmax(m, fabs(u[i]));
    }
    m = block_max(m);
    if (threadIdx.x == 0) atomicMax(mx, (unsigned long long)__double_as_longlong(m));
}

__global__ void k_scalar_init(double *scal, int which, double v)
{
    if (threadIdx.x == 0) scal[which] = v;
}

// Blocks of up to 600 points: a wavefront each (with the read-back, 4096
// blocks of 24^2: 38 us, by workgroups 50; 64 of 32^2: 21.7, by workgroups
// 20.4).
static bool dt_by_waves(const Geo &G) { return G.bs0 * G.bs1 * G.bs2 <= 600; }

int launch_dt(wh_pool *P, const AcmDev &a, const TimeDev *step)
{
    const Geo G = make_geo(P);
    const TimeDev tc = step ? *step : TimeDev{};
    const bool waves = dt_by_waves(G);
    // At most 1 (wavefronts) or 2 (workgroups per block) workgroups per compute
    // unit, as each ends with a release of its own: 4096 blocks of 16^2 31 / 33
    // / 44 us with 1 / 2 / 4, of 24^3 344 / 314 / 335 us.
    const dim3 grid(std::max(1, waves ? std::min(P->n_cu, (P->nact + 3) / 4) : std::min(2 * P->n_cu, P->nact)));
#define LDT(W, ST)                                                                                                 \
    hipLaunchKernelGGL((k_dt<W, ST>), grid, dim3(256), 0, P->stream, P->block, P->d_active, P->d_x0dx, G, a,        \
                       (unsigned long long *)nullptr, (const int32_t *)nullptr, (const AcmDev *)nullptr, P->nact, \
                       P->scal, tc)
    if (waves && step) LDT(1, true);
    else if (waves) LDT(1, false);
    else if (step) LDT(0, true);
    else LDT(0, false);
#undef LDT
    WH_HIP(hipGetLastError());
    return WH_OK;
}

__global__ void k_fill_u64(unsigned long long *p, int n, unsigned long long v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

int launch_dt_groups(wh_pool *P, const AcmDev &a)
{
    const int n = P->ngrp;
    unsigned long long bits;
    std::memcpy(&bits, &DT_NONE, sizeof bits);
    hipLaunchKernelGGL(k_fill_u64, dim3((n + 255) / 256), dim3(256), 0, P->stream, P->d_dtg, n,
                       bits);
    if (P->nact > 0) {
        const Geo G = make_geo(P);
        const AcmDev *gacm = P->ngacm == P->ngrp ? P->d_gacm : nullptr;
        const bool waves = dt_by_waves(G);
        const dim3 grid(waves ? (P->nact + 3) / 4 : P->nact);
        if (waves)
            hipLaunchKernelGGL((k_dt<1, false>), grid, dim3(256), 0, P->stream, P->block, P->d_active, P->d_x0dx, G, a,
                               P->d_dtg, (const int32_t *)P->d_grp, gacm, P->nact, P->scal, TimeDev{});
        else
            hipLaunchKernelGGL((k_dt<0, false>), grid, dim3(256), 0, P->stream, P->block, P->d_active, P->d_x0dx, G, a,
                               P->d_dtg, (const int32_t *)P->d_grp, gacm, P->nact, P->scal, TimeDev{});
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_maxabs(wh_pool *P, const double *in)
{
    hipLaunchKernelGGL(k_scalar_init, dim3(1), dim3(64), 0, P->stream, P->scal,
                       (int)DS_MAXABS_BITS, 0.0);
    if (P->nact > 0) {
        const Geo G = make_geo(P);
        hipLaunchKernelGGL(k_maxabs, dim3(P->nact), dim3(256), 0, P->stream, in, P->d_active, G,
                           P->d.neq, (unsigned long long *)(P->scal + DS_MAXABS_BITS));
    }
    WH_HIP(hipGetLastError());
    return WH_OK;
}

// time, iteration and dt of the device-side time loop in one launch
__global__ void k_time_set(double *scal, double time, double iter)
{
    if (threadIdx.x != 0) return;
    scal[DS_TIME] = time;
    scal[DS_ITER] = iter;
    scal[DS_DT] = 0.0;
}

int launch_time_set(wh_pool *P, double time, double iter)
{
    hipLaunchKernelGGL(k_time_set, dim3(1), dim3(64), 0, P->stream, P->scal, time, iter);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

int launch_set_scalar(wh_pool *P, int which, double v)
{
    hipLaunchKernelGGL(k_scalar_init, dim3(1), dim3(64), 0, P->stream, P->scal, which, v);
    WH_HIP(hipGetLastError());
    return WH_OK;
}

AcmDev make_acm_dev(const wh_acm_params *p)
{
    AcmDev a{};
    a.c02 = p->c_0 * p->c_0;
    a.c_0 = p->c_0;
    a.nu = p->nu;
    a.gamma_p = p->gamma_p;
    a.C_eta = p->C_eta;
    a.Cinv = 1.0 / p->C_eta;
    a.C_sponge = p->C_sponge;
    a.Csp_inv = 1.0 / p->C_sponge;
    for (int i = 0; i < 3; ++i) a.ums[i] = p->u_mean_set[i];
    a.CFL = p->CFL;
    a.CFL_nu = p->CFL_nu;
    a.CFL_eta = p->CFL_eta;
    a.dim = p->dim;
    a.scheme = p->scheme;
    a.skew = p->skew_symmetry ? 1 : 0;
    a.penal = p->penalization ? 1 : 0;
    a.sponge = p->use_sponge ? 1 : 0;
    return a;
}

}  // namespace wh
