// adjoint_fast.hip -- the tile-sorted adjoint engine's particle kernels (gfx950).
//
// The FP32 engine steps its particles with the production push kernel
// (k_push2d_split, index-carrying variant), the FP64 engine with k_fa_push64
// below: every step's particles sit in the tile bins of that step, and the push
// records for every input slot the slot its particle was written to.  The
// reverse step walks the
// same bins as the forward push of that step, one workgroup per tile: the
// tile's cell-corner E and B (of that step) in LDS, the adjoint current
// -s * Eb of the (T+5)^2 window in LDS, and the adjoint of the tile's corner
// fields accumulated in LDS and flushed with global atomics.  A particle's
// incoming adjoint is read at its output slot, its outgoing adjoint written
// at its input slot.
#include <type_traits>

#include "adjoint.h"
#include "adjoint_math.h"
#include "push_common.h"

namespace pictor {
namespace {
using namespace pushdev;
using namespace adjm;

// cell-corner E/B of the tile's T x T cells (the reference's VecE/VecB), component-major
template <typename R, int T, int BS>
__device__ inline void stage_corners(const GridP &g, int tx, int ty, const R *Ex, const R *Ey, const R *Ez,
                                     const R *Bx, const R *By, const R *Bz, typename V4<R>::T *sC)
{
    const int mx = g.mx;
    const int iw = 1 + tx * T, jw = 1 + ty * T;
    const R half = (R)0.5;
    for (int lc = threadIdx.x; lc < T * T; lc += BS) {
        const long long o = (long long)(iw + 2 + lc % T - 1) + (long long)mx * (jw + 2 + lc / T - 1);
        R v[6][4];
#pragma unroll
        for (int cn = 0; cn < 4; cn++) {
            const long long p = o + (cn & 1) + (cn >> 1) * (long long)mx;
            v[0][cn] = (Ex[p - 1] + Ex[p]) * half;
            v[1][cn] = (Ey[p - mx] + Ey[p]) * half;
            v[2][cn] = Ez[p];
            v[3][cn] = (Bx[p - mx] + Bx[p]) * half;
            v[4][cn] = (By[p - 1] + By[p]) * half;
            v[5][cn] = (Bz[p - 1 - mx] + Bz[p - 1] + Bz[p - mx] + Bz[p]) * (R)0.25;
        }
#pragma unroll
        for (int cc = 0; cc < 6; cc++) sC[6 * lc + cc] = {v[cc][0], v[cc][1], v[cc][2], v[cc][3]};
    }
}

// bins of a tile in the production kernel's order: centre bins of every species first
__device__ inline void vbin_of(int v, int nsp, int &s, int &d)
{
    if (v < nsp) { s = v; d = 4; return; }
    const int r = v - nsp;
    s = r >> 3;
    const int q = r & 7;
    d = q < 4 ? q : q + 1;
}

// one particle of the reverse sweep: its slot, species, state before the step
// and the slot it went to (where the adjoint of its state after the step is)
template <typename R>
struct AdjRec {
    unsigned slot;
    int s, to, ci, cj;
    R ox, oy, oz, u, v, w;
};

__device__ inline void load_rec(const PartSplit &st, const int *dst, AdjRec<float> &r)
{
    const unsigned sl = r.slot;
    r.to = dst[sl];
    const int cell = st.cell[sl];
    r.ci = cell & 0xFFFF; r.cj = cell >> 16;
    r.ox = st.ox[sl]; r.oy = st.oy[sl]; r.oz = kZMid;
    r.u = st.u[sl]; r.v = st.v[sl]; r.w = st.w[sl];
}
__device__ inline void load_rec(const PartE64 &st, const int *dst, AdjRec<double> &r)
{
    const unsigned sl = r.slot;
    r.to = dst[sl];
    const uint32_t cs = st.p.cs[sl];
    r.ci = (int)(cs & 0xFFFFu); r.cj = (int)((cs >> 16) & 0x7FFFu); r.s = (int)(cs >> 31);
    r.ox = st.p.ox[sl]; r.oy = st.p.oy[sl]; r.oz = st.p.oz[sl];
    r.u = st.p.u[sl]; r.v = st.p.v[sl]; r.w = st.p.w[sl];
}

// ---------------------------------------------------------------------------
// FP64 forward push on the tile bins.  The arithmetic of a particle is that of the unsorted
// engine (push_fwd, seg_values in FP64), bit for bit; what the tiles change is where the field
// comes from (LDS instead of 24 scattered loads a particle) and where the current goes: an LDS
// window flushed once per tile instead of 16 global FP64 atomics a particle.
// 128 x 128, 524288 particles: a forward step with its fields 270 -> 35 us, a reverse step
// 560 -> 70 us (k_eng_push and k_eng_adjoint of the unsorted engine: 246 and 518 us of these).
// The reverse sweep's state takes 233 registers, two waves per SIMD.
// ---------------------------------------------------------------------------
template <int T, int BS>
__global__ __launch_bounds__(BS) void k_fa_push64(GridP g, TileP tp, AdjP ap, const double *__restrict__ Ex,
                                                  const double *__restrict__ Ey, const double *__restrict__ Ez,
                                                  const double *__restrict__ Bx, const double *__restrict__ By,
                                                  const double *__restrict__ Bz, double *__restrict__ Jx,
                                                  double *__restrict__ Jy, double *__restrict__ Jz, PartE64 A,
                                                  PartE64 O, BinsP bins, SpillP sp, int *__restrict__ dst)
{
    constexpr int W = T + 5, WW = W * W, kLogT = T == 8 ? 3 : 4;
    __shared__ double4 sC[6 * T * T];
    __shared__ double sJ[3][WW];
    __shared__ int sStart[10], sCnt[9], sDstCap[9], sDstBin[9];
    __shared__ unsigned sSrc[9], sDstBase[9];
    if (sp.stop && *sp.stop < sp.step) return;
    const int tile = tile_remap(tp, blockIdx.x);
    const int tx = tile % tp.ntx, ty = tile / tp.ntx;
    const int iw = 1 + tx * T, jw = 1 + ty * T, cx0 = tx * T - 2, cy0 = ty * T - 2;
    const int tid = threadIdx.x;
    int bcnt = 0;
    if (tid < 9) {
        bcnt = bins.cnt_in[tile * tp.NB + tid];
        sSrc[tid] = (unsigned)bins.base[tile * tp.NB + tid];
        const int dt = wrap_tile(ty + tid / 3 - 1, tp.nty) * tp.ntx + wrap_tile(tx + tid % 3 - 1, tp.ntx);
        const int db = dt * tp.NB + tid;
        sDstBin[tid] = db;
        sDstBase[tid] = (unsigned)bins.base[db];
        sDstCap[tid] = bins.cap[db];
        sCnt[tid] = 0;
    }
    if (tid < 64) bin_starts(bcnt, 9, sStart);
    stage_corners<double, T, BS>(g, tx, ty, Ex, Ey, Ez, Bx, By, Bz, sC);
    for (int e = tid; e < WW; e += BS) { sJ[0][e] = 0.0; sJ[1][e] = 0.0; sJ[2][e] = 0.0; }
    __syncthreads();
    const int total = sStart[9];
    int bin = 0, binEnd = sStart[1];
    unsigned binOff = sSrc[0];
    for (int base = 0; base < total; base += BS) {
        const int k = base + tid;
        const bool active = k < total;
        int d = -1, id = 0;
        unsigned slot_in = 0;
        uint32_t ncs = 0;
        double ox = 0, oy = 0, oz = 0, un[3] = {0, 0, 0};
        if (active) {
            if (k >= binEnd) {
                do bin++; while (k >= sStart[bin + 1]);
                binEnd = sStart[bin + 1];
                binOff = sSrc[bin] - (unsigned)sStart[bin];
            }
            slot_in = binOff + (unsigned)k;
            const uint32_t cs = A.p.cs[slot_in];
            id = A.id[slot_in];
            const int ci = (int)(cs & 0xFFFFu), cj = (int)((cs >> 16) & 0x7FFFu), s = (int)(cs >> 31);
            const int li = ci - cx0 - 2, lj = cj - cy0 - 2;
            if (li < 0 || li >= T || lj < 0 || lj >= T) {
                atomicOr(sp.err, (int)kErrBounds);
            } else {
                const double x0 = A.p.ox[slot_in], y0 = A.p.oy[slot_in], z0 = A.p.oz[slot_in];
                PState<double> q;
                push_fwd<double>(ap, s, x0, y0, z0, A.p.u[slot_in], A.p.v[slot_in], A.p.w[slot_in],
                                 &sC[6 * (lj * T + li)], q);
                int di = q.d[0], dj = q.d[1];
                // offsets; a position rounded onto the upper face belongs to the next cell
                ox = q.x1[0] - (double)di;
                if (ox >= 1.0) { ox = 0.0; di += 1; }
                oy = q.x1[1] - (double)dj;
                if (oy >= 1.0) { oy = 0.0; dj += 1; }
                oz = q.x1[2] - (double)q.d[2];
                if (oz >= 1.0) oz = 0.0;
                un[0] = q.un1[0]; un[1] = q.un1[1]; un[2] = q.un1[2];
                double a[8], b[8];
                seg_values<double>(q.F1, q.W1, a);
                seg_values<double>(q.F2, q.W2, b);
                const int ei = q.d[0], ej = q.d[1];
                const bool cross = ei != 0 || ej != 0;
                if (!cross) {
#pragma unroll
                    for (int m = 0; m < 8; m++) a[m] += b[m];
                }
                auto add = [&](const double *u, int e) {
                    atomicAdd(&sJ[0][e], u[0]); atomicAdd(&sJ[0][e + W], u[1]);
                    atomicAdd(&sJ[1][e], u[2]); atomicAdd(&sJ[1][e + 1], u[3]);
                    atomicAdd(&sJ[2][e], u[4]); atomicAdd(&sJ[2][e + 1], u[5]);
                    atomicAdd(&sJ[2][e + W], u[6]); atomicAdd(&sJ[2][e + W + 1], u[7]);
                };
                const int e0 = (lj + 2) * W + li + 2;
                add(a, e0);
                if (cross) add(b, e0 + min(max(ej, -1), 1) * W + min(max(ei, -1), 1));
                int nci = ci + di, ncj = cj + dj;
                nci = nci < 0 ? nci + g.nx : (nci >= g.nx ? nci - g.nx : nci);
                ncj = ncj < 0 ? ncj + g.ny : (ncj >= g.ny ? ncj - g.ny : ncj);
                ncs = (uint32_t)nci | ((uint32_t)ncj << 16) | (cs & 0x80000000u);
                const int mi = (li + di) >> kLogT, mj = (lj + dj) >> kLogT;
                if (mi < -1 || mi > 1 || mj < -1 || mj > 1) atomicOr(sp.err, (int)kErrBounds);
                else d = 4 + mi + 3 * mj;
            }
        }
        const int slot = reserve_slot(d, 4, sCnt);
        if (active) {
            int to = -1;
            if (d >= 0 && slot < sDstCap[d]) {
                const unsigned o = sDstBase[d] + (unsigned)slot;
                O.p.cs[o] = ncs; O.id[o] = id;
                O.p.ox[o] = ox; O.p.oy[o] = oy; O.p.oz[o] = oz;
                O.p.u[o] = un[0]; O.p.v[o] = un[1]; O.p.w[o] = un[2];
                to = (int)o;
            } else if (d >= 0) {
                // centre bins grow with the tile's own population when the pass is repeated; a side
                // bin, or the centre of a nearly empty tile, would only overflow again
                spill_slot(sp);
                if (d != 4 || sDstCap[4] <= 80) atomicOr(sp.err, (int)kErrCapacity);
            }
            if (dst) dst[slot_in] = to;
        }
    }
    __syncthreads();
    for (int e = tid; e < WW; e += BS) {
        const long long o = (long long)(iw + e % W - 1) + (long long)g.mx * (jw + e / W - 1);
        const double a = sJ[0][e], b = sJ[1][e], cz = sJ[2][e];
        if (a != 0.0) unsafeAtomicAdd(&Jx[o], a);
        if (b != 0.0) unsafeAtomicAdd(&Jy[o], b);
        if (cz != 0.0) unsafeAtomicAdd(&Jz[o], cz);
    }
    if (tid < 9) bins.cnt_out[sDstBin[tid]] = min(sCnt[tid], sDstCap[tid]);
}

// the FP64 engine's particles from the caller's arrays (k_eng_load's rounding and checks)
__global__ __launch_bounds__(256) void k_fa_range64(AdjP ap, const double *__restrict__ x, const double *__restrict__ y,
                                                    const double *__restrict__ z, long long n, int *__restrict__ err)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int ci = (int)floor(x[p]) - 3, cj = (int)floor(y[p]) - 3;
    if (ci < 0 || ci >= ap.nx || cj < 0 || cj >= ap.ny || !(z[p] >= 1.0 && z[p] < 2.0)) atomicOr(err, 1);
}
__global__ __launch_bounds__(256) void k_fa_load64(const double *__restrict__ x, const double *__restrict__ y,
                                                   const double *__restrict__ z, const double *__restrict__ u,
                                                   const double *__restrict__ v, const double *__restrict__ w,
                                                   const int *__restrict__ flv, long long n,
                                                   const int *__restrict__ tile_of, const long long *__restrict__ off,
                                                   int *__restrict__ fill, const int *__restrict__ count, PartE64 O)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int t = tile_of[p];
    // neighbours in the caller's order usually share a cell: a stride spreads them over the bin,
    // so that the lanes of a wave do not add to one LDS address (1000003 is prime: a permutation
    // unless it divides their count)
    const long long m = count[t], r = atomicAdd(&fill[t], 1);
    const long long o = off[t] + (m % 1000003 ? r * 1000003 % m : r);
    const double fx = floor(x[p]), fy = floor(y[p]), fz = floor(z[p]);
    O.p.cs[o] = (uint32_t)((int)fx - 3) | ((uint32_t)((int)fy - 3) << 16) | ((uint32_t)(flv[p] == 2 ? 1 : 0) << 31);
    O.p.ox[o] = x[p] - fx; O.p.oy[o] = y[p] - fy; O.p.oz[o] = z[p] - fz;
    O.p.u[o] = u[p]; O.p.v[o] = v[p]; O.p.w[o] = w[p];
    O.id[o] = (int)p;
}

template <typename R, int T, int BS, int WAVES>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void k_fa_adjoint(GridP g, TileP tp, AdjP ap, const R *__restrict__ Ex,
                                                   const R *__restrict__ Ey, const R *__restrict__ Ez,
                                                   const R *__restrict__ Bx, const R *__restrict__ By,
                                                   const R *__restrict__ Bz, const double *__restrict__ Ebx,
                                                   const double *__restrict__ Eby, const double *__restrict__ Ebz,
                                                   const long long *__restrict__ base, const int *__restrict__ cnt,
                                                   typename FaState<R>::T st, const int *__restrict__ dst, EPart<R> ain,
                                                   EPart<R> aout, double *__restrict__ gEx,
                                                   double *__restrict__ gEy, double *__restrict__ gEz,
                                                   double *__restrict__ gBx, double *__restrict__ gBy,
                                                   double *__restrict__ gBz)
{
    constexpr int W = T + 5, WW = W * W;
    constexpr int N1 = T + 1, NN = N1 * N1;
    constexpr int MB = 18;
    constexpr bool kF64 = sizeof(R) == 8;
    __shared__ typename V4<R>::T sC[6 * T * T];
    __shared__ R sJb[3 * WW];
    // FP64: an LDS FP32 atomic add runs at about 1/8 the rate of an FP64 one on
    // gfx950 (0.33 vs 2.6 lanes per CU per clock); the 32 x 32 tile keeps FP32,
    // whose FP64 window would not fit beside its corner staging in 160 KB
    using GA = typename std::conditional<(T <= 16), double, float>::type;
    __shared__ GA sG[6 * NN];
    __shared__ int sStart[MB + 1], sVs[MB];
    __shared__ unsigned sSrc[MB];
    const int tile = tile_remap(tp, blockIdx.x);
    const int tx = tile % tp.ntx, ty = tile / tp.ntx;
    const int cx0 = tx * T - 2, cy0 = ty * T - 2;
    const int mx = g.mx;
    const int iw = 1 + tx * T, jw = 1 + ty * T;
    const int nsp = tp.nsp, NV = nsp * 9;
    if ((int)threadIdx.x < NV) {
        int s, d;
        vbin_of(threadIdx.x, nsp, s, d);
        sSrc[threadIdx.x] = (unsigned)base[tile * tp.NB + s * 9 + d];
        sVs[threadIdx.x] = s;
    }
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int v = 0; v < NV; v++) {
            int s, d;
            vbin_of(v, nsp, s, d);
            sStart[v] = acc;
            acc += cnt[tile * tp.NB + s * 9 + d];
        }
        sStart[NV] = acc;
    }
    stage_corners<R, T, BS>(g, tx, ty, Ex, Ey, Ez, Bx, By, Bz, sC);
    const R js = (R)(-ap.jscale);
    for (int e = threadIdx.x; e < WW; e += BS) {
        const long long o = (long long)(iw + e % W - 1) + (long long)mx * (jw + e / W - 1);
        sJb[e] = js * (R)Ebx[o];
        sJb[WW + e] = js * (R)Eby[o];
        sJb[2 * WW + e] = js * (R)Ebz[o];
    }
    for (int e = threadIdx.x; e < 6 * NN; e += BS) sG[e] = (GA)0;
    __syncthreads();
    const int total = sStart[NV];
    // software pipeline: the next particle's state and output slot are loaded
    // while the current one is processed; the current one's incoming adjoint
    // (whose address is its output slot) is loaded first and used only after
    // the recomputed forward push
    // bin of position k: the last v < NV with sStart[v] <= k (an empty bin shares
    // its start with the next one).  A fixed-depth search with no loop: a loop
    // inside the particle loop makes the compiler wait for every outstanding
    // load before entering it, which would undo the pipelining.
    static_assert(MB <= 32, "bin search depth");
    auto slot_of = [&](int k, unsigned &slot, int &s) {
        int v = 0;
#pragma unroll
        for (int step = 16; step >= 1; step >>= 1) {
            const int c = v + step;
            const int sv = sStart[c < NV ? c : NV - 1];
            v = ((c < NV) & (sv <= k)) ? c : v;
        }
        slot = sSrc[v] + (unsigned)(k - sStart[v]);
        s = sVs[v];
    };
    AdjRec<R> nxt{};
    if ((int)threadIdx.x < total) {
        slot_of(threadIdx.x, nxt.slot, nxt.s);
        load_rec(st, dst, nxt);
    }
    // the loads below are unconditional (clamped indices): a load under a branch
    // makes the compiler wait for all outstanding loads where the paths join
    for (int k = (int)threadIdx.x; k < total; k += BS) {
        const AdjRec<R> cur = nxt;
        const int t = cur.to >= 0 ? cur.to : 0;
        // z is not stored in the 2-D split form (kZMid): no adjoint flows through it
        const R a[6] = {ain.ox[t], ain.oy[t], kF64 ? ain.oz[t] : (R)0, ain.u[t], ain.v[t], ain.w[t]};
        slot_of(k + BS < total ? k + BS : k, nxt.slot, nxt.s);
        load_rec(st, dst, nxt);
        int ii0 = cur.ci - cx0, jj0 = cur.cj - cy0;
        // a particle the forward checks excluded goes through the same
        // instructions on a clamped cell and contributes zeros (no branch: see above)
        const bool ok = ii0 >= 2 && ii0 <= T + 1 && jj0 >= 2 && jj0 <= T + 1 && cur.to >= 0;
        ii0 = min(max(ii0, 2), T + 1);
        jj0 = min(max(jj0, 2), T + 1);
        const int lc = (jj0 - 2) * T + (ii0 - 2);
        const typename V4<R>::T gc[6] = {sC[6 * lc], sC[6 * lc + 1], sC[6 * lc + 2], sC[6 * lc + 3], sC[6 * lc + 4], sC[6 * lc + 5]};
        PState<R> q;
        push_fwd<R>(ap, cur.s, cur.ox, cur.oy, cur.oz, cur.u, cur.v, cur.w, gc, q);
        const int e0 = jj0 * W + ii0;
        const int e2 = e0 + min(max(q.d[1], -1), 1) * W + min(max(q.d[0], -1), 1);
        const R jb1[8] = {sJb[e0], sJb[e0 + W], sJb[WW + e0], sJb[WW + e0 + 1],
                              sJb[2 * WW + e0], sJb[2 * WW + e0 + 1], sJb[2 * WW + e0 + W], sJb[2 * WW + e0 + W + 1]};
        const R jb2[8] = {sJb[e2], sJb[e2 + W], sJb[WW + e2], sJb[WW + e2 + 1],
                              sJb[2 * WW + e2], sJb[2 * WW + e2 + 1], sJb[2 * WW + e2 + W], sJb[2 * WW + e2 + W + 1]};
        const R x1b[3] = {a[0], a[1], a[2]};
        const R u1b[3] = {a[3], a[4], a[5]};
        R x0b[3], unb[3], PEb[3], PBb[3];
        reverse<R>(ap, cur.s, q, gc, jb1, jb2, x1b, u1b, x0b, unb, PEb, PBb);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            PEb[c] = ok ? PEb[c] : (R)0;
            PBb[c] = ok ? PBb[c] : (R)0;
        }
        const int n0 = (jj0 - 2) * N1 + (ii0 - 2);
        const int nc[4] = {n0, n0 + 1, n0 + N1, n0 + N1 + 1};
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const R w = ok ? q.w[m] : (R)0;
            atomicAdd(&sG[nc[m]], (GA)(w * PEb[0]));
            atomicAdd(&sG[NN + nc[m]], (GA)(w * PEb[1]));
            atomicAdd(&sG[2 * NN + nc[m]], (GA)(w * PEb[2]));
            atomicAdd(&sG[3 * NN + nc[m]], (GA)(w * PBb[0]));
            atomicAdd(&sG[4 * NN + nc[m]], (GA)(w * PBb[1]));
            atomicAdd(&sG[5 * NN + nc[m]], (GA)(w * PBb[2]));
        }
        const unsigned slot = cur.slot;
        aout.ox[slot] = ok ? x0b[0] : (R)0; aout.oy[slot] = ok ? x0b[1] : (R)0; aout.oz[slot] = kF64 && ok ? x0b[2] : (R)0;
        aout.u[slot] = ok ? unb[0] : (R)0; aout.v[slot] = ok ? unb[1] : (R)0; aout.w[slot] = ok ? unb[2] : (R)0;
    }
    __syncthreads();
    // node (gi, gj) of the tile is reference node (3 + tx T + gi, 3 + ty T + gj)
    double *gdst[6] = {gEx, gEy, gEz, gBx, gBy, gBz};
    for (int e = threadIdx.x; e < NN; e += BS) {
        const long long o = (long long)(2 + tx * T + e % N1) + (long long)mx * (2 + ty * T + e / N1);
#pragma unroll
        for (int cc = 0; cc < 6; cc++) {
            const double val = (double)sG[cc * NN + e];
            if (val != 0.0) unsafeAtomicAdd(&gdst[cc][o], val);
        }
    }
}

// Operations over the occupied slots of a bin layout, one workgroup per tile.
// mode 0: pos[id[slot]] = slot
// mode 1: aout[slot] = ain[pos[id[slot]]]          (adjoint to a new slot order)
// mode 2: du[id[slot]] = scale * ain.u[slot], ...  (adjoint to the caller's order)
template <typename R>
__global__ __launch_bounds__(256) void k_fa_slots(TileP tp, int mode, const long long *__restrict__ base,
                                                  const int *__restrict__ cnt, const int *__restrict__ id,
                                                  int *__restrict__ pos, EPart<R> ain, EPart<R> aout,
                                                  double scale, double *__restrict__ du, double *__restrict__ dv,
                                                  double *__restrict__ dw)
{
    const int tile = blockIdx.x;
    for (int b = 0; b < tp.NB; b++) {
        const long long b0 = base[tile * tp.NB + b];
        const int n = cnt[tile * tp.NB + b];
        for (int k = threadIdx.x; k < n; k += blockDim.x) {
            const long long slot = b0 + k;
            const int p = id[slot];
            if (mode == 0) {
                pos[p] = (int)slot;
            } else if (mode == 1) {
                const int o = pos[p];
                aout.ox[slot] = ain.ox[o]; aout.oy[slot] = ain.oy[o]; aout.oz[slot] = ain.oz[o];
                aout.u[slot] = ain.u[o]; aout.v[slot] = ain.v[o]; aout.w[slot] = ain.w[o];
            } else {
                du[p] = scale * (double)ain.u[slot];
                dv[p] = scale * (double)ain.v[slot];
                dw[p] = scale * (double)ain.w[slot];
            }
        }
    }
}

}  // namespace

template <typename R>
void launch_fa_adjoint(const GridP &g, const TileP &tp, const AdjP &ap, R *const E[3], R *const B[3],
                       double *const Eb[3], const long long *base, const int *cnt, typename FaState<R>::T st,
                       const int *dst, EPart<R> ain, EPart<R> aout, double *const gE[3], double *const gB[3],
                       hipStream_t s)
{
#define FA_ADJ(TT, BSZ, WV)                                                                                          \
    hipLaunchKernelGGL((k_fa_adjoint<R, TT, BSZ, WV>), dim3(tp.ntiles), dim3(BSZ), 0, s, g, tp, ap, E[0], E[1],      \
                       E[2], B[0], B[1], B[2], Eb[0], Eb[1], Eb[2], base, cnt, st, dst, ain, aout, gE[0], gE[1],     \
                       gE[2], gB[0], gB[1], gB[2])
    if constexpr (sizeof(R) == 8) {
        // FP64: the linearisation takes all registers of two waves per SIMD
        switch (tp.T) {
        case 8: FA_ADJ(8, 256, 2); break;
        case 16: FA_ADJ(16, 256, 2); break;
        default: break;
        }
    } else {
        switch (tp.T) {
        case 8: FA_ADJ(8, 256, 4); break;
        case 16: FA_ADJ(16, 256, 4); break;
        case 32: FA_ADJ(32, 512, 2); break;
        default: break;
        }
    }
#undef FA_ADJ
}

template <typename R>
void launch_fa_slots(const TileP &tp, int mode, const long long *base, const int *cnt, const int *id, int *pos,
                     EPart<R> ain, EPart<R> aout, double scale, double *du, double *dv, double *dw, hipStream_t s)
{
    hipLaunchKernelGGL(k_fa_slots<R>, dim3(tp.ntiles), dim3(256), 0, s, tp, mode, base, cnt, id, pos, ain, aout, scale,
                       du, dv, dw);
}

void launch_fa_push64(const GridP &g, const TileP &tp, const AdjP &ap, double *const E[3], double *const B[3],
                      double *const J[3], PartE64 A, PartE64 O, BinsP bins, SpillP sp, int *dst, hipStream_t s)
{
#define FA_PUSH(TT, BSZ)                                                                                             \
    hipLaunchKernelGGL((k_fa_push64<TT, BSZ>), dim3(tp.ntiles), dim3(BSZ), 0, s, g, tp, ap, E[0], E[1], E[2], B[0],  \
                       B[1], B[2], J[0], J[1], J[2], A, O, bins, sp, dst)
    if (tp.T == 8) FA_PUSH(8, 256);
    else if (tp.T == 16) FA_PUSH(16, 512);
#undef FA_PUSH
}

void launch_fa_range64(const AdjP &ap, const double *const raw[6], long long n, int *err, hipStream_t s)
{
    if (n > 0)
        hipLaunchKernelGGL(k_fa_range64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ap, raw[0], raw[1], raw[2],
                           n, err);
}

void launch_fa_load64(const AdjP &, const double *const raw[6], const int *flv, long long n, const int *tile_of,
                      const long long *off, int *fill, const int *count, PartE64 out, hipStream_t s)
{
    if (n > 0)
        hipLaunchKernelGGL(k_fa_load64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, raw[0], raw[1], raw[2],
                           raw[3], raw[4], raw[5], flv, n, tile_of, off, fill, count, out);
}

#define INST(R)                                                                                                     \
    template void launch_fa_adjoint<R>(const GridP &, const TileP &, const AdjP &, R *const[3], R *const[3],        \
                                       double *const[3], const long long *, const int *, FaState<R>::T, const int *, \
                                       EPart<R>, EPart<R>, double *const[3], double *const[3], hipStream_t);        \
    template void launch_fa_slots<R>(const TileP &, int, const long long *, const int *, const int *, int *, EPart<R>, \
                                     EPart<R>, double, double *, double *, double *, hipStream_t);
INST(float)
INST(double)
#undef INST

}  // namespace pictor
