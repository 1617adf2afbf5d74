// kernels_push3d.hip -- 3-D tile-local Boris push + zigzag deposit + binning (gfx950).
//
// Same structure as the 2-D kernels (kernels_push.hip) on T x T x T tiles:
// node-centred E and B of the window staged in LDS (the reference's 8-corner
// VecE/VecB, movdep_routines.F90:6-223, corner nn of cell (i,j,k) is node
// (i + a, j + b, k + c), nn = 1 + a + 2b + 4c), the 12-value zigzag deposit of
// movdep.F90:187-234 into an LDS current window, the exchange of
// loadprtlout.F90:22-97 with its z rules, and 27 arrival bins per tile.
//
// The loop is that of the 2-D kernels (one prefetched particle, its bin kept between
// iterations, one LDS add for both halves of a move inside a cell).  The split form's deposit
// makes one component's counts at a time: 75 instead of 91 VGPRs and 51 KB of LDS let three
// workgroups share a CU instead of two.  128^3, 33.5M particles: push 684 -> 622 us (18.5 ps
// per particle; VALU 74 %, LDS 72 % of the cycles); 48 x 40 x 32 in FP64 (tile 4): 60 -> 53 us.
#include "pictor_common.h"
#include "push_common.h"

namespace pictor {
namespace {
using namespace pushdev;

// ---------------------------------------------------------------------------
// FP64 form, 3-D.  Gather window: nodes [i0-1, i0+T+1] (particles may sit one
// cell into a ghost layer after the exchange); current window [i0-2, i0+T+2].
// ---------------------------------------------------------------------------
template <int T, int BS, bool BC, bool TAG = false>
__global__ __launch_bounds__(BS) void k_push3d_f64(GridP g, PhysP ph, TileP tp, const double *__restrict__ Ex,
                                                   const double *__restrict__ Ey, const double *__restrict__ Ez,
                                                   const double *__restrict__ Bx, const double *__restrict__ By,
                                                   const double *__restrict__ Bz, double *__restrict__ Jx,
                                                   double *__restrict__ Jy, double *__restrict__ Jz, PartF64 A,
                                                   PartF64 Bo, BinsP bins, PartF64 spill, SpillP sp)
{
    constexpr int WN = T + 3, WN3 = WN * WN * WN;   // gather nodes
    constexpr int WJ = T + 5, WJ3 = WJ * WJ * WJ;   // current nodes
    __shared__ double sN[6][WN3];
    __shared__ double sJ[3][WJ3];
    __shared__ int sStart[28];
    __shared__ long long sSrc[27], sDstBase[27];
    __shared__ int sDstCap[27], sDstBin[27], sCnt[27];

    if (sp.stop && *sp.stop < sp.step) return;
    const int tile = tile_remap(tp, blockIdx.x);
    const int tx = tile % tp.ntx, ty = (tile / tp.ntx) % tp.nty, tz = tile / (tp.ntx * tp.nty);
    const int i0 = 3 + tx * T, j0 = 3 + ty * T, k0 = 3 + tz * T;   // first cell of the tile
    const int tid = threadIdx.x;
    const int mx = g.mx;
    const long long mxy = (long long)g.mx * g.my;

    int bcnt = 0;
    if (tid < 27) {
        const int b = tile * tp.NB + tid;
        bcnt = bins.cnt_in[b];
        sSrc[tid] = bins.base[b];
        const int ddx = tid % 3 - 1, ddy = (tid / 3) % 3 - 1, ddz = tid / 9 - 1;
        const int dt = (wrap_tile(tz + ddz, tp.ntz) * tp.nty + wrap_tile(ty + ddy, tp.nty)) * tp.ntx +
                       wrap_tile(tx + ddx, tp.ntx);
        const int db = dt * tp.NB + tid;
        sDstBin[tid] = db;
        sDstBase[tid] = bins.base[db];
        sDstCap[tid] = bins.cap[db];
        sCnt[tid] = 0;
    }
    if (tid < 64) bin_starts(bcnt, 27, sStart);
    const double bx0 = ph.bext[0], by0 = ph.bext[1], bz0 = ph.bext[2];
    for (int e = tid; e < WN3; e += BS) {
        const int ii = e % WN, jj = (e / WN) % WN, kk = e / (WN * WN);
        const long long o = fidx(g, i0 - 1 + ii, j0 - 1 + jj, k0 - 1 + kk);
        const long long oi = o - 1, oj = o - mx, ok = o - mxy;
        sN[0][e] = (Ex[oi] + Ex[o]) * 0.5;
        sN[1][e] = (Ey[oj] + Ey[o]) * 0.5;
        sN[2][e] = (Ez[ok] + Ez[o]) * 0.5;
        sN[3][e] = (Bx[oj - mxy] + Bx[ok] + Bx[oj] + Bx[o]) * 0.25 + bx0;
        sN[4][e] = (By[oi - mxy] + By[oi] + By[ok] + By[o]) * 0.25 + by0;
        sN[5][e] = (Bz[oi - mx] + Bz[oi] + Bz[oj] + Bz[o]) * 0.25 + bz0;
    }
    for (int e = tid; e < WJ3; e += BS) { sJ[0][e] = 0.0; sJ[1][e] = 0.0; sJ[2][e] = 0.0; }
    __syncthreads();

    const double c = ph.c, sqc = ph.sqc, cinv = ph.cinv, qi = ph.qi;
    const int total = sStart[27];
    // position k lies in bin `bin` while k < binEnd, at slot k + binOff; a thread's k only grows
    int bin = 0, binEnd = sStart[1];
    long long binOff = sSrc[0];
    auto load = [&](int k, RecF64 &r) {
        if (k >= binEnd) {
            bin = bin_of<27>(k, sStart, 27);
            binEnd = sStart[bin + 1];
            binOff = sSrc[bin] - sStart[bin];
        }
        const long long src = binOff + k;
        r.x = A.x[src]; r.y = A.y[src]; r.z = A.z[src];
        r.u = A.u[src]; r.v = A.v[src]; r.w = A.w[src];
        r.q = A.q[src]; r.flv = A.flv[src];
        if (TAG) r.tag = A.tag[src];
    };
    RecF64 cur;
    if (tid < total) load(tid, cur);
    settle(cur.x, cur.y, cur.z, cur.u, cur.v, cur.w, cur.q, cur.flv);
    for (int base = 0; base < total; base += BS) {
        const int k = base + tid;
        const bool active = k < total;
        RecF64 nxt;
        load(min(k + BS, total - 1), nxt);   // prefetch the next particle of this thread
        double x0 = 0, y0 = 0, z0 = 0, un = 0, vn = 0, wn = 0, q = 0;
        double xn = 0, yn = 0, zn = 0;
        int flv = 0, d = -1, tg = 0;
        if (active) {
            x0 = cur.x; y0 = cur.y; z0 = cur.z;
            un = cur.u; vn = cur.v; wn = cur.w;
            q = cur.q; flv = cur.flv;
            if (TAG) tg = cur.tag;
            const int ip0 = (int)x0, jp0 = (int)y0, kp0 = (int)z0;
            // node-window coordinates of the cell (origin i0-1)
            const int gi = ip0 - (i0 - 1), gj = jp0 - (j0 - 1), gk = kp0 - (k0 - 1);
            xn = x0; yn = y0; zn = z0;   // a particle refused below stays where it is
            if (gi < 0 || gi > T + 1 || gj < 0 || gj > T + 1 || gk < 0 || gk > T + 1 || flv < 1 || flv > ph.nflvr) {
                flag_error(sp, kErrBounds);
                d = 13;
            } else {
                const double dx = x0 - ip0, dy = y0 - jp0, dz = z0 - kp0;
                double wt[8];
#pragma unroll
                for (int cn = 0; cn < 8; cn++) {
                    const double fx = (cn & 1) ? dx : 1.0 - dx;
                    const double fy = (cn & 2) ? dy : 1.0 - dy;
                    const double fz = (cn & 4) ? dz : 1.0 - dz;
                    wt[cn] = fx * fy * fz;
                }
                const int e0 = (gk * WN + gj) * WN + gi;
                double pf[6];
#pragma unroll
                for (int cc = 0; cc < 6; cc++) {
                    double a = 0.0;
#pragma unroll
                    for (int cn = 0; cn < 8; cn++)
                        a = a + wt[cn] * sN[cc][e0 + (cn & 1) + ((cn >> 1) & 1) * WN + (cn >> 2) * WN * WN];
                    pf[cc] = a;
                }
                const double qm = ph.flvrqm[flv - 1] * 0.5;
                double pEx = pf[0] * qm, pEy = pf[1] * qm, pEz = pf[2] * qm;
                double pBx = pf[3] * qm, pBy = pf[4] * qm, pBz = pf[5] * qm;
                double u0 = c * un + pEx;
                double v0 = c * vn + pEy;
                double w0 = c * wn + pEz;
                double gg = 1.0 / sqrt(sqc + u0 * u0 + v0 * v0 + w0 * w0);
                pBx = gg * pBx; pBy = gg * pBy; pBz = gg * pBz;
                const double f = 2.0 / (1.0 + pBx * pBx + pBy * pBy + pBz * pBz);
                const double u1 = (u0 + v0 * pBz - w0 * pBy) * f;
                const double v1 = (v0 + w0 * pBx - u0 * pBz) * f;
                const double w1 = (w0 + u0 * pBy - v0 * pBx) * f;
                u0 = u0 + v1 * pBz - w1 * pBy + pEx;
                v0 = v0 + w1 * pBx - u1 * pBz + pEy;
                w0 = w0 + u1 * pBy - v1 * pBx + pEz;
                un = u0 * cinv; vn = v0 * cinv; wn = w0 * cinv;
                gg = sqc / sqrt(sqc + u0 * u0 + v0 * v0 + w0 * w0);
                xn = x0 + un * gg * ph.inv_dx;
                yn = y0 + vn * gg * ph.inv_dy;
                zn = z0 + wn * gg * ph.inv_dz;
                const int ip = (int)xn, jp = (int)yn, kp = (int)zn;
                const double xr = dmin((double)(min(ip0, ip) + 1), dmax((double)max(ip0, ip), 0.5 * (x0 + xn)));
                const double yr = dmin((double)(min(jp0, jp) + 1), dmax((double)max(jp0, jp), 0.5 * (y0 + yn)));
                const double zr = dmin((double)(min(kp0, kp) + 1), dmax((double)max(kp0, kp), 0.5 * (z0 + zn)));
                const double qthis = q * qi;
                const double Fx[2] = {qthis * (xr - x0), qthis * (xn - xr)};
                const double Fy[2] = {qthis * (yr - y0), qthis * (yn - yr)};
                const double Fz[2] = {qthis * (zr - z0), qthis * (zn - zr)};
                const double Wx[2] = {0.5 * (x0 + xr) - ip0, 0.5 * (xn + xr) - ip};
                const double Wy[2] = {0.5 * (y0 + yr) - jp0, 0.5 * (yn + yr) - jp};
                const double Wz[2] = {0.5 * (z0 + zr) - kp0, 0.5 * (zn + zr) - kp};
                // a particle that stays in its cell deposits both halves on the same nodes: one
                // LDS add for their sum
                const bool cross = ip != ip0 || jp != jp0 || kp != kp0;
                constexpr int sy = WJ, sz = WJ * WJ;
                const int ea = ((kp0 - (k0 - 2)) * WJ + (jp0 - (j0 - 2))) * WJ + (ip0 - (i0 - 2));
                const int eb = ((kp - (k0 - 2)) * WJ + (jp - (j0 - 2))) * WJ + (ip - (i0 - 2));
                // F (1 - P, P) x (1 - Q, Q) on the nodes 0, sp, sq, sp + sq of a component
                auto deposit = [&](double *w, const double *F, const double *P, const double *Q, int sp_, int sq_) {
                    double v[2][4];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const double l = F[h] * (1.0 - P[h]), u = F[h] * P[h];
                        v[h][0] = l * (1.0 - Q[h]); v[h][1] = u * (1.0 - Q[h]); v[h][2] = l * Q[h]; v[h][3] = u * Q[h];
                    }
                    if (!cross) {
#pragma unroll
                        for (int m = 0; m < 4; m++) v[0][m] = v[0][m] + v[1][m];
                    }
                    atomicAdd(w + ea, v[0][0]); atomicAdd(w + ea + sp_, v[0][1]);
                    atomicAdd(w + ea + sq_, v[0][2]); atomicAdd(w + ea + sp_ + sq_, v[0][3]);
                    if (cross) {
                        atomicAdd(w + eb, v[1][0]); atomicAdd(w + eb + sp_, v[1][1]);
                        atomicAdd(w + eb + sq_, v[1][2]); atomicAdd(w + eb + sp_ + sq_, v[1][3]);
                    }
                };
                // Jx(i, j..j+1, k..k+1), Jy(i..i+1, j, k..k+1), Jz(i..i+1, j..j+1, k)
                deposit(sJ[0], Fx, Wy, Wz, sy, sz);
                deposit(sJ[1], Fy, Wx, Wz, 1, sz);
                deposit(sJ[2], Fz, Wx, Wy, 1, sy);
                // EnforceBC_PostMovDep (bc.F90:238-287)
                bool keep = true;
                if (BC) keep = particle_faces<double>(ph, g, xn, yn, zn, un, vn);
                // periodic exchange, loadprtlout.F90:31-96 (3-D rules); a face of a
                // non-periodic axis sends to a null neighbour (the particle is gone)
                bool sent = false;
                if (keep) {
                    if (xn < ph.xmin) {
                        if ((yn <= (ph.ymax + ph.xmin - xn)) && (yn >= (ph.ymin - ph.xmin + xn)) &&
                            (zn <= (ph.zmax + ph.xmin - xn)) && (zn >= (ph.zmin - ph.xmin + xn))) {
                            if (BC && !g.per[0]) keep = false; else xn = xn + ph.xlen;
                            sent = true;
                        }
                    } else if (xn > ph.xmax) {
                        if ((yn <= (ph.ymax - ph.xmax + xn)) && (yn >= (ph.ymin + ph.xmax - xn)) &&
                            (zn <= (ph.zmax - ph.xmax + xn)) && (zn >= (ph.zmin + ph.xmax - xn))) {
                            if (BC && !g.per[0]) keep = false; else xn = xn - ph.xlen;
                            sent = true;
                        }
                    }
                }
                if (keep && !sent) {
                    if (yn < ph.ymin) {
                        if ((yn < (ph.ymin - ph.xmin + xn)) && (yn < (ph.ymin + ph.xmax - xn)) &&
                            (zn >= (ph.zmin - ph.ymin + yn)) && (zn <= (ph.zmax + ph.ymin - yn))) {
                            if (BC && !g.per[1]) keep = false; else yn = yn + ph.ylen;
                            sent = true;
                        }
                    } else if (yn > ph.ymax) {
                        if ((yn > (ph.ymax + ph.xmin - xn)) && (yn > (ph.ymax - ph.xmax + xn)) &&
                            (zn >= (ph.zmin + ph.ymax - yn)) && (zn <= (ph.zmax - ph.ymax + yn))) {
                            if (BC && !g.per[1]) keep = false; else yn = yn - ph.ylen;
                            sent = true;
                        }
                    }
                }
                if (keep && !sent) {
                    if (zn < ph.zmin) {
                        if ((zn < (ph.zmin - ph.xmin + xn)) && (zn < (ph.zmin + ph.xmax - xn)) &&
                            (zn < (ph.zmin - ph.ymin + yn)) && (zn < (ph.zmin + ph.ymax - yn))) {
                            if (BC && !g.per[2]) keep = false; else zn = zn + ph.zlen;
                        }
                    } else if (zn > ph.zmax) {
                        if ((zn > (ph.zmax + ph.xmin - xn)) && (zn > (ph.zmax - ph.xmax + xn)) &&
                            (zn > (ph.zmax + ph.ymin - yn)) && (zn > (ph.zmax - ph.ymax + yn))) {
                            if (BC && !g.per[2]) keep = false; else zn = zn - ph.zlen;
                        }
                    }
                }
                if (keep) {
                    int cx = (int)xn - 3, cy = (int)yn - 3, cz = (int)zn - 3;
                    cx = cx < 0 ? 0 : (cx > g.nx - 1 ? g.nx - 1 : cx);
                    cy = cy < 0 ? 0 : (cy > g.ny - 1 ? g.ny - 1 : cy);
                    cz = cz < 0 ? 0 : (cz > g.nz - 1 ? g.nz - 1 : cz);
                    const int ddx = norm_dir(cx / T - tx, tp.ntx), ddy = norm_dir(cy / T - ty, tp.nty);
                    const int ddz = norm_dir(cz / T - tz, tp.ntz);
                    if (ddx < -1 || ddx > 1 || ddy < -1 || ddy > 1 || ddz < -1 || ddz > 1) {
                        flag_error(sp, kErrBounds);
                        d = 13;
                    } else {
                        d = (ddx + 1) + 3 * (ddy + 1) + 9 * (ddz + 1);
                    }
                }
            }
        }
        const int slot = reserve_slot(d, 13, sCnt);
        settle(nxt.x, nxt.y, nxt.z, nxt.u, nxt.v, nxt.w, nxt.q, nxt.flv);
        if (active && d >= 0) {
            if (slot < sDstCap[d]) {
                const long long o = sDstBase[d] + slot;
                Bo.x[o] = xn; Bo.y[o] = yn; Bo.z[o] = zn;
                Bo.u[o] = un; Bo.v[o] = vn; Bo.w[o] = wn;
                Bo.q[o] = q; Bo.flv[o] = flv;
                if (TAG) Bo.tag[o] = tg;
            } else {
                const int s = spill_slot(sp);
                if (s < sp.cap) {
                    spill.x[s] = xn; spill.y[s] = yn; spill.z[s] = zn;
                    spill.u[s] = un; spill.v[s] = vn; spill.w[s] = wn;
                    spill.q[s] = q; spill.flv[s] = flv;
                    if (TAG) spill.tag[s] = tg;
                } else {
                    flag_error(sp, kErrCapacity);
                }
            }
        }
        cur = nxt;
    }
    __syncthreads();
    for (int e = tid; e < WJ3; e += BS) {
        const long long o = fidx(g, i0 - 2 + e % WJ, j0 - 2 + (e / WJ) % WJ, k0 - 2 + e / (WJ * WJ));
        const double a = sJ[0][e], b = sJ[1][e], cz = sJ[2][e];
        if (a != 0.0) unsafeAtomicAdd(&Jx[o], a);
        if (b != 0.0) unsafeAtomicAdd(&Jy[o], b);
        if (cz != 0.0) unsafeAtomicAdd(&Jz[o], cz);
    }
    if (tid < 27) bins.cnt_out[sDstBin[tid]] = min(sCnt[tid], sDstCap[tid]);
}

// ---------------------------------------------------------------------------
// FP32 split form, 3-D.  Particles always sit inside their tile: gather nodes
// [i0, i0+T], current window [i0-1, i0+T+1].
// ---------------------------------------------------------------------------
struct SplitRec3 {
    int cell;
    float ox, oy, oz, u, v, w;
    int id;     // tag (TAG)
    float wq;   // charge weight (WQ)
};

template <int T, int BS, bool BC, bool TAG = false, bool WQ = false>
__global__ __launch_bounds__(BS) void k_push3d_split(GridP g, PhysP ph, TileP tp, const float *__restrict__ Ex,
                                                     const float *__restrict__ Ey, const float *__restrict__ Ez,
                                                     const float *__restrict__ Bx, const float *__restrict__ By,
                                                     const float *__restrict__ Bz, double *__restrict__ Jx,
                                                     double *__restrict__ Jy, double *__restrict__ Jz, PartSplit A,
                                                     PartSplit Bo, BinsP bins, PartSplit spill, SpillP sp)
{
#pragma clang fp contract(fast)
    constexpr int WN = T + 1, WN3 = WN * WN * WN;
    constexpr int WJ = T + 3, WJ3 = WJ * WJ * WJ;
    constexpr int MB = 54;   // species (<= 2) x 27 directions
    constexpr int kLogT = T == 4 ? 2 : 3;
    // node e: sNa[e] = (Ex, Ey, Ez, Bx), sNb[e] = (By, Bz); 24 B per node keeps the LDS of a
    // tile-8 workgroup under a third of the CU's
    __shared__ float4 sNa[WN3];
    __shared__ float2 sNb[WN3];
    __shared__ unsigned long long sJ[3][WJ3];
    __shared__ int sStart[MB + 1], sVs[MB];
    __shared__ unsigned sSrc[MB], sDstBase[MB];
    __shared__ int sDstCap[MB], sDstBin[MB], sCnt[MB];

    if (sp.stop && *sp.stop < sp.step) return;
    const int tile = tile_remap(tp, blockIdx.x);
    const int tx = tile % tp.ntx, ty = (tile / tp.ntx) % tp.nty, tz = tile / (tp.ntx * tp.nty);
    const int i0 = 3 + tx * T, j0 = 3 + ty * T, k0 = 3 + tz * T;
    const int tid = threadIdx.x;
    const int mx = g.mx, nx = g.nx, ny = g.ny, nz = g.nz;
    const long long mxy = (long long)g.mx * g.my;
    const bool edge = tx == 0 || ty == 0 || tz == 0 || tx == tp.ntx - 1 || ty == tp.nty - 1 || tz == tp.ntz - 1;
    const int nsp = tp.nsp, NV = nsp * 27;

    int bcnt = 0;
    if (tid < NV) {
        // virtual bins: centre bins of every species first, then the 26 others
        int s, d;
        if (tid < nsp) { s = tid; d = 13; }
        else { const int r = tid - nsp; s = r / 26; const int q = r % 26; d = q < 13 ? q : q + 1; }
        bcnt = bins.cnt_in[tile * tp.NB + s * 27 + d];
        sSrc[tid] = (unsigned)bins.base[tile * tp.NB + s * 27 + d];
        sVs[tid] = s;
        const int ds = tid / 27, dd = tid % 27;
        const int ddx = dd % 3 - 1, ddy = (dd / 3) % 3 - 1, ddz = dd / 9 - 1;
        const int dt = (wrap_tile(tz + ddz, tp.ntz) * tp.nty + wrap_tile(ty + ddy, tp.nty)) * tp.ntx +
                       wrap_tile(tx + ddx, tp.ntx);
        const int db = dt * tp.NB + ds * 27 + dd;
        sDstBin[tid] = db;
        sDstBase[tid] = (unsigned)bins.base[db];
        sDstCap[tid] = bins.cap[db];
        sCnt[tid] = 0;
    }
    if (tid < 64) bin_starts(bcnt, NV, sStart);
    const float bx0 = (float)ph.bext[0], by0 = (float)ph.bext[1], bz0 = (float)ph.bext[2];
    for (int e = tid; e < WN3; e += BS) {
        const int ii = e % WN, jj = (e / WN) % WN, kk = e / (WN * WN);
        const long long o = fidx(g, i0 + ii, j0 + jj, k0 + kk);
        const long long oi = o - 1, oj = o - mx, ok = o - mxy;
        sNa[e] = make_float4((Ex[oi] + Ex[o]) * 0.5f, (Ey[oj] + Ey[o]) * 0.5f, (Ez[ok] + Ez[o]) * 0.5f,
                             (Bx[oj - mxy] + Bx[ok] + Bx[oj] + Bx[o]) * 0.25f + bx0);
        sNb[e] = make_float2((By[oi - mxy] + By[oi] + By[ok] + By[o]) * 0.25f + by0,
                             (Bz[oi - mx] + Bz[oi] + Bz[oj] + Bz[o]) * 0.25f + bz0);
    }
    for (int e = tid; e < WJ3; e += BS) { sJ[0][e] = 0ull; sJ[1][e] = 0ull; sJ[2][e] = 0ull; }
    __syncthreads();

    const float c = (float)ph.c, sqc = (float)ph.sqc, cinv = (float)ph.cinv;
    const float idx_ = (float)ph.inv_dx, idy_ = (float)ph.inv_dy, idz_ = (float)ph.inv_dz;
    // q/m / 2 and the charge pre-scaled by 2^30 (exact) for the fixed-point current
    const float qm0 = (float)(ph.flvrqm[0] * 0.5), qm1 = (float)(ph.flvrqm[1] * 0.5);
    const float qs0 = (float)(ph.flvq[0] * kFixScale), qs1 = (float)(ph.flvq[1] * kFixScale);
    const int total = sStart[NV];

    // position k lies in bin `bin` while k < binEnd, at slot k + binOff; a thread's k only grows
    int bin = 0, binEnd = sStart[1], spc = sVs[0];
    unsigned binOff = sSrc[0];
    auto load = [&](int k, SplitRec3 &r) {
        if (k >= binEnd) {
            bin = bin_of<MB>(k, sStart, NV);
            binEnd = sStart[bin + 1];
            binOff = sSrc[bin] - (unsigned)sStart[bin];
            spc = sVs[bin];
        }
        const unsigned off = (binOff + (unsigned)k) * 4u;
        r.cell = ldo(A.cell, off);
        r.ox = ldo(A.ox, off); r.oy = ldo(A.oy, off); r.oz = ldo(A.oz, off);
        r.u = ldo(A.u, off); r.v = ldo(A.v, off); r.w = ldo(A.w, off);
        if (TAG) r.id = ldo(A.id, off);
        if (WQ) r.wq = ldo(A.wq, off);
    };

    SplitRec3 cur;
    if (tid < total) load(tid, cur);
    settle(cur.cell, cur.ox, cur.oy, cur.oz, cur.u, cur.v, cur.w);
    for (int base = 0; base < total; base += BS) {
        const int k = base + tid;
        const bool active = k < total;
        const int spn = spc;   // the species of `cur`
        SplitRec3 nxt;
        load(min(k + BS, total - 1), nxt);   // prefetch the next particle of this thread
        int d = -1, ncell;
        float ox, oy, oz, un, vn, wn;
        if (active) {
            int ci, cj, ck;
            cell_unpack(3, cur.cell, ci, cj, ck);
            const int gi = ci - (i0 - 3), gj = cj - (j0 - 3), gk = ck - (k0 - 3);   // 0..T-1 inside the tile
            if (gi < 0 || gi >= T || gj < 0 || gj >= T || gk < 0 || gk >= T) {
                flag_error(sp, kErrBounds);
                d = spn * 27 + 13;
                ncell = cur.cell;
                ox = cur.ox; oy = cur.oy; oz = cur.oz; un = cur.u; vn = cur.v; wn = cur.w;
            } else {
                const float x0 = cur.ox, y0 = cur.oy, z0 = cur.oz;
                const float qm = spn ? qm1 : qm0, qsp = spn ? qs1 : qs0, qs = WQ ? qsp * cur.wq : qsp;
                float wt[8];
#pragma unroll
                for (int cn = 0; cn < 8; cn++)
                    wt[cn] = ((cn & 1) ? x0 : 1.0f - x0) * ((cn & 2) ? y0 : 1.0f - y0) * ((cn & 4) ? z0 : 1.0f - z0);
                const int e0 = (gk * WN + gj) * WN + gi;
                float pE[3] = {0.f, 0.f, 0.f}, hB[3] = {0.f, 0.f, 0.f};
#pragma unroll
                for (int cn = 0; cn < 8; cn++) {
                    const int e = e0 + (cn & 1) + ((cn >> 1) & 1) * WN + (cn >> 2) * WN * WN;
                    const float4 a = sNa[e];
                    const float2 b = sNb[e];
                    pE[0] += wt[cn] * a.x; pE[1] += wt[cn] * a.y; pE[2] += wt[cn] * a.z;
                    hB[0] += wt[cn] * a.w; hB[1] += wt[cn] * b.x; hB[2] += wt[cn] * b.y;
                }
                const float pEx = pE[0] * qm, pEy = pE[1] * qm, pEz = pE[2] * qm;
                float u0 = c * cur.u + pEx;
                float v0 = c * cur.v + pEy;
                float w0 = c * cur.w + pEz;
                float gg = __builtin_amdgcn_rsqf(sqc + u0 * u0 + v0 * v0 + w0 * w0);
                const float pBx = gg * hB[0] * qm, pBy = gg * hB[1] * qm, pBz = gg * hB[2] * qm;
                const float f = 2.0f * __builtin_amdgcn_rcpf(1.0f + pBx * pBx + pBy * pBy + pBz * pBz);
                const float u1 = (u0 + v0 * pBz - w0 * pBy) * f;
                const float v1 = (v0 + w0 * pBx - u0 * pBz) * f;
                const float w1b = (w0 + u0 * pBy - v0 * pBx) * f;
                u0 = u0 + v1 * pBz - w1b * pBy + pEx;
                v0 = v0 + w1b * pBx - u1 * pBz + pEy;
                w0 = w0 + u1 * pBy - v1 * pBx + pEz;
                un = u0 * cinv; vn = v0 * cinv; wn = w0 * cinv;
                gg = sqc * __builtin_amdgcn_rsqf(sqc + u0 * u0 + v0 * v0 + w0 * w0);
                const float x1 = x0 + un * gg * idx_;
                const float y1 = y0 + vn * gg * idy_;
                const float z1 = z0 + wn * gg * idz_;
                int di = (int)floorf(x1), dj = (int)floorf(y1), dk = (int)floorf(z1);
                const float xr = fminf((float)(min(0, di) + 1), fmaxf((float)max(0, di), 0.5f * (x0 + x1)));
                const float yr = fminf((float)(min(0, dj) + 1), fmaxf((float)max(0, dj), 0.5f * (y0 + y1)));
                const float zr = fminf((float)(min(0, dk) + 1), fmaxf((float)max(0, dk), 0.5f * (z0 + z1)));
                const float Fx[2] = {qs * (xr - x0), qs * (x1 - xr)};
                const float Fy[2] = {qs * (yr - y0), qs * (y1 - yr)};
                const float Fz[2] = {qs * (zr - z0), qs * (z1 - zr)};
                const float Wx[2] = {0.5f * (x0 + xr), 0.5f * (x1 + xr) - (float)di};
                const float Wy[2] = {0.5f * (y0 + yr), 0.5f * (y1 + yr) - (float)dj};
                const float Wz[2] = {0.5f * (z0 + zr), 0.5f * (z1 + zr) - (float)dk};
                const bool cross = (di != 0) || (dj != 0) || (dk != 0);
                constexpr int sy = WJ, sz = WJ * WJ;
                const int ea = ((gk + 1) * WJ + (gj + 1)) * WJ + (gi + 1);
                const int eb = ((gk + 1 + dk) * WJ + (gj + 1 + dj)) * WJ + (gi + 1 + di);
                // F (1 - P, P) x (1 - Q, Q) on the nodes 0, sp, sq, sp + sq of a component, as counts;
                // one component at a time keeps few of them in registers
                auto deposit = [&](unsigned long long *w, const float *F, const float *P, const float *Q, int sp_, int sq_) {
                    int v[2][4];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const float l = F[h] * (1.0f - P[h]), u = F[h] * P[h];
                        v[h][0] = quanti(l * (1.0f - Q[h])); v[h][1] = quanti(u * (1.0f - Q[h]));
                        v[h][2] = quanti(l * Q[h]); v[h][3] = quanti(u * Q[h]);
                    }
                    long long t[4] = {v[0][0], v[0][1], v[0][2], v[0][3]};
                    if (!cross) {
#pragma unroll
                        for (int m = 0; m < 4; m++) t[m] += v[1][m];
                    }
                    atomicAdd(w + ea, (unsigned long long)t[0]); atomicAdd(w + ea + sp_, (unsigned long long)t[1]);
                    atomicAdd(w + ea + sq_, (unsigned long long)t[2]); atomicAdd(w + ea + sp_ + sq_, (unsigned long long)t[3]);
                    if (cross) {
                        atomicAdd(w + eb, (unsigned long long)(long long)v[1][0]);
                        atomicAdd(w + eb + sp_, (unsigned long long)(long long)v[1][1]);
                        atomicAdd(w + eb + sq_, (unsigned long long)(long long)v[1][2]);
                        atomicAdd(w + eb + sp_ + sq_, (unsigned long long)(long long)v[1][3]);
                    }
                };
                deposit(sJ[0], Fx, Wy, Wz, sy, sz);
                deposit(sJ[1], Fy, Wx, Wz, 1, sz);
                deposit(sJ[2], Fz, Wx, Wy, 1, sy);
                ox = x1 - (float)di;
                if (ox >= 1.0f) { ox = 0.0f; di += 1; }
                oy = y1 - (float)dj;
                if (oy >= 1.0f) { oy = 0.0f; dj += 1; }
                oz = z1 - (float)dk;
                if (oz >= 1.0f) { oz = 0.0f; dk += 1; }
                if (BC) {
                    // the boundary faces on the FP64 position; a reflected coordinate is
                    // split again into cell and offset
                    int nci = ci + di, ncj = cj + dj, nck = ck + dk;
                    double X = 3.0 + (double)nci + (double)ox, Y = 3.0 + (double)ncj + (double)oy;
                    const double Z = 3.0 + (double)nck + (double)oz;
                    const double X0 = X, Y0 = Y;
                    bool keep = particle_faces<float>(ph, g, X, Y, Z, un, vn);
                    if (keep && X != X0) {
                        const double f = floor(X);
                        nci = (int)f - 3;
                        ox = (float)(X - f);
                        if (ox >= 1.0f) { ox = 0.0f; nci += 1; }
                    }
                    if (keep && Y != Y0) {
                        const double f = floor(Y);
                        ncj = (int)f - 3;
                        oy = (float)(Y - f);
                        if (oy >= 1.0f) { oy = 0.0f; ncj += 1; }
                    }
                    if ((nci < 0 || nci >= nx) && !g.per[0]) keep = false;
                    if ((ncj < 0 || ncj >= ny) && !g.per[1]) keep = false;
                    if ((nck < 0 || nck >= nz) && !g.per[2]) keep = false;
                    if (keep) {
                        nci = nci < 0 ? nci + nx : (nci >= nx ? nci - nx : nci);
                        ncj = ncj < 0 ? ncj + ny : (ncj >= ny ? ncj - ny : ncj);
                        nck = nck < 0 ? nck + nz : (nck >= nz ? nck - nz : nck);
                        ncell = cell_pack(3, nci, ncj, nck);
                        const int ddx = norm_dir(nci / T - tx, tp.ntx), ddy = norm_dir(ncj / T - ty, tp.nty);
                        const int ddz = norm_dir(nck / T - tz, tp.ntz);
                        d = spn * 27 + (ddx + 1) + 3 * (ddy + 1) + 9 * (ddz + 1);
                    }
                } else {
                    // |di|, |dj|, |dk| <= 1: the destination is this tile or a neighbour, given by
                    // the cell counted from the tile's corner (-1 .. T); only the tiles at the edge
                    // of the box have cells to wrap
                    ncell = cur.cell + di + dj * (1 << 11) + dk * (1 << 22);
                    if (edge) {
                        int nci = ci + di, ncj = cj + dj, nck = ck + dk;
                        nci = nci < 0 ? nci + nx : (nci >= nx ? nci - nx : nci);
                        ncj = ncj < 0 ? ncj + ny : (ncj >= ny ? ncj - ny : ncj);
                        nck = nck < 0 ? nck + nz : (nck >= nz ? nck - nz : nck);
                        ncell = cell_pack(3, nci, ncj, nck);
                    }
                    d = spn * 27 + 13 + ((gi + di) >> kLogT) + 3 * ((gj + dj) >> kLogT) + 9 * ((gk + dk) >> kLogT);
                }
            }
        }
        const int slot = reserve_slot(d, __builtin_amdgcn_readfirstlane(spn) * 27 + 13, sCnt);
        settle(nxt.cell, nxt.ox, nxt.oy, nxt.oz, nxt.u, nxt.v, nxt.w);
        if (active && d >= 0) {
            if (slot < sDstCap[d]) {
                const unsigned off = (sDstBase[d] + (unsigned)slot) * 4u;
                sto(Bo.cell, off, ncell); sto(Bo.ox, off, ox); sto(Bo.oy, off, oy); sto(Bo.oz, off, oz);
                sto(Bo.u, off, un); sto(Bo.v, off, vn); sto(Bo.w, off, wn);
                if (TAG) sto(Bo.id, off, cur.id);
                if (WQ) sto(Bo.wq, off, cur.wq);
            } else {
                const int si = spill_slot(sp);
                if (si < sp.cap) {
                    spill.cell[si] = ncell; spill.ox[si] = ox; spill.oy[si] = oy; spill.oz[si] = oz;
                    spill.u[si] = un; spill.v[si] = vn; spill.w[si] = wn; spill.sp[si] = spn;
                    if (TAG) spill.id[si] = cur.id;
                    if (WQ) spill.wq[si] = cur.wq;
                } else {
                    flag_error(sp, kErrCapacity);
                }
            }
        }
        cur = nxt;
    }
    __syncthreads();
    if (tid < NV) bins.cnt_out[sDstBin[tid]] = min(sCnt[tid], sDstCap[tid]);
    constexpr double lim = kFixLimit * kFixScale;
    bool big = false;
    for (int e = tid; e < WJ3; e += BS) {
        const long long o = fidx(g, i0 - 1 + e % WJ, j0 - 1 + (e / WJ) % WJ, k0 - 1 + e / (WJ * WJ));
        const double a = (double)(long long)sJ[0][e], b = (double)(long long)sJ[1][e];
        const double cz = (double)(long long)sJ[2][e];
        big = big || fabs(a) >= lim || fabs(b) >= lim || fabs(cz) >= lim;
        if (a != 0.0) unsafeAtomicAdd(&Jx[o], a);
        if (b != 0.0) unsafeAtomicAdd(&Jy[o], b);
        if (cz != 0.0) unsafeAtomicAdd(&Jz[o], cz);
    }
    if (big) flag_error(sp, kErrPrecision);
}

}  // namespace

// the kernel variant for the boundary faces (BC) and carried tags (TAG) of this context
#define PICK_BC_TAG(K, bc, tag, ...)                                                                                \
    do {                                                                                                           \
        if (bc) { if (tag) K(true, true, __VA_ARGS__); else K(true, false, __VA_ARGS__); }                           \
        else { if (tag) K(false, true, __VA_ARGS__); else K(false, false, __VA_ARGS__); }                            \
    } while (0)

// the split form's variant for the faces (BC), carried tags (TAG) and charge weights (WQ)
#define PICK_BC_TAG_WQ(K, bc, tag, wq, ...)                                                                         \
    do {                                                                                                           \
        if (wq) {                                                                                                  \
            if (bc) { if (tag) K(true, true, true, __VA_ARGS__); else K(true, false, true, __VA_ARGS__); }           \
            else { if (tag) K(false, true, true, __VA_ARGS__); else K(false, false, true, __VA_ARGS__); }            \
        } else {                                                                                                   \
            if (bc) { if (tag) K(true, true, false, __VA_ARGS__); else K(true, false, false, __VA_ARGS__); }         \
            else { if (tag) K(false, true, false, __VA_ARGS__); else K(false, false, false, __VA_ARGS__); }          \
        }                                                                                                          \
    } while (0)

void launch_push3d_f64(int T, const GridP &g, const PhysP &ph, const TileP &tp, double *const E[3],
                       double *const B[3], double *const J[3], PartF64 A, PartF64 Bo, BinsP bins, PartF64 spill,
                       SpillP sp, hipStream_t s)
{
    dim3 grid(tp.ntiles);
#define K3_F64(BCV, TAGV, TT, BSZ)                                                                                 \
    hipLaunchKernelGGL((k_push3d_f64<TT, BSZ, BCV, TAGV>), grid, dim3(BSZ), 0, s, g, ph, tp, E[0], E[1], E[2], B[0], \
                       B[1], B[2], J[0], J[1], J[2], A, Bo, bins, spill, sp)
    const bool bc = ph.pbc_on != 0, tag = A.tag != nullptr;
    switch (T) {
    case 4: PICK_BC_TAG(K3_F64, bc, tag, 4, 256); break;
    case 8: PICK_BC_TAG(K3_F64, bc, tag, 8, 1024); break;
    default: break;
    }
#undef K3_F64
}

void launch_push3d_split(int T, const GridP &g, const PhysP &ph, const TileP &tp, float *const E[3],
                         float *const B[3], double *const J[3], PartSplit A, PartSplit Bo, BinsP bins,
                         PartSplit spill, SpillP sp, hipStream_t s)
{
    dim3 grid(tp.ntiles);
#define K3_SPLIT(BCV, TAGV, WQV, TT, BSZ)                                                                          \
    hipLaunchKernelGGL((k_push3d_split<TT, BSZ, BCV, TAGV, WQV>), grid, dim3(BSZ), 0, s, g, ph, tp, E[0], E[1],      \
                       E[2], B[0], B[1], B[2], J[0], J[1], J[2], A, Bo, bins, spill, sp)
    const bool bc = ph.pbc_on != 0, tag = A.id != nullptr, wq = A.wq != nullptr;
    switch (T) {
    case 4: PICK_BC_TAG_WQ(K3_SPLIT, bc, tag, wq, 4, 256); break;
    case 8: PICK_BC_TAG_WQ(K3_SPLIT, bc, tag, wq, 8, 512); break;
    default: break;
    }
#undef K3_SPLIT
}
#undef PICK_BC_TAG
#undef PICK_BC_TAG_WQ

}  // namespace pictor
