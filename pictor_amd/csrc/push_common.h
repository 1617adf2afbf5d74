// push_common.h -- device helpers shared by the 2-D and 3-D push kernels.
#pragma once
#include "pictor_common.h"

namespace pictor {
namespace pushdev {

__device__ inline double dmin(double a, double b) { return (b < a) ? b : a; }
__device__ inline double dmax(double a, double b) { return (b > a) ? b : a; }

// an error of this step, and a spilled particle: both stop the steps enqueued behind it
__device__ inline void flag_error(const SpillP &sp, int bits)
{
    atomicOr(sp.err, bits);
    if (sp.stop) atomicMin(sp.stop, sp.step);
}
__device__ inline int spill_slot(const SpillP &sp)
{
    if (sp.stop) atomicMin(sp.stop, sp.step);
    return atomicAdd(sp.count, 1);
}

// Bin of position k (0 <= k < sStart[n]) among n bins laid end to end: the last b < n with
// sStart[b] <= k (an empty bin shares its start with the next).  A search of fixed depth (5 or 6
// LDS reads) for the 27-direction bins of the 3-D layout, where a linear walk from the first bin
// takes up to 53 steps; the 2-D kernels, whose centre bins come first, keep the walk.
template <int NMAX>
__device__ inline int bin_of(int k, const int *sStart, int n)
{
    constexpr int top = NMAX > 32 ? 32 : NMAX > 16 ? 16 : NMAX > 8 ? 8 : NMAX > 4 ? 4 : NMAX > 2 ? 2 : 1;
    static_assert(NMAX <= 64, "bin search depth");
    int b = 0;
#pragma unroll
    for (int step = top; step >= 1; step >>= 1) {
        const int c = b + step;
        const int sv = sStart[c < n ? c : n - 1];
        b = ((c < n) & (sv <= k)) ? c : b;
    }
    return b;
}

// Reservation of slots in the LDS counters of the destinations; every lane of the wave
// must call it (d = -1 for idle lanes).  The lanes of the wave's usual destination `home`
// (wave-uniform: the tile's own bin) take consecutive slots from one add by their first
// lane; the few that leave the tile add for themselves, in the same LDS instruction.
__device__ inline int reserve_slot(int d, int home, int *sCnt)
{
    const bool stay = d == home;
    const unsigned long long m = __ballot(stay);
    const unsigned rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    int b = 0;
    if (d >= 0 && (!stay || rank == 0u)) b = atomicAdd(&sCnt[d], stay ? __popcll(m) : 1);
    const int b0 = __builtin_amdgcn_readlane(b, m ? __ffsll(m) - 1 : 0);
    return stay ? b0 + (int)rank : b;
}

// a particle of the FP64 form as loaded
struct RecF64 {
    double x, y, z, u, v, w, q;
    int flv, tag;
};

// Wait for the loads that fill `r`..., before the stores that follow in program order: loads
// and stores share one counter, so a wait placed after them would last until they are done.
template <typename... T>
__device__ inline void settle(T &...r)
{
    (..., [](auto &v) { asm volatile("" : "+v"(v) : : "memory"); }(r));
}

// sStart[v] for v = 0..n from the counts `cnt` of the bins v = lane < n (n < 64), by one wave
__device__ inline void bin_starts(int cnt, int n, int *sStart)
{
    const int lane = (int)__lane_id();
    int acc = lane < n ? cnt : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(acc, o);
        if (lane >= o) acc += up;
    }
    if (lane < n) sStart[lane + 1] = acc;
    if (lane == 0) sStart[0] = 0;
}

__device__ inline int wrap_tile(int t, int n)
{
    return (t < 0) ? t + n : (t >= n ? t - n : t);
}

__device__ inline int norm_dir(int dd, int n)
{
    if (dd > 1) dd -= n;
    else if (dd < -1) dd += n;
    return dd;
}

// FP32 -> exact integer count of 2^-30 units (the argument is already scaled by 2^30;
// |v| < 2^31, so one conversion)
__device__ inline int quanti(float v) { return (int)__builtin_rintf(v); }

// F * W, a product in FP64, as a count: rounded to the nearest integer (ties to even) by adding
// 1.5 * 2^52, whose sum's bit pattern minus the constant's is that integer for |F W| < 2^51.
constexpr double kCountBias = 6755399441055744.0;
constexpr unsigned long long kCountBits = 0x4338000000000000ull;
__device__ inline unsigned long long count_of(double F, double W)
{
    return (unsigned long long)__double_as_longlong(F * W + kCountBias) - kCountBits;
}

// The two zigzag half-segments of the 2-D split form (movdep.F90:177-237)
// from the old offsets (x0, y0, kZMid) to the new position as stored: offsets
// (ox, oy) in the cell displaced by (di, dj), each -1, 0 or 1, z advanced to z1.
// Evaluated in FP64, every relay point, flux F and weight W is exact for FP32
// inputs (F up to its product with the charge) and each node value is rounded
// once to a 2^-30 count, so the deposited Jx, Jy carry exactly the charge moved
// between the stored positions up to that last rounding.  qs: charge times 2^30.
// Index 0: the first half-segment (nodes of the old cell), 1: the second (nodes
// of the new cell).  The node counts are left to jx, jy, jz, so that a kernel
// holds one component's at a time.
struct Zigzag {
    double Fx[2], Fy[2], Fz[2], Wx[2], Wy[2];

    __device__ Zigzag(double qs, float x0, float y0, float ox, float oy, float z1, int di, int dj)
    {
        // relay point: the midpoint, or the face that was crossed
        auto relay = [](double p0, double p1, int d) { return d == 0 ? 0.5 * (p0 + p1) : (d > 0 ? 1.0 : 0.0); };
        const double X0 = x0, Y0 = y0, Z0 = kZMid;
        const double dx = di, dy = dj;
        const double X1 = (double)ox + dx, Y1 = (double)oy + dy, Z1 = z1;
        const double xr = relay(X0, X1, di), yr = relay(Y0, Y1, dj);
        const double zr = relay(Z0, Z1, z1 < 0.0f ? -1 : (z1 >= 1.0f ? 1 : 0));
        Fx[0] = qs * (xr - X0); Fy[0] = qs * (yr - Y0); Fz[0] = qs * (zr - Z0);
        Fx[1] = qs * (X1 - xr); Fy[1] = qs * (Y1 - yr); Fz[1] = qs * (Z1 - zr);
        Wx[0] = 0.5 * (X0 + xr); Wy[0] = 0.5 * (Y0 + yr);
        Wx[1] = __builtin_fma(0.5, X1 + xr, -dx); Wy[1] = __builtin_fma(0.5, Y1 + yr, -dy);
    }
    // counts at (i, j), (i, j+1)
    __device__ void jx(int h, unsigned long long n[2]) const
    {
        n[0] = count_of(Fx[h], 1.0 - Wy[h]); n[1] = count_of(Fx[h], Wy[h]);
    }
    // counts at (i, j), (i+1, j)
    __device__ void jy(int h, unsigned long long n[2]) const
    {
        n[0] = count_of(Fy[h], 1.0 - Wx[h]); n[1] = count_of(Fy[h], Wx[h]);
    }
    // counts at (i, j), (i+1, j), (i, j+1), (i+1, j+1)
    __device__ void jz(int h, unsigned long long n[4]) const
    {
        const double lo = Fz[h] * (1.0 - Wx[h]), hi = Fz[h] * Wx[h], Vy = 1.0 - Wy[h];
        n[0] = count_of(lo, Vy); n[1] = count_of(hi, Vy); n[2] = count_of(lo, Wy[h]); n[3] = count_of(hi, Wy[h]);
    }
};

// EnforceBC_PostMovDep (bc.F90:238-287) on one pushed particle, in the
// reference's order: the reflecting faces top, bottom, right, left
// (RefBC_Prtl_*, bc_reflect.F90:76-186: specular image 2 x_w - x with the
// normal momentum reversed, only where the wall lies inside the array), then
// every face again in order x lo .. z hi, reflecting once more (which changes
// nothing then) or removing the particle beyond a 'remv' face (bc_open.F90).
// Positions are the reference's local coordinates.  Returns false when the
// particle is removed.  The current of a reflected particle is folded back by
// the face kernels after the push.
template <typename R>
__device__ inline bool particle_faces(const PhysP &ph, const GridP &g, double &x, double &y, double z, R &u, R &v)
{
    const int *t = ph.pbc;
    const double *p = ph.pbc_pos;
    auto top = [&]() { if (p[3] < g.my - 1 && y > p[3]) { v = -v; y = 2.0 * p[3] - y; } };
    auto bottom = [&]() { if (p[2] > 1 && y < p[2]) { v = -v; y = 2.0 * p[2] - y; } };
    auto right = [&]() { if (p[1] < g.mx - 1 && x > p[1]) { u = -u; x = 2.0 * p[1] - x; } };
    auto left = [&]() { if (p[0] > 1 && x < p[0]) { u = -u; x = 2.0 * p[0] - x; } };
    if (t[3] == kBcRefl) top();
    if (t[2] == kBcRefl) bottom();
    if (t[1] == kBcRefl) right();
    if (t[0] == kBcRefl) left();
    if (t[0] == kBcRefl) left();
    else if (t[0] == kBcRemv && x < p[0]) return false;
    if (t[1] == kBcRefl) right();
    else if (t[1] == kBcRemv && x > p[1]) return false;
    if (t[2] == kBcRefl) bottom();
    else if (t[2] == kBcRemv && y < p[2]) return false;
    if (t[3] == kBcRefl) top();
    else if (t[3] == kBcRemv && y > p[3]) return false;
    if (t[4] == kBcRemv && z < p[4]) return false;
    if (t[5] == kBcRemv && z > p[5]) return false;
    return true;
}

// byte-offset accessors: a uniform base plus a 32-bit lane offset lets the
// compiler use SGPR-base addressing (one VALU op per access)
template <typename T>
__device__ inline T ldo(const T *base, unsigned off)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + off);
}
template <typename T>
__device__ inline void sto(T *base, unsigned off, T v)
{
    *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + off) = v;
}


}  // namespace pushdev
}  // namespace pictor
