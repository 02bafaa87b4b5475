// advec_mom (advec_mom_kernel.f90:29-428) for one sweep and all three
// velocity components, as one kernel that keeps every intermediate on chip.
//
// Per sweep along axis s the reference forms, node by node,
//   node_flux     nf(n)  = 0.125 * (8 mass fluxes around n)
//   node_mass_post  mp(n) = 0.125 * (8 x density1 * post_vol of the cells around n)
//   node_mass_pre   mq(n) = mp(n) - nf(n-s) + nf(n)
//   mom_flux      F(f)   = advec_vel_s(f) * nf(f)      (face f between n and n+s)
//   vel(n) <- (vel(n) * mq(n) + F(n-s) - F(n)) / mp(n)
// and needs, for node n, nf at n-2s..n+s, mp at n-s..n+s and vel at n-2s..n+2s.
// The per-call path stores nf, mp, mq and mom_flux in work arrays; here
// every value is formed once, in registers, with the same expression and
// operand order (so the FP64 form's results are bit-identical; the FP32 form
// runs the same expressions in FP32), and shared with the neighbours that
// need it:
//   * lanes of a wavefront lie along x (coalesced rows); neighbours along x
//     come from lane shifts (x sweep) or LDS;
//   * the waves of a workgroup lie along the second axis; a neighbour row is
//     read from LDS (double-buffered, one barrier per plane).  Wave 0 is the
//     halo row and stores nothing;
//   * the workgroup marches along the third axis, keeping the previous
//     planes' values in registers.
// The y and z sweeps march along the sweep axis itself, so the +-2 window
// along s is a register pipeline; the x sweep marches along z and takes its
// +-2 window from the lanes (60 of 64 lanes store).
//
// Each face's momentum flux is formed once (the per-call kernel, like the
// reference, forms mom_flux once per face too) and each input element is
// read about once, instead of the 8 density/volume reads per node mass and
// 16 mass-flux reads per pair of node fluxes of a plain per-node kernel.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "batch.h"
#include "fast.h"
#include "launch.h"

namespace clover {

// waves per workgroup (wave 0 is the halo row) of the x (DIR 1), y (2) and
// z (3) sweeps: the y/z marches run faster in 4-wave workgroups despite the
// larger share of halo rows, the x sweep in 8-wave ones
constexpr int mw_of(int dir) { return dir == 1 ? 8 : 4; }

template <typename S>
struct Vel3 {
    const S *in[3];
    S *out[3];
};

// post_vol of advec_mom_kernel.f90:95-163 for the sweep `mode`:
// 1 sweep 1 along x (formed in mom_x_body), 2 sweep 1 along z, 3 sweep 2 with
// advect_x, 4 sweep 2 without, 5 and 6 sweep 3
template <typename S>
// (dxt: the offset of the column vol_flux_y and vol_flux_z are read at, on a
// mirrored x face, launch.h tan_xm)
__device__ inline S mom_post_vol(int mode, const Lay &g, int i, S V0, const S *__restrict__ vfx,
                                 const S *__restrict__ vfy, const S *__restrict__ vfz, int dxt)
{
#define D(x) (x)
    const int t = i + dxt;
    switch (mode) {
    case 2: return V0 + D(vfx[i + 1]) - D(vfx[i]) + D(vfy[t + g.ld]) - D(vfy[t]);
    case 3: return V0 + D(vfz[t + g.plane]) - D(vfz[t]);
    case 4: return V0 + D(vfx[i + 1]) - D(vfx[i]);
    default: return V0;
    }
#undef D
}

// momentum flux through the face between nodes n and n+s
// (advec_mom_kernel.f90:213-249 and its y/z twins); vm1..vp2 are the
// velocity at n-s, n, n+s, n+2s; sigma is |nf| / node_mass_pre(donor); d the
// node spacing along the sweep (rd: the same as a divisor), r6: 6 as a divisor
template <typename T>
__device__ inline T mom_face_flux(T nf, T sigma, T d, const Recip &rd, const Recip &r6, T vm1, T v0, T vp1, T vp2)
{
    T upwind, donor, downwind;
    if (nf < (T)0) {
        upwind = vp2; donor = vp1; downwind = v0;
    } else {
        upwind = vm1; donor = v0; downwind = vp1;
    }
    const T width = d;
    const T vdiffuw = donor - upwind;
    const T vdiffdw = downwind - donor;
    T limiter = 0;
    if (vdiffuw * vdiffdw > (T)0) {
        const T auw = fabs(vdiffuw);
        const T adw = fabs(vdiffdw);
        T wind = 1;
        if (vdiffdw <= (T)0) wind = -1;
        limiter = wind * tmin(tmin(by_const<T>(width * (by_const<T>(((T)2 - sigma) * adw, rd) +
                                                        by_const<T>(((T)1 + sigma) * auw, rd)),
                                               r6),
                                   auw),
                              adw);
    }
    const T advec_vel_s = donor + ((T)1 - sigma) * limiter;
    return advec_vel_s * nf;
}

template <typename T>
__device__ inline T face_sigma(T nf, T mq_lo, T mq_hi)
{
    return quo(fabs(nf), nf < (T)0 ? mq_hi : mq_lo);
}

// A value and its neighbours: one column along x (-1 in the y and z sweeps; in
// the x sweep +1 for mass fluxes, -1 for cell masses), one down the wave axis, both.
template <typename T>
struct Quad {
    T c, x, w, xw;
};

// The loads of one plane, kept raw so that they can be issued a plane ahead
// (after the barrier of the plane in hand) and consumed by the next plane:
// the sweep's mass flux, density1 and the volume fluxes post_vol needs.
template <typename S>
struct Raw {
    S a, rho, v0, v1, v2, v3;  // storage type: converted where used, so the loads stay in flight
};

// dxc: offset of the density read (a mirrored x face, launch.h cell_xm);
// dxt: of the vol_flux_y and vol_flux_z reads (tan_xm); dma: of the mass
// flux read (the same in the y and z sweeps, whose mass fluxes follow
// tan_xm too)
template <typename S>
__device__ inline Raw<S> load_raw(int mode, const Lay &g, int i, bool ok_a, bool ok_p, const S *__restrict__ mf,
                                  const S *__restrict__ vfx, const S *__restrict__ vfy, const S *__restrict__ vfz,
                                  const S *__restrict__ density1, int dxc, int dxt, int dma)
{
    Raw<S> r{0, 0, 0, 0, 0, 0};
    if (ok_a) r.a = mf[i + dma];
    if (ok_p) {
        r.rho = density1[i + dxc];
        const int t = i + dxt;
        switch (mode) {
        case 2: r.v0 = vfx[i + 1]; r.v1 = vfx[i]; r.v2 = vfy[t + g.ld]; r.v3 = vfy[t]; break;
        case 3: r.v0 = vfz[t + g.plane]; r.v1 = vfz[t]; break;
        case 4: r.v0 = vfx[i + 1]; r.v1 = vfx[i]; break;
        default: break;
        }
    }
    return r;
}

// density1 * post_vol with mom_post_vol's expression order
template <typename S>
__device__ inline S raw_cell_mass(int mode, S V0, const Raw<S> &r, bool ok_p)
{
    if (!ok_p) return 0;
    S pv;
    switch (mode) {
    case 2: pv = V0 + r.v0 - r.v1 + r.v2 - r.v3; break;
    case 3:
    case 4: pv = V0 + r.v0 - r.v1; break;
    default: pv = V0; break;
    }
    return r.rho * pv;
}

__device__ inline double shfl_d(double x, int src) { return __shfl(x, src, 64); }
__device__ inline float shfl_d(float x, int src) { return __shfl(x, src, 64); }

// ---------------------------------------------------------------------------
// y and z sweeps: lanes along x on 64 line-aligned columns, all of which
// store; lane 0 also loads and publishes column j-1, which the first column's
// node needs.  (A 63-column layout with lane 0 as the j-1
// halo read rows that straddle cache lines: measured at 512^3 the aligned
// one runs FP32 mom_y 1.35 -> 1.28 ms and mom_z 1.33 -> 1.20 ms, FP64 the
// same.)  Waves lie along the other axis; the workgroup marches along the
// sweep axis.
//
// In (x, m = sweep axis, w = wave axis) offsets both sweeps have the same
// node flux (advec_mom_kernel.f90:260-265 for y, 345-350 for z):
//   nf(m) = 0.125*(f(-1,0,0)+f(0,0,0)+f(-1,1,0)+f(0,1,0)+f(-1,0,-1)+f(0,0,-1)+f(-1,1,-1)+f(0,1,-1))
// and node_mass_post (advec_mom_kernel.f90:267-275, 352-360) sums the cells
// (dj,dk,dl) = (0,-1,0),(0,0,0),(-1,-1,0),(-1,0,0),(0,-1,-1),(0,0,-1),(-1,-1,-1),(-1,0,-1),
// which is a different order in (x, m, w) for the two sweeps.
template <int DIR, typename T>
__device__ inline T march_node_flux(const Quad<T> &f0, const Quad<T> &f1)
{
    return (T)0.125 * (f0.x + f0.c + f1.x + f1.c + f0.xw + f0.w + f1.xw + f1.w);
}

template <int DIR, typename T>
__device__ inline T march_node_mass(const Quad<T> &pm, const Quad<T> &p0)  // cell planes m-1, m
{
    if (DIR == 2)  // k = m, l = w
        return (T)0.125 * (pm.c + p0.c + pm.x + p0.x + pm.w + p0.w + pm.xw + p0.xw);
    // DIR == 3: k = w, l = m
    return (T)0.125 * (p0.w + p0.c + p0.xw + p0.x + pm.w + pm.c + pm.xw + pm.x);
}

// The last x tile of a sweep holds the node columns left over by the
// 64-column tiles: one (x_max+1) on a mesh a multiple of 64 cells wide.  In
// the lane-along-x layout its workgroups march every plane with one live
// lane, and at 512^3 they held 1/9 of the launch's workgroup slots (the y and
// z sweeps ran 8 % faster on 511^3, whose nodes fill 8 tiles).  In the FP64
// form a tail of one column (a mesh a multiple of 64 cells wide) is marched
// instead with lanes along the wave axis: one wave per column and 63 rows (lane
// 0 is the halo row), each lane loading both x neighbours itself and taking the
// row below from lane-1, in the grid's first workgroups (mom_march).  Every value is
// formed by the same expressions from the same operands as in the 64-column
// layout.  Measured at 512^3 FP64: mom_y 2.38 -> 2.32 ms, mom_z 2.26 -> 2.22
// ms; 640^3 as 8 tiles (320^3 tiles, one tail column in six tiles): the
// batched momentum launches 4.41 -> 4.16 ms.  The FP32 form keeps the
// 64-column layout: there the tail's loads (a line per lane, 4 bytes used)
// cost more than the slots save (mom_y 1.29 -> 1.35 ms, mom_z 1.20 -> 1.25
// ms, batched 2.29 -> 2.64 ms).
constexpr int kTailCols = 1;  // 4 columns at 131x75x93 ran mom_y 28.0 -> 33.7 us, mom_z 29.2 -> 36.0
static_assert(kTailCols <= mw_of(2) && kTailCols <= mw_of(3), "the tail's waves fit in the tile's workgroups");

__host__ __device__ inline int mom_tail_cols(const Lay &g, int gx)
{
    const int tw = g.x_max - g.x_min + 2 - 64 * (gx - 1);  // node columns of the last x tile
    return tw <= kTailCols ? tw : 0;
}

// The tail's waves march at most about kTailPlanes planes of a chunk each
// (nsub pieces of the chunk, as many as the tile's workgroups hold), so
// that they end with the chunk's 64-column workgroups.
constexpr int kTailPlanes = 16;

struct TailSplit {
    int tw, nrg, nsub, tb;  // columns, row groups, pieces per chunk, workgroups per chunk
};

template <int DIR>
__device__ inline TailSplit mom_tail_split(const Lay &g, const Blk &bk, int tw)
{
    constexpr int MW = mw_of(DIR);
    const int nrow = DIR == 3 ? g.y_max - g.y_min + 2 : g.z_max - g.z_min + 2;  // storing rows
    const int npos = DIR == 3 ? g.z_max - g.z_min + 2 : g.y_max - g.y_min + 2;  // march positions
    TailSplit t;
    t.tw = tw;
    t.nrg = (nrow + 62) / 63;
    const int per = (npos + bk.gz - 1) / bk.gz;  // chunk_range's chunk length
    t.nsub = max(1, min((per + kTailPlanes - 1) / kTailPlanes, bk.gy * MW / (tw * t.nrg)));
    t.tb = (tw * t.nrg * t.nsub + MW - 1) / MW;  // <= bk.gy: tw * nrg <= MW * ceil(nrow / (MW-1))
    return t;
}

// The tail: one wave's columns, a lane per row (no barrier on this path)
template <int DIR, typename S>
__device__ __forceinline__ void mom_tail_body(const Blk &bk, TailSplit ts, Lay g, Geo geo, int mode,
                                              const S *__restrict__ mf, const S *__restrict__ vfx,
                                              const S *__restrict__ vfy, const S *__restrict__ vfz,
                                              const S *__restrict__ density1, Vel3<S> v)
{
    using T = S;  // arithmetic type of the form
    constexpr int MW = mw_of(DIR);
    const int lane = threadIdx.x, w = threadIdx.y;
    const int sM = DIR == 3 ? g.plane : g.ld;
    const int wmin = DIR == 3 ? g.y_min : g.z_min, wmax = DIR == 3 ? g.y_max : g.z_max;
    const int mmin = DIR == 3 ? g.z_min : g.y_min, mmax = DIR == 3 ? g.z_max : g.y_max;
    const T d = (T)(DIR == 3 ? geo.dz : geo.dy);
    const Recip rd = DIR == 3 ? geo.rz : geo.ry;
    const T V0 = (T)geo.vol;

    int m0, m1;
    chunk_range(bk, mmin, mmax + 1, m0, m1);
    // wave item: piece fastest, then row group (rows wmin..wmax+1 store), then column
    const int item = bk.y * MW + w;
    if (item >= ts.tw * ts.nrg * ts.nsub) return;
    const int sub = item % ts.nsub, rest = item / ts.nsub;
    const int j = g.x_min + 64 * (bk.gx - 1) + rest / ts.nrg;
    const int wp = wmin - 1 + (rest % ts.nrg) * 63 + lane;
    const int len = (m1 - m0 + 1 + ts.nsub - 1) / ts.nsub;
    m0 += sub * len;
    m1 = min(m0 + len - 1, m1);
    if (m0 > m1) return;
    // j >= x_min-1 and wp >= wmin-1 always; upper limits of the arrays read:
    // cells and the sweep's mass flux end at +2 across the sweep, vertices at +3
    const bool ok_cell = j <= g.x_max + 2 && wp <= wmax + 2;
    const bool ok_cm = j - 1 <= g.x_max + 2 && wp <= wmax + 2;
    const bool store = lane >= 1 && j <= g.x_max + 1 && wp <= wmax + 1;
    const int i0 = DIR == 3 ? idx(g, j, wp, mmin) : idx(g, j, mmin, wp);  // offset at march position mmin
#define OFF(q) (i0 + ((q) - mmin) * sM)

    constexpr int MA = DIR - 1, WA = DIR == 3 ? 1 : 2;
    const int sW = DIR == 3 ? g.ld : g.plane, dwc = (cell_m(g, WA, wp) - wp) * sW;  // a mirrored row of density
    auto dmc = [&](int q) { return (cell_m(g, MA, q) - q) * sM; };                    // a mirrored plane
    const int dxc = cell_xm(g, j) - j;  // a mirrored x face: the interior cell its halo copies
    const int dxm = cell_xm(g, j - 1) - (j - 1);
    const int dxt = tan_xm(g, j) - j, dxtm = tan_xm(g, j - 1) - (j - 1);  // vol_flux_y/z, the sweep's mass flux
    // the quads of a plane: columns j-1, j of rows wp-1, wp (Quad x, c, xw, w)
    auto xchg = [&](T a, T p, T am, T pm, Quad<T> &F, Quad<T> &P) {
        const int src = lane > 0 ? lane - 1 : 0;  // lane 0 (the halo row) stores nothing
        F.c = a;
        F.x = am;
        F.w = shfl_d(a, src);
        F.xw = shfl_d(am, src);
        P.c = p;
        P.x = pm;
        P.w = shfl_d(p, src);
        P.xw = shfl_d(pm, src);
    };
    auto plane = [&](int q, Quad<T> &F, Quad<T> &P) {
        const int i = OFF(q);
        const T a = ok_cell ? (T)mf[i + dxt] : (T)0;  // q <= mmax+3: inside the sweep's face extent
        const T p = (ok_cell && q <= mmax + 2)
                        ? (T)density1[i + dxc + dwc + dmc(q)] * mom_post_vol(mode, g, i, V0, vfx, vfy, vfz, dxt)
                        : (T)0;
        const T am = ok_cm ? (T)mf[i - 1 + dxtm] : (T)0;
        const T pm = (ok_cm && q <= mmax + 2)
                         ? (T)density1[i - 1 + dxm + dwc + dmc(q)] * mom_post_vol(mode, g, i - 1, V0, vfx, vfy, vfz, dxtm)
                         : (T)0;
        xchg(a, p, am, pm, F, P);
    };
    auto vel_at = [&](int c, int q) -> T {
        const int qn = node_m(g, MA, q);
        const T x = store ? (T)v.in[c][OFF(qn)] : (T)0;
        return c == MA && qn != q ? -x : x;
    };

    Quad<T> Fa, Pa, Fb, Pb;
    // prologue: nf(m0-2..m0), node masses at m0-1, m0, m0+1, velocities m0-2..m0+1
    plane(m0 - 2, Fa, Pa);
    plane(m0 - 1, Fb, Pb);
    const T nf_m2 = march_node_flux<DIR, T>(Fa, Fb);
    const T mp_m1 = march_node_mass<DIR, T>(Pa, Pb);
    plane(m0, Fa, Pa);
    T nf_lo = march_node_flux<DIR, T>(Fb, Fa);  // nf(m-1)
    T mp0 = march_node_mass<DIR, T>(Pb, Pa);    // mp(m)
    const T mq_m1 = mp_m1 - nf_m2 + nf_lo;
    plane(m0 + 1, Fb, Pb);
    T nf0 = march_node_flux<DIR, T>(Fa, Fb);     // nf(m)
    T mp1 = march_node_mass<DIR, T>(Pa, Pb);     // mp(m+1)
    T mq0 = mp0 - nf_lo + nf0;                // mq(m)
    // Fb, Pb hold plane m+1

    T vm1[3], v0[3], vp1[3], flo[3];
    {
        const T sig = face_sigma(nf_lo, mq_m1, mq0);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const T vm2 = vel_at(c, m0 - 2);
            vm1[c] = vel_at(c, m0 - 1);
            v0[c] = vel_at(c, m0);
            vp1[c] = vel_at(c, m0 + 1);
            flo[c] = mom_face_flux(nf_lo, sig, d, rd, geo.r6, vm2, vm1[c], v0[c], vp1[c]);  // F(m0-1)
        }
    }

    // each step loads its own plane m+2 first.  Loading the next plane's
    // values one step ahead instead held them in registers across the step:
    // at 512^3 that measured FP32 mom_y 1.42 against 1.35 ms and mom_z 1.36
    // against 1.31 ms, and FP64 (125 against 95 VGPRs, four waves per SIMD
    // against five) mom_y 2.55 against 2.43 ms and mom_z 2.47 against 2.33.
    for (int m = m0; m <= m1; m++) {
        const Raw<S> rc = load_raw(mode, g, OFF(m + 2), ok_cell, ok_cell && m + 2 <= mmax + 2, mf, vfx, vfy, vfz,
                                   density1, dxc + dwc + dmc(m + 2), dxt, dxt);
        const Raw<S> rcm = load_raw(mode, g, OFF(m + 2) - 1, ok_cm, ok_cm && m + 2 <= mmax + 2, mf, vfx, vfy, vfz,
                                    density1, dxm + dwc + dmc(m + 2), dxtm, dxtm);
        T vp2[3];
#pragma unroll
        for (int c = 0; c < 3; c++) vp2[c] = vel_at(c, m + 2);
        const T a = (T)rc.a, p = raw_cell_mass(mode, V0, rc, ok_cell && m + 2 <= mmax + 2);
        const T am = (T)rcm.a, pm = raw_cell_mass(mode, V0, rcm, ok_cm && m + 2 <= mmax + 2);
        Quad<T> Fc, Pc;
        xchg(a, p, am, pm, Fc, Pc);
        const T nf1 = march_node_flux<DIR, T>(Fb, Fc);  // nf(m+1)
        const T mp2 = march_node_mass<DIR, T>(Pb, Pc);  // mp(m+2), garbage at mmax+3 (never used)
        const T mq1 = mp1 - nf0 + nf1;              // mq(m+1)
        const T sig = face_sigma(nf0, mq0, mq1);
        const int i = OFF(m);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const T fhi = mom_face_flux(nf0, sig, d, rd, geo.r6, vm1[c], v0[c], vp1[c], vp2[c]);  // F(m)
            if (store) v.out[c][i] = quo(v0[c] * mq0 + flo[c] - fhi, mp0);
            flo[c] = fhi;
            vm1[c] = v0[c];
            v0[c] = vp1[c];
            vp1[c] = vp2[c];
        }
        nf0 = nf1;
        mp0 = mp1;
        mp1 = mp2;
        mq0 = mq1;
        Fb = Fc;
        Pb = Pc;
    }
#undef OFF
}

// sign-bit mask of x in the high word of its type
__device__ inline unsigned sign_of(double x) { return (unsigned)(__builtin_bit_cast(unsigned long long, x) >> 32) & 0x80000000u; }
__device__ inline unsigned sign_of(float x) { return __builtin_bit_cast(unsigned, x) & 0x80000000u; }
__device__ inline double flip_sign(double x, unsigned m)
{
    return __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, x) ^ ((unsigned long long)m << 32));
}
__device__ inline float flip_sign(float x, unsigned m) { return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) ^ m); }

// mom_face_flux from the velocity differences d0 = v0 - vm1, d1 = vp1 - v0,
// d2 = vp2 - vp1, which successive faces share: for nf < 0 the reference's
// differences are -d2 and -d1, exactly, and only their product, magnitudes and
// the sign of the second count.  `wind` becomes a flip of the sign bit (sgn:
// the sign bit where nf < 0).
template <typename T>
__device__ inline T mom_flux_of(T nf, bool neg, unsigned sgn, T one_m, T two_m, T one_p, T d, const Recip &rd,
                                const Recip &r6, T v0, T vp1, T d0, T d1, T d2)
{
    const T du = neg ? d2 : d0;
    const T donor = neg ? vp1 : v0;
    const T auw = fabs(du), adw = fabs(d1);
    const T lim = tmin(tmin(by_const<T>(d * (by_const<T>(two_m * adw, rd) + by_const<T>(one_p * auw, rd)), r6), auw), adw);
    const T limiter = du * d1 > (T)0 ? flip_sign(lim, sign_of(d1) ^ sgn) : (T)0;
    return (donor + one_m * limiter) * nf;
}

// The 64-column layout of the y and z sweeps.  mom_tail_body's expressions
// (MODE: the sweep's post_vol, mom_post_vol), with the work per plane cut to
// what they need, since at 344 (FP64) and 253 (FP32) VALU instructions per wave
// and plane the sweeps ran at or near the VALU's rate:
//   * row addresses are scalar (the wave's row and the plane), a lane adds a
//     byte offset; lanes and planes outside the arrays read clamped ones;
//   * the march is unrolled by four, so the window of velocities, their
//     differences and the planes' quads stay in their registers;
//   * the halo row (wave 0) only loads and publishes;
//   * the prologue's planes are loaded two at a time and exchanged past one
//     barrier.
// Now 205 and 107 instructions.  The old form against this one, best shapes, one
// machine: 512^3 FP64 mom_y 2.37 -> 2.30 ms, mom_z 2.16 -> 2.15, FP32 1.24 -> 1.17
// and 1.12 -> 1.06; 256^3 FP64 0.362 -> 0.328 and 0.338 -> 0.313; 131x75x93 38.6 ->
// 28.0 and 41.8 -> 29.2 us (with the tail rule below); 64^3 18.5 -> 17.0 and
// 17.7 -> 16.9; FP32 101x143x67 20.7 -> 17.5 and 20.1 -> 16.8; 320^3 as 8 tiles,
// the three batched launches 2.13 -> 2.00 ms.  8-wave workgroups (fewer halo rows)
// were within 1.5 % at 512^3 and 12-25 % slower at 64^3 to 131x75x93.
template <int DIR, int MODE, typename S>
__device__ __forceinline__ void mom_cols_body(const Blk &bk, S (*xbuf)[2][mw_of(DIR)][65], Lay g, Geo geo,
                                              const S *__restrict__ mf, const S *__restrict__ vfx,
                                              const S *__restrict__ vfy, const S *__restrict__ vfz,
                                              const S *__restrict__ density1, Vel3<S> v)
{
    using T = S;  // arithmetic type of the form
    constexpr int MW = mw_of(DIR);
    const int lane = (int)threadIdx.x, w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int wmin = DIR == 3 ? g.y_min : g.z_min, wmax = DIR == 3 ? g.y_max : g.z_max;
    const int mmin = DIR == 3 ? g.z_min : g.y_min, mmax = DIR == 3 ? g.z_max : g.y_max;
    const T d = (T)(DIR == 3 ? geo.dz : geo.dy);
    const Recip rd = DIR == 3 ? geo.rz : geo.ry;
    const T V0 = (T)geo.vol;
    int m0, m1;
    chunk_range(bk, mmin, mmax + 1, m0, m1);
    if (m0 > m1) return;  // the whole workgroup, before any barrier
    const int j = g.x_min + bk.x * 64 + lane;
    const int wp = wmin - 1 + bk.y * (MW - 1) + w;
    const bool row = w >= 1 && wp <= wmax + 1;  // an owned row (uniform)
    const bool store = j <= g.x_max + 1;
    // cells and the sweep's mass flux end at +2 across the sweep
    const int jr = min(j, g.x_max + 2), wr = min(wp, wmax + 2);
    // byte offsets from column x_min-2: the lane's column, density's and the
    // tangential fluxes' on a mirrored x face; lane 0's column j-1 likewise
    auto off = [&](int col) { return (unsigned)(col - g.x_min + 2) * (unsigned)sizeof(S); };
    unsigned oj = off(jr), orho = off(cell_xm(g, jr)), ot = off(tan_xm(g, jr));
    const int jm = min(j - 1, g.x_max + 2);
    unsigned ojm = off(jm), orhom = off(cell_xm(g, jm)), otm = off(tan_xm(g, jm));
    // the wave's row at march position q (elements)
    const int sM = DIR == 3 ? g.plane : g.ld;
    const int row0 = DIR == 3 ? idx(g, g.x_min - 2, wr, 0) : idx(g, g.x_min - 2, 0, wr);
    auto row_at = [&](int q) { return row0 + q * sM; };
    // on a mirrored face density and the velocities are read at the interior
    // cell or node their halo copies (the component along the sweep with its
    // sign flipped): from the row at q, to that one.  The first position past
    // each face (out of reach where it is not mirrored); q below mmin: prologue.
    constexpr int MA = DIR - 1, WA = DIR == 3 ? 1 : 2;  // the march's axis and the waves'
    constexpr int far = 1 << 29;
    const int dw = (cell_m(g, WA, wr) - wr) * (DIR == 3 ? g.ld : g.plane);
    const int lo = (g.mirror >> (2 * MA)) & 1 ? mmin : -far, hi = (g.mirror >> (2 * MA)) & 2 ? mmax : far;
    auto cell_shift = [&](int q, bool pro) { return q > hi ? 2 * (hi - q) + 1 : pro && q < lo ? 2 * (lo - q) - 1 : 0; };
    auto node_shift = [&](int q, bool pro) { return q > hi + 1 ? 2 * (hi + 1 - q) : pro && q < lo ? 2 * (lo - q) : 0; };
    const int up = DIR == 3 ? g.ld : g.plane;  // to the next row across the sweep

    // the values of a plane: the sweep's mass flux, density and the volume
    // fluxes of post_vol (as stored, so that their loads can stay in flight), of
    // column j and, in lane 0, of j-1
    constexpr int NF = MODE == 2 ? 4 : MODE == 6 ? 0 : 2;
    struct Col {
        S a, rho, f[NF > 0 ? NF : 1];
    };
    struct Pl {
        Col c, m;
    };
    auto load_col = [&](Col &x, int r, int rc, int rr, unsigned o, unsigned orh, unsigned otan) {
        x.a = at(mf + r, otan);
        x.rho = at(density1 + rr, orh);
        if constexpr (MODE == 2 || MODE == 4) {
            x.f[0] = at(vfx + rc + 1, o);
            x.f[1] = at(vfx + rc, o);
        }
        if constexpr (MODE == 2) {
            x.f[2] = at(vfy + rc + up, otan);
            x.f[3] = at(vfy + rc, otan);
        }
        if constexpr (MODE == 3) {
            x.f[0] = at(vfz + rc + up, otan);
            x.f[1] = at(vfz + rc, otan);
        }
    };
    auto load = [&](int q, int r, Pl &x, bool pro) {  // r: row_at(q)
        const int qc = min(q, mmax + 2);  // mass fluxes end at mmax+3, cells at mmax+2
        const int rc = q > mmax + 2 ? r - sM : r, rr = rc + cell_shift(qc, pro) * sM + dw;
        load_col(x.c, r, rc, rr, oj, orho, ot);
        if (lane == 0) load_col(x.m, r, rc, rr, ojm, orhom, otm);
    };
    auto cell_mass = [&](const Col &x) -> T {  // mom_post_vol's expressions
        if constexpr (NF == 4) return x.rho * (V0 + x.f[0] - x.f[1] + x.f[2] - x.f[3]);
        else if constexpr (NF == 2) return x.rho * (V0 + x.f[0] - x.f[1]);
        else return x.rho * V0;
    };
    // publishes the plane's mass flux and cell mass; returns the cell mass of column j
    auto publish = [&](int b, const Pl &x) {
        const T p = cell_mass(x.c);
        xbuf[b][0][w][lane + 1] = x.c.a;
        xbuf[b][1][w][lane + 1] = p;
        if (lane == 0) {
            xbuf[b][0][w][0] = x.m.a;
            xbuf[b][1][w][0] = cell_mass(x.m);
        }
        return p;
    };
    auto gather = [&](int b, T a, T p, Quad<T> &F, Quad<T> &P) {
        F = Quad<T>{a, xbuf[b][0][w][lane], xbuf[b][0][w - 1][lane + 1], xbuf[b][0][w - 1][lane]};
        P = Quad<T>{p, xbuf[b][1][w][lane], xbuf[b][1][w - 1][lane + 1], xbuf[b][1][w - 1][lane]};
    };
    auto vel_at = [&](int c, int q, int r, bool pro) -> T {
        const int dq = node_shift(q, pro);
        const T x = at(v.in[c] + (r + dq * sM), oj);
        return c == MA ? flip_sign(x, dq ? 0x80000000u : 0u) : x;
    };

    // waves without an owned row only load and publish; the barriers are the
    // same in number: two, then one per position
    if (!row) {
        for (int q = 0; q < 4; q++) {
            Pl x;
            load(m0 - 2 + q, row_at(m0 - 2 + q), x, true);
            publish(q, x);
        }
        __syncthreads();
        __syncthreads();
        for (int m = m0; m <= m1; m++) {
            Pl x;
            load(m + 2, row_at(m + 2), x, false);
            publish((m - m0) & 1, x);
            __syncthreads();
        }
        return;
    }

    // by position mod 4 (quads mod 2): velocities, differences vel(q) = v(q+1)
    // - v(q), node flux, node masses; the momentum flux through the face below
    Quad<T> F[2], P[2];
    T vel[4][3], dv[4][3], nf[4], mp[4], mq[4], flo[3];
    {
        // two planes at a time: all four would take the kernel's registers past the march's own
        T a[4], p[4];
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
            Pl x, y;
            load(m0 - 2 + q, row_at(m0 - 2 + q), x, true);
            load(m0 - 1 + q, row_at(m0 - 1 + q), y, true);
            a[q] = x.c.a;
            p[q] = publish(q, x);
            a[q + 1] = y.c.a;
            p[q + 1] = publish(q + 1, y);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            vel[2][c] = vel_at(c, m0 - 2, row_at(m0 - 2), true);
            vel[3][c] = vel_at(c, m0 - 1, row_at(m0 - 1), true);
            vel[0][c] = vel_at(c, m0, row_at(m0), true);
            vel[1][c] = vel_at(c, m0 + 1, row_at(m0 + 1), true);
        }
        __syncthreads();
        gather(0, a[0], p[0], F[0], P[0]);
        gather(1, a[1], p[1], F[1], P[1]);
        const T nf_m2 = march_node_flux<DIR, T>(F[0], F[1]);
        const T mp_m1 = march_node_mass<DIR, T>(P[0], P[1]);
        gather(2, a[2], p[2], F[0], P[0]);
        nf[3] = march_node_flux<DIR, T>(F[1], F[0]);
        mp[0] = march_node_mass<DIR, T>(P[1], P[0]);
        const T mq_m1 = mp_m1 - nf_m2 + nf[3];
        gather(3, a[3], p[3], F[1], P[1]);
        nf[0] = march_node_flux<DIR, T>(F[0], F[1]);
        mp[1] = march_node_mass<DIR, T>(P[0], P[1]);
        mq[0] = mp[0] - nf[3] + nf[0];
        const T sig = face_sigma(nf[3], mq_m1, mq[0]);
        const bool neg = nf[3] < (T)0;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            dv[2][c] = vel[3][c] - vel[2][c];
            dv[3][c] = vel[0][c] - vel[3][c];
            dv[0][c] = vel[1][c] - vel[0][c];
            flo[c] = mom_flux_of<T>(nf[3], neg, neg ? 0x80000000u : 0u, (T)1 - sig, (T)2 - sig, (T)1 + sig, d, rd,
                                    geo.r6, vel[3][c], vel[0][c], dv[2][c], dv[3][c], dv[0][c]);
        }
        __syncthreads();  // slots 0 and 1 are read before the march rewrites them
    }

    // a plane's loads go out before the barrier of the plane before (AHEAD: up
    // to 124 VGPRs in FP64, four waves per SIMD either way; 512^3 mom_y 2.39 ->
    // 2.30 ms FP64, FP32 mom_z 1.04 -> 0.98), except where four volume fluxes
    // would spill: FP64 mode 2, at the top of its own step (mom_z over both of its
    // modes 2.15 ms that way, 2.26 with 20 values spilled)
    constexpr bool AHEAD = sizeof(S) == 4 || MODE != 2;
    Pl nx;
    auto load_plane = [&](int q, int r, T(&vq)[3]) {
        Pl x;  // lanes other than 0 leave its column j-1 unset
        load(q, r, x, false);
#pragma unroll
        for (int c = 0; c < 3; c++) vq[c] = vel_at(c, q, r, false);
        return x;
    };
    int r = row_at(m0);
    if (AHEAD) nx = load_plane(m0 + 2, r + 2 * sM, vel[2]);
    auto step = [&](auto ic, int m) {
        constexpr int i = decltype(ic)::value, i1 = (i + 1) & 3, i2 = (i + 2) & 3, im = (i + 3) & 3, e = i & 1;
        // keeps the compiler from hoisting array + offset into vector registers
        // and from walking a pointer per array
        asm volatile("" : "+v"(oj), "+v"(orho), "+v"(ot), "+v"(ojm), "+v"(orhom), "+v"(otm), "+s"(r));
        const Pl x = AHEAD ? nx : load_plane(m + 2, r + 2 * sM, vel[i2]);
        const T a = x.c.a, p = publish(e, x);
        if (AHEAD && m < m1) nx = load_plane(m + 3, r + 3 * sM, vel[im]);  // vel(m-1) is done with
        __syncthreads();
        // F[1-e], P[1-e] hold plane m+1
        gather(e, a, p, F[e], P[e]);
        nf[i1] = march_node_flux<DIR, T>(F[1 - e], F[e]);  // nf(m+1)
        mp[i2] = march_node_mass<DIR, T>(P[1 - e], P[e]);  // mp(m+2), not used at mmax+3
        mq[i1] = mp[i1] - nf[i] + nf[i1];
        const T sig = face_sigma(nf[i], mq[i], mq[i1]);
        const bool neg = nf[i] < (T)0;
        const unsigned sgn = neg ? 0x80000000u : 0u;
        const T one_m = (T)1 - sig, two_m = (T)2 - sig, one_p = (T)1 + sig;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            dv[i1][c] = vel[i2][c] - vel[i1][c];
            const T fhi = mom_flux_of<T>(nf[i], neg, sgn, one_m, two_m, one_p, d, rd, geo.r6, vel[i][c], vel[i1][c],
                                         dv[im][c], dv[i][c], dv[i1][c]);  // F(m)
            const T out = quo(vel[i][c] * mq[i] + flo[c] - fhi, mp[i]);
            if (store) at(v.out[c] + r, oj) = out;
            flo[c] = fhi;
        }
        r += sM;
    };
    for (int m = m0;;) {
        step(std::integral_constant<int, 0>{}, m);
        if (++m > m1) break;
        step(std::integral_constant<int, 1>{}, m);
        if (++m > m1) break;
        step(std::integral_constant<int, 2>{}, m);
        if (++m > m1) break;
        step(std::integral_constant<int, 3>{}, m);
        if (++m > m1) break;
    }
}

// One workgroup of a y or z sweep.  With a narrow tail the grid's first
// workgroups (in launch order) march the tail, TailSplit::tb per chunk: its
// marches take longest per plane (each load touches a line per lane), and
// dispatched last they ran past the rest of the launch.  The 64-column
// tiles follow in the grid's order with gx-1 tiles to a row, and the
// workgroups left over exit at once.
// lin: the workgroup's place in launch order on a gx x gy x gz grid; xcd: the
// XCD order (launch.h xcd_layer_block, single-tile launches) for the 64-column
// tiles.
template <int DIR, int MODE, typename S>
__device__ __forceinline__ void mom_march(int lin, int gx, int gy, int gz, int xcd, Lay g, Geo geo,
                                          const S *__restrict__ mf, const S *__restrict__ vfx,
                                          const S *__restrict__ vfy, const S *__restrict__ vfz,
                                          const S *__restrict__ density1, Vel3<S> v)
{
    __shared__ S xbuf[4][2][mw_of(DIR)][65];
    int off = 0;
    if constexpr (sizeof(S) == 8) {  // the tail form: FP64 only (mom_tail_cols)
        const int tw = mom_tail_cols(g, gx);
        if (tw) {
            const TailSplit ts = mom_tail_split<DIR>(g, Blk{0, 0, 0, gx, gy, gz}, tw);
            if (lin < ts.tb * gz) {
                mom_tail_body<DIR, S>(Blk{gx - 1, lin % ts.tb, lin / ts.tb, gx, gy, gz}, ts, g, geo, MODE, mf, vfx,
                                      vfy, vfz, density1, v);
                return;
            }
            off = ts.tb * gz;
            gx -= 1;  // the 64-column tiles
            if (lin - off >= gx * gy * gz) return;
        }
    }
    const int id = xcd ? xcd_layer_block(lin, gx * gy, off) : lin - off;
    mom_cols_body<DIR, MODE, S>(Blk{id % gx, (id / gx) % gy, id / (gx * gy), gx, gy, gz}, xbuf, g, geo, mf, vfx, vfy,
                                vfz, density1, v);
}

template <int DIR, int MODE, typename S>
__global__ void __launch_bounds__(64 * mw_of(DIR), sizeof(S) == 8 ? 4 : 1) k_fast_mom_march(const DtDev *__restrict__ dt, int xcd, Lay g, Geo geo, const S *__restrict__ mf, const S *__restrict__ vfx,
                 const S *__restrict__ vfy, const S *__restrict__ vfz,
                 const S *__restrict__ density1, Vel3<S> v)
{
    if (dt->small) return;  // a small step (launch_dt_final)
    const int gx = (int)gridDim.x, gy = (int)gridDim.y, gz = (int)gridDim.z;
    mom_march<DIR, MODE, S>((int)blockIdx.x + gx * ((int)blockIdx.y + gy * (int)blockIdx.z), gx, gy, gz, xcd, g, geo,
                            mf, vfx, vfy, vfz, density1, v);
}

// ---------------------------------------------------------------------------
// x sweep: lanes along x with lanes 0-1 and 62-63 as halo (60 store), waves
// along y, march along z.  advec_mom_kernel.f90:172-206:
//   nf(j)  = 0.125*(f(0,-1,0)+f(0,0,0)+f(1,-1,0)+f(1,0,0)+f(0,-1,-1)+f(0,0,-1)+f(1,-1,-1)+f(1,0,-1))
//   mp(j)  = cells (0,-1,0),(0,0,0),(-1,-1,0),(-1,0,0),(0,-1,-1),(0,0,-1),(-1,-1,-1),(-1,0,-1)

//
// Laid out like mom_cols_body (scalar rows, MODE a template argument, the halo
// row's wave only loads and publishes); a neighbour along x is a DPP shift, so
// LDS carries the row below alone, 4 accesses per wave and plane instead of 34,
// and the VALU issues 239 (FP64) and 125 (FP32) instructions instead of 305 and
// 190.  The form before against this one, three rounds on one machine: 64^3 FP64
// 16.2 -> 14.1 us, 131x75x93 24.6 -> 21.1, 256^3 278 -> 256, FP32 101x143x67 16.0
// -> 15.4; 512^3, at its ten arrays' bandwidth, within the memory's spread.  Of
// 4, 8 and 16 waves per workgroup: 13.2, 14.1, 17.4 us at 64^3, 21.8, 21.1, 28.3 at
// 131x75x93.
template <int MODE, typename S>
__device__ __forceinline__ void mom_x_body(const Blk &bk, Lay g, Geo geo, const S *__restrict__ mf,
                                           const S *__restrict__ vfy, const S *__restrict__ vfz,
                                           const S *__restrict__ density1, Vel3<S> v)
{
    static_assert(MODE == 1 || MODE == 5, "the x sweep's modes");
    using T = S;  // arithmetic type of the form
    constexpr int MW = mw_of(1);
    __shared__ T xbuf[2][2][MW][64];
    const int lane = (int)threadIdx.x, w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const T d = (T)geo.dx;
    const Recip rd = geo.rx;
    const T V0 = (T)geo.vol;
    int l0, l1;
    chunk_range(bk, g.z_min, g.z_max + 1, l0, l1);
    if (l0 > l1) return;  // the whole workgroup: before any barrier
    const int j = g.x_min - 2 + bk.x * 60 + lane;
    const int k = g.y_min - 1 + bk.y * (MW - 1) + w;
    const bool row = w >= 1 && k <= g.y_max + 1;  // an owned row (uniform)
    const bool store = lane >= 2 && lane <= 61 && j <= g.x_max + 1;
    // Lanes and rows outside the arrays read clamped ones, which no stored node
    // needs: mass_flux_x and the vertices end at x_max+3, cells at x_max+2, and
    // every row read at y_max+2.  Byte offsets from column x_min-2: faces, nodes,
    // density and the tangential fluxes on a mirrored x face (launch.h).
    const int jf = min(j, g.x_max + 3), jc = min(j, g.x_max + 2), kr = min(k, g.y_max + 2);
    auto off = [&](int col) { return (unsigned)(col - g.x_min + 2) * (unsigned)sizeof(S); };
    unsigned oj = off(jf), on = off(node_xm(g, jf)), orho = off(cell_xm(g, jc)), ot = off(tan_xm(g, jc));
    const unsigned sx = node_xsign(g, jf) ? 0x80000000u : 0u;  // the reflection of the x velocity (update_halo_kernel.f90:604-1004)
    const int dk = (cell_m(g, 1, kr) - kr) * g.ld;  // density's row on a mirrored y face

    // a plane's values as stored, so that their loads can stay in flight; the
    // flux through its lower z face is the upper one of the plane before
    struct Pl {
        S a, rho, f[MODE == 1 ? 3 : 1];
    };
    auto load = [&](int q, int r) {  // r: the wave's row in plane q
        Pl x;
        x.a = at(mf + r, oj);
        x.rho = at(density1 + (r + dk + (cell_m(g, 2, q) - q) * g.plane), orho);
        if constexpr (MODE == 1) {
            x.f[0] = at(vfy + r + g.ld, ot);
            x.f[1] = at(vfy + r, ot);
            x.f[2] = at(vfz + r + g.plane, ot);
        }
        return x;
    };
    T zlo = 0;  // MODE 1: vol_flux_z through the lower face of the plane in hand
    auto publish = [&](int b, const Pl &x) {  // returns the cell mass, post_vol as in advec_mom_kernel.f90:95-163
        T p;
        if constexpr (MODE == 1) {
            p = x.rho * (V0 + x.f[0] - x.f[1] + x.f[2] - zlo);
            zlo = x.f[2];
        } else {
            p = x.rho * V0;
        }
        xbuf[b][0][w][lane] = x.a;
        xbuf[b][1][w][lane] = p;
        return p;
    };

    int r = idx(g, g.x_min - 2, kr, l0 - 1);
    if constexpr (MODE == 1) zlo = at(vfz + r, ot);
    if (!row) {  // loads and publishes only; as many barriers as below
        publish(1, load(l0 - 1, r));
        __syncthreads();
        for (int l = l0; l <= l1; l++) {
            r += g.plane;
            publish((l - l0) & 1, load(l, r));
            __syncthreads();
        }
        return;
    }

    Quad<T> F[2], P[2];
    auto gather = [&](int b, T a, T p) {
        const T aw = xbuf[b][0][w - 1][lane], pw = xbuf[b][1][w - 1][lane];
        F[b] = Quad<T>{a, next_lane(a), aw, next_lane(aw)};
        P[b] = Quad<T>{p, prev_lane(p), pw, prev_lane(pw)};
    };
    // a plane's loads go out before the barrier of the plane before; in FP32 that
    // ran 101x143x67 15.6 -> 15.4 us and 512^3 1.04 -> 1.01 ms against loads at the
    // top of the plane's own step
    Pl nx;
    S vn[3];
    auto load_plane = [&](int q, int rq) {
        nx = load(q, rq);
#pragma unroll
        for (int c = 0; c < 3; c++) vn[c] = at(v.in[c] + rq, on);
    };
    {
        const Pl x = load(l0 - 1, r);
        r += g.plane;
        const T p = publish(1, x);
        load_plane(l0, r);
        __syncthreads();
        gather(1, x.a, p);
    }
    auto step = [&](auto ic, int l) {
        constexpr int e = decltype(ic)::value;
        // keeps array + offset out of vector registers
        asm volatile("" : "+v"(oj), "+v"(on), "+v"(orho), "+v"(ot), "+s"(r));
        const Pl x = nx;
        T v0[3];
#pragma unroll
        for (int c = 0; c < 3; c++) v0[c] = vn[c];
        v0[0] = flip_sign(v0[0], sx);
        const T p = publish(e, x);
        if (l < l1) load_plane(l + 1, r + g.plane);
        __syncthreads();
        gather(e, x.a, p);
        // F.x = f(+1,0), F.w = f(0,-1), F.xw = f(+1,-1); P.x = cell(-1,0), ...
        const Quad<T> &Fc = F[e], &Fp = F[1 - e], &Pc = P[e], &Pp = P[1 - e];
        const T nf = (T)0.125 * (Fc.w + Fc.c + Fc.xw + Fc.x + Fp.w + Fp.c + Fp.xw + Fp.x);
        const T mp = (T)0.125 * (Pc.w + Pc.c + Pc.xw + Pc.x + Pp.w + Pp.c + Pp.xw + Pp.x);
        const T mq = mp - prev_lane(nf) + nf;
        const T sig = face_sigma(nf, mq, next_lane(mq));
        const bool neg = nf < (T)0;
        const unsigned sgn = neg ? 0x80000000u : 0u;
        const T one_m = (T)1 - sig, two_m = (T)2 - sig, one_p = (T)1 + sig;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const T vp1 = next_lane(v0[c]), d1 = vp1 - v0[c];
            const T fhi = mom_flux_of<T>(nf, neg, sgn, one_m, two_m, one_p, d, rd, geo.r6, v0[c], vp1, prev_lane(d1),
                                         d1, next_lane(d1));  // face j | j+1
            const T out = quo(v0[c] * mq + prev_lane(fhi) - fhi, mp);
            if (store) at(v.out[c] + r, oj) = out;
        }
        r += g.plane;
    };
    for (int l = l0;;) {
        step(std::integral_constant<int, 0>{}, l);
        if (++l > l1) break;
        step(std::integral_constant<int, 1>{}, l);
        if (++l > l1) break;
    }
}

template <int MODE, typename S>
__global__ void __launch_bounds__(64 * mw_of(1), sizeof(S) == 8 ? 6 : 1)
k_fast_mom_x(const DtDev *__restrict__ dt, int xcd, Lay g, Geo geo, const S *__restrict__ mf,
             const S *__restrict__ vfy, const S *__restrict__ vfz, const S *__restrict__ density1, Vel3<S> v)
{
    if (dt->small) return;  // a small step (launch_dt_final)
    mom_x_body<MODE, S>(hw_blk(xcd), g, geo, mf, vfy, vfz, density1, v);
}

// mom_post_vol's mode of a sweep of advection.f90 (x and z in sweeps 1 and 3,
// y in sweep 2); 0: no such sweep
static int mom_mode(int advect_x, int sweep_number, int direction)
{
    if (direction == 1) return sweep_number == 1 ? 1 : sweep_number == 3 ? 5 : 0;
    if (direction == 2) return sweep_number != 2 ? 0 : advect_x ? 3 : 4;
    if (direction == 3) return sweep_number == 1 ? 2 : sweep_number == 3 ? 6 : 0;
    return 0;
}

template <typename S>
static hipError_t fast_advec_mom_t(const DtDev *dt, const Lay &g, const Geo &m, int mode, int direction, const S *mass_flux_x,
                                   const S *vol_flux_x, const S *mass_flux_y, const S *vol_flux_y,
                                   const S *mass_flux_z, const S *vol_flux_z, const S *density1,
                                   const void *const *vel_in, void *const *vel_out, const Shape &sh, hipStream_t st)
{
    Vel3<S> v;
    for (int c = 0; c < 3; c++) {
        v.in[c] = static_cast<const S *>(vel_in[c]);
        v.out[c] = static_cast<S *>(vel_out[c]);
    }
    const int nxn = g.x_max - g.x_min + 2, nyn = g.y_max - g.y_min + 2, nzn = g.z_max - g.z_min + 2;  // nodes
    const int MW = mw_of(direction);
    const dim3 blk(64, MW, 1);
    if (direction == 1) {
        const dim3 grid((nxn + 59) / 60, (nyn + MW - 2) / (MW - 1), nchunks(nzn, sh.planes));
        const auto kern = mode == 1 ? k_fast_mom_x<1, S> : k_fast_mom_x<5, S>;
        TIMED_LAUNCH("k_fast_mom_x", st, kern, grid, blk, 0, st, dt, sh.xcd, g, m, mass_flux_x, vol_flux_y, vol_flux_z,
                     density1, v);
    } else if (direction == 2) {
        const dim3 grid((nxn + 63) / 64, (nzn + MW - 2) / (MW - 1), nchunks(nyn, sh.planes));
        const auto kern = mode == 3 ? k_fast_mom_march<2, 3, S> : k_fast_mom_march<2, 4, S>;
        TIMED_LAUNCH("k_fast_mom_y", st, kern, grid, blk, 0, st, dt, sh.xcd, g, m, mass_flux_y, vol_flux_x, vol_flux_y,
                     vol_flux_z, density1, v);
    } else {
        const dim3 grid((nxn + 63) / 64, (nyn + MW - 2) / (MW - 1), nchunks(nzn, sh.planes));
        const auto kern = mode == 2 ? k_fast_mom_march<3, 2, S> : k_fast_mom_march<3, 6, S>;
        TIMED_LAUNCH("k_fast_mom_z", st, kern, grid, blk, 0, st, dt, sh.xcd, g, m, mass_flux_z, vol_flux_x, vol_flux_y,
                     vol_flux_z, density1, v);
    }
    return hipGetLastError();
}

hipError_t launch_fast_advec_mom(Store s, const DtDev *dt, const Lay &g, const Geo &m, int advect_x, int sweep_number,
                                 int direction, const void *mass_flux_x, const void *vol_flux_x,
                                 const void *mass_flux_y, const void *vol_flux_y, const void *mass_flux_z,
                                 const void *vol_flux_z, const void *density1, const void *const *vel_in,
                                 void *const *vel_out, const Shape &sh, hipStream_t st)
{
    const int mode = mom_mode(advect_x, sweep_number, direction);
    if (!mode) return hipErrorInvalidValue;  // the resident driver issues only the reference's sweeps
#define CALL(T)                                                                                                 \
    fast_advec_mom_t<T>(dt, g, m, mode, direction, static_cast<const T *>(mass_flux_x),                             \
                        static_cast<const T *>(vol_flux_x), static_cast<const T *>(mass_flux_y),                \
                        static_cast<const T *>(vol_flux_y), static_cast<const T *>(mass_flux_z),                \
                        static_cast<const T *>(vol_flux_z), static_cast<const T *>(density1), vel_in, vel_out, sh, st)
    return s == ST_F32 ? CALL(float) : CALL(double);
#undef CALL
}

// ---------------------------------------------------------------------------
// Batched over many decks (batch.h): the new velocities go to X_W5..X_W7,
// wherever those and the step's arrays are at this point of it.
struct MomSlots {
    int rho, in[3], out[3];
};

__host__ __device__ inline void dims_mom(int dir, const Lay &g, int planes, int &gx, int &gy, int &gz)
{
    const int nxn = g.x_max - g.x_min + 2, nyn = g.y_max - g.y_min + 2, nzn = g.z_max - g.z_min + 2;  // nodes
    const int MW = mw_of(dir);
    if (dir == 1) {
        gx = (nxn + 59) / 60; gy = (nyn + MW - 2) / (MW - 1); gz = nchunks(nzn, planes);
    } else if (dir == 2) {
        gx = (nxn + 63) / 64; gy = (nzn + MW - 2) / (MW - 1); gz = nchunks(nyn, planes);
    } else {
        gx = (nxn + 63) / 64; gy = (nyn + MW - 2) / (MW - 1); gz = nchunks(nzn, planes);
    }
}

int batch_blocks_mom(int dir, const Lay &g, int planes)
{
    int gx, gy, gz;
    dims_mom(dir, g, planes, gx, gy, gz);
    return gx * gy * gz;
}

template <int DIR, int MODE, typename S>
__device__ __forceinline__ void mom_tile(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd,
                                         int planes, const MomSlots &ms, int hb)
{
    const int d = deck_of(start, nd, hb);
    const DeckDev &D = decks[d];
    int gx, gy, gz;
    dims_mom(DIR, D.g, planes, gx, gy, gz);
    const int lb = hb - start[d];
    const Blk bk{lb % gx, (lb / gx) % gy, lb / (gx * gy), gx, gy, gz};
    Vel3<S> v;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        v.in[c] = static_cast<const S *>(D.f[ms.in[c]]);
        v.out[c] = static_cast<S *>(D.f[ms.out[c]]);
    }
    const S *vfx = static_cast<const S *>(D.f[F_VOL_FLUX_X]);
    const S *vfy = static_cast<const S *>(D.f[F_VOL_FLUX_Y]);
    const S *vfz = static_cast<const S *>(D.f[F_VOL_FLUX_Z]);
    const S *rho = static_cast<const S *>(D.f[ms.rho]);
    if constexpr (DIR == 1)
        mom_x_body<MODE, S>(bk, D.g, D.m, static_cast<const S *>(D.f[F_MASS_FLUX_X]), vfy, vfz, rho, v);
    else
        mom_march<DIR, MODE, S>(lb, gx, gy, gz, 0, D.g, D.m,
                                static_cast<const S *>(D.f[DIR == 2 ? F_MASS_FLUX_Y : F_MASS_FLUX_Z]), vfx, vfy, vfz,
                                rho, v);
}

template <int DIR, int MODE, typename S>
// The FP64 y/z sweeps held to four waves per SIMD (128 VGPRs): at five they
// spill 18-34 values and the launches of 320^3 as 8 tiles ran 2.00 -> 2.42 ms.
__global__ void __launch_bounds__(64 * mw_of(DIR), DIR != 1 && sizeof(S) == 8 ? 4 : 1)
kb_mom(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd, int planes, int xcd, MomSlots ms)
{
    int hb, end, step;  // the tiles of this workgroup (persistent when the grid is short)
    tile_walk(start[nd], xcd, hb, end, step);
    for (; hb < end; hb += step) {
        mom_tile<DIR, MODE, S>(decks, start, nd, planes, ms, hb);
        __syncthreads();  // the next tile reuses the workgroup's LDS
    }
}

hipError_t batch_advec_mom(Store s, const DeckDev *decks, int nd, const BatchGrid &bg, int advect_x, int dir,
                           int sweep_number, const Slots &sl, const Shape &sh, hipStream_t st)
{
    const int mode = mom_mode(advect_x, sweep_number, dir);
    if (!mode) return hipErrorInvalidValue;
    if (bg.total == 0) return hipSuccess;
    const dim3 grid(batch_wgs(bg, sh)), blk(64, mw_of(dir));
    const MomSlots ms{sl[F_DENSITY1], {sl[F_XVEL1], sl[F_YVEL1], sl[F_ZVEL1]}, {sl[X_W5], sl[X_W6], sl[X_W7]}};
#define L(D_, M_, T_)                                                                                        \
    TIMED_LAUNCH("kb_mom", st, (kb_mom<D_, M_, T_>), grid, blk, 0, st, decks, bg.start, nd, sh.planes, sh.xcd, ms)
#define LM(T_)                                                                                               \
    if (mode == 1) L(1, 1, T_);                                                                              \
    else if (mode == 5) L(1, 5, T_);                                                                         \
    else if (mode == 3) L(2, 3, T_);                                                                         \
    else if (mode == 4) L(2, 4, T_);                                                                         \
    else if (mode == 2) L(3, 2, T_);                                                                         \
    else L(3, 6, T_)
    if (s == ST_F32) {
        LM(float);
    } else {
        LM(double);
    }
#undef LM
#undef L
    return hipGetLastError();
}

}  // namespace clover
