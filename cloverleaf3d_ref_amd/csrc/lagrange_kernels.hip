// The Lagrangian phase of a step as one z-march, for tiles whose six faces
// are all external and mirrored (Lay::mirror): the PdV predictor and its
// ideal_gas (PdV_kernel.f90:78-116, ideal_gas_kernel.f90:50-51), accelerate
// (accelerate_kernel.f90:61-109), the PdV corrector (PdV_kernel.f90:126-164)
// and flux_calc (flux_calc_kernel.f90:56-90), which hydro.f90:52-60 runs one
// after the other.  Such a tile needs no exchange between them: the predicted
// pressure's halo is the mirrored interior cell's.  Tiled and thin chunks
// exchange that pressure: they run the predictor of fast_kernels.hip, then this
// march without its own (k_fast_accel_pdv).
//
// Bytes.  Those two read the level-0 state twice and pass the predicted
// pressure through memory: 7 + 15 arrays per cell.  Here the state is read once
// and the predicted pressure never leaves the chip: 6 reads and 8 writes.
//
// Exactness.  Every value is formed by the expressions of the separate kernels
// on the same operands in the same order.  Sums that two faces or two stages
// share are formed once: a cell's right face is its x neighbour's left face,
// its front face the back face of the plane above (the same nodes in the same
// order), and the corrector's 8-term face sums continue from the predictor's
// 4-term partial over the same level-0 nodes.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "batch.h"
#include "fast.h"
#include "launch.h"

namespace clover {

// Layout.  A workgroup is 64 lanes (x) by LW waves (y); thread (lane, w) is
// node and cell (j, k) = (J + lane - 1, K + w - 1).  Owned are lanes 1..61 and
// waves 1..LW-2: a cell's corrector needs the level-1 nodes of lane+1 and w+1,
// these the predicted cells of lanes and waves around them, and those the
// level-0 nodes of lane+1 and w+1 (wave 0, which only predicts, loads the row
// above the last wave's).
//
// At node plane lp the march runs two phases, each ended by a barrier:
//   X: level-1 velocities of node plane lp from the cells of planes lp-1, lp;
//      the level-0 nodes of plane lp+2 go to LDS; the next plane's loads go out
//      first, so they have both phases to arrive;
//   Y: z faces of node plane lp, corrector and x/y faces of cell plane lp-1,
//      predictor of cell plane lp+1.
// LDS holds two planes each of level-0 and level-1 nodes, by parity, and one of
// cells.  X(lp) rewrites the slot of level-0 nodes lp+2, last read by other
// threads (plane lp) in Y(lp-1), and of level-1 nodes lp, last read (plane
// lp-2) in Y(lp-1); Y(lp) writes cells lp+1 over cells lp, read in X(lp).
//
// 512^3: the two kernels took 4.03 + 1.44 ms FP64 and 2.33 + 0.75 FP32, this one
// 3.96 (14 arrays, 3.8 TB/s) and 2.08; 131x75x93 FP64 40 + 16 -> 41 us.  The first
// form issued about 650 VALU instructions per wave and plane (now 340) and ran at
// the VALU's rate (4.05 ms, 64^3 26.8 us against 22.5).  Hence: terms
// that the next plane, lane or stage uses again are kept or shifted
// (next_lane) instead of formed again; the march is unrolled by two so that
// what alternates between planes stays in its registers; row addresses are
// scalar, with one byte offset per lane; mirrored halo cells are copies
// in LDS (x) or another row's index (y) instead of selects at each use; lanes
// outside the mesh load clamped addresses instead of branching.
//
// Waves.  FP64 takes 158 VGPRs, three waves per SIMD: one 12-wave workgroup per
// CU (512^3: 3.96 ms; 8, 10 and 11 waves 3.88-3.93, but 64^3 23.1-24.6 us
// against 22.5; held to 128 VGPRs for 16 waves, 28 values spill and it ran
// 7.1).  FP32 takes 90, five waves per SIMD: two 8-wave workgroups (512^3:
// 2.08 ms; 10, 14, 16 waves 2.07, 2.10, 2.14; 101x143x67 24.9 us, 26.2, 24.3,
// 24.5; held to 80 VGPRs for two 12-wave ones it spilled: 2.78 ms).
template <typename S>
constexpr int lw_of() { return sizeof(S) == 4 ? 8 : 12; }

__host__ __device__ inline void dims_lagrange(const Lay &g, int lw, int planes, int &gx, int &gy, int &gz)
{
    gx = (g.x_max - g.x_min + 2 + kLagrangeCols - 1) / kLagrangeCols;
    gy = (g.y_max - g.y_min + 2 + lw - 3) / (lw - 2);
    gz = nchunks(g.z_max - g.z_min + 2, planes);
}

// What accelerate uses of one pressure-like field (pressure, viscosity) in one
// cell plane, for the node (j, k): the area-weighted differences along x in
// rows k and k-1, along y in column j, and the cells of column j in rows k, k-1
template <typename T>
struct AccelTerms {
    T x0, x1, y0, c0, c1;
};

template <typename T>
__device__ inline AccelTerms<T> accel_terms(T c0, T c1, T xa, T ya)
{
    AccelTerms<T> t;
    t.x0 = xa * (c0 - prev_lane(c0));
    t.x1 = xa * (c1 - prev_lane(c1));
    t.y0 = ya * (c0 - c1);
    t.c0 = c0;
    t.c1 = c1;
    return t;
}

// accelerate_kernel.f90:75-101: u, v, w less st times the field's differences
// around the node (hi: the cell plane above it, lo: below)
template <typename T>
__device__ inline void accel_by(const AccelTerms<T> &hi, const AccelTerms<T> &lo, T st, T za, T &u, T &v, T &w)
{
    u = u - st * (hi.x0 + hi.x1 + lo.x0 + lo.x1);
    v = v - st * (hi.y0 + prev_lane(hi.y0) + lo.y0 + prev_lane(lo.y0));
    const T z0 = za * (hi.c0 - lo.c0), z1 = za * (hi.c1 - lo.c1);
    w = w - st * (z0 + z1 + prev_lane(z0) + prev_lane(z1));
}

// PRED: the whole phase, on a lagrange_tile (512^3: see above).  Otherwise accelerate, the
// corrector and flux_calc of any tile, after its predicted pressure (`pressure`)
// has been exchanged: the cells around the tile are read from its halo, or where
// a face is mirrored from the interior.  That form's own kernel before (quads
// read from memory and selected at mirrored faces, both velocity levels through
// LDS, 378 VALU instructions per plane against 252) ran 320^3 as 8 tiles FP64
// 1.31 -> 1.10 ms, FP32 0.584 -> 0.588, 160^3 as 8 227 -> 179 us and 89 -> 86,
// 512^3 as 4 tiles 4.90 -> 4.43 ms, 48x40x44 as 8 the same (three rounds on one
// machine).
template <bool PRED, typename S>
__device__ __forceinline__ void lagrange_body(const Blk &bk, Lay g, Geo m, double dt,
                                              const S *__restrict__ density0, S *__restrict__ density1,
                                              const S *__restrict__ energy0, S *__restrict__ energy1,
                                              const S *__restrict__ pressure, const S *__restrict__ viscosity, const S *__restrict__ xvel0,
                                              S *__restrict__ xvel1, const S *__restrict__ yvel0,
                                              S *__restrict__ yvel1, const S *__restrict__ zvel0,
                                              S *__restrict__ zvel1, S *__restrict__ vol_flux_x,
                                              S *__restrict__ vol_flux_y, S *__restrict__ vol_flux_z)
{
    using T = S;  // arithmetic type of the form
    constexpr int LW = lw_of<S>();
    __shared__ S n0[2][3][LW + 1][64];  // level-0 nodes
    __shared__ S n1[2][3][LW][64];      // level-1 nodes
    __shared__ S cb[3][LW][64];         // density, predicted pressure, viscosity of the cells
    const int lane = (int)threadIdx.x, w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int j = lagrange_col(g, bk.x, lane);
    const int k = g.y_min - 1 + bk.y * (LW - 2) + w;
    int l0, l1;
    chunk_range(bk, g.z_min, g.z_max + 1, l0, l1);
    if (l0 > l1) return;  // the whole workgroup, before any barrier
    const bool cols = lane >= 1 && lane <= kLagrangeCols && j <= g.x_max + 1;  // owned columns of nodes
    const bool ccols = cols && j <= g.x_max;                            // and of cells
    const bool march = w >= 1 && w <= LW - 2 && k <= g.y_max + 1;       // owned row of nodes (uniform)
    const bool crow = march && k <= g.y_max;                            // and of cells
    const int wu = min(w + 1, LW - 1);
    // rows of cb that hold the cells of rows k-1 and k: across a mirrored y
    // face the halo row is the interior one, which without the predictor was
    // loaded there
    const int r1 = PRED && k <= g.y_min ? w : w - 1, r0 = PRED && k > g.y_max ? w - 1 : w;
    const bool xedge = lagrange_halo_cells(g, bk.x);
    const T xa = (T)m.xa, ya = (T)m.ya, za = (T)m.za, vol = (T)m.vol, tdt = (T)dt;
    // the fluxes' factors 0.125 and 0.5 are powers of two: scaling dt by them
    // instead of the product gives the same bits (short of subnormal products,
    // which the sums and the state absorb)
    const T c0 = (T)0.125 * tdt, cp = c0 * (T)0.5;
    const T cx = c0 * xa, cy = c0 * ya, cz = c0 * za;
    const T recip_volume = (T)1 / vol;
    const int lend = min(l1 + 1, g.z_max + 1);  // last node plane accelerated
    // last and first cell plane predicted (the planes past mirrored z faces are
    // not), or loaded
    const int clast = PRED ? min(lend, g.z_max) : lend;
    const int lp0 = !PRED || l0 > g.z_min ? l0 - 1 : l0;
    // lanes outside the mesh read the nearest column and row inside it: nodes
    // to x_max+1, cells (mirrored halo cells among them) to x_max; without the
    // predictor cells are read one into the halo where that is not mirrored
    const int jn = min(max(j, g.x_min), g.x_max + 1);
    const int kn = min(max(k, g.y_min), g.y_max + 1);
    const int jc = PRED ? min(max(j, g.x_min), g.x_max) : cell_m(g, 0, min(j, g.x_max + 1));
    const int kc = PRED ? min(max(k, g.y_min), g.y_max) : cell_m(g, 1, min(k, g.y_max + 1));
    const int kn2 = min(k + LW, g.y_max + 1);  // wave 0: the row above the last wave's
    const int xb = PRED ? g.x_min : g.x_min - 1;  // rows are addressed from here
    unsigned on = (unsigned)(jn - xb) * (unsigned)sizeof(S);
    unsigned oc = (unsigned)(jc - xb) * (unsigned)sizeof(S);

    S un, vn, wn, u2n = 0, v2n = 0, w2n = 0, dn, en, pn = 0, qn;  // the next planes' loads
    auto load_nodes = [&](int l) {
        const int64_t r = idx(g, xb, kn, l);
        un = at(xvel0 + r, on);
        vn = at(yvel0 + r, on);
        wn = at(zvel0 + r, on);
        if (w == 0) {
            const int64_t r2 = idx(g, xb, kn2, l);
            u2n = at(xvel0 + r2, on);
            v2n = at(yvel0 + r2, on);
            w2n = at(zvel0 + r2, on);
        }
    };
    auto load_cells = [&](int l) {
        const int64_t r = idx(g, xb, kc, PRED ? l : cell_m(g, 2, l));
        dn = at(density0 + r, oc);
        en = at(energy0 + r, oc);
        if constexpr (!PRED) pn = at(pressure + r, oc);
        qn = at(viscosity + r, oc);
    };
    auto put_nodes = [&](int s) {
        n0[s][0][w][lane] = un;
        n0[s][1][w][lane] = vn;
        n0[s][2][w][lane] = wn;
        if (w == 0) {
            n0[s][0][LW][lane] = u2n;
            n0[s][1][LW][lane] = v2n;
            n0[s][2][LW][lane] = w2n;
        }
    };

    // Per cell plane, by parity: the corrector's 4-term level-0 sums of the
    // left, bottom and top faces, density, energy and (p + q) / density
    struct {
        T sl, sb, st, d, e, a;
    } cell[2] = {};
    // per z face, by parity: the 4-term level-0 sums of the corrector and of
    // vol_flux_z (its own node order)
    T sz[2], qz[2];
    T zp, zc = 0;  // the predictor's flux through its back face, the corrector's
    // per cell plane, by parity: accelerate's terms and the cell masses of rows k, k-1
    AccelTerms<T> pt[2] = {}, qt[2] = {};
    T m0[2] = {0, 0}, m1[2] = {0, 0};

    // a z face's level-0 sums from its nodes: column j rows k, k+1
    auto z_face = [&](T wa, T wb, T &s4, T &q4) {
        const T wan = next_lane(wa), wbn = next_lane(wb);
        s4 = wa + wan + wb + wbn;
        q4 = wa + wan + wan + wbn;
        return (za * (s4 + wa + wan + wb + wbn)) * cp;  // the predictor's flux: each node twice
    };
    // PdV predictor and ideal_gas of a cell plane of parity p, between the
    // node planes of parity p (below) and 1-p; without PRED the level-0 sums
    // alone, and pp is the predicted pressure
    auto predict = [&](auto par, T d0, T e0, T pp, T q0) {
        constexpr int p = decltype(par)::value;
        auto &C = cell[p];
        const T ua = n0[p][0][w][lane], ub = n0[p][0][w + 1][lane];
        const T uc = n0[1 - p][0][w][lane], ud = n0[1 - p][0][w + 1][lane];
        const T va = n0[p][1][w][lane], vb = n0[p][1][w + 1][lane];
        const T vc = n0[1 - p][1][w][lane], vd = n0[1 - p][1][w + 1][lane];
        const T wa = n0[1 - p][2][w][lane], wb = n0[1 - p][2][w + 1][lane];
        const T van = next_lane(va), vbn = next_lane(vb), vcn = next_lane(vc), vdn = next_lane(vd);
        C.sl = ua + ub + uc + ud;
        C.sb = va + van + vc + vcn;
        C.st = vb + vbn + vd + vdn;
        T qd;
        if constexpr (!PRED) {
            z_face(wa, wb, sz[1 - p], qz[1 - p]);
            qd = quo_sparse(q0, d0);
        } else {
            const T left_flux = (xa * (C.sl + ua + ub + uc + ud)) * cp;
            const T right_flux = next_lane(left_flux);
            const T bottom_flux = (ya * (C.sb + va + van + vc + vcn)) * cp;
            const T top_flux = (ya * (C.st + vb + vbn + vd + vdn)) * cp;
            const T front_flux = z_face(wa, wb, sz[1 - p], qz[1 - p]);
            const T total_flux = right_flux - left_flux + top_flux - bottom_flux + front_flux - zp;
            zp = front_flux;
            const T p0 = pressure_of<T>(d0, e0);
            const T vol_change_s = quo(vol, vol + total_flux);
            qd = quo_sparse(q0, d0);
            const T energy_change = (quo(p0, d0) + qd) * total_flux * recip_volume;
            const T e1 = e0 - energy_change;
            const T d1 = d0 * vol_change_s;
            pp = (T)(1.4 - 1.0) * d1 * e1;
            if (xedge) {  // mirrored halo columns take their neighbour's (density and viscosity were loaded there)
                const T lo = next_lane(pp), hi = prev_lane(pp);
                pp = j < g.x_min ? lo : j > g.x_max ? hi : pp;
            }
        }
        C.a = quo(pp, d0) + qd;
        C.d = d0;
        C.e = e0;
        cb[0][w][lane] = d0;
        cb[1][w][lane] = pp;
        cb[2][w][lane] = q0;
    };

    // one node plane of parity s
    auto plane = [&](auto par, int lp) {
        constexpr int s = decltype(par)::value;
        // keeps the compiler from hoisting array + offset, 17 address pairs in
        // VGPRs, instead of adding the offset to a scalar row address
        asm volatile("" : "+v"(on), "+v"(oc));
        // ---- X
        T u = n0[s][0][w][lane], v = n0[s][1][w][lane], ww = n0[s][2][w][lane];
        put_nodes(s);
        const T d0 = dn, e0 = en, p0 = pn, q0 = qn;
        if (lp + 3 <= clast + PRED) load_nodes(lp + 3);
        if (lp + 2 <= clast) load_cells(lp + 2);
        if (w >= 1) {
            if (!PRED || lp <= g.z_max) {
                pt[s] = accel_terms<T>(cb[1][r0][lane], cb[1][r1][lane], xa, ya);
                qt[s] = accel_terms<T>(cb[2][r0][lane], cb[2][r1][lane], xa, ya);
                m0[s] = cb[0][r0][lane] * vol;
                m1[s] = cb[0][r1][lane] * vol;
            } else {  // the plane above z_max mirrors z_max
                pt[s] = pt[1 - s], qt[s] = qt[1 - s], m0[s] = m0[1 - s], m1[s] = m1[1 - s];
            }
            if (PRED && lp == g.z_min)  // the plane below z_min mirrors z_min
                pt[1 - s] = pt[s], qt[1 - s] = qt[s], m0[1 - s] = m0[s], m1[1 - s] = m1[s];
            if (lp >= l0) {
                const T nodal_mass = (prev_lane(m1[s]) + m1[s] + m0[s] + prev_lane(m0[s]) + prev_lane(m1[1 - s]) +
                                      m1[1 - s] + m0[1 - s] + prev_lane(m0[1 - s])) *
                                     (T)0.125;
                const T st = quo((T)0.25 * tdt, nodal_mass);
                accel_by(pt[s], pt[1 - s], st, za, u, v, ww);
                accel_by(qt[s], qt[1 - s], st, za, u, v, ww);
                n1[s][0][w][lane] = u;
                n1[s][1][w][lane] = v;
                n1[s][2][w][lane] = ww;
                if (march && lp <= l1 && cols) {
                    const int64_t r = idx(g, xb, k, lp);
                    at(xvel1 + r, on) = u;
                    at(yvel1 + r, on) = v;
                    at(zvel1 + r, on) = ww;
                }
            }
        }
        __syncthreads();
        // ---- Y
        if (march && lp >= l0) {
            const T wa = n1[s][2][w][lane], wb = n1[s][2][wu][lane];
            const T wan = next_lane(wa), wbn = next_lane(wb);
            const T zflux = (za * (sz[s] + wa + wan + wb + wbn)) * c0;
            if (crow && lp <= l1 && ccols)
                at(vol_flux_z + (int64_t)idx(g, xb, k, lp), oc) = cz * (qz[s] + wa + wan + wb + wbn);
            if (lp > l0) {  // cell plane lp-1
                const auto &C = cell[1 - s];
                const T ua = n1[1 - s][0][w][lane], ub = n1[1 - s][0][wu][lane];
                const T uc = n1[s][0][w][lane], ud = n1[s][0][wu][lane];
                const T va = n1[1 - s][1][w][lane], vb = n1[1 - s][1][wu][lane];
                const T vc = n1[s][1][w][lane], vd = n1[s][1][wu][lane];
                const T sl = C.sl + ua + ub + uc + ud;
                const T sb = C.sb + va + next_lane(va) + vc + next_lane(vc);
                const T stp = C.st + vb + next_lane(vb) + vd + next_lane(vd);
                const T left_flux = (xa * sl) * c0;
                const T right_flux = next_lane(left_flux);
                const T bottom_flux = (ya * sb) * c0;
                const T top_flux = (ya * stp) * c0;
                const T total_flux = right_flux - left_flux + top_flux - bottom_flux + zflux - zc;
                const T energy_change = C.a * total_flux * recip_volume;
                const T e1 = C.e - energy_change;
                const T d1 = C.d * quo(vol, vol + total_flux);
                const int64_t r = idx(g, xb, k, lp - 1);
                if (crow && cols) at(vol_flux_x + r, on) = cx * sl;
                if (ccols) at(vol_flux_y + r, oc) = cy * sb;
                if (crow && ccols) {
                    at(energy1 + r, oc) = e1;
                    at(density1 + r, oc) = d1;
                }
            }
            zc = zflux;
        }
        if (lp + 1 <= clast) predict(std::integral_constant<int, 1 - s>{}, d0, e0, p0, q0);
        __syncthreads();
    };

    load_nodes(lp0);
    put_nodes(0);
    load_nodes(lp0 + 1);
    load_cells(lp0);
    put_nodes(1);
    const T d0 = dn, e0 = en, p0 = pn, q0 = qn;
    if (lp0 + 2 <= clast + PRED) load_nodes(lp0 + 2);
    if (lp0 + 1 <= clast) load_cells(lp0 + 1);
    __syncthreads();
    zp = z_face(n0[0][2][w][lane], n0[0][2][w + 1][lane], sz[0], qz[0]);
    predict(std::integral_constant<int, 0>{}, d0, e0, p0, q0);
    __syncthreads();
    for (int lp = lp0;; lp++) {
        plane(std::integral_constant<int, 0>{}, lp);
        if (++lp > lend) break;
        plane(std::integral_constant<int, 1>{}, lp);
        if (lp >= lend) break;
    }
}

template <typename S>
__global__ void __launch_bounds__(64 * lw_of<S>())
    k_fast_lagrange(int xcd, Lay g, Geo m, const DtDev *__restrict__ dtp, const S *__restrict__ density0, S *__restrict__ density1,
                    const S *__restrict__ energy0, S *__restrict__ energy1, const S *__restrict__ viscosity,
                    const S *__restrict__ xvel0, S *__restrict__ xvel1, const S *__restrict__ yvel0,
                    S *__restrict__ yvel1, const S *__restrict__ zvel0, S *__restrict__ zvel1,
                    S *__restrict__ vol_flux_x, S *__restrict__ vol_flux_y, S *__restrict__ vol_flux_z)
{
    const double dt = dtp->dt;
    if (dtp->small) return;
    lagrange_body<true, S>(hw_blk(xcd), g, m, dt, density0, density1, energy0, energy1, nullptr, viscosity, xvel0,
                           xvel1, yvel0, yvel1, zvel0, zvel1, vol_flux_x, vol_flux_y, vol_flux_z);
}

template <typename S>
__global__ void __launch_bounds__(64 * lw_of<S>())
    k_fast_accel_pdv(int xcd, Lay g, Geo m, const DtDev *__restrict__ dtp, const S *__restrict__ density0, S *__restrict__ density1,
                     const S *__restrict__ energy0, S *__restrict__ energy1, const S *__restrict__ pressure,
                     const S *__restrict__ viscosity, const S *__restrict__ xvel0, S *__restrict__ xvel1,
                     const S *__restrict__ yvel0, S *__restrict__ yvel1, const S *__restrict__ zvel0,
                     S *__restrict__ zvel1, S *__restrict__ vol_flux_x, S *__restrict__ vol_flux_y,
                     S *__restrict__ vol_flux_z)
{
    const double dt = dtp->dt;
    if (dtp->small) return;
    lagrange_body<false, S>(hw_blk(xcd), g, m, dt, density0, density1, energy0, energy1, pressure, viscosity, xvel0,
                            xvel1, yvel0, yvel1, zvel0, zvel1, vol_flux_x, vol_flux_y, vol_flux_z);
}

hipError_t launch_fast_lagrange(Store s, const Lay &g, const Geo &m, const DtDev *dt, const void *density0, void *density1,
                                const void *energy0, void *energy1, const void *viscosity, const void *xvel0,
                                void *xvel1, const void *yvel0, void *yvel1, const void *zvel0, void *zvel1,
                                void *vol_flux_x, void *vol_flux_y, void *vol_flux_z, const Shape &sh, hipStream_t st)
{
    if (!lagrange_tile(g)) return hipErrorInvalidValue;
    int gx, gy, gz;
    dims_lagrange(g, s == ST_F32 ? lw_of<float>() : lw_of<double>(), sh.planes, gx, gy, gz);
#define CP(p) static_cast<const T *>(p)
#define MP(p) static_cast<T *>(p)
#define CALL(T_)                                                                                              \
    do {                                                                                                      \
        using T = T_;                                                                                         \
        TIMED_LAUNCH("k_fast_lagrange", st, k_fast_lagrange<T>, dim3(gx, gy, gz), dim3(64, lw_of<T>()), 0, st, sh.xcd, g, m, \
                     dt, CP(density0), MP(density1), CP(energy0), MP(energy1), CP(viscosity), CP(xvel0), MP(xvel1),  \
                     CP(yvel0), MP(yvel1), CP(zvel0), MP(zvel1), MP(vol_flux_x), MP(vol_flux_y), MP(vol_flux_z));    \
    } while (0)
    if (s == ST_F32) CALL(float);
    else CALL(double);
#undef CALL
#undef CP
#undef MP
    return hipGetLastError();
}

hipError_t launch_fast_accel_pdv(Store s, const Lay &g, const Geo &m, const DtDev *dt, const void *density0,
                                 void *density1, const void *energy0, void *energy1, const void *pressure,
                                 const void *viscosity, const void *xvel0, void *xvel1, const void *yvel0,
                                 void *yvel1, const void *zvel0, void *zvel1, void *vol_flux_x, void *vol_flux_y,
                                 void *vol_flux_z, const Shape &sh, hipStream_t st)
{
    int gx, gy, gz;
    dims_lagrange(g, s == ST_F32 ? lw_of<float>() : lw_of<double>(), sh.planes, gx, gy, gz);
#define CP(p) static_cast<const T *>(p)
#define MP(p) static_cast<T *>(p)
#define CALL(T_)                                                                                              \
    do {                                                                                                      \
        using T = T_;                                                                                         \
        TIMED_LAUNCH("k_fast_accel_pdv", st, k_fast_accel_pdv<T>, dim3(gx, gy, gz), dim3(64, lw_of<T>()), 0, st, sh.xcd, g, m, \
                     dt, CP(density0), MP(density1), CP(energy0), MP(energy1), CP(pressure), CP(viscosity), CP(xvel0),  \
                     MP(xvel1), CP(yvel0), MP(yvel1), CP(zvel0), MP(zvel1), MP(vol_flux_x), MP(vol_flux_y),   \
                     MP(vol_flux_z));                                                                         \
    } while (0)
    if (s == ST_F32) CALL(float);
    else CALL(double);
#undef CALL
#undef CP
#undef MP
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Batched over many decks (batch.h)
int batch_blocks_lagrange(const Lay &g, int planes, Store s)
{
    int gx, gy, gz;
    dims_lagrange(g, s == ST_F32 ? lw_of<float>() : lw_of<double>(), planes, gx, gy, gz);
    return gx * gy * gz;
}

template <bool PRED, typename S>
__device__ __forceinline__ void lagrange_tiles(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd,
                                               int planes, int xcd)
{
    int hb, end, step;  // the tiles of this workgroup (persistent when the grid is short)
    tile_walk(start[nd], xcd, hb, end, step);
    for (; hb < end; hb += step) {
        const int d = deck_of(start, nd, hb);
        const DeckDev &D = decks[d];
        int gx, gy, gz;
        dims_lagrange(D.g, lw_of<S>(), planes, gx, gy, gz);
        const int lb = hb - start[d];
        const Blk bk{lb % gx, (lb / gx) % gy, lb / (gx * gy), gx, gy, gz};
#define CF(id) static_cast<const S *>(D.f[id])
#define MF(id) static_cast<S *>(D.f[id])
        lagrange_body<PRED, S>(bk, D.g, D.m, D.dt, CF(F_DENSITY0), MF(F_DENSITY1), CF(F_ENERGY0), MF(F_ENERGY1),
                               CF(F_PRESSURE), CF(F_VISCOSITY), CF(F_XVEL0), MF(F_XVEL1), CF(F_YVEL0), MF(F_YVEL1),
                               CF(F_ZVEL0), MF(F_ZVEL1), MF(F_VOL_FLUX_X), MF(F_VOL_FLUX_Y), MF(F_VOL_FLUX_Z));
#undef CF
#undef MF
        __syncthreads();  // the next tile reuses the workgroup's LDS
    }
}

template <typename S>
__global__ void __launch_bounds__(64 * lw_of<S>())
kb_lagrange(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd, int planes, int xcd)
{
    lagrange_tiles<true, S>(decks, start, nd, planes, xcd);
}

template <typename S>
__global__ void __launch_bounds__(64 * lw_of<S>())
kb_accel_pdv(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd, int planes, int xcd)
{
    lagrange_tiles<false, S>(decks, start, nd, planes, xcd);
}

hipError_t batch_lagrange(Store s, const DeckDev *decks, int nd, const BatchGrid &bg, const Shape &sh, hipStream_t st)
{
    if (bg.total == 0) return hipSuccess;
    const dim3 grid(batch_wgs(bg, sh)), blk(64, s == ST_F32 ? lw_of<float>() : lw_of<double>());
    if (s == ST_F32)
        TIMED_LAUNCH("kb_lagrange", st, kb_lagrange<float>, grid, blk, 0, st, decks, bg.start, nd, sh.planes, sh.xcd);
    else
        TIMED_LAUNCH("kb_lagrange", st, kb_lagrange<double>, grid, blk, 0, st, decks, bg.start, nd, sh.planes, sh.xcd);
    return hipGetLastError();
}

hipError_t batch_accel_pdv(Store s, const DeckDev *decks, int nd, const BatchGrid &bg, const Shape &sh, hipStream_t st)
{
    if (bg.total == 0) return hipSuccess;
    const dim3 grid(batch_wgs(bg, sh)), blk(64, s == ST_F32 ? lw_of<float>() : lw_of<double>());
    if (s == ST_F32)
        TIMED_LAUNCH("kb_accel_pdv", st, kb_accel_pdv<float>, grid, blk, 0, st, decks, bg.start, nd, sh.planes, sh.xcd);
    else
        TIMED_LAUNCH("kb_accel_pdv", st, kb_accel_pdv<double>, grid, blk, 0, st, decks, bg.start, nd, sh.planes, sh.xcd);
    return hipGetLastError();
}

}  // namespace clover
