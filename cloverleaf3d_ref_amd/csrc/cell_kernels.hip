// advec_cell (advec_cell_kernel.f90:30-383) for one sweep as one kernel:
// the mass and energy fluxes of every face along the sweep and the cell
// update that consumes them, with the energy flux and pre_vol kept in
// registers.  The fluxes of a face depend only on cells along the sweep
// (upwind, donor, downwind), so
//   * the x sweep works on rows: lanes along x, each lane forms the flux of
//     its face from its neighbours' values (lane shuffles) and updates its
//     cell from its own and the next lane's flux (60 of 64 lanes store);
//   * the y and z sweeps march each (x, cross) column along the sweep
//     axis with the upwind..downwind window in registers.
// The reference computes every flux with the old density1/energy1 before
// it updates any cell, so the new values go to separate arrays (rho_out,
// e_out) which then take the place of density1/energy1; only interior cells
// of those are written (the halo update that follows every advec_cell
// sweep in advection.f90 refreshes their halos before anything reads them).
// The step's last sweep can also write the pressure of the new state (p_out;
// null otherwise): after reset_field that state is the
// next step's level 0, so these are the values the next ideal_gas call
// (timestep.f90:48 or field_summary.f90:49-60) would compute.
// In the FP64 form every value is formed with the expression and operand
// order of the per-call kernels, so the results are bit-identical.  The FP32
// form computes the face fluxes in FP32 and keeps pre_vol and the cell's
// mass and energy update in FP64.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "batch.h"
#include "fast.h"
#include "launch.h"

namespace clover {

constexpr int CROWS = 4;   // rows (or columns) per workgroup

// pre_vol (advec_cell_kernel.f90:97-116, 193-210, 289-306) has a `mode`:
// 1 x sweep 1, 2 x sweep 3, 3 y sweep with advect_x, 4 y without,
// 5 z sweep 1, 6 z sweep 3

template <typename T>
__device__ inline T cell_limiter(T sigma, T sigma3, T sigma4, T diffuw, T diffdw)
{
    const T one_by_six = (T)(1.0 / 6.0);
    if (diffuw * diffdw > (T)0)
        return ((T)1 - sigma) * copysign((T)1, diffdw) *
               tmin(tmin(fabs(diffuw), fabs(diffdw)), one_by_six * (sigma3 * fabs(diffuw) + sigma4 * fabs(diffdw)));
    return (T)0;
}

// Mass and energy flux through one face (advec_cell_kernel.f90:123-186 and
// twins): ru/rd/rw, eu/ed/ew the density and energy of the upwind, donor and
// downwind cells, pv the donor's pre_vol, vd the vertex spacing; T is the
// form's arithmetic type.
template <typename T>
__device__ inline void cell_face_flux(T vf, T pv, T vd, T ru, T rd, T rw, T eu, T ed, T ew, T &mf, T &ef)
{
    const T sigmat = quo(fabs(vf), pv);
    const T sigma3 = ((T)1 + sigmat) * (vd / vd);  // vertexd*(j)/vertexd*(dif) on the uniform mesh
    const T sigma4 = (T)2 - sigmat;
    T limiter = cell_limiter(sigmat, sigma3, sigma4, rd - ru, rw - rd);
    mf = vf * (rd + limiter);
    const T sigmam = quo(fabs(mf), rd * pv);
    limiter = cell_limiter(sigmam, sigma3, sigma4, ed - eu, ew - ed);
    ef = mf * (ed + limiter);
}

// cell update (advec_cell_kernel.f90:188-191 and twins), FP64 in both forms
__device__ inline void cell_update(double rho, double e, double pv, double mf_lo, double mf_hi, double ef_lo,
                                   double ef_hi, double vf_lo, double vf_hi, double &rho_new, double &e_new)
{
    const double pm = rho * pv;
    const double pom = pm + mf_lo - mf_hi;
    const double pe = (e * pm + ef_lo - ef_hi) / pom;
    const double av = pv + vf_lo - vf_hi;
    rho_new = pom / av;
    e_new = pe;
}

__device__ inline double shfl_c(double x, int src) { return __shfl(x, src, 64); }
__device__ inline float shfl_c(float x, int src) { return __shfl(x, src, 64); }

// ---------------------------------------------------------------------------
// x sweep: faces j in [x_min, x_max+2], rows k, l interior.  Lane i holds
// cell/face j = jt - 2 + i.  A wave walks `rows` consecutive rows (k
// fastest) and issues the next row's loads before the current row's work;
// one row per wave leaves too few bytes in flight in the FP32 form.
template <typename S>
__device__ __forceinline__ void cell_x_body(const Blk &bk, Lay g, Geo m, int mode, int rows, const S *__restrict__ vfx,
              const S *__restrict__ vfy, const S *__restrict__ vfz, const S *__restrict__ density1,
              const S *__restrict__ energy1, S *__restrict__ mass_flux_x, S *__restrict__ rho_out,
              S *__restrict__ e_out, S *__restrict__ p_out)
{
    const int lane = threadIdx.x;
    const int ny = g.y_max - g.y_min + 1, nz = g.z_max - g.z_min + 1;
    const int nrows = ny * nz;
    const int r0 = (bk.y * CROWS + (int)threadIdx.y) * rows;
    if (r0 >= nrows) return;  // whole wave: no shuffle partner is lost
    const int r1 = min(r0 + rows, nrows) - 1;
    const int j = g.x_min - 2 + bk.x * 60 + lane;
    using T = S;  // arithmetic type of the fluxes
    const bool ok_cell = j <= g.x_max + 2;  // j >= x_min-2 always
    const bool ok_face = j <= g.x_max + 3;
    // pre_vol's volume fluxes (advec_cell_kernel.f90:97-116): all three axes
    // in sweep 1 (mode 1), x only in sweep 3 (mode 2)
    const bool all3 = mode == 1;
    // the next row's values, raw (converted where used, so the loads stay
    // in flight): density, energy, vol_flux_x at j and j+1, vol_flux_y at k
    // and k+1, vol_flux_z at l and l+1
    S rn = 0, en = 0, fx0 = 0, fx1 = 0, fy0 = 0, fy1 = 0, fz0 = 0, fz1 = 0;
    auto row_at = [&](int r) { return idx(g, j, g.y_min + r % ny, g.z_min + r / ny); };
    const int dxc = cell_xm(g, j) - j;  // a mirrored x face: the interior cell its halo copies
    const int dxt = tan_xm(g, j) - j;  // the same for vol_flux_y and vol_flux_z
    auto load = [&](int ii) {
        rn = ok_cell ? density1[ii + dxc] : (S)0;
        en = ok_cell ? energy1[ii + dxc] : (S)0;
        fx0 = ok_face ? vfx[ii] : (S)0;
        fx1 = ok_cell ? vfx[ii + 1] : (S)0;
        fy0 = (ok_cell && all3) ? vfy[ii + dxt] : (S)0;
        fy1 = (ok_cell && all3) ? vfy[ii + dxt + g.ld] : (S)0;
        fz0 = (ok_cell && all3) ? vfz[ii + dxt] : (S)0;
        fz1 = (ok_cell && all3) ? vfz[ii + dxt + g.plane] : (S)0;
    };
    int in = row_at(r0);
    load(in);
    for (int r = r0; r <= r1; r++) {
        const int i = in;
        const T rho = rn, e = en;
        const S x0 = fx0, x1 = fx1, y0 = fy0, y1 = fy1, z0 = fz0, z1 = fz1;
        if (r < r1) {
            in = row_at(r + 1);
            load(in);
        }
        double pv = 0.0;
        if (ok_cell)
            pv = all3 ? m.vol + ((double)x1 - (double)x0 + (double)y1 - (double)y0 + (double)z1 - (double)z0)
                      : m.vol + (double)x1 - (double)x0;
        const T vf = x0;
        const int lm2 = max(lane - 2, 0), lm1 = max(lane - 1, 0), lp1 = min(lane + 1, 63);
        const T rm2 = shfl_c(rho, lm2), rm1 = shfl_c(rho, lm1), rp1 = shfl_c(rho, lp1);
        const T em2 = shfl_c(e, lm2), em1 = shfl_c(e, lm1), ep1 = shfl_c(e, lp1);
        const double pvm1 = shfl_c(pv, lm1);
        const T vd = (T)m.dx;
        // face j: upwind/donor/downwind (advec_cell_kernel.f90:123-132); the
        // upwind index is clamped at x_max+2
        T mf, ef;
        if (vf > (T)0) {
            cell_face_flux(vf, (T)pvm1, vd, rm2, rm1, rho, em2, em1, e, mf, ef);
        } else {
            const bool clamp = j + 1 > g.x_max + 2;
            cell_face_flux(vf, (T)pv, vd, clamp ? rho : rp1, rho, rm1, clamp ? e : ep1, e, em1, mf, ef);
        }
        const T mf_hi = shfl_c(mf, lp1), ef_hi = shfl_c(ef, lp1), vf_hi = shfl_c(vf, lp1);
        if (lane < 2 || lane > 61) continue;
        if (j <= g.x_max + 2) mass_flux_x[i] = mf;
        if (j <= g.x_max) {
            double rnew, enew;
            cell_update(rho, e, pv, mf, mf_hi, ef, ef_hi, vf, vf_hi, rnew, enew);
            const S rs = (S)rnew, es = (S)enew;
            rho_out[i] = rs;
            e_out[i] = es;
            if (p_out) p_out[i] = pressure_of<S>(rs, es);
        }
    }
}

template <typename S>
__global__ void __launch_bounds__(64 * CROWS) k_fast_cell_x(const DtDev *__restrict__ dt, int xcd, Lay g, Geo m, int mode, const S *__restrict__ vfx, const S *__restrict__ vfy,
              const S *__restrict__ vfz, const S *__restrict__ density1,
              const S *__restrict__ energy1, S *__restrict__ mass_flux_x, S *__restrict__ rho_out,
              S *__restrict__ e_out, S *__restrict__ p_out, int rows)
{
    if (dt->small) return;  // a small step (launch_dt_final)
    cell_x_body<S>(hw_blk(xcd), g, m, mode, rows, vfx, vfy, vfz, density1, energy1, mass_flux_x, rho_out, e_out,
                   p_out);
}

// the order of the y and z marches' positions (launch.h linear_sweep); along z the
// lanes' 32-bit byte offsets span the array
template <int DIR>
__host__ __device__ inline bool linear_cell(const Lay &g)
{
    return linear_sweep(g.x_max - g.x_min + 1) &&
           (DIR == 3 || (long long)g.plane * (g.z_max - g.z_min + 6) < (1LL << 29));
}

template <int DIR>
__host__ __device__ inline void dims_march(const Lay &g, int planes, int &gx, int &gy, int &gz)
{
    const int nx = g.x_max - g.x_min + 1, ny = g.y_max - g.y_min + 1, nz = g.z_max - g.z_min + 1;
    dims_rows(linear_cell<DIR>(g), nx, DIR == 3 ? ny : nz + 2, 64, CROWS, gx, gy);
    gz = nchunks(DIR == 3 ? nz + 2 : ny + 2, planes);
}

// ---------------------------------------------------------------------------
// y and z sweeps: lanes along x (interior j), threadIdx.y along the cross
// axis, march along the sweep axis over faces [smin, smax+2] in chunks.
// Faces of the y sweep run over l in [z_min, z_max+2] (advec_cell_kernel.f90:
// 215-217); the cells updated are interior.  MODE: pre_vol's,
// 3-6.  Row addresses are scalar (the wave's cross row and the face), a
// lane adds a byte offset; density and energy across a mirrored face are read
// at the interior cell.
template <bool LIN, int DIR, int MODE, typename S>
__device__ __forceinline__ void cell_march_body(const Blk &bk, Lay g, Geo m, const S *__restrict__ vfx, const S *__restrict__ vfy,
                  const S *__restrict__ vfz, const S *__restrict__ density1,
                  const S *__restrict__ energy1, S *__restrict__ mass_flux, S *__restrict__ rho_out,
                  S *__restrict__ e_out, S *__restrict__ p_out)
{
    int pos, row0;
    place_rows<LIN>(bk, g.x_max - g.x_min + 1, 0, 0, pos, row0);
    const int crmin = DIR == 3 ? g.y_min : g.z_min;
    const int j = g.x_min + pos, cr = crmin + row0;
    const int crmax = DIR == 3 ? g.y_max : g.z_max + 2;  // last cross position with faces
    if (j > g.x_max || cr > crmax) return;                 // no cross-lane traffic in this kernel
    const bool cross_in = DIR == 3 || cr <= g.z_max;       // updates only on interior cells
    const int smin = DIR == 3 ? g.z_min : g.y_min, smax = DIR == 3 ? g.z_max : g.y_max;
    using T = S;  // arithmetic type of the fluxes
    const T vd = (T)(DIR == 3 ? m.dz : m.dy);
    const S *__restrict__ vfs = DIR == 3 ? vfz : vfy;
    int f0, f1;
    chunk_range(bk, smin, smax + 2, f0, f1);
    if (f0 > f1) return;
    // the scalar rows' cross positions, of faces and of cells, and the lane's
    // byte offsets from them: the wave's own, or the first where lanes lie in
    // several rows
    const int crc = DIR == 3 ? cr : cell_m(g, 2, cr);
    const int cb = LIN ? crmin : cr, cbc = LIN ? crmin : crc;
    const int sC = DIR == 3 ? g.ld : g.plane;
    unsigned oj = (unsigned)(pos + (LIN ? row0 * sC : 0)) * (unsigned)sizeof(S);
    unsigned ojc = LIN ? (unsigned)(pos + (crc - crmin) * sC) * (unsigned)sizeof(S) : 0;
    auto row = [&](int q) { return (int64_t)(DIR == 3 ? idx(g, g.x_min, cb, q) : idx(g, g.x_min, q, cb)); };
    auto cell = [&](const S *__restrict__ p, int q) -> S {  // density or energy
        const int qc = cell_m(g, DIR - 1, q);
        return at(p + (int64_t)(DIR == 3 ? idx(g, g.x_min, cbc, qc) : idx(g, g.x_min, qc, cbc)), LIN ? ojc : oj);
    };
    // pre_vol's volume fluxes of the cell at q, raw (converted where used, so
    // that a face's loads can be issued a step ahead of their use)
    struct Pre {
        S v[MODE == 5 ? 6 : MODE == 6 ? 2 : 4];
    };
    auto load_pre = [&](int q) {
        const int64_t r = row(q);
        Pre x;
        int n = 0;
        auto pair = [&](const S *__restrict__ p, int up) {
            x.v[n++] = at(p + r + up, oj);
            x.v[n++] = at(p + r, oj);
        };
        if constexpr (MODE == 5) pair(vfx, 1);
        if constexpr (MODE == 5 || MODE == 3 || MODE == 4) pair(vfy, g.ld);
        if constexpr (MODE == 4) pair(vfx, 1);
        if constexpr (MODE != 4) pair(vfz, g.plane);
        return x;
    };
    // its expressions
    auto pre_of = [&](const Pre &x) -> double {
#define D(i) ((double)x.v[i])
        if constexpr (MODE == 5) return m.vol + (D(0) - D(1) + D(2) - D(3) + D(4) - D(5));
        else if constexpr (MODE == 6) return m.vol + D(0) - D(1);
        else return m.vol + D(0) - D(1) + D(2) - D(3);
#undef D
    };

    // window of old values at f-2, f-1, f, f+1 and pre_vol at f-1, f
    T r_m2 = cell(density1, f0 - 2), r_m1 = cell(density1, f0 - 1), r_0 = cell(density1, f0);
    T e_m2 = cell(energy1, f0 - 2), e_m1 = cell(energy1, f0 - 1), e_0 = cell(energy1, f0);
    const Pre pr_m1 = load_pre(f0 - 1);
    // face f0's loads; each step issues the next face's before its arithmetic
    S vf_n = at(vfs + row(f0), oj);
    Pre pr_n = load_pre(f0);
    S r_n = (S)0, e_n = (S)0;  // upwind for vf <= 0 is min(f+1, smax+2)
    if (f0 + 1 <= smax + 2) {
        r_n = cell(density1, f0 + 1);
        e_n = cell(energy1, f0 + 1);
    }
    double pv_m1 = pre_of(pr_m1);
    // flux of face f0-1, needed when cell f0-1 is updated here (f0 > smin)
    T mf_lo = 0, ef_lo = 0, vf_lo = 0;
    if (f0 > smin) {
        vf_lo = at(vfs + row(f0 - 1), oj);
        const T r_m3 = cell(density1, f0 - 3), e_m3 = cell(energy1, f0 - 3);
        const double pv_m2 = pre_of(load_pre(f0 - 2));
        if (vf_lo > (T)0)
            cell_face_flux(vf_lo, (T)pv_m2, vd, r_m3, r_m2, r_m1, e_m3, e_m2, e_m1, mf_lo, ef_lo);
        else
            cell_face_flux(vf_lo, (T)pv_m1, vd, r_0, r_m1, r_m2, e_0, e_m1, e_m2, mf_lo, ef_lo);  // f0 <= smax+1
    }
    for (int f = f0; f <= f1; f++) {
        asm volatile("" : "+v"(oj));  // no array + offset hoisted into vector registers
        if constexpr (LIN) asm volatile("" : "+v"(ojc));
        const T vf = vf_n;
        const double pv_0 = pre_of(pr_n);
        const T r_p1 = f + 1 <= smax + 2 ? r_n : r_0, e_p1 = f + 1 <= smax + 2 ? e_n : e_0;
        if (f < f1) {
            vf_n = at(vfs + row(f + 1), oj);
            pr_n = load_pre(f + 1);
            if (f + 2 <= smax + 2) {
                r_n = cell(density1, f + 2);
                e_n = cell(energy1, f + 2);
            }
        }
        T mf, ef;
        if (vf > (T)0)
            cell_face_flux(vf, (T)pv_m1, vd, r_m2, r_m1, r_0, e_m2, e_m1, e_0, mf, ef);
        else
            cell_face_flux(vf, (T)pv_0, vd, r_p1, r_0, r_m1, e_p1, e_0, e_m1, mf, ef);
        at(mass_flux + row(f), oj) = mf;
        const int c = f - 1;  // cell between faces f-1 and f
        if (cross_in && c >= smin && c <= smax) {
            double rn, en;
            cell_update(r_m1, e_m1, pv_m1, mf_lo, mf, ef_lo, ef, vf_lo, vf, rn, en);
            const S rs = (S)rn, es = (S)en;
            const int64_t rc = row(c);
            at(rho_out + rc, oj) = rs;
            at(e_out + rc, oj) = es;
            if (p_out) at(p_out + rc, oj) = pressure_of<S>(rs, es);
        }
        mf_lo = mf;
        ef_lo = ef;
        vf_lo = vf;
        r_m2 = r_m1;
        r_m1 = r_0;
        r_0 = r_p1;
        e_m2 = e_m1;
        e_m1 = e_0;
        e_0 = e_p1;
        pv_m1 = pv_0;
    }
}

template <int DIR, int MODE, typename S, bool LIN>
__global__ void __launch_bounds__(64 * CROWS) k_fast_cell_march(const DtDev *__restrict__ dt, int xcd, Lay g, Geo m, const S *__restrict__ vfx, const S *__restrict__ vfy,
                  const S *__restrict__ vfz, const S *__restrict__ density1,
                  const S *__restrict__ energy1, S *__restrict__ mass_flux, S *__restrict__ rho_out,
                  S *__restrict__ e_out, S *__restrict__ p_out)
{
    if (dt->small) return;
    cell_march_body<LIN, DIR, MODE, S>(hw_blk(xcd), g, m, vfx, vfy, vfz, density1, energy1, mass_flux, rho_out, e_out,
                                  p_out);
}

template <typename S>
static hipError_t fast_advec_cell_t(const DtDev *dt, const Lay &g, const Geo &m, int mode, int dir, const S *density1,
                                    const S *energy1, S *mass_flux_x, const S *vol_flux_x, S *mass_flux_y,
                                    const S *vol_flux_y, S *mass_flux_z, const S *vol_flux_z, S *rho_out, S *e_out,
                                    S *p_out, const Shape &sh, hipStream_t st)
{
    const int nx = g.x_max - g.x_min + 1, ny = g.y_max - g.y_min + 1, nz = g.z_max - g.z_min + 1;
    const dim3 blk(64, CROWS, 1);
    if (dir == 1) {
        const int rows = cell_x_rows(sh.planes);
        const dim3 grid((nx + 2 + 59) / 60, ((ny * nz + rows - 1) / rows + CROWS - 1) / CROWS, 1);
        TIMED_LAUNCH("k_fast_cell_x", st, k_fast_cell_x<S>, grid, blk, 0, st, dt, sh.xcd, g, m, mode, vol_flux_x, vol_flux_y,
                     vol_flux_z, density1, energy1, mass_flux_x, rho_out, e_out, p_out, rows);
    } else if (dir == 2) {
        int gx, gy, gz;
        dims_march<2>(g, sh.planes, gx, gy, gz);
        const dim3 grid(gx, gy, gz);
        const bool lin = linear_cell<2>(g);
        const auto kern = mode == 3 ? lin ? k_fast_cell_march<2, 3, S, true> : k_fast_cell_march<2, 3, S, false>
                          : lin     ? k_fast_cell_march<2, 4, S, true>
                                    : k_fast_cell_march<2, 4, S, false>;
        TIMED_LAUNCH("k_fast_cell_y", st, kern, grid, blk, 0, st, dt, sh.xcd, g, m, vol_flux_x, vol_flux_y, vol_flux_z, density1, energy1, mass_flux_y, rho_out, e_out, p_out);
    } else {
        int gx, gy, gz;
        dims_march<3>(g, sh.planes, gx, gy, gz);
        const dim3 grid(gx, gy, gz);
        const bool lin = linear_cell<3>(g);
        const auto kern = mode == 5 ? lin ? k_fast_cell_march<3, 5, S, true> : k_fast_cell_march<3, 5, S, false>
                          : lin     ? k_fast_cell_march<3, 6, S, true>
                                    : k_fast_cell_march<3, 6, S, false>;
        TIMED_LAUNCH("k_fast_cell_z", st, kern, grid, blk, 0, st, dt, sh.xcd, g, m, vol_flux_x, vol_flux_y, vol_flux_z, density1, energy1, mass_flux_z, rho_out, e_out, p_out);
    }
    return hipGetLastError();
}

hipError_t launch_fast_advec_cell(Store s, const DtDev *dt, const Lay &g, const Geo &m, int advect_x, int dir, int sweep_number,
                                  const void *density1, const void *energy1, void *mass_flux_x,
                                  const void *vol_flux_x, void *mass_flux_y, const void *vol_flux_y,
                                  void *mass_flux_z, const void *vol_flux_z, void *rho_out, void *e_out,
                                  void *pressure, const Shape &sh, hipStream_t st)
{
    int mode = 0;
    if (dir == 1) mode = sweep_number == 1 ? 1 : sweep_number == 3 ? 2 : 0;
    else if (dir == 2) mode = sweep_number == 2 ? (advect_x ? 3 : 4) : 0;
    else if (dir == 3) mode = sweep_number == 1 ? 5 : sweep_number == 3 ? 6 : 0;
    if (!mode) return hipErrorInvalidValue;  // the resident driver issues only the reference's sweeps
    if (pressure && sweep_number != 3) return hipErrorInvalidValue;  // only the last sweep's state is final
#define CALL(T)                                                                                                 \
    fast_advec_cell_t<T>(dt, g, m, mode, dir, static_cast<const T *>(density1), static_cast<const T *>(energy1),     \
                         static_cast<T *>(mass_flux_x), static_cast<const T *>(vol_flux_x),                      \
                         static_cast<T *>(mass_flux_y), static_cast<const T *>(vol_flux_y),                      \
                         static_cast<T *>(mass_flux_z), static_cast<const T *>(vol_flux_z),                      \
                         static_cast<T *>(rho_out), static_cast<T *>(e_out), static_cast<T *>(pressure), sh, st)
    return s == ST_F32 ? CALL(float) : CALL(double);
#undef CALL
}

// ---------------------------------------------------------------------------
// Batched over many decks (batch.h): new density1/energy1 go to X_W1/X_W2,
// wherever those and density1/energy1 are at this point of the step.
struct CellSlots {
    int rho, e, rho_out, e_out;
};

__host__ __device__ inline void dims_cell(int dir, const Lay &g, int planes, int &gx, int &gy, int &gz)
{
    const int nx = g.x_max - g.x_min + 1, ny = g.y_max - g.y_min + 1, nz = g.z_max - g.z_min + 1;
    if (dir == 1) {
        const int rows = cell_x_rows(planes);
        gx = (nx + 2 + 59) / 60; gy = ((ny * nz + rows - 1) / rows + CROWS - 1) / CROWS; gz = 1;
    } else if (dir == 2) {
        dims_march<2>(g, planes, gx, gy, gz);
    } else {
        dims_march<3>(g, planes, gx, gy, gz);
    }
}

int batch_blocks_cell(int dir, const Lay &g, int planes)
{
    int gx, gy, gz;
    dims_cell(dir, g, planes, gx, gy, gz);
    return gx * gy * gz;
}

template <int DIR, int MODE, typename S>  // MODE: 0 for the x sweep, which takes `mode`
__global__ void __launch_bounds__(64 * CROWS)
kb_cell(const DeckDev *__restrict__ decks, const int *__restrict__ start, int nd, int mode, int gas, int planes,
        int xcd, CellSlots cs)
{
    int hb, end, step;  // the tiles of this workgroup (persistent when the grid is short)
    tile_walk(start[nd], xcd, hb, end, step);
    for (; hb < end; hb += step) {
        const int d = deck_of(start, nd, hb);
        const DeckDev &D = decks[d];
        int gx, gy, gz;
        dims_cell(DIR, D.g, planes, gx, gy, gz);
        const int lb = hb - start[d];
        const Blk bk{lb % gx, (lb / gx) % gy, lb / (gx * gy), gx, gy, gz};
#define CF(id) static_cast<const S *>(D.f[id])
#define MF(id) static_cast<S *>(D.f[id])
        if constexpr (DIR == 1) {
            cell_x_body<S>(bk, D.g, D.m, mode, cell_x_rows(planes), CF(F_VOL_FLUX_X), CF(F_VOL_FLUX_Y), CF(F_VOL_FLUX_Z), CF(cs.rho),
                           CF(cs.e), MF(F_MASS_FLUX_X), MF(cs.rho_out), MF(cs.e_out), gas ? MF(F_PRESSURE) : nullptr);
        } else {
            auto body = [&](auto lin) {
                cell_march_body<decltype(lin)::value, DIR, MODE, S>(
                    bk, D.g, D.m, CF(F_VOL_FLUX_X), CF(F_VOL_FLUX_Y), CF(F_VOL_FLUX_Z), CF(cs.rho), CF(cs.e),
                    MF(DIR == 2 ? F_MASS_FLUX_Y : F_MASS_FLUX_Z), MF(cs.rho_out), MF(cs.e_out),
                    gas ? MF(F_PRESSURE) : nullptr);
            };
            if (linear_cell<DIR>(D.g)) body(std::true_type{});
            else body(std::false_type{});
        }
#undef CF
#undef MF
        __syncthreads();  // the next tile reuses the workgroup's LDS
    }
}

hipError_t batch_advec_cell(Store s, const DeckDev *decks, int nd, const BatchGrid &bg, int advect_x, int dir,
                            int sweep_number, bool gas, const Slots &sl, const Shape &sh, hipStream_t st)
{
    int mode = 0;
    if (dir == 1) mode = sweep_number == 1 ? 1 : sweep_number == 3 ? 2 : 0;
    else if (dir == 2) mode = sweep_number == 2 ? (advect_x ? 3 : 4) : 0;
    else if (dir == 3) mode = sweep_number == 1 ? 5 : sweep_number == 3 ? 6 : 0;
    if (!mode) return hipErrorInvalidValue;
    if (bg.total == 0) return hipSuccess;
    const dim3 grid(batch_wgs(bg, sh)), blk(64, CROWS);
    const CellSlots cs{sl[F_DENSITY1], sl[F_ENERGY1], sl[X_W1], sl[X_W2]};
    if (gas && sweep_number != 3) return hipErrorInvalidValue;
#define L(D_, M_, T_)                                                                                         \
    TIMED_LAUNCH("kb_cell", st, (kb_cell<D_, M_, T_>), grid, blk, 0, st, decks, bg.start, nd, mode, gas ? 1 : 0, \
                 sh.planes, sh.xcd, cs)
#define LM(T_)                                                                                                \
    if (dir == 1) L(1, 0, T_);                                                                                \
    else if (mode == 3) L(2, 3, T_);                                                                          \
    else if (mode == 4) L(2, 4, T_);                                                                          \
    else if (mode == 5) L(3, 5, T_);                                                                          \
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
