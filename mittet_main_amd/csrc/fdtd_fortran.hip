// fdtd_fortran.hip -- the Fortran lineage's step (ver0040), variant 1 of the
// library: magnetic Hz source points applied before the E update
// (ver0040/cpu_waveform.f90:6-58, cpu_main.f90:104-148), E and H updates over
// the Fortran loop ranges (cpu_eh_field_cpml42.f90:116-252), CPML over its
// shells with every other axis in full range (cpu_cpml4.f90:271-474, including
// the c2 in place of c1 of the psi_Hyx stencil, :400, 413), and per-cell
// permeability in the H coefficients (cpu_eh_field_cpml42.f90:51-53).
//
// A block owns a tile of one plane, a lane one of its cells (the tiles, LDS stencils and
// plane-relative addresses of the C variant's per-cell kernels, fdtd_kernels.hip), and
// applies, in the Fortran order, the field update (where the loop range contains the
// cell) and then the x, y and z CPML corrections (where the shell contains it).  The
// per-cell order of operations is the Fortran one, so the result is that of the
// operator-by-operator loops bit for bit.  Cells of a Fortran shell range outside the
// stored slabs ([0, nc) and [n - nc, n)) have zero profiles there (their psi stays 0 and
// adds 0) and are skipped.  Where an axis' CPML sigma is zero its coefficients are
// exactly 1 and dt/eps' (dt/mu), so their divisions are skipped.
//
// Bound by latency and the 64-bit divisions on the grids this variant is run on: 121 x 51
// x 51 11.2 us per E and H launch, 14.3 and 13.9 with every stencil value loaded from
// global memory and every coefficient divided out on every cell (100 and 108 VGPRs; kept
// below 96 for five waves by computing psi first, or by spilling, 11.2 + 11.6 and 11.4 +
// 14.0).  The source points of a step used to be a launch of their own before it (3.4
// us); both launches now take them off the values they load.
// Non-temporal field loads and stores, which the C variant has beyond the Infinity
// Cache, do not pay here: 200^3 425 us a step without, 431 with.

#include "fdtd_tile.h"

namespace mt {

namespace {

__device__ __forceinline__ const GLOBAL double *cg(const double *p) { return (const GLOBAL double *)p; }
__device__ __forceinline__ GLOBAL double *mg(double *p) { return (GLOBAL double *)p; }

// x / c of a complex x by a real c, as the reference's Fortran evaluates it
// compiled with amdflang: c becomes the complex (c, 0) and each part of the
// quotient is (x c) / (c c) (the textbook complex quotient with zero
// imaginary divisor), which differs from x / c in the last place.  Applies to
// every stencil division, psi update and the source scaling; the real and
// imaginary runs of a complex field take it part by part.
__device__ __forceinline__ double cdivr(double x, double c) { return (x * c) / (c * c); }

// Hz source points of step n in plane k, in their order: Hz(src) -= s[n] dt / mu(src) /
// dx / dy / dz (ver0040/cpu_waveform.f90:6-58), on a value just loaded from plane offset
// o.  Until the step's H launch stores the cell, memory holds the value before.
__device__ __forceinline__ double hz_source(const ShotDev &S, int k, int n, unsigned o, double v)
{
    const int plane = (int)(S.pb >> 3);
    for (int p = 0; p < S.nsrc_h && p < 4; ++p) {
        const int rel = S.src_h[p] - k * plane;
        if ((unsigned)rel < (unsigned)plane && o == (unsigned)rel * 8u)
            v = v - cg(S.amp)[(size_t)p * (S.it - 1) + n];
    }
    return v;
}
__device__ __forceinline__ bool hz_plane(const ShotDev &S, int k)
{
    const int plane = (int)(S.pb >> 3);
    bool any = false;
    for (int p = 0; p < S.nsrc_h && p < 4; ++p)
        any |= (unsigned)(S.src_h[p] - k * plane) < (unsigned)plane;
    return any;
}

// An axis' coefficients (1 - s)/(1 + s) and m/(1 + s), s = sigma dt/(2 eps')
// (cpu_eh_field_cpml42.f90:26-53), m = dt/eps' or dt/mu: the first scales v where the
// component's range holds the cell, the second takes the place of m
__device__ __forceinline__ void coeff(double sigma, double dt, double eps2, double &v, double &m,
                                      bool range)
{
    if (sigma != 0.0) {
        const double s = (sigma * dt) / (2.0 * eps2);
        const double ca = (1.0 - s) / (1.0 + s);
        m = m / (1.0 + s);
        v = range ? ca * v : v;
    }
}

}  // namespace

// Trace samples of step n, components [c0, c0 + 3) of Ex .. Hz, from F [3][n]
__device__ __forceinline__ void rec_v(const ShotDev &S, int n, const double *F, int c0)
{
    for (int q = threadIdx.x; q < 3 * S.nrec; q += blockDim.x) {
        const int comp = q / S.nrec, r = q - comp * S.nrec;
        const double v = cg(F)[(size_t)comp * S.n + S.rec_cell[r]];
        mg(S.traces)[((size_t)(c0 + comp) * S.nrec + r) * S.it + n] = v;
        if (!__builtin_isfinite(v))
            *S.flag = 1;
    }
}

// The first recn blocks gather H of step j - 1 at the receivers, block s for shot s (H is
// not written by this launch).  MANY: launches over several shots, whose members may have
// finished.  They look the step up before their loads; in those of one shot that look
// costs 0.4 % (121 x 51 x 51, 200^3), and they end with its time loop.
template <bool MANY>
__global__ __launch_bounds__(PT) void k_efield_v(const ShotDev *__restrict__ D, int ns,
                                                 const int *__restrict__ pre, int j, int recn)
{
    __shared__ double sh[3 * PT_TILE];
    if ((int)blockIdx.x < recn) {
        if ((int)blockIdx.x < ns) {
            const ShotDev &R = D[blockIdx.x];
            const int n = chunk_step(R) + j - 1;
            if (n < R.it - 1)
                rec_v(R, n, R.h, 3);
        }
        return;
    }
    const int b = blockIdx.x - recn;
    const int s = MANY ? find_shot(pre, ns, b) : 0;
    const ShotDev &S = D[s];
    const int nm = MANY ? chunk_step(S) + j : 0;
    FTile T;
    if (!ftile<false>(S, MANY ? b - pre[s] : b, T))
        return;   // uniform over the block
    if (MANY && nm >= S.it - 1)
        return;   // a member of a batch that has finished its time loop loads nothing
    const int k = T.k, nc = S.nc, ix = S.ix, iy = S.iy, iz = S.iz;
    const bool ax = T.x0 < nc || T.x0 + T.w > ix - nc, ay = T.y0 < nc || T.y0 + T.h > iy - nc;
    const bool az = k < nc || k >= iz - nc, shell = ax || ay || az;
    const int si = ring_slot(S, S.cur + j), so = ring_slot(S, S.cur + j + 1);
    const size_t nb = (size_t)S.n * 8, pb = S.pb, kp = (size_t)k * pb;
    const size_t zm1 = k >= 1 ? kp - pb : kp, zm2 = k >= 2 ? kp - 2 * pb : kp;
    const size_t zp1 = k + 1 < iz ? kp + pb : kp;
    const gcp Hb = cb(S.h), Ein = cb(S.e + (size_t)si * S.sstride) + kp;
    const FLane<2> q(S, T);
    const int hc = halo_comp(q.hk);

    // ---- loads
    double z0 = at(Hb + 2 * nb + kp, q.o);
    const double y0 = at(Hb + nb + kp, q.o), x0 = at(Hb + kp, q.o);
    double hv = 0.0;
    if (q.halo)
        hv = *(const GLOBAL double *)(Hb + kp + (size_t)hc * nb + q.ho);
    const double yzm1 = at(Hb + nb + zm1, q.o), yzp1 = at(Hb + nb + zp1, q.o), yzm2 = at(Hb + nb + zm2, q.o);
    const double xzm1 = at(Hb + zm1, q.o), xzp1 = at(Hb + zp1, q.o), xzm2 = at(Hb + zm2, q.o);
    double ex = at(Ein, q.o), ey = at(Ein + nb, q.o), ez = at(Ein + 2 * nb, q.o);
    const double dte = at(cb(S.cbi) + kp, q.o);   // dt / eps'
    const double eps2 = shell ? at(cb(S.eps) + kp, q.o) : 1.0;
    const int ci = min(q.i, ix - 1), cj = min(q.jj, iy - 1);
    const bool fx = ax && in_face(ci, 2, nc, ix - nc, ix - 1), fy = ay && in_face(cj, 2, nc, iy - nc, iy - 1);
    const bool fz = in_face(k, 2, nc, iz - nc, iz - 1);
    Quad X{0.0, 0.0, 0.0, 0.0}, Y = X;
    const Quad Z = uquad<false>(S.cq[2], k);
    const size_t L0 = (size_t)S.slab[0] * 8, L1 = (size_t)S.slab[1] * 8, L2 = (size_t)S.slab[2] * 8;
    const gmp P0 = mb(S.psi[0]) + (size_t)(unsigned)k * (unsigned)(iy * nc * 16);
    const gmp P1 = mb(S.psi[1]) + (size_t)(unsigned)k * (unsigned)(ix * nc * 16);
    const gmp P2 = mb(S.psi[2]) + (fz ? (size_t)(unsigned)slab_pos(k, iz, nc) * pb : 0);
    unsigned q0 = 0, q1 = 0;
    double ax0 = 0.0, ax1 = 0.0, ay0 = 0.0, ay1 = 0.0, az0 = 0.0, az1 = 0.0;
    if (ax)
        X = quad<false>(S.prof[0], ix, ci);
    else
        X.k = uload(S.cq[0] + (size_t)T.x0 * CQ_N + CQ_E + 1);
    if (ay)
        Y = quad<false>(S.prof[1], iy, cj);
    else
        Y.k = uload(S.cq[1] + (size_t)T.y0 * CQ_N + CQ_E + 1);
    if (fx) {
        q0 = (unsigned)(cj * (2 * nc) + slab_pos(ci, ix, nc)) * 8u;
        ax0 = at(P0, q0);
        ax1 = at(P0 + L0, q0);
    }
    if (fy) {
        q1 = (unsigned)(slab_pos(cj, iy, nc) * ix + ci) * 8u;
        ay0 = at(P1, q1);
        ay1 = at(P1 + L1, q1);
    }
    if (fz) {
        az0 = at(P2, q.o);
        az1 = at(P2 + L2, q.o);
    }
    const int n = MANY ? nm : chunk_step(S) + j;
    if (!MANY && n >= S.it - 1)
        return;   // uniform over the block
    if (hz_plane(S, k)) {
        z0 = hz_source(S, k, n, q.o, z0);
        if (q.halo && hc == 2)
            hv = hz_source(S, k, n, q.ho, hv);
    }
    if (q.own) {
        lds_put(sh, q.a, x0);
        lds_put(sh + PT_TILE, q.a, y0);
        lds_put(sh + 2 * PT_TILE, q.a, z0);
    }
    if (q.halo)
        lds_put(sh, q.ha + (unsigned)hc * (PT_TILE * 8u), hv);
    __syncthreads();
    if (!q.own || q.i >= ix || q.jj >= iy)
        return;

    // ---- arithmetic
    const double c1 = S.c1, c2 = S.c2, dt = S.dt;
    const double *sx = sh, *sy = sh + PT_TILE, *sz = sh + 2 * PT_TILE;
    const unsigned am1 = q.a - q.p, am2 = am1 - q.p, ap1 = q.a + q.p;
    const double hzy = dm(z0, lds_at(sz, am1), lds_at(sz, ap1), lds_at(sz, am2), c1, c2);
    const double hyz = dm(y0, yzm1, yzp1, yzm2, c1, c2);
    const double hxz = dm(x0, xzm1, xzp1, xzm2, c1, c2);
    const double hzx = dm(z0, lds_at(sz, q.a, -8), lds_at(sz, q.a, 8), lds_at(sz, q.a, -16), c1, c2);
    const double hyx = dm(y0, lds_at(sy, q.a, -8), lds_at(sy, q.a, 8), lds_at(sy, q.a, -16), c1, c2);
    const double hxy = dm(x0, lds_at(sx, am1), lds_at(sx, ap1), lds_at(sx, am2), c1, c2);
    const double cux = cdivr(hzy, Y.k) - cdivr(hyz, Z.k);
    const double cuy = cdivr(hxz, Z.k) - cdivr(hzx, X.k);
    const double cuz = cdivr(hyx, X.k) - cdivr(hxy, Y.k);
    // e_field_cpml4 (:125-155)
    const bool ri = q.i >= 2 && q.i < ix - 1, rj = q.jj >= 2 && q.jj < iy - 1, rk = k >= 2 && k < iz - 1;
    double cbx = dte, cby = dte, cbz = dte;
    if (ax)
        coeff(X.s, dt, eps2, ex, cbx, rk && rj);
    if (rk && rj)
        ex = ex + cbx * cux;
    if (ay)
        coeff(Y.s, dt, eps2, ey, cby, rk && ri);
    if (rk && ri)
        ey = ey + cby * cuy;
    if (az)
        coeff(Z.s, dt, eps2, ez, cbz, rj && ri);
    if (rj && ri)
        ez = ez + cbz * cuz;
    // CPML_E4 (cpu_cpml4.f90:281-358): x, then y, then z
    if (ax && fx) {
        const double h = S.dl[0];
        ax0 = X.b * ax0 + cdivr(X.c * hyx, h);   // psi_Ezx
        ax1 = X.b * ax1 + cdivr(X.c * hzx, h);   // psi_Eyx
        put_s<false>(P0, q0, ax0);
        put_s<false>(P0 + L0, q0, ax1);
        ez = ez + cbz * ax0;
        ey = ey - cby * ax1;
    }
    if (ay && fy) {
        const double h = S.dl[1];
        ay0 = Y.b * ay0 + cdivr(Y.c * hzy, h);   // psi_Exy
        ay1 = Y.b * ay1 + cdivr(Y.c * hxy, h);   // psi_Ezy
        put_s<false>(P1, q1, ay0);
        put_s<false>(P1 + L1, q1, ay1);
        ex = ex + cbx * ay0;
        ez = ez - cbz * ay1;
    }
    if (az && fz) {
        const double h = S.dl[2];
        az0 = Z.b * az0 + cdivr(Z.c * hxz, h);   // psi_Eyz
        az1 = Z.b * az1 + cdivr(Z.c * hyz, h);   // psi_Exz
        put_s<false>(P2, q.o, az0);
        put_s<false>(P2 + L2, q.o, az1);
        ey = ey + cby * az0;
        ex = ex - cbx * az1;
    }
    const gmp Eout = mb(S.e + (size_t)so * S.sstride) + kp;
    put_s<false>(Eout, q.o, ex);
    put_s<false>(Eout + nb, q.o, ey);
    put_s<false>(Eout + 2 * nb, q.o, ez);
}

// The first recn blocks gather E of step j at the receivers, block s for shot s
// (E is not written by this launch).
template <bool MANY>
__global__ __launch_bounds__(PT) void k_hfield_v(const ShotDev *__restrict__ D, int ns,
                                                 const int *__restrict__ pre, int j, int recn)
{
    __shared__ double sh[3 * PT_TILE];
    if ((int)blockIdx.x < recn) {
        if ((int)blockIdx.x < ns) {
            const ShotDev &R = D[blockIdx.x];
            const int n = chunk_step(R) + j;
            if (n < R.it - 1)
                rec_v(R, n, R.e + (size_t)((R.cur + j + 1) % R.ring) * R.sstride, 0);
        }
        return;
    }
    const int b = blockIdx.x - recn;
    const int s = MANY ? find_shot(pre, ns, b) : 0;
    const ShotDev &S = D[s];
    const int nm = MANY ? chunk_step(S) + j : 0;
    FTile T;
    if (!ftile<false>(S, MANY ? b - pre[s] : b, T))
        return;   // uniform over the block
    if (MANY && nm >= S.it - 1)
        return;   // a member of a batch that has finished its time loop loads nothing
    const int k = T.k, nc = S.nc, ix = S.ix, iy = S.iy, iz = S.iz;
    const bool ax = T.x0 < nc || T.x0 + T.w > ix - nc, ay = T.y0 < nc || T.y0 + T.h > iy - nc;
    const bool az = k < nc || k >= iz - nc, shell = ax || ay || az;
    const int so = ring_slot(S, S.cur + j + 1);
    const size_t nb = (size_t)S.n * 8, pb = S.pb, kp = (size_t)k * pb;
    const size_t zm1 = k >= 1 ? kp - pb : kp;
    const size_t zp1 = k + 1 < iz ? kp + pb : kp, zp2 = k + 2 < iz ? kp + 2 * pb : kp;
    const gcp Eb = cb(S.e + (size_t)so * S.sstride);
    const gmp Hk = mb(S.h) + kp;
    const FLane<1> q(S, T);
    const int hc = halo_comp(q.hk);

    // ---- loads
    const double z0 = at(Eb + 2 * nb + kp, q.o), y0 = at(Eb + nb + kp, q.o), x0 = at(Eb + kp, q.o);
    double hv = 0.0;
    if (q.halo)
        hv = *(const GLOBAL double *)(Eb + kp + (size_t)hc * nb + q.ho);
    const double yzp1 = at(Eb + nb + zp1, q.o), yzp2 = at(Eb + nb + zp2, q.o), yzm1 = at(Eb + nb + zm1, q.o);
    const double xzp1 = at(Eb + zp1, q.o), xzp2 = at(Eb + zp2, q.o), xzm1 = at(Eb + zm1, q.o);
    double hx = at(Hk, q.o), hy = at(Hk + nb, q.o), hz = at(Hk + 2 * nb, q.o);
    const double mu = at(cb(S.mu) + kp, q.o), eps2 = shell ? at(cb(S.eps) + kp, q.o) : 1.0;
    const int ci = min(q.i, ix - 1), cj = min(q.jj, iy - 1);
    const bool fx = ax && in_face(ci, 1, nc, ix - nc, ix - 2), fy = ay && in_face(cj, 1, nc, iy - nc, iy - 2);
    const bool fz = in_face(k, 1, nc, iz - nc, iz - 2);
    Quad X{0.0, 0.0, 0.0, 0.0}, Y = X;
    const Quad Z = uquad<true>(S.cq[2], k);
    const size_t L0 = (size_t)S.slab[0] * 8, L1 = (size_t)S.slab[1] * 8, L2 = (size_t)S.slab[2] * 8;
    const gmp P0 = mb(S.psi[0]) + PSI_HP * L0 + (size_t)(unsigned)k * (unsigned)(iy * nc * 16);
    const gmp P1 = mb(S.psi[1]) + PSI_HP * L1 + (size_t)(unsigned)k * (unsigned)(ix * nc * 16);
    const gmp P2 = mb(S.psi[2]) + PSI_HP * L2 + (fz ? (size_t)(unsigned)slab_pos(k, iz, nc) * pb : 0);
    unsigned q0 = 0, q1 = 0;
    double ax0 = 0.0, ax1 = 0.0, ay0 = 0.0, ay1 = 0.0, az0 = 0.0, az1 = 0.0;
    if (ax)
        X = quad<true>(S.prof[0], ix, ci);
    else
        X.k = uload(S.cq[0] + (size_t)T.x0 * CQ_N + CQ_H + 1);
    if (ay)
        Y = quad<true>(S.prof[1], iy, cj);
    else
        Y.k = uload(S.cq[1] + (size_t)T.y0 * CQ_N + CQ_H + 1);
    if (fx) {
        q0 = (unsigned)(cj * (2 * nc) + slab_pos(ci, ix, nc)) * 8u;
        ax0 = at(P0, q0);
        ax1 = at(P0 + L0, q0);
    }
    if (fy) {
        q1 = (unsigned)(slab_pos(cj, iy, nc) * ix + ci) * 8u;
        ay0 = at(P1, q1);
        ay1 = at(P1 + L1, q1);
    }
    if (fz) {
        az0 = at(P2, q.o);
        az1 = at(P2 + L2, q.o);
    }
    if (q.own) {
        lds_put(sh, q.a, x0);
        lds_put(sh + PT_TILE, q.a, y0);
        lds_put(sh + 2 * PT_TILE, q.a, z0);
    }
    if (q.halo)
        lds_put(sh, q.ha + (unsigned)hc * (PT_TILE * 8u), hv);
    __syncthreads();
    // the step is looked up behind the loads
    const int n = MANY ? nm : chunk_step(S) + j;
    if (n >= S.it - 1 || !q.own || q.i >= ix || q.jj >= iy)
        return;
    if (hz_plane(S, k))
        hz = hz_source(S, k, n, q.o, hz);

    // ---- arithmetic
    const double c1 = S.c1, c2 = S.c2, dt = S.dt;
    const double *sx = sh, *sy = sh + PT_TILE, *sz = sh + 2 * PT_TILE;
    const unsigned am1 = q.a - q.p, ap1 = q.a + q.p, ap2 = ap1 + q.p;
    const double zxp1 = lds_at(sz, q.a, 8), zxp2 = lds_at(sz, q.a, 16), zxm1 = lds_at(sz, q.a, -8);
    const double ezy = dp(lds_at(sz, ap1), z0, lds_at(sz, ap2), lds_at(sz, am1), c1, c2);
    const double eyz = dp(yzp1, y0, yzp2, yzm1, c1, c2);
    const double exz = dp(xzp1, x0, xzp2, xzm1, c1, c2);
    const double ezx = dp(zxp1, z0, zxp2, zxm1, c1, c2);
    const double eyx = dp(lds_at(sy, q.a, 8), y0, lds_at(sy, q.a, 16), lds_at(sy, q.a, -8), c1, c2);
    const double exy = dp(lds_at(sx, ap1), x0, lds_at(sx, ap2), lds_at(sx, am1), c1, c2);
    const double cux = cdivr(ezy, Y.k) - cdivr(eyz, Z.k);
    const double cuy = cdivr(exz, Z.k) - cdivr(ezx, X.k);
    const double cuz = cdivr(eyx, X.k) - cdivr(exy, Y.k);
    const double dtm = dt / mu;
    // h_field_cpml4 (:221-251)
    const bool ri = q.i >= 1 && q.i < ix - 2, rj = q.jj >= 1 && q.jj < iy - 2, rk = k >= 1 && k < iz - 2;
    double dbx = dtm, dby = dtm, dbz = dtm;
    if (ax)
        coeff(X.s, dt, eps2, hx, dbx, rk && rj);
    if (rk && rj)
        hx = hx - dbx * cux;
    if (ay)
        coeff(Y.s, dt, eps2, hy, dby, rk && ri);
    if (rk && ri)
        hy = hy - dby * cuy;
    if (az)
        coeff(Z.s, dt, eps2, hz, dbz, rj && ri);
    if (rj && ri)
        hz = hz - dbz * cuz;
    // CPML_H4 (cpu_cpml4.f90:394-471): x, then y, then z
    if (ax && fx) {
        const double h = S.dl[0];
        // psi_Hyx takes c2 where the stencil has c1 (cpu_cpml4.f90:400, 413)
        const double zx = c1 * zxp1 - c2 * z0 + c2 * zxp2 - c2 * zxm1;
        ax0 = X.b * ax0 + cdivr(X.c * eyx, h);   // psi_Hzx
        ax1 = X.b * ax1 + cdivr(X.c * zx, h);    // psi_Hyx
        put_s<false>(P0, q0, ax0);
        put_s<false>(P0 + L0, q0, ax1);
        hz = hz - dbz * ax0;
        hy = hy + dby * ax1;
    }
    if (ay && fy) {
        const double h = S.dl[1];
        ay0 = Y.b * ay0 + cdivr(Y.c * ezy, h);   // psi_Hxy
        ay1 = Y.b * ay1 + cdivr(Y.c * exy, h);   // psi_Hzy
        put_s<false>(P1, q1, ay0);
        put_s<false>(P1 + L1, q1, ay1);
        hx = hx - dbx * ay0;
        hz = hz + dbz * ay1;
    }
    if (az && fz) {
        const double h = S.dl[2];
        az0 = Z.b * az0 + cdivr(Z.c * exz, h);   // psi_Hyz
        az1 = Z.b * az1 + cdivr(Z.c * eyz, h);   // psi_Hxz
        put_s<false>(P2, q.o, az0);
        put_s<false>(P2 + L2, q.o, az1);
        hy = hy - dby * az0;
        hx = hx + dbx * az1;
    }
    put_s<false>(Hk, q.o, hx);
    put_s<false>(Hk + nb, q.o, hy);
    put_s<false>(Hk + 2 * nb, q.o, hz);
}

hipError_t launch_efield_v(const ShotDev *d, int ns, const int *pre, int nblocks, int j, hipStream_t st,
                           bool rec_prev)
{
    if (nblocks <= 0)
        return rec_prev ? hipErrorInvalidValue : hipSuccess;
    const int recn = rec_prev && j > 0 ? (ns + 7) & ~7 : 0;
    if (ns > 1)
        hipLaunchKernelGGL(k_efield_v<true>, dim3(recn + nblocks), dim3(PT), 0, st, d, ns, pre, j, recn);
    else
        hipLaunchKernelGGL(k_efield_v<false>, dim3(recn + nblocks), dim3(PT), 0, st, d, ns, pre, j, recn);
    return hipGetLastError();
}

hipError_t launch_hfield_v(const ShotDev *d, int ns, const int *pre, int nblocks, int j, hipStream_t st,
                           bool rec_e)
{
    if (nblocks <= 0)
        return rec_e ? hipErrorInvalidValue : hipSuccess;
    const int recn = rec_e ? (ns + 7) & ~7 : 0;
    if (ns > 1)
        hipLaunchKernelGGL(k_hfield_v<true>, dim3(recn + nblocks), dim3(PT), 0, st, d, ns, pre, j, recn);
    else
        hipLaunchKernelGGL(k_hfield_v<false>, dim3(recn + nblocks), dim3(PT), 0, st, d, ns, pre, j, recn);
    return hipGetLastError();
}

}  // namespace mt
