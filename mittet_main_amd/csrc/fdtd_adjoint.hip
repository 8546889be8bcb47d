// fdtd_adjoint.hip -- exact discrete adjoint of the fused forward step and the
// gradient of a receiver misfit with respect to eps' (hence sigma).
//
// Forward step n (state u = (E, H, psiE, psiH), all linear for fixed sigma):
//   E-phase : E' = ca.E + cb.curl-(H)  on the reference's update ranges,
//             psiE' = be.psiE + ce.D-(H)/dl on the CPML faces, E += +-cb.psiE'
//   source  : E'[src] -= amp[n],  amp ~ 1/sigma[src]
//   H-phase : H' = da.H - db.curl+(E'), psiH' = bh.psiH + ch.D+(E')/dl, H += +-db.psiH'
// (satan_i/fwi3d_cpu_function_v1.4.c:1184-1290, fwi3d_cpu_cpmlabc_v1.4.c:402-679).
// The adjoint applies the transposed sub-steps in reverse order.  Transposes
// are written as gathers: the transpose of D+ is -D- and of D- is -D+, taken
// over the same range masks and with the weights of the cell the forward
// stencil was centred on.  Gradient terms use
//   d ca/de = 2K/(e+K)^2, d cb/de = -dt/(e+K)^2          (K = esig*dt/2)
//   d da/de = 2Km/(e+Km)^2, d db/de = (dt/mu0) Km/(e+Km)^2 (Km = msig*dt/2)
// with e = eps' = sigma/(2 omega0): ca = (e-K)/(e+K), cb = dt/(e+K) are the
// reference's coefficients rewritten.
//
// Order of a step, per cell outside the LDS region (phase H gathers with the
// weights of the H update, phase E with those of the E update):
//   H local  w = db lH, psi-H adjoint, gradient through db and da, lH <- da lH
//   H gather lE += transposed curl+ (w) and transposed psi-H stencils
//   E local  w = cb lE, psi-E adjoint, gradient through cb and ca, lE <- ca lE
//   E gather lH += transposed curl- (w) and transposed psi-E stencils
// A gather needs every cell's weights, a local part only its own cell, so each
// gather shares its launch with the local part after it: (H gather, E local) and
// (E gather, H local of the step before).
//
// Weights: for axis a with p = a+1, q = a+2 (mod 3) a gather along a needs the
// weight of component q and of component p, each over kappa of that axis, and
// the two psi rows of the axis, which take the same stencil.  Both are summed
// where they arise into two arrays per axis, P_a (weight of component q) and Q_a
// (of component p), so a gather along a is two plain stencils wherever the cell
// lies:
//   H: P_a = w_q/khd_a - t1, Q_a = w_p/khd_a + t0;  lE_p += D-_a P_a, lE_q -= D-_a Q_a
//   E: P_a = w_q/ked_a + t0, Q_a = w_p/ked_a - t1;  lH_p -= D+_a P_a, lH_q += D+_a Q_a
// with t0, t1 the psi weights (c m h of the two rows, 0 off the faces).
//
// In the LDS region (ca = da = 1, kappa = 1, no psi) the arrays lE and lH hold the
// weights themselves, cb lE and db lH, so that its kernels march plain stencils
// over them as the forward LDS kernels do; its gradient term is then
// -cb lE . (E' + amp - E)/dt.  Beyond the region's faces these read P_a of axis
// d + 1 as the weight of component d, and next to them they write P_a and Q_a for
// the per-cell passes' stencils.
//
// Gradient terms need no stencil: the forward step itself holds what multiplies
// the coefficients.  With K = esig dt/2, r = 1/(e + K) and E' = ca E + cb X - amp,
//   dca/de E + dcb/de X = 2 K r^2 E - r (E' + amp - ca E) = -r (E' + amp - E),
// for cells that only a psi correction changes (ca = 1) as well, and with
// Km = msig dt/2, r = 1/(e + Km)
//   dda/de H - ddb/de X = (Km r/e) (H' + H)   (H' - H where only psi acts).
// E' - E cancels where the field changes little in a step.  Its rounding is that of E, as
// large as that of the curl it stands for while the field is a wave (cb |H| / dl is about
// |E| / 2).  Against 64-bit values the gradient's relative error is 6.4e-15 at 152^3 with 200
// steps (5.8e-15 with the stencils) and 1.3e-15 at 61 x 50 x 44 with 160 (1.4e-15), and in one
// dimension 2.9e-15 after 16 000 steps (2.2e-15).
#include "fdtd_tile.h"

namespace mt {

namespace {

__device__ __forceinline__ bool in_region(const AdjArgs &A, int i, int j, int k)
{
    return i >= A.lo[0] && i < A.hi[0] && j >= A.lo[1] && j < A.hi[1] && k >= A.lo[2] &&
           k < A.hi[2];
}

}  // namespace

// adjoint receiver source: lE[comp][rec] += g[comp][rec] (state after step n).  At most
// one receiver of a cell has a sensitivity that is not zero (the host sums those on one
// cell), and only that lane touches the cell: each lane loads, adds and stores by itself.
__global__ void k_adj_inject(AdjArgs A, const double *__restrict__ g, int nrec,
                             const int *__restrict__ rec)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 3 * nrec)
        return;
    const double gq = g[q];
    if (gq == 0.0)
        return;
    const int comp = q / nrec, r = q - comp * nrec, c = rec[r];
    const int i = c % A.ix, t = c / A.ix, j = t % A.iy, k = t / A.iy;
    if (in_region(A, i, j, k))
        A.lE[(size_t)comp * A.n + c] += A.cbi[c] * gq;
    else
        A.lE[(size_t)comp * A.n + c] += gq;
}

// Per-cell pass over the tiles outside the LDS region (every tile without one).
// EP = false: H gather into lE, then the E local part; EP = true: E gather into
// lH, then the H local part of the step before (gather or local switched off at
// the ends of a replayed segment).  The x and y stencils go through LDS as in the
// forward per-cell kernels (four weight arrays, one halo value per lane), the z
// stencils are loaded directly.  Bound by memory: 6 weights read and 6 written,
// lambda, the forward states, the gradient and psi are about 250 B per cell and
// pass.  152^3 with a 12-cell CPML, per step: 101 and 98 us of events around the two
// launches, 72 and 44 us around those of the region.  With the step's replay a step
// takes 512 us there, 574 before each gather shared its launch with a local part (then
// 8 launches a step); 45 us at 61 x 50 x 44, where every cell is this kernel's, 89 then.
template <bool EP>
__global__ __launch_bounds__(PT) void k_adj_cell(AdjArgs A, int gather, int local)
{
    __shared__ double sh[4 * PT_TILE];   // P_x, Q_x (x stencils), P_y, Q_y (y stencils)
    FTile T;
    if (!ftile<false>(A, blockIdx.x, T))
        return;   // uniform over the block
    const int k = T.k, nc = A.nc;
    const bool ax = T.x0 < nc || T.x0 + T.w > A.ix - nc, ay = T.y0 < nc || T.y0 + T.h > A.iy - nc;
    const bool az = k < nc || k >= A.iz - nc;
    const size_t nb = (size_t)A.n * 8, pb = A.pb, kp = (size_t)k * pb;
    const FLane<EP ? 1 : 2> q(A, T);
    const bool ing = q.own && q.i < A.ix && q.jj < A.iy;
    // cells of the LDS region belong to its kernels
    const bool mine = ing && q.jj < T.yend && !in_region(A, q.i, q.jj, k);
    const int ci = min(q.i, A.ix - 1), cj = min(q.jj, A.iy - 1);

    // ---- loads
    const gcp U = cb(EP ? A.ue : A.uh), Uk = U + kp;   // arrays P_x, Q_x, P_y, Q_y, P_z, Q_z
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0, hv = 0.0, pz[4], qz[4];
    if (gather) {
        s0 = at(Uk, q.o);
        s1 = at(Uk + nb, q.o);
        s2 = at(Uk + 2 * nb, q.o);
        s3 = at(Uk + 3 * nb, q.o);
        if (q.halo && q.hin)   // rows of P_y, Q_y, columns of P_x, Q_x
            hv = *(const GLOBAL double *)(Uk + (size_t)(q.hk ^ 2) * nb + q.ho);
        // planes of the z stencil: D- (k, k-1, k+1, k-2), D+ (k+1, k, k+2, k-1)
        const int off[4] = {EP ? 1 : 0, EP ? 0 : -1, EP ? 2 : 1, EP ? -1 : -2};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int z = k + off[r];
            pz[r] = qz[r] = 0.0;
            if (z >= 0 && z < A.iz) {
                pz[r] = at(U + 4 * nb + (size_t)z * pb, q.o);
                qz[r] = at(U + 5 * nb + (size_t)z * pb, q.o);
            }
        }
    }
    const gmp LO = mb(EP ? A.lH : A.lE) + kp;
    double l[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        l[d] = at(LO + (size_t)d * nb, q.o);
    const bool shell = ax || ay || az;
    // forward state of the gradient terms: E on every cell, H only where a
    // magnetic CPML conductivity is nonzero (a shell)
    const bool grd = local && (!EP || shell);
    double f0[3] = {0.0, 0.0, 0.0}, f1[3] = {0.0, 0.0, 0.0}, e = 1.0, g0 = 0.0;
    if (grd) {
        e = at(cb(A.eps) + kp, q.o);
        g0 = at(cb(A.grad) + kp, q.o);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            f0[d] = at_s<false>(cb(EP ? A.H0 : A.E0) + (size_t)d * nb + kp, q.o);
            f1[d] = at_s<false>(cb(EP ? A.H1 : A.E1) + (size_t)d * nb + kp, q.o);
        }
    }
    // an axis' sigma, b, c and 1/(kappa dl), and the cell's psi of that axis
    const int PS = EP ? PR_MSIG : PR_ESIG, PB = EP ? PR_BH : PR_BE, PC = EP ? PR_CH : PR_CE;
    const int idx[3] = {ci, cj, k}, len[3] = {A.ix, A.iy, A.iz};
    const bool act[3] = {ax, ay, az};
    double sg[3] = {0.0, 0.0, 0.0}, pbv[3], pcv[3], rk[3], m0[3], m1[3];
    gmp psi[3];
    unsigned qo[3];
    bool face[3] = {false, false, false};
    int fl = 0;
    if (local) {
        fl = uload(A.fl[2] + k) &
             (ax ? *(const GLOBAL int *)(cb(A.fl[0]) + (unsigned)(ci * 4)) : uload(A.fl[0] + T.x0)) &
             (ay ? *(const GLOBAL int *)(cb(A.fl[1]) + (unsigned)(cj * 4)) : uload(A.fl[1] + T.y0));
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            rk[a] = A.rdl[a];
            if (!act[a])
                continue;
            const gcp P = cb(A.prof[a]);
            const unsigned o = (unsigned)idx[a] * 8u, rw = (unsigned)len[a] * 8u;
            sg[a] = at(P, o + PS * rw);
            rk[a] = at(cb(A.rp[a]), o + (EP ? rw : 0u));
            face[a] = (fl & ((EP ? FL_PHX : FL_PEX) << a)) != 0;
            if (!face[a])
                continue;
            const int sp = idx[a] < nc ? idx[a] : idx[a] - (len[a] - 2 * nc);
            psi[a] = mb(A.lpsi[a]) + (size_t)A.slab[a] * (EP ? 16 : 0);
            if (a == 0) {
                psi[a] += (size_t)(unsigned)k * (unsigned)(A.iy * nc * 16);
                qo[a] = (unsigned)(cj * (2 * nc) + sp) * 8u;
            } else if (a == 1) {
                psi[a] += (size_t)(unsigned)k * (unsigned)(A.ix * nc * 16);
                qo[a] = (unsigned)(sp * A.ix + ci) * 8u;
            } else {
                psi[a] += (size_t)(unsigned)sp * pb;
                qo[a] = q.o;
            }
            pbv[a] = at(P, o + PB * rw);
            pcv[a] = at(P, o + PC * rw) * A.rdl[a];
            m0[a] = at(psi[a], qo[a]);
            m1[a] = at(psi[a] + (size_t)A.slab[a] * 8, qo[a]);
        }
    }

    // ---- gather
    const double c1 = A.c1, c2 = A.c2;
    if (gather) {
        if (q.own) {
            lds_put(sh, q.a, ing ? s0 : 0.0);
            lds_put(sh + PT_TILE, q.a, ing ? s1 : 0.0);
            lds_put(sh + 2 * PT_TILE, q.a, ing ? s2 : 0.0);
            lds_put(sh + 3 * PT_TILE, q.a, ing ? s3 : 0.0);
        }
        if (q.halo)
            lds_put(sh, q.ha + (unsigned)((q.hk ^ 2) * PT_TILE) * 8u, hv);
        __syncthreads();
        if (!mine)
            return;
        const unsigned am1 = q.a - q.p, ap1 = q.a + q.p;
        double D[6];   // P_x, Q_x, P_y, Q_y, P_z, Q_z
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const double *sx = sh + m * PT_TILE, *sy = sh + (2 + m) * PT_TILE;
            const double ox = m ? s1 : s0, oy = m ? s3 : s2;
            if (EP) {
                D[m] = c1 * lds_at(sx, q.a, 8) - c1 * ox + c2 * lds_at(sx, q.a, 16) - c2 * lds_at(sx, q.a, -8);
                D[2 + m] = c1 * lds_at(sy, ap1) - c1 * oy + c2 * lds_at(sy, ap1 + q.p) - c2 * lds_at(sy, am1);
            } else {
                D[m] = c1 * ox - c1 * lds_at(sx, q.a, -8) + c2 * lds_at(sx, q.a, 8) - c2 * lds_at(sx, q.a, -16);
                D[2 + m] = c1 * oy - c1 * lds_at(sy, am1) + c2 * lds_at(sy, ap1) - c2 * lds_at(sy, am1 - q.p);
            }
            const double *z = m ? qz : pz;
            D[4 + m] = c1 * z[0] - c1 * z[1] + c2 * z[2] - c2 * z[3];
        }
        // H: lE_p += D-P, lE_q -= D-Q; E: lH_p -= D+P, lH_q += D+Q
        const double d0 = D[4] - D[3], d1 = D[0] - D[5], d2 = D[2] - D[1];
        l[0] += EP ? -d0 : d0;
        l[1] += EP ? -d1 : d1;
        l[2] += EP ? -d2 : d2;
    } else if (!mine) {
        return;
    }
    const int c = (int)(k * (A.pb >> 3) + (q.o >> 3));
    const bool src = !EP && c == A.src_cell;
    if (src) {
        // E[src] -= amp (amp ~ 1/sigma): d/dsigma = +amp/sigma  (kept in sigma units)
        A.grad_src[0] += (A.src_comp == 0 ? l[0] : (A.src_comp == 1 ? l[1] : l[2])) * A.amp_n / A.sig_src;
    }

    // ---- local part
    double w[6];
    if (local) {
        double w3[3], cf[3], g = 0.0, ln[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const bool up = (fl & ((EP ? FL_UHX : FL_UEX) << d)) != 0;
            const double K = sg[d] * A.dt / 2.0;
            ln[d] = l[d];
            if (EP && !shell) {   // e was not loaded: db = dt/mu0, da = 1
                cf[d] = A.dbi;
            } else {
                const double r = 1.0 / (e + K);
                if (EP) {
                    cf[d] = K != 0.0 ? A.dbi * e * r : A.dbi;
                    g += l[d] * (K * r / e) * (up ? f1[d] + f0[d] : f1[d] - f0[d]);
                } else {
                    cf[d] = A.dt * r;
                    const double df = f1[d] - f0[d] + (src && A.src_comp == d ? A.amp_n : 0.0);
                    g -= l[d] * r * df;
                }
                if (up && K != 0.0)
                    ln[d] = l[d] * (e - K) * r;
            }
            w3[d] = up ? cf[d] * l[d] : 0.0;
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int p = (a + 1) % 3, qq = (a + 2) % 3;
            double t0 = 0.0, t1 = 0.0;
            if (face[a]) {
                // psi0 feeds E_q (+cb_q) or H_p (+db_p), psi1 E_p (-cb_p) or H_q (-db_q)
                m0[a] = EP ? m0[a] + cf[p] * l[p] : m0[a] + cf[qq] * l[qq];
                m1[a] = EP ? m1[a] - cf[qq] * l[qq] : m1[a] - cf[p] * l[p];
                t0 = pcv[a] * m0[a];
                t1 = pcv[a] * m1[a];
            }
            w[2 * a] = EP ? w3[qq] * rk[a] - t1 : w3[qq] * rk[a] + t0;
            w[2 * a + 1] = EP ? w3[p] * rk[a] + t0 : w3[p] * rk[a] - t1;
        }
        const gmp W = mb(EP ? A.uh : A.ue) + kp;
#pragma unroll
        for (int r = 0; r < 6; ++r)
            put_s<false>(W + (size_t)r * nb, q.o, w[r]);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (face[a]) {
                put_s<false>(psi[a], qo[a], pbv[a] * m0[a]);
                put_s<false>(psi[a] + (size_t)A.slab[a] * 8, qo[a], pbv[a] * m1[a]);
            }
        if (grd)
            put_s<false>(mb(A.grad) + kp, q.o, g0 + g);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            l[d] = ln[d];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d)
        put_s<false>(LO + (size_t)d * nb, q.o, l[d]);
}

// ------------------------------------------------------------------------
// LDS z-marching kernels of the adjoint over its region.  A block owns a 64 x LY
// column and marches lkb planes along z, as the forward LDS kernels.  The H-phase
// kernel adds cb times the transposed curl+ of kH to kE (the stencil pattern of
// the forward E kernel) and the gradient term; the E-phase kernel adds db times
// the transposed curl- of kE to kH (the pattern of the forward H kernel).

namespace {

constexpr int ANT = LX * LY;

template <int XL, int XR, int YL, int YR> struct ATile {
    static constexpr int W = LX + XL + XR, H = LY + YL + YR, N = W * H;
    static constexpr int R = (N + ANT - 1) / ANT;   // elements per lane
};

// Weight of component d at cells outside the region: P of axis d + 1 (kappa = 1 and
// no psi row within the stencils' reach of the region), times that axis' dl
__device__ __forceinline__ gcp wout(const AdjArgs &A, const double *u, int d)
{
    return cb(u) + (size_t)(2 * ((d + 1) % 3)) * A.n * 8;
}

// Weights of component d on the planes of a tile (halo XL/YL before the tile), f the
// region's array and u the passes' weights.  Which of the two a tile element reads
// follows from its column, once for all planes of the region's z range; it keeps
// its byte offset in a plane and that choice, so a plane costs one scalar-base load
// per element.  Coordinates beyond (xmax, ymax) are clamped onto them: those
// elements are read only by the idle lanes of a partial tile.
template <class T, int XL, int YL> struct WTile {
    unsigned o[T::R];
    bool in[T::R];
    double r[T::R];
    gcp fin, fout;
    double dl;
    __device__ __forceinline__ WTile(const AdjArgs &A, const double *f, const double *u, int d,
                                     int x0, int y0, int xmax, int ymax)
        : fin(cb(f) + (size_t)d * A.n * 8), fout(wout(A, u, d)), dl(A.dl[(d + 1) % 3])
    {
#pragma unroll
        for (int q = 0; q < T::R; ++q) {
            const int e = min((int)threadIdx.x + q * ANT, T::N - 1);
            const int gx = min(x0 - XL + e % T::W, xmax), gy = min(y0 - YL + e / T::W, ymax);
            o[q] = (unsigned)gy * A.row + (unsigned)gx * 8u;
            in[q] = gx >= A.lo[0] && gx < A.hi[0] && gy >= A.lo[1] && gy < A.hi[1];
        }
    }
    __device__ __forceinline__ void load(const AdjArgs &A, int k)
    {
        const bool zin = k >= A.lo[2] && k < A.hi[2];
        const gcp pi = fin + (size_t)k * A.pb, po = fout + (size_t)k * A.pb;
#pragma unroll
        for (int q = 0; q < T::R; ++q) {
            if (zin && in[q])
                r[q] = at(pi, o[q]);
            else
                r[q] = at(po, o[q]);
        }
    }
    __device__ __forceinline__ void store(const AdjArgs &A, int k, double *lds) const
    {
        const bool zin = k >= A.lo[2] && k < A.hi[2];
#pragma unroll
        for (int q = 0; q < T::R; ++q) {
            const int e = threadIdx.x + q * ANT;
            if (e < T::N)
                lds[e] = zin && in[q] ? r[q] : dl * r[q];
        }
    }
};

// weight of component d at the lane's own column (in the region's xy range)
__device__ __forceinline__ double wcol(const AdjArgs &A, const double *f, const double *u, int d,
                                       int k, unsigned o)
{
    const size_t kp = (size_t)k * A.pb;
    if (k < A.lo[2] || k >= A.hi[2])
        return at(wout(A, u, d) + kp, o) * A.dl[(d + 1) % 3];
    return at(cb(f) + (size_t)d * A.n * 8 + kp, o);
}

// Weight arrays of a region cell that the per-cell passes' stencils reach: along
// an axis, the two cells next to the region's faces on that axis
__device__ __forceinline__ void rim(const AdjArgs &A, double *u, int i, int j, int k, unsigned o,
                                    double w0, double w1, double w2)
{
    const size_t nb = (size_t)A.n * 8;
    const gmp W = mb(u) + (size_t)k * A.pb;
    if (i < A.lo[0] + 2 || i >= A.hi[0] - 2) {
        put_s<false>(W, o, w2 * A.rdl[0]);
        put_s<false>(W + nb, o, w1 * A.rdl[0]);
    }
    if (j < A.lo[1] + 2 || j >= A.hi[1] - 2) {
        put_s<false>(W + 2 * nb, o, w0 * A.rdl[1]);
        put_s<false>(W + 3 * nb, o, w2 * A.rdl[1]);
    }
    if (k < A.lo[2] + 2 || k >= A.hi[2] - 2) {
        put_s<false>(W + 4 * nb, o, w1 * A.rdl[2]);
        put_s<false>(W + 5 * nb, o, w0 * A.rdl[2]);
    }
}

// block -> (region tile, z-chunk), XCD-contiguous numbering
__device__ __forceinline__ bool acol(const AdjArgs &A, int &x0, int &y0, int &k0, int &k1)
{
    const int b = blockIdx.x;
    const int L = (b & 7) * (A.lb_pad >> 3) + (b >> 3);
    if (L >= A.lb)
        return false;
    const int tx = L % A.ltx, r = L / A.ltx;
    const int ty = r % A.lty, kz = r / A.lty;
    x0 = A.lo[0] + tx * LX;
    y0 = A.lo[1] + ty * LY;
    k0 = A.lo[2] + kz * A.lkb;
    k1 = min(k0 + A.lkb, A.hi[2]);
    return true;
}

}  // namespace

__global__ __launch_bounds__(ANT) void k_adj_hl(AdjArgs A)
{
    // weights of Hz: x -2..+1, y -2..+1; of Hy: x -2..+1; of Hx: y -2..+1
    using TZ = ATile<2, 1, 2, 1>;
    using TY = ATile<2, 1, 0, 0>;
    using TX = ATile<0, 0, 2, 1>;
    __shared__ double sz[3][TZ::N], sy[3][TY::N], sx[3][TX::N];
    int x0, y0, k0, k1;
    if (!acol(A, x0, y0, k0, k1))
        return;
    const int lx = threadIdx.x % LX, ly = threadIdx.x / LX;
    const int i = x0 + lx, jj = y0 + ly;
    const bool valid = i < A.hi[0] && jj < A.hi[1];
    // idle lanes of a partial tile work on their row's last cell (in bounds)
    const int ci = min(i, A.hi[0] - 1), cj = min(jj, A.hi[1] - 1);
    const unsigned o = (unsigned)cj * A.row + (unsigned)ci * 8u;
    const size_t nb = (size_t)A.n * 8, pb = A.pb;
    const int xmax = min(x0 + LX, A.hi[0]), ymax = min(y0 + LY, A.hi[1]);
    const double c1 = A.c1, c2 = A.c2, rx = A.rdl[0], ry = A.rdl[1], rz = A.rdl[2];
    const int src_k = A.src_cell >= 0 ? A.src_cell / (int)(A.pb >> 3) : -1;
    const unsigned src_o = A.src_cell >= 0 ? (unsigned)(A.src_cell % (int)(A.pb >> 3)) * 8u : 0u;
    // own column's weights of Hy and Hx at planes k-2, k-1
    double yq2 = wcol(A, A.lH, A.uh, 1, k0 - 2, o), yq1 = wcol(A, A.lH, A.uh, 1, k0 - 1, o);
    double xq2 = wcol(A, A.lH, A.uh, 0, k0 - 2, o), xq1 = wcol(A, A.lH, A.uh, 0, k0 - 1, o);
    WTile<TZ, 2, 2> wz(A, A.lH, A.uh, 2, x0, y0, xmax, ymax);
    WTile<TY, 2, 0> wy(A, A.lH, A.uh, 1, x0, y0, xmax, ymax);
    WTile<TX, 0, 2> wx(A, A.lH, A.uh, 0, x0, y0, xmax, ymax);
    int b0 = 0, b1 = 1, b2 = 2;   // LDS buffers of planes k, k+1 and the one being filled
    wz.load(A, k0);
    wy.load(A, k0);
    wx.load(A, k0);
    wz.store(A, k0, sz[b0]);
    wy.store(A, k0, sy[b0]);
    wx.store(A, k0, sx[b0]);
    wz.load(A, k0 + 1);
    wy.load(A, k0 + 1);
    wx.load(A, k0 + 1);
    gmp lE = mb(A.lE) + (size_t)k0 * pb, grad = mb(A.grad) + (size_t)k0 * pb;
    gcp E0 = cb(A.E0) + (size_t)k0 * pb, E1 = cb(A.E1) + (size_t)k0 * pb, CB = cb(A.cbi) + (size_t)k0 * pb;
    double l0 = at(lE, o), l1 = at(lE + nb, o), l2 = at(lE + 2 * nb, o);
    // forward E after and before the step, dt/eps' and the gradient of the plane
    double p0 = at_s<true>(E1, o), p1 = at_s<true>(E1 + nb, o), p2 = at_s<true>(E1 + 2 * nb, o);
    double q0 = at_s<true>(E0, o), q1 = at_s<true>(E0 + nb, o), q2 = at_s<true>(E0 + 2 * nb, o);
    double cbv = at(CB, o), g0 = at(grad, o);
    for (int k = k0; k < k1; ++k) {
        wz.store(A, k + 1, sz[b1]);
        wy.store(A, k + 1, sy[b1]);
        wx.store(A, k + 1, sx[b1]);
        __syncthreads();
        const double f0 = p0 - q0, f1 = p1 - q1, f2 = p2 - q2, cc = cbv, gg = g0;
        const double m0 = l0, m1 = l1, m2 = l2;
        if (k + 1 < k1) {
            wz.load(A, k + 2);
            wy.load(A, k + 2);
            wx.load(A, k + 2);
            l0 = at(lE + pb, o);
            l1 = at(lE + pb + nb, o);
            l2 = at(lE + pb + 2 * nb, o);
            p0 = at_s<true>(E1 + pb, o);
            p1 = at_s<true>(E1 + pb + nb, o);
            p2 = at_s<true>(E1 + pb + 2 * nb, o);
            q0 = at_s<true>(E0 + pb, o);
            q1 = at_s<true>(E0 + pb + nb, o);
            q2 = at_s<true>(E0 + pb + 2 * nb, o);
            cbv = at(CB + pb, o);
            g0 = at(grad + pb, o);
        }
        const double *Z = sz[b0], *Y = sy[b0], *X = sx[b0];
        const int zc = (ly + 2) * TZ::W + lx + 2;
        const double z0 = Z[zc], zym1 = Z[zc - TZ::W], zyp1 = Z[zc + TZ::W], zym2 = Z[zc - 2 * TZ::W];
        const double zxm1 = Z[zc - 1], zxp1 = Z[zc + 1], zxm2 = Z[zc - 2];
        const int yc = ly * TY::W + lx + 2;
        const double y0v = Y[yc], yxm1 = Y[yc - 1], yxp1 = Y[yc + 1], yxm2 = Y[yc - 2];
        const double yzp1 = sy[b1][yc];
        const int xc = (ly + 2) * TX::W + lx;
        const double x0v = X[xc], xym1 = X[xc - TX::W], xyp1 = X[xc + TX::W], xym2 = X[xc - 2 * TX::W];
        const double xzp1 = sx[b1][xc];
        // D-_a of the weights of component d
        const double dxy = c1 * x0v - c1 * xym1 + c2 * xyp1 - c2 * xym2;
        const double dxz = c1 * x0v - c1 * xq1 + c2 * xzp1 - c2 * xq2;
        const double dyz = c1 * y0v - c1 * yq1 + c2 * yzp1 - c2 * yq2;
        const double dyx = c1 * y0v - c1 * yxm1 + c2 * yxp1 - c2 * yxm2;
        const double dzx = c1 * z0 - c1 * zxm1 + c2 * zxp1 - c2 * zxm2;
        const double dzy = c1 * z0 - c1 * zym1 + c2 * zyp1 - c2 * zym2;
        if (valid) {
            const double e0 = m0 + cc * (dyz * rz - dzy * ry), e1 = m1 + cc * (dzx * rx - dxz * rz),
                         e2 = m2 + cc * (dxy * ry - dyx * rx);
            put_s<false>(lE, o, e0);
            put_s<false>(lE + nb, o, e1);
            put_s<false>(lE + 2 * nb, o, e2);
            double g = e0 * f0 + e1 * f1 + e2 * f2;
            if (k == src_k && o == src_o) {
                const double le = A.src_comp == 0 ? e0 : (A.src_comp == 1 ? e1 : e2);
                A.grad_src[0] += le / cc * A.amp_n / A.sig_src;
                g += le * A.amp_n;
            }
            put_s<false>(grad, o, gg - g * A.rdt);
            rim(A, A.ue, i, jj, k, o, e0, e1, e2);
        }
        yq2 = yq1;
        yq1 = y0v;
        xq2 = xq1;
        xq1 = x0v;
        lE += pb;
        grad += pb;
        E0 += pb;
        E1 += pb;
        CB += pb;
        const int t = b0;
        b0 = b1;
        b1 = b2;
        b2 = t;
    }
}

__global__ __launch_bounds__(ANT) void k_adj_el(AdjArgs A)
{
    // weights of Ez: x -1..+2, y -1..+2; of Ey: x -1..+2; of Ex: y -1..+2
    using TZ = ATile<1, 2, 1, 2>;
    using TY = ATile<1, 2, 0, 0>;
    using TX = ATile<0, 0, 1, 2>;
    __shared__ double sz[4][TZ::N], sy[4][TY::N], sx[4][TX::N];
    int x0, y0, k0, k1;
    if (!acol(A, x0, y0, k0, k1))
        return;
    const int lx = threadIdx.x % LX, ly = threadIdx.x / LX;
    const int i = x0 + lx, jj = y0 + ly;
    const bool valid = i < A.hi[0] && jj < A.hi[1];
    const int ci = min(i, A.hi[0] - 1), cj = min(jj, A.hi[1] - 1);
    const unsigned o = (unsigned)cj * A.row + (unsigned)ci * 8u;
    const size_t nb = (size_t)A.n * 8, pb = A.pb;
    const int xmax = min(x0 + LX, A.hi[0]) + 1, ymax = min(y0 + LY, A.hi[1]) + 1;
    const double c1 = A.c1, c2 = A.c2, rx = A.rdl[0], ry = A.rdl[1], rz = A.rdl[2];
    // own column's weights of Ey and Ex at plane k-1
    double yq1 = wcol(A, A.lE, A.ue, 1, k0 - 1, o), xq1 = wcol(A, A.lE, A.ue, 0, k0 - 1, o);
    WTile<TZ, 1, 1> wz(A, A.lE, A.ue, 2, x0, y0, xmax, ymax);
    WTile<TY, 1, 0> wy(A, A.lE, A.ue, 1, x0, y0, xmax, ymax);
    WTile<TX, 0, 1> wx(A, A.lE, A.ue, 0, x0, y0, xmax, ymax);
    int b0 = 0, b1 = 1, b2 = 2, b3 = 3;   // planes k, k+1, k+2 (being filled), free
    for (int p = 0; p < 2; ++p) {
        const int bp = p == 0 ? b0 : b1;
        wz.load(A, k0 + p);
        wy.load(A, k0 + p);
        wx.load(A, k0 + p);
        wz.store(A, k0 + p, sz[bp]);
        wy.store(A, k0 + p, sy[bp]);
        wx.store(A, k0 + p, sx[bp]);
    }
    wz.load(A, k0 + 2);
    wy.load(A, k0 + 2);
    wx.load(A, k0 + 2);
    gmp lH = mb(A.lH) + (size_t)k0 * pb;
    const double dbi = A.dbi;
    double h0 = at(lH, o), h1 = at(lH + nb, o), h2 = at(lH + 2 * nb, o);
    for (int k = k0; k < k1; ++k) {
        wz.store(A, k + 2, sz[b2]);
        wy.store(A, k + 2, sy[b2]);
        wx.store(A, k + 2, sx[b2]);
        __syncthreads();
        const double m0 = h0, m1 = h1, m2 = h2;
        if (k + 1 < k1) {
            wz.load(A, k + 3);
            wy.load(A, k + 3);
            wx.load(A, k + 3);
            h0 = at(lH + pb, o);
            h1 = at(lH + pb + nb, o);
            h2 = at(lH + pb + 2 * nb, o);
        }
        const double *Z = sz[b0], *Y = sy[b0], *X = sx[b0];
        const int zc = (ly + 1) * TZ::W + lx + 1;
        const double z0 = Z[zc], zyp1 = Z[zc + TZ::W], zyp2 = Z[zc + 2 * TZ::W], zym1 = Z[zc - TZ::W];
        const double zxp1 = Z[zc + 1], zxp2 = Z[zc + 2], zxm1 = Z[zc - 1];
        const int yc = ly * TY::W + lx + 1;
        const double y0v = Y[yc], yxp1 = Y[yc + 1], yxp2 = Y[yc + 2], yxm1 = Y[yc - 1];
        const double yzp1 = sy[b1][yc], yzp2 = sy[b2][yc];
        const int xc = (ly + 1) * TX::W + lx;
        const double x0v = X[xc], xyp1 = X[xc + TX::W], xyp2 = X[xc + 2 * TX::W], xym1 = X[xc - TX::W];
        const double xzp1 = sx[b1][xc], xzp2 = sx[b2][xc];
        // D+_a of the weights of component d
        const double pxy = c1 * xyp1 - c1 * x0v + c2 * xyp2 - c2 * xym1;
        const double pxz = c1 * xzp1 - c1 * x0v + c2 * xzp2 - c2 * xq1;
        const double pyz = c1 * yzp1 - c1 * y0v + c2 * yzp2 - c2 * yq1;
        const double pyx = c1 * yxp1 - c1 * y0v + c2 * yxp2 - c2 * yxm1;
        const double pzx = c1 * zxp1 - c1 * z0 + c2 * zxp2 - c2 * zxm1;
        const double pzy = c1 * zyp1 - c1 * z0 + c2 * zyp2 - c2 * zym1;
        if (valid) {
            const double n0 = m0 + dbi * (pzy * ry - pyz * rz), n1 = m1 + dbi * (pxz * rz - pzx * rx),
                         n2 = m2 + dbi * (pyx * rx - pxy * ry);
            put_s<false>(lH, o, n0);
            put_s<false>(lH + nb, o, n1);
            put_s<false>(lH + 2 * nb, o, n2);
            rim(A, A.uh, i, jj, k, o, n0, n1, n2);
        }
        yq1 = y0v;
        xq1 = x0v;
        lH += pb;
        const int t = b0;
        b0 = b1;
        b1 = b2;
        b2 = b3;
        b3 = t;
    }
}

// rim weights of the H update from the region's lH: they do not outlive a replayed
// segment in uh
__global__ __launch_bounds__(256) void k_adj_rim(AdjArgs A)
{
    const unsigned w = (unsigned)(A.hi[0] - A.lo[0]), h = (unsigned)(A.hi[1] - A.lo[1]);
    const unsigned q = blockIdx.x * 256u + threadIdx.x, t = q / w;
    const int i = A.lo[0] + (int)(q - t * w), j = A.lo[1] + (int)(t % h), k = A.lo[2] + (int)(t / h);
    if (k >= A.hi[2])
        return;
    const bool inner = i >= A.lo[0] + 2 && i < A.hi[0] - 2 && j >= A.lo[1] + 2 && j < A.hi[1] - 2 &&
                       k >= A.lo[2] + 2 && k < A.hi[2] - 2;
    if (inner)
        return;
    const size_t nb = (size_t)A.n * 8;
    const gcp lH = cb(A.lH) + (size_t)k * A.pb;
    const unsigned o = (unsigned)j * A.row + (unsigned)i * 8u;
    rim(A, A.uh, i, j, k, o, at(lH, o), at(lH + nb, o), at(lH + 2 * nb, o));
}

hipError_t launch_adjoint_local(const AdjArgs &A, hipStream_t st)
{
    if (A.lb_pad > 0) {
        const unsigned cells = (unsigned)(A.hi[0] - A.lo[0]) * (unsigned)(A.hi[1] - A.lo[1]) *
                               (unsigned)(A.hi[2] - A.lo[2]);
        hipLaunchKernelGGL(k_adj_rim, dim3((cells + 255) / 256), dim3(256), 0, st, A);
    }
    hipLaunchKernelGGL(k_adj_cell<true>, dim3(A.fb_pad), dim3(PT), 0, st, A, 0, 1);
    return hipGetLastError();
}

hipError_t launch_adjoint_step(const AdjArgs &A, const double *g, int nrec, const int *rec,
                               bool next_local, hipStream_t st)
{
    if (nrec > 0) {
        hipLaunchKernelGGL(k_adj_inject, dim3((3 * nrec + 255) / 256), dim3(256), 0, st, A, g,
                           nrec, rec);
    }
    hipLaunchKernelGGL(k_adj_cell<false>, dim3(A.fb_pad), dim3(PT), 0, st, A, 1, 1);
    if (A.lb_pad > 0)
        hipLaunchKernelGGL(k_adj_hl, dim3(A.lb_pad), dim3(ANT), 0, st, A);
    hipLaunchKernelGGL(k_adj_cell<true>, dim3(A.fb_pad), dim3(PT), 0, st, A, 1, next_local ? 1 : 0);
    if (A.lb_pad > 0)
        hipLaunchKernelGGL(k_adj_el, dim3(A.lb_pad), dim3(ANT), 0, st, A);
    return hipGetLastError();
}

}  // namespace mt
