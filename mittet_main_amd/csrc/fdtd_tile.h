// fdtd_tile.h -- device helpers shared by the per-cell forward kernels
// (fdtd_kernels.hip) and the adjoint's (fdtd_adjoint.hip): global-memory and
// scalar loads, plane-relative addressing, and the tiles of a plane with their
// LDS layout and halo items.
#pragma once

#include "fdtd_dev.h"

// Pointers read out of the shot descriptor are generic; casting them to the
// global address space lets the compiler emit global_load/store instead of
// flat accesses (which also count against the LDS wait counter).
#define GLOBAL __attribute__((address_space(1)))

namespace mt {

__device__ __forceinline__ const GLOBAL double *gc(const double *p) { return (const GLOBAL double *)p; }
__device__ __forceinline__ GLOBAL double *gm(double *p) { return (GLOBAL double *)p; }
__device__ __forceinline__ const GLOBAL int *gc(const int *p) { return (const GLOBAL int *)p; }
__device__ __forceinline__ const GLOBAL double *gc(const GLOBAL double *p) { return p; }
__device__ __forceinline__ GLOBAL double *gm(GLOBAL double *p) { return p; }

// Field values each half-step reads or writes once (own E or H, coefficient,
// the updated field, psi).  With NT they are non-temporal, so they do not
// evict the stencil neighbours that other tiles still read from L2 and the
// Infinity Cache; the host sets NT only for launches whose fields do not fit
// that cache anyway.
template <bool NT> __device__ __forceinline__ double ld_s(const GLOBAL double *p)
{
    if constexpr (NT)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}
template <bool NT> __device__ __forceinline__ void st_s(GLOBAL double *p, double v)
{
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

// A wave-uniform double (a z-profile value of the current plane) through the
// scalar cache.  A vector load issued after a plane's prefetch would make the
// wait for it also wait for every prefetch load issued before it.
__device__ __forceinline__ double uload(const double *p)
{
    return *(const __attribute__((address_space(4))) double *)p;
}

// Addresses of the per-cell kernels.  A block's cells lie in one plane, so every
// access is a wave-uniform base (component and plane, scalar arithmetic) plus a
// 32-bit byte offset within the plane: one scalar-base load instruction, no
// 64-bit vector arithmetic per access.  A grid below 2^31 cells has at least 8
// planes (two CPML shells of 2 cells and 4 more), so a plane is below 2^31
// bytes.
typedef const GLOBAL char *gcp;
typedef GLOBAL char *gmp;
__device__ __forceinline__ gcp cb(const void *p) { return (gcp)p; }
__device__ __forceinline__ gmp mb(void *p) { return (gmp)p; }
__device__ __forceinline__ double at(gcp b, unsigned o, int d = 0)
{
    return *(const GLOBAL double *)(b + o + d);
}
template <bool NT> __device__ __forceinline__ double at_s(gcp b, unsigned o)
{
    return ld_s<NT>((const GLOBAL double *)(b + o));
}
template <bool NT> __device__ __forceinline__ void put_s(gmp b, unsigned o, double v)
{
    st_s<NT>((GLOBAL double *)(b + o), v);
}

__device__ __forceinline__ int uload(const int *p)
{
    return *(const __attribute__((address_space(4))) int *)p;
}
namespace {

// Tile of a block, the same for its lanes: rows [y0, yend) x columns [x0, x0 + w)
// of plane k, th = rows of lanes
struct FTile {
    int x0, y0, k, w, h, yend;
    bool region;   // may hold cells of the LDS kernels' region
};

// Order of the tiles.  Blocks go to the XCDs in turn (block b to XCD b mod 8).
// Without a list, each XCD owns a contiguous run of planes: what a launch wrote is
// then in the L2 that the next one reads it from (84^3: 16.7 us a launch, in layers
// 17.4).  LAYERS (the launches with non-temporal fields, which pass through the
// caches anyway): all XCDs work on the same planes, each on its eighth of the
// plane's tiles, so that what their stencils share is read about when it is in the
// Infinity Cache, and each XCD gets the same part of the costly CPML planes (four
// shots of 84^3 to 120^3: 127 us a launch with runs, 117 in layers).  Eighths of a
// plane move on by one XCD every 8 planes: an XCD that kept the y faces' tiles
// through all planes would finish last (132 us).  The shell list has this order too
// (complement_tiles).
template <bool LAYERS, class G> __device__ __forceinline__ bool ftile(const G &S, int b, FTile &T)
{
    if (!S.shell) {
        if constexpr (LAYERS) {
            const unsigned m = (unsigned)b >> 3, tpp = (unsigned)(S.ftx * S.fty), e = (tpp + 7u) >> 3;
            T.k = (int)(((unsigned long long)m * S.emul) >> S.esh);   // m / e
            const unsigned r = ((b + (T.k >> 3)) & 7) * e + (m - (unsigned)T.k * e);
            if (T.k >= S.iz || r >= tpp)
                return false;
            const unsigned ty = (unsigned)(((unsigned long long)r * S.fmul) >> S.fsh);   // r / ftx
            T.w = ZX;
            T.h = ZY;
            T.x0 = (int)(r - ty * S.ftx) * ZX;
            T.y0 = (int)ty * ZY;
        } else {
            const unsigned q = (b & 7) * (S.fb_pad >> 3) + (b >> 3);
            if (q >= (unsigned)S.fb)
                return false;
            T.k = (int)(((unsigned long long)q * S.tmul) >> S.tsh);
            const unsigned r = q - (unsigned)T.k * S.tpp;
            const unsigned ty = (unsigned)(((unsigned long long)r * S.xmul) >> S.xsh);
            T.w = S.tw;
            T.h = S.th;
            T.x0 = (int)(r - ty * S.ttx) * T.w;
            T.y0 = (int)ty * T.h;
        }
        T.yend = S.iy;
        T.region = false;
        return true;
    }
    if (b >= S.fb)
        return false;
    const int *t = (const int *)(S.shell + b);   // {x0, y0, k, yend}
    T.x0 = uload(t);
    T.y0 = uload(t + 1);
    T.k = uload(t + 2);
    const int yend = uload(t + 3);
    T.w = yend ? 16 : ZX;
    T.h = yend ? 16 : ZY;
    T.yend = yend ? yend : S.iy;
    T.region = !yend && T.k >= S.lo[2] && T.k < S.hi[2];
    return T.k >= 0;
}

// A lane's cell in its tile, its LDS position (pitch w + 3, two cells before
// the tile for E, one for H) and its halo item.  LO cells before the tile and
// 3 - LO after it on each axis, two arrays with halo rows and two with halo
// columns (hk: 0 and 1 the rows of the first and second, 2 and 3 the columns).
template <int LO> struct FLane {
    int i, jj;
    unsigned o;        // byte offset of the (clamped) cell in its plane
    unsigned a, p;     // LDS byte address of the cell, pitch in bytes
    bool own;          // the lane's cell is one of the tile's
    bool halo;         // the lane has a halo item
    int hk;            // its array
    bool hin;          // it lies in the grid
    int hx, hy;        // its cell, clamped into the grid
    unsigned ho, ha;   // its plane offset and LDS byte address in its array
    template <class G> __device__ __forceinline__ FLane(const G &S, const FTile &T)
    {
        const int t = threadIdx.x, w = T.w, h = T.h;
        const unsigned wm = (65535u + w) / (unsigned)w;   // t / w = t wm >> 16 for t < 256, w <= PT_WH
        const int ly = (int)((t * wm) >> 16), lx = t - ly * w;
        p = (unsigned)(w + 3) * 8u;
        i = T.x0 + lx;
        jj = T.y0 + ly;
        own = ly < h;
        o = (unsigned)min(jj, S.iy - 1) * S.row + (unsigned)min(i, S.ix - 1) * 8u;
        a = (unsigned)(ly + LO) * p + (unsigned)(lx + LO) * 8u;
        int u, v;   // halo position relative to the tile
        if (t < 6 * w) {
            const bool second = t >= 3 * w;
            const int m = second ? t - 3 * w : t;
            const int r = (int)((m * wm) >> 16);
            u = m - r * w;
            v = r < LO ? r - LO : h + r - LO;
            hk = second ? 1 : 0;
        } else {
            int m = t - 6 * w;
            const bool second = m >= 3 * h;
            m = second ? m - 3 * h : m;
            v = (m * 21846) >> 16;   // m / 3
            const int r = m - 3 * v;
            u = r < LO ? r - LO : w + r - LO;
            hk = second ? 3 : 2;
        }
        halo = t < 6 * (w + h);
        hx = min(max(T.x0 + u, 0), S.ix - 1);
        hy = min(max(T.y0 + v, 0), S.iy - 1);
        hin = hx == T.x0 + u && hy == T.y0 + v;
        ho = (unsigned)hy * S.row + (unsigned)hx * 8u;
        ha = (unsigned)(v + LO) * p + (unsigned)(u + LO) * 8u;
    }
};

// r in [a, b) U [c, d): an axis' CPML face (a superset of a cell's face flag, so
// psi loads need not wait for the flag words)
__device__ __forceinline__ bool in_face(int r, int a, int b, int c, int d)
{
    return (r >= a && r < b) || (r >= c && r < d);
}
__device__ __forceinline__ double lds_at(const double *b, unsigned o, int d = 0)
{
    return *(const double *)((const char *)b + o + d);
}
__device__ __forceinline__ void lds_put(double *b, unsigned o, double v)
{
    *(double *)((char *)b + o) = v;
}

__device__ __forceinline__ int find_shot(const int *__restrict__ pre, int ns, int b)
{
    int s = 0;
    while (s + 1 < ns && b >= pre[s + 1])
        ++s;
    return s;
}

// slab position of index r on an axis of length n with nc-cell shells
__device__ __forceinline__ int slab_pos(int r, int n, int nc)
{
    return r < nc ? r : r - (n - 2 * nc);
}

// Absolute step of local index 0 of the current chunk.  Every lane of a launch
// reads the same word, which the previous chunk's k_advance wrote: a scalar
// load through the constant address space serves it from the scalar cache
// instead of a vector round trip to L2 per wave.
__device__ __forceinline__ int chunk_step(const ShotDev &S)
{
    return *(const __attribute__((address_space(4))) int *)S.step;
}

// ring slot q of a descriptor, q < 2 * ring (or any q when there is one slot)
__device__ __forceinline__ int ring_slot(const ShotDev &S, int q)
{
    return S.ring == 1 ? 0 : (q >= S.ring ? q - S.ring : q);
}

// An axis' sigma, kappa*dl, b and c: of a lane's x or y index (rows, so that
// neighbouring lanes read neighbouring words), or of one index for the whole
// wave (a record, scalar loads)
struct Quad {
    double s, k, b, c;
};
template <bool H> __device__ __forceinline__ Quad quad(const double *prof, int n, int r)
{
    const gcp p = cb(prof);
    const unsigned o = (unsigned)r * 8u, m = (unsigned)n * 8u;
    return {at(p, o + m * (H ? PR_MSIG : PR_ESIG)), at(p, o + m * (H ? PR_KHD : PR_KED)),
            at(p, o + m * (H ? PR_BH : PR_BE)), at(p, o + m * (H ? PR_CH : PR_CE))};
}
template <bool H> __device__ __forceinline__ Quad uquad(const double *cq, int r)
{
    const double *p = cq + (size_t)r * CQ_N + (H ? CQ_H : CQ_E);
    return {uload(p), uload(p + 1), uload(p + 2), uload(p + 3)};
}

// D- and D+ of the fourth-order stencil: f0 at the cell, fp1 one cell up and so on
__device__ __forceinline__ double dm(double f0, double fm1, double fp1, double fm2, double c1,
                                     double c2)
{
    return c1 * f0 - c1 * fm1 + c2 * fp1 - c2 * fm2;
}
__device__ __forceinline__ double dp(double fp1, double f0, double fp2, double fm1, double c1,
                                     double c2)
{
    return c1 * fp1 - c1 * f0 + c2 * fp2 - c2 * fm1;
}

// Component of a halo item: components 2 and 0 have halo rows, 2 and 1 columns
__device__ __forceinline__ int halo_comp(int hk) { return hk == 1 ? 0 : (hk == 3 ? 1 : 2); }

}  // namespace

}  // namespace mt
